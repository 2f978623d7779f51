"""The ring of a large transfer (csrc/ring.h) on the CPU, its device one of
memory copies: whole blocks both ways with any number of helpers, threads that
cannot be had, and errors of the device, each of which has to come up (and not
leave the caller waiting, or a thread behind)."""
import ctypes as C
import os
import subprocess
import threading

import numpy as np
import pytest

from conftest import PKG_DIR, ROOT


@pytest.fixture(scope="module")
def ring(tmp_path_factory):
    so = os.path.join(str(tmp_path_factory.mktemp("ring")), "core.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-pthread", "-I",
                    os.path.join(PKG_DIR, "csrc"), "-o", so, os.path.join(ROOT, "tests", "transfer_ring.cpp")], check=True)
    lib = C.CDLL(so)

    def run(runs, each, down, helpers, threads, late=0, fail=-1, how=0, piece=4096, slots=8):
        g = np.random.default_rng(runs * each + down)
        data = g.integers(0, 256, runs * each, dtype=np.uint8)
        src, dst = data.copy(), np.zeros_like(data)
        host, block = (dst, src) if down else (src, dst)
        had = C.c_int(-1)
        p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
        rc = lib.ring_copy(runs, C.c_int64(each), p(host), p(block), int(down), C.c_int64(piece), slots, helpers,
                               threads, late, fail, how, C.byref(had))
        return rc, had.value, np.array_equal(dst, data)
    run.lib = lib
    return run


@pytest.mark.parametrize("down", [0, 1])
@pytest.mark.parametrize("runs,each", [(1, 4097), (3, 1000), (11, 8000), (19, 24593), (2, 200000)])
@pytest.mark.parametrize("helpers,threads", [(0, 0), (3, 0), (3, 1), (3, 2), (3, 3)])
def test_whole_blocks(ring, runs, each, down, helpers, threads):
    """... with fewer threads than asked for the rest of them and the caller do."""
    for late in (0, 3):
        rc, had, same = ring(runs, each, down, helpers, threads, late)
        assert rc == 0 and same
        assert had == min(helpers, threads)


@pytest.mark.timeout(60)
@pytest.mark.parametrize("down", [0, 1])
@pytest.mark.parametrize("how", [0, 1])
@pytest.mark.parametrize("fail", [0, 1, 7, 8, 30])
@pytest.mark.parametrize("threads", [0, 3])
def test_errors_come_up(ring, down, how, fail, threads):
    before = threading.active_count(), len(os.listdir("/proc/self/task"))
    rc, _, _ = ring(16, 16384, down, 3, threads, 2, fail, how)   # 64 pieces
    assert rc == -1
    assert (threading.active_count(), len(os.listdir("/proc/self/task"))) == before


def test_a_buffer_left_early_is_not_kept(ring):
    """Copies may still be under way in the buffer of a transfer that failed."""
    assert ring.lib.lease_steps(1, 1) == 13
    assert ring.lib.lease_steps(1, 0) == 14
    assert ring.lib.lease_steps(0, 1) == 124
    assert ring.lib.lease_steps(0, 0) == 124
