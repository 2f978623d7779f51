// What tests/test_transfer_ring.py drives of csrc/ring.h.
#include <cerrno>
#include <cstdint>
#include <stdexcept>
#include <system_error>

#include "ring.h"

using ag2::Ring;
using ag2::Run;

// A transfer's ring (ring.h) between `runs` host arrays of `each` bytes and a
// device of memory copies that complete `late` polls after they are queued.
// threads: helpers that can be had before starting one fails; fail: the piece
// whose completion is an error (-1: none), as its copy queues (how 0), is polled
// or waited for (1).  Returns 0, or -1 where the error came up; *had: helpers.
struct CopyDevice {
    char *block, *slots;
    const Ring<CopyDevice> *ring = nullptr;
    bool down;
    int late, fail, how;
    std::vector<int> polls;
    void copy(int p) {
        if (down) std::memcpy(ring->slot(p), block + ring->off(p), ring->len(p));
        else std::memcpy(block + ring->off(p), ring->slot(p), ring->len(p));
    }
    void issue(int p) {
        if (p == fail && how == 0) throw std::runtime_error("issue");
        polls.push_back(late);
    }
    void wait(int p) {
        if (p == fail && how == 1) throw std::runtime_error("wait");
        copy(p);
    }
    bool left(int p) {
        if (p == fail && how == 1) throw std::runtime_error("left");
        if (polls[(size_t)p]-- > 0) return false;
        copy(p);
        return true;
    }
};

extern "C" int ring_copy(int runs, int64_t each, char *host, char *block, int down, int64_t piece, int n_slots,
                             int helpers, int threads, int late, int fail, int how, int *had) {
    std::vector<Run> r;
    for (int k = 0; k < runs; k++) r.push_back({host + (size_t)k * (size_t)each, (size_t)each});
    std::vector<char> slots((size_t)piece * (size_t)n_slots);
    CopyDevice dev{block, slots.data(), nullptr, down != 0, late, fail, how, {}};
    int started = 0;
    try {
        Ring<CopyDevice> ring(dev, slots.data(), n_slots, (size_t)piece, r, (size_t)runs * (size_t)each, down != 0,
                              helpers, [&](std::function<void()> f) {
                                  if (started >= threads) throw std::system_error(EAGAIN, std::generic_category());
                                  started++;
                                  return std::thread(std::move(f));
                              });
        dev.ring = &ring;
        *had = ring.helpers();
        ring.run();
        // copies still on their way when the last one had been queued
        if (!down)
            for (size_t p = 0; p < dev.polls.size(); p++)
                if (dev.polls[p] >= 0) dev.copy((int)p);
    } catch (const std::runtime_error &) {
        return -1;
    }
    return 0;
}

// A lease that ends whole or early, with room on the shelf or not: what became
// of its buffer, as decimal digits in order (1 taken, 2 drained, 3 kept, 4 destroyed).
extern "C" int lease_steps(int whole, int room) {
    struct Ops {
        int *log, room;
        void note(int d) { *log = *log * 10 + d; }
        int take() { note(1); return 7; }
        void drain() { note(2); }
        bool keep(int) {
            if (room) note(3);
            return room != 0;
        }
        void destroy(int) { note(4); }
    };
    int log = 0;
    try {
        ag2::Lease<int, Ops> lease(Ops{&log, room});
        if (!whole) throw std::runtime_error("a copy failed");
        lease.whole();
    } catch (const std::runtime_error &) {
    }
    return log;
}
