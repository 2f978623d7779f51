"""The split form's walk either side of the particle count where its groups go
from 16 to 64 targets, against the oracle."""
import pytest

from test_gpu_walk_groups import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [262144, 262145])
def test_split_form_group_limit(ag2, orc, n):
    nh, nd = n // 2, (3 * n) // 10
    check(ag2, orc, ag2.ics.disk_galaxy(nh, nd, n - nh - nd, seed=2), 0.5, ag2.engine.AG2_FP32_SPLIT)
