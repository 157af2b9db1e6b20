"""Prompt chunks at 64-wide heads on every side of the rule that gives a launch to the general kernel or
to one of the chunk kernel's splits: one KV head (or an odd number in a workgroup) at long block tables,
many chunks of one tile of 16 columns, tables of one and of two tiles of keys, one round of workgroups and
more, all beside decode rows; against the CPU oracle (the tolerance of the other head widths)."""
import numpy as np
import pytest

from tests import workloads
from tests.test_gpu_paged_attn_head_dims import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("new,prior,hq,hkv,blocks", [
    ([20, 1], [100, 30], 8, 1, 32), ([20, 1], [100, 30], 8, 1, 33),   # one KV head: tables of 512 keys, 528
    ([700], [0], 8, 1, 50), ([20, 2], [70, 9], 5, 5, 40),             # ... more tiles than units; five heads
    ([2] * 32, [20] * 32, 8, 8, 8), ([2] * 33, [20] * 33, 8, 8, 8),   # chunks of one tile, 256 and 264
    ([3] * 33, [20] * 33, 64, 8, 8),                                  # ... of two tiles
    ([40, 1, 9], [24, 60, 3], 14, 2, 4), ([40, 1, 9], [24, 60, 3], 14, 2, 5),   # one tile of keys, two
    ([100, 1], [28, 5], 14, 2, 8), ([100, 1], [28, 5], 14, 2, 9),     # ... two, three
    ([512], [10], 16, 16, 40), ([544], [10], 16, 16, 40),             # a round of workgroups, more
    ([30] * 40, [50] * 40, 8, 8, 8),                                  # no column beyond 32
])
def test_rule(new, prior, hq, hkv, blocks):
    rng = np.random.default_rng(sum(new) + hq)
    c = workloads.paged_case(rng, new, prior, hq=hq, hkv=hkv, d=64, min_max_blocks=blocks)
    _check(c, what=f"{len(new)} x {new[0]}, {hq}/{hkv}, {blocks} blocks")
