"""Decode rows at heads of 32 and 64: whole contexts in one workgroup where a block table holds at most
256 keys, partitions and a merge beyond, both against the CPU oracle (the tolerance of the other head
widths), at contexts around a tile, around the sixteen waves of a workgroup, and at none."""
import numpy as np
import pytest

from tests import workloads
from tests.gpu_harness import PagedAttnRunner
from tests.test_gpu_decode_step import _rel_l2, _run_both
from tests.test_gpu_paged_attn_head_dims import _check

pytestmark = pytest.mark.gpu

CTX = [1, 15, 16, 17, 31, 33, 127, 128, 129, 240, 255, 256]


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("hq,hkv", [(14, 2), (3, 3), (16, 1), (32, 4), (5, 1)])
@pytest.mark.parametrize("blocks", [16, 17])  # whole contexts, partitions
def test_contexts(d, hq, hkv, blocks):
    rng = np.random.default_rng(d + hq)
    c = workloads.paged_case(rng, np.ones(len(CTX), np.int32), np.array(CTX) - 1, hq=hq, hkv=hkv, d=d,
                             min_max_blocks=blocks)
    _check(c, what=f"{hq}/{hkv} x {d}, {blocks} blocks")


def test_a_context_of_no_keys():
    rng = np.random.default_rng(3)
    c = workloads.paged_case(rng, [1, 1, 1], [20, 0, 5], hq=14, hkv=2, d=64)
    c["context_lens"] = np.array([21, 0, 6], c["context_lens"].dtype)
    r = PagedAttnRunner(c)
    r.launch()
    got = r.result().reshape(3, -1)
    assert not np.any(got[1]) and np.any(got[0]) and np.any(got[2])


@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (4, 2, 32), (6, 3, 64), (8, 1, 64)])
@pytest.mark.parametrize("rows", [1, 5, 17, 40])
@pytest.mark.parametrize("longest", [200, 700])  # whole contexts, partitions
def test_as_the_next_operand(hq, hkv, d, rows, longest):
    # the step's o projection reads the prepared layout that the attention or the merge writes (or,
    # where a workgroup's heads are no whole groups of 128 columns, rows prepared behind it)
    rng = np.random.default_rng(hq * 10 + rows)
    cfg, layers, batch = workloads.decode_step_problem(
        rng, num_layers=1, hidden=256, hq=hq, hkv=hkv, d=d, inter=384, ctx=np.append(rng.integers(1, longest, size=rows - 1), longest))
    _, got, want, _, _ = _run_both(cfg, layers, batch)
    assert _rel_l2(got, want) < 6e-3  # the decode batch's bound (tests/test_gpu_decode_step.py)
