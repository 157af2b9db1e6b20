"""Decode rows of many sequences at heads of 32 and 64 and short block tables, on both sides of the line
between whole contexts in one workgroup and partitions with their merge (one workgroup per compute unit;
beyond it by the table, the width and the KV heads), against the CPU oracle (the tolerance of the other
head widths)."""
import numpy as np
import pytest

from tests import workloads
from tests.test_gpu_paged_attn_head_dims import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seqs,hq,hkv,d,blocks", [
    (64, 8, 8, 64, 16), (65, 8, 8, 64, 16),          # at the line, and one sequence more
    (260, 4, 4, 32, 8), (260, 4, 4, 32, 7),          # heads of 32: tables of 128 keys and of 112
    (257, 6, 2, 64, 16), (257, 6, 2, 64, 3),         # two KV heads
    (90, 6, 3, 64, 8), (90, 4, 4, 64, 8), (300, 5, 5, 64, 8),
])
def test_many_sequences(seqs, hq, hkv, d, blocks):
    rng = np.random.default_rng(seqs + hkv)
    ctx = rng.integers(1, 16 * blocks + 1, size=seqs)
    ctx[:3] = 16 * blocks, 1, 16 * blocks - 1
    c = workloads.paged_case(rng, np.ones(seqs, np.int32), ctx - 1, hq=hq, hkv=hkv, d=d,
                             min_max_blocks=blocks)
    _check(c, what=f"{seqs} x {hq}/{hkv} x {d}, {blocks} blocks")
