"""Decode rows at heads of 32 and 64: the merge (or the whole-context kernel) that writes the o projection's
operand itself gives the bits of the rows and the operator that prepares them, which a step takes whose
batch is declared to hold chunks (max_seqlen_q 2, and none is there)."""
import numpy as np
import pytest

from tests import workloads
from tests.gpu_harness import DecodeStepRunner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (8, 2, 32), (16, 1, 64)])
@pytest.mark.parametrize("rows,longest", [
    (2, 4000), (5, 700), (17, 130),  # a static split: many partitions, some, a whole context each
    (40, 3000),                      # workers with equal shares (at two KV heads)
])
@pytest.mark.parametrize("empty", [False, True])
def test_same_bits_as_prepared_rows(hq, hkv, d, rows, longest, empty):
    rng = np.random.default_rng(rows + hq)
    ctx = rng.integers(1, longest, size=rows)
    ctx[-1] = longest
    cfg, layers, batch = workloads.decode_step_problem(rng, num_layers=1, hidden=256, hq=hq, hkv=hkv, d=d,
                                                       inter=384, ctx=ctx)
    if empty:
        batch["context_lens"][0] = 0
    got = []
    for max_q in (1, 2):
        r = DecodeStepRunner(cfg, layers, batch)
        r.batch.total_tokens, r.batch.max_seqlen_q = rows, max_q
        r.launch()
        got.append((r.result_bits(), r.h.to_numpy(np.uint32, (rows, cfg["hidden"]))))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
