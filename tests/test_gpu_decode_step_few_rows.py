"""The step's fused few-row projections (up to 16 packed rows) against the oracle at the edges of
their dispatch: 1 to 17 rows (17 is the other path), one to 32 groups of K per projection,
shares of K that do not divide by the waves, heads of 32 to 256, a bias, 3-bit pools, a chunk."""
import numpy as np
import pytest

from tests import workloads
from tests.test_gpu_decode_step import _rel_l2, _run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("hidden,hq,hkv,d,inter", [
    (128, 1, 1, 128, 128),      # one group of K everywhere
    (896, 14, 2, 64, 4864),     # 7 and 38 groups, tiles that do not fill the last workgroup
    (1152, 8, 4, 96, 2176),     # 9, 6 and 17 groups
    (2176, 17, 17, 128, 1152),  # 17 groups of the norm, one KV head per query head
])
def test_rows_and_widths(rows, hidden, hq, hkv, d, inter):
    rng = np.random.default_rng(1000 * rows + hidden)
    ctx = rng.integers(1, 90, size=rows)
    cfg, layers, batch = workloads.decode_step_problem(
        rng, num_layers=1, hidden=hidden, hq=hq, hkv=hkv, d=d, inter=inter, ctx=ctx,
        qkv_bias=bool(rows & 1))
    r, got, want, lay, bat = _run_both(cfg, layers, batch)
    # one layer: the decode batch's bounds (tests/test_gpu_decode_step.py)
    assert _rel_l2(got, want) < 6e-3
    assert np.all(np.abs(got - want) <= 1.5e-2 + 2e-2 * np.abs(want))
    assert _rel_l2(r.h.to_numpy(np.float32, bat["h"].shape), bat["h"]) < 6e-3
    for (kp, vp), L in zip(r.pools, lay):
        for buf, ref in ((kp, L["k_pool"]), (vp, L["v_pool"])):
            diff = np.abs(buf.to_numpy(np.float16, ref.shape).astype(np.float32)
                          - ref.astype(np.float32))
            assert np.all((diff <= 4e-3) | (diff <= 1e-2 * np.abs(ref.astype(np.float32))))


@pytest.mark.parametrize("rows", [1, 16])
def test_widest_norm(rows):
    rng = np.random.default_rng(77 + rows)
    cfg, layers, batch = workloads.decode_step_problem(
        rng, num_layers=1, hidden=4096, hq=8, hkv=2, inter=8960, ctx=rng.integers(1, 60, size=rows))
    _, got, want, _, _ = _run_both(cfg, layers, batch)
    assert _rel_l2(got, want) < 6e-3
    assert np.all(np.abs(got - want) <= 1.5e-2 + 2e-2 * np.abs(want))


def test_three_bit_pools_and_a_chunk():
    rng = np.random.default_rng(78)
    cfg, layers, batch = workloads.decode_step_problem(
        rng, num_layers=1, hidden=512, hq=4, hkv=2, inter=1024, ctx=[40, 9, 77], kv_turbo3=True)
    _, got, want, _, _ = _run_both(cfg, layers, batch)
    assert _rel_l2(got, want) < 1e-2  # the bound of the steps over 3-bit pools
    cfg, layers, batch = workloads.decode_step_problem(
        rng, num_layers=1, hidden=512, hq=4, hkv=2, inter=1024, ctx=[40, 21, 77],
        new_tokens=[1, 13, 1])
    _, got, want, _, _ = _run_both(cfg, layers, batch)
    assert _rel_l2(got, want) < 6e-3


def test_sum_of_squares_past_fp32():
    # a row whose sum of squares overflows: its norm is 0 (1 / sqrt(inf)), not a NaN, so that the
    # layer adds nothing to that row; the other row is untouched by it
    rng = np.random.default_rng(79)
    cfg, layers, batch = workloads.decode_step_problem(
        rng, num_layers=1, hidden=512, hq=4, hkv=2, inter=1024, ctx=[1, 9])
    batch["h"][0] = np.float32(1e20)
    with np.errstate(over="ignore"):
        r, got, want, _, bat = _run_both(cfg, layers, batch)
    h = r.h.to_numpy(np.float32, bat["h"].shape)
    assert np.all(got[0] == 0) and np.all(h[0] == np.float32(1e20))
    assert _rel_l2(got[1], want[1]) < 6e-3
