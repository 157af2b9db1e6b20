"""The step's fused few-row projections (up to 16 packed rows) against the oracle at the edges of
their dispatch: 1 to 17 rows (17 is the other path), one to 32 groups of K per projection,
shares of K that do not divide by the waves, heads of 32 to 256, a bias, 3-bit pools, a chunk."""
import numpy as np
import pytest

import oracle as O
from tests import workloads
from tests.gpu_harness import DecodeStepRunner
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


def _tie_gain(a, odd):
    """A gain whose fp32 product with `a` lies exactly between two bf16 values, the lower of which
    is odd (the product rounds up, one step less rounds down) or even (the other way round)."""
    a = np.float32(a)
    for lower in range(0x3f40 + odd, 0x3fc0, 2):
        tie = np.array([(lower << 16) | 0x8000], np.uint32).view(np.float32)[0] * np.sign(a)
        g = np.float32(tie / a)
        for _ in range(4):
            g = np.nextafter(g, np.float32(0))
        for _ in range(9):
            if a * g == tie:
                return g
            g = np.nextafter(g, np.float32(np.inf))
    raise AssertionError("no gain found")


@pytest.mark.parametrize("rows", [1, 3, 8, 16, 17])
@pytest.mark.parametrize("hidden", [384, 896, 1536, 2176, 4096])
def test_norm_to_the_last_bit(rows, hidden):
    # 1 / sqrt(mean + eps) with every operation rounded once: whole numbers whose sum of squares is
    # exact in any order, one gain per group of K that puts a value halfway between two bf16 ones,
    # and value-projection rows that read one column each.  A last bit more or less in the root,
    # the mean or the reciprocal turns about half of the values over.
    for trial in range(6):
        rng = np.random.default_rng(100 * hidden + trial)
        cfg, layers, batch = workloads.decode_step_problem(
            rng, num_layers=1, hidden=hidden, hq=1, hkv=1, inter=128, ctx=[5] * rows)
        h = rng.integers(1, 9, size=hidden).astype(np.float32) * rng.choice([-1, 1], hidden)
        h = (h * np.float32(2.0) ** rng.integers(-3, 4)).astype(np.float32)
        total = np.float32((h.astype(np.float64) ** 2).sum())
        inv = np.float32(1) / np.sqrt(total / np.float32(hidden) + np.float32(cfg["eps"]))
        groups = hidden // 128
        col = 128 * np.arange(groups) + rng.integers(0, 128, groups)
        gains = np.zeros(hidden, np.float32)
        for i, c in enumerate(col):
            gains[c] = _tie_gain(h[c] * inv, i & 1)
        want = O.bf16_bits_to_f32(O.f32_to_bf16_bits(h[col] * inv * gains[col]))
        q = np.zeros((3 * 128, hidden), np.uint8)
        q[256 + np.arange(groups), col] = 1
        scale = np.zeros((3 * 128, groups), np.float16)
        scale[256:] = 1
        layers[0]["qkv"] = (q[:, 0::2] | (q[:, 1::2] << 4), scale, np.zeros_like(scale))
        layers[0]["norm1"] = gains
        batch["h"][:] = h
        r = DecodeStepRunner(cfg, layers, batch)
        r.launch()
        r.result_bits()
        pool = r.pools[0][1].to_numpy(np.float16, layers[0]["v_pool"].shape)
        got = pool[np.asarray(batch["slots"])][:, :groups].astype(np.float32)
        assert np.array_equal(got, np.broadcast_to(want, got.shape)), trial
