"""Steps of 33 to 96 packed rows: every operator takes all rows in one launch, the projections in
chunks of 32 rows side by side, the last one with 1 to 32 rows.  Against the oracle, on each of the
projection kernels (x in registers: K a multiple of 2048; streaming: 8 groups and many tiles; split
over K: the rest), with decode rows, chunks, and 3-bit pools (whose last chunk of up to 16 rows stays
by itself when there are chunks)."""
import numpy as np
import pytest

from logismos_amd import hip
from tests import workloads
from tests.gpu_harness import DecodeStepRunner
from tests.test_gpu_decode_step import _rel_l2, _run_both

pytestmark = pytest.mark.gpu

WIDTHS = [
    (2048, 16, 4, 128, 2048),   # x in registers
    (1024, 8, 2, 128, 16384),   # streaming gate/up projection, x in registers behind it
    (896, 14, 2, 64, 1152),     # 7 and 9 groups, heads of 64
    (384, 3, 1, 128, 640),      # fewer rows than a workgroup takes
]


def _check(cfg, layers, batch, rel, kv_ok=True):
    r, got, want, lay, bat = _run_both(cfg, layers, batch)
    assert _rel_l2(got, want) < rel
    assert _rel_l2(r.h.to_numpy(np.float32, bat["h"].shape), bat["h"]) < rel
    return got, want


@pytest.mark.parametrize("rows", [33, 34, 48, 49, 64, 65, 96])
@pytest.mark.parametrize("hidden,hq,hkv,d,inter", WIDTHS)
def test_decode_rows(rows, hidden, hq, hkv, d, inter):
    rng = np.random.default_rng(rows * 7 + hidden)
    cfg, layers, batch = workloads.decode_step_problem(
        rng, num_layers=2, hidden=hidden, hq=hq, hkv=hkv, d=d, inter=inter,
        ctx=rng.integers(1, 60, size=rows), qkv_bias=bool(rows & 1))
    # the decode batch's bounds (tests/test_gpu_decode_step.py), two layers
    got, want = _check(cfg, layers, batch, 8e-3)
    assert np.all(np.abs(got - want) <= 2e-2 + 3e-2 * np.abs(want))


@pytest.mark.parametrize("new", [[1, 31, 1], [20, 1, 1, 30], [1, 64, 1, 1]])
@pytest.mark.parametrize("hidden,hq,hkv,d,inter", WIDTHS[:3])
def test_chunks_beside_decode_rows(new, hidden, hq, hkv, d, inter):
    rng = np.random.default_rng(sum(new) + hidden)
    cfg, layers, batch = workloads.decode_step_problem(
        rng, num_layers=2, hidden=hidden, hq=hq, hkv=hkv, d=d, inter=inter,
        ctx=[n + 9 * i for i, n in enumerate(new)], new_tokens=new)
    got, want = _check(cfg, layers, batch, 8e-3)
    assert np.all(np.abs(got - want) <= 2e-2 + 3e-2 * np.abs(want))


@pytest.mark.parametrize("new", [[1] * 40, [1, 30, 2, 4], [1, 40, 20]])  # one pass, two, one
def test_three_bit_pools(new):
    rng = np.random.default_rng(len(new))
    cfg, layers, batch = workloads.decode_step_problem(
        rng, num_layers=1, hidden=512, hq=4, hkv=2, inter=1024,
        ctx=[n + 40 + i for i, n in enumerate(new)], new_tokens=new, kv_turbo3=True)
    _check(cfg, layers, batch, 1e-2)  # the bound of the steps over 3-bit pools


@pytest.mark.parametrize("rows", [64, 96])
@pytest.mark.parametrize("hidden,hq,hkv,d,inter", WIDTHS)
def test_whole_chunks_are_steps_of_32_rows(rows, hidden, hq, hkv, d, inter):
    """Every chunk's rows, bit for bit, as a step of those 32 rows by themselves: a norm, rotation or
    activation that took another row's value, group sum or place in a later chunk's buffer would not be.
    (One key per sequence: attention is that key's value however a batch is split.)"""
    rng = np.random.default_rng(rows + hidden)
    cfg, layers, batch = workloads.decode_step_problem(
        rng, num_layers=2, hidden=hidden, hq=hq, hkv=hkv, d=d, inter=inter, ctx=np.ones(rows, np.int32),
        qkv_bias=True)

    def run(r0, r1):
        part = dict(batch, cu_seqlens=np.arange(r1 - r0 + 1, dtype=np.int32))
        for name in ("h", "block_tables", "context_lens", "positions", "slots"):
            part[name] = batch[name][r0:r1]
        r = DecodeStepRunner(cfg, layers, part)
        r.launch()
        pools = [p.to_numpy(np.uint16, L["k_pool"].shape)[part["slots"]]
                 for kv, L in zip(r.pools, layers) for p in kv]
        return r.result_bits(), r.h.to_numpy(np.uint32, (r1 - r0, hidden)), *pools

    whole = run(0, rows)
    for r0 in range(0, rows, 32):
        for got, want in zip(whole, run(r0, r0 + 32)):
            assert np.array_equal(got[r0:r0 + 32], want)


@pytest.mark.parametrize("new", [[1] * 17, [1] * 33, [1] * 65, [1, 30, 2, 4]])  # (the last over 3-bit pools: two passes)
@pytest.mark.parametrize("hidden,hq,hkv,d,inter", WIDTHS)
def test_nothing_behind_the_workspace(new, hidden, hq, hkv, d, inter):
    rng = np.random.default_rng(hidden)
    cfg, layers, batch = workloads.decode_step_problem(
        rng, num_layers=1, hidden=hidden, hq=hq, hkv=hkv, d=d, inter=inter, ctx=[n + 5 for n in new],
        new_tokens=new, kv_turbo3=max(new) > 1 and d == 128)
    r = DecodeStepRunner(cfg, layers, batch)
    r.launch()
    want, size = r.result_bits(), r.ws.nbytes
    r = DecodeStepRunner(cfg, layers, batch)
    r.ws = hip.DeviceBuffer(size + 4096)
    r.ws.fill(0xA5)
    r.launch()
    assert np.array_equal(r.result_bits(), want)
    assert (r.ws.to_numpy(np.uint8, (size + 4096,))[size:] == 0xA5).all()
