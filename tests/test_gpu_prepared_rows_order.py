"""The norm and the activation that write the prepared layout at every kind of row count: each row exactly
once, the norm within a rounding of the oracle, the activation bit for bit the plain one's, and nothing in
the places of rows that there are not."""
import numpy as np
import pytest

import oracle as O
from logismos_amd import hip, kernels
from oracle import decode_step as OS

pytestmark = pytest.mark.gpu


def _rows(buf, b, k):
    """prepared layout -> bf16 bits and group sums of all row places"""
    bp = 16 if b <= 16 else 32
    xp = buf[: k // 8 * bp * 16].view(np.uint16).reshape(k // 8, bp, 8)[..., [0, 2, 4, 6, 1, 3, 5, 7]]
    return (xp.transpose(1, 0, 2).reshape(bp, k),
            buf[k // 8 * bp * 16:].view(np.uint32)[: k // 128 * bp].reshape(k // 128, bp).T)


def _empty_places(x, sums, rows):
    return (x[rows:] == 0xFFFF).all() and (sums[rows:] == 0xFFFFFFFF).all()


@pytest.mark.parametrize("rows", [1, 7, 8, 9, 15, 16, 17, 24, 25, 31, 32])
@pytest.mark.parametrize("n", [128, 1152])
def test_every_row_once(rows, n):
    rng = np.random.default_rng(rows * 10000 + n)
    dev = hip.DeviceBuffer.from_numpy
    h = rng.standard_normal((rows, n), np.float32)
    parts = rng.standard_normal((2, rows, n), np.float32)
    w = (1 + 0.02 * rng.standard_normal(n)).astype(np.float32)
    d_h, d_parts, d_w = dev(h), dev(parts), dev(w)
    out = hip.DeviceBuffer(kernels.q4_xprep_bytes(rows, n))
    out.fill(0xFF)
    kernels.launch_add_rms_norm_f32p_xprep(d_h, d_parts, 2, d_w, out, rows, n, 1e-6)
    hip.synchronize()
    x, sums = _rows(out.to_numpy(np.uint8, (out.nbytes,)), rows, n)
    h_want = h.copy()
    want = O.bf16_bits_to_f32(OS.add_rms_norm_bf16(h_want, parts[0] + parts[1], w, 1e-6))
    got = O.bf16_bits_to_f32(x[:rows])
    # h: two fp32 additions on each side, in another order; the normed value: those, and one bf16 step
    apart = 4 * 2.0**-24 * (np.abs(h) + np.abs(parts).sum(0))
    assert (np.abs(d_h.to_numpy(np.float32, (rows, n)) - h_want) <= apart).all()
    scale = np.abs(w) / np.sqrt((h_want * h_want).mean(1, keepdims=True) + 1e-6)
    assert (np.abs(got - want) <= 2.0**-7 * np.abs(want) + 1.01 * scale * apart).all()
    # a group's 128 values added up in fp32, at most nine roundings behind one another
    group = got.astype(np.float64).reshape(rows, n // 128, 128)
    assert (np.abs(sums[:rows].view(np.float32) - group.sum(2)) <= 9 * 2.0**-24 * np.abs(group).sum(2)).all()
    assert _empty_places(x, sums, rows)

    gp = rng.standard_normal((2, rows, 2 * n), np.float32)
    d_gp, plain = dev(gp), hip.DeviceBuffer(rows * n * 2)
    want_op = hip.DeviceBuffer(kernels.q4_xprep_bytes(rows, n))
    out.fill(0xFF)
    kernels.launch_silu_mul_f32p(d_gp, 2, plain, rows, n)
    kernels.launch_q4_prepare_x_bf16(plain, want_op, rows, n)
    kernels.launch_silu_mul_f32p_xprep(d_gp, 2, out, rows, n)
    hip.synchronize()
    x, sums = _rows(out.to_numpy(np.uint8, (out.nbytes,)), rows, n)
    x_want, sums_want = _rows(want_op.to_numpy(np.uint8, (want_op.nbytes,)), rows, n)
    assert np.array_equal(x[:rows], x_want[:rows]) and np.array_equal(sums[:rows], sums_want[:rows])
    assert _empty_places(x, sums, rows)
