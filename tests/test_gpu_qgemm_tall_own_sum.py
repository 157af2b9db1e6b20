"""Products over many rows by themselves, on both sides of the line between 128 x 256 tiles split over K (with
a launch that adds up the parts) and smaller tiles that take all of K: two parts and three, nine large tiles and
ten, rows and columns that end inside a tile.  The fp32 result is always on the smaller ones; the bf16
result and the activation have its bits whichever they are on."""
import numpy as np
import pytest

import oracle as O
from logismos_amd import hip, kernels
from tests.gpu_harness import assert_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1, 2, 1280), (129, 258, 1280), (100, 512, 2048), (300, 260, 2048),  # two parts
    (97, 300, 1536), (300, 768, 1536),                                   # three, up to nine large tiles
    (100, 2560, 1536), (513, 514, 1536), (200, 1100, 1792),              # ... ten and more
])
def test_one_result_on_every_tile(m, n, k):
    rng = np.random.default_rng(m + n + k)
    qw, s, z = O.quantize_q4g128(rng.standard_normal((n, k), np.float32) * np.float32(0.02), n, k)
    xb = O.f32_to_bf16_bits(rng.standard_normal((m, k), np.float32))
    up = hip.DeviceBuffer.from_numpy
    weights = up(qw), up(s.view(np.uint16)), up(z.view(np.uint16))
    ws = hip.DeviceBuffer(kernels.qgemm_q4g128_tall_workspace_bytes(m, k))
    ws.fill(0xFF)
    y32, y16, act = (hip.DeviceBuffer(m * n * 4) for _ in range(3))
    for y in (y32, y16, act):
        y.fill(0xA5)
    kernels.launch_qgemm_q4g128_tall(up(xb), *weights, y32, ws, m, n, k, f32_out=True)
    kernels.launch_qgemm_q4g128_tall_prepared(*weights, y16, ws, m, n, k)
    kernels.launch_qgemm_q4g128_tall_swiglu_prepared(*weights, act, ws, m, n // 2, k)
    hip.synchronize()
    got = y32.to_numpy(np.float32, (m, n))
    assert_parity(got, O.qgemm_q4g128_f32(xb, qw, s, z, m, n, k), max_abs=2e-4, max_rel=1e-3)
    bits = y16.to_numpy(np.uint16, (2 * m * n,))
    assert np.array_equal(bits[:m * n], O.f32_to_bf16_bits(got).ravel())
    a = act.to_numpy(np.uint16, (2 * m * n,))
    g, u = got[:, :n // 2].astype(np.float64), got[:, n // 2:].astype(np.float64)
    want = g / (1 + np.exp(-g)) * u
    # one bf16 rounding (eight significant bits: 2^-8), the fp32 ones of the exponential and of three
    # operations in front of it are under 2^-20
    assert (np.abs(O.bf16_bits_to_f32(a[:m * (n // 2)]).reshape(want.shape) - want) <= (2.0**-8 + 2.0**-20) * np.abs(want)).all()
    # and nothing behind the results
    assert (bits[m * n:] == 0xA5A5).all() and (a[m * (n // 2):] == 0xA5A5).all()
