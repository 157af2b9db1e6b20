"""The many-row rotation + K/V write (64 tokens and more at heads of 128 and wider, 2400 (token, head)
pairs and more at narrower ones) at head widths other than 128: bit for bit the per-head kernel that
launches of fewer tokens take, from split-K parts with a bias, with a token that has no slot.  Widths
that are no multiple of 8 stay on the per-head kernel."""
import numpy as np
import pytest

import oracle as O
from logismos_amd import hip, kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [131, 266, 267])  # 9 heads: 2394 and 2403 pairs
@pytest.mark.parametrize("d", [8, 24, 64, 96, 256, 12])
def test_same_bits_as_the_per_head_kernel(d, t):
    rng = np.random.default_rng(d)
    hq, hkv, rows, max_pos = 7, 1, t + 29, 300
    width = (hq + 2 * hkv) * d
    parts = rng.standard_normal((2, t, width), np.float32)
    bias = rng.standard_normal(width).astype(np.float32)
    positions = rng.integers(0, max_pos, size=t).astype(np.int32)
    slots = rng.permutation(rows)[:t].astype(np.int64)
    slots[70] = -1
    cos, sin = O.build_rope_table_f32(max_pos, d, 10_000.0)
    dev = hip.DeviceBuffer.from_numpy

    def run(chunk):
        k, v = dev(np.zeros((rows, hkv * d), np.float16)), dev(np.zeros((rows, hkv * d), np.float16))
        q = []
        for r0 in range(0, t, chunk):
            n = min(chunk, t - r0)
            d_q = hip.DeviceBuffer(n * hq * d * 2)
            kernels.launch_rope_kv_write_f32p(
                dev(np.ascontiguousarray(parts[:, r0:r0 + n])), 2, dev(positions[r0:r0 + n]), dev(cos),
                dev(sin), dev(slots[r0:r0 + n]), d_q, k, v, n, hq, hkv, d, max_pos, bias=dev(bias))
            hip.synchronize()
            q.append(d_q.to_numpy(np.uint16, (n, hq, d)))
        return np.concatenate(q), k.to_numpy(np.uint16, (rows, hkv * d)), v.to_numpy(np.uint16, (rows, hkv * d))

    for a, b in zip(run(t), run(50)):
        assert np.array_equal(a, b)
