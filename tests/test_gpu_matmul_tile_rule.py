"""The fp16 matmul at shapes that the rule over rounds gives to each of its tiles: one, two, three and more
slabs than a ring holds, ragged last tiles and slabs, a few more tiles than the chip holds at once."""
import numpy as np
import pytest

from logismos_amd import hip, kernels
from tests.test_gpu_reference_ops_pieces import _f16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (2100, 1024, 776), (2900, 776, 264), (700, 3072, 72),     # 33 rows of 64-row tiles, 17 of 128-row ones
    (1300, 3080, 64), (1300, 3080, 128), (1300, 3080, 136), (1300, 3080, 192), (1300, 3080, 200),
    (520, 2056, 8), (64, 520, 320), (2050, 4104, 40)])
def test_tiles_by_rounds(m, n, k):
    rng = np.random.default_rng(m + k)
    a, b = _f16(rng, m, k), _f16(rng, k, n)
    d = hip.DeviceBuffer(m * n * 2 + 64)
    d.fill(0x55)
    kernels.launch_matmul_fp16("wmma", hip.DeviceBuffer.from_numpy(a), hip.DeviceBuffer.from_numpy(b), d, m, n, k)
    hip.synchronize()
    raw = d.to_numpy(np.uint8, (m * n * 2 + 64,))
    assert (raw[m * n * 2:] == 0x55).all()
    got = raw[:m * n * 2].view(np.float16).reshape(m, n).astype(np.float64)
    a, b = a.astype(np.float64), b.astype(np.float64)
    want = a @ b
    # the rounding to fp16, and of each of the k fp32 sums at most one unit of what their terms add up to
    assert np.all(np.abs(got - want) <= 2.0 ** -11 * np.abs(want) + 2.0 ** -25
                  + k * 2.0 ** -23 * (np.abs(a) @ np.abs(b)))
