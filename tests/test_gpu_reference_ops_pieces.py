"""The forms of the reference's launchers that work on whole 16-byte pieces, at the edges of their
tiles, slabs and registers, with the reference's metric and tolerance
(tests/test_gpu_reference_ops.py)."""
import numpy as np
import pytest

import oracle as O
from tests.test_gpu_reference_ops import _dev, _f16, _matmul, _parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1, 8, 8), (63, 64, 128), (65, 72, 136), (64, 128, 120), (17, 200, 1032),  # 64 x 64, long slabs
    (1500, 1608, 72), (1537, 1544, 64),                                        # 64 x 64
    (2900, 2888, 72), (2817, 2952, 136)])                                      # 128 x 128
def test_matmul_of_whole_pieces(m, n, k):
    got, want = _matmul("wmma", m, n, k, 5)
    _parity(got, want)


def test_matmul_leaves_out_what_lies_behind_k():
    # the piece behind a row's last column belongs to the next row: infinities there do not count
    from logismos_amd import hip, kernels
    m, n, k = 3, 8, 72
    rng = np.random.default_rng(6)
    a, b = _f16(rng, m, k), _f16(rng, k, n)
    a[1] = np.inf
    d = hip.DeviceBuffer(m * n * 2)
    kernels.launch_matmul_fp16("wmma", _dev(a), _dev(b), d, m, n, k)
    hip.synchronize()
    got = d.to_numpy(np.float16, (m, n))
    want = O.matmul_fp16_ref(a, b, m, n, k).reshape(m, n)
    _parity(got[[0, 2]].ravel(), want[[0, 2]].ravel())


@pytest.mark.parametrize("m,n", [(1, 8), (5, 1024), (6, 1032), (3, 2048), (7, 2056), (4, 4096), (2, 4104)])
def test_rms_norm_of_whole_pieces(m, n):
    from logismos_amd import hip, kernels
    rng = np.random.default_rng(n)
    x, w = _f16(rng, m, n), _f16(rng, n)
    y = hip.DeviceBuffer(m * n * 2)
    y.fill(0xFF)
    kernels.launch_rms_norm_fp16(_dev(x), _dev(w), y, m, n, 1e-5)
    hip.synchronize()
    _parity(y.to_numpy(np.float16, (m * n,)), O.rms_norm_fp16_ref(x, w, m, n, 1e-5))


@pytest.mark.parametrize("batch,seq,heads,d", [(1, 1, 1, 8), (2, 3, 5, 24), (3, 33, 12, 64), (1, 7, 33, 72)])
def test_rope_of_whole_pieces(batch, seq, heads, d):
    from logismos_amd import hip, kernels
    rng = np.random.default_rng(seq)
    qk = _f16(rng, batch, seq, heads, d)
    table = O.build_cos_sin_table(seq, d, 10_000.0)
    dev = _dev(qk)
    kernels.launch_rope_fp16_in_place(dev, _dev(table), batch, seq, heads, d)
    hip.synchronize()
    _parity(dev.to_numpy(np.float16, (qk.size,)), O.rope_apply_fp16_ref(qk, table, batch, seq, heads, d))
