"""The forms of the reference's launchers that work on whole 16-byte pieces, at the edges of their
tiles, slabs and registers, with the reference's metric and tolerance
(tests/test_gpu_reference_ops.py)."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from logismos_amd import hip, kernels
from tests.test_gpu_reference_ops import _dev, _f16, _matmul, _parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1, 8, 8), (63, 64, 128), (65, 72, 136), (64, 128, 120), (17, 200, 1032),  # 64 x 64, long slabs
    (1500, 1608, 72), (1537, 1544, 64),                                        # 64 x 64
    (2900, 2888, 72), (2817, 2952, 136)])                                      # 128 x 128
def test_matmul_of_whole_pieces(m, n, k):
    got, want = _matmul("wmma", m, n, k, 5)
    _parity(got, want)


@pytest.mark.parametrize("m,n,k", [
    (640, 2056, 72), (700, 1992, 320),                    # 64 x 128
    (1409, 1672, 392), (1536, 1664, 328),                 # 128 x 128
    (1793, 3464, 200), (2048, 3080, 256), (1900, 3336, 8)])  # 256 x 128
def test_matmul_tiles(m, n, k):
    # ragged last tiles and slabs, fewer and more slabs than the ring holds.  Bound: the rounding to
    # fp16, and of each of the k fp32 sums at most one unit of what their terms add up to
    rng = np.random.default_rng(m)
    a, b = _f16(rng, m, k), _f16(rng, k, n)
    da, db, d = hip.DeviceBuffer.from_numpy(a), hip.DeviceBuffer.from_numpy(b), hip.DeviceBuffer(m * n * 2)
    kernels.launch_matmul_fp16("wmma", da, db, d, m, n, k)
    hip.synchronize()
    got = d.to_numpy(np.float16, (m, n)).astype(np.float64)
    a, b = a.astype(np.float64), b.astype(np.float64)
    want = a @ b
    assert np.all(np.abs(got - want) <= 2.0 ** -11 * np.abs(want) + 2.0 ** -25
                  + k * 2.0 ** -23 * (np.abs(a) @ np.abs(b)))


@pytest.mark.parametrize("m,n,k", [(70, 136, 72), (1500, 1608, 72)])
def test_matmul_into_rows_off_sixteen_bytes(m, n, k):
    rng = np.random.default_rng(m)
    a, b = _f16(rng, m, k), _f16(rng, k, n)
    da, db = hip.DeviceBuffer.from_numpy(a), hip.DeviceBuffer.from_numpy(b)
    d = hip.DeviceBuffer(m * n * 2 + 16)
    d.fill(0xA5)
    d2 = hip.DeviceBuffer(m * n * 2)
    kernels.launch_matmul_fp16("wmma", da, db, C.c_void_p(d.ptr.value + 2), m, n, k)
    kernels.launch_matmul_fp16("wmma", da, db, d2, m, n, k)
    hip.synchronize()
    got = d.to_numpy(np.uint16, (m * n + 8,))
    assert np.array_equal(got[1:1 + m * n], d2.to_numpy(np.uint16, (m * n,)))
    assert got[0] == 0xA5A5 and (got[1 + m * n:] == 0xA5A5).all()  # and nothing beside them


def test_matmul_leaves_out_what_lies_behind_k():
    # the piece behind a row's last column belongs to the next row: infinities there do not count
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
    rng = np.random.default_rng(n)
    x, w = _f16(rng, m, n), _f16(rng, n)
    y = hip.DeviceBuffer(m * n * 2)
    y.fill(0xFF)
    kernels.launch_rms_norm_fp16(_dev(x), _dev(w), y, m, n, 1e-5)
    hip.synchronize()
    _parity(y.to_numpy(np.float16, (m * n,)), O.rms_norm_fp16_ref(x, w, m, n, 1e-5))


@pytest.mark.parametrize("batch,seq,heads,d", [(1, 1, 1, 8), (2, 3, 5, 24), (3, 33, 12, 64), (1, 7, 33, 72)])
def test_rope_of_whole_pieces(batch, seq, heads, d):
    rng = np.random.default_rng(seq)
    qk = _f16(rng, batch, seq, heads, d)
    table = O.build_cos_sin_table(seq, d, 10_000.0)
    dev = _dev(qk)
    kernels.launch_rope_fp16_in_place(dev, _dev(table), batch, seq, heads, d)
    hip.synchronize()
    _parity(dev.to_numpy(np.float16, (qk.size,)), O.rope_apply_fp16_ref(qk, table, batch, seq, heads, d))


@pytest.mark.parametrize("n", [328, 656, 1000, 1536, 2504, 4040])
def test_rms_norm_to_the_last_bit(n):
    # 1 / sqrt(mean + eps) with every operation rounded once, over whole numbers whose sum of
    # squares is exact in any order.  The inputs tell it from a mean that is a product with 1 / n.
    rng = np.random.default_rng(n)
    m, eps, one = 400, np.float32(1e-5), np.float32(1)
    x = rng.integers(-9, 10, size=(m, n)).astype(np.float32)
    w = rng.normal(1, 0.1, n).astype(np.float16)
    total = (x.astype(np.float64) ** 2).sum(1, keepdims=True).astype(np.float32)
    mean = total / np.float32(n)

    def norm(mean):
        return (x * (one / np.sqrt(mean + eps)) * w.astype(np.float32)).astype(np.float16)

    want = norm(mean)
    assert (want != norm(total * (one / np.float32(n)))).any()
    up = hip.DeviceBuffer.from_numpy
    d_y = hip.DeviceBuffer(m * n * 2)
    kernels.launch_rms_norm_fp16(up(x.astype(np.float16)), up(w), d_y, m, n, float(eps))
    hip.synchronize()
    assert np.array_equal(d_y.to_numpy(np.float16, (m, n)), want)
