// The five launchers the reference's kernels crate already declares and its `praxis` layer
// already calls, for gfx950 (the reference builds them for gfx1100, wave32):
//
//   logismos_launch_rms_norm_fp16       crates/kernels/src/rms_norm/hip/rms_norm.hip:58-84
//   logismos_launch_softmax_fp16        crates/kernels/src/softmax/hip/softmax.hip:66-87
//   logismos_launch_rope_fp16           crates/kernels/src/rope/hip/rope.hip:45-68
//   logismos_launch_matmul_naive_fp16   crates/kernels/src/matmul/hip/matmul_launchers.cpp:14-32
//   logismos_launch_matmul_wmma_fp16    crates/kernels/src/matmul/hip/matmul_launchers.cpp:34-52
//
// Same symbols, argument lists and meaning (fp16 in and out, fp32 arithmetic inside, one
// rounding at the output; the CPU references crates/kernels/src/{rms_norm,softmax,rope,
// matmul}/cpu.rs define the results), so the crate's `extern "C"` blocks link against this
// archive unchanged.  "wmma" names the reference's RDNA3 instruction; here that entry point
// runs on the CDNA4 matrix cores (v_mfma_f32_32x32x16_f16) and, unlike the reference's,
// takes any M, N, K.
#include "device_utils.hpp"
#include "launch_common.hpp"
#include "q4_common.hpp"

#include <hip/hip_fp16.h>
#include <math.h>

#include <algorithm>

namespace lg {

constexpr int kRowThreads = 256;

// sum / max over the 256 threads of a workgroup; every thread gets the result
__device__ __forceinline__ float block_sum_256(float v, float* red) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    const float r = red[0] + red[1] + red[2] + red[3];
    __syncthreads();
    return r;
}
__device__ __forceinline__ float block_max_256(float v, float* red) {
    v = row16_max(v);
    v = fmaxf(fmaxf(__shfl(v, 0, kWave), __shfl(v, 16, kWave)),
              fmaxf(__shfl(v, 32, kWave), __shfl(v, 48, kWave)));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    const float r = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    __syncthreads();
    return r;
}

// y[r][j] = fp16( x[r][j] * (1 / sqrt(mean_j x[r][j]^2 + eps)) * w[j] ), one workgroup per row
// (`rms_norm_fp16_ref`, crates/kernels/src/rms_norm/cpu.rs:13-45)
__global__ __launch_bounds__(kRowThreads) void rms_norm_fp16_kernel(
    const __half* __restrict__ x, const __half* __restrict__ w, __half* __restrict__ y, int n,
    float eps) {
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    const __half* xr = x + row * n;
    __half* yr = y + row * n;
    float part = 0.0f;
    for (int j = threadIdx.x; j < n; j += kRowThreads) {
        const float v = __half2float(xr[j]);
        part = fmaf(v, v, part);
    }
    const float sum_sq = block_sum_256(part, red);
    const float inv_rms = 1.0f / sqrtf(sum_sq / (float)n + eps);
    for (int j = threadIdx.x; j < n; j += kRowThreads)
        yr[j] = __float2half_rn(__half2float(xr[j]) * inv_rms * __half2float(w[j]));
}

// The same for rows of whole 16-byte pieces that fit a wave's registers (n a multiple of 8, at
// most 512 * NP): one wave per row, read once, four rows per workgroup, instead of two passes of
// 2-byte accesses by a workgroup per row.  For 2036 x 1536 this and the rotation below together
// went from 11.8 to 5.7 us (12 MB each way through memory).
template <int NP>
__global__ __launch_bounds__(256) void rms_norm_fp16_wave_kernel(const uint4_t* __restrict__ x,
                                                                 const uint4_t* __restrict__ w,
                                                                 uint4_t* __restrict__ y, int m,
                                                                 int pieces, float eps) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= m) return;
    uint4_t xv[NP], wv[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        xv[p] = wv[p] = uint4_t{0u, 0u, 0u, 0u};
        if (p * 64 + lane < pieces) {
            xv[p] = x[(int64_t)row * pieces + p * 64 + lane];
            wv[p] = w[p * 64 + lane];
        }
    }
    // squares in pairs, pieces in pairs: no longer chains than a workgroup's 256 partial sums have
    float part[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const half8_t v = __builtin_bit_cast(half8_t, xv[p]);
        float pair[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            pair[e] = fmaf((float)v[2 * e + 1], (float)v[2 * e + 1], (float)v[2 * e] * (float)v[2 * e]);
        part[p] = (pair[0] + pair[1]) + (pair[2] + pair[3]);
    }
#pragma unroll
    for (int d = 1; d < NP; d *= 2)
#pragma unroll
        for (int p = 0; p < NP; p += 2 * d) part[p] += part[p + d];
    const float inv_rms = 1.0f / sqrtf(wave_sum(part[0]) / (float)(8 * pieces) + eps);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        if (p * 64 + lane >= pieces) continue;
        const half8_t v = __builtin_bit_cast(half8_t, xv[p]), g = __builtin_bit_cast(half8_t, wv[p]);
        half8_t o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (_Float16)((float)v[e] * inv_rms * (float)g[e]);
        y[(int64_t)row * pieces + p * 64 + lane] = __builtin_bit_cast(uint4_t, o);
    }
}

// Row softmax, fp32 inside: max-subtracted exponentials times the reciprocal of their sum; a
// row whose maximum is -inf (every entry -inf) becomes uniform 1/n
// (`softmax_fp16_ref`, crates/kernels/src/softmax/cpu.rs:14-74)
__global__ __launch_bounds__(kRowThreads) void softmax_fp16_kernel(const __half* __restrict__ x,
                                                                   __half* __restrict__ y, int n) {
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    const __half* xr = x + row * n;
    __half* yr = y + row * n;
    float mx = -INFINITY;
    for (int j = threadIdx.x; j < n; j += kRowThreads) mx = fmaxf(mx, __half2float(xr[j]));
    mx = block_max_256(mx, red);
    if (mx == -INFINITY) {
        const __half u = __float2half_rn(1.0f / (float)n);
        for (int j = threadIdx.x; j < n; j += kRowThreads) yr[j] = u;
        return;
    }
    float part = 0.0f;
    for (int j = threadIdx.x; j < n; j += kRowThreads) part += expf(__half2float(xr[j]) - mx);
    const float inv = 1.0f / block_sum_256(part, red);
    for (int j = threadIdx.x; j < n; j += kRowThreads)
        yr[j] = __float2half_rn(expf(__half2float(xr[j]) - mx) * inv);
}

// In place on fp16 (batch, seq, heads, head_dim): pair (2i, 2i+1) of every head row at
// position s is rotated by (cos, sin) = table[s][2i], table[s][2i+1]
// (`rope_apply_fp16_ref`, crates/kernels/src/rope/cpu.rs:56-127).  One thread per pair: a
// pair is one aligned 32-bit word of the tensor and one 64-bit entry of the table.
__global__ __launch_bounds__(256) void rope_fp16_kernel(unsigned* __restrict__ qk_pairs,
                                                        const float2* __restrict__ cos_sin,
                                                        int64_t total_pairs, int seq, int heads,
                                                        int pairs) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total_pairs) return;
    const int i = (int)(idx % pairs);
    const int64_t row = idx / pairs;           // (b * seq + s) * heads + h
    const int s = (int)((row / heads) % seq);
    const float2 cs = cos_sin[(int64_t)s * pairs + i];
    const unsigned word = qk_pairs[idx];
    const float x0 = __half2float(__ushort_as_half((unsigned short)(word & 0xffffu)));
    const float x1 = __half2float(__ushort_as_half((unsigned short)(word >> 16)));
    const float y0 = x0 * cs.x - x1 * cs.y;
    const float y1 = x0 * cs.y + x1 * cs.x;
    qk_pairs[idx] = (unsigned)__half_as_ushort(__float2half_rn(y0)) |
                    ((unsigned)__half_as_ushort(__float2half_rn(y1)) << 16);
}

// The same for head rows of whole 16-byte pieces (head_dim a multiple of 8): one thread per four
// pairs, grid (pieces of a token, seq, batch), no 64-bit division.
__global__ __launch_bounds__(256) void rope_fp16_pieces_kernel(uint4_t* __restrict__ qk,
                                                               const float4_t* __restrict__ cos_sin,
                                                               int token_pieces, int head_pieces) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= token_pieces) return;
    const int s = blockIdx.y;
    const unsigned i = (unsigned)t % (unsigned)head_pieces;
    uint4_t* const at = qk + ((int64_t)blockIdx.z * gridDim.y + s) * token_pieces + t;
    const float4_t* const cs = cos_sin + ((int64_t)s * head_pieces + i) * 2;
    const half8_t v = __builtin_bit_cast(half8_t, *at);
    half8_t o;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const float4_t c = cs[q];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const float x0 = (float)v[4 * q + 2 * p], x1 = (float)v[4 * q + 2 * p + 1];
            o[4 * q + 2 * p] = (_Float16)(x0 * c[2 * p] - x1 * c[2 * p + 1]);
            o[4 * q + 2 * p + 1] = (_Float16)(x0 * c[2 * p + 1] + x1 * c[2 * p]);
        }
    }
    *at = __builtin_bit_cast(uint4_t, o);
}

// D = A[M,K] . B[K,N], one thread per output element, fp32 accumulation in ascending k with
// separate multiply and add -- the order and the roundings of `matmul_fp16_ref`
// (crates/kernels/src/matmul/cpu.rs:12-30), so the result is bit-identical to it.
__global__ __launch_bounds__(256) void matmul_naive_fp16_kernel(const __half* __restrict__ a,
                                                                const __half* __restrict__ b,
                                                                __half* __restrict__ d, int m,
                                                                int n, int k) {
    const int col = blockIdx.x * 64 + (threadIdx.x & 63);
    const int row = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (row >= m || col >= n) return;
    const __half* ar = a + (int64_t)row * k;
    float acc = 0.0f;
    for (int p = 0; p < k; ++p)
        acc = __fadd_rn(acc, __fmul_rn(__half2float(ar[p]), __half2float(b[(int64_t)p * n + col])));
    d[(int64_t)row * n + col] = __float2half_rn(acc);
}

// The matrix-core version: a workgroup of four waves owns a 128 x 128 tile of D, each wave a
// 64 x 64 quarter (2 x 2 accumulators of v_mfma_f32_32x32x16_f16).  Per 32-wide slab of K the
// workgroup stages A[128 x 32] and B[32 x 128] in LDS -- B transposed to [n][k] on the way,
// because the MFMA B operand wants eight consecutive k of one column and B is row-major: two
// k rows per thread, merged into (k, k+1) words, with the four 16-byte chunks of an LDS row
// XOR-swizzled by (row / 16) % 4 so that these transposed 4-byte stores are two-way instead
// of eight-way bank conflicts.  The LDS tiles are double buffered: slab s + 1 is fetched
// from memory while slab s is multiplied, one barrier per slab.  Rows, columns and k beyond
// the matrix are zero-filled.
constexpr int kMmTile = 128, kMmK = 32;
constexpr int kMmStride = kMmK + 8;  // halfs per LDS row: 80 bytes, 16-byte reads stay aligned
constexpr int kMmBuf = kMmTile * kMmStride;

__global__ __launch_bounds__(256) void matmul_mfma_fp16_kernel(const _Float16* __restrict__ a,
                                                               const _Float16* __restrict__ b,
                                                               _Float16* __restrict__ d, int m,
                                                               int n, int k) {
    __shared__ __attribute__((aligned(16))) _Float16 as[2 * kMmBuf];
    __shared__ __attribute__((aligned(16))) _Float16 bs[2 * kMmBuf];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int row0 = blockIdx.y * kMmTile;
    const int col0 = blockIdx.x * kMmTile;
    const int wr = (wave >> 1) * 64;  // this wave's quarter
    const int wc = (wave & 1) * 64;
    const int r = lane & 31;
    const int h = lane >> 5;

    float16_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    // staging roles.  A: thread -> rows tid / 4 and tid / 4 + 64, eight consecutive k at
    // 8 * (tid % 4).  B: thread -> k rows 2 * (tid / 16) and + 1, eight consecutive columns at
    // 8 * (tid % 16).
    const int a_row = tid >> 2, a_k = (tid & 3) * 8;
    const int b_kp = tid >> 4, b_col = (tid & 15) * 8;
    const bool a_vec = (k & 7) == 0, b_vec = (n & 7) == 0;
    half8_t ra[2], rb[2];
    auto gload = [&](int k0) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            half8_t v = {0, 0, 0, 0, 0, 0, 0, 0};
            const int gr = row0 + a_row + 64 * u, gk = k0 + a_k;
            if (gr < m && gk < k) {
                const _Float16* src = a + (int64_t)gr * k + gk;
                if (a_vec && gk + 8 <= k) {
                    v = *reinterpret_cast<const half8_t*>(src);
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (gk + i < k) v[i] = src[i];
                }
            }
            ra[u] = v;
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            half8_t v = {0, 0, 0, 0, 0, 0, 0, 0};
            const int gk = k0 + 2 * b_kp + u, gc = col0 + b_col;
            if (gk < k && gc < n) {
                const _Float16* src = b + (int64_t)gk * n + gc;
                if (b_vec && gc + 8 <= n) {
                    v = *reinterpret_cast<const half8_t*>(src);
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (gc + i < n) v[i] = src[i];
                }
            }
            rb[u] = v;
        }
    };
    // LDS column (halfs) of k pair b_kp in a B row whose swizzle key is `key`
    auto lstore = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
            *reinterpret_cast<half8_t*>(as + buf * kMmBuf + (a_row + 64 * u) * kMmStride + a_k) =
                ra[u];
        const uint4_t lo = __builtin_bit_cast(uint4_t, rb[0]);
        const uint4_t hi = __builtin_bit_cast(uint4_t, rb[1]);
        const int key = (b_col >> 4) & 3;  // (row / 16) % 4 of rows b_col .. b_col + 7
        _Float16* dst =
            bs + buf * kMmBuf + 8 * ((b_kp >> 2) ^ key) + 2 * (b_kp & 3);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const unsigned sel = (e & 1) ? 0x07060302u : 0x05040100u;
            const unsigned pr = __builtin_amdgcn_perm(hi[e >> 1], lo[e >> 1], sel);
            *reinterpret_cast<unsigned*>(dst + (b_col + e) * kMmStride) = pr;
        }
    };

    const int slabs = (k + kMmK - 1) / kMmK;
    gload(0);
    lstore(0);
    __syncthreads();
    for (int sl = 0; sl < slabs; ++sl) {
        const int buf = sl & 1;
        if (sl + 1 < slabs) gload((sl + 1) * kMmK);
        const _Float16* at = as + buf * kMmBuf;
        const _Float16* bt = bs + buf * kMmBuf;
#pragma unroll
        for (int kk = 0; kk < kMmK; kk += 16) {
            half8_t av[2], bv[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                av[i] = *reinterpret_cast<const half8_t*>(at + (wr + 32 * i + r) * kMmStride + kk +
                                                          8 * h);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int row = wc + 32 * j + r;
                bv[j] = *reinterpret_cast<const half8_t*>(
                    bt + row * kMmStride + 8 * (((kk >> 3) + h) ^ ((row >> 4) & 3)));
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[i], bv[j], acc[i][j], 0,
                                                                       0, 0);
        }
        if (sl + 1 < slabs) lstore(buf ^ 1);  // last read of that buffer: before the last barrier
        __syncthreads();
    }
    // lane (h, r) holds column r, rows 8 * (e / 4) + 4h + e % 4 of each 32 x 32 block
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int gc = col0 + wc + 32 * j + r;
            if (gc >= n) continue;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int gr = row0 + wr + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3);
                if (gr < m) d[(int64_t)gr * n + gc] = (_Float16)acc[i][j][e];
            }
        }
}

// The same product for rows that are whole 16-byte pieces (n and k multiples of 8): a workgroup
// owns a 32 MB WR x 32 NB WC tile, its WR x WC waves 32 MB x 32 NB each.  Slabs of 64 columns of A
// (TM rows of 128 bytes) and 64 rows of B (TN columns) go from global memory straight into a ring of
// BUFS buffers in LDS (global_load_lds, 1 KiB of consecutive LDS per request), BUFS - 1 slabs ahead,
// two requests behind each of the last two steps of 16 columns.  As in the tiled Q4 GEMM the wait and
// the barrier stand in the middle of a slab and the first operands of the next slab are read in its
// last step.  Rows cannot be padded; the 16-byte chunks of a row are swizzled instead: A's by half
// the row index (a ds_read_b128 of 32 rows x 2 chunks touches every bank once per 16 lanes), B's in
// pairs (the transposing read takes 4 rows x 32 bytes per 16 lanes).  The B operand -- eight
// consecutive k of one column -- is two ds_read_b64_tr_b16: inside 16 lanes, lane L receives element
// L % 4 of the 8-byte pieces that the lanes L / 4 + 4 i point at, so lanes pointing at 4 k x 16 columns
// come back with 4 k of one column each.  LDS is only touched through inline assembly inside the
// loop: the compiler would order every access it can see behind all outstanding requests.
typedef __attribute__((address_space(3))) void* mm_lds_ptr_t;
template <int MB, int NB, int WR, int WC, int BUFS>
__global__ __launch_bounds__(64 * WR * WC) void matmul_ring_fp16_kernel(
    const _Float16* __restrict__ a, const _Float16* __restrict__ b, _Float16* __restrict__ d, int m,
    int n, int k, int tiles_m, int tiles_n, int vec_out) {
    constexpr int W = WR * WC, TM = 32 * MB * WR, TN = 32 * NB * WC, KS = 64;
    constexpr int kA = TM * KS * 2, kBuf = kA + KS * TN * 2;   // bytes
    constexpr int RA = TM / 8 / W, RB = TN / 8 / W;            // requests per wave and slab
    static_assert(RA * W * 8 == TM && RB * W * 8 == TN , "whole requests");
    static_assert(TN == 64 || TN == 128, "the swizzle of B");
    constexpr int kReq = RA + RB;
    extern __shared__ uint4_t mm_lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, h = lane >> 5;

    // Workgroups go round the eight XCDs in the order of their ids: each XCD takes a run of tiles,
    // four row tiles by as many column tiles as that makes, and reads its part of A and B once.
    const int tiles = tiles_m * tiles_n;
    int t = blockIdx.x;
    {
        const int per = tiles / 8, more = tiles % 8, xcd = t % 8;
        t = xcd * per + min(xcd, more) + t / 8;
    }
    const int band = t / (4 * tiles_n), in_band = t - band * 4 * tiles_n;
    const int band_rows = min(4, tiles_m - 4 * band);
    const int row0 = (4 * band + in_band % band_rows) * TM, col0 = (in_band / band_rows) * TN;

    const unsigned lds_base = (unsigned)(uintptr_t)(mm_lds_ptr_t)mm_lds;
    // ---- requests: q of A covers rows 8 (RA wave + q) .. + 7, lane -> row + lane / 8, position lane
    // % 8, which holds chunk (position ^ row / 2 % 8); q of B covers 1 KiB of rows of TN columns.  What
    // lies past m, n or k re-reads what is there (past k it is taken as zero below, past m and n it
    // only reaches results that are not stored).
    constexpr int BR = 512 / TN;                        // rows of B per request
    auto b_swizzle = [](int row) { return TN == 128 ? 2 * (row & 3) : 2 * ((row >> 1) & 1); };
    unsigned a_row[RA], b_col[RB];
    int a_chunk[RA], b_row[RB];
#pragma unroll
    for (int q = 0; q < RA; ++q) {
        const int row = 8 * (RA * wave + q) + (lane >> 3);
        a_chunk[q] = 8 * ((lane & 7) ^ ((row >> 1) & 7));
        a_row[q] = (unsigned)min(row0 + row, m - 1) * (unsigned)k;
    }
#pragma unroll
    for (int q = 0; q < RB; ++q) {
        b_row[q] = BR * (RB * wave + q) + lane / (TN / 8);
        b_col[q] = (unsigned)min(col0 + 8 * ((lane % (TN / 8)) ^ b_swizzle(b_row[q])), n - 8);
    }
    auto request_a = [&](int s, int buf_off) LG_INLINE {
#pragma unroll
        for (int q = 0; q < RA; ++q)
            request_lds16(a, (a_row[q] + (unsigned)min(s * KS + a_chunk[q], k - 8)) * 2u,
                    __builtin_amdgcn_readfirstlane(lds_base + (unsigned)buf_off + (unsigned)(RA * wave + q) * 1024u));
    };
    auto request_b = [&](int s, int buf_off) LG_INLINE {
#pragma unroll
        for (int q = 0; q < RB; ++q)
            request_lds16(b, ((unsigned)min(s * KS + b_row[q], k - 1) * (unsigned)n + b_col[q]) * 2u,
                    __builtin_amdgcn_readfirstlane(lds_base + (unsigned)buf_off + kA + (unsigned)(RB * wave + q) * 1024u));
    };

    // ---- operand reads.  A: lane (r, h) at step kk (16 columns) wants chunk 2 kk + h of row wr + 32 i +
    // r.  B: rows 16 kk + 8 h + lane % 16 / 4 and four on, columns wc + 32 j + 16 (lane / 16 % 2) + 4 (lane % 4).
    const int wr = (wave / WC) * 32 * MB, wc = (wave % WC) * 32 * NB;
    const unsigned a_base = lds_base + (unsigned)(wr + r) * 128u;
    const unsigned a_pos = (unsigned)(h ^ ((r >> 1) & 7)) * 16u;
    const int s16 = lane & 15, b_k = 8 * h + (s16 >> 2);
    unsigned b_base[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int col = wc + 32 * j + 16 * ((lane >> 4) & 1) + 4 * (s16 & 3);
        b_base[j] = lds_base + kA + (unsigned)b_k * (TN * 2u) +
                    (unsigned)((col >> 3) ^ b_swizzle(b_k)) * 16u + (unsigned)(col & 4) * 2u;
    }
    half8_t av[2][MB];
    uint2_t bl[2][NB], bh[2][NB];  // rows 0 .. 3 and 4 .. 7 of the lane's eight
    auto read_step = [&](auto kk_c, int buf_off) LG_INLINE {
        constexpr int KK = decltype(kk_c)::value, P = KK & 1;
        const unsigned aa = (a_base + (a_pos ^ (32u * KK))) + (unsigned)buf_off;
        static_for<MB>([&](auto i_c) LG_INLINE {
            constexpr int at = decltype(i_c)::value * 32 * 128;
            half8_t& dst = av[P][decltype(i_c)::value];
            const unsigned from = aa;
            asm volatile("ds_read_b128 %0, %1 offset:%c2" : "=&v"(dst) : "v"(from), "n"(at) : "memory");
        });
        static_for<NB>([&](auto j_c) LG_INLINE {
            constexpr int J = decltype(j_c)::value;
            uint2_t& lo = bl[P][J];
            uint2_t& hi = bh[P][J];
            const unsigned from = b_base[J] + (unsigned)buf_off;
            // (four rows on: the swizzle repeats every four rows)
            asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%c3\n\tds_read_b64_tr_b16 %1, %2 offset:%c4"
                         : "=&v"(lo), "=&v"(hi)
                         : "v"(from), "n"(KK * 16 * TN * 2), "n"((KK * 16 + 4) * TN * 2)
                         : "memory");
        });
    };
    auto step_landed = [&](auto kk_c) LG_INLINE {
        constexpr int P = decltype(kk_c)::value & 1;
        half8_t& a0 = av[P][0];
        uint2_t& l0 = bl[P][0];
        uint2_t& h0 = bh[P][0];
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a0), "+v"(l0), "+v"(h0)::"memory");
        static_for<MB - 1>([&](auto i_c) LG_INLINE {
            half8_t& x = av[P][decltype(i_c)::value + 1];
            asm volatile("" : "+v"(x)::"memory");
        });
        static_for<NB - 1>([&](auto j_c) LG_INLINE {
            uint2_t& x = bl[P][decltype(j_c)::value + 1];
            uint2_t& y = bh[P][decltype(j_c)::value + 1];
            asm volatile("" : "+v"(x), "+v"(y)::"memory");
        });
    };
    float16_t acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    const int slabs = (k + KS - 1) / KS;
    // (LAST: the slab is the last one, which may end past k)
    auto multiply = [&](auto kk_c, auto last_c, int s) LG_INLINE {
        constexpr int KK = decltype(kk_c)::value, P = KK & 1;
        uint4_t bv[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) bv[j] = uint4_t{bl[P][j][0], bl[P][j][1], bh[P][j][0], bh[P][j][1]};
        if (decltype(last_c)::value && s * KS + KS > k) {
            // past k: zeros on both sides (what lies there may be an infinity)
            const bool in = s * KS + 16 * KK + 8 * h < k;
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                uint4_t v = __builtin_bit_cast(uint4_t, av[P][i]);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = in ? v[e] : 0u;
                av[P][i] = __builtin_bit_cast(half8_t, v);
            }
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) bv[j][e] = in ? bv[j][e] : 0u;
        }
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[P][i], __builtin_bit_cast(half8_t, bv[j]),
                                                                   acc[i][j], 0, 0, 0);
    };

    // ---- the first BUFS - 1 slabs, then slab by slab
#pragma unroll
    for (int u = 0; u < BUFS - 1; ++u)
        if (u < slabs) {
            request_a(u, u * kBuf);
            request_b(u, u * kBuf);
        }
    if (slabs >= BUFS - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((BUFS - 2) * kReq) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    read_step(ic<0>{}, 0);
    step_landed(ic<0>{});
    // MORE: there is a slab behind this one.  (A constant: whether a read is waited for has to be known where
    // it is asked for, or the compiler may join the two ways with a copy of what is still in flight.)
    auto slab = [&](auto more_c, int s, int buf_off) LG_INLINE {
        constexpr bool more = decltype(more_c)::value != 0;
        constexpr ic<!more> last{};
        const int next_off = buf_off + kBuf == BUFS * kBuf ? 0 : buf_off + kBuf;
        const int last_off = buf_off == 0 ? (BUFS - 1) * kBuf : buf_off - kBuf;  // of slab s - 1
        const bool ahead = more && s + BUFS - 1 < slabs;
        read_step(ic<1>{}, buf_off);
        __builtin_amdgcn_sched_barrier(0);
        multiply(ic<0>{}, last, s);
        __builtin_amdgcn_sched_barrier(0);
        step_landed(ic<1>{});
        read_step(ic<2>{}, buf_off);
        __builtin_amdgcn_sched_barrier(0);
        multiply(ic<1>{}, last, s);
        __builtin_amdgcn_sched_barrier(0);
        step_landed(ic<2>{});
        if constexpr (more) {
            // slab s + 1 has landed (its requests are the oldest of BUFS - 2 slabs'; this wave's
            // requests complete in the order they were issued), behind the barrier everybody's has,
            // and everybody has left slab s - 1, whose buffer slab s + BUFS - 1 takes
            if (s + BUFS - 2 < slabs) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((BUFS - 3) * kReq) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
        }
        read_step(ic<3>{}, buf_off);
        if (ahead) request_a(s + BUFS - 1, last_off);
        __builtin_amdgcn_sched_barrier(0);
        multiply(ic<2>{}, last, s);
        __builtin_amdgcn_sched_barrier(0);
        step_landed(ic<3>{});
        if constexpr (more) read_step(ic<0>{}, next_off);
        if (ahead) request_b(s + BUFS - 1, last_off);
        __builtin_amdgcn_sched_barrier(0);
        multiply(ic<3>{}, last, s);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (more) step_landed(ic<0>{});
        return next_off;
    };
    int buf_off = 0;
    for (int s = 0; s + 1 < slabs; ++s) buf_off = slab(ic<1>{}, s, buf_off);
    slab(ic<0>{}, slabs - 1, buf_off);

    // lane (h, r) holds column r, rows 8 * (e / 4) + 4h + e % 4 of each 32 x 32 block
    if (!vec_out) {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                const int gc = col0 + wc + 32 * j + r;
                if (gc >= n) continue;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int gr = row0 + wr + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3);
                    if (gr < m) d[(int64_t)gr * n + gc] = (_Float16)acc[i][j][e];
                }
            }
        return;
    }
    // ... through LDS, and out in 16-byte pieces
    __syncthreads();  // the ring is done with once every wave has read its last operands
    constexpr int kPitch = TN + 8;
    _Float16* const out = reinterpret_cast<_Float16*>(mm_lds);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                out[(wr + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3)) * kPitch + wc + 32 * j + r] = (_Float16)acc[i][j][e];
    __syncthreads();
    constexpr int kPieces = TN / 8;
#pragma unroll
    for (int u = 0; u < TM * kPieces / (64 * W); ++u) {
        const int id = u * 64 * W + tid, row = id / kPieces, c = id % kPieces;
        const int gr = row0 + row, gc = col0 + 8 * c;
        if (gr < m && gc < n)
            *reinterpret_cast<uint4_t*>(d + (int64_t)gr * n + gc) = *reinterpret_cast<const uint4_t*>(out + row * kPitch + 8 * c);
    }
}

template <int MB, int NB, int WR, int WC, int BUFS>
static hipError_t matmul_ring_launch(const void* a, const void* b, void* d, int m, int n, int k,
                                     hipStream_t st) {
    constexpr int TM = 32 * MB * WR, TN = 32 * NB * WC;
    constexpr int kMost = BUFS * (TM + TN) * 128;
    const auto kernel = matmul_ring_fp16_kernel<MB, NB, WR, WC, BUFS>;
    static const hipError_t opt = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kMost);
    if (opt != hipSuccess) return opt;
    // few slabs: the ring is no longer than they are (and the product's way out needs its tile), so that
    // more workgroups share a compute unit
    const int slabs = (k + 63) / 64;
    const int lds = std::max(std::min(slabs, BUFS) * (TM + TN) * 128, TM * (TN + 8) * 2);
    static_assert(TM * (TN + 8) * 2 <= kMost, "the tile fits the ring");
    const int tm = (m + TM - 1) / TM, tn = (n + TN - 1) / TN;
    const int vec_out = (reinterpret_cast<uintptr_t>(d) & 15u) == 0;
    kernel<<<dim3((unsigned)((int64_t)tm * tn)), dim3(64 * WR * WC), lds, st>>>(
        static_cast<const _Float16*>(a), static_cast<const _Float16*>(b), static_cast<_Float16*>(d), m, n, k,
        tm, tn, vec_out);
    return hipGetLastError();
}

// Which tile: the one whose rounds take the least.  A compute unit holds as many workgroups of a tile as
// the ring (min(slabs, buffers) slabs of LDS) and the registers allow; a round of r of them takes the tile's
// ramp and, per slab of 64 columns, the longer of its own chain of dependent steps and r times its share of
// the unit.  The share is larger by `uneven` where the rows of A or B are not whole 128-byte lines: what a
// request asks for lies in more of them, the more so the narrower the tile.  All in us, fitted to 2380 shapes
// (64 to 5000 rows, 512 to 4096 columns, K 64 to 4096, half of them uneven): the tile taken is 2.1 % off the
// fastest of the six on the mean.  us, 256 x 128 / 128 x 128 / 64 x 128 / 64 x 64 (the last two on the better of
// their rings):
//   3200 x 768 x 2048   28.2 / 16.9 / 19.5 / 18.4   2100 x 1024 x 512   9.1 / 6.6 / 6.6 / 5.9
//   1700 x 4096 x 512   12.3 / 13.4 / 14.4 / 16.2   200 x 4096 x 512    8.6 / 6.2 / 4.4 / 4.3
// A shorter ring (three buffers) lets more workgroups share a unit.  Where the longer one holds all there are, it
// is taken: at a long K the shorter one waits for memory (200 x 3072 x 3560 26.0 / 17.0, 700 x 512 x 3560 25.5 /
// 16.5).  Up to three slabs there is no difference but the code; the shorter one then.
// What bounds it: the operands' way from L2 where tiles are many, where they are few a slab's chain of four
// dependent steps, 0.24 us on 64 x 64, 0.34 on 128 x 128.
struct MatmulTile {
    int rows, cols, bufs, most;  // most: workgroups of a compute unit by its registers
    float once, ramp, chain, share, uneven;
    decltype(&matmul_ring_launch<2, 2, 4, 2, 3>) launch;
    int64_t held(int64_t slabs) const {  // workgroups of a unit
        const int64_t lds = std::max(std::min<int64_t>(slabs, bufs) * (rows + cols) * 128,
                                     (int64_t)rows * (cols + 8) * 2);
        return std::min<int64_t>(160 * 1024 / lds, most);
    }
    float time(int64_t per_cu, int64_t slabs, bool whole_lines) const {
        const int64_t h = held(slabs);
        const float part = whole_lines ? share : share * (1.0f + uneven);
        auto round = [&](int64_t r) { return ramp + (float)slabs * std::max(chain, (float)r * part); };
        return once + (float)(per_cu / h) * round(h) + (per_cu % h ? round(per_cu % h) : 0.0f);
    }
};
static hipError_t matmul_tiled(const void* a, const void* b, void* d, int m, int n, int k, void* stream) {
    static const MatmulTile tiles[] = {
        {256, 128, 3, 2, 0.0f, 3.71f, 0.25f, 0.90f, 0.19f, matmul_ring_launch<2, 2, 4, 2, 3>},
        {128, 128, 5, 3, 0.02f, 3.56f, 0.34f, 0.48f, 0.13f, matmul_ring_launch<2, 1, 2, 4, 5>},
        {64, 128, 5, 4, 0.67f, 1.97f, 0.32f, 0.32f, 0.10f, matmul_ring_launch<1, 1, 2, 4, 5>},
        {64, 128, 3, 4, 1.15f, 1.72f, 0.50f, 0.32f, 0.10f, matmul_ring_launch<1, 1, 2, 4, 3>},
        {64, 64, 5, 8, 1.48f, 1.10f, 0.24f, 0.24f, 0.20f, matmul_ring_launch<1, 1, 2, 2, 5>},
        {64, 64, 3, 8, 1.55f, 1.15f, 0.22f, 0.18f, 0.27f, matmul_ring_launch<1, 1, 2, 2, 3>},
    };
    const int64_t slabs = ((int64_t)k + 63) / 64, cus = device_cu_count();
    const bool whole_lines = n % 64 == 0 && k % 64 == 0;
    const MatmulTile* best = nullptr;
    float best_time = 0.0f;
    bool all_held = false;  // of the tile in front, on the longer ring
    for (const MatmulTile& t : tiles) {
        const int64_t count = (((int64_t)m + t.rows - 1) / t.rows) * (((int64_t)n + t.cols - 1) / t.cols);
        const int64_t per_cu = (count + cus - 1) / cus;
        if (t.rows == 64) {
            if (t.bufs == 5) {
                if (slabs <= 3) continue;
                all_held = per_cu <= t.held(slabs);
            } else if (slabs > 3 && all_held) {
                continue;
            }
        }
        const float time = t.time(per_cu, slabs, whole_lines);
        if (!best || time < best_time) best = &t, best_time = time;
    }
    return best->launch(a, b, d, m, n, k, static_cast<hipStream_t>(stream));
}

// `check_matmul_shape` (crates/kernels/src/matmul/mod.rs:89-117)
static bool matmul_shape_ok(int m, int n, int k) {
    if (m <= 0 || n <= 0 || k <= 0) return false;
    const int64_t lim = INT32_MAX;
    return (int64_t)m * k <= lim && (int64_t)k * n <= lim && (int64_t)m * n <= lim;
}

}  // namespace lg

namespace lg {

// scores[r][c] = -inf where mask[r / repeat][c] == 0 (one mask row serves `repeat` consecutive
// score rows: the heads of one batch row), 16 bytes of mask per thread where n allows
template <typename T>
__global__ __launch_bounds__(256) void mask_additive_kernel(T* __restrict__ scores,
                                                            const uint8_t* __restrict__ mask,
                                                            int64_t rows, int64_t n,
                                                            int64_t repeat, T neg_inf) {
    const int64_t total = rows * n;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int64_t r = i / n;
        const int64_t c = i - r * n;
        if (mask[(r / repeat) * n + c] == 0) scores[i] = neg_inf;
    }
}

static logismos_status_t mask_additive_check(const void* scores, const void* mask,
                                             size_t mask_len, size_t rows, size_t n,
                                             int64_t* repeat) {
    *repeat = 0;
    // `mask_additive_in_place` (crates/kernels/src/cpu_f32/mod.rs:451-486): nothing to do
    // without columns, rows or a mask, or with a mask shorter than one row
    if (n == 0 || rows == 0 || mask_len == 0 || mask_len / n == 0) return hipSuccess;
    if (!scores || !mask) return hipErrorInvalidValue;
    const size_t mask_rows = mask_len / n;
    // (the reference's debug assertion: the mask is whole rows)
    if (mask_rows * n != mask_len) return hipErrorInvalidValue;
    // the reference panics here: a row count that the mask rows do not divide would leave
    // the trailing rows unmasked
    if (rows % mask_rows != 0) return hipErrorInvalidValue;
    if (rows > (size_t)INT32_MAX || n > (size_t)INT32_MAX ||
        (uint64_t)rows * (uint64_t)n > ((uint64_t)1 << 40))
        return hipErrorInvalidValue;
    *repeat = (int64_t)(rows / mask_rows);
    return hipSuccess;
}

template <typename T>
static logismos_status_t mask_additive_launch(void* scores, const void* mask, size_t mask_len,
                                              size_t rows, size_t n, T neg_inf,
                                              logismos_stream_t stream) {
    int64_t repeat;
    const logismos_status_t st = mask_additive_check(scores, mask, mask_len, rows, n, &repeat);
    if (st != hipSuccess || repeat == 0) return st;
    const int64_t total = (int64_t)rows * (int64_t)n;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 256 * 32) blocks = 256 * 32;
    mask_additive_kernel<T><<<dim3((unsigned)blocks), dim3(256), 0,
                              static_cast<hipStream_t>(stream)>>>(
        static_cast<T*>(scores), static_cast<const uint8_t*>(mask), (int64_t)rows, (int64_t)n,
        repeat, neg_inf);
    return hipGetLastError();
}

}  // namespace lg

extern "C" logismos_status_t logismos_launch_mask_additive_f32(void* scores_f32,
                                                               const void* mask_u8,
                                                               size_t mask_len, size_t rows,
                                                               size_t n,
                                                               logismos_stream_t stream) {
    return lg::mask_additive_launch<float>(scores_f32, mask_u8, mask_len, rows, n, -INFINITY,
                                           stream);
}

extern "C" logismos_status_t logismos_launch_mask_additive_fp16(void* scores_fp16,
                                                                const void* mask_u8,
                                                                size_t mask_len, size_t rows,
                                                                size_t n,
                                                                logismos_stream_t stream) {
    return lg::mask_additive_launch<unsigned short>(scores_fp16, mask_u8, mask_len, rows, n,
                                                    (unsigned short)0xFC00u, stream);
}

extern "C" logismos_status_t logismos_launch_rms_norm_fp16(const void* x_fp16, const void* w_fp16,
                                                           void* y_fp16, int m, int n, float eps,
                                                           logismos_stream_t stream) {
    if (m <= 0 || n <= 0 || (int64_t)m * n > (int64_t)INT32_MAX) return hipErrorInvalidValue;
    if (!x_fp16 || !w_fp16 || !y_fp16) return hipErrorInvalidValue;
    if (n % 8 == 0 && n <= 4096 &&
        ((reinterpret_cast<uintptr_t>(x_fp16) | reinterpret_cast<uintptr_t>(w_fp16) |
          reinterpret_cast<uintptr_t>(y_fp16)) & 15u) == 0) {
        const auto kernel = n <= 1024   ? lg::rms_norm_fp16_wave_kernel<2>
                            : n <= 2048 ? lg::rms_norm_fp16_wave_kernel<4>
                                        : lg::rms_norm_fp16_wave_kernel<8>;
        kernel<<<dim3((m + 3) / 4), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(
            static_cast<const lg::uint4_t*>(x_fp16), static_cast<const lg::uint4_t*>(w_fp16),
            static_cast<lg::uint4_t*>(y_fp16), m, n / 8, eps);
        return hipGetLastError();
    }
    lg::rms_norm_fp16_kernel<<<dim3(m), dim3(lg::kRowThreads), 0,
                               static_cast<hipStream_t>(stream)>>>(
        static_cast<const __half*>(x_fp16), static_cast<const __half*>(w_fp16),
        static_cast<__half*>(y_fp16), n, eps);
    return hipGetLastError();
}

extern "C" logismos_status_t logismos_launch_softmax_fp16(const void* x_fp16, void* y_fp16, int m,
                                                          int n, logismos_stream_t stream) {
    if (m <= 0 || n <= 0 || (int64_t)m * n > (int64_t)INT32_MAX) return hipErrorInvalidValue;
    if (!x_fp16 || !y_fp16) return hipErrorInvalidValue;
    lg::softmax_fp16_kernel<<<dim3(m), dim3(lg::kRowThreads), 0,
                              static_cast<hipStream_t>(stream)>>>(
        static_cast<const __half*>(x_fp16), static_cast<__half*>(y_fp16), n);
    return hipGetLastError();
}

extern "C" logismos_status_t logismos_launch_rope_fp16(void* qk_fp16, const void* cos_sin_f32,
                                                       int batch, int seq, int heads, int head_dim,
                                                       logismos_stream_t stream) {
    // `check_rope_shape` (crates/kernels/src/rope/mod.rs:79-130): positive dimensions, an even
    // head_dim, element counts within i32
    if (batch <= 0 || seq <= 0 || heads <= 0 || head_dim <= 0 || (head_dim & 1))
        return hipErrorInvalidValue;
    // the product is bounded factor by factor: four i32 factors can overflow i64 as well
    int64_t total = 1;
    for (int f : {batch, seq, heads, head_dim}) {
        if (total > (int64_t)INT32_MAX / f) return hipErrorInvalidValue;
        total *= f;
    }
    if (!qk_fp16 || !cos_sin_f32) return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(qk_fp16) & 3u) || (reinterpret_cast<uintptr_t>(cos_sin_f32) & 7u))
        return hipErrorInvalidValue;
    if (head_dim % 8 == 0 && seq <= 65535 && batch <= 65535 &&
        ((reinterpret_cast<uintptr_t>(qk_fp16) | reinterpret_cast<uintptr_t>(cos_sin_f32)) & 15u) == 0) {
        const int token_pieces = heads * (head_dim / 8);
        lg::rope_fp16_pieces_kernel<<<dim3((token_pieces + 255) / 256, seq, batch), dim3(256), 0,
                                      static_cast<hipStream_t>(stream)>>>(
            static_cast<lg::uint4_t*>(qk_fp16), static_cast<const lg::float4_t*>(cos_sin_f32),
            token_pieces, head_dim / 8);
        return hipGetLastError();
    }
    const int64_t total_pairs = total / 2;
    lg::rope_fp16_kernel<<<dim3((unsigned)((total_pairs + 255) / 256)), dim3(256), 0,
                           static_cast<hipStream_t>(stream)>>>(
        static_cast<unsigned*>(qk_fp16), static_cast<const float2*>(cos_sin_f32), total_pairs, seq,
        heads, head_dim / 2);
    return hipGetLastError();
}

extern "C" logismos_status_t logismos_launch_matmul_naive_fp16(const void* a_fp16,
                                                               const void* b_fp16, void* d_fp16,
                                                               int m, int n, int k,
                                                               logismos_stream_t stream) {
    if (!lg::matmul_shape_ok(m, n, k) || !a_fp16 || !b_fp16 || !d_fp16) return hipErrorInvalidValue;
    lg::matmul_naive_fp16_kernel<<<dim3((n + 63) / 64, (m + 3) / 4), dim3(256), 0,
                                   static_cast<hipStream_t>(stream)>>>(
        static_cast<const __half*>(a_fp16), static_cast<const __half*>(b_fp16),
        static_cast<__half*>(d_fp16), m, n, k);
    return hipGetLastError();
}

extern "C" logismos_status_t logismos_launch_matmul_wmma_fp16(const void* a_fp16,
                                                              const void* b_fp16, void* d_fp16,
                                                              int m, int n, int k,
                                                              logismos_stream_t stream) {
    if (!lg::matmul_shape_ok(m, n, k) || !a_fp16 || !b_fp16 || !d_fp16) return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(a_fp16) | reinterpret_cast<uintptr_t>(b_fp16)) & 15u)
        return hipErrorInvalidValue;
    if (n % 8 == 0 && k % 8 == 0) return lg::matmul_tiled(a_fp16, b_fp16, d_fp16, m, n, k, stream);
    lg::matmul_mfma_fp16_kernel<<<dim3((n + lg::kMmTile - 1) / lg::kMmTile,
                                       (m + lg::kMmTile - 1) / lg::kMmTile),
                                  dim3(256), 0, static_cast<hipStream_t>(stream)>>>(
        static_cast<const _Float16*>(a_fp16), static_cast<const _Float16*>(b_fp16),
        static_cast<_Float16*>(d_fp16), m, n, k);
    return hipGetLastError();
}
