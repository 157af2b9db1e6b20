// The fused few-row projections (qgemm_q4_rows.hip): arguments and launcher.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_utils.hpp"
#include "q4_common.hpp"

namespace lg {

constexpr int kRowsMax = 16;               // packed rows
constexpr int kRowsMaxNormWidth = 4096;    // residual width that fits the waves' registers
constexpr int kRowsMaxPrepWidth = 32768;   // K of the o and down projections (scales in registers)
constexpr int kRowsMaxQkv = 1 << 17;        // its tiles divide by a 20-bit reciprocal

// What is done to the products of a projection.
enum RowsEpilogue {
    kRowsF32 = 0,   // out_f32[b][N]
    kRowsRes = 1,   // h += product (N = the residual width)
    kRowsQkv = 2,   // bias, rotation, q out, K/V rows into fp16 pools
    kRowsSilu = 3,  // weights [2 * inter][K], gate rows first: act = bf16(silu(gate) * up) in
                    // the prepared layout (16 rows, no group sums) of the down projection
};

struct RowsEpilogueArgs {
    float* out_f32;  // kRowsF32; kRowsRes in two parts: the second part's products
    // what is still to be added to the residual stream, [b][its width], or null: the norm reads the stream with
    // it, kRowsRes adds it before its product
    const float* pending;
    uint4_t* act;    // kRowsSilu
    int inter;
    // kRowsQkv; tiles_per_head_inv = ceil(2^20 / (head_dim / 16))
    int hq, hkv, head_dim, max_pos;
    unsigned tiles_per_head_inv;
    const float* bias;
    const int32_t* positions;
    const float *cos_t, *sin_t;
    const int64_t* slots;
    __half *q_out, *k_pool, *v_pool;
};

struct RowsArgs {
    const uint4_t* xprep;  // without the norm: x in the prepared layout of 16 rows
    float* h;              // residual stream, row-major: input of the norm, and what kRowsRes adds to
    const float* gain;
    float eps;
    const uint8_t* qw;
    const __half *scale, *zero;
    int b, k, tiles;       // tiles of 16 weight rows
    RowsEpilogueArgs e;
};

// Whether a step of b rows with this residual width, widest other K and q/k/v outputs can run on
// these kernels with such weights.
bool qgemm_q4_rows_applies(int b, int hidden, int widest, int qkv, const void* scale,
                           const void* zero);
// norm: kRowsQkv, kRowsSilu, kRowsF32; otherwise kRowsRes.
hipError_t qgemm_q4_rows_launch(bool norm, int epilogue, const RowsArgs& args, hipStream_t st);
// Parts of K that kRowsRes takes for this product where out_f32 is given: of two, the second one's products go there.
int qgemm_q4_rows_res_parts(int tiles, int k);

// ---- device helpers of the kernels that multiply few rows by 16 weight rows at a time

__device__ __forceinline__ unsigned pack_bf16(float lo, float hi) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    const f2 v = {lo, hi};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2_t));
}

// The unpack's magic number and the ones of the sum MFMA, kept in registers.
struct RowsConst {
    unsigned magic;
    bf16x8_t ones;
    __device__ __forceinline__ RowsConst() {
        unsigned one;
        asm volatile("v_mov_b32 %0, 0x43004300" : "=v"(magic));
        asm volatile("v_mov_b32 %0, 0x3f803f80" : "=v"(one));
        ones = __builtin_bit_cast(bf16x8_t, uint4_t{one, one, one, one});
    }
};

// Sum of x over a group of K, per batch row, in the layout of the products.
__device__ __forceinline__ float4_t rows_group_sum(const uint4_t (&x)[4], const RowsConst& c) {
    float4_t s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4)
        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x[s4]), c.ones, s, 0, 0, 0);
    return s;
}

// x . q over one group of 128 columns of K, nibbles as bf16 128 + q.
__device__ __forceinline__ float4_t rows_product(const uint4_t& wv, const uint4_t (&x)[4], const RowsConst& c) {
    float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
        uint4_t h;
#pragma unroll
        for (int sft = 0; sft < 4; ++sft) h[sft] = ((wv[s4] >> (4 * sft)) & kNibMask) | c.magic;
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x[s4]),
                                                      __builtin_bit_cast(bf16x8_t, h), acc, 0, 0, 0);
    }
    return acc;
}

// y += one group: scale * (x . q - zero * sum(x)).
__device__ __forceinline__ void rows_group(float4_t& y, const uint4_t& wv, const uint4_t (&x)[4],
                                           const float4_t& xs, uint16_t scale, uint16_t zero,
                                           const RowsConst& c) {
    const float sf = __half2float(__ushort_as_half(scale));
    const float zf = 128.0f + __half2float(__ushort_as_half(zero));
    const float4_t acc = rows_product(wv, x, c);
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = fmaf(sf, fmaf(-zf, xs[e], acc[e]), y[e]);
}

// Groups [first, first + count) of wave w when `groups` are dealt to `waves` evenly.
__device__ __forceinline__ int2 rows_share(int groups, int waves, int w) {
    const int each = groups / waves, more = groups - each * waves;
    return int2{w * each + min(w, more), each + (w < more ? 1 : 0)};
}

}  // namespace lg
