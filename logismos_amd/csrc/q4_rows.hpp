// The fused few-row projections (qgemm_q4_rows.hip): arguments and launcher.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_utils.hpp"

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
    float* out_f32;  // kRowsF32
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

}  // namespace lg
