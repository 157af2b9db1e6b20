// Q4G128 projections of a step with few packed rows (up to 16; one row over fp16 pools mostly takes
// decode_resident.hip, which is 1.18 to 1.34 times as fast there), with what surrounds them folded
// in: one launch is "norm -> projection -> what is done to each output".
//
//   A step of few rows is a chain of dependent launches whose inputs are a few KiB of
//   activations and the weights of one projection; each launch costs its boundary, one trip to
//   memory and its drain whatever it computes, so the chain's length is the step's time.  With
//   fp32 K parts between the operators a layer is ten launches; here it is six (five with one
//   attention partition; one more where attention cannot write the o projection's operand -- heads of
//   other widths than 128 with a chunk in the batch, or not 32 or 64 wide -- and a launch of its own
//   prepares its rows, and one more over 3-bit pools, where rotation and encoding follow the projection):
//     rows_norm<QKV>   RMSNorm of the residual rows, q/k/v projection, bias, rotation, q out,
//                      K/V rows into the pools
//     attention, merge
//     rows_prep<RES>   o projection added into the residual stream
//     rows_norm<SILU>  RMSNorm, gate and up projections, SwiGLU
//     rows_prep<RES>   down projection added into the residual stream
//
// * A workgroup owns tiles of 16 weight rows and ALL of K, so that a finished product exists in
//   one place: the waves split the groups of K between them and meet once in LDS.  That is what
//   lets the epilogue rotate, activate or add into the residual stream (nobody else reads or
//   writes those elements in the launch), and no K parts go to memory.
// * Everything a wave needs is requested before anything is waited for: its slices of the
//   weight rows as whole runs of 64 * GPW bytes (four lanes on 64 consecutive bytes), the
//   activations, and the tiles' scales and zeros, which are one contiguous block per eight
//   rows.  The weights pass through a private piece of LDS (written as loaded, read in the
//   operand layout: row stride 4 * GPW + 1 pieces, conflict-free; a wave's LDS queue is in
//   order, so nothing waits in between).
// * The norm: every workgroup normalises the rows for itself.  With up to 16 rows of up to 4096
//   columns that costs less than the launch it replaces.
// * The group sums of x for the zero-point term come from one more MFMA per operand against
//   ones: they land in the layout of the products.  (Without them the down projection would take
//   0.3-0.4 us less; having the producer deliver them costs more than that.)
//
// What bounds it, from clock stamps: 0.4-0.8 us until the workgroup's waves are there, about
// 0.5 us of address arithmetic, one trip to memory, then instructions: with four waves per SIMD
// every instruction of the prologue costs 16 clocks, so it is written for their number (one tile
// in flight, eight waves up to 8 rows of at most 2048 columns, a tile's head by a reciprocal from
// the host).  The root, the mean and its reciprocal are divisions and a root all the same, 0.1-0.2
// us of a launch, as in every other norm.  More
// tiles in flight are slower (six: 16.8 us instead of 12.9 for the 24576 x 4096 product): a
// wave whose requests fill the compute unit's queue stands still, and the others wait for its
// rows at the next barrier.
//
// The four projections of a layer with their norms, rotation and activation, us per layer, traced
// (the ten launches they replace):
//   hidden  896, 14 / 2 heads of 64, MLP 4864, one row       16.5 (40)
//   hidden 1536, 12 / 2 heads of 128, MLP 8960, 16 rows      29.8 (52)
//   hidden 4096, 32 / 8 heads of 128, MLP 12288, one row     36.7 (62)
// Whole steps: 24 layers of the first 1323 -> 784 us (674 since attention writes the operand), 28 of the second 1796 -> 1172, 36 of the third
// 2769 -> 1882.
#include "device_utils.hpp"
#include "launch_common.hpp"
#include "q4_common.hpp"
#include "q4_rows.hpp"

#include <hip/hip_fp16.h>
#include <math.h>

namespace lg {

namespace {

// A tile is two runs of eight weight rows, `rows_tile_first` and `rows_tile_apart` further on:
// for the rotation the two halves of its pairs, for the SwiGLU the gate and the up rows of the
// same outputs.
template <int EPI>
__device__ __forceinline__ int rows_tile_first(const RowsEpilogueArgs& e, int t) {
    if constexpr (EPI == kRowsSilu) {
        return 8 * t;
    } else if constexpr (EPI == kRowsQkv) {
        // head_dim / 16 tiles per head; the division through the reciprocal the host made
        const int h = (int)(((unsigned)t * e.tiles_per_head_inv) >> 20);
        return 8 * t + h * (e.head_dim >> 1);
    } else {
        return 16 * t;
    }
}
template <int EPI>
__device__ __forceinline__ int rows_tile_apart(const RowsEpilogueArgs& e) {
    return EPI == kRowsSilu ? e.inter : (EPI == kRowsQkv ? e.head_dim >> 1 : 8);
}

// A wave's slices (GPW groups) of the 16 weight rows of a tile, 16 bytes per lane and request,
// as whole runs of 64 * GPW bytes; put down row by row (stride 4 * GPW + 1 pieces) and read back
// as MFMA operands (lane = 16 rows x 4 pieces of a group).
template <int GPW>
struct RowsStage {
    static constexpr int PIECES = 4 * GPW;
    static constexpr int STRIDE = (PIECES + 1) * 16;
    static constexpr int BYTES = 16 * STRIDE;
    unsigned at[GPW];  // this lane's pieces, from the slice's start in the tile's first row
    __device__ __forceinline__ RowsStage(int apart, unsigned khalf, int lane) {
#pragma unroll
        for (int i = 0; i < GPW; ++i) {
            const int p = i * 64 + lane, row = p / PIECES, pc = p % PIECES;
            at[i] = (unsigned)((row & 7) + (row < 8 ? 0 : apart)) * khalf + (unsigned)pc * 16u;
        }
    }
    // slice: the wave's first group in the tile's first row (uniform)
    __device__ __forceinline__ void request(uint4_t (&wr)[GPW], const uint8_t* slice) const {
#pragma unroll
        for (int i = 0; i < GPW; ++i) {
            const uint4_t* src = reinterpret_cast<const uint4_t*>(slice + at[i]);
            // whole 128-byte lines past the caches (the activations stay there); a line that two
            // waves share goes through them
            if constexpr (GPW % 2 == 0)
                wr[i] = __builtin_nontemporal_load(src);
            else
                wr[i] = *src;
        }
    }
    static __device__ __forceinline__ void put(char* stage, const uint4_t (&wr)[GPW], int lane) {
#pragma unroll
        for (int i = 0; i < GPW; ++i) {
            const int p = i * 64 + lane;
            *reinterpret_cast<uint4_t*>(stage + (p / PIECES) * STRIDE + (p % PIECES) * 16) = wr[i];
        }
    }
    static __device__ __forceinline__ uint4_t get(const char* stage, int i, int lane) {
        return *reinterpret_cast<const uint4_t*>(stage + (lane & 15) * STRIDE + (4 * i + (lane >> 4)) * 16);
    }
};

// Scales and zeros of TILES tiles into LDS: eight weight rows are one contiguous block of 4 * G
// dwords of either array, a block is one wave's (or, with few blocks, several waves'): DW dwords
// per lane and block.  dst: [tile][16 rows][G] halves of scales, then of zeros.
template <int EPI, int WAVES, int TILES, int DW>
struct RowsScales {
    static constexpr int BLOCKS = 4 * TILES;
    static constexpr int PARTS = WAVES >= 2 * BLOCKS ? WAVES / BLOCKS : 1;
    static constexpr int STEP = WAVES / PARTS;
    static constexpr int ROUNDS = (BLOCKS + STEP - 1) / STEP;
    unsigned v[ROUNDS][DW];
    __device__ __forceinline__ void request(const __half* scale, const __half* zero,
                                            const RowsEpilogueArgs& e, int t0, int tiles, int G,
                                            int wave, int lane) {
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            const int block = wave / PARTS + r * STEP;  // (tile, array, half of its rows)
            const int row = rows_tile_first<EPI>(e, min(t0 + (block >> 2), tiles - 1)) +
                            ((block & 1) ? rows_tile_apart<EPI>(e) : 0);
            const unsigned* src = reinterpret_cast<const unsigned*>((block & 2) ? zero : scale) +
                                  (unsigned)row * (unsigned)G / 2;
#pragma unroll
            for (int d = 0; d < DW; ++d) {
                const int o = (d * PARTS + wave % PARTS) * 64 + lane;
                if (block < BLOCKS && o < 4 * G) v[r][d] = src[o];
            }
        }
    }
    __device__ __forceinline__ void put(int G, int wave, int lane, unsigned* dst) const {
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            const int block = wave / PARTS + r * STEP;
            unsigned* to = dst + ((block & 2) ? 8 * TILES * G : 0) + ((block >> 2) * 2 + (block & 1)) * 4 * G;
#pragma unroll
            for (int d = 0; d < DW; ++d) {
                const int o = (d * PARTS + wave % PARTS) * 64 + lane;
                if (block < BLOCKS && o < 4 * G) to[o] = v[r][d];
            }
        }
    }
};

// What is done to the finished product v of batch row r and weight row n (0..15) of a tile.  The
// 16 lanes of a row of lanes hold the 16 weight rows; all of them take part.  What it needs from
// memory is asked for long before (`early`, then `late`: the rotation factors are found by the
// token's position).
template <int EPI>
struct RowsFinish {
    float a = 0.0f, b = 0.0f;  // RES: the residual; QKV: cos, sin
    int pos = 0;
    int64_t slot = -1;
    float bias = 0.0f;

    template <bool PENDING = false>
    __device__ __forceinline__ void early(const RowsEpilogueArgs& e, const float* h, int tile,
                                          int tiles, int r, int n, bool ok) {
        if (!ok) return;
        if constexpr (EPI == kRowsRes) {
            const unsigned at = (unsigned)r * (unsigned)(16 * tiles) + (unsigned)(16 * tile + n);
            a = h[at];
            if constexpr (PENDING) a += e.pending[at];
        } else if constexpr (EPI == kRowsQkv) {
            pos = e.positions[r];
            slot = e.slots[r];
            if (e.bias)
                bias = e.bias[rows_tile_first<EPI>(e, tile) + (n & 7) + (n < 8 ? 0 : e.head_dim >> 1)];
        }
    }
    __device__ __forceinline__ void late(const RowsEpilogueArgs& e, int tile, int n, bool ok) {
        if constexpr (EPI == kRowsQkv) {
            const int head = (int)(((unsigned)tile * e.tiles_per_head_inv) >> 20);
            if (!ok || head >= e.hq + e.hkv) return;
            const int half = e.head_dim >> 1;
            const int i = 8 * (tile - head * (e.head_dim >> 4)) + (n & 7);  // rotation pair (i, i + d/2)
            const int p = pos < 0 ? 0 : (pos >= e.max_pos ? e.max_pos - 1 : pos);
            a = e.cos_t[(int64_t)p * half + i];
            b = e.sin_t[(int64_t)p * half + i];
        }
    }
    __device__ __forceinline__ void finish(const RowsEpilogueArgs& e, float* h, int tile, int tiles,
                                           int r, int n, float v, bool ok) const {
        if constexpr (EPI == kRowsRes) {
            if (ok) h[(unsigned)r * (unsigned)(16 * tiles) + (unsigned)(16 * tile + n)] = a + v;
        } else if constexpr (EPI == kRowsF32) {
            if (ok) e.out_f32[(unsigned)r * (unsigned)(16 * tiles) + (unsigned)(16 * tile + n)] = v;
        } else if constexpr (EPI == kRowsSilu) {
            const float up = lane_xor_f32<8>(v);
            if (ok && n < 8) {
                const float act = v / (1.0f + expf(-v)) * up;
                uint16_t* dst = reinterpret_cast<uint16_t*>(e.act + (unsigned)tile * 16u + r);
                dst[2 * (n & 3) + (n >> 2)] = f32_to_bf16_rne(act);
            }
        } else {
            v += bias;
            const float other = lane_xor_f32<8>(v);
            if (!ok) return;
            const int d = e.head_dim, hq = e.hq, hkv = e.hkv;
            const int head = (int)(((unsigned)tile * e.tiles_per_head_inv) >> 20);
            const int at = 8 * (tile - head * (d >> 4)) + (n & 7) + (n < 8 ? 0 : d >> 1);
            float res = v;
            if (head < hq + hkv) {
                // the two halves of rope_rotate (step_ops.hip), rounded alike
                res = n < 8 ? fmaf(v, a, -(other * b)) : fmaf(other, b, v * a);
                asm volatile("" : "+v"(res));
            }
            if (head < hq) {
                e.q_out[((int64_t)r * hq + head) * d + at] = __float2half_rn(res);
            } else if (slot >= 0) {
                __half* pool = head < hq + hkv ? e.k_pool : e.v_pool;
                const int kvh = head < hq + hkv ? head - hq : head - hq - hkv;
                pool[(slot * hkv + kvh) * d + at] = __float2half_rn(res);
            }
        }
    }
};

// Waves that share a batch row while the rows are normalised (nw >= b).
__host__ __device__ __forceinline__ int rows_waves_per_row(int nw, int b) {
    return nw / (b > 8 ? 16 : (b > 4 ? 8 : (b > 2 ? 4 : b)));
}

// The sums of W waves' partial products (16 x 16 floats in the MFMA layout, 1 KiB apart by
// `step`) of batch row r and weight row n.
template <int W>
__device__ __forceinline__ float rows_meet(const char* src, int step, int r, int n) {
    float v[W];
#pragma unroll
    for (int w = 0; w < W; ++w)
        v[w] = *reinterpret_cast<const float*>(src + w * step + ((r >> 2) * 16 + n) * 16 + (r & 3) * 4);
    float s = v[0];
#pragma unroll
    for (int w = 1; w < W; ++w) s += v[w];
    return s;
}

// RMSNorm -> projection.  NW waves as NW / W teams of W waves; a team's waves split the groups
// of K (at most GPW each) and the team takes every (NW / W)-th tile of the workgroup's
// TN * NW / W tiles.  The workgroup normalises the rows once, through LDS, and each wave keeps
// its slice of them in registers for all its tiles.
constexpr int kRowsLds = 160 * 1024;

// LDS: [scales and zeros][sums of squares][rows, gains][staging, exchange]; the last two share
// their place where the whole does not fit otherwise.
struct RowsNormLds {
    int ssq, x, stage, bytes;
    __host__ RowsNormLds(int tiles, int stage_bytes, int red_bytes, int b, int k) {
        ssq = tiles * 16 * (k >> 7) * 4;
        x = ssq + 16 * 16 * 4;
        const int rows = b * (2 * k + 16) + 4 * k, rest = stage_bytes + red_bytes;
        const bool apart = x + rows + rest <= kRowsLds;
        stage = apart ? x + rows : x;
        bytes = apart ? stage + rest : x + (rows > rest ? rows : rest);
    }
};

// CR: chunks of the rows per lane.  PENDING: the stream is h with what is pending.
template <int EPI, int NW, int W, int GPW, int TN, int CR, bool PENDING>
__global__ __launch_bounds__(64 * NW) void qgemm_q4g128_rows_norm_kernel(
    const float* __restrict__ h, const float* __restrict__ gain, const uint8_t* __restrict__ qw,
    const __half* __restrict__ scale, const __half* __restrict__ zero, int b, int k, int tiles,
    float eps, int lds_ssq, int lds_x, int lds_stage, const RowsEpilogueArgs e) {
    using Stage = RowsStage<GPW>;
    constexpr int TEAMS = NW / W;
    constexpr int TILES = TN * TEAMS;
    constexpr int THREADS = 64 * NW;
    constexpr int GR = 1024 / THREADS;  // gain chunks of four columns per thread
    extern __shared__ __attribute__((aligned(16))) char lds[];
    uint16_t* const sz = reinterpret_cast<uint16_t*>(lds);
    float* const ssq = reinterpret_cast<float*>(lds + lds_ssq);  // [row][part of the row]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int team = wave / W, member = wave % W;
    const int G = k >> 7;
    const unsigned khalf = (unsigned)k >> 1;
    const int t0 = blockIdx.x * TILES;

    // ---- the rows: wpr waves share a row, a lane takes whole chunks of 8 columns
    const int wpr = rows_waves_per_row(NW, b);
    const int row = wave / wpr, part = wave - row * wpr;
    const int chunks = k >> 3;
    const bool mine = row < b;
    float4_t hv[CR][2];
    const float* hrow = h + (unsigned)(mine ? row : 0) * (unsigned)k;
#pragma unroll
    for (int i = 0; i < CR; ++i) {
        if (i * wpr * 64 < chunks) {  // uniform
            const int c = min((i * wpr + part) * 64 + lane, chunks - 1);
            hv[i][0] = *reinterpret_cast<const float4_t*>(hrow + 8 * c);
            hv[i][1] = *reinterpret_cast<const float4_t*>(hrow + 8 * c + 4);
        }
    }
    if constexpr (PENDING) {
        const float* prow = e.pending + (unsigned)(mine ? row : 0) * (unsigned)k;
#pragma unroll
        for (int i = 0; i < CR; ++i) {
            if (i * wpr * 64 < chunks) {
                const int c = min((i * wpr + part) * 64 + lane, chunks - 1);
                hv[i][0] += *reinterpret_cast<const float4_t*>(prow + 8 * c);
                hv[i][1] += *reinterpret_cast<const float4_t*>(prow + 8 * c + 4);
            }
        }
    }
    const unsigned xrow = (unsigned)(2 * k + 16);  // bytes per row of x, off the banks' period
    float4_t* const gains = reinterpret_cast<float4_t*>(lds + lds_x + (unsigned)b * xrow);
    float4_t gv[GR];
#pragma unroll
    for (int i = 0; i < GR; ++i)
        if (4 * (i * THREADS + tid) < k) gv[i] = *reinterpret_cast<const float4_t*>(gain + 4 * (i * THREADS + tid));
    RowsScales<EPI, NW, TILES, W * GPW <= 16 ? 1 : 2> scales;
    scales.request(scale, zero, e, t0, tiles, G, wave, lane);
    // this wave's groups: a slice of GPW groups (moved back to end with the last one), of which
    // the groups lo .. hi - 1 are its own
    const int2 share = rows_share(G, W, member);
    const int g0 = min(share.x, G - GPW);
    const int lo = share.x - g0, hi = lo + share.y;
    const Stage slices(rows_tile_apart<EPI>(e), khalf, lane);
    uint4_t wr[GPW];
    auto request = [&](int u) {
        const int first = rows_tile_first<EPI>(e, min(t0 + u * TEAMS + team, tiles - 1));
        slices.request(wr, qw + ((unsigned)first * khalf + (unsigned)g0 * 64u));
    };
    request(0);
    const int fr = (tid >> 4) & 15, fn = tid & 15, ft = t0 + (tid >> 8);
    const bool fok = (4 * TILES >= NW || tid < TILES * 256) && ft < tiles && fr < b;
    RowsFinish<EPI> first;
    first.early(e, nullptr, ft, tiles, fr, fn, fok);

    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < CR; ++i) {
        if (i * wpr * 64 < chunks) {
            float s = 0.0f;
#pragma unroll
            for (int v = 0; v < 2; ++v)
#pragma unroll
                for (int c = 0; c < 4; ++c) s = fmaf(hv[i][v][c], hv[i][v][c], s);
            ss += (i * wpr + part) * 64 + lane < chunks ? s : 0.0f;
        }
    }
    ss = wave_sum(ss);
    if (lane == 0) ssq[row * 16 + part] = mine ? ss : 0.0f;
#pragma unroll
    for (int i = 0; i < GR; ++i)
        if (4 * (i * THREADS + tid) < k) gains[i * THREADS + tid] = gv[i];
    __syncthreads();
    const float total = row16_sum((lane & 15) < wpr ? ssq[row * 16 + (lane & 15)] : 0.0f);
    const float inv = 1.0f / sqrtf(total / (float)k + eps);
#pragma unroll
    for (int i = 0; i < CR; ++i) {
        const int c = (i * wpr + part) * 64 + lane;
        if (i * wpr * 64 < chunks && mine && c < chunks) {
            const float4_t w0 = gains[2 * c], w1 = gains[2 * c + 1];
            uint4_t o;  // pair order: (x0, x4) (x1, x5) (x2, x6) (x3, x7)
#pragma unroll
            for (int p = 0; p < 4; ++p) o[p] = pack_bf16(hv[i][0][p] * inv * w0[p], hv[i][1][p] * inv * w1[p]);
            *reinterpret_cast<uint4_t*>(lds + lds_x + (unsigned)row * xrow + c * 16) = o;
        }
    }
    scales.put(G, wave, lane, reinterpret_cast<unsigned*>(sz));
    __syncthreads();
    // (rows past the batch repeat its last one: a row of x only reaches its own row of the product)
    uint4_t x[GPW][4];
    float4_t xs[GPW];
    const RowsConst cst;
    const char* const xsrc = lds + lds_x + (unsigned)min(lane & 15, b - 1) * xrow + (lane >> 4) * 64 + g0 * 256;
#pragma unroll
    for (int i = 0; i < GPW; ++i)
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4)
            x[i][s4] = *reinterpret_cast<const uint4_t*>(xsrc + i * 256 + s4 * 16);
#pragma unroll
    for (int i = 0; i < GPW; ++i) xs[i] = rows_group_sum(x[i], cst);
    first.late(e, ft, fn, fok);
    if (lds_stage == lds_x) __syncthreads();  // the staging area takes the place of the rows

    char* const stage = lds + lds_stage + wave * Stage::BYTES;
    char* const red = lds + lds_stage + NW * Stage::BYTES;  // [tile of the team][wave][lane]
#pragma unroll
    for (int u = 0; u < TN; ++u) {
        Stage::put(stage, wr, lane);
        if (u + 1 < TN) request(u + 1);
        float4_t y = {0.0f, 0.0f, 0.0f, 0.0f};
        const uint16_t* s = sz + ((u * TEAMS + team) * 16 + (lane & 15)) * G + g0;
#pragma unroll
        for (int i = 0; i < GPW; ++i) {
            if (i < lo || i >= hi) continue;  // uniform
            rows_group(y, Stage::get(stage, i, lane), x[i], xs[i], s[i], s[TILES * 16 * G + i], cst);
        }
        *reinterpret_cast<float4_t*>(red + (u * NW + wave) * 1024 + lane * 16) = y;
    }
    __syncthreads();
#pragma unroll
    for (int o0 = 0; o0 < TILES * 256; o0 += THREADS) {
        const int o = o0 + tid;
        if (o >= TILES * 256) break;
        const int t = o >> 8;
        const float v = rows_meet<W>(red + ((t / TEAMS) * NW + (t % TEAMS) * W) * 1024, 1024, fr, fn);
        if (o0 == 0) {
            first.finish(e, nullptr, ft, tiles, fr, fn, v, fok);
        } else {
            RowsFinish<EPI> f;
            const bool ok = t0 + t < tiles && fr < b;
            f.early(e, nullptr, t0 + t, tiles, fr, fn, ok);
            f.late(e, t0 + t, fn, ok);
            f.finish(e, nullptr, t0 + t, tiles, fr, fn, v, ok);
        }
    }
}

// Projection of prepared rows: one tile per workgroup, the waves split the groups of K, SETS
// groups of a wave in flight.  K may be cut in two parts (grid y): the first adds to the residual stream, the
// second's products are left to the operators behind it.  (Modes of their own: an argument that a launch does not
// need is a load in front of everything else, 1.5 % of a step of 8 rows at width 4096.)
enum RowsPrepMode { kPrepPlain = 0, kPrepPending = 1, kPrepTwoParts = 2 };
template <int EPI, int W, int DW, int MODE>
__global__ __launch_bounds__(64 * W) void qgemm_q4g128_rows_prep_kernel(
    const uint4_t* __restrict__ xprep, const uint8_t* __restrict__ qw, const __half* __restrict__ scale,
    const __half* __restrict__ zero, float* __restrict__ h, int b, int k, int tiles,
    const RowsEpilogueArgs e) {
    using Stage = RowsStage<1>;
    constexpr int SETS = 3;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    uint16_t* const sz = reinterpret_cast<uint16_t*>(lds + W * Stage::BYTES);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = k >> 7;
    const unsigned khalf = (unsigned)k >> 1;
    const int tile = blockIdx.x;
    const bool second = MODE == kPrepTwoParts && blockIdx.y != 0;
    const int half = (G + 1) >> 1;
    int2 share = rows_share(MODE != kPrepTwoParts ? G : (second ? G - half : half), W, wave);
    if (second) share.x += half;
    const int end = share.x + share.y;
    char* const stage = lds + wave * Stage::BYTES;

    RowsScales<EPI, W, 1, DW> scales;
    scales.request(scale, zero, e, tile, tiles, G, wave, lane);
    const Stage slices(rows_tile_apart<EPI>(e), khalf, lane);
    const uint8_t* const wtile = qw + (unsigned)rows_tile_first<EPI>(e, tile) * khalf;
    uint4_t wr[SETS][1], x[SETS][4];
    const unsigned xlane = (unsigned)((lane >> 4) * 4 * 16 + min(lane & 15, b - 1));
    auto request = [&](int set, int g) {
        slices.request(wr[set], wtile + g * 64);
        const uint4_t* src = xprep + g * 256;
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) x[set][s4] = src[xlane + s4 * 16];
    };
#pragma unroll
    for (int s = 0; s < SETS; ++s)
        if (share.x + s < end) request(s, share.x + s);
    const int fr = (tid >> 4) & 15, fn = tid & 15;
    const bool fok = tid < 256 && fr < b;
    RowsFinish<EPI> fin;
    fin.template early<MODE == kPrepPending>(e, h, tile, tiles, fr, fn, fok && !second);
    const RowsConst cst;
    float4_t y = {0.0f, 0.0f, 0.0f, 0.0f};
    scales.put(G, wave, lane, reinterpret_cast<unsigned*>(sz));
    __syncthreads();
    const uint16_t* const srow = sz + (lane & 15) * G;
    for (int g = share.x; g < end; g += SETS) {
#pragma unroll
        for (int s = 0; s < SETS; ++s) {
            if (g + s >= end) break;  // uniform
            Stage::put(stage, wr[s], lane);
            rows_group(y, Stage::get(stage, 0, lane), x[s], rows_group_sum(x[s], cst), srow[g + s],
                       srow[16 * G + g + s], cst);
            if (g + s + SETS < end) request(s, g + s + SETS);
        }
    }
    *reinterpret_cast<float4_t*>(stage + lane * 16) = y;
    __syncthreads();
    if (tid < 256) {
        const float v = rows_meet<W>(lds, Stage::BYTES, fr, fn);
        if (!second) fin.finish(e, h, tile, tiles, fr, fn, v, fok);
        else if (fok) e.out_f32[(unsigned)fr * (unsigned)(16 * tiles) + (unsigned)(16 * tile + fn)] = v;
    }
}

template <typename K>
hipError_t rows_opt_in(K kernel) {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, kRowsLds);
}

template <int EPI, int NW, int W, int GPW, int TN, int CR, bool PENDING = false>
hipError_t rows_norm_launch(const RowsArgs& a, hipStream_t st) {
    // (only widths of up to 2048 have something pending, in front of the q/k/v projection)
    if constexpr (!PENDING && EPI != kRowsSilu && W * GPW <= 16)
        if (a.e.pending) return rows_norm_launch<EPI, NW, W, GPW, TN, CR, true>(a, st);
    const auto kernel = qgemm_q4g128_rows_norm_kernel<EPI, NW, W, GPW, TN, CR, PENDING>;
    static const hipError_t opt_in = rows_opt_in(kernel);
    if (opt_in != hipSuccess) return opt_in;
    constexpr int tiles = TN * NW / W;
    const RowsNormLds l(tiles, NW * RowsStage<GPW>::BYTES, TN * NW * 1024, a.b, a.k);
    kernel<<<dim3((unsigned)((a.tiles + tiles - 1) / tiles)), dim3(64 * NW), (size_t)l.bytes, st>>>(
        a.h, a.gain, a.qw, a.scale, a.zero, a.b, a.k, a.tiles, a.eps, l.ssq, l.x, l.stage, a.e);
    return hipGetLastError();
}

template <int EPI, int NW, int W, int GPW, int CR>
hipError_t rows_norm_by_n(const RowsArgs& a, hipStream_t st) {
    const int per = (a.tiles * W / NW + device_cu_count() - 1) / device_cu_count();
    if (per <= 1) return rows_norm_launch<EPI, NW, W, GPW, 1, CR>(a, st);
    if (per <= 2) return rows_norm_launch<EPI, NW, W, GPW, 2, CR>(a, st);
    if (per <= 3 || EPI != kRowsSilu) return rows_norm_launch<EPI, NW, W, GPW, 3, CR>(a, st);
    if constexpr (EPI == kRowsSilu) {
        if (per <= 4) return rows_norm_launch<EPI, NW, W, GPW, 4, CR>(a, st);
        if (per <= 5) return rows_norm_launch<EPI, NW, W, GPW, 5, CR>(a, st);
        return rows_norm_launch<EPI, NW, W, GPW, 6, CR>(a, st);
    }
    return hipErrorInvalidValue;
}

// chunks of 8 columns a lane holds: waves_per_row waves share a row.  (More than four only with
// more than 2048 columns, one only where fewer than nine rows share the waves or K is short.)
template <int EPI, int NW, int W, int GPW>
hipError_t rows_norm_by_b(const RowsArgs& a, hipStream_t st) {
    const int wpr = rows_waves_per_row(NW, a.b);
    const int cr = ((a.k >> 3) + 64 * wpr - 1) / (64 * wpr);
    if constexpr (W * GPW > 16)
        if (cr > 4) return rows_norm_by_n<EPI, NW, W, GPW, 8>(a, st);
    if constexpr (NW == W || GPW == 1)
        if (cr <= 1) return rows_norm_by_n<EPI, NW, W, GPW, 1>(a, st);
    return rows_norm_by_n<EPI, NW, W, GPW, 4>(a, st);
}

template <int EPI>
hipError_t rows_norm(const RowsArgs& a, hipStream_t st) {
    const int g = a.k >> 7;
    if (a.b <= 8) {
        if (g <= 8) return rows_norm_by_b<EPI, 8, 8, 1>(a, st);
        if (g <= 16) return rows_norm_by_b<EPI, 8, 8, 2>(a, st);
    }
    if (g <= 8) return rows_norm_by_b<EPI, 16, 8, 1>(a, st);
    if (g <= 16) return rows_norm_by_b<EPI, 16, 8, 2>(a, st);
    return rows_norm_by_b<EPI, 16, 16, 2>(a, st);
}

template <int W, int DW, int MODE>
hipError_t rows_prep_launch(const RowsArgs& a, hipStream_t st) {
    const auto kernel = qgemm_q4g128_rows_prep_kernel<kRowsRes, W, DW, MODE>;
    static const hipError_t opt_in = rows_opt_in(kernel);
    if (opt_in != hipSuccess) return opt_in;
    const int lds = W * RowsStage<1>::BYTES + 16 * (a.k >> 7) * 4;
    kernel<<<dim3((unsigned)a.tiles, MODE == kPrepTwoParts ? 2u : 1u), dim3(64 * W), (size_t)lds, st>>>(
        a.xprep, a.qw, a.scale, a.zero, a.h, a.b, a.k, a.tiles, a.e);
    return hipGetLastError();
}
template <int W, int DW>
hipError_t rows_prep(const RowsArgs& a, hipStream_t st) {
    if constexpr (W == 16)  // (two parts are of more groups than eight waves ever take)
        if (a.e.out_f32 && qgemm_q4_rows_res_parts(a.tiles, a.k) == 2) return rows_prep_launch<W, DW, kPrepTwoParts>(a, st);
    if (a.e.pending) return rows_prep_launch<W, DW, kPrepPending>(a, st);
    return rows_prep_launch<W, DW, kPrepPlain>(a, st);
}

}  // namespace

bool qgemm_q4_rows_applies(int b, int hidden, int widest, int qkv, const void* scale,
                           const void* zero) {
    const uintptr_t al = reinterpret_cast<uintptr_t>(scale) | reinterpret_cast<uintptr_t>(zero);
    return b >= 1 && b <= kRowsMax && hidden % 128 == 0 && hidden <= kRowsMaxNormWidth &&
           widest <= kRowsMaxPrepWidth && qkv <= kRowsMaxQkv && (al & 3u) == 0;
}

// Two parts where a wave of one has more groups than it keeps in flight (16 waves of three groups), both
// parts' workgroups, one to a compute unit, run at once, and the norm that takes the rest is one of the narrow ones
// (up to 2048 columns): 1536 x 8960 is 96 workgroups of 70 groups.  28 layers of it, us per step, one part / two:
// 2 rows 899 / 854, 8 rows 936 / 912, 12 rows 1055 / 1010, 16 rows 1157 / 1108.  Eight layers of widths 512 to 2048 with
// 6400 to 16384, 2 to 16 rows: 0.935 to 0.99 of one part's time up to 1536, 0.96 to 1.006 at 2048 (2 rows of 512 x 6400
// 207.7 / 201.2, 16 of 2048 x 16384 364.4 / 364.4).  The norm that reads the rest pays part of it back: q/k/v of 1536 at 16
// rows takes 7.8 instead of 6.5, the down projection 6.9 instead of 10.1.  (From 24 groups on, 896 x 4864 of 56
// workgroups too: no difference.)
int qgemm_q4_rows_res_parts(int tiles, int k) {
    return (k >> 7) > 48 && tiles <= 128 && 2 * tiles <= device_cu_count() ? 2 : 1;
}

hipError_t qgemm_q4_rows_launch(bool norm, int epilogue, const RowsArgs& a, hipStream_t st) {
    if (norm) {
        if (epilogue == kRowsQkv) return rows_norm<kRowsQkv>(a, st);
        if (epilogue == kRowsSilu) return rows_norm<kRowsSilu>(a, st);
        return rows_norm<kRowsF32>(a, st);
    }
    // DW: 4 * K / 128 dwords of scales over 64 * W / 4 lanes
    if (a.k <= 2048) return rows_prep<8, 1>(a, st);
    if (a.k <= 8192) return rows_prep<16, 1>(a, st);
    if (a.k <= 16384) return rows_prep<16, 2>(a, st);
    return rows_prep<16, 4>(a, st);
}

}  // namespace lg
