// Q4G128 GEMM for a tall x over a workspace: the tiled kernel of qgemm_q4_tall.hip with the
// work that does not belong in its inner loop taken out of it.
//   y[m][n] = sum_k x[m][k] * (q[n][k] - zero[n][k/128]) * scale[n][k/128] (+ bias[n])
// `cpu_f32::linear_t` (crates/kernels/src/cpu_f32/mod.rs:271-345) at m = hundreds to thousands
// of rows over the dequantised matrix.
//
// Counters of the workspace-less kernel show its vector pipe, not its matrix pipe, setting the
// pace: per 32 MFMAs a wave issues ~500 vector instructions -- the nibble unpack (112), the
// staging of x through registers into LDS with the pair-order permute and the group sums
// (~130), and two multiply-adds per result and group for scale and zero point (128).  Here:
//
// * a first pass (`q4_tall_prepare_kernel`, x read once, ~1 % of the product's time) writes x
//   in the order the nibble unpack produces ("pair order": (x0,x4)(x1,x5)(x2,x6)(x3,x7) per
//   16-byte chunk), rows padded with zeros to a multiple of 128, and every row's sum over each
//   group of 128 columns;
// * the product kernel (128 x 256 tiles of eight waves, one workgroup per CU; where K is
//   short also 64 x 256, one per CU, and 64 x 128 of four waves, two per CU) moves a
//   group's slab of that copy (128 columns) and its tile of nibbles from global
//   memory STRAIGHT into LDS (global_load_lds, 16 bytes per lane, no registers, no vector
//   instructions) into a ring of three buffers, requested two groups ahead, one barrier per
//   group.  A request writes 1 KiB of consecutive LDS, so instead of padding rows the
//   16-byte chunks of a row are stored XOR-swizzled by the row index and the ds_read_b128 of
//   the MFMA operands stay conflict-free;
// * a wave takes ALL rows of the tile by 32 weight rows, so that no two waves unpack the same nibbles:
//   56 vector instructions of unpack per 32 MFMAs instead of the 112 of 64 x 64 parts, for an LDS
//   operand read per MFMA instead of one per two (at 256 bytes per clock, the rate of 16-byte reads, these
//   take 1100 clocks by count, of the 3600 that a group's 1.75 us are at about 2.05 GHz);
// * the requests go out one per step of 16 columns.  Issued together behind the barrier, all eight
//   waves waited in front of the texture addresser (48 requests x 16 cycles) with the matrix pipe
//   idle: a build without any requests was 15 % faster, and this one gets most of that back.
//   The wait and the barrier stand in the middle of a group and the first operands of the next are
//   read in its last step, so that nothing is waited for between two groups.  Bit for bit the
//   same products.  4000 rows, us before / now: 6144 x 4096 206 / 180, 4096 x 12288 380 / 347,
//   24576 x 4096 with the activation 778 / 737, 1536 x 8960 144 / 113; 195 rows: 30.0 / 27.9,
//   44.0 / 40.7, 59.7 / 55.2, 26.8 / 24.4;
// * scales, zeros and the group sums of x reach a lane's registers for four (or two) pairs
//   of groups per load where K allows: a lane's row of scales is 64 bytes apart from the
//   next lane's, so each such load costs the address path a cache line per lane -- one per
//   pair and array, they took it twice as long as the tiles themselves and held every wave
//   up behind each barrier.  The first pass writes the group sums in the layout these loads
//   want ([row tile][block of pairs][group's place in its pair][row][pair]);
// * the zero-point term -scale * (128 + zero) * sum_x is a rank-(K/128) product of its own:
//   one v_mfma_f32_32x32x2_f32 per output tile and PAIR of groups, accumulating into the same
//   registers, in place of a multiply-add per result and group (an odd number of groups: one per
//   group, into the group's own sum);
// * what is left per group and wave: the unpack (a lane of the v_mfma_f32_32x32x16_bf16 B
//   operand is one weight row and one dword of nibbles, made bf16 `128 + q` with an and-or per
//   pair, exact), one multiply-add per result for the group's scale, 32 MFMAs.  At 4000 rows a group
//   takes 1.75 us, of which the matrix pipe needs 1.12 at the clock the board's power leaves.
//
// * workgroups all take the same time and a CU holds one, so a launch whose tile count is not
//   a multiple of the CU count ends on a round that leaves most CUs idle (config 4's o and
//   down projections: 1040 tiles on 256 CUs, a fifth round for 16 tiles).  The tiles of that
//   last partial round are split over K into parts, one workgroup each, that write fp32
//   partial tiles into the workspace; `q4_tall_reduce_kernel` sums a tile's parts in part
//   order (deterministic), adds the bias and writes y.  A launch of fewer tiles than CUs is
//   all "last round": the split also fills the device at a few hundred rows.
//
// LDS is only touched through inline assembly inside the loop: the compiler would order
// every LDS access it can see behind all outstanding global_load_lds.
#include "device_utils.hpp"
#include "launch_common.hpp"
#include "q4_common.hpp"

#include <hip/hip_fp16.h>
#include <type_traits>

namespace lg {

typedef __attribute__((address_space(3))) void* tp_lds_ptr_t;

// A workgroup's tile: 32 * BLOCKS rows of x by 32 weight rows for each of its WAVES waves.
// CUTS: adds up in the parts a 128 x 256 tile would be split into (32 more registers; the code for it
// costs 0.3-0.9 us of a launch, about 0.2 us of one that has no parts).
template <int BLOCKS, int WAVES, bool CUTS = false>
struct TpTile {
    static constexpr int kBlocks = BLOCKS, kWaves = WAVES;
    static constexpr int kM = 32 * BLOCKS, kN = 32 * WAVES;
    static constexpr int kSlabBytes = kM * 256;  // one group's slab of x: kM rows x 128 bf16
    static constexpr int kBufBytes = kSlabBytes + kN * 64;  // ... and its tile of nibbles
    static constexpr int kXRequests = kM / 4 / kWaves;      // 1 KiB requests of x per wave
    static constexpr bool kBig = BLOCKS == 4 && WAVES == 8;
    static constexpr bool kCuts = CUTS;
    static_assert(BLOCKS == 2 || BLOCKS == 4, "what the operand reads spell out");
    static_assert(kXRequests == 2 || kXRequests == 4, "what request_x spells out");
};
using TpBig = TpTile<4, 8>;
template <bool CUTS>
using TpHalf = TpTile<2, 8, CUTS>;
template <bool CUTS>
using TpSmall = TpTile<2, 4, CUTS>;
constexpr int kTpTileM = TpBig::kM;  // 128 rows of x per workgroup
constexpr int kTpTileN = TpBig::kN;  // 256 weight rows per workgroup
constexpr int kTpBufs = 3;                // groups in LDS: one in use, two on their way

constexpr int kTpTileElems = kTpTileM * kTpTileN;
constexpr int kTpMaxParts = 512;          // partial tiles the workspace holds (fp32, 128 KiB each)
constexpr int kTpMinGroupsPerPart = 4;    // a part of a tile takes at least four groups of K

static_assert(kTpTileM == kTallTileRows, "the layout helpers of q4_common.hpp are for this tile");
__host__ __device__ inline int tp_padded_rows(int m) { return tall_padded_rows(m); }
__host__ __device__ inline size_t tp_sums_offset(int m, int k) { return tall_sums_offset(m, k); }
__host__ __device__ inline size_t tp_partials_offset(int m, int k) {
    // (whole pairs of groups: the sums of a missing last group have a place, which nothing uses)
    return (tp_sums_offset(m, k) + (size_t)tp_padded_rows(m) * ((k / 128 + 1) & ~1) * 4 + 255) &
           ~(size_t)255;
}

// How a launch of `tiles` workgroup tiles is laid over `cus` CUs: the first `full` tiles whole,
// the other `tiles - full` (the last, partial round) in `split` parts over K each.
struct TpPlan {
    int full, split;
};
inline TpPlan tp_plan(int tiles, int groups, int block_groups, int cus) {
    const int rem = tiles % cus;
    TpPlan p{tiles, 1};
    if (rem == 0) return p;
    int split = cus / rem;
    // parts are whole blocks of the kernel's small loads and at least four groups
    const int most = groups / (block_groups > kTpMinGroupsPerPart ? block_groups : kTpMinGroupsPerPart);
    if (split > most) split = most;
    if (split > 1 && rem * split <= kTpMaxParts) p = TpPlan{tiles - rem, split};
    return p;
}

// x [m][k] bf16 -> xp [m_pad][k] bf16 in pair order (rows >= m: zeros), xs: the fp32 sum of the
// bf16 values of every row and group, laid out for the product kernel's loads as
// [row tile of 128][block of w pairs of groups][group's place in its pair][row][pair].
// One thread per 16-byte chunk; the 16 lanes of a row of lanes hold one group of one row.
__global__ __launch_bounds__(256) void q4_tall_prepare_kernel(const uint16_t* __restrict__ x,
                                                             uint16_t* __restrict__ xp,
                                                             float* __restrict__ xs, int m,
                                                             int m_pad, int k, int w) {
    const int64_t chunks_per_row = k >> 3;
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= (int64_t)m_pad * chunks_per_row) return;  // (whole rows of 16 lanes: k % 128 == 0)
    const int64_t row = id / chunks_per_row;
    const int64_t c = id - row * chunks_per_row;
    uint4_t v = {0u, 0u, 0u, 0u};
    if (row < m) v = *reinterpret_cast<const uint4_t*>(x + row * k + c * 8);
    const float gs = row16_sum(sum8_bf16(v));
    *reinterpret_cast<uint4_t*>(xp + row * k + c * 8) = pair_order(v);
    if ((threadIdx.x & 15) == 0) xs[tall_sum_index(row, (int)(c >> 4), k, w)] = gs;
}

// W values a lane loads at once, as one register operand of an assembly statement: a vector
// of W, or the plain value for W = 1 (a vector of one is no register operand).
template <typename T, int W>
struct TpRegs {
    typedef T raw_t __attribute__((ext_vector_type(W)));
    raw_t raw;
    __device__ __forceinline__ T operator[](int i) const { return raw[i]; }
};
template <typename T>
struct TpRegs<T, 1> {
    typedef T raw_t;
    raw_t raw;
    __device__ __forceinline__ T operator[](int) const { return raw; }
};

// What a launch writes.  kTpOutSwiglu: the weights are a gate/up pair [gate rows | up rows]
// (2 n rows) and y [m][n] is bf16 silu(gate) * up -- a workgroup tile takes as many gate rows as
// up rows of the same outputs, a wave's first 16 columns the gate and its other 16 the up values of
// the same 16 outputs, which the two halves of a row of 32 lanes exchange at the end, so that the fp32
// gate/up products (a gigabyte at 8240 rows of a 12288-wide MLP) never go to memory.
// kTpOutSwigluOperand: the same product, written as the operand of a following launch of this
// kernel over K = n (n a multiple of 256): y is that launch's workspace -- the bf16 values in
// pair order, rows up to the padded count (the padding rows of x are zeros, and so are their
// activations), and the group sums (a tile's 128 outputs are one group), added up in the order
// of the first pass (`q4_tall_prepare_kernel`), so that the workspace is bit for bit what that
// pass makes of the bf16 activations.
constexpr int kTpOutBf16 = 0, kTpOutF32 = 1, kTpOutSwiglu = 2, kTpOutSwigluOperand = 3;
__host__ __device__ constexpr bool tp_is_swiglu(int out) { return out >= kTpOutSwiglu; }

// 16-bit slot of element j of a 16-byte chunk in pair order ((x0,x4)(x1,x5)(x2,x6)(x3,x7))
__device__ __forceinline__ int tp_pair_slot(int j) { return 2 * (j & 3) + (j >> 2); }

// The sum of a chunk's eight values as `sum8_bf16` adds them, for values that sit one per lane
// in eight consecutive lanes (x_j in lane 8 c + j): the chunk's first lane gets
// (((0 + (x0 + x1)) + (x2 + x3)) + (x4 + x5)) + (x6 + x7).
__device__ __forceinline__ float tp_chunk_sum_across_lanes(float v) {
    const float p = v + __shfl_down(v, 1, 64);  // x_j + x_(j+1): even j count
    float s = 0.0f + p;
    s += __shfl_down(p, 2, 64);
    s += __shfl_down(p, 4, 64);
    s += __shfl_down(p, 6, 64);
    return s;
}
// ... and of a row's 16 chunk sums as `row16_sum` adds them (chunk c with c + 8, those with
// the pair of c + 4, then c + 2, then c + 1), from sums[wave column wq = c / 4][c % 4]
__device__ __forceinline__ float tp_group_sum(const float (&cs)[4][4]) {
    float quad[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) quad[q] = (cs[0][q] + cs[2][q]) + (cs[1][q] + cs[3][q]);
    return (quad[0] + quad[2]) + (quad[1] + quad[3]);
}

// The lane's number, computed where it is asked for: to the compiler a new value, so that a lane constant
// that is needed once per block or behind the loop holds no register inside it.  Without it six of the
// 128 x 256 instances are short of 1 to 7 registers, and a register that goes to scratch while a read
// into it is in flight would hold what was there before (the build refuses spills in this kernel).
__device__ __forceinline__ int tp_lane_again() {
    int v;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(v));
    return v;
}

// out_pairs (kTpOutSwigluOperand): the following launch's W.  (kTpOutF32): 1 where the K parts are
// left to the consumer (a launch that has nothing but parts), 0 otherwise.
// W: pairs of groups whose scales, zeros and group sums a lane loads at once (1, 2 or 4: a
// dword, two or four per load; K a multiple of 256 W).
// ODD (W = 1): an odd number of groups.  Rows of scales are then only 2-byte aligned and come
// as halves; the last pair has one group.  The zero-point term is taken off group by group, halfway
// through a group's columns: error against 64 bits at 896 columns 5.3e-7, 9.7e-7 with a term per pair
// as below, 6.5e-7 on the kernel of qgemm_q4_tall.hip.  1030 rows x 896 (seven groups): 9728 gate/up
// rows with the activation 39.7 us, 52.6 + 11.0 on the kernel of qgemm_q4_tall.hip with the activation
// behind it; 1152 rows of q/k/v 13.5 (24.5), both on the smaller tiles of `tp_less`.
template <int OUT, int W, bool ODD, class T>
__global__ __launch_bounds__(64 * T::kWaves) void qgemm_q4g128_tallp_kernel(
    const uint16_t* __restrict__ xp, const float* __restrict__ xs, const uint8_t* __restrict__ qw,
    const __half* __restrict__ scale, const __half* __restrict__ zero,
    const float* __restrict__ bias, void* __restrict__ y_out, float* __restrict__ partials, int m,
    int n, int k, int tiles_n, int full_tiles, int split, int out_pairs) {
    extern __shared__ uint4_t tp_lds[];  // kTpBufs x {slab of x, tile of weights}
    constexpr int BL = 2 * W;            // groups per block of small loads
    constexpr int MI = T::kBlocks;
    constexpr int kSlab = T::kSlabBytes, kBuf = T::kBufBytes;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31;
    const int h = lane >> 5;
    // workgroup -> tile (columns fastest) and, for 128 x 256 tiles past the whole ones, part of a
    // tile: groups [g_begin, groups) of K, both multiples of BL
    static_assert(!ODD || W == 1, "an odd number of groups is taken pair by pair");
    int tile = blockIdx.x, part = -1;
    int g_begin = 0, groups = k >> 7;
    if (T::kBig && tile >= full_tiles) {
        const int p = tile - full_tiles;
        tile = full_tiles + p / split;
        part = p;
        const int blocks = (groups + BL - 1) / BL, q = p % split;
        g_begin = BL * (int)((int64_t)blocks * q / split);
        groups = min(groups, BL * (int)((int64_t)blocks * (q + 1) / split));
    }
    const int row_tile = tile / tiles_n;
    const int row0 = row_tile * T::kM;
    // (SwiGLU: a tile is half as many outputs wide, as many gate as up rows of the weights)
    constexpr int kTileOutputs = tp_is_swiglu(OUT) ? T::kN / 2 : T::kN;
    const int col0 = (tile % tiles_n) * kTileOutputs;
    // weight row behind row L of the tile in LDS (a wave's B operand rows are L = 32 wave + r)
    auto weight_row = [&](int L) {
        if constexpr (tp_is_swiglu(OUT)) {
            const int out_col = min(col0 + (L >> 5) * 16 + (L & 15), n - 1);
            return ((L >> 4) & 1) ? n + out_col : out_col;
        } else {
            return min(col0 + L, n - 1);  // a row past n re-reads the last row
        }
    };
    const int wc = wave * 32;  // this wave's weight rows of the tile
    const int groups_row = k >> 7;    // scales and zeros: groups per weight row
    unsigned magic;
    asm volatile("v_mov_b32 %0, 0x43004300" : "=v"(magic));
    const unsigned lds_base = (unsigned)(uintptr_t)(tp_lds_ptr_t)tp_lds;

    // ---- requests of a group, straight into LDS (a request writes 1 KiB of consecutive LDS).
    // x: request q of this wave covers rows 4 kXReq wave + 4 q .. + 3, lane -> row + lane / 16, LDS
    // position lane % 16 of that row, which holds the row's chunk (position ^ row % 16).
    // weights: request q covers rows 32 wave + 16 q .. + 15 of the tile, lane -> row + lane / 4,
    // position lane % 4 of the row's 64 bytes, which holds piece (position ^ (row / 4) % 4).
    // Byte offsets fit 32 bits (m_pad * K * 2 and N * K < 2^31 are checked on the host).
    constexpr int kXReq = T::kXRequests;
    // (Request q of x is four rows on, whose chunks are swizzled by another 4 q: rows are multiples of
    // 256 bytes apart, so its offsets are the first one's ^ 64 q from a base 4 q rows on.)
    const int xrow = 4 * kXReq * wave + (lane >> 4);
    const unsigned xoff = ((unsigned)(row0 + xrow) * (unsigned)k +
                           (unsigned)((lane & 15) ^ (xrow & 15)) * 8u) * 2u;
    unsigned woff[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int row = 32 * wave + 16 * q + (lane >> 2);
        const int piece = (lane & 3) ^ ((row >> 2) & 3);
        woff[q] = (unsigned)weight_row(row) * (unsigned)(k >> 1) + (unsigned)piece * 16u;
    }
    // request q of group g's x and weights, into the buffer at byte `buf_off` of the ring
    auto request_x = [&](auto q_c, int g, int buf_off) LG_INLINE {
        constexpr int Q = decltype(q_c)::value;
        // (scalar registers for sure: a value the compiler takes for lane-dependent would be
        // handed to the statement in vector registers)
        request_lds16(reinterpret_cast<const char*>(xp) + ((size_t)g * 256 + (size_t)Q * 8 * (unsigned)k),
                xoff ^ (64u * Q),
                __builtin_amdgcn_readfirstlane(lds_base + (unsigned)buf_off +
                                               (unsigned)(wave * kXReq + Q) * 1024u));
    };
    auto request_w = [&](auto q_c, int g, int buf_off) LG_INLINE {
        constexpr int Q = decltype(q_c)::value;
        request_lds16(reinterpret_cast<const char*>(qw) + (size_t)g * 64, woff[Q],
                __builtin_amdgcn_readfirstlane(lds_base + (unsigned)buf_off + kSlab +
                                               (unsigned)(wave * 2 + Q) * 1024u));
    };
    auto request_group = [&](int g, int buf_off) LG_INLINE {
        static_for<kXReq>([&](auto q) LG_INLINE { request_x(q, g, buf_off); });
        static_for<2>([&](auto q) LG_INLINE { request_w(q, g, buf_off); });
    };
    // ---- A operand reads: lane (r, h) at step s8 wants chunk 8 h + s8 of row 32 i + r,
    // stored at position (8 h + s8) ^ (r % 16): a0 ^ (s8 << 4), the i-tile as an immediate
    // (a buffer's offset in the ring is a multiple of 8 KiB: adding it commutes with the XOR)
    const unsigned a0 = lds_base + (unsigned)r * 256u +
                        (unsigned)(((8 * h) ^ (r & 8)) | (r & 7)) * 16u;
    // ---- B operand reads: lane (r, h) wants the pieces 2 h, 2 h + 1 of row wc + r (dword s8 % 4 of
    // piece 2 h + s8 / 4 feeds step s8)
    // (piece 2 h + 1 sits at the address ^ 16)
    const unsigned b_addr = lds_base + kSlab + (unsigned)(wc + r) * 64u +
                            (unsigned)((2 * h) ^ ((r >> 2) & 3)) * 16u;

    // ---- The small loads of a block of W pairs of groups, from global memory into registers:
    // scales and zeros of this lane's weight row (a lane's results all belong to one weight row;
    // pair p in dword p: group 2 p in the low half), and the group sums of x
    // for the zero-point product (lane (r, h) holds row 32 i + r, group 2 p + h of pair
    // p; the first pass wrote them as [row tile][block][h][row][p], so a wave reads 512
    // consecutive bytes x W).  Per block and wave one load of scales and one of zeros (ODD: a
    // second one of scales, of the second group) and MI of group sums, written as assembly
    // with the wait for them spelled out below, once per block: for loads it can see the
    // compiler waits with vmcnt(0) wherever a value is used, in every group, which also waits
    // for every request of the groups ahead and takes the ring's depth away.  A register
    // loaded here must not be touched before `small_loads_landed` has named it.
    // (The group sums of four pairs come as two loads of two, the second behind the first half of the
    // block: 8 registers less.)
    constexpr int WX = W == 4 ? 2 : W;
    struct Small {
        TpRegs<unsigned, W> s, z;
        TpRegs<float, WX> xs[MI];
        unsigned s_hi;  // ODD, on its way: the scale of the pair's second group (then the high half
                        // of s); z is the zero of this lane's group of the pair
    };
    // (kept where registers are left: with small loads for every pair of groups it is 1-2 % of 4000 x
    // 1536 x 8960 to compute their offsets anew)
    constexpr bool kLaneAgain = T::kBig && (ODD || (W > 1 && OUT != kTpOutSwigluOperand));
    auto lane_for_loads = [&]() LG_INLINE { return kLaneAgain ? tp_lane_again() : lane; };
    // the sums of the WX pairs from group g on
    auto gload_sums = [&](int g, Small& v) LG_INLINE {
        const float* xb = xs + ((size_t)(row0 / kTallTileRows) * ((groups_row + BL - 1) / BL) + g / BL) *
                                   (2 * kTallTileRows * W) + (g % BL) / 2;
        const int ln = lane_for_loads();
        const unsigned xsoff =
            (unsigned)(((ln >> 5) * kTallTileRows + (row0 % kTallTileRows) + (ln & 31)) * W) * 4u;
        // (the row tiles 32 W floats apart, as immediates)
        static_for<MI>([&](auto i_c) LG_INLINE {
            constexpr int at = decltype(i_c)::value * 32 * W * 4;
            typename TpRegs<float, WX>::raw_t& dst = v.xs[decltype(i_c)::value].raw;
            const unsigned off = xsoff;
            const float* const base = xb;
            if constexpr (WX == 1)
                asm volatile("global_load_dword %0, %1, %2 offset:%c3" : "=&v"(dst) : "v"(off), "s"(base), "n"(at) : "memory");
            else
                asm volatile("global_load_dwordx2 %0, %1, %2 offset:%c3" : "=&v"(dst) : "v"(off), "s"(base), "n"(at) : "memory");
        });
    };
    auto gload_small = [&](int g, Small& v) LG_INLINE {
        const __half* sb = scale + g;
        const __half* zb = zero + g;
        const int ln = lane_for_loads();
        const unsigned soff = (unsigned)weight_row(wc + (ln & 31)) * (unsigned)groups_row * 2u;
        if constexpr (ODD) {
            // (a missing second group re-reads the first)
            const unsigned second = soff + (g + 1 < groups_row ? 2u : 0u);
            const unsigned own = ln & 32 ? second : soff;
            asm volatile("global_load_ushort %0, %1, %2" : "=&v"(v.s.raw) : "v"(soff), "s"(sb) : "memory");
            asm volatile("global_load_ushort %0, %1, %2" : "=&v"(v.s_hi) : "v"(second), "s"(sb) : "memory");
            asm volatile("global_load_ushort %0, %1, %2" : "=&v"(v.z.raw) : "v"(own), "s"(zb) : "memory");
        } else if constexpr (W == 1) {
            asm volatile("global_load_dword %0, %1, %2" : "=&v"(v.s.raw) : "v"(soff), "s"(sb) : "memory");
            asm volatile("global_load_dword %0, %1, %2" : "=&v"(v.z.raw) : "v"(soff), "s"(zb) : "memory");
        } else if constexpr (W == 2) {
            asm volatile("global_load_dwordx2 %0, %1, %2" : "=&v"(v.s.raw) : "v"(soff), "s"(sb) : "memory");
            asm volatile("global_load_dwordx2 %0, %1, %2" : "=&v"(v.z.raw) : "v"(soff), "s"(zb) : "memory");
        } else {
            asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(v.s.raw) : "v"(soff), "s"(sb) : "memory");
            asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(v.z.raw) : "v"(soff), "s"(zb) : "memory");
        }
        gload_sums(g, v);
    };
    // Waits for everything this wave has outstanding and hands the registers over.  (Not
    // "at most the requests issued behind them": whether loads into registers and requests
    // into LDS complete in order with each other is not relied on.)
    auto small_loads_landed = [&](Small& v) LG_INLINE {
        asm volatile("s_waitcnt vmcnt(0)"
                     : "+v"(v.s.raw), "+v"(v.z.raw), "+v"(v.xs[0].raw), "+v"(v.xs[1].raw)
                     :
                     : "memory");
        if constexpr (MI == 4) asm volatile("" : "+v"(v.xs[MI - 2].raw), "+v"(v.xs[MI - 1].raw)::"memory");
        if constexpr (ODD) {
            asm volatile("" : "+v"(v.s_hi)::"memory");
            v.s.raw |= v.s_hi << 16;
        }
    };
    // The next block's values are loaded over a block's behind their last use; they are waited for
    // in the middle of the next group, and first used behind that.
    Small cur;

    float16_t yacc[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) yacc[i][e] = 0.0f;
    // (kCuts) A smaller tile takes all of K, and adds up what it has at the places where the 128 x 256
    // tile it lies in would be split over K (`split` parts): a product's bits do not depend on the tile
    // a launch takes (in front of a 3-bit K/V row a last bit flips whole codes).
    float16_t parts_sum[MI];  // the parts before this one
    const int part_blocks = (groups + BL - 1) / BL;
    int cut = 0, next_cut = 0;   // next_cut: the first group behind this part
    auto next_part = [&]() LG_INLINE {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                parts_sum[i][e] += yacc[i][e];
                yacc[i][e] = 0.0f;
            }
        ++cut;
        next_cut = BL * (part_blocks * (cut + 1) / split);
    };
    if constexpr (T::kCuts) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) parts_sum[i][e] = 0.0f;
        next_cut = BL * (part_blocks / split);
    }

    // The buffer `ahead` groups on in the ring.
    auto ring = [&](int off, int ahead) LG_INLINE {
        off += ahead * kBuf;
        return off >= kTpBufs * kBuf ? off - kTpBufs * kBuf : off;
    };
    gload_small(g_begin, cur);
    request_group(g_begin, 0);
    if (g_begin + 1 < groups) request_group(g_begin + 1, kBuf);
    small_loads_landed(cur);
    __builtin_amdgcn_s_barrier();

    // zero-point term of a pair of groups (lanes h = 0 the first, h = 1 the second):
    // y[m][n] += sum_x[m][g'] * (-scale[n][g'] * (128 + zero[n][g']))
    auto zero_term = [&](auto pair_c) LG_INLINE {
        constexpr int P = decltype(pair_c)::value;
        const unsigned sd = cur.s[P], zd = cur.z[P];
        const unsigned short sb = (unsigned short)(h ? (sd >> 16) : sd);
        const unsigned short zb = (unsigned short)(h ? (zd >> 16) : zd);
        const float cv = -__half2float(__builtin_bit_cast(__half, sb)) *
                         (128.0f + __half2float(__builtin_bit_cast(__half, zb)));
#pragma unroll
        for (int i = 0; i < MI; ++i)
            yacc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur.xs[i][P % WX], cv, yacc[i], 0, 0, 0);
    };
    // ODD: the same term of one group, -sum_x[m][g] * (128 + zero[n][g]) (the lanes of the pair's other
    // group give 0), added to the group's sum halfway through its columns: the sum then runs from 0 to
    // half of the large term, to minus half of it and back, is small when it is scaled, and the large
    // term is never rounded at its full size nor into y.
    auto zero_halfway = [&](int par, float16_t(&acc)[MI]) LG_INLINE {
        const bool own = h == par;
        const unsigned short zb = (unsigned short)cur.z[0];
        const float off = own ? -(128.0f + __half2float(__builtin_bit_cast(__half, zb))) : 0.0f;
#pragma unroll
        for (int i = 0; i < MI; ++i)
            acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(own ? cur.xs[i][0] : 0.0f, off, acc[i], 0, 0, 0);
    };

    float16_t acc[MI];
    bf16x8_t av[2][MI];  // [step parity][i]
    bf16x8_t bv[2];      // [step parity]
    uint4_t wq[2];       // [half of the group]: the group's nibbles of this lane's row
    // the x operands of a step, at byte address `a` of row r
    auto read_x = [&](bf16x8_t(&v)[MI], unsigned a) LG_INLINE {
        if constexpr (MI == 4)
            asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:8192\n\t"
                         "ds_read_b128 %2, %4 offset:16384\n\tds_read_b128 %3, %4 offset:24576"
                         : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[MI - 2]), "=&v"(v[MI - 1])
                         : "v"(a)
                         : "memory");
        else
            asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:8192"
                         : "=&v"(v[0]), "=&v"(v[1])
                         : "v"(a)
                         : "memory");
    };
    auto x_landed = [&](bf16x8_t(&v)[MI]) LG_INLINE {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0]), "+v"(v[1])::"memory");
        if constexpr (MI == 4) asm volatile("" : "+v"(v[MI - 2]), "+v"(v[MI - 1])::"memory");
    };
    // a group's nibbles and its first x operands, from the buffer at byte `buf_off` of the ring (the
    // offset is added here: LDS offsets of up to 144 KiB do not fit the 16-bit immediate of a read)
    auto read_first = [&](int buf_off) LG_INLINE {
        unsigned t0, t1;
        asm volatile("v_add_u32 %2, %5, %4\n\tv_xor_b32 %3, 16, %2\n\t"
                     "ds_read_b128 %0, %2\n\tds_read_b128 %1, %3"
                     : "=&v"(wq[0]), "=&v"(wq[1]), "=&v"(t0), "=&v"(t1)
                     : "v"(b_addr), "s"(buf_off)
                     : "memory");
        read_x(av[0], a0 + (unsigned)buf_off);
    };
    auto first_landed = [&]() LG_INLINE {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(wq[0]), "+v"(wq[1])::"memory");
        x_landed(av[0]);
    };
    // the x operands of step S (1 .. 7) of the group at a_buf
    auto read_step = [&](auto s_c, unsigned a_buf) LG_INLINE {
        constexpr int S = decltype(s_c)::value;
        read_x(av[S & 1], a_buf ^ (unsigned)(S << 4));
    };
    auto step_landed = [&](auto s_c) LG_INLINE { x_landed(av[decltype(s_c)::value & 1]); };
    auto unpack = [&](auto s_c) LG_INLINE {
        constexpr int S = decltype(s_c)::value;
        const unsigned wd = wq[S >> 2][S & 3];
        uint4_t e4;
#pragma unroll
        for (int sft = 0; sft < 4; ++sft) e4[sft] = ((wd >> (4 * sft)) & kNibMask) | magic;
        bv[S & 1] = __builtin_bit_cast(bf16x8_t, e4);
    };
    // the MFMA of step 0 of one tile of the wave
    auto first_product = [&](int i) LG_INLINE {
        float16_t z16;
#pragma unroll
        for (int e = 0; e < 16; ++e) z16[e] = 0.0f;
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[0][i], bv[0], z16, 0, 0, 0);
    };

    // One group of 128 columns out of the buffer at byte `buf_off` of the ring; U: the group's
    // place in its block.  Its step 0 has been issued by the group before it, so that nothing is
    // waited for between two groups:
    // * the wait for the next group's requests and the workgroup's barrier stand in the middle of a
    //   group, the reads of the next group's nibbles and first x operands in its step 7;
    // * the tile by tile `y += scale * acc` is followed by that tile's first MFMA of the next group.
    // LEFT: at least so many groups follow this one; LAST: exactly so many.  par: U % 2, but for the
    // last group of an odd number of groups, which may be either of its pair.
    auto group = [&](auto u_c, auto left_c, auto last_c, int g, int buf_off, int par) LG_INLINE {
        constexpr int U = decltype(u_c)::value;
        constexpr int LEFT = decltype(left_c)::value;
        constexpr bool LAST = decltype(last_c)::value;
        constexpr bool more = LEFT > 0;
        auto follows = [&](int d) LG_INLINE { return LEFT >= d || (!LAST && g + d < groups); };
        const unsigned a_buf = a0 + (unsigned)buf_off;
        // Step s8 issues the reads of step s8 + 1, then its four MFMAs with the unpack of step
        // s8 + 1 between them (the matrix pipe takes 32 cycles per MFMA, eight issue slots of
        // the vector pipe), and only then waits for the reads.  The order is pinned: left
        // alone the scheduler sinks the MFMAs below the wait, which then sits right behind the
        // reads it waits for.
        static_for<7>([&](auto sc) LG_INLINE {
            constexpr int s8 = decltype(sc)::value + 1;
            if constexpr (s8 == 4) {
                // The requests of the next group's x and weights (issued one and two groups ago)
                // have landed; those of the weights behind it, the youngest two, may be on their
                // way.  (Requests complete in the order they were issued.  Behind a block's
                // small loads everything is waited for: whether loads into registers complete in
                // order with the requests is not relied on.)
                if (U == 0 || (W == 4 && U == 4)) small_loads_landed(cur);
                else if (!follows(2)) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                else asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
                // Behind the barrier everybody's have; everybody has left the group before this
                // one, whose x slab the group after next takes, and has read this group's nibbles.
                if constexpr (more) {
                    __builtin_amdgcn_s_barrier();
                }
            }
            // One request per step: issued together they keep every wave from its next operands until
            // the texture addresser has taken all of them.
            if (follows(2)) {
                if constexpr (s8 >= 4 && s8 - 4 < kXReq)
                    request_x(ic<(s8 >= 4 && s8 - 4 < kXReq ? s8 - 4 : 0)>{}, g + 2, ring(buf_off, 2));
                constexpr int kFirstW = U == 0 || (W == 4 && U == 4) ? 5 : 1;
                if constexpr (s8 == kFirstW || s8 == kFirstW + 1)
                    request_w(ic<(s8 == kFirstW ? 0 : 1)>{}, g + 2, ring(buf_off, 2));
            }
            if constexpr (s8 < 7) read_step(ic<(s8 < 7 ? s8 + 1 : 7)>{}, a_buf);
            else if constexpr (more) read_first(ring(buf_off, 1));
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (ODD && s8 == 4) {
                zero_halfway(par, acc);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (s8 < 7) unpack(ic<(s8 < 7 ? s8 + 1 : 7)>{});
#pragma unroll
            for (int i = 0; i < MI; ++i)
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[s8 & 1][i], bv[s8 & 1], acc[i], 0,
                                                                 0, 0);
#pragma unroll
            for (int q = 0; q < MI; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);       // one MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, 8 / MI, 0);  // vector instructions
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (s8 < 7) step_landed(ic<(s8 < 7 ? s8 + 1 : 7)>{});
        });
        if constexpr (more) {
            first_landed();
            unpack(ic<0>{});
            read_step(ic<1>{}, a0 + (unsigned)ring(buf_off, 1));
        }
        __builtin_amdgcn_sched_barrier(0);
        const unsigned sd = cur.s[U >> 1];
        const unsigned short sb = (unsigned short)(par ? (sd >> 16) : sd);
        const float sf = __half2float(__builtin_bit_cast(__half, sb));
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int e = 0; e < 16; ++e) yacc[i][e] = fmaf(sf, acc[i][e], yacc[i][e]);
            if constexpr (more) first_product(i);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (more) {
            unpack(ic<1>{});
            step_landed(ic<1>{});
        }
        if constexpr (U % 2 == 1 && !ODD) zero_term(ic<(U >> 1)>{});
        if constexpr (U == BL - 1 && more) gload_small(g + 1, cur);
        if constexpr (W == 4 && U == 3) gload_sums(g + 1, cur);
    };
    // the first group's step 0
    read_first(0);
    first_landed();
    unpack(ic<0>{});
    read_step(ic<1>{}, a0);
#pragma unroll
    for (int i = 0; i < MI; ++i) first_product(i);
    unpack(ic<1>{});
    step_landed(ic<1>{});
    // ranges are whole blocks (K is a multiple of 256 W); buffers go round in threes
    int buf_off = 0;
    auto one_group = [&](auto u_c, auto left_c, auto last_c, int g) LG_INLINE {
        group(u_c, left_c, last_c, g, buf_off, decltype(u_c)::value & 1);
        buf_off = ring(buf_off, 1);
    };
    // whole blocks with more behind them, then the last one (an odd number of groups: of one or two)
    int g0 = g_begin;
    for (; g0 + BL < groups; g0 += BL) {
        if constexpr (T::kCuts)
            if (g0 == next_cut) next_part();
        static_for<BL>([&](auto uc) LG_INLINE {
            constexpr int U = decltype(uc)::value;
            one_group(uc, ic<BL - 1 - U + (ODD ? 1 : BL)>{}, ic<0>{}, g0 + U);
        });
    }
    if constexpr (T::kCuts)
        if (g0 == next_cut) next_part();
    if constexpr (ODD) {
        const int par = groups - 1 - g0;
        if (par != 0) one_group(ic<0>{}, ic<1>{}, ic<1>{}, g0);
        group(ic<0>{}, ic<0>{}, ic<1>{}, groups - 1, buf_off, par);
    } else {
        static_for<BL>([&](auto uc) LG_INLINE {
            constexpr int U = decltype(uc)::value;
            one_group(uc, ic<BL - 1 - U>{}, ic<1>{}, g0 + U);
        });
    }
    if constexpr (T::kCuts) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) yacc[i][e] = parts_sum[i][e] + yacc[i][e];
    }

    const int lane_e = tp_lane_again(), r_e = lane_e & 31, h_e = lane_e >> 5, tid_e = 64 * wave + lane_e;
    if (OUT == kTpOutF32 && T::kBig && part >= 0 && out_pairs != 0) {
        // a part of a launch whose consumer adds up the parts: rows of an [m][n] matrix each
        float* dst = partials + (size_t)(part % split) * ((size_t)m * n);
        const int gn = col0 + wc + r_e;
        if (gn >= n) return;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int gr = row0 + 32 * i + 8 * (e >> 2) + 4 * h_e + (e & 3);
                if (gr < m) dst[(int64_t)gr * n + gn] = yacc[i][e];
            }
        return;
    }
    if (T::kBig && part >= 0) {
        // a part of a tile: the wave's 128 x 32 results as they lie in registers, lane fastest
        float* dst = partials + (size_t)part * kTpTileElems + (size_t)wave * 4096 + lane_e;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) dst[(i * 16 + e) * 64] = yacc[i][e];
        return;
    }
    if constexpr (tp_is_swiglu(OUT)) {
        // Lanes r < 16 hold the gate, r >= 16 the up products of outputs 16 wave + r % 16.  Result e of
        // the upper lanes and result e + 8 of the lower ones change places, and every lane has both
        // products of eight rows per block: e of the lower, e + 8 of the upper lanes.
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const auto sw = __builtin_amdgcn_permlane16_swap(
                    __float_as_uint(yacc[i][e]), __float_as_uint(yacc[i][e + 8]), false, false);
                yacc[i][e] = __uint_as_float(sw[0]);      // gate
                yacc[i][e + 8] = __uint_as_float(sw[1]);  // up
            }
        // the row of result e (0 .. 7) of block i
        auto row_of = [&](int i, int e) { return 32 * i + 8 * (e >> 2) + (r_e & 16) + 4 * h_e + (e & 3); };
        auto activation = [&](int i, int e) {
            const float g = yacc[i][e], u = yacc[i][e + 8];
            return f32_to_bf16_rne(g / (1.0f + expf(-g)) * u);
        };
        if constexpr (OUT == kTpOutSwigluOperand) {
            // (n is a multiple of 128 here: every column of the tile is a result)
            uint16_t* const xo = static_cast<uint16_t*>(y_out);
            float* const so = reinterpret_cast<float*>(static_cast<char*>(y_out) + tall_sums_offset(m, n));
            // The bf16 tile goes through LDS, rows 16 bytes apart from a multiple of their 256, and
            // comes back as the first pass of a product takes it: a thread a chunk of eight, the 16
            // lanes of a row of lanes a row's group.
            __syncthreads();  // the ring is done with once every wave has read its last operands
            constexpr int kPitch = 128 + 8;
            uint16_t* const tile_b = reinterpret_cast<uint16_t*>(tp_lds);
            static_assert(T::kWaves == 8, "a tile's outputs are one group of the next K");
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    tile_b[row_of(i, e) * kPitch + 16 * wave + (r_e & 15)] = activation(i, e);
            __syncthreads();
#pragma unroll
            for (int u = 0; u < T::kM / 32; ++u) {
                const int row = 32 * u + (tid_e >> 4), c = tid_e & 15;
                const uint4_t v = *reinterpret_cast<const uint4_t*>(tile_b + row * kPitch + 8 * c);
                const float gs = row16_sum(sum8_bf16(v));
                *reinterpret_cast<uint4_t*>(xo + (int64_t)(row0 + row) * n + col0 + 8 * c) = pair_order(v);
                if (c == 0) so[tall_sum_index(row0 + row, col0 >> 7, n, out_pairs)] = gs;
            }
        } else {
            const int gn = col0 + (wc >> 1) + (r_e & 15);
            if (gn >= n) return;
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int gr = row0 + row_of(i, e);
                    if (gr < m) static_cast<uint16_t*>(y_out)[(int64_t)gr * n + gn] = activation(i, e);
                }
        }
        return;
    }
    const int gn = col0 + wc + r_e;
    if (gn >= n) return;
    float bv_n = bias ? bias[gn] : 0.0f;
    // (waited for here: left to the compiler the wait stands in front of every store, and behind the
    // stores before it: 281 us instead of 263 for 4096 x 4096 at 8240 rows)
    asm volatile("" : "+v"(bv_n));
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int gr = row0 + 32 * i + 8 * (e >> 2) + 4 * h_e + (e & 3);
            if (gr < m) {
                if constexpr (OUT == kTpOutF32)
                    static_cast<float*>(y_out)[(int64_t)gr * n + gn] = yacc[i][e] + bv_n;
                else
                    static_cast<uint16_t*>(y_out)[(int64_t)gr * n + gn] = f32_to_bf16_rne(yacc[i][e] + bv_n);
            }
        }
}

// Sums the `split` fp32 parts of each tile of the last round, in part order, adds the bias and
// writes y.  One thread per result; a part's element index is (wave, i, e, lane) as the
// product kernel left it.  (SwiGLU: lane % 32 < 16 is the gate and the lane 16 on the up product of the
// same result; one thread takes both.)
template <int OUT>
__global__ __launch_bounds__(256) void q4_tall_reduce_kernel(const float* __restrict__ partials,
                                                            const float* __restrict__ bias,
                                                            void* __restrict__ y_out, int m, int n,
                                                            int tiles_n, int full_tiles,
                                                            int split) {
    static_assert(OUT != kTpOutSwigluOperand, "q4_tall_reduce_operand_kernel");
    constexpr int kPerTile = OUT == kTpOutSwiglu ? kTpTileElems / 2 : kTpTileElems;
    // a tile's workgroups by its blocks of 32 rows first: of a tile whose rows end early the first ones
    // have work and the rest none (every other run of them, with the waves first: 280 to 320 rows of
    // 1536 x 8960 in 14 parts 9.8 us, 6.3 this way)
    constexpr int kWgs = kPerTile / 256, kSub = kWgs / 32;  // kSub: of a wave's block
    const int t = blockIdx.x / kWgs, b = blockIdx.x % kWgs;
    int idx = (((b / kSub) % 8 * 4 + b / (8 * kSub)) * kSub + b % kSub) * 256 + threadIdx.x;
    if constexpr (OUT == kTpOutSwiglu) idx = ((idx >> 4) << 5) | (idx & 15);  // the gate's lanes
    const int lane = idx & 63, e = (idx >> 6) & 15, i = (idx >> 10) & 3, wave = idx >> 12;
    const int tile = full_tiles + t;
    const int gr = (tile / tiles_n) * kTpTileM + 32 * i + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
    const float* src = partials + (size_t)t * split * kTpTileElems + idx;
    if constexpr (OUT == kTpOutSwiglu) {
        const int gn = (tile % tiles_n) * (kTpTileN / 2) + wave * 16 + (lane & 15);
        if (gr >= m || gn >= n) return;
        float g = 0.0f, u = 0.0f;
        for (int q = 0; q < split; ++q) {
            g += src[(size_t)q * kTpTileElems];
            u += src[(size_t)q * kTpTileElems + 16];
        }
        static_cast<uint16_t*>(y_out)[(int64_t)gr * n + gn] =
            f32_to_bf16_rne(g / (1.0f + expf(-g)) * u);
    } else {
        const int gn = (tile % tiles_n) * kTpTileN + wave * 32 + (lane & 31);
        if (gr >= m || gn >= n) return;
        float acc = 0.0f;
        for (int q = 0; q < split; ++q) acc += src[(size_t)q * kTpTileElems];
        if (bias) acc += bias[gn];
        if constexpr (OUT == kTpOutF32) static_cast<float*>(y_out)[(int64_t)gr * n + gn] = acc;
        else static_cast<uint16_t*>(y_out)[(int64_t)gr * n + gn] = f32_to_bf16_rne(acc);
    }
}

// The same for kTpOutSwigluOperand: a workgroup takes four rows-of-registers (e = 4 eq .. + 3)
// of one block i of a tile across all eight waves, i.e. eight rows of the tile with
// all their 128 outputs, so that it can add up their group sums: thread (wave, h, output of the wave)
// sums the parts of the gate and the up product of its result in part order, applies the
// activation and writes the bf16 value in pair order; chunk and group sums as in the product
// kernel.  grid: 16 workgroups per tile.
__global__ __launch_bounds__(256) void q4_tall_reduce_operand_kernel(
    const float* __restrict__ partials, void* __restrict__ y_out, int m, int n, int tiles_n,
    int full_tiles, int split, int out_pairs) {
    __shared__ float red[16][8];  // [chunk of the group][row of the eight]
    const int t = blockIdx.x >> 4;
    const int i = (blockIdx.x >> 2) & 3, eq = blockIdx.x & 3;
    const int wave = threadIdx.x >> 5, h = (threadIdx.x >> 4) & 1, c = threadIdx.x & 15;
    const int tile = full_tiles + t;
    const int row0 = (tile / tiles_n) * kTpTileM, col0 = (tile % tiles_n) * (kTpTileN / 2);
    const int gn = col0 + 16 * wave + c;
    uint16_t* const xo = static_cast<uint16_t*>(y_out);
    float* const so = reinterpret_cast<float*>(static_cast<char*>(y_out) + tall_sums_offset(m, n));
    const float* src = partials + (size_t)t * split * kTpTileElems + (size_t)wave * 4096 +
                       (size_t)i * 1024 + h * 32 + c;
#pragma unroll
    for (int el = 0; el < 4; ++el) {
        const int e = 4 * eq + el;
        float g = 0.0f, u = 0.0f;
        for (int q = 0; q < split; ++q) {
            g += src[(size_t)q * kTpTileElems + e * 64];
            u += src[(size_t)q * kTpTileElems + e * 64 + 16];
        }
        const int row = 32 * i + 8 * (e >> 2) + 4 * h + (e & 3);
        const uint16_t b = f32_to_bf16_rne(g / (1.0f + expf(-g)) * u);
        xo[(int64_t)(row0 + row) * n + (gn & ~7) + tp_pair_slot(gn & 7)] = b;
        const float cs = tp_chunk_sum_across_lanes(__uint_as_float((unsigned)b << 16));
        if ((c & 7) == 0) red[2 * wave + (c >> 3)][2 * el + h] = cs;
    }
    __syncthreads();
    if (threadIdx.x < 8) {
        const int el = threadIdx.x >> 1, hh = threadIdx.x & 1, e = 4 * eq + el;
        float cs[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) cs[a][b] = red[4 * a + b][threadIdx.x];
        const int row = 32 * i + 8 * (e >> 2) + 4 * hh + (e & 3);
        so[tall_sum_index(row0 + row, col0 >> 7, n, out_pairs)] = tp_group_sum(cs);
    }
}

inline int tp_pairs_per_load(int k, const void* scale, const void* zero) {
    return tall_pairs_per_load(k, scale, zero);
}

// 32-bit offsets of the kernels
static bool tp_sizes_ok(int m, int n, int k) {
    const int64_t lim = INT32_MAX;
    return (int64_t)n * k <= lim && (int64_t)tp_padded_rows(m) * k * 2 <= lim && (int64_t)m * n <= lim;
}

bool qgemm_q4_tallp_applies(int m, int n, int k) {
    return m > 0 && n > 0 && k > 0 && k % 128 == 0 && tp_sizes_ok(m, n, k);
}

// The plan of a launch's 128 x 256 tiles (which the smaller tiles add up by).
template <int OUT>
static TpPlan tp_big_plan(int m, int n, int k, int block_groups, int cus) {
    constexpr int outputs = tp_is_swiglu(OUT) ? kTpTileN / 2 : kTpTileN;
    // (an operand's padding rows are written too: whole tiles as well)
    return tp_plan(((n + outputs - 1) / outputs) * ((m + kTpTileM - 1) / kTpTileM), k >> 7, block_groups,
                   cus);
}

// Whether a launch takes the smaller tiles.  A 128 x 256 tile takes about 1.8 us a group of 128 columns
// whatever else runs, so with few groups of K and few tiles the smaller ones win by filling the chip.
// us, 128 x 256 / 64 x 128 (the first with the sum of its K parts, both at K 896 with the first pass
// over x):
//   K  896, 1152 columns:  100 rows 23.2 / 13.9, 1030 26.4 / 17.0, 2060 29.1 / 21.7, 4120 32.4 / 33.3
//   K 1536, 2048 columns:  100 rows 13.1 / 13.4,  520 20.6 / 14.4, 1030 23.6 / 17.1, 2060 28.5 / 29.7
// hence: at most 16 groups (at 32 a small tile's chain costs what the large one's parts do) and all tiles
// resident at once (two per compute unit).  Where the big tiles could be split over K, it matters who adds
// up the parts:
// * the next operator of a step, which reads its operand anyway: at least 20 big tiles (28 layers of 1536,
//   200 rows, 2048 columns of q/k/v, which are 16: 3418 us a step, 3491 on small ones);
// * a launch of its own, 4 us: always in two parts and for fp32 results, else from ten big tiles on.  1440
//   products of 16 to 1000 rows, 256 to 4608 columns, the first pass over x included:
//     K 1280, 2 parts:  128 x 256 fp32 16.2 / 12.8, 300 x 256 bf16 16.6 / 14.1;  K 2048, 2 parts:  128 x 256 bf16 19.4 / 17.5
//     K 1536, 3 parts:  128 x 256 fp32 14.3 / 14.0, bf16 14.2 / 14.9, with SwiGLU 11.5 / 12.4 (from ten tiles on:
//     128 x 2560 16.5 / 14.2, 16.4 / 15.1, 13.1 / 12.6; 200 x 2048 18.1 / 14.7, 18.0 / 15.7, 13.8 / 12.6)
// A next product's operand is written by 64 x 256 tiles, one per compute unit, whose round takes
// five eighths of a big one's (a last round that is split over K about six of them):
//   K  896, 4864 outputs:  195 rows 23.4 / 15.7,  520 25.2 / 28.2, 1030 45.8 / 40.8, 2060 69.4 / 77.4
//   K 1536, 8960 outputs:  100 rows 23.6 / 16.8,  195 25.5 / 31.9,  300 28.3 / 33.9, 2060 148 / 168
// Whole large tiles in front of split ones keep the large tiles (none of the above is lost by it), so
// that a launch on the smaller ones adds up all of its tiles alike.
// parts_out: the launch may leave its K parts to the next operator.
template <int OUT>
static bool tp_less(int m, int n, int k, int block_groups, int cus, bool parts_out) {
    const int groups = k >> 7;
    if (groups > 16) return false;
    auto tiles = [&](int rows, int tm, int tn) {
        return (int64_t)((rows + tm - 1) / tm) * ((n + tn - 1) / tn);
    };
    const TpPlan plan = tp_big_plan<OUT>(m, n, k, block_groups, cus);
    if (plan.split > 1 && plan.full > 0) return false;
    if (OUT == kTpOutSwigluOperand) {
        const int rows = tp_padded_rows(m);
        const int64_t big = plan.split > 1 ? 6 : 8 * ((plan.full + cus - 1) / cus);
        const int64_t half = (tiles(rows, TpHalf<false>::kM, TpHalf<false>::kN / 2) + cus - 1) / cus;
        return 5 * half < big;
    }
    const int div = tp_is_swiglu(OUT) ? 2 : 1;
    if (tiles(m, TpSmall<false>::kM, TpSmall<false>::kN / div) > 2 * cus) return false;
    const int64_t big = tiles(m, TpBig::kM, TpBig::kN / div);
    if (parts_out) return plan.split == 1 || big >= 20;
    return plan.split <= 2 || OUT == kTpOutF32 || big >= 10;
}

template <int OUT, int W, bool ODD, class T>
static hipError_t tallp_launch_tile(const uint16_t* xp, const float* xs, float* partials,
                               const uint8_t* qw, const __half* scale, const __half* zero,
                                    const float* bias, void* y, int m, int n, int k, hipStream_t st,
                                    int out_pairs) {
    constexpr size_t lds = (size_t)kTpBufs * T::kBufBytes;
    static const hipError_t opt = hipFuncSetAttribute(
        reinterpret_cast<const void*>(qgemm_q4g128_tallp_kernel<OUT, W, ODD, T>),
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (opt != hipSuccess) return opt;
    constexpr int tile_outputs = tp_is_swiglu(OUT) ? T::kN / 2 : T::kN;
    const int tiles_n = (n + tile_outputs - 1) / tile_outputs;
    // (an operand's padding rows are written too)
    const int rows = OUT == kTpOutSwigluOperand ? tp_padded_rows(m) : m;
    const int tiles = tiles_n * ((rows + T::kM - 1) / T::kM);
    const int cus = device_cu_count();
    if (cus <= 0) return hipErrorInvalidDevice;
    const TpPlan plan = tp_big_plan<OUT>(m, n, k, 2 * W, cus);
    const int parts = T::kBig && plan.split > 1 ? (tiles - plan.full) * plan.split : 0;
    qgemm_q4g128_tallp_kernel<OUT, W, ODD, T>
        <<<dim3(parts ? plan.full + parts : tiles), dim3(64 * T::kWaves), lds, st>>>(
            xp, xs, qw, scale, zero, bias, y, partials, m, n, k, tiles_n, plan.full, plan.split,
            out_pairs);
    if (parts && !(OUT == kTpOutF32 && out_pairs != 0)) {
        if constexpr (OUT == kTpOutSwigluOperand) {
            q4_tall_reduce_operand_kernel<<<dim3((tiles - plan.full) * 16), dim3(256), 0, st>>>(
                partials, y, m, n, tiles_n, plan.full, plan.split, out_pairs);
        } else {
            constexpr int per_tile = OUT == kTpOutSwiglu ? kTpTileElems / 2 : kTpTileElems;
            q4_tall_reduce_kernel<OUT>
                <<<dim3((tiles - plan.full) * (per_tile / 256)), dim3(256), 0, st>>>(
                    partials, bias, y, m, n, tiles_n, plan.full, plan.split);
        }
    }
    return hipGetLastError();
}

template <int OUT, int W, bool ODD = false>
static hipError_t tallp_launch(const uint16_t* xp, const float* xs, float* partials,
                               const uint8_t* qw, const __half* scale, const __half* zero,
                               const float* bias, void* y, int m, int n, int k, hipStream_t st,
                               int out_pairs = 0) {
    constexpr bool operand = OUT == kTpOutSwigluOperand;
    using Less = std::conditional_t<operand, TpHalf<false>, TpSmall<false>>;
    using LessCuts = std::conditional_t<operand, TpHalf<true>, TpSmall<true>>;
    const int cus = device_cu_count();
    if (cus <= 0) return hipErrorInvalidDevice;
    if (tp_less<OUT>(m, n, k, 2 * W, cus, OUT == kTpOutF32 && out_pairs != 0)) {
        if (tp_big_plan<OUT>(m, n, k, 2 * W, cus).split > 1)
            return tallp_launch_tile<OUT, W, ODD, LessCuts>(xp, xs, partials, qw, scale, zero, bias, y,
                                                            m, n, k, st, out_pairs);
        return tallp_launch_tile<OUT, W, ODD, Less>(xp, xs, partials, qw, scale, zero, bias, y, m, n,
                                                    k, st, out_pairs);
    }
    return tallp_launch_tile<OUT, W, ODD, TpBig>(xp, xs, partials, qw, scale, zero, bias, y, m, n, k,
                                                 st, out_pairs);
}

template <int OUT>
static hipError_t tallp_launch_w(int w, const uint16_t* xp, const float* xs, float* partials,
                                 const uint8_t* qw, const __half* scale, const __half* zero,
                                 const float* bias, void* y, int m, int n, int k, hipStream_t st,
                                 int out_pairs = 0) {
    if ((k >> 7) & 1) {
        // (bf16 products are the exported entry points', which take pairs of groups)
        if constexpr (OUT == kTpOutBf16)
            return hipErrorInvalidValue;
        else
            return tallp_launch<OUT, 1, true>(xp, xs, partials, qw, scale, zero, bias, y, m, n, k, st,
                                              out_pairs);
    }
    switch (w) {
        case 4:
            return tallp_launch<OUT, 4>(xp, xs, partials, qw, scale, zero, bias, y, m, n, k, st,
                                        out_pairs);
        case 2:
            return tallp_launch<OUT, 2>(xp, xs, partials, qw, scale, zero, bias, y, m, n, k, st,
                                        out_pairs);
        default:
            return tallp_launch<OUT, 1>(xp, xs, partials, qw, scale, zero, bias, y, m, n, k, st,
                                        out_pairs);
    }
}

}  // namespace lg

extern "C" logismos_status_t logismos_check_qgemm_q4g128_tall_shape(int m, int n, int k, char* msg,
                                                                    size_t msg_cap) {
    const char* kn = "qgemm_q4g128_tall";
    if (m <= 0) return lg::reject(msg, msg_cap, "%s: rows must be positive, got %d", kn, m);
    if (n <= 0) return lg::reject(msg, msg_cap, "%s: N must be positive, got %d", kn, n);
    if (k <= 0 || k % 256 != 0)
        return lg::reject(msg, msg_cap,
                          "%s: K = %d is not a positive multiple of 256 (pairs of groups of 128)",
                          kn, k);
    const int64_t lim = INT32_MAX;
    if ((int64_t)n * k > lim)
        return lg::reject(msg, msg_cap, "%s: N*K = %lld exceeds i32::MAX", kn,
                          (long long)((int64_t)n * k));
    if ((int64_t)lg::tp_padded_rows(m) * k * 2 > lim || (int64_t)m * n > lim)
        return lg::reject(msg, msg_cap, "%s: rows*K*2 or rows*N exceeds i32::MAX", kn);
    return 0;
}

extern "C" size_t logismos_qgemm_q4g128_tall_workspace_bytes(int m, int k) {
    if (m <= 0 || k <= 0 || k % 128 != 0) return 0;
    return lg::tp_partials_offset(m, k) + (size_t)lg::kTpMaxParts * lg::kTpTileElems * 4;
}

extern "C" int logismos_qgemm_q4g128_tall_pairs_per_load(int k, const void* scale_f16,
                                                         const void* zero_f16) {
    return lg::tall_pairs_per_load(k, scale_f16, zero_f16);
}

namespace lg {

// (an odd number of groups: the rows of scales and zeros are halves, loaded as halves)
static hipError_t tall_args_ok(const void* qw_u8, const void* scale_f16,
                                      const void* zero_f16, const void* y, const void* workspace,
                                      int m, int n, int k) {
    if (!qgemm_q4_tallp_applies(m, n, k)) return hipErrorInvalidValue;
    if (!qw_u8 || !scale_f16 || !zero_f16 || !y || !workspace) return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(qw_u8) | reinterpret_cast<uintptr_t>(workspace)) & 15u)
        return hipErrorInvalidValue;
    const uintptr_t align = k % 256 == 0 ? 3u : 1u;
    if ((reinterpret_cast<uintptr_t>(scale_f16) | reinterpret_cast<uintptr_t>(zero_f16)) & align)
        return hipErrorInvalidValue;
    return hipSuccess;
}

// How many K parts the launch leaves to a consumer that asks for them; 1: the finished product.
static int tallp_parts(const void* scale_f16, const void* zero_f16, int m, int n, int k) {
    const int cus = device_cu_count();
    if (cus <= 0) return 1;
    const int block_groups = ((k >> 7) & 1) ? 2 : 2 * tp_pairs_per_load(k, scale_f16, zero_f16);
    if (tp_less<kTpOutF32>(m, n, k, block_groups, cus, true)) return 1;
    const int tiles = ((m + kTpTileM - 1) / kTpTileM) * ((n + kTpTileN - 1) / kTpTileN);
    const TpPlan plan = tp_plan(tiles, k >> 7, block_groups, cus);
    return plan.full == 0 ? plan.split : 1;
}

hipError_t qgemm_q4_tallp_prepared_parts(const void* qw_u8, const void* scale_f16,
                                         const void* zero_f16, void* y_f32, void* workspace, int m,
                                         int n, int k, TallParts* out, hipStream_t st) {
    if (const hipError_t e = tall_args_ok(qw_u8, scale_f16, zero_f16, y_f32, workspace, m, n, k))
        return e;
    out->count = tallp_parts(scale_f16, zero_f16, m, n, k);
    out->src = out->count > 1 ? static_cast<char*>(workspace) + tp_partials_offset(m, k)
                              : static_cast<char*>(y_f32);
    const int w = tp_pairs_per_load(k, scale_f16, zero_f16);
    return tallp_launch_w<kTpOutF32>(
        w, static_cast<const uint16_t*>(workspace),
        reinterpret_cast<const float*>(static_cast<char*>(workspace) + tp_sums_offset(m, k)),
        reinterpret_cast<float*>(static_cast<char*>(workspace) + tp_partials_offset(m, k)),
        static_cast<const uint8_t*>(qw_u8), static_cast<const __half*>(scale_f16),
        static_cast<const __half*>(zero_f16), nullptr, y_f32, m, n, k, st, out->count > 1 ? 1 : 0);
}

hipError_t qgemm_q4_tallp_prepare(const void* x_bf16, const void* scale_f16, const void* zero_f16,
                                  void* workspace, int m, int k, hipStream_t st) {
    if (!x_bf16 || ((reinterpret_cast<uintptr_t>(x_bf16) | reinterpret_cast<uintptr_t>(workspace)) & 15u))
        return hipErrorInvalidValue;
    const int m_pad = tp_padded_rows(m);
    const int64_t chunks = (int64_t)m_pad * (k / 8);
    q4_tall_prepare_kernel<<<dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, st>>>(
        static_cast<const uint16_t*>(x_bf16), static_cast<uint16_t*>(workspace),
        reinterpret_cast<float*>(static_cast<char*>(workspace) + tp_sums_offset(m, k)), m, m_pad, k,
        tp_pairs_per_load(k, scale_f16, zero_f16));
    return hipGetLastError();
}

hipError_t qgemm_q4_tallp_prepared(
    const void* qw_u8, const void* scale_f16, const void* zero_f16, const void* bias_f32, void* y,
    int y_is_f32, void* workspace, int m, int n, int k, hipStream_t st) {
    if (const hipError_t e = tall_args_ok(qw_u8, scale_f16, zero_f16, y, workspace, m, n, k))
        return e;
    const uint16_t* xp = static_cast<const uint16_t*>(workspace);
    const float* xs =
        reinterpret_cast<const float*>(static_cast<char*>(workspace) + tp_sums_offset(m, k));
    float* partials = reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                               tp_partials_offset(m, k));
    const int w = tp_pairs_per_load(k, scale_f16, zero_f16);
    if (y_is_f32)
        return tallp_launch_w<kTpOutF32>(w, xp, xs, partials, static_cast<const uint8_t*>(qw_u8),
                                        static_cast<const __half*>(scale_f16),
                                        static_cast<const __half*>(zero_f16),
                                        static_cast<const float*>(bias_f32), y, m, n, k, st);
    return tallp_launch_w<kTpOutBf16>(w, xp, xs, partials, static_cast<const uint8_t*>(qw_u8),
                                     static_cast<const __half*>(scale_f16),
                                     static_cast<const __half*>(zero_f16),
                                     static_cast<const float*>(bias_f32), y, m, n, k, st);
}

hipError_t qgemm_q4_tallp_swiglu(
    const void* gate_up_qw_u8, const void* scale_f16, const void* zero_f16, void* act_bf16,
    void* workspace, int m, int inter, int k, hipStream_t st) {
    // the weights are 2 * inter rows (gate, then up); the output is m x inter
    if (inter <= 0 || inter > INT32_MAX / 2) return hipErrorInvalidValue;
    if (const hipError_t e = tall_args_ok(gate_up_qw_u8, scale_f16, zero_f16, act_bf16,
                                                 workspace, m, 2 * inter, k))
        return e;
    const uint16_t* xp = static_cast<const uint16_t*>(workspace);
    const float* xs =
        reinterpret_cast<const float*>(static_cast<char*>(workspace) + tp_sums_offset(m, k));
    float* partials = reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                               tp_partials_offset(m, k));
    const int w = tp_pairs_per_load(k, scale_f16, zero_f16);
    return tallp_launch_w<kTpOutSwiglu>(
        w, xp, xs, partials, static_cast<const uint8_t*>(gate_up_qw_u8),
        static_cast<const __half*>(scale_f16), static_cast<const __half*>(zero_f16), nullptr,
        act_bf16, m, inter, k, st);
}

hipError_t qgemm_q4_tallp_swiglu_operand(
    const void* gate_up_qw_u8, const void* scale_f16, const void* zero_f16, void* next_workspace,
    int next_pairs_per_load, void* workspace, int m, int inter, int k, hipStream_t st) {
    // the output is the operand of a product over K = inter: whole pairs of groups, and as many
    // pairs per load as the caller's next launch will ask for (whole blocks of them)
    if (inter <= 0 || inter > INT32_MAX / 2 || inter % 256 != 0) return hipErrorInvalidValue;
    if (next_pairs_per_load != 1 && next_pairs_per_load != 2 && next_pairs_per_load != 4)
        return hipErrorInvalidValue;
    if (inter % (256 * next_pairs_per_load) != 0) return hipErrorInvalidValue;
    if (const hipError_t e = tall_args_ok(gate_up_qw_u8, scale_f16, zero_f16,
                                                 next_workspace, workspace, m, 2 * inter, k))
        return e;
    // (the next launch's own shape: rows * inter * 2 within 32 bits)
    if (!qgemm_q4_tallp_applies(m, 1, inter))
        return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(next_workspace) & 15u) || next_workspace == workspace)
        return hipErrorInvalidValue;
    const uint16_t* xp = static_cast<const uint16_t*>(workspace);
    const float* xs =
        reinterpret_cast<const float*>(static_cast<char*>(workspace) + tp_sums_offset(m, k));
    float* partials = reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                               tp_partials_offset(m, k));
    const int w = tp_pairs_per_load(k, scale_f16, zero_f16);
    return tallp_launch_w<kTpOutSwigluOperand>(
        w, xp, xs, partials, static_cast<const uint8_t*>(gate_up_qw_u8),
        static_cast<const __half*>(scale_f16), static_cast<const __half*>(zero_f16), nullptr,
        next_workspace, m, inter, k, st, next_pairs_per_load);
}

hipError_t qgemm_q4_tallp(
    const void* x_bf16, const void* qw_u8, const void* scale_f16, const void* zero_f16,
    const void* bias_f32, void* y, int y_is_f32, void* workspace, int m, int n, int k,
    hipStream_t st) {
    if (const hipError_t e = tall_args_ok(qw_u8, scale_f16, zero_f16, y, workspace, m, n, k))
        return e;
    if (!x_bf16 || (reinterpret_cast<uintptr_t>(x_bf16) & 15u)) return hipErrorInvalidValue;
    if (const hipError_t e = qgemm_q4_tallp_prepare(x_bf16, scale_f16, zero_f16, workspace, m, k, st))
        return e;
    return qgemm_q4_tallp_prepared(qw_u8, scale_f16, zero_f16, bias_f32, y,
                                                      y_is_f32, workspace, m, n, k, st);
}

}  // namespace lg

// The exported entry points take whole pairs of groups.
extern "C" logismos_status_t logismos_launch_qgemm_q4g128_tall_prepared(
    const void* qw_u8, const void* scale_f16, const void* zero_f16, const void* bias_f32, void* y,
    int y_is_f32, void* workspace, int m, int n, int k, logismos_stream_t stream) {
    if (k % 256 != 0) return hipErrorInvalidValue;
    return lg::qgemm_q4_tallp_prepared(qw_u8, scale_f16, zero_f16, bias_f32, y, y_is_f32, workspace,
                                       m, n, k, static_cast<hipStream_t>(stream));
}

extern "C" logismos_status_t logismos_launch_qgemm_q4g128_tall_swiglu_prepared(
    const void* gate_up_qw_u8, const void* scale_f16, const void* zero_f16, void* act_bf16,
    void* workspace, int m, int inter, int k, logismos_stream_t stream) {
    if (k % 256 != 0) return hipErrorInvalidValue;
    return lg::qgemm_q4_tallp_swiglu(gate_up_qw_u8, scale_f16, zero_f16, act_bf16, workspace, m,
                                     inter, k, static_cast<hipStream_t>(stream));
}

extern "C" logismos_status_t logismos_launch_qgemm_q4g128_tall_swiglu_operand(
    const void* gate_up_qw_u8, const void* scale_f16, const void* zero_f16, void* next_workspace,
    int next_pairs_per_load, void* workspace, int m, int inter, int k, logismos_stream_t stream) {
    if (k % 256 != 0) return hipErrorInvalidValue;
    return lg::qgemm_q4_tallp_swiglu_operand(gate_up_qw_u8, scale_f16, zero_f16, next_workspace,
                                             next_pairs_per_load, workspace, m, inter, k,
                                             static_cast<hipStream_t>(stream));
}

extern "C" logismos_status_t logismos_launch_qgemm_q4g128_tall(
    const void* x_bf16, const void* qw_u8, const void* scale_f16, const void* zero_f16,
    const void* bias_f32, void* y, int y_is_f32, void* workspace, int m, int n, int k,
    logismos_stream_t stream) {
    if (k % 256 != 0) return hipErrorInvalidValue;
    return lg::qgemm_q4_tallp(x_bf16, qw_u8, scale_f16, zero_f16, bias_f32, y, y_is_f32, workspace, m,
                              n, k, static_cast<hipStream_t>(stream));
}
