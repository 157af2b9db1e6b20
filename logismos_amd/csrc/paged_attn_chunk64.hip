// Rows of sequences with several new tokens (prompt chunks) at 64-wide heads, fp16 pools: the general
// kernel of paged_attn_anydim.hip gives 16 / G tokens one pass over all their keys, so the chunk of a
// group of seven heads reads its keys 256 times; here 32 columns -- (token, head) pairs of one KV
// head, in that order over the whole chunk -- take a wave, and CW waves share the keys in LDS.
//
// * A tile is 64 keys: 8 KiB of K and of V, straight from the pools into LDS (global_load_lds, 16
//   bytes per lane, eight keys per request; block_size is a multiple of 16, so a request lies in one
//   block), a ring of four tiles (two where every wave has its own), requested three (one) ahead.  The
//   16-byte chunks of a row are swizzled by its index so that the operand reads below touch every
//   bank once.
// * Scores transposed: S^T = K . Q^T on v_mfma_f32_32x32x16_f16 (A = K from LDS, B = the queries, in
//   registers for the whole launch).  A lane then holds 16 keys of ONE column: maximum, sum and
//   rescaling are per-lane values (the lane 32 on holds the column's other 16 keys).
// * O^T = V^T . P^T: a lane's probabilities are the B operand as they lie, which fixes the order of the
//   keys inside an MFMA: k = (h, i) is key 4 h + i for i < 4 and 8 + 4 h + i - 4 behind it, and two
//   transposing LDS reads (ds_read_b64_tr_b16: four keys of one column each) fetch V in that order.
//   Probabilities go in as two fp16 terms, as in the general kernel.
// * KP key phases: the workgroup's four waves are CW column groups by KP phases, phase f taking
//   the tiles f, f + KP, ... out of a ring of its own; their (m, l, O) states meet in LDS at the
//   end.  Many columns: CW = 4.  Few: every wave a phase (a workgroup's walk over the keys is
//   what sets the time then).
//
// What bounds it: a step of 64 keys is a chain of reads, products, exponentials and products of about
// 0.7 us for a wave alone on its SIMD, 300 vector instructions of it the softmax.  24 layers of 14 query
// and 2 KV heads: 1030 rows, two chunks of 512 in contexts of up to 1500, 34 -> 20.8 us a layer.
//
// Semantics as in the general kernel: column (token i, head) sees the first ctx - n_new + i + 1 keys
// (all ctx where not causal); a column that sees none is a row of zeros.
#include "device_utils.hpp"
#include "launch_common.hpp"
#include "paged_attn_params.hpp"
#include "q4_common.hpp"

namespace lg {

typedef __attribute__((address_space(3))) void* c64_lds_ptr_t;

// Lengths and block ids are the same for a whole wave and are not written while the kernel runs: read
// through the constant address space they come as scalar loads.  (As vector loads, which is what the
// compiler makes of them beside assembly that touches memory, each waited for every request in flight:
// two chunks of 512 29 us instead of 22.)
typedef const __attribute__((address_space(4))) int32_t* c64_scalar_ptr_t;
__device__ __forceinline__ c64_scalar_ptr_t c64_scalar(const int32_t* p) {
    return (c64_scalar_ptr_t)(uintptr_t)p;
}

constexpr int kC64Keys = 64;                 // keys per tile
constexpr int kC64Tile = kC64Keys * 64 * 2;  // bytes of a tile of K (or V)
constexpr int c64_bufs(int kp) { return kp == 4 ? 2 : 4; }

template <int CW, int KP>
__global__ __launch_bounds__(256, KP == 1 ? 2 : 1) void paged_attn_chunk64_kernel(const AttnParams p, int G, int block_shift) {
    static_assert(CW * KP == 4, "four waves");
    constexpr int kBuf = 2 * kC64Tile;       // K, then V
    constexpr int kReq = kC64Keys / 8 / CW;  // requests of K (and of V) per wave and tile
    constexpr int kBufs = c64_bufs(KP), kRing = kBufs * kBuf;
    extern __shared__ uint4_t c64_lds[];     // KP rings
    __shared__ unsigned odd_waves[4];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cw = wave % CW, phase = wave / CW;
    const int col = lane & 31, h = lane >> 5;
    const int s = blockIdx.z, kvh = blockIdx.y;
    const c64_scalar_ptr_t cu = c64_scalar(p.cu_seqlens_q);
    const int row0 = cu[s];
    const int n_new = cu[s + 1] - row0;
    if (n_new <= 1) return;
    const int cols = n_new * G;
    // (the last columns see the most keys: they start first)
    const int groups = (cols + 32 * CW - 1) / (32 * CW);
    const int group = groups - 1 - (int)blockIdx.x;
    if (group < 0) return;
    const int ctx = c64_scalar(p.context_lens)[s];
    const int c0 = (group * CW + cw) * 32;   // this wave's first column
    const int gc = c0 + col;
    const bool live = gc < cols;
    const int tok = (live ? gc : cols - 1) / G, head = (live ? gc : cols - 1) - tok * G;
    const int vis = p.causal ? ctx - n_new + tok + 1 : ctx;  // keys of this lane's column
    const int last_tok = min(n_new - 1, ((group + 1) * 32 * CW - 1) / G);
    const int visible = p.causal ? ctx - n_new + last_tok + 1 : ctx;  // of the workgroup's last
    const int first_vis = p.causal ? ctx - n_new + min(c0, cols - 1) / G + 1 : ctx;  // of the wave's first
    const int last_vis = p.causal ? ctx - n_new + min(c0 + 31, cols - 1) / G + 1 : ctx;  // ... and last

    // the queries as the B operand: column col, elements 16 st + 8 h .. + 7
    half8_t qb[4];
    {
        const _Float16* q = p.q + ((int64_t)(row0 + tok) * p.hq + (int64_t)kvh * G + head) * 64 + 8 * h;
#pragma unroll
        for (int st = 0; st < 4; ++st) qb[st] = *reinterpret_cast<const half8_t*>(q + 16 * st);
    }
    // waited for here: left to the compiler the wait sits at the first use inside the loop, and
    // empties the ring in every step
#pragma unroll
    for (int st = 0; st < 4; ++st) asm volatile("" : "+v"(qb[st]));

    const unsigned ring = (unsigned)(uintptr_t)(c64_lds_ptr_t)c64_lds + (unsigned)phase * kRing;
    const int tiles = visible > 0 ? (visible + kC64Keys - 1) / kC64Keys : 0;
    // (every wave of the workgroup goes through the same number of steps)
    const int steps = (tiles + KP - 1) / KP;
    const c64_scalar_ptr_t table = c64_scalar(p.block_tables + (int64_t)s * p.max_blocks_per_seq);
    const unsigned row_bytes = (unsigned)p.hkv * 128u;
    const char* const kp = reinterpret_cast<const char*>(p.k_pool) + (int64_t)kvh * 128;
    const char* const vp = reinterpret_cast<const char*>(p.v_pool) + (int64_t)kvh * 128;
    // request q of a tile: keys 8 (kReq cw + q) .. + 7, lane -> key lane / 8, position lane % 8 of its
    // row, which holds K's chunk (position ^ key / 2 % 8), V's (position ^ 2 (key / 2 % 2))
    const int rk = lane >> 3;
    // (a step past the phase's last tile re-reads the last tile of the context, and past its last key
    // that key: they are there, and not used)
    auto first_key = [&](int step, int q) LG_INLINE {
        const int tile = min(step * KP + phase, tiles - 1);
        return min(tile * kC64Keys + 8 * (kReq * cw + q), (visible - 1) & ~7);
    };
    // (block_shift >= 0: log2 of the block size)
    auto block_of = [&](int key) LG_INLINE { return block_shift >= 0 ? key >> block_shift : key / p.block_size; };
    // Block ids are read a step ahead of the requests that need them.
    int ids[kReq];
    auto load_ids = [&](int step) LG_INLINE {
#pragma unroll
        for (int q = 0; q < kReq; ++q) ids[q] = table[block_of(first_key(step, q))];
    };
    auto request_tile = [&](int step, int buf) LG_INLINE {
#pragma unroll
        for (int q = 0; q < kReq; ++q) {
            const int k8 = 8 * (kReq * cw + q);  // first key of the request in the tile
            const int key0 = first_key(step, q);
            const int in_block = key0 - block_of(key0) * p.block_size;
            const int64_t base = ((int64_t)ids[q] * p.block_size + in_block) * row_bytes;
            const unsigned at = (unsigned)min(rk, visible - 1 - key0) * row_bytes;
            const int key = k8 + rk;  // its place in the tile
            const unsigned ko = at + (unsigned)((lane & 7) ^ ((key >> 1) & 7)) * 16u;
            const unsigned vo = at + (unsigned)((lane & 7) ^ (2 * ((key >> 1) & 1))) * 16u;
            const unsigned dst = __builtin_amdgcn_readfirstlane(ring + (unsigned)buf * kBuf + (unsigned)k8 * 128u);
            const char* ks = kp + base;
            const char* vs = vp + base;
            request_lds16(ks, ko, dst);
            request_lds16(vs, vo, dst + kC64Tile);
        }
    };

    const unsigned k_rd = ring + (unsigned)col * 128u;
    const int s16 = lane & 15, vrow = 4 * h + (s16 >> 2);
    unsigned v_rd[2];  // by 32 elements of the head
#pragma unroll
    for (int dt = 0; dt < 2; ++dt) {
        const int el = 32 * dt + 16 * ((lane >> 4) & 1) + 4 * (s16 & 3);
        v_rd[dt] = ring + kC64Tile + (unsigned)vrow * 128u +
                   (unsigned)((el >> 3) ^ (2 * ((vrow >> 1) & 1))) * 16u + (unsigned)(el & 4) * 2u;
    }

    float m = -INFINITY, l = 0.0f;
    float16_t o[2] = {};

    const unsigned k_swz = (unsigned)((col >> 1) & 7);
    // CAREFUL: a key that a column does not see has the probability 0 there, and 0 times an infinity or NaN
    // of its V row is a NaN.  The first walk over the keys takes no notice; if its results are not all
    // finite, a second one takes a pass of its own for every number of keys that a column of the wave
    // sees in a tile.  (Looked for in the V rows of the tiles in which a column ends, non-finite values
    // cost 1 to 7 % of a launch.)
    auto tile_step = [&](auto careful_c, int step, int buf) LG_INLINE {
        constexpr bool CAREFUL = decltype(careful_c)::value != 0;
        const unsigned off = (unsigned)buf * kBuf;
        half8_t ka[2][4];  // [32 keys][16 elements]
        {
            const unsigned a = k_rd + off;
            const unsigned a0 = a + ((unsigned)h ^ k_swz) * 16u, a1 = a + ((unsigned)(2 + h) ^ k_swz) * 16u;
            const unsigned a2 = a + ((unsigned)(4 + h) ^ k_swz) * 16u, a3 = a + ((unsigned)(6 + h) ^ k_swz) * 16u;
            asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\tds_read_b128 %2, %10\n\t"
                         "ds_read_b128 %3, %11\n\tds_read_b128 %4, %8 offset:4096\n\t"
                         "ds_read_b128 %5, %9 offset:4096\n\tds_read_b128 %6, %10 offset:4096\n\t"
                         "ds_read_b128 %7, %11 offset:4096\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(ka[0][0]), "=&v"(ka[0][1]), "=&v"(ka[0][2]), "=&v"(ka[0][3]),
                           "=&v"(ka[1][0]), "=&v"(ka[1][1]), "=&v"(ka[1][2]), "=&v"(ka[1][3])
                         : "v"(a0), "v"(a1), "v"(a2), "v"(a3)
                         : "memory");
        }
        uint2_t vl[4][2], vh[4][2];  // [16 keys][32 elements]: keys 4 h .. + 3, 8 + 4 h .. + 3
        static_for<4>([&](auto kb_c) LG_INLINE {
            constexpr int at = decltype(kb_c)::value * 2048;
            uint2_t(&lo)[2] = vl[decltype(kb_c)::value];
            uint2_t(&hi)[2] = vh[decltype(kb_c)::value];
            const unsigned v0 = v_rd[0] + off, v1 = v_rd[1] + off;
            asm volatile("ds_read_b64_tr_b16 %0, %4 offset:%c6\n\tds_read_b64_tr_b16 %1, %4 offset:%c7\n\t"
                         "ds_read_b64_tr_b16 %2, %5 offset:%c6\n\tds_read_b64_tr_b16 %3, %5 offset:%c7"
                         : "=&v"(lo[0]), "=&v"(hi[0]), "=&v"(lo[1]), "=&v"(hi[1])
                         : "v"(v0), "v"(v1), "n"(at), "n"(at + 1024)
                         : "memory");
        });
        float16_t sc[2];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 16; ++e) sc[b][e] = 0.0f;
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
            for (int b = 0; b < 2; ++b)
                sc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka[b][st], qb[st], sc[b], 0, 0, 0);
        const int key0 = (step * KP + phase) * kC64Keys;
        if (key0 + kC64Keys > first_vis) {  // (a whole-wave branch) some column ends in the tile
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    sc[b][e] = key0 + 32 * b + 8 * (e >> 2) + 4 * h + (e & 3) < vis ? sc[b][e] : -INFINITY;
        }
        float mx[2] = {sc[0][0], sc[1][0]};
#pragma unroll
        for (int e = 1; e < 16; ++e)
#pragma unroll
            for (int b = 0; b < 2; ++b) mx[b] = fmaxf(mx[b], sc[b][e]);
        mx[0] = fmaxf(mx[0], mx[1]);
        const float tmax = fmaxf(mx[0], lane_xor_f32<32>(mx[0])) * p.scale_log2e;
        if (__builtin_amdgcn_ballot_w64(tmax > m) != 0) {
            const float m_new = fmaxf(m, tmax);
            const float alpha = m_new == -INFINITY ? 1.0f : fast_exp2(m - m_new);
            m = m_new;
            l *= alpha;
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[dt][e] *= alpha;
        }
        const float mref = m == -INFINITY ? 0.0f : m;
        // probabilities as two fp16 terms: the rounded value, and what the rounding left
        uint4_t pa[4], pb[4];
        float ps[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 16; e += 2) {
                const float p0 = fast_exp2(fmaf(sc[b][e], p.scale_log2e, -mref));
                const float p1 = fast_exp2(fmaf(sc[b][e + 1], p.scale_log2e, -mref));
                ps[e & 3] += p0;
                ps[(e & 3) + 1] += p1;
                unsigned hi = __builtin_bit_cast(unsigned, half2_t{(_Float16)p0, (_Float16)p1});
                asm("" : "+v"(hi));  // (else each half is converted a second time by itself)
                const half2_t hv = __builtin_bit_cast(half2_t, hi);
                pa[2 * b + (e >> 3)][(e & 7) >> 1] = hi;
                const half2_t lo = {(_Float16)(p0 - (float)hv[0]), (_Float16)(p1 - (float)hv[1])};
                pb[2 * b + (e >> 3)][(e & 7) >> 1] = __builtin_bit_cast(unsigned, lo);
            }
        l += (ps[0] + ps[1]) + (ps[2] + ps[3]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        static_for<4>([&](auto kb_c) LG_INLINE {
            uint2_t(&lo)[2] = vl[decltype(kb_c)::value];
            uint2_t(&hi)[2] = vh[decltype(kb_c)::value];
            asm volatile("" : "+v"(lo[0]), "+v"(hi[0]), "+v"(lo[1]), "+v"(hi[1])::"memory");
        });
        // O += V^T . P^T of the tile (ALL), or of its keys in front of key `keys` + 4 h of it
        auto products = [&](auto all_c, int keys, float16_t(&acc)[2]) LG_INLINE {
            static_for<4>([&](auto kb_c) LG_INLINE {
                constexpr int kb = decltype(kb_c)::value;
                uint4_t v[2];
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) v[dt] = uint4_t{vl[kb][dt][0], vl[kb][dt][1], vh[kb][dt][0], vh[kb][dt][1]};
                if constexpr (!decltype(all_c)::value) {
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const int at = 16 * kb + 2 * w + (w > 1 ? 4 : 0);  // (and 4 h: its first key)
                        const unsigned m = keys >= at + 2 ? ~0u : keys == at + 1 ? 0xffffu : 0u;
                        v[0][w] &= m;
                        v[1][w] &= m;
                    }
                }
                half8_t va[2];
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) va[dt] = __builtin_bit_cast(half8_t, v[dt]);
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
                    acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[dt], __builtin_bit_cast(half8_t, pa[kb]), acc[dt], 0, 0, 0);
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
                    acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[dt], __builtin_bit_cast(half8_t, pb[kb]), acc[dt], 0, 0, 0);
            });
        };
        if (!CAREFUL || key0 + kC64Keys <= first_vis) {
            products(ic<1>{}, kC64Keys, o);
        } else {
            for (int seen = first_vis; seen <= last_vis; ++seen) {
                float16_t t[2] = {o[0], o[1]};
                products(ic<0>{}, seen - key0 - 4 * h, t);
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int e = 0; e < 16; ++e) o[dt][e] = vis == seen ? t[dt][e] : o[dt][e];
            }
        }
    };

    auto walk = [&](auto careful_c) LG_INLINE {
        m = -INFINITY;
        l = 0.0f;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[dt][e] = 0.0f;
        for (int u = 0; u < kBufs - 1; ++u)
            if (u < steps) {
                load_ids(u);
                request_tile(u, u);
            }
        load_ids(kBufs - 1);
        int buf = 0;
        for (int i = 0; i < steps; ++i) {
            // this wave's requests of step i have landed (those of the steps behind it may be on their
            // way; they complete in the order they were issued), behind the barrier everybody's have,
            // and everybody has left step i - 1, whose buffer step i + kBufs - 1 takes
            if (i + kBufs - 2 < steps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kBufs - 2) * 2 * kReq) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (KP < 4 || i == 0) __builtin_amdgcn_s_barrier();
            if (i + kBufs - 1 < steps) {
                request_tile(i + kBufs - 1, (buf + kBufs - 1) & (kBufs - 1));
                load_ids(i + kBufs);
            }
            if (i * KP + phase < tiles) tile_step(careful_c, i, buf);
            buf = (buf + 1) & (kBufs - 1);
        }
    };
    if (steps > 0) {
        walk(ic<0>{});
        float odd = 0.0f;  // NaN if a result is not finite
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) odd = fmaf(o[dt][e], 0.0f, odd);
        if (lane == 0) odd_waves[wave] = 0u;
        if (odd != odd) odd_waves[wave] = 1u;
        __syncthreads();  // (and behind it the rings are free)
        if (__builtin_amdgcn_readfirstlane(odd_waves[0] | odd_waves[1] | odd_waves[2] | odd_waves[3]) != 0) {
            walk(ic<1>{});
            __syncthreads();
        }
    }

    l += lane_xor_f32<32>(l);
    if constexpr (KP > 1) {
        // the phases' states into phase 0's; a phase without a key of the column has m = -inf, l = 0, o = 0
        float* const sm = reinterpret_cast<float*>(c64_lds);  // [phase - 1][cw][34][lane]
        if (phase > 0) {
            float* dst = sm + (size_t)((phase - 1) * CW + cw) * 34 * 64 + lane;
            dst[0] = m;
            dst[64] = l;
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int e = 0; e < 16; ++e) dst[(2 + 16 * dt + e) * 64] = o[dt][e];
        }
        __syncthreads();
        if (phase > 0) return;
        float mall = m;
#pragma unroll
        for (int f = 0; f < KP - 1; ++f) mall = fmaxf(mall, sm[(size_t)(f * CW + cw) * 34 * 64 + lane]);
        const float ref = mall == -INFINITY ? 0.0f : mall;
        const float own = fast_exp2(m - ref);
        l *= own;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[dt][e] *= own;
#pragma unroll
        for (int f = 0; f < KP - 1; ++f) {
            const float* src = sm + (size_t)(f * CW + cw) * 34 * 64 + lane;
            const float w = fast_exp2(src[0] - ref);
            l = fmaf(w, src[64], l);
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[dt][e] = fmaf(w, src[(2 + 16 * dt + e) * 64], o[dt][e]);
        }
    }
    if (!live) return;
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;  // a column that sees no key: zeros
    unsigned short* const out = reinterpret_cast<unsigned short*>(p.out) +
                                ((int64_t)(row0 + tok) * p.hq + (int64_t)kvh * G + head) * 64;
    // (one branch for all elements)
    auto write = [&](auto bf16_c) LG_INLINE {
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                uint2_t w;
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    w[e] = (unsigned)attn_out_elem(o[dt][4 * g + 2 * e] * inv, decltype(bf16_c)::value) |
                           ((unsigned)attn_out_elem(o[dt][4 * g + 2 * e + 1] * inv, decltype(bf16_c)::value) << 16);
                *reinterpret_cast<uint2_t*>(out + 32 * dt + 8 * g + 4 * h) = w;
            }
    };
    if (p.out_bf16) write(ic<1>{});
    else write(ic<0>{});
}

template <int CW, int KP>
static hipError_t launch_chunk64(const AttnParams& p, int max_seqlen_q, hipStream_t stream) {
    constexpr int lds = KP * c64_bufs(KP) * 2 * kC64Tile;  // (and 34 * 64 floats per wave of a later phase)
    static_assert(lds >= (KP - 1) * CW * 34 * 64 * 4, "the phases' states fit the rings");
    const auto kernel = paged_attn_chunk64_kernel<CW, KP>;
    static const hipError_t opt = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (opt != hipSuccess) return opt;
    const int g = p.hq / p.hkv;
    const int64_t groups = ((int64_t)max_seqlen_q * g + 32 * CW - 1) / (32 * CW);
    int shift = -1;
    if ((p.block_size & (p.block_size - 1)) == 0)
        for (shift = 0; (1 << shift) < p.block_size;) ++shift;
    kernel<<<dim3((unsigned)groups, p.hkv, p.num_seqs), dim3(256), lds, stream>>>(p, g, shift);
    return hipGetLastError();
}

// Which split a launch takes, from what the host knows: the tokens of the longest chunk, all packed rows and
// the block tables' length.  If all rows came in chunks of that length there would be `chunks` of them.
// us, the general kernel / CW = 4 / 2 / 1:
//   8 x 512 tokens, contexts to 4600, 14 / 2 heads: 257 / 116 / 131 / 157; 2 x 512 to 1500: 36 / 29.8 / 20.8 / 26.0
//   1 x 20, a context of 4000, 14 / 2:              34 / 46 / 30 / 23
//   1 x 512 at 8000, 16 / 16:                       101 / 160 / 99 / 68 (256 workgroups at CW = 1: one round)
//   1 x 2000 at 6000, 16 / 2:                       316 / 151 / 161 / 207
//   1 x 128 and 1 x 32 alone, 14 / 2:               8.8 / 8.5 / 7.6 / 7.9 and 7.6 / 7.2 / 7.5 / 7.9
//   200 x 2 at 300, 8 / 8:                          34 / 44 / 54 / 54;  64 x 2 at 300: 18.1 / 19.1 / 20.4 / 20.5
//   1 x 32 at 16000, 8 / 1:                         95 / 296 / 178 / 114;  1 x 512 at 8000: 55 / 159 / 97 / 65
//   1 x 2000 alone, 8 / 1:                          40 / 44 / 29 / 26
constexpr int kC64General = 0;
static int chunk64_columns(const AttnParams& p, int64_t total_tokens, int64_t max_seqlen_q) {
    const int64_t g = p.hq / p.hkv, cols = max_seqlen_q * g, cus = device_cu_count();
    const int64_t keys = (int64_t)p.block_size * p.max_blocks_per_seq;
    const int64_t chunks_hkv = total_tokens * p.hkv;  // (chunks x hkv x max_seqlen_q)
    auto workgroups = [&](int64_t cw) { return chunks_hkv * ((cols + 32 * cw - 1) / (32 * cw)) / max_seqlen_q; };
    // The general kernel: where a KV head has all eight of its waves, which walk a long context faster
    // than four here, as long as its tiles of 16 columns are about one per unit; and where a whole chunk is
    // one such tile and there are more chunks than units (a tile of 32 columns here is half empty).
    const int64_t tile = 16 / g;
    if (anydim_wg_heads(p.hkv) % 2 == 1 && keys > 512 &&
        (total_tokens + tile - 1) / tile * p.hkv <= cus + cus / 4)
        return kC64General;
    if (max_seqlen_q <= tile && workgroups(1) > cus) return kC64General;
    if (keys <= kC64Keys) return 4;  // (a key phase needs a tile)
    if (total_tokens * p.hq / 128 >= cus && cols > 32) return 4;
    if (keys <= 2 * kC64Keys) return 2;
    return workgroups(1) <= cus || cols <= 32 ? 1 : 2;
}

bool paged_attn_chunk64_applies(const AttnParams& p, int head_dim, int total_tokens, int max_seqlen_q) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(p.k_pool) | reinterpret_cast<uintptr_t>(p.v_pool) |
                         reinterpret_cast<uintptr_t>(p.q) | reinterpret_cast<uintptr_t>(p.out);
    return head_dim == 64 && (at & 15u) == 0 && chunk64_columns(p, total_tokens, max_seqlen_q) != kC64General;
}

hipError_t paged_attn_chunk64_launch(const AttnParams& p, int total_tokens, int max_seqlen_q,
                                     hipStream_t stream) {
    switch (chunk64_columns(p, total_tokens, max_seqlen_q)) {
        case 4: return launch_chunk64<4, 1>(p, max_seqlen_q, stream);
        case 2: return launch_chunk64<2, 2>(p, max_seqlen_q, stream);
        default: return launch_chunk64<1, 4>(p, max_seqlen_q, stream);
    }
}

}  // namespace lg
