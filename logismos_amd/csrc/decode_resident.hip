// All layers of a decode step of one row as ONE resident launch.
//
//   A step of one row is a chain of dependent products over a few KiB of activations.  As six launches
//   a layer (qgemm_q4_rows.hip) each link costs a launch boundary, the ramp of its weights from
//   memory and its drain: 4.6 us, of which the weights need 0.2-2 us.  Here one workgroup per compute
//   unit stays for the whole step and two things overlap that a launch boundary keeps apart:
//
// * Weights (and K/V tiles) do not depend on activations.  Eight STREAMING waves per workgroup walk
//   the step's whole sequence of weight tiles and K/V tiles through private rings in LDS, requested
//   straight into it (global_load_lds) as far ahead as the ring holds, across operators and layers: while
//   the workgroups exchange activations, the next operator's weights arrive.
// * Activations pass between workgroups as 8-byte words {value, tag}, written and read past the L2s
//   (device scope): a reader polls the values themselves, there is no barrier, flag or counter, and an
//   exchange costs one store and one load through the fabric.  Four FRONT waves per workgroup poll them,
//   normalise, and lay the operand out in LDS; after the product they add up the streaming waves' parts,
//   apply the epilogue and publish.  256 workgroups that all read 32 KiB of such words: 2.4 us a round; a
//   barrier over counters took 7.6-11.4 us, flags beside the data 4.6.
//
// Per layer: row normed -> q/k/v, bias, rotation, K/V row into the pools | attention of one piece of
// the context for one KV head per workgroup | (merge of the pieces) | o projection + residual | row
// normed -> gate/up, SwiGLU | down projection + residual.
//
// What bounds it, from clock stamps at widths 896 / 4096 (us per layer 20 / 40): five exchanges of 2-4 us (six where the
// pieces are merged), of which the poll 1.3-2 and what follows it up to the barrier 1; products 0.6-2 / 1-8 (at
// 4096 they wait for memory: 370 KiB per compute unit and layer at 23-27 B/ns, 192 of them gate/up); epilogues 0.6 each.
// A compute unit's requests return in order, so a poll also waits for what the streaming waves asked for before it.
// Every instruction of a front wave is on the chain: for two to four rows the same kernel was slower than the launches it
// replaces (0.81-1.01 of their speed), hence one row.  (More uniform values are alive than there are scalar registers: 80-odd
// of each instance lie in lanes of vector registers.  The build refuses one that spills a vector register.)
//
// Steps of one row, us (six launches a layer / here): 24 layers of 896 at 500 keys 674 / 502, 28 of 1536 at 4000 keys
// 912 / 773, 36 of 4096 at 1500 keys 1885 / 1524.
//
// Work is cut for V workgroups (one per compute unit) before the launch: a small kernel writes, for each and
// for each of its streaming waves, the list of a layer's batches (up to four groups of K of a tile, or a
// K/V tile), which a wave keeps in its registers.
//
// Waits end: a launch does not assume that all of its workgroups run at once.  Each takes a ticket;
// the last one, or one that has waited 100 us, closes the step to the n workgroups that hold tickets so
// far, which are all running; later ones leave.  Workgroup r does the parts r, r + n, ... of the V, so
// results do not depend on n.  Times do (us with 256 | 255 | 128 | 64 | 32 | 10 workgroups: 24 layers of 896 473 | 635 | 580 |
// 833 | 1470 | 4591, 36 of 4096 1425 | 2317 | 2398 | 4441 | 8427 | 26900): a wave with several parts requests no
// weights ahead of its phase.  Waiting longer than 100 us was measured beside GEMMs, prompt attention and other steps on a
// second stream and gained in none of them.  A tag is written by whoever owns the value in every case, whatever the
// batch holds.  A budget of polls bounds the kernel even so.  A wave that has spent it says so in the region, and
// all that its workgroup publishes from there on is NaN, which every product behind it hands on: the residual stream
// ends as NaN, and K/V rows that are NaN on that account are left out of the pools.
//
// A buffer of words is reused by the next layer without a wait: between two writes of a word lies the
// whole chain of a layer, and the workgroups of every link read all of what the one before it wrote.
#include "decode_resident.hpp"

#include "device_utils.hpp"
#include "launch_common.hpp"
#include "paged_attn_params.hpp"
#include "q4_common.hpp"
#include "q4_rows.hpp"

#include <hip/hip_fp16.h>
#include <math.h>

namespace lg {

namespace {

constexpr int kStreamWaves = 8;
constexpr int kFrontWaves = 4;
constexpr int kFrontThreads = 64 * kFrontWaves;
constexpr int kThreads = 64 * (kStreamWaves + kFrontWaves);
constexpr int kSlot = 4096;         // bytes of a ring slot: four requests of a wave
// (24 layers of 896 with 2 | 3 | 4 | 5 slots: 505 | 485 | 480 | 480 us; 28 of 1536 792 | 777 | 777 | 777)
constexpr int kMaxSlots = 4;
constexpr int kResLds = 160 * 1024;
constexpr int kMaxParts = 256;      // V: parts the work is cut into, and pieces of its attention
constexpr int kMaxTilesHeld = 15;   // tiles of a projection in a part
constexpr int kMaxList = 512;       // batches of a wave's part of a layer
constexpr int kNormChunks = 2;      // chunks of eight columns a front thread normalises
// The partials of the context's pieces: the o projection's workgroups read them themselves where a thread has one chunk of
// eight columns and they are few words, otherwise a workgroup per head merges them, which is one exchange more.  us of 16
// layers, read / merged: 512 columns of heads, 1 | 4 | 8 pieces 241 / 273 | 247 / 274 | 262 / 274; 896, 325 / 353 | 326 / 357 |
// 341 / 340; 1536 (width 1536), 429 / 449 | 434 / 460; but 2048 (width 2048), 1 | 2 pieces 397 / 374 | 414 / 377 (width 1024, one
// piece 297 / 308); 2560, 551 / 513 | 574 / 525; 4096, 692 / 640 | 780 / 716.
constexpr int kDirectWords = 8192, kDirectColumns = 1536;
constexpr int kCloseAfter = 10000;  // ticks of 10 ns that a workgroup waits for the others
constexpr int kPollBudget = 1 << 21;  // of a wave and step: seconds, where a step's waits are some hundred polls

// What a merge of pieces starts from: below every score, and finite, so that a piece whose keys all score -inf weighs
// nothing (from -inf the difference of the two maxima is NaN).
constexpr float kNoKey = -3.402823466e38f;

// the projections, in the order of a layer; attention stands between the first two
enum { kQkv = 0, kO = 1, kGateUp = 2, kDown = 3 };
enum { kPhaseQkv = 0, kPhaseAttn = 1, kPhaseO = 2, kPhaseGateUp = 3, kPhaseDown = 4, kPhases = 5 };

struct ResidentLayer {
    const uint8_t* qw[4];
    const __half* scale[4];
    const __half* zero[4];
    const float *norm1, *norm2, *bias;
    __half *k_pool, *v_pool;
};
constexpr int kLayersPerInit = 24;  // what the arguments of one launch hold
struct ResidentLayers {
    ResidentLayer l[kLayersPerInit];
};

// One batch of a streaming wave.  at: byte offset of its first weight group, or the K/V head row of its
// first key.  what: groups c (bits 0..2; kKvTile; 0: nothing to multiply), last of its tile (bit 3), tile of
// the part (4..7), first group (8..15) or keys that are seen (8..15), projection (16..17).  form: of a K/V
// tile, 1 + the key at which this step appends its row, or 0; otherwise bytes of a weight row and rows to the
// tile's second run, less 8 (16 bits each).
struct Batch {
    unsigned at, what, form, none;
};
constexpr int kKvTile = 5;
// Of a part: the attention piece it computes.
struct Piece {
    int count, unit, kvh, none;  // count: pieces of the context; 0: this part has none
};
// Of the step: pieces of the context (0: no key is seen), and whether a workgroup per head merges them.
struct StepInfo {
    int pieces, merged;
};

struct ResidentPlan {
    int layers, hidden, inter, hq, hkv, group;
    int block_size, max_blocks, max_pos;
    float eps, scale_log2e;
    int parts;           // V
    int list;            // batches that a wave's list has room for
    int slots;           // per streaming wave
    // LDS, bytes from the start
    unsigned group_inv[4];  // of the projections' groups of K: 2^20 / groups, rounded up
    int lds_x, lds_red, lds_scale[2], lds_ssq, lds_misc;
    // the region: bytes from its start
    unsigned at_step, at_pieces, at_starts, at_lists, at_h, at_qkv, at_part, at_x, at_act, bytes;
    char* region;
    const ResidentLayer* table;
    float* h;
    const int32_t *block_tables, *cu, *ctx, *positions;
    const int64_t* slot_mapping;
    const float *cos_t, *sin_t;
    int polls;  // after which a front wave gives up (at the end: further up it moves fields that are loaded together, 1.3 %)
    unsigned all;  // tickets with which the step is closed at once
};

#define LG_CONST __attribute__((address_space(4)))
// The kernel's arguments where they are, in constant memory: fields are loaded where they are used (as a
// value all of them are held in scalar registers from the start, more than there are).
using Plan = const LG_CONST ResidentPlan;
__device__ __forceinline__ Plan& arguments() {
    Plan* a = (Plan*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    return *a;
}

// a scalar load (the address is uniform)
template <typename T>
__device__ __forceinline__ T uniform_load(const T* p) {
    return *reinterpret_cast<const LG_CONST T*>(reinterpret_cast<uintptr_t>(p));
}
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ void block_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ---- words {value, tag}
constexpr int kPastCaches = 16;  // sc1 of a buffer load: device scope
struct Words {
    __amdgpu_buffer_rsrc_t rsrc;
    char* base;
    __device__ __forceinline__ Words(char* b, unsigned bytes)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc(b, 0, bytes, 0x00020000)), base(b) {}
    // two words: {value, tag, value, tag}
    __device__ __forceinline__ uint4_t get2(unsigned at) const {
        return __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, at, 0, kPastCaches));
    }
    __device__ __forceinline__ uint2_t get(unsigned at) const {
        return __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(rsrc, at, 0, kPastCaches));
    }
    __device__ __forceinline__ void put(unsigned at, unsigned value, unsigned tag) const {
        __hip_atomic_store(reinterpret_cast<unsigned long long*>(base + at),
                           ((unsigned long long)tag << 32) | value, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
};
__device__ __forceinline__ bool tagged(const uint4_t& v, unsigned tag) { return v[1] == tag && v[3] == tag; }

struct Shape {  // of a projection
    int tiles, k;
};
template <typename P>
__device__ __forceinline__ Shape proj_shape(P& p, int which, int d) {
    if (which == kQkv) return {(p.hq + 2 * p.hkv) * d / 16, p.hidden};
    if (which == kO) return {p.hidden / 16, p.hq * d};
    if (which == kGateUp) return {p.inter / 8, p.hidden};
    return {p.hidden / 16, p.inter};
}
// A tile is two runs of eight weight rows: for the rotation the two halves of its pairs, for the
// SwiGLU the gate and the up rows of the same outputs.
template <int D>
__device__ __forceinline__ int tile_first(int which, int t) {
    if (which == kQkv) return 8 * t + t / (D / 16) * (D / 2);
    return which == kGateUp ? 8 * t : 16 * t;
}
template <int D, typename P>
__device__ __forceinline__ int tile_apart(P& p, int which) {
    return which == kQkv ? D / 2 : (which == kGateUp ? p.inter : 8);
}
// tiles of part v
__device__ __forceinline__ int tiles_of(int v, int parts, int tiles) {
    return v < tiles ? (tiles - v + parts - 1) / parts : 0;
}

// 16-byte piece pc of row r of a batch of c groups lies where piece pc ^ swizzle(r, c) would: eight rows
// read at the same piece are on eight different runs of banks.
__device__ __forceinline__ int swizzle(int r, int c) { return c == 1 ? (r >> 1) & 3 : r & 7; }

// all but the newest `left` requests are there (or a few of those too: an exact count takes more branches than
// the rounding costs; rings of whole batches of four ask for multiples of four)
__device__ __forceinline__ void wait_requests(int left) {
    if (left >= 4) {
        if (left >= 8) {
            if (left >= 12) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        }
    } else {
        if (left >= 2) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
}

// bytes of the attention's part of the operand area: queries, the token's K and V row, partials
__host__ __device__ inline int attn_q_stride(int d) { return 2 * d + 16; }
__host__ __device__ inline int attn_new_at(int d) { return 16 * attn_q_stride(d); }
__host__ __device__ inline int attn_part_at(int d) { return attn_new_at(d) + 2 * d * 2; }
__host__ __device__ inline int attn_part_floats(int d, int group) { return 32 + group * d; }

// ---------------------------------------------------------------------------- streaming waves
// A wave keeps 64 batches of its list in registers, one per lane: for the requests with their
// addresses in the present layer, for the products without.
template <int D>
struct Stream {
    static constexpr int KV = D / 32;  // requests of a K or V tile
    char* const lds;
    const int rank, n, wave, lane;
    const int parts, layers, slots;
    const unsigned ring, row_bytes;  // of the wave's ring; of a K/V pool's row
    const bool alone;                // one part: requests run ahead across operators and layers

    // the request side: batches [at, end) of the layer, `room` slots free
    int layer = 0, part, at = 0, end = 0, room;
    int have = -64;  // first batch held
    unsigned lo = 0, hi = 0, what_ = 0, form = 0;
    int64_t v_from_k = 0;  // from a layer's K pool to its V pool
    unsigned key = ~0u, off0 = 0, off1 = 0;
    int key_c = 0;
    int in = 0, out = 0, issued = 0, used = 0;
    // the computing side
    int now = -64, now_part = -1;
    unsigned now_what = 0, now_form = 0;

    __device__ __forceinline__ Stream(Plan& p, char* l, int r, int n_, int w, int ln)
        : lds(l), rank(r), n(n_), wave(w), lane(ln), parts(p.parts), layers(p.layers), slots(p.slots),
          ring((unsigned)(w * p.slots * kSlot)), row_bytes((unsigned)p.hkv * (2u * D)), alone(n_ == p.parts),
          part(r), room(p.slots) {}

    __device__ __forceinline__ const uint4_t* list(Plan& p, int v) const {
        return reinterpret_cast<const uint4_t*>(p.region + p.at_lists) + ((size_t)v * kStreamWaves + wave) * p.list;
    }
    // this lane, so that what follows from it is worked out where it is used: carried through the whole kernel it
    // costs registers that the operand needs
    __device__ __forceinline__ int here() const {
        int l = lane;
        asm volatile("" : "+v"(l));
        return l;
    }
    // batches [x, y) of a phase in a part's list
    __device__ __forceinline__ int2 range(Plan& p, int v, int ph) const {
        const int* s = reinterpret_cast<const int*>(p.region + p.at_starts) + ((size_t)v * kStreamWaves + wave) * 8 + ph;
        return int2{uniform_load(s), uniform_load(s + 1)};
    }
    // batches from i on, with their addresses in the present layer
    __device__ __forceinline__ void hold(int v, int i) {
        Plan& p = arguments();
        const uint4_t b = list(p, v)[min(i + lane, p.list - 1)];
        const ResidentLayer* const L = p.table + layer;
        const unsigned which = (b[1] >> 16) & 3u;
        const bool kv = (b[1] & 7u) == kKvTile;
        uint64_t base = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint64_t q = reinterpret_cast<uint64_t>(uniform_load(&L->qw[j]));
            base = which == (unsigned)j ? q : base;
        }
        const uint64_t k = reinterpret_cast<uint64_t>(uniform_load(&L->k_pool));
        v_from_k = (int64_t)(reinterpret_cast<uint64_t>(uniform_load(&L->v_pool)) - k);
        base = kv ? k + (uint64_t)b[0] * (2 * D) : base + b[0];
        lo = (unsigned)base;
        hi = (unsigned)(base >> 32);
        what_ = b[1];
        form = b[2];
        have = i;
    }
    static __device__ __forceinline__ unsigned of(unsigned v, int i) {
        return (unsigned)__builtin_amdgcn_readlane((int)v, i);
    }
    static __device__ __forceinline__ const char* address(unsigned l, unsigned h) {
        return reinterpret_cast<const char*>(((uint64_t)h << 32) | l);
    }
    // This lane's bytes from the first weight row, of a batch of c = 1, 2 or 4 groups: a request is 16, 8 or
    // 4 rows, and those of a tile's second run are as far from each other as those of its first.
    __device__ __forceinline__ void weight_offsets(int c, unsigned khalf, unsigned second) {
        const int pieces = 4 * c, shift = c == 4 ? 4 : (c == 2 ? 3 : 2), lane = here();
        const int row = lane >> shift, pc = lane & (pieces - 1);
        off0 = __umul24((unsigned)(row & 7), khalf) + (row < 8 ? 0u : second) + (unsigned)((pc ^ swizzle(row, c)) * 16);
        off1 = __umul24((unsigned)(row + 4), khalf) + (unsigned)((pc ^ swizzle(row + 4, c)) * 16);
    }
    // The next batch of the sequence, its slots taken: c = 0 where the ring has no room or the step has no
    // more.  A K/V tile's requests are sent here.
    struct Next {
        unsigned lo, hi;       // address of its first row
        unsigned second, dst;  // the second run of its rows from the first; its slot
        int c;
    };
    __device__ __forceinline__ Next next() {
        Next q{0, 0, 0, 0, 0};
#pragma unroll 1
        while (room) {
            if (at == end) {
                if (!alone || end == 0 || layer + 1 >= layers) return q;  // (0: a part without work)
                layer = uniform(layer + 1);
                at = 0;
                have = -64;
            }
            if ((unsigned)(at - have) >= 64u) hold(part, at);
            const int i = at - have;
            const unsigned what = of(what_, i);
            const int c = what & 7;
            if (c == kKvTile && room < 2) return q;
            ++at;
            if (c == 0) continue;
            q.dst = ring + (unsigned)in * kSlot;
            q.lo = of(lo, i);
            q.hi = of(hi, i);
            in = in + 1 == slots ? 0 : in + 1;
            --room;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slots' last reads are through
            if (c != kKvTile) {
                const unsigned f = of(form, i);
                q.second = (f & 0xffffu) * ((f >> 16) + 8u);
                q.c = c;
                if (f != key || c != key_c) {
                    weight_offsets(c, f & 0xffffu, q.second);
                    key = f;
                    key_c = c;
                }
                return q;
            }
            constexpr int PER = D / 8, KEYS = 64 / PER;  // pieces of a row, rows per request
            const int lane = here();
            const unsigned vdst = ring + (unsigned)in * kSlot;
            const char *const ksrc = address(q.lo, q.hi), *const vsrc = ksrc + v_from_k;
            in = in + 1 == slots ? 0 : in + 1;
            --room;
            const unsigned pos = lane % PER;
            const int last = (int)((what >> 8) & 255u) - 1;  // keys past the context: its last one again
#pragma unroll
            for (int r = 0; r < KV; ++r) {
                const int kk = r * KEYS + lane / PER;
                const unsigned row = (unsigned)min(kk, last) * row_bytes;
                request_lds16(ksrc, row + ((pos ^ (unsigned)(kk & 7)) * 16u), q.dst + r * 1024);
                request_lds16(vsrc, row + pos * 16u, vdst + r * 1024);
            }
            issued += 2 * KV;
        }
        return q;
    }
    // request r (0 .. 3) of a batch of weights, where it has one
    __device__ __forceinline__ void send(const Next& q, int r) {
        if (r == 0 ? q.c == 0 : (r == 2 ? q.c < 2 : q.c != 4)) return;
        const char* const src = address((unsigned)uniform((int)q.lo), (unsigned)uniform((int)q.hi));
        request_lds16(r < 2 ? src : src + (unsigned)uniform((int)q.second), (r & 1) ? off1 : off0,
                      (unsigned)uniform((int)(q.dst + (r == 2 ? q.c * 512 : r * 1024))));
        ++issued;
    }
    __device__ __forceinline__ void fill() {
#pragma unroll 1
        while (true) {
            const Next q = next();
            if (q.c == 0) return;
#pragma unroll
            for (int r = 0; r < 4; ++r) send(q, r);
        }
    }
    // several parts: the requests of a phase's range only, when it is its turn
    __device__ __forceinline__ void start(int v, int l, const int2& r) {
        if (alone) return;
        layer = l;
        part = v;
        at = r.x;
        end = r.y;
        have = -64;
        fill();
    }
    __device__ __forceinline__ char* next_slot() {
        char* s = lds + ring + out * kSlot;
        out = out + 1 == slots ? 0 : out + 1;
        return s;
    }
    // the oldest batch is in LDS
    __device__ __forceinline__ void arrive(int requests) {
        used += requests;
        wait_requests(issued - used);
    }
    // batch i of part v for the computing side: the lane that holds it
    __device__ __forceinline__ int reach(Plan& p, int v, int i) {
        if (v != now_part || (unsigned)(i - now) >= 64u) {
            const uint4_t b = list(p, v)[min(i + lane, p.list - 1)];
            now_what = b[1];
            now_form = b[2];
            now = i;
            now_part = v;
        }
        return i - now;
    }

    // ---- a projection of the operand in LDS: batches [x, y) of at most C groups
    template <int C>
    __device__ __forceinline__ void multiply(Plan& p, int wh, int v, const int2& r) {
        const int G = proj_shape(p, wh, D).k >> 7, lane = here();
        const int row = lane & 15, quarter = lane >> 4;
        const char* const xsrc = lds + p.lds_x + quarter * 64;
        const char* const scales = lds + ((wh & 1) ? p.lds_scale[1] : p.lds_scale[0]) + (row >> 3) * 16 * G +
                                   (row & 7) * G * 2;
        float* const red = reinterpret_cast<float*>(lds + p.lds_red) + wave * 16 + lane;
        const RowsConst cst;
        uint4_t x[C][4];
        float xs[C], y = 0.0f;
        int xg = -1;  // the group that x starts with
        unsigned what = of(now_what, r.x - now);
        block_barrier();  // operand and scales are there
#pragma unroll 1
        for (int i = r.x;;) {
            const int c = what & 7, t = (what >> 4) & 15, g = (what >> 8) & 255;
            if (C > 1 || c) {
                if (g != xg) {
                    // (groups past a shorter batch are not used: what is read lies in LDS)
#pragma unroll
                    for (int u = 0; u < C; ++u) {
#pragma unroll
                        for (int s4 = 0; s4 < 4; ++s4)
                            x[u][s4] = *reinterpret_cast<const uint4_t*>(xsrc + (g + u) * 256 + s4 * 16);
                    }
                    // (the matrix cores have time; a front wave's sums would be on the chain)
#pragma unroll
                    for (int u = 0; u < C; ++u) xs[u] = rows_group_sum(x[u], cst)[0];
                    xg = g;
                }
                const char* const sc = scales + t * 64 * G + g * 2;
                arrive(c);
                const char* const wsrc = next_slot() + row * 64 * c;
                const int sw = swizzle(row, c);
                uint4_t w[C];
                uint16_t scale[C], zero[C];
#pragma unroll
                for (int u = 0; u < C; ++u) {
                    w[u] = *reinterpret_cast<const uint4_t*>(wsrc + (((4 * u + quarter) ^ sw) * 16));
                    scale[u] = *reinterpret_cast<const uint16_t*>(sc + 2 * u);
                    zero[u] = *reinterpret_cast<const uint16_t*>(sc + 32 * G + 2 * u);
                }
                ++room;
                // the next requests between the products: sent together they hold the wave up for as long as
                // the products take
                Next q{0, 0, 0, 0, 0};
                if (r.y - i > slots - room) q = next();
                auto part_of = [&](auto uu) LG_INLINE {
                    constexpr int U = decltype(uu)::value % C;
                    // (all rows of the operand are the token's: any result row will do)
                    const float sf = __half2float(__ushort_as_half(scale[U]));
                    const float zf = 128.0f + __half2float(__ushort_as_half(zero[U]));
                    y = fmaf(sf, fmaf(-zf, xs[U], rows_product(w[U], x[U], cst)[0]), y);
                };
                part_of(ic<0>{});
                send(q, 0);
                if (C > 1 && c > 1) part_of(ic<1>{});
                send(q, 1);
                if (C > 2 && c > 2) part_of(ic<2>{});
                send(q, 2);
                if (C > 2 && c > 2) part_of(ic<3>{});
                send(q, 3);
            }
            if (what & 8) {
                if (lane < 16) red[t * (kStreamWaves * 16)] = y;
                y = 0.0f;
            }
            if (++i == r.y) break;
            const int held = reach(p, v, i);
            what = of(now_what, held);
        }
        block_barrier();  // the parts are there
    }
    __device__ __forceinline__ void project(int wh, int v, int l) {
        Plan& p = arguments();
        const int2 r = range(p, v, wh == kQkv ? kPhaseQkv : wh + 1);
        if (r.x == r.y) return;
        start(v, l, r);
        // a tile's first batches are its longest ones
        const int first = reach(p, v, r.x);
        const int c = of(now_what, first) & 7;
        if (c == 4) multiply<4>(p, wh, v, r);
        else if (c == 2) multiply<2>(p, wh, v, r);
        else multiply<1>(p, wh, v, r);
        fill();
    }

    // ---- attention: this wave's tiles of the part's piece
    __device__ __forceinline__ void attend(int v, int l) {
        constexpr int E = D / 16;  // elements of a value row per lane
        Plan& p = arguments();
        const Piece* const piece = reinterpret_cast<const Piece*>(p.region + p.at_pieces) + v;
        if (uniform_load(&piece->count) == 0) return;
        const int2 range_ = range(p, v, kPhaseAttn);
        start(v, l, range_);
        const int lane = here(), tg = lane >> 4, c = lane & 15, G = p.group;
        const float scale = p.scale_log2e;
        char* const area = lds + p.lds_x;
        block_barrier();  // the queries and the token's K/V row are there
        {
            half8_t q[KV];
#pragma unroll
            for (int j = 0; j < KV; ++j)
                q[j] = *reinterpret_cast<const half8_t*>(area + min(c, G - 1) * attn_q_stride(D) + (4 * j + tg) * 16);
            float m = -INFINITY, sum = 0.0f;
            float4_t acc[E];
#pragma unroll
            for (int e = 0; e < E; ++e) acc[e] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
            for (int i = range_.x; i < range_.y; ++i) {
                const int at_ = reach(p, v, i);
                const int seen = (int)((of(now_what, at_) >> 8) & 255u);
                const unsigned fresh = of(now_form, at_);
                arrive(2 * KV);
                char* const kt = next_slot();
                char* const vt = next_slot();
                room += 2;
                if (fresh && lane < D / 8) {
                    // the row that this step appends comes from the other workgroups' words, not from memory
                    const int k_ = (int)fresh - 1;
                    const uint4_t* src = reinterpret_cast<const uint4_t*>(area + attn_new_at(D));
                    *reinterpret_cast<uint4_t*>(kt + k_ * 2 * D + ((lane ^ (k_ & 7)) * 16)) = src[lane];
                    *reinterpret_cast<uint4_t*>(vt + k_ * 2 * D + lane * 16) = src[D / 8 + lane];
                }
                // keys past the context have no weight; what stands there must not be a NaN
                if (seen < kTileKeys)
                    for (int j = seen * (D / 8) + lane; j < kTileKeys * (D / 8); j += 64)
                        *reinterpret_cast<uint4_t*>(vt + j * 16) = uint4_t{0, 0, 0, 0};
                asm volatile("" ::: "memory");  // (one wave: its LDS accesses stay in this order)
                half8_t kk[KV];
#pragma unroll
                for (int j = 0; j < KV; ++j)
                    kk[j] = *reinterpret_cast<const half8_t*>(kt + c * 2 * D + (((4 * j + tg) ^ (c & 7)) * 16));
                unsigned val[4][E / 2];
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int e = 0; e < E / 4; ++e) {
                        const uint2_t w = *reinterpret_cast<const uint2_t*>(vt + (4 * tg + j) * 2 * D + c * 2 * E + e * 8);
                        val[j][2 * e] = w[0];
                        val[j][2 * e + 1] = w[1];
                    }
                float4_t sc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < KV; ++j) sc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kk[j], q[j], sc, 0, 0, 0);
                float mx = m;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    sc[r] = 4 * tg + r < seen ? sc[r] * scale : -INFINITY;
                    mx = fmaxf(mx, sc[r]);
                }
                mx = fmaxf(mx, lane_xor_f32<16>(mx));
                mx = fmaxf(mx, lane_xor_f32<32>(mx));
                const float safe = mx == -INFINITY ? 0.0f : mx;
                const float alpha = fast_exp2(m - safe);
                // the probabilities as two fp16 terms: the rounded value and the remainder
                half4_t pa, pb;
                float ps = 0.0f;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float pr = fast_exp2(sc[r] - safe);
                    ps += pr;
                    pa[r] = (_Float16)pr;
                    pb[r] = (_Float16)(pr - (float)pa[r]);
                }
                sum = sum * alpha + ps;
                m = mx;
                float ar[4];  // of the heads 4 tg + r
#pragma unroll
                for (int r = 0; r < 4; ++r) ar[r] = __shfl(alpha, 4 * tg + r, 64);
#pragma unroll
                for (int e = 0; e < E; ++e) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[e][r] *= ar[r];
                    const unsigned sel = (e & 1) ? 0x07060302u : 0x05040100u;
                    uint2_t b;
                    b[0] = __builtin_amdgcn_perm(val[1][e >> 1], val[0][e >> 1], sel);
                    b[1] = __builtin_amdgcn_perm(val[3][e >> 1], val[2][e >> 1], sel);
                    acc[e] = __builtin_amdgcn_mfma_f32_16x16x16f16(pa, __builtin_bit_cast(half4_t, b), acc[e], 0, 0, 0);
                    acc[e] = __builtin_amdgcn_mfma_f32_16x16x16f16(pb, __builtin_bit_cast(half4_t, b), acc[e], 0, 0, 0);
                }
                if (i + 1 < range_.y) fill();
            }
            sum += lane_xor_f32<16>(sum);
            sum += lane_xor_f32<32>(sum);
            float* const part_ = reinterpret_cast<float*>(area + attn_part_at(D)) + wave * attn_part_floats(D, G);
            if (tg == 0) {
                part_[c] = m;
                part_[16 + c] = sum;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (4 * tg + r < G)
#pragma unroll
                    for (int e = 0; e < E; e += 4)
                        *reinterpret_cast<float4_t*>(part_ + 32 + (4 * tg + r) * D + E * c + e) =
                            float4_t{acc[e][r], acc[e + 1][r], acc[e + 2][r], acc[e + 3][r]};
            block_barrier();  // the waves' parts are there
            fill();
        }
    }

    __device__ __forceinline__ void run() {
        if (alone) {
            end = range(arguments(), rank, kPhases - 1).y;
            fill();
        }
#pragma unroll 1
        for (int l = 0; l < layers; ++l)
#pragma unroll 1
            for (int ph = 0; ph < kPhases; ++ph)
#pragma unroll 1
                for (int v = rank; v < parts; v += n) {
                    if (ph == kPhaseAttn) attend(v, l);
                    else project(ph == kPhaseQkv ? kQkv : ph - 1, v, l);
                }
    }
};

// ---------------------------------------------------------------------------- front waves
template <int D>
struct Front {
    char* const lds;
    const int rank, n, tid, lane, wave;  // tid 0 .. 255
    const int parts, layers;
    const Words words;
    int budget;
    unsigned meets = 0;
    const int pieces;  // of the context
    const bool many;   // more partials than the o projection's workgroups read themselves
    const int pos;
    const int64_t slot;
    // this lane's tile and weight row in every epilogue
    const int et, en;

    __device__ __forceinline__ Front(Plan& p, char* l, int r, int n_, int t)
        : lds(l), rank(r), n(n_), tid(t), lane(t & 63), wave(uniform(t >> 6)), parts(p.parts), layers(p.layers),
          words(p.region, p.bytes), budget(p.polls), pieces(uniform_load(&info(p)->pieces)),
          many(uniform_load(&info(p)->merged)), pos(uniform_load(p.positions)),
          slot(uniform_load(p.slot_mapping)), et(t >> 4), en(t & 15) {}
    static __device__ __forceinline__ const StepInfo* info(Plan& p) {
        return reinterpret_cast<const StepInfo*>(p.region + p.at_step);
    }

    // barrier of the front waves
    __device__ __forceinline__ void meet() {
        meets += kFrontWaves;
        unsigned* const count = reinterpret_cast<unsigned*>(lds + arguments().lds_misc);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (lane == 0) __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        while (__hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < meets) {
        }
        asm volatile("" ::: "memory");
    }
    // once more around a poll?
    __device__ __forceinline__ bool again(bool ok) {
        asm volatile("" ::: "memory");
        if (__all(ok)) return false;
        return --budget > 0;
    }
    // Where a wave has words that it waited for, on the way to what follows from them (in the polls themselves it cost a
    // step 1 to 2 %, here at most 0.7 %).
    __device__ __forceinline__ void arrived() {
        if (__builtin_expect(budget > 0, 1)) return;
        if (lane == 0) {
            __hip_atomic_store(gave_up_word(), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *whole() = NAN;
        }
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // known before anything that follows is
    }
    // 1, or NaN from where a wave of this workgroup has gone on without words that it waited for: a factor of all
    // that the workgroup publishes
    __device__ __forceinline__ float* whole() const {
        return reinterpret_cast<float*>(lds + arguments().lds_misc) + 3;
    }
    static __device__ __forceinline__ unsigned* gave_up_word() {
        return reinterpret_cast<unsigned*>(arguments().region) + 2;
    }
    // ... a wave of any workgroup
    static __device__ __forceinline__ bool any_gave_up() {
        return __hip_atomic_load(gave_up_word(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    }

    // ---- scales and zeros of a part's tiles: [tile][scales, zeros][eight rows][16 G bytes] straight into LDS
    __device__ __forceinline__ void fetch_scales(int which, int l, int v) {
        Plan& p = arguments();
        const Shape s = proj_shape(p, which, D);
        const int G = s.k >> 7, total = tiles_of(v, parts, s.tiles) * 4 * G;
        if (total == 0) return;
        const unsigned inv = p.group_inv[which];
        const __half* const sc = uniform_load(&p.table[l].scale[which]);
        const __half* const ze = uniform_load(&p.table[l].zero[which]);
        const unsigned dst = (unsigned)((which & 1) ? p.lds_scale[1] : p.lds_scale[0]);
        const int apart = tile_apart<D>(p, which);
#pragma unroll 1
        for (int i0 = wave * 64; i0 < total; i0 += kFrontThreads) {
            const int i = min(i0 + lane, total - 1);
            const int run = (int)(((unsigned)i * inv) >> 20), pc = i - run * G;
            const int row = tile_first<D>(which, v + (run >> 2) * parts) + ((run & 1) ? apart : 0);
            const char* src = reinterpret_cast<const char*>((run & 2) ? ze : sc) + (size_t)row * G * 2 + pc * 16;
            const unsigned to = dst + (unsigned)i0 * 16u;
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                         :
                         : "v"(src), "s"(to)
                         : "memory");
        }
    }

    // ---- the operand: the row normed
    __device__ __forceinline__ void norm_row(int which, int l) {
        Plan& p = arguments();
        const int hidden = p.hidden, chunks = hidden >> 3;
        const unsigned at_h = p.at_h;
        const float eps = p.eps;
        const float* const gain = which == kQkv ? uniform_load(&p.table[l].norm1) : uniform_load(&p.table[l].norm2);
        float4_t w[kNormChunks][2];
        float v[kNormChunks][8];
#pragma unroll
        for (int i = 0; i < kNormChunks; ++i) {
            if (i * kFrontThreads >= chunks) continue;
            const float* const g = gain + 8 * min(i * kFrontThreads + tid, chunks - 1);
            w[i][0] = *reinterpret_cast<const float4_t*>(g);
            w[i][1] = *reinterpret_cast<const float4_t*>(g + 4);
        }
        if (which == kQkv && l == 0) {
            const float* const h = p.h;
#pragma unroll
            for (int i = 0; i < kNormChunks; ++i) {
                if (i * kFrontThreads >= chunks) continue;
                const float* src = h + 8 * min(i * kFrontThreads + tid, chunks - 1);
                const float4_t a = *reinterpret_cast<const float4_t*>(src);
                const float4_t b = *reinterpret_cast<const float4_t*>(src + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[i][e] = a[e];
                    v[i][4 + e] = b[e];
                }
            }
        } else {
            const unsigned tag = which == kQkv ? 2u * l : 2u * l + 1u;
            uint4_t raw[kNormChunks][4];
            bool ok;
            do {
                ok = true;
#pragma unroll
                for (int i = 0; i < kNormChunks; ++i) {
                    if (i * kFrontThreads >= chunks) continue;
                    const unsigned at = at_h + (unsigned)min(i * kFrontThreads + tid, chunks - 1) * 64u;
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        raw[i][q] = words.get2(at + q * 16);
                }
#pragma unroll
                for (int i = 0; i < kNormChunks; ++i) {
                    if (i * kFrontThreads >= chunks) continue;
#pragma unroll
                    for (int q = 0; q < 4; ++q) ok = ok && tagged(raw[i][q], tag);
                }
            } while (again(ok));
#pragma unroll
            for (int i = 0; i < kNormChunks; ++i) {
                if (i * kFrontThreads >= chunks) continue;
#pragma unroll
                for (int e = 0; e < 8; ++e) v[i][e] = __uint_as_float(raw[i][e >> 1][2 * (e & 1)]);
            }
        }
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < kNormChunks; ++i) {
            if (i * kFrontThreads >= chunks) continue;
            float t = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) t = fmaf(v[i][e], v[i][e], t);
            s += i * kFrontThreads + tid < chunks ? t : 0.0f;
        }
        s = wave_sum(s);
        float* const ssq = reinterpret_cast<float*>(lds + p.lds_ssq);
        if (lane == 0) ssq[wave] = s;
        meet();
        const float4_t all = *reinterpret_cast<const float4_t*>(ssq);
        const float inv = 1.0f / sqrtf((all[0] + all[1] + all[2] + all[3]) / (float)hidden + eps);
#pragma unroll
        for (int i = 0; i < kNormChunks; ++i) {
            if (i * kFrontThreads >= chunks) continue;
            uint4_t o;  // pair order: (x0, x4) (x1, x5) (x2, x6) (x3, x7)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                o[e] = pack_bf16(v[i][e] * inv * w[i][0][e], v[i][4 + e] * inv * w[i][1][e]);
            put_operand(o, i * kFrontThreads + tid, chunks);
        }
    }
    // chunk c (eight columns in pair order)
    __device__ __forceinline__ void put_operand(const uint4_t& o, int c, int chunks) {
        if (c < chunks) *reinterpret_cast<uint4_t*>(lds + arguments().lds_x + c * 16) = o;
    }

    // ---- the operand: bf16 values that are there as words of two
    __device__ __forceinline__ void take_row(unsigned at, int k, unsigned tag) {
        constexpr int R = 6;  // chunks per thread and round
        const int chunks = k >> 3;
#pragma unroll 1
        for (int c0 = 0; c0 < chunks; c0 += R * kFrontThreads) {
            uint4_t raw[R][2];
            bool ok;
            do {
                ok = true;
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    if (c0 + i * kFrontThreads >= chunks) continue;
                    const unsigned ch = (unsigned)min(c0 + i * kFrontThreads + tid, chunks - 1);
#pragma unroll
                    for (int q = 0; q < 2; ++q)
                        raw[i][q] = words.get2(at + ch * 32u + q * 16u);
                }
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    if (c0 + i * kFrontThreads >= chunks) continue;
                    ok = ok && tagged(raw[i][0], tag) && tagged(raw[i][1], tag);
                }
            } while (again(ok));
#pragma unroll
            for (int i = 0; i < R; ++i) {
                if (c0 + i * kFrontThreads >= chunks) continue;
                const uint4_t d = {raw[i][0][0], raw[i][0][2], raw[i][1][0], raw[i][1][2]};
                put_operand(pair_order(d), c0 + i * kFrontThreads + tid, chunks);
            }
        }
    }

    // ---- the operand of the o projection from the partials themselves (few of them)
    __device__ __forceinline__ unsigned part_at(Plan& p, int unit, int head) const {
        return p.at_part + (unsigned)((unit * p.group + head) * (D + 2)) * 8u;
    }
    __device__ __forceinline__ void take_partials(unsigned tag) {
        Plan& p = arguments();
        constexpr int R = 4;  // pieces asked for together
        const int chunks = p.hq * (D / 8);
        if (pieces == 0) {
            // no key is seen: the projection before has no reader, but the chain has to pass through it
            const int count = (p.hq + 2 * p.hkv) * (D / 4);
#pragma unroll 1
            for (int i = tid; i - tid < count; i += kFrontThreads)
                while (again(tagged(words.get2(p.at_qkv + (unsigned)min(i, count - 1) * 16u), tag))) {
                }
        }
#pragma unroll 1
        for (int c0 = 0; c0 < chunks; c0 += kFrontThreads) {
            const int ch = min(c0 + tid, chunks - 1);
            const int head = ch / (D / 8), c = ch % (D / 8);
            const int kvh = head / p.group, hin = head - kvh * p.group, u0 = kvh * pieces;
            float M = kNoKey, L = 0.0f, o[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = 0.0f;
#pragma unroll 1
            for (int j0 = 0; j0 < pieces; j0 += R) {
                uint4_t ml[R], raw[R][4];
                bool ok;
                do {
                    ok = true;
#pragma unroll
                    for (int j = 0; j < R; ++j) {
                        const unsigned at = part_at(p, u0 + min(j0 + j, pieces - 1), hin);
                        ml[j] = words.get2(at);
#pragma unroll
                        for (int q = 0; q < 4; ++q) raw[j][q] = words.get2(at + 16u + c * 64u + q * 16u);
                    }
#pragma unroll
                    for (int j = 0; j < R; ++j) {
                        ok = ok && tagged(ml[j], tag);
#pragma unroll
                        for (int q = 0; q < 4; ++q) ok = ok && tagged(raw[j][q], tag);
                    }
                } while (again(ok));
#pragma unroll
                for (int j = 0; j < R; ++j) {
                    if (j0 + j >= pieces) continue;
                    const float mj = __uint_as_float(ml[j][0]), lj = __uint_as_float(ml[j][2]);
                    const float mx = fmaxf(M, mj);
                    const float a = fast_exp2(M - mx), b = fast_exp2(mj - mx);
                    M = mx;
                    L = L * a + lj * b;
#pragma unroll
                    for (int e = 0; e < 8; ++e) o[e] = o[e] * a + __uint_as_float(raw[j][e >> 1][2 * (e & 1)]) * b;
                }
            }
            const float inv = pieces ? 1.0f / L : 0.0f;
            uint4_t x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = pack_bf16(o[e] * inv, o[4 + e] * inv);
            put_operand(x, c0 + tid, chunks);
        }
    }
    // ... or, with more of them, one head per workgroup, published as bf16 pairs
    // (apart: a barrier lies between the q/k/v epilogue and here)
    __device__ __forceinline__ void merge_pieces(unsigned tag, bool apart) {
        Plan& p = arguments();
        constexpr int TEAMS = kFrontThreads / D;
        const int team = tid / D, c = tid % D;
        float* const area = reinterpret_cast<float*>(lds + p.lds_red);  // [team]{M, L, o[D]}
        // The area lies over the parts of the q/k/v product, which a wave with a tile of it may still be adding up:
        // a workgroup without a piece of the context comes here without a barrier, and the words it waits for
        // are those of another KV head.
        if (!apart && n - 1 - rank < p.hq) meet();
#pragma unroll 1
        for (int head = n - 1 - rank; head < p.hq; head += n) {
            const int kvh = head / p.group, hin = head - kvh * p.group, u0 = kvh * pieces;
            float M = kNoKey, L = 0.0f, o = 0.0f;
            constexpr int R = 8;
#pragma unroll 1
            for (int j0 = 0; j0 < pieces; j0 += R * TEAMS) {
                uint4_t ml[R];
                uint2_t raw[R];
                bool ok;
                do {
                    ok = true;
#pragma unroll
                    for (int j = 0; j < R; ++j) {
                        const unsigned at = part_at(p, u0 + min(j0 + j * TEAMS + team, pieces - 1), hin);
                        ml[j] = words.get2(at);
                        raw[j] = words.get(at + 16u + c * 8u);
                    }
#pragma unroll
                    for (int j = 0; j < R; ++j) ok = ok && tagged(ml[j], tag) && raw[j][1] == tag;
                } while (again(ok));
#pragma unroll
                for (int j = 0; j < R; ++j) {
                    if (j0 + j * TEAMS + team >= pieces) continue;
                    const float mj = __uint_as_float(ml[j][0]), lj = __uint_as_float(ml[j][2]);
                    const float mx = fmaxf(M, mj);
                    const float a = fast_exp2(M - mx), b = fast_exp2(mj - mx);
                    M = mx;
                    L = L * a + lj * b;
                    o = o * a + __uint_as_float(raw[j][0]) * b;
                }
            }
            area[team * (D + 2)] = M;
            area[team * (D + 2) + 1] = L;
            area[team * (D + 2) + 2 + c] = o;
            arrived();
            meet();
            if (tid < D / 2) {
                float mx = -INFINITY, den = 0.0f, o0 = 0.0f, o1 = 0.0f;
#pragma unroll
                for (int t = 0; t < TEAMS; ++t) mx = fmaxf(mx, area[t * (D + 2)]);
#pragma unroll
                for (int t = 0; t < TEAMS; ++t) {
                    const float a = fast_exp2(area[t * (D + 2)] - mx);
                    den += area[t * (D + 2) + 1] * a;
                    o0 += area[t * (D + 2) + 2 + 2 * tid] * a;
                    o1 += area[t * (D + 2) + 3 + 2 * tid] * a;
                }
                const float inv = *whole() / den;
                words.put(p.at_x + (unsigned)(head * (D / 2) + tid) * 8u, pack_bf16(o0 * inv, o1 * inv), tag);
            }
            meet();
        }
    }

    // ---- attention: queries and the token's K and V row into LDS, the waves' parts out of it
    // returns whether the workgroup had a piece
    __device__ __forceinline__ bool attend(int l) {
        Plan& p = arguments();
        const unsigned tag = l + 1;
        const int G = p.group;
        bool any = false;
#pragma unroll 1
        for (int v = rank; v < parts; v += n) {
            const Piece* const pp = reinterpret_cast<const Piece*>(p.region + p.at_pieces) + v;
            if (uniform_load(&pp->count) == 0) continue;
            any = true;
            const int unit = uniform_load(&pp->unit), kvh = uniform_load(&pp->kvh);
            char* const area = lds + p.lds_x;
            const int nq = G * (D / 4), total = nq + D / 2;  // runs of four values
#pragma unroll 1
            for (int i0 = 0; i0 < total; i0 += 2 * kFrontThreads) {
                uint4_t raw[2];
                unsigned at[2], to[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int i = min(i0 + j * kFrontThreads + tid, total - 1);
                    int e;
                    if (i < nq) {
                        const int head = i / (D / 4), c = i % (D / 4);
                        e = (kvh * G + head) * D + 4 * c;
                        to[j] = (unsigned)(head * attn_q_stride(D) + c * 8);
                    } else {
                        const int c = i - nq;  // K, then V
                        e = (p.hq + kvh + (c >= D / 4 ? p.hkv : 0)) * D + 4 * (c % (D / 4));
                        to[j] = (unsigned)(attn_new_at(D) + c * 8);
                    }
                    at[j] = p.at_qkv + (unsigned)e * 4u;
                }
                bool ok;
                do {
                    raw[0] = words.get2(at[0]);
                    raw[1] = words.get2(at[1]);
                    ok = tagged(raw[0], tag) && tagged(raw[1], tag);
                } while (again(ok));
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    *reinterpret_cast<uint2_t*>(area + to[j]) = uint2_t{raw[j][0], raw[j][2]};
            }
            arrived();
            block_barrier();
            block_barrier();  // the waves' parts are there
            const float* const part = reinterpret_cast<const float*>(area + attn_part_at(D));
            const int step = attn_part_floats(D, G);
#pragma unroll 1
            for (int i = tid; i < G * (D / 2); i += kFrontThreads) {
                const int head = i / (D / 2), c = 2 * (i % (D / 2));
                typedef float float2_t __attribute__((ext_vector_type(2)));
                float m[kStreamWaves], sum[kStreamWaves];
                float2_t v[kStreamWaves];
#pragma unroll
                for (int w = 0; w < kStreamWaves; ++w) {
                    m[w] = part[w * step + head];
                    sum[w] = part[w * step + 16 + head];
                    v[w] = *reinterpret_cast<const float2_t*>(part + w * step + 32 + 2 * i);
                }
                float M = m[0];
#pragma unroll
                for (int w = 1; w < kStreamWaves; ++w) M = fmaxf(M, m[w]);
                const float safe = M == -INFINITY ? 0.0f : M;
                float L = 0.0f, o0 = 0.0f, o1 = 0.0f;
#pragma unroll
                for (int w = 0; w < kStreamWaves; ++w) {
                    // (a wave without a tile: maximum -inf, sums zero)
                    const float b = fast_exp2(m[w] - safe);
                    L = fmaf(sum[w], b, L);
                    o0 = fmaf(v[w][0], b, o0);
                    o1 = fmaf(v[w][1], b, o1);
                }
                const unsigned at = part_at(p, unit, head);
                words.put(at + 16u + c * 8u, __float_as_uint(o0), tag);
                words.put(at + 24u + c * 8u, __float_as_uint(o1), tag);
                if (c == 0) {
                    words.put(at, __float_as_uint(M), tag);
                    words.put(at + 8u, __float_as_uint(L * *whole()), tag);
                }
            }
            meet();  // the area's readers are through
        }
        return any;
    }

    // ---- a projection: its operand, then the epilogue, a weight row of a tile per lane
    __device__ __forceinline__ void project(int which, int l) {
        Plan& p = arguments();
        const Shape s = proj_shape(p, which, D);
        const bool alone = n == parts;  // one part: the next projection's scales are asked for ahead
        bool first = true;
#pragma unroll 1
        for (int v = rank; v < parts; v += n) {
            const int count = tiles_of(v, parts, s.tiles);
            if (count == 0) break;  // (so have the parts behind it)
            if (!alone) fetch_scales(which, l, v);
            // what this lane's epilogue needs from memory (the residual that an owner adds to is its own store of
            // the projection before)
            const int t = v + min(et, count - 1) * parts;
            const int head = t / (D / 16), at = 8 * (t - head * (D / 16)) + (en & 7);
            float a = 0.0f, b = 0.0f, bias = 0.0f;  // residual; or cos, sin, bias
            if (which == kQkv) {
                const int q = pos < 0 ? 0 : (pos >= p.max_pos ? p.max_pos - 1 : pos);
                const float* const bp = uniform_load(&p.table[l].bias);
                a = p.cos_t[(int64_t)q * (D / 2) + at];
                b = p.sin_t[(int64_t)q * (D / 2) + at];
                if (bp) bias = bp[head * D + at + (en < 8 ? 0 : D / 2)];
            } else if (which != kGateUp) {
                a = p.h[16 * t + en];
            }
            if (first) {  // (the parts of a workgroup have the same operand)
                if (which == kQkv || which == kGateUp) norm_row(which, l);
                else if (which == kO && !many) take_partials(l + 1);
                else take_row(which == kO ? p.at_x : p.at_act, s.k, l + 1);
            }
            first = false;
            arrived();
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the scales
            block_barrier();
            if (alone) fetch_next_scales(which, l);
            block_barrier();  // the streaming waves' parts are there
            if (wave * 4 >= count) continue;
            const float* const red = reinterpret_cast<const float*>(lds + p.lds_red) + et * (kStreamWaves * 16) + en;
            float sum = red[0];
#pragma unroll
            for (int w = 1; w < kStreamWaves; ++w) sum += red[w * 16];
            sum *= *whole();
            const bool ok = et < count;
            if (which == kO || which == kDown) {
                if (ok) {
                    const float res = a + sum;
                    words.put(p.at_h + (unsigned)(16 * t + en) * 8u, __float_as_uint(res),
                              which == kO ? 2 * l + 1 : 2 * l + 2);
                    p.h[16 * t + en] = res;
                }
            } else if (which == kGateUp) {
                const float up = lane_xor_f32<8>(sum);
                const float act = sum / (1.0f + expf(-sum)) * up;
                const float next = lane_xor_f32<1>(act);
                if (ok && en < 8 && (en & 1) == 0)
                    words.put(p.at_act + (unsigned)(4 * t + (en >> 1)) * 8u, pack_bf16(act, next), l + 1);
            } else {
                sum += bias;
                const float other = lane_xor_f32<8>(sum);
                float res = sum;
                if (head < p.hq + p.hkv) {
                    // the two halves of rope_rotate (step_ops.hip), rounded alike
                    res = en < 8 ? fmaf(sum, a, -(other * b)) : fmaf(other, b, sum * a);
                    asm volatile("" : "+v"(res));
                }
                const __half r16 = __float2half_rn(res);
                const unsigned lo = __half_as_ushort(r16), hi = (unsigned)lane_xor_i32<1>((int)lo);
                const int col = head * D + at + (en < 8 ? 0 : D / 2);
                if (ok && (en & 1) == 0) words.put(p.at_qkv + (unsigned)col * 4u, lo | (hi << 16), l + 1);
                if (ok && head >= p.hq && slot >= 0 && !(res != res && any_gave_up())) {
                    const bool is_k = head < p.hq + p.hkv;
                    __half* const kp = uniform_load(&p.table[l].k_pool);
                    __half* const vp = uniform_load(&p.table[l].v_pool);
                    (is_k ? kp : vp)[slot * p.hkv * D + col - (is_k ? p.hq : p.hq + p.hkv) * D] = r16;
                }
            }
        }
        if (first && alone) fetch_next_scales(which, l);
    }
    __device__ __forceinline__ void fetch_next_scales(int which, int l) {
        if (which == kDown && l + 1 == layers) return;
        fetch_scales((which + 1) & 3, which == kDown ? l + 1 : l, rank);
    }
    __device__ __forceinline__ void run() {
        if (n == parts) fetch_scales(kQkv, 0, rank);
#pragma unroll 1
        for (int l = 0; l < layers; ++l)
#pragma unroll 1
            for (int which = kQkv; which <= kDown; ++which) {
                project(which, l);
                if (which == kQkv) {
                    const bool any = attend(l);
                    if (many) merge_pieces(l + 1, any);
                }
            }
    }
};

template <int D>
__global__ __launch_bounds__(kThreads) void decode_resident_kernel(const ResidentPlan) {
    Plan& p = arguments();
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x;
    const int wave = uniform(tid >> 6);
    unsigned* const misc = reinterpret_cast<unsigned*>(lds + p.lds_misc);  // {front barrier, rank, n, Front::whole}
    if (tid == 0) {
        unsigned* const ctl = reinterpret_cast<unsigned*>(p.region);  // {tickets, closed, a wave gave up}
        const unsigned ticket = __hip_atomic_fetch_add(ctl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        unsigned n = 0;
        if (const unsigned all = p.all; ticket == all - 1) {
            __hip_atomic_compare_exchange_strong(ctl + 1, &n, all, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
            if (n == 0) n = all;
        }
        const unsigned long long start = __builtin_readsteadycounter();  // 100 MHz
        while (n == 0) {
            n = __hip_atomic_load(ctl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (n == 0 && __builtin_readsteadycounter() - start > kCloseAfter) {
                const unsigned now = __hip_atomic_load(ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_compare_exchange_strong(ctl + 1, &n, now, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
                if (n == 0) n = now;
            }
        }
        misc[0] = 0;
        misc[1] = ticket;
        misc[2] = n;
        misc[3] = __float_as_uint(1.0f);
    }
    __syncthreads();
    const int rank = uniform((int)misc[1]), n = uniform((int)misc[2]);
    if (rank >= n) return;
    if (wave < kStreamWaves) Stream<D>(p, lds, rank, n, wave, tid & 63).run();
    else Front<D>(p, lds, rank, n, tid - 64 * kStreamWaves).run();
}

// Before the step: its words without a tag and its tickets at zero; the layers' operands as a table; and
// the lists of the parts, one workgroup per part, one wave per streaming wave.
template <int D>
__global__ __launch_bounds__(64 * kStreamWaves) void decode_resident_init_kernel(const ResidentPlan p,
                                                                                 ResidentLayer* table, int first,
                                                                                 int count,
                                                                                 const ResidentLayers layers) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, v = blockIdx.x;
    if (v == 0 && tid < count) table[first + tid] = layers.l[tid];
    if (first) return;
    {
        uint4_t* const words = reinterpret_cast<uint4_t*>(p.region + p.at_h);
        for (unsigned i = v * blockDim.x + tid; i < (p.bytes - p.at_h) / 16; i += gridDim.x * blockDim.x)
            words[i] = uint4_t{0, 0, 0, 0};
    }
    // the context in pieces: a tile per streaming wave, as long as there are parts
    // (a list has room for the keys that the block table can hold, and the table no entries past them)
    const int ctx = p.cu[1] - p.cu[0] == 1 ? min(p.ctx[0], p.max_blocks * p.block_size) : 0;
    Piece piece{0, 0, 0, 0};
    int pieces = 0, t0 = 0, t1 = 0;
    if (ctx > 0) {
        const int tiles = (ctx + kTileKeys - 1) / kTileKeys;
        const int want = min(p.parts / p.hkv, (tiles + kStreamWaves - 1) / kStreamWaves);
        const int per = (tiles + want - 1) / want;
        pieces = (tiles + per - 1) / per;
        const int unit = p.parts - 1 - v;  // (the parts with two q/k/v tiles are the first ones)
        if (unit < p.hkv * pieces) {
            piece = Piece{pieces, unit, unit / pieces, 0};
            t0 = (unit - piece.kvh * pieces) * per;
            t1 = min(t0 + per, tiles);
        }
    }
    if (tid == 0) {
        reinterpret_cast<Piece*>(p.region + p.at_pieces)[v] = piece;
        if (v == 0) {
            unsigned* const ctl = reinterpret_cast<unsigned*>(p.region);
            ctl[0] = ctl[1] = ctl[2] = 0;
            *reinterpret_cast<StepInfo*>(p.region + p.at_step) =
                StepInfo{pieces, pieces && (p.hq * D > kDirectColumns || pieces * p.hq * (D + 2) > kDirectWords)};
        }
    }
    uint4_t* const list = reinterpret_cast<uint4_t*>(p.region + p.at_lists) + ((size_t)v * kStreamWaves + wave) * p.list;
    int at = 0, starts[kPhases + 1];
#pragma unroll
    for (int ph = 0; ph < kPhases; ++ph) {
        starts[ph] = at;
        if (ph == kPhaseAttn) {
            const int tiles = piece.count && t0 + wave < t1 ? (t1 - t0 - wave + kStreamWaves - 1) / kStreamWaves : 0;
            for (int i = lane; i < tiles; i += 64) {
                const int tok = (t0 + wave + i * kStreamWaves) * kTileKeys, bi = tok / p.block_size;
                const int64_t row0 = (int64_t)p.block_tables[bi] * p.block_size + (tok - bi * p.block_size);
                const int64_t slot = p.slot_mapping[0];
                const bool here = slot >= 0 && slot >= row0 && slot < row0 + kTileKeys;
                list[at + i] = uint4_t{(unsigned)(row0 * p.hkv + piece.kvh),
                                       kKvTile | ((unsigned)min(ctx - tok, kTileKeys) << 8),
                                       here ? (unsigned)(slot - row0) + 1u : 0u, 0};
            }
            at += tiles;
            continue;
        }
        const int which = ph == kPhaseQkv ? kQkv : ph - 1;
        const Shape s = proj_shape(p, which, D);
        const int2 share = rows_share(s.k >> 7, kStreamWaves, wave);
        // batches of a tile: four groups each, then two, then one
        const int fours = share.y >> 2, twos = (share.y >> 1) & 1, ones = share.y & 1;
        const int each = max(fours + twos + ones, 1), batches = tiles_of(v, p.parts, s.tiles) * each;
        for (int i = lane; i < batches; i += 64) {
            const int t = i / each, b = i - t * each;
            const int c = b < fours ? 4 : (b < fours + twos ? 2 : ones);
            const int g = share.x + 4 * min(b, fours) + 2 * max(b - fours, 0);  // (the one behind no two: b = fours)
            list[at + i] = uint4_t{(unsigned)tile_first<D>(which, v + t * p.parts) * (unsigned)(s.k >> 1) + g * 64u,
                                   (unsigned)c | (b == each - 1 ? 8u : 0u) | ((unsigned)t << 4) | ((unsigned)g << 8) |
                                       ((unsigned)which << 16),
                                   (unsigned)(s.k >> 1) | ((unsigned)(tile_apart<D>(p, which) - 8) << 16), 0};
        }
        at += batches;
    }
    starts[kPhases] = at;
    if (lane == 0) {
        int* const dst = reinterpret_cast<int*>(p.region + p.at_starts) + ((size_t)v * kStreamWaves + wave) * 8;
#pragma unroll
        for (int i = 0; i <= kPhases; ++i) dst[i] = starts[i];
    }
}

size_t pad256(size_t v) { return (v + 255) & ~(size_t)255; }

// Offsets and sizes; false: not a geometry for this launch.
bool resident_plan(const logismos_decode_config_t& c, ResidentPlan* p) {
    const int d = c.head_dim;
    if (c.kv_turbo3 || (d != 64 && d != 128) || c.hidden > 8 * kNormChunks * kFrontThreads || c.block_size % 16 != 0)
        return false;
    const int group = c.num_q_heads / c.num_kv_heads;
    const int64_t qd = (int64_t)c.num_q_heads * d, width = qd + 2 * (int64_t)c.num_kv_heads * d;
    // a batch's first group has eight bits; words and a projection's bytes are found by 32-bit offsets, scales
    // by a 20-bit reciprocal of their groups
    if (group > 16 || c.intermediate > 16384 || qd > 16384 || width > 32768) return false;
    const int cus = device_cu_count(), parts = cus < kMaxParts ? cus : kMaxParts;
    if (c.num_kv_heads > parts) return false;
    *p = ResidentPlan{};
    p->layers = c.num_layers;
    p->hidden = c.hidden;
    p->inter = c.intermediate;
    p->hq = c.num_q_heads;
    p->hkv = c.num_kv_heads;
    p->group = group;
    p->block_size = c.block_size;
    p->max_blocks = c.max_blocks_per_seq;
    p->max_pos = c.max_pos;
    p->eps = c.rms_eps;
    p->scale_log2e = 1.4426950408889634f / sqrtf((float)d);
    p->parts = parts;
    const int tiles[4] = {(int)(width / 16), c.hidden / 16, c.intermediate / 8, c.hidden / 16};
    const int ks[4] = {c.hidden, (int)qd, c.hidden, c.intermediate};
    // a wave's list: the batches of its share of K for every tile, and its K/V tiles
    int list = 0, held = 1, scale[2] = {0, 0}, x = 0;
    for (int i = 0; i < 4; ++i) {
        const int per = (tiles[i] + parts - 1) / parts, groups = ks[i] / 128;
        if (per > kMaxTilesHeld) return false;
        const int share = (groups + kStreamWaves - 1) / kStreamWaves;
        list += per * ((share >> 2) + 2);
        if (per > held) held = per;
        // requests of whole waves of 1 KiB
        const int bytes = (per * 64 * groups + 1023) / 1024 * 1024;
        if (bytes > scale[i & 1]) scale[i & 1] = bytes;
        const int op = 2 * ks[i];
        if (op > x) x = op;
        p->group_inv[i] = ((1u << 20) + groups - 1) / groups;
    }
    {
        const int64_t longest = ((int64_t)c.max_blocks_per_seq * c.block_size + kTileKeys - 1) / kTileKeys;
        const int most = parts / c.num_kv_heads;
        const int64_t per = (longest + most - 1) / most;
        const int64_t of_wave = ((per > kStreamWaves ? per : kStreamWaves) + kStreamWaves - 1) / kStreamWaves;
        if (list + of_wave > kMaxList) return false;
        list += (int)of_wave;
    }
    p->list = list;
    size_t at = 256;
    auto take = [&](size_t bytes) {
        const size_t o = at;
        at += pad256(bytes);
        return (unsigned)o;
    };
    p->at_step = take(sizeof(StepInfo));
    p->at_pieces = take(sizeof(Piece) * parts);
    p->at_starts = take((size_t)parts * kStreamWaves * 8 * 4);
    p->at_lists = take((size_t)parts * kStreamWaves * list * 16);
    p->at_h = take((size_t)c.hidden * 8);
    p->at_qkv = take((size_t)width * 4);
    p->at_x = take((size_t)qd * 4);
    p->at_act = take((size_t)c.intermediate * 4);
    p->at_part = take((size_t)parts * group * (d + 2) * 8);
    p->bytes = (unsigned)at;
    // LDS, from its end; the rings take the rest
    const int attn = attn_part_at(d) + kStreamWaves * attn_part_floats(d, group) * 4;
    if (attn > x) x = attn;
    // (the merge of pieces lies where the parts of a product do)
    const int merge = kFrontThreads / d * (d + 2) * 4, parts_of = held * kStreamWaves * 64;
    const int red = merge > parts_of ? merge : parts_of;
    int rest = kResLds;
    auto lds = [&](int bytes) {
        rest -= (bytes + 15) / 16 * 16;
        return rest;
    };
    p->lds_misc = lds(16);
    p->lds_ssq = lds(kFrontWaves * 4);
    p->lds_red = lds(red);
    p->lds_x = lds(x);
    p->lds_scale[0] = lds(scale[0]);
    p->lds_scale[1] = lds(scale[1]);
    const int slots = rest / (kStreamWaves * kSlot);
    p->slots = slots < kMaxSlots ? slots : kMaxSlots;
    return rest > 0 && slots >= 2;
}

// the layer table, in front of the region
size_t table_bytes(const logismos_decode_config_t& c) { return pad256((size_t)c.num_layers * sizeof(ResidentLayer)); }

template <int D>
hipError_t resident_launch(const ResidentPlan& p, const logismos_decode_config_t& c,
                           const logismos_decode_layer_t* layers, ResidentLayer* table, int workgroups, hipStream_t st) {
    const auto kernel = decode_resident_kernel<D>;
    static const hipError_t opt_in = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kResLds);
    if (opt_in != hipSuccess) return opt_in;
    for (int l0 = 0; l0 < c.num_layers; l0 += kLayersPerInit) {
        ResidentLayers arg{};
        const int count = c.num_layers - l0 < kLayersPerInit ? c.num_layers - l0 : kLayersPerInit;
        for (int i = 0; i < count; ++i) {
            const logismos_decode_layer_t& L = layers[l0 + i];
            ResidentLayer& r = arg.l[i];
            const logismos_q4_weight_t* W[4] = {&L.qkv, &L.o, &L.gate_up, &L.down};
            for (int j = 0; j < 4; ++j) {
                r.qw[j] = static_cast<const uint8_t*>(W[j]->qw);
                r.scale[j] = static_cast<const __half*>(W[j]->scale);
                r.zero[j] = static_cast<const __half*>(W[j]->zero);
            }
            r.norm1 = static_cast<const float*>(L.norm1_w_f32);
            r.norm2 = static_cast<const float*>(L.norm2_w_f32);
            r.bias = static_cast<const float*>(L.qkv_bias_f32);
            r.k_pool = static_cast<__half*>(L.k_pool_f16);
            r.v_pool = static_cast<__half*>(L.v_pool_f16);
        }
        decode_resident_init_kernel<D><<<dim3(l0 ? 1 : (unsigned)p.parts), dim3(64 * kStreamWaves), 0, st>>>(
            p, table, l0, count, arg);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    }
    kernel<<<dim3((unsigned)workgroups), dim3(kThreads), kResLds, st>>>(p);
    return hipGetLastError();
}

}  // namespace

size_t decode_resident_bytes(const logismos_decode_config_t& c) {
    ResidentPlan p;
    return resident_plan(c, &p) ? p.bytes + table_bytes(c) : 0;
}

// Few layers: the lists, the words' zeros and the start of the kernel are 10 to 15 us that the layers have to earn.  us at
// 500 keys, launches / here, 2 | 4 | 8 layers: width 512 44 / 42 | 91 / 72 | 179 / 129; 896 51 / 52 | 103 / 92 | 206 / 167; 1536
// (MLP of 8960) 59 / 63 | 117 / 112 | 229 / 213.  Wider, where a layer's weights take up more of it, 8 | 16 | 28 layers: 2048
// (MLP of 11008, two KV heads) 254 / 276 | 520 / 543 | 934 / 940; 3072 (four KV heads) 329 / 339 | 681 / 667; 3584 (MLP of
// 9472) 315 / 340 | 660 / 668 | 1155 / 1156; but 2048 (MLP of 6144) 257 / 190 and 4096 394 / 326 at 8.  40 geometries at 500 and
// 4000 keys and 4, 8, 16 or 28 layers past the lines below take 0.60 to 1.05 of the launches' time, 0.83 on average.
// More than 1 % longer: the first of these at 500 keys (at 4000 552 / 531 and 997 / 921), and 3584 with 28 KV heads at 4000
// keys (803 / 826, at 500 714 / 687).
//
// Long contexts: this kernel's attention reads K and V at 5.7 TB/s, the launches' at 7 (with one or two KV heads less), so
// that from some size on their stream outweighs the chain of launches.  us of eight layers with a full table, launches /
// here, at 256 | 384 | 512 MiB of K and V per layer: 32 KV heads of 128 762 / 740 | 916 / 926 | 1085 / 1117; 8 heads
// 795 / 737 | 963 / 935 | 1117 / 1133; 4 heads 711 / 661 | 887 / 860 | 1059 / 1058; 16 heads of 64 790 / 721 | 960 / 920 |
// 1112 / 1110; at 512 and 768 MiB 2 heads of 128 1184 / 1049 and 1520 / 1441, of 64 1017 / 997 and 1365 / 1383.  The
// host knows what the table can hold, not what it holds: the lines lie where a full one is still no slower.
bool decode_resident_pays(const logismos_decode_config_t& c) {
    const int64_t kv_bytes = 4 * (int64_t)c.num_kv_heads * c.head_dim * c.block_size * c.max_blocks_per_seq;
    return c.num_layers >= (c.hidden <= 1536 ? 4 : 16) && kv_bytes <= (c.num_kv_heads <= 2 ? (int64_t)512 : 320) << 20;
}

bool decode_resident_applies(const logismos_decode_config_t& c, const logismos_decode_layer_t* layers,
                             const logismos_decode_batch_t& b, int t) {
    ResidentPlan p;
    if (t != 1 || !resident_plan(c, &p)) return false;
    uintptr_t at = reinterpret_cast<uintptr_t>(b.hidden_f32);
    for (int l = 0; l < c.num_layers; ++l) {
        const logismos_decode_layer_t& L = layers[l];
        at |= reinterpret_cast<uintptr_t>(L.norm1_w_f32) | reinterpret_cast<uintptr_t>(L.norm2_w_f32) |
              reinterpret_cast<uintptr_t>(L.k_pool_f16) | reinterpret_cast<uintptr_t>(L.v_pool_f16);
        for (const logismos_q4_weight_t* W : {&L.qkv, &L.o, &L.gate_up, &L.down})
            at |= reinterpret_cast<uintptr_t>(W->scale) | reinterpret_cast<uintptr_t>(W->zero);
    }
    return (at & 15u) == 0;
}

hipError_t decode_resident_launch(const logismos_decode_config_t& c, const logismos_decode_layer_t* layers,
                                  const logismos_decode_batch_t& b, void* region, hipStream_t st,
                                  const ResidentLimits& limits) {
    ResidentPlan p;
    if (!resident_plan(c, &p)) return hipErrorInvalidValue;
    p.polls = limits.polls > 0 ? limits.polls : kPollBudget;
    const int workgroups = limits.workgroups > 0 && limits.workgroups < p.parts ? limits.workgroups : p.parts;
    p.all = limits.tickets > 0 && limits.tickets < workgroups ? limits.tickets : workgroups;
    ResidentLayer* const table = static_cast<ResidentLayer*>(region);
    p.region = static_cast<char*>(region) + table_bytes(c);
    p.table = table;
    p.h = static_cast<float*>(b.hidden_f32);
    p.block_tables = b.block_tables;
    p.cu = b.cu_seqlens;
    p.ctx = b.context_lens;
    p.positions = b.positions;
    p.slot_mapping = b.slot_mapping;
    p.cos_t = static_cast<const float*>(b.rope_cos_f32);
    p.sin_t = static_cast<const float*>(b.rope_sin_f32);
    return c.head_dim == 64 ? resident_launch<64>(p, c, layers, table, workgroups, st)
                            : resident_launch<128>(p, c, layers, table, workgroups, st);
}

}  // namespace lg

// The launch by itself and its rule, for the tests (the header does not declare them).
extern "C" int lg_decode_resident_pays(const logismos_decode_config_t* cfg) { return lg::decode_resident_pays(*cfg); }
extern "C" size_t lg_decode_resident_bytes(const logismos_decode_config_t* cfg) {
    return lg::decode_resident_bytes(*cfg);
}
extern "C" logismos_status_t lg_decode_resident_launch(const logismos_decode_config_t* cfg,
                                                       const logismos_decode_layer_t* layers,
                                                       const logismos_decode_batch_t* batch, void* region,
                                                       const lg::ResidentLimits* limits, logismos_stream_t stream) {
    return lg::decode_resident_launch(*cfg, layers, *batch, region, static_cast<hipStream_t>(stream), *limits);
}
