// One continuous-batching decode step (one new token per live sequence) as a
// sequence of asynchronous launches on one stream: the executor the reference
// does not have yet (crates/decoders/src/lib.rs is a scaffold), written against
// the launchers of this library only.  Nothing is allocated, nothing
// synchronises; a caller may capture the whole step into a HIP graph.
#include "decode_resident.hpp"
#include "launch_common.hpp"
#include "q4_rows.hpp"

#include <math.h>

namespace {

constexpr int kChunkRows = 32;  // rows the prepared layout and the decode GEMMs hold

// A step with this many packed rows or more takes the projections on the tiled GEMM (plain bf16
// activations, fp32 products for the whole batch at once) instead of 32-row chunks.
constexpr int kTallRows = 97;

struct Workspace {
    char* xn;        // prepared activations of width hidden, one buffer per 32-row chunk (input of
                     // qkv / gate_up; they carry the normed rows from the end of one layer to
                     // the start of the next)
    char* qkv;       // f32  [Jqkv][rows][(hq+2hkv)*d]   split-K parts of a pass
    char* q;         // f16  [T][hq*d]
    char* attn_b;    // prepared activations of width hq*d (input of the o projection)
    char* attn_out;  // bf16 [T][hq*d]: attention output where it does not go straight into attn_b
    char* proj;      // f32  [max(Jo,Jdown)][rows][hidden]  (o projection, then down projection)
    char* gate_up;   // f32  [Jgu][rows][2*inter]
    char* act;       // prepared activations of width inter (input of the down projection)
    char* attn_ws;   // split-K workspace of the attention
    char* head_ws;   // per-workgroup candidates of the token selection (vocab > 0)
    // many-row steps (tall): plain buffers for all T rows
    char* t_xn;    // bf16 [T][hidden]
    char* t_qkv;   // f32  [T][(hq+2hkv)*d]
    char* t_proj;  // f32  [T][hidden]
    char* t_gu;    // f32  [T][2*inter]
    char* t_act;   // bf16 [T][inter] (or the down projection's own workspace, see carve)
    bool t_act_is_workspace;
    char* t_gemm;  // workspace of the tiled GEMM (its copy of x in unpack order + group sums)
    // tokens for the last row of every sequence (vocab > 0)
    char* norm_out;   // bf16 [T][hidden]: the normed rows when the caller takes none (chunked
                      // steps; a many-row step has t_xn free by then)
    char* last_rows;  // bf16 [num_seqs][hidden]: the normed last rows, gathered
    char* last_xn;    // prepared activations of one chunk of them
    char* resident;   // of the resident launch, where one row would take it; in every step's workspace, so
                      // that one for many rows is one for few
    bool tall;
    size_t xn_stride;
    int chunks;        // of 32 rows
    size_t total;
};

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

Workspace carve(const logismos_decode_config_t& c, int num_seqs, int t, int num_splits,
                char* base) {
    Workspace w{};
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char* p = base ? base + off : nullptr;
        off += align256(bytes);
        return p;
    };
    const size_t qd = (size_t)c.num_q_heads * c.head_dim;
    const size_t kvd = (size_t)c.num_kv_heads * c.head_dim;
    w.tall = t >= kTallRows;
    if (w.tall) {
        w.attn_ws = take(
            logismos_paged_attn_workspace_bytes(num_seqs, c.num_q_heads, c.head_dim, num_splits));
        w.t_xn = take((size_t)t * c.hidden * 2);
        w.t_qkv = take((size_t)t * (qd + 2 * kvd) * 4);
        w.q = take((size_t)t * qd * 2);
        w.attn_out = take((size_t)t * qd * 2);
        w.t_proj = take((size_t)t * c.hidden * 4);
        w.t_gu = take((size_t)t * 2 * c.intermediate * 4);
        // bf16 [T][inter], or (inter a multiple of 256) a whole workspace of the tiled GEMM over
        // K = inter: the gate/up projection then writes the down projection's operand there
        const size_t act_rows = (size_t)t * c.intermediate * 2;
        const size_t act_ws = c.intermediate % 256 == 0
                                  ? logismos_qgemm_q4g128_tall_workspace_bytes(t, c.intermediate)
                                  : 0;
        w.t_act_is_workspace = act_ws >= act_rows && act_ws > 0;
        w.t_act = take(w.t_act_is_workspace ? act_ws : act_rows);
        const int kmax = c.intermediate > (int)qd ? (c.intermediate > c.hidden ? c.intermediate : c.hidden)
                                                  : ((int)qd > c.hidden ? (int)qd : c.hidden);
        w.t_gemm = take(logismos_qgemm_q4g128_tall_workspace_bytes(t, kmax));
        if (c.vocab > 0) {
            w.last_rows = take((size_t)num_seqs * c.hidden * 2);
            w.last_xn = take(logismos_q4_xprep_bytes(kChunkRows, c.hidden));
            w.head_ws =
                take(logismos_qgemm_q4g128_greedy_workspace_bytes(kChunkRows, c.vocab, c.hidden));
        }
        w.resident = take(lg::decode_resident_pays(c) ? lg::decode_resident_bytes(c) : 0);
        w.total = off;
        return w;
    }
    w.chunks = (t + kChunkRows - 1) / kChunkRows;
    const int b = t < kChunkRows ? t : kChunkRows;
    // fp32 rows that the K parts of a product take: those of all rows on the plan of a chunk, and of a
    // ragged last chunk by itself, which may have more parts (few rows are split further).  The size
    // asked for (no base) holds the most over all smaller batches too, so that a workspace for many rows
    // is one for fewer; a launch lays out what its batch takes, which is no more (32 plans of four products
    // are 3 to 6 us of a host core).
    const int last = t - (w.chunks - 1) * kChunkRows;
    auto part_rows = [&](int n, int k) {
        int most = logismos_qgemm_q4g128_splitk_xprep_parts(b, n, k) * t;
        for (int rows = base ? last : 1; rows <= (base ? last : b); ++rows) {
            const int r = logismos_qgemm_q4g128_splitk_xprep_parts(rows, n, k) * rows;
            most = r > most ? r : most;
        }
        return (size_t)most;
    };
    const size_t o_rows = part_rows(c.hidden, (int)qd), down_rows = part_rows(c.hidden, c.intermediate);
    // prepared activations of all rows: one buffer, or one per chunk of 32
    auto xprep = [&](int k) {
        return w.chunks == 1 ? align256(logismos_q4_xprep_bytes(b, k))
                             : w.chunks * lg::xprep_rows_stride(k);
    };
    w.xn_stride = lg::xprep_rows_stride(c.hidden);
    w.xn = take(xprep(c.hidden));
    w.qkv = take(part_rows((int)(qd + 2 * kvd), c.hidden) * (qd + 2 * kvd) * 4);
    w.q = take((size_t)t * qd * 2);
    w.attn_b = take(xprep((int)qd));
    w.attn_out = take((size_t)t * qd * 2);
    w.proj = take((o_rows > down_rows ? o_rows : down_rows) * c.hidden * 4);
    w.gate_up = take(part_rows(2 * c.intermediate, c.hidden) * 2 * c.intermediate * 4);
    w.act = take(xprep(c.intermediate));
    w.attn_ws =
        take(logismos_paged_attn_workspace_bytes(num_seqs, c.num_q_heads, c.head_dim, num_splits));
    if (c.vocab > 0) {
        const int hb = num_seqs < kChunkRows ? (b > num_seqs ? b : num_seqs) : kChunkRows;
        w.head_ws = take(logismos_qgemm_q4g128_greedy_workspace_bytes(hb, c.vocab, c.hidden));
        w.norm_out = take((size_t)t * c.hidden * 2);
        w.last_rows = take((size_t)num_seqs * c.hidden * 2);
        w.last_xn = take(logismos_q4_xprep_bytes(kChunkRows, c.hidden));
    }
    w.resident = take(lg::decode_resident_pays(c) ? lg::decode_resident_bytes(c) : 0);
    w.total = off;
    return w;
}

bool config_ok(const logismos_decode_config_t* c, int num_seqs, int t, int max_seqlen_q) {
    if (!c || num_seqs <= 0 || t < num_seqs || max_seqlen_q < 1 || max_seqlen_q > t) return false;
    if (num_seqs > 65535 || t > 65535) return false;
    if (c->num_layers <= 0 || c->hidden <= 0 || c->intermediate <= 0 || c->max_pos <= 0)
        return false;
    if (c->num_q_heads <= 0 || c->num_kv_heads <= 0) return false;
    // heads of 128 on the kernels built for them; other multiples of 32 up to 256 on the general
    // attention kernel (fp16 pools only: a turbo3 head row is 128 wide)
    if (c->head_dim <= 0 || c->head_dim % 32 != 0 || c->head_dim > 256) return false;
    if (c->head_dim != 128 && c->kv_turbo3) return false;
    // what the attention launcher accepts, checked here so that no step is launched in part:
    // GQA groups up to 8 (16 on the general kernel), whose packed rows end at 65520
    if (c->num_q_heads % c->num_kv_heads != 0 ||
        c->num_q_heads / c->num_kv_heads > (c->head_dim == 128 ? 8 : 16))
        return false;
    if (c->head_dim != 128 && t > 65520) return false;
    if (c->hidden % 128 != 0 || c->intermediate % 128 != 0) return false;
    if (((int64_t)c->num_q_heads * c->head_dim) % 128 != 0) return false;
    // every position a block table can hold must have a row in the RoPE tables
    if (c->block_size <= 0 || c->max_blocks_per_seq <= 0 ||
        (int64_t)c->max_pos < (int64_t)c->block_size * c->max_blocks_per_seq)
        return false;
    if ((int64_t)t * (c->num_q_heads + 2 * c->num_kv_heads) * c->head_dim > (int64_t)INT32_MAX ||
        (int64_t)t * c->hidden > (int64_t)INT32_MAX)
        return false;
    if (c->vocab < 0) return false;
    // tokens in / tokens out for every packed row is a decode-step feature: one chunk
    if (c->vocab > 0 && t <= kChunkRows &&
        logismos_check_qgemm_q4g128_greedy_shape(t, c->vocab, c->hidden, nullptr, 0))
        return false;
    const int b = t < kChunkRows ? t : kChunkRows;
    const int qd = c->num_q_heads * c->head_dim;
    const int kvd = c->num_kv_heads * c->head_dim;
    if (t >= kTallRows) {
        // the tiled GEMM's own limits (the products of the whole batch are held in fp32)
        const int64_t lim = INT32_MAX;
        const int64_t widest = 2 * (int64_t)c->intermediate > qd + 2 * kvd
                                   ? 2 * (int64_t)c->intermediate
                                   : (int64_t)qd + 2 * kvd;
        return (int64_t)t * widest <= lim && (int64_t)widest * c->hidden <= lim &&
               (int64_t)c->hidden * c->intermediate <= lim && c->hidden >= 128 && qd >= 128;
    }
    // every projection must have a plan for a full chunk of rows and for the ragged last chunk
    const int last = t - (t - 1) / kChunkRows * kChunkRows;
    for (const int rows : {b, last}) {
        if (logismos_qgemm_q4g128_splitk_xprep_parts(rows, qd + 2 * kvd, c->hidden) <= 0 ||
            logismos_qgemm_q4g128_splitk_xprep_parts(rows, c->hidden, qd) <= 0 ||
            logismos_qgemm_q4g128_splitk_xprep_parts(rows, 2 * c->intermediate, c->hidden) <= 0 ||
            logismos_qgemm_q4g128_splitk_xprep_parts(rows, c->hidden, c->intermediate) <= 0)
            return false;
    }
    return true;
}

// The operands that every step on the 32-row or the few-row projections reads: all there, and the
// nibbles of every projection on 16 bytes (their loads).  Looked at for all layers before the first
// launch: the fused kernels check no pointer themselves, and no step is launched in part.
bool operands_ok(const logismos_decode_config_t& c, const logismos_decode_layer_t* layers,
                 const logismos_decode_batch_t& b) {
    if (!b.hidden_f32 || !b.final_norm_w_f32 || !b.block_tables || !b.cu_seqlens ||
        !b.context_lens || !b.positions || !b.slot_mapping || !b.rope_cos_f32 || !b.rope_sin_f32)
        return false;
    for (int l = 0; l < c.num_layers; ++l) {
        const logismos_decode_layer_t& L = layers[l];
        if (!L.norm1_w_f32 || !L.norm2_w_f32 || !L.k_pool_f16 || !L.v_pool_f16) return false;
        for (const logismos_q4_weight_t* W : {&L.qkv, &L.o, &L.gate_up, &L.down})
            if (!W->qw || !W->scale || !W->zero || (reinterpret_cast<uintptr_t>(W->qw) & 15u))
                return false;
    }
    return true;
}

// Whether every projection of the step can run on the fused few-row kernels.
bool few_rows(const logismos_decode_config_t& c, const logismos_decode_layer_t* layers, int t) {
    const int qd = c.num_q_heads * c.head_dim;
    const int widest = qd > c.intermediate ? qd : c.intermediate;
    for (int l = 0; l < c.num_layers; ++l)
        for (const logismos_q4_weight_t* W : {&layers[l].qkv, &layers[l].o, &layers[l].gate_up, &layers[l].down})
            if (!lg::qgemm_q4_rows_applies(t, c.hidden, widest,
                                           qd + 2 * c.num_kv_heads * c.head_dim, W->scale, W->zero))
                return false;
    return true;
}

// Whether the last chunk of a step of 33 to 96 rows goes through the projections by itself.  Tiles of
// 16 rows (and other K parts) add up in another order than the 32-row chunks beside them.  In front
// of 3-bit K/V rows a last bit flips whole codes: over chunks that read mostly their own new rows another
// order of the same sums moves the hidden state of 36 layers by up to 19 %, over decode rows, which
// read encoded rows that are there already, by 1.8 %.
bool split_last_chunk(const logismos_decode_config_t& c, int max_q, int last_rows) {
    if (!c.kv_turbo3 || max_q == 1) return false;
    const int qd = c.num_q_heads * c.head_dim, kvd = c.num_kv_heads * c.head_dim;
    return !(lg::qgemm_q4_splitk_same_sums(last_rows, qd + 2 * kvd, c.hidden) &&
             lg::qgemm_q4_splitk_same_sums(last_rows, c.hidden, qd) &&
             lg::qgemm_q4_splitk_same_sums(last_rows, 2 * c.intermediate, c.hidden) &&
             lg::qgemm_q4_splitk_same_sums(last_rows, c.hidden, c.intermediate));
}

#define LG_TRY(call)                                  \
    do {                                              \
        logismos_status_t st__ = (call);              \
        if (st__ != 0) return st__;                   \
    } while (0)

// The layers of a step of up to 16 rows on the fused few-row projections (qgemm_q4_rows.hip):
// every projection is one launch with the norm in front of it and what follows it folded in.
logismos_status_t few_rows_layers(const logismos_decode_config_t& c,
                                  const logismos_decode_layer_t* layers,
                                  const logismos_decode_batch_t* batch, const Workspace& w, int t,
                                  int max_q, bool direct, int* res_parts, logismos_stream_t stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int qd = c.num_q_heads * c.head_dim;
    const int width = qd + 2 * c.num_kv_heads * c.head_dim;
    const float scale = 1.0f / sqrtf((float)c.head_dim);
    lg::RowsArgs base{};
    base.b = t;
    base.eps = c.rms_eps;
    base.h = static_cast<float*>(batch->hidden_f32);
    auto with = [&](const logismos_q4_weight_t& W, int n, int k) {
        lg::RowsArgs a = base;
        a.qw = static_cast<const uint8_t*>(W.qw);
        a.scale = static_cast<const __half*>(W.scale);
        a.zero = static_cast<const __half*>(W.zero);
        a.tiles = n / 16;
        a.k = k;
        return a;
    };
    // the down projection in two parts leaves the second to the next layer's norm and o projection, and of
    // the last layer to the final norm
    const bool two = lg::qgemm_q4_rows_res_parts(c.hidden / 16, c.intermediate) == 2;
    const float* const pending = two ? reinterpret_cast<const float*>(w.proj) : nullptr;
    *res_parts = two ? 1 : 0;
    for (int l = 0; l < c.num_layers; ++l) {
        const logismos_decode_layer_t& L = layers[l];
        lg::RowsArgs a = with(L.qkv, width, c.hidden);
        a.gain = static_cast<const float*>(L.norm1_w_f32);
        a.e.pending = l ? pending : nullptr;
        if (c.kv_turbo3) {
            // the encoder wants whole head rows: the product as it is, then the operator
            a.e.out_f32 = reinterpret_cast<float*>(w.qkv);
            LG_TRY(lg::qgemm_q4_rows_launch(true, lg::kRowsF32, a, st));
            LG_TRY(logismos_launch_rope_kv_write_f32p_turbo3_bias(
                w.qkv, 1, L.qkv_bias_f32, batch->positions, batch->rope_cos_f32,
                batch->rope_sin_f32, batch->slot_mapping, w.q, L.k_pool_f16, L.v_pool_f16, t,
                c.num_q_heads, c.num_kv_heads, c.head_dim, c.max_pos, stream));
        } else {
            a.e.bias = static_cast<const float*>(L.qkv_bias_f32);
            a.e.positions = batch->positions;
            a.e.cos_t = static_cast<const float*>(batch->rope_cos_f32);
            a.e.sin_t = static_cast<const float*>(batch->rope_sin_f32);
            a.e.slots = batch->slot_mapping;
            a.e.q_out = reinterpret_cast<__half*>(w.q);
            a.e.k_pool = static_cast<__half*>(L.k_pool_f16);
            a.e.v_pool = static_cast<__half*>(L.v_pool_f16);
            a.e.hq = c.num_q_heads;
            a.e.hkv = c.num_kv_heads;
            a.e.head_dim = c.head_dim;
            a.e.max_pos = c.max_pos;
            a.e.tiles_per_head_inv = (unsigned)(((1 << 20) + c.head_dim / 16 - 1) / (c.head_dim / 16));
            LG_TRY(lg::qgemm_q4_rows_launch(true, lg::kRowsQkv, a, st));
        }
        LG_TRY(lg::paged_attn_launch(
            w.q, L.k_pool_f16, L.v_pool_f16, batch->block_tables, batch->cu_seqlens,
            batch->context_lens, direct ? w.attn_b : w.attn_out, w.attn_ws, batch->num_seqs, t, max_q,
            c.num_q_heads, c.num_kv_heads, c.head_dim, c.block_size, c.max_blocks_per_seq,
            batch->num_splits, scale, 1, LOGISMOS_ATTN_PHASE_ALL, direct ? 2 : 1,
            c.kv_turbo3 ? 1 : 0, stream));
        if (!direct)
            LG_TRY(logismos_launch_q4_prepare_x_bf16(w.attn_out, w.attn_b, t, qd, stream));
        a = with(L.o, c.hidden, qd);
        a.xprep = reinterpret_cast<const lg::uint4_t*>(w.attn_b);
        a.e.pending = l ? pending : nullptr;
        LG_TRY(lg::qgemm_q4_rows_launch(false, lg::kRowsRes, a, st));
        a = with(L.gate_up, 2 * c.intermediate, c.hidden);
        a.gain = static_cast<const float*>(L.norm2_w_f32);
        a.e.inter = c.intermediate;
        a.e.act = reinterpret_cast<lg::uint4_t*>(w.act);
        LG_TRY(lg::qgemm_q4_rows_launch(true, lg::kRowsSilu, a, st));
        a = with(L.down, c.hidden, c.intermediate);
        a.xprep = reinterpret_cast<const lg::uint4_t*>(w.act);
        a.e.out_f32 = reinterpret_cast<float*>(w.proj);
        LG_TRY(lg::qgemm_q4_rows_launch(false, lg::kRowsRes, a, st));
    }
    return 0;
}

// total_tokens / max_seqlen_q of a batch: 0 means "one new token per sequence"
int batch_tokens(const logismos_decode_batch_t* b) {
    return b->total_tokens > 0 ? b->total_tokens : b->num_seqs;
}
int batch_max_q(const logismos_decode_batch_t* b) {
    return b->max_seqlen_q > 0 ? b->max_seqlen_q : 1;
}

// How the layers of a step of one row are launched.
enum OneRow { kWhatIsFaster, kPerOperator, kOneLaunch };

logismos_status_t launch_step(const logismos_decode_config_t* cfg, const logismos_decode_layer_t* layers,
                              const logismos_decode_batch_t* batch, void* workspace, OneRow one_row,
                              logismos_stream_t stream);

}  // namespace

extern "C" size_t logismos_decode_step_workspace_bytes(const logismos_decode_config_t* cfg,
                                                       int num_seqs, int num_splits) {
    return logismos_decode_step_workspace_bytes_tokens(cfg, num_seqs, num_seqs, num_splits);
}

extern "C" size_t logismos_decode_step_workspace_bytes_tokens(const logismos_decode_config_t* cfg,
                                                              int num_seqs, int total_tokens,
                                                              int num_splits) {
    if (!config_ok(cfg, num_seqs, total_tokens, 1) || num_splits <= 0) return 0;
    return carve(*cfg, num_seqs, total_tokens, num_splits, nullptr).total;
}

extern "C" logismos_status_t logismos_launch_decode_step(const logismos_decode_config_t* cfg,
                                                         const logismos_decode_layer_t* layers,
                                                         const logismos_decode_batch_t* batch,
                                                         void* workspace,
                                                         logismos_stream_t stream) {
    return launch_step(cfg, layers, batch, workspace, kWhatIsFaster, stream);
}
extern "C" logismos_status_t logismos_launch_decode_step_per_operator(const logismos_decode_config_t* cfg,
                                                                      const logismos_decode_layer_t* layers,
                                                                      const logismos_decode_batch_t* batch,
                                                                      void* workspace,
                                                                      logismos_stream_t stream) {
    return launch_step(cfg, layers, batch, workspace, kPerOperator, stream);
}
// For the tests (the header does not declare it): one launch where it is possible at all, otherwise refused.  The
// workspace holds lg_decode_resident_bytes() more.
extern "C" logismos_status_t lg_launch_decode_step_one_launch(const logismos_decode_config_t* cfg,
                                                              const logismos_decode_layer_t* layers,
                                                              const logismos_decode_batch_t* batch, void* workspace,
                                                              logismos_stream_t stream) {
    return launch_step(cfg, layers, batch, workspace, kOneLaunch, stream);
}

namespace {

logismos_status_t launch_step(const logismos_decode_config_t* cfg, const logismos_decode_layer_t* layers,
                              const logismos_decode_batch_t* batch, void* workspace, OneRow one_row,
                              logismos_stream_t stream) {
    if (!cfg || !layers || !batch || !workspace) return hipErrorInvalidValue;
    const int num_seqs = batch->num_seqs;
    const int t = batch_tokens(batch);
    const int max_q = batch_max_q(batch);
    if (!config_ok(cfg, num_seqs, t, max_q) || batch->num_splits <= 0) return hipErrorInvalidValue;
    if (reinterpret_cast<uintptr_t>(workspace) & 255u) return hipErrorInvalidValue;
    const logismos_decode_config_t& c = *cfg;
    const bool tokens_in = batch->token_ids != nullptr;
    const bool tokens_out = batch->lm_head != nullptr;
    if ((tokens_in || tokens_out) && c.vocab <= 0) return hipErrorInvalidValue;
    if (tokens_in && !batch->embed_table_bf16) return hipErrorInvalidValue;
    if (tokens_out && !batch->out_tokens_u32) return hipErrorInvalidValue;
    if (!tokens_out && !batch->out_bf16) return hipErrorInvalidValue;
    const bool last_only = tokens_out && batch->tokens_for_last_rows != 0;
    if (last_only) {
        // the sequences' last rows go through the vocabulary projection 32 at a time
        const int full = num_seqs < kChunkRows ? num_seqs : kChunkRows;
        const int rest = num_seqs % kChunkRows;
        for (const int rows : {full, rest ? rest : full})
            if (logismos_check_qgemm_q4g128_greedy_shape(rows, c.vocab, c.hidden, nullptr, 0))
                return hipErrorInvalidValue;
    }
    // the vocabulary projection with its token choice takes one chunk of rows: every packed
    // row of a step of up to 32, or (tokens_for_last_rows) the last row of every sequence
    if (tokens_out && !last_only && t > kChunkRows) return hipErrorInvalidValue;
    const Workspace w = carve(c, num_seqs, t, batch->num_splits, static_cast<char*>(workspace));
    if (!w.tall && !operands_ok(c, layers, *batch)) return hipErrorInvalidValue;
    const int qd = c.num_q_heads * c.head_dim;
    const int kvd = c.num_kv_heads * c.head_dim;
    const int width = qd + 2 * kvd;
    const float scale = 1.0f / sqrtf((float)c.head_dim);
    // Steps of up to 96 rows: every launch takes all rows, except where a last chunk of few rows by
    // itself would add up in another order and that order matters (see below).
    const int last_rows = t - (w.chunks - 1) * kChunkRows;
    const bool one_pass = !w.tall && (w.chunks == 1 || !split_last_chunk(c, max_q, last_rows));
    // tokens for last rows: the normed rows of the whole batch, in the caller's buffer or in
    // the workspace, are gathered afterwards
    char* const norm_dst = batch->out_bf16 ? static_cast<char*>(batch->out_bf16)
                                           : (w.tall ? w.t_xn : w.norm_out);
    auto project_last_rows = [&]() -> logismos_status_t {
        LG_TRY(lg::gather_last_rows_bf16_launch(norm_dst, batch->cu_seqlens, w.last_rows, num_seqs,
                                                c.hidden, static_cast<hipStream_t>(stream)));
        const logismos_q4_weight_t& H = *batch->lm_head;
        for (int s0 = 0; s0 < num_seqs; s0 += kChunkRows) {
            const int rows = num_seqs - s0 < kChunkRows ? num_seqs - s0 : kChunkRows;
            LG_TRY(logismos_launch_q4_prepare_x_bf16(w.last_rows + (size_t)s0 * c.hidden * 2,
                                                     w.last_xn, rows, c.hidden, stream));
            LG_TRY(logismos_launch_qgemm_q4g128_greedy_xprep(
                w.last_xn, H.qw, H.scale, H.zero,
                static_cast<uint32_t*>(batch->out_tokens_u32) + s0,
                batch->logits_f32 ? static_cast<float*>(batch->logits_f32) + (size_t)s0 * c.vocab
                                  : nullptr,
                w.head_ws, rows, c.vocab, c.hidden, stream));
        }
        return 0;
    };
    // attention writes the o projection's input
    const bool direct = one_pass && lg::paged_attn_prepared_out(num_seqs, c.head_dim, c.num_q_heads,
                                                                c.num_kv_heads, c.block_size,
                                                                c.max_blocks_per_seq, max_q, batch->num_splits);
    float* const h = static_cast<float*>(batch->hidden_f32);
    const bool one_launch = (one_row == kOneLaunch || (one_row == kWhatIsFaster && lg::decode_resident_pays(c))) &&
                            lg::decode_resident_applies(c, layers, *batch, t);
    if (one_row == kOneLaunch && !one_launch) return hipErrorInvalidValue;

    if (tokens_in)
        LG_TRY(logismos_launch_embed_lookup_bf16(batch->embed_table_bf16, batch->token_ids,
                                                 batch->hidden_f32, t, c.hidden, c.vocab, stream));
    if (w.tall) {
        // ---- many rows: every projection is one launch of the tiled GEMM over all T rows
        // (fp32 products, consumed un-rounded by the next operator as in the chunked path), the
        // small operators run over all rows at once
        hipStream_t st = static_cast<hipStream_t>(stream);
        // The tiled GEMM over a workspace.  An odd number of groups of K only where its 16-byte
        // loads are aligned (the kernel that stages x itself takes any address; a layer of width
        // 896 at 1030 rows takes 215 us on that one, 177 here).
        auto tiled = [&](const logismos_q4_weight_t& W, const void* gains, int n, int k) {
            if (!lg::qgemm_q4_tallp_applies(t, n, k)) return false;
            const uintptr_t at = reinterpret_cast<uintptr_t>(W.qw) |
                                 reinterpret_cast<uintptr_t>(gains) |
                                 reinterpret_cast<uintptr_t>(batch->hidden_f32);
            return k % 256 == 0 || (at & 15u) == 0;
        };
        // A launch of fewer tiles than compute units is split over K; its fp32 parts are added up
        // by the operator that follows instead of by a launch of their own, which took 7.5 us three
        // times per layer (200 rows of the 4096-wide layers): in part order from zero, the same
        // sum, which is then added to the residual stream or rotated.  The parts lie in
        // the launch's workspace behind its operand, K wide; the norm that adds them up writes an
        // operand hidden wide to the front of t_gemm, hence `keep`.
        auto product = [&](const logismos_q4_weight_t& W, char* y_f32, char* workspace, int n, int k,
                           bool keep, lg::TallParts* out) -> logismos_status_t {
            if (keep)
                return lg::qgemm_q4_tallp_prepared_parts(W.qw, W.scale, W.zero, y_f32, workspace, t, n,
                                                         k, out, st);
            *out = {y_f32, 1};
            return lg::qgemm_q4_tallp_prepared(W.qw, W.scale, W.zero, nullptr, y_f32, 1, workspace, t,
                                               n, k, st);
        };
        auto gemm = [&](const void* x_bf16, const logismos_q4_weight_t& W, char* y_f32, int n, int k,
                        bool keep, lg::TallParts* out) -> logismos_status_t {
            // the kernel that takes x through a first pass into the workspace; past its sizes the
            // one that stages x itself
            if (tiled(W, nullptr, n, k)) {
                LG_TRY(lg::qgemm_q4_tallp_prepare(x_bf16, W.scale, W.zero, w.t_gemm, t, k, st));
                return product(W, y_f32, w.t_gemm, n, k, keep, out);
            }
            *out = {y_f32, 1};
            return lg::qgemm_q4_tall_f32_launch(x_bf16, W.qw, W.scale, W.zero, nullptr, y_f32, t, n, k,
                                                st);
        };
        lg::TallParts res{w.t_proj, 0};  // what is to be added to the residual stream
        // add + norm followed by a projection of the normed rows: where the tiled GEMM with a
        // workspace takes the shape, the normed rows go straight into its workspace in the
        // kernel's operand order (no first pass over them)
        auto norm_then_gemm = [&](const void* gains, const logismos_q4_weight_t& W, char* y_f32, int n,
                                  bool keep, lg::TallParts* out) -> logismos_status_t {
            if (tiled(W, gains, n, c.hidden) && c.hidden <= 16384) {
                LG_TRY(lg::add_rms_norm_tall(
                    batch->hidden_f32, res.src, res.count, true, gains, w.t_gemm, t, c.hidden, c.rms_eps,
                    logismos_qgemm_q4g128_tall_pairs_per_load(c.hidden, W.scale, W.zero), st));
                return product(W, y_f32, w.t_gemm, n, c.hidden, keep, out);
            }
            LG_TRY(lg::add_rms_norm_f32p(batch->hidden_f32, res.src, res.count, true, gains, w.t_xn, t,
                                         c.hidden, c.rms_eps, st));
            return gemm(w.t_xn, W, y_f32, n, c.hidden, keep, out);
        };
        for (int l = 0; l < c.num_layers; ++l) {
            const logismos_decode_layer_t& L = layers[l];
            lg::TallParts qkv;
            LG_TRY(norm_then_gemm(L.norm1_w_f32, L.qkv, w.t_qkv, width, true, &qkv));
            const auto rope_kv_write = c.kv_turbo3 ? logismos_launch_rope_kv_write_f32p_turbo3_bias
                                                   : logismos_launch_rope_kv_write_f32p_bias;
            LG_TRY(rope_kv_write(qkv.src, qkv.count, L.qkv_bias_f32, batch->positions,
                                 batch->rope_cos_f32, batch->rope_sin_f32, batch->slot_mapping, w.q, L.k_pool_f16,
                                 L.v_pool_f16, t, c.num_q_heads, c.num_kv_heads, c.head_dim,
                                 c.max_pos, stream));
            LG_TRY(lg::paged_attn_launch(
                w.q, L.k_pool_f16, L.v_pool_f16, batch->block_tables, batch->cu_seqlens,
                batch->context_lens, w.attn_out, w.attn_ws, num_seqs, t, max_q, c.num_q_heads,
                c.num_kv_heads, c.head_dim, c.block_size, c.max_blocks_per_seq, batch->num_splits,
                scale, 1, LOGISMOS_ATTN_PHASE_ALL, 1, c.kv_turbo3 ? 1 : 0, stream));
            LG_TRY(gemm(w.attn_out, L.o, w.t_proj, c.hidden, qd, qd >= c.hidden, &res));
            if (tiled(L.gate_up, L.norm2_w_f32, 2 * c.intermediate, c.hidden) && c.hidden <= 16384) {
                // the gate/up projection with the SwiGLU where its products are summed: the
                // fp32 gate and up products never go to memory
                LG_TRY(lg::add_rms_norm_tall(
                    batch->hidden_f32, res.src, res.count, true, L.norm2_w_f32, w.t_gemm, t, c.hidden,
                    c.rms_eps,
                    logismos_qgemm_q4g128_tall_pairs_per_load(c.hidden, L.gate_up.scale,
                                                              L.gate_up.zero),
                    st));
                if (w.t_act_is_workspace &&
                    logismos_check_qgemm_q4g128_tall_shape(t, c.hidden, c.intermediate, nullptr,
                                                           0) == 0) {
                    // ... and the activations written as the down projection's operand, in its
                    // own workspace: no bf16 rows in between, no first pass over them
                    LG_TRY(lg::qgemm_q4_tallp_swiglu_operand(
                        L.gate_up.qw, L.gate_up.scale, L.gate_up.zero, w.t_act,
                        logismos_qgemm_q4g128_tall_pairs_per_load(c.intermediate, L.down.scale,
                                                                  L.down.zero),
                        w.t_gemm, t, c.intermediate, c.hidden, st));
                    LG_TRY(product(L.down, w.t_proj, w.t_act, c.hidden, c.intermediate, true, &res));
                } else {
                    LG_TRY(lg::qgemm_q4_tallp_swiglu(L.gate_up.qw, L.gate_up.scale, L.gate_up.zero,
                                                     w.t_act, w.t_gemm, t, c.intermediate, c.hidden,
                                                     st));
                    LG_TRY(gemm(w.t_act, L.down, w.t_proj, c.hidden, c.intermediate,
                                c.intermediate >= c.hidden, &res));
                }
                continue;
            }
            lg::TallParts gu;
            LG_TRY(norm_then_gemm(L.norm2_w_f32, L.gate_up, w.t_gu, 2 * c.intermediate, false, &gu));
            if (logismos_check_qgemm_q4g128_tall_shape(t, c.hidden, c.intermediate, nullptr, 0) == 0) {
                // the activation goes straight into the down projection's workspace, in the
                // kernel's operand order: no first pass over it
                LG_TRY(logismos_launch_silu_mul_f32p_tall(
                    gu.src, gu.count, w.t_gemm, t, c.intermediate,
                    logismos_qgemm_q4g128_tall_pairs_per_load(c.intermediate, L.down.scale,
                                                              L.down.zero),
                    stream));
                LG_TRY(logismos_launch_qgemm_q4g128_tall_prepared(L.down.qw, L.down.scale, L.down.zero,
                                                                  nullptr, w.t_proj, 1, w.t_gemm, t,
                                                                  c.hidden, c.intermediate, stream));
                res = {w.t_proj, 1};
            } else {
                LG_TRY(logismos_launch_silu_mul_f32p(gu.src, gu.count, w.t_act, t, c.intermediate, stream));
                LG_TRY(gemm(w.t_act, L.down, w.t_proj, c.hidden, c.intermediate,
                            c.intermediate >= c.hidden, &res));
            }
        }
        LG_TRY(lg::add_rms_norm_f32p(batch->hidden_f32, res.src, res.count, true,
                                     batch->final_norm_w_f32, norm_dst, t, c.hidden, c.rms_eps, st));
        return last_only ? project_last_rows() : 0;
    }
    int res_parts = 0;  // split-K parts of the last down projection not yet folded into h
    if (one_launch) {
        LG_TRY(lg::decode_resident_launch(c, layers, *batch, w.resident, static_cast<hipStream_t>(stream)));
    } else if (few_rows(c, layers, t)) {
        LG_TRY(few_rows_layers(c, layers, batch, w, t, max_q, direct, &res_parts, stream));
    } else {
        // All rows in one launch of every operator, the projections in chunks of 32 side by side (48
        // rows of the 4096-wide layers, chunk after chunk: 19 launches a layer, 117 us beside the
        // attention; 10 launches now).  Two passes where the last chunk stays by itself.
        hipStream_t st = static_cast<hipStream_t>(stream);
        struct {
            int row0, rows;
            char* xn;
        } passes[2] = {{0, one_pass ? t : t - last_rows, w.xn},
                       {t - last_rows, last_rows, w.xn + (w.chunks - 1) * w.xn_stride}};
        const int num_passes = one_pass ? 1 : 2;
        // The normed input of a layer's first half is produced where the residual stream is
        // completed: before layer 0 here, afterwards by the add + norm that folds a pass's down
        // projection into h (with the NEXT layer's gains).
        for (int i = 0; i < num_passes; ++i)
            LG_TRY(lg::add_rms_norm_xprep_rows(h + (int64_t)passes[i].row0 * c.hidden, nullptr, 0,
                                               layers[0].norm1_w_f32, passes[i].xn, passes[i].rows,
                                               c.hidden, c.rms_eps, st));
        for (int l = 0; l < c.num_layers; ++l) {
            const logismos_decode_layer_t& L = layers[l];
            const bool last_layer = l + 1 == c.num_layers;
            // ---- first half: q/k/v projection, RoPE, K/V rows into the pools
            for (int i = 0; i < num_passes; ++i) {
                const int r0 = passes[i].row0, rows = passes[i].rows;
                LG_TRY(lg::qgemm_q4_splitk_rows(passes[i].xn, L.qkv.qw, L.qkv.scale, L.qkv.zero, w.qkv,
                                                rows, width, c.hidden, st));
                const int j = lg::qgemm_q4_splitk_rows_parts(rows, width, c.hidden);
                const auto rope_kv_write = c.kv_turbo3 ? logismos_launch_rope_kv_write_f32p_turbo3_bias
                                                       : logismos_launch_rope_kv_write_f32p_bias;
                LG_TRY(rope_kv_write(w.qkv, j, L.qkv_bias_f32, batch->positions + r0,
                                     batch->rope_cos_f32, batch->rope_sin_f32,
                                     batch->slot_mapping + r0, w.q + (size_t)r0 * qd * 2, L.k_pool_f16,
                                     L.v_pool_f16, rows, c.num_q_heads, c.num_kv_heads, c.head_dim,
                                     c.max_pos, stream));
            }
            // ---- attention over the whole ragged batch.  One pass: the result goes straight into
            // the prepared layout of the o projection; otherwise bf16 rows that each pass prepares
            // for itself.
            LG_TRY(lg::paged_attn_launch(
                w.q, L.k_pool_f16, L.v_pool_f16, batch->block_tables, batch->cu_seqlens,
                batch->context_lens, direct ? w.attn_b : w.attn_out,
                w.attn_ws, num_seqs, t, max_q, c.num_q_heads, c.num_kv_heads, c.head_dim, c.block_size,
                c.max_blocks_per_seq, batch->num_splits, scale, 1, LOGISMOS_ATTN_PHASE_ALL,
                direct ? 2 : 1, c.kv_turbo3 ? 1 : 0, stream));
            // ---- second half
            for (int i = 0; i < num_passes; ++i) {
                const int r0 = passes[i].row0, rows = passes[i].rows;
                char* const xn = passes[i].xn;
                float* hp = h + (int64_t)r0 * c.hidden;
                if (!direct)
                    LG_TRY(lg::q4_prepare_x_rows(w.attn_out + (size_t)r0 * qd * 2, w.attn_b, rows, qd,
                                                 st));
                LG_TRY(lg::qgemm_q4_splitk_rows(w.attn_b, L.o.qw, L.o.scale, L.o.zero, w.proj, rows,
                                                c.hidden, qd, st));
                LG_TRY(lg::add_rms_norm_xprep_rows(
                    hp, w.proj, lg::qgemm_q4_splitk_rows_parts(rows, c.hidden, qd), L.norm2_w_f32, xn,
                    rows, c.hidden, c.rms_eps, st));
                LG_TRY(lg::qgemm_q4_splitk_rows(xn, L.gate_up.qw, L.gate_up.scale, L.gate_up.zero,
                                                w.gate_up, rows, 2 * c.intermediate, c.hidden, st));
                LG_TRY(lg::silu_mul_xprep_rows(
                    w.gate_up, lg::qgemm_q4_splitk_rows_parts(rows, 2 * c.intermediate, c.hidden),
                    w.act, rows, c.intermediate, st));
                LG_TRY(lg::qgemm_q4_splitk_rows(w.act, L.down.qw, L.down.scale, L.down.zero, w.proj,
                                                rows, c.hidden, c.intermediate, st));
                const int j_down = lg::qgemm_q4_splitk_rows_parts(rows, c.hidden, c.intermediate);
                if (!last_layer) {
                    // fold the down projection into h and norm for the next layer's first half
                    LG_TRY(lg::add_rms_norm_xprep_rows(hp, w.proj, j_down, layers[l + 1].norm1_w_f32,
                                                       xn, rows, c.hidden, c.rms_eps, st));
                } else if (!one_pass) {
                    // last layer of two passes: the final norm of this pass's rows
                    LG_TRY(logismos_launch_add_rms_norm_f32p(
                        hp, w.proj, j_down, batch->final_norm_w_f32,
                        norm_dst + (size_t)r0 * c.hidden * 2, rows, c.hidden, c.rms_eps, stream));
                } else {
                    res_parts = j_down;
                }
            }
        }
    }
    if (!one_pass) return last_only ? project_last_rows() : 0;
    if (last_only) {
        LG_TRY(logismos_launch_add_rms_norm_f32p(batch->hidden_f32, w.proj, res_parts,
                                                 batch->final_norm_w_f32, norm_dst, t, c.hidden,
                                                 c.rms_eps, stream));
        return project_last_rows();
    }
    if (tokens_out) {
        // the normed state in the layout of the vocabulary projection, then the projection
        // with the token choice fused into it
        LG_TRY(logismos_launch_add_rms_norm_f32p_xprep(batch->hidden_f32, w.proj, res_parts,
                                                       batch->final_norm_w_f32, w.xn, t, c.hidden,
                                                       c.rms_eps, stream));
        res_parts = 0;  // folded into h by the call above
        const logismos_q4_weight_t& H = *batch->lm_head;
        LG_TRY(logismos_launch_qgemm_q4g128_greedy_xprep(w.xn, H.qw, H.scale, H.zero,
                                                         batch->out_tokens_u32, batch->logits_f32,
                                                         w.head_ws, t, c.vocab, c.hidden, stream));
    }
    if (batch->out_bf16)
        LG_TRY(logismos_launch_add_rms_norm_f32p(batch->hidden_f32, w.proj, res_parts,
                                                 batch->final_norm_w_f32, batch->out_bf16, t,
                                                 c.hidden, c.rms_eps, stream));
    return 0;
}

}  // namespace
