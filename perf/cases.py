"""The work a user of this library has it do, as timed cases.

Three kinds of call, all through the public wrappers of `logismos_amd.kernels`:

* `step`: one pass of the continuous-batching executor (packing of the ragged batch, embedding
  lookup, every layer, and where the geometry allows it the vocabulary projection with the token
  choice) over a paged KV cache, for decode batches, prefill chunks and mixtures of both;
* `linear`: one quantized `linear_t` (Q8G32, Q4G32, Q4G128), what a program that runs its own
  layers calls;
* `front`: the fp16 operators of the `kernels` crate in the order an encoder block calls them
  (rms_norm, matmul, rope).

Sizes are those of the repository's own configurations, tests and benchmark: the 24-layer
geometry with heads of 64, the one of 12 query and 2 KV heads, and the 36-layer one the
headline is quoted on.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from logismos_amd import kernels

BLOCK = 16  # rows per KV block

# layers, hidden, query heads, KV heads, head width, MLP width, q/k/v bias, tokens out.  The
# vocabulary projection of the library takes widths that are a multiple of 1024; the two small
# geometries stop at the normed state.
GEOMETRIES = {
    "h896": dict(layers=24, hidden=896, hq=14, hkv=2, d=64, inter=4864, bias=True, head=False),
    "h1536": dict(layers=28, hidden=1536, hq=12, hkv=2, d=128, inter=8960, bias=True, head=False),
    "h4096": dict(layers=36, hidden=4096, hq=32, hkv=8, d=128, inter=12288, bias=False, head=True),
}
VOCAB = 151936


def _step(name, geometry, decode, lo, hi, chunks=0, chunk=0, prior=0, turbo3=False, ragged=1):
    return dict(name=name, kind="step", geometry=geometry, decode=decode, ctx_lo=lo, ctx_hi=hi,
                chunks=chunks, chunk=chunk, prior=prior, turbo3=turbo3, ragged=ragged)


def listed():
    return [
        # One projection of a ggml Q8_0 model at one token: the smallest call there is.
        dict(name="q8 gemv 8960x1536", kind="linear", format="q8g32", rows=1, n=8960, k=1536),
        # One Q4G128 projection for a handful of concurrent sequences.
        dict(name="q4g128 8 rows", kind="linear", format="q4g128", rows=8, n=12288, k=4096),
        # The same of a ggml Q4_1 model.
        dict(name="q4g32 16 rows", kind="linear", format="q4g32", rows=16, n=12288, k=4096),
        # The front of an fp16 encoder block over a batch of documents.
        dict(name="fp16 block front", kind="front", batch=4, seq=509, hidden=1536, heads=12, d=128),
        # One user alone on the smallest model: nothing but launches and latency.
        _step("h896 1 user", "h896", 1, 500, 500),
        # Prompts arriving while others generate, small model, heads of 64.
        _step("h896 two prompts", "h896", 6, 256, 2048, chunks=2, chunk=512, prior=1000),
        # A small model serving sixteen short conversations.
        _step("h1536 16 users", "h1536", 16, 64, 2048),
        # One user alone on the large model: every weight read for one row.
        _step("h4096 1 user", "h4096", 1, 1500, 1500),
        # The headline: 32 conversations of up to 8192 tokens.
        _step("h4096 32 users", "h4096", 32, 256, 8192),
        # More users than one 32-row tile, on the 3-bit cache that makes room for them.
        _step("h4096 48 users turbo3", "h4096", 48, 256, 4096, turbo3=True),
        # One prompt chunk next to a few generating users.
        _step("h4096 chunk of 195", "h4096", 5, 256, 4096, chunks=1, chunk=195, prior=700),
        # A full server: 48 generating users with long contexts and 16 prompt chunks of 512.
        _step("h4096 full batch", "h4096", 48, 128, 16384, chunks=16, chunk=512, prior=8192),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: seven of ten are executor steps, as in real use."""
    what = rng.random()
    if what < 0.2:
        fmt = rng.choice(["q8g32", "q4g32", "q4g128"])
        unit = 32 if fmt == "q8g32" else 128
        k = max(4, _log(rng, 896 / unit, 12288 / unit)) * unit
        return dict(kind="linear", format=fmt, rows=1 if fmt == "q8g32" else _log(rng, 1, 64),
                    n=_log(rng, 1024, 24576), k=k)
    if what < 0.3:
        heads = rng.choice([8, 12, 16, 32])
        return dict(kind="front", batch=rng.randint(1, 8), seq=_log(rng, 16, 512),
                    hidden=8 * _log(rng, 96, 512), heads=heads, d=rng.choice([64, 128]))
    geometry = rng.choice(sorted(GEOMETRIES))
    g = GEOMETRIES[geometry]
    hi = _log(rng, 128, 8192)
    c = _step("", geometry, _log(rng, 1, 64), min(128, hi), hi, ragged=rng.randint(2, 1 << 20),
              turbo3=g["d"] == 128 and rng.random() < 0.2)
    if rng.random() < 0.5:
        c.update(chunks=_log(rng, 1, 8), chunk=_log(rng, 16, 512), prior=_log(rng, 1, 4096),
                 decode=_log(rng, 1, 48))
    del c["name"]
    return c


# ---------------------------------------------------------------------------- what a case holds
def _batch_shape(case):
    """(new tokens, prior context) of every sequence, from the case's own numbers."""
    r = np.random.default_rng(case["ragged"])
    dec = np.exp(r.uniform(math.log(case["ctx_lo"]), math.log(case["ctx_hi"] + 1), case["decode"])) \
        if case["ctx_hi"] > 8192 else r.integers(case["ctx_lo"], case["ctx_hi"] + 1, case["decode"])
    new = np.concatenate([np.ones(case["decode"], np.int64),
                          np.full(case["chunks"], case["chunk"], np.int64)])
    prior = np.concatenate([np.asarray(dec, np.int64).clip(1) - 1,
                            r.integers(0, case["prior"] + 1, case["chunks"])])
    order = r.permutation(len(new))
    return new[order], prior[order].astype(np.int64)


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _q4_weight(gen, n, k, group, keep=False):
    """Normal weights of deviation 0.02 in 4 bits: codes around the middle of the range, one
    scale and one zero point per group."""
    q = torch.empty(n, k, device="cuda").normal_(7.5, 15 / 5.6, generator=gen)
    q = q.round_().clamp_(0, 15).to(torch.uint8)
    qw = (q[:, 0::2] | (q[:, 1::2] << 4)).contiguous()
    scale = torch.empty(n, k // group, device="cuda").normal_(1, 0.08, generator=gen)
    scale = (scale * (0.02 * 5.6 / 15)).half()
    zero = torch.empty(n, k // group, device="cuda").normal_(7.5, 0.4, generator=gen).half()
    return (qw, scale, zero, q) if keep else (qw, scale, zero)


def _bf16(gen, *shape):
    return torch.empty(*shape, device="cuda").normal_(0, 1, generator=gen).bfloat16()


# ---------------------------------------------------------------------------- linear
def _prepare_linear(case, gen):
    m, n, k, fmt = case["rows"], case["n"], case["k"], case["format"]
    s = dict(case=case)
    if fmt == "q8g32":
        s["x"] = torch.empty(k, device="cuda").normal_(0, 1, generator=gen)
        w = torch.empty(n, k, device="cuda").normal_(0, 127 / 2.7, generator=gen)
        s["w"] = (w.round_().clamp_(-127, 127).to(torch.int8),
                  torch.empty(n, k // 32, device="cuda").normal_(1, 0.15, generator=gen)
                  .mul_(0.02 * 2.7 / 127).half())
        s["y"] = torch.empty(n, device="cuda")
        return s
    one = fmt == "q4g32" and m == 1  # the fp32 GEMV of the ggml formats
    s["x"] = _bf16(gen, m, k).float() if one else _bf16(gen, m, k)
    qw, scale, zero = _q4_weight(gen, n, k, 32 if fmt == "q4g32" else 128)
    if fmt == "q4g32":  # w = q * scale + min
        zero = (-(zero.float() * scale.float())).half()
    s["w"] = (qw, scale, zero)
    s["y"] = torch.empty(m, n, device="cuda", dtype=torch.float32 if one else torch.bfloat16)
    if fmt == "q4g128" and m > 32 and k % 256 == 0:  # many rows: the entry point with a workspace
        s["ws"] = torch.empty(kernels.qgemm_q4g128_tall_workspace_bytes(m, k), device="cuda",
                              dtype=torch.uint8)
    return s


def _run_linear(s):
    c = s["case"]
    x, y, w = _ptr(s["x"]), _ptr(s["y"]), [_ptr(t) for t in s["w"]]
    if c["format"] == "q8g32":
        kernels.launch_qgemv_q8g32_f32(x, *w, y, c["n"], c["k"])
    elif c["format"] == "q4g32" and c["rows"] == 1:
        kernels.launch_qgemv_q4g32_f32(x, *w, y, c["n"], c["k"])
    elif c["format"] == "q4g32":
        kernels.launch_qgemm_q4g32_bf16(x, *w, y, c["rows"], c["n"], c["k"])
    elif "ws" in s:
        kernels.launch_qgemm_q4g128_tall(x, *w, y, _ptr(s["ws"]), c["rows"], c["n"], c["k"])
    else:
        kernels.launch_qgemm_q4g128_bf16(x, *w, y, c["rows"], c["n"], c["k"])
    return s["y"]


# ---------------------------------------------------------------------------- front
def _prepare_front(case, gen):
    m, hidden, width = case["batch"] * case["seq"], case["hidden"], case["heads"] * case["d"]
    half = dict(device="cuda", dtype=torch.float16)
    s = dict(case=case)
    s["x"] = torch.empty(m, hidden, device="cuda").normal_(0, 1, generator=gen).half()
    s["gain"] = torch.empty(hidden, device="cuda").normal_(1, 0.02, generator=gen).half()
    s["w"] = torch.empty(hidden, width, device="cuda").normal_(0, 0.02, generator=gen).half()
    s["xn"], s["q"] = torch.empty(m, hidden, **half), torch.empty(m, width, **half)
    inv = 1e4 ** (-torch.arange(0, case["d"], 2, device="cuda", dtype=torch.float32) / case["d"])
    ang = torch.arange(case["seq"], device="cuda", dtype=torch.float32)[:, None] * inv
    s["table"] = torch.stack([ang.cos(), ang.sin()], -1).reshape(case["seq"], case["d"]).contiguous()
    return s


def _run_front(s):
    c = s["case"]
    m, width = c["batch"] * c["seq"], c["heads"] * c["d"]
    kernels.launch_rms_norm_fp16(_ptr(s["x"]), _ptr(s["gain"]), _ptr(s["xn"]), m, c["hidden"], 1e-6)
    kernels.launch_matmul_fp16("wmma", _ptr(s["xn"]), _ptr(s["w"]), _ptr(s["q"]), m, width,
                               c["hidden"])
    kernels.launch_rope_fp16_in_place(_ptr(s["q"]), _ptr(s["table"]), c["batch"], c["seq"],
                                      c["heads"], c["d"])
    return dict(xn=s["xn"], q=s["q"])


# ---------------------------------------------------------------------------- step
def _prepare_step(case, gen):
    g = GEOMETRIES[case["geometry"]]
    L, hidden, hq, hkv, d, inter = (g[x] for x in ("layers", "hidden", "hq", "hkv", "d", "inter"))
    new, prior = _batch_shape(case)
    ctx = new + prior
    S, T = len(new), int(new.sum())
    dev = dict(device="cuda")
    i32 = dict(device="cuda", dtype=torch.int32)
    s = dict(case=case, keep=[])

    def hold(t):
        s["keep"].append(t)
        return _ptr(t)

    # ---- the paged cache: block ids in random order, those that receive the new rows first, so
    # that what the step writes is one range of every pool
    nblk = -(-ctx // BLOCK)
    first = prior // BLOCK
    fresh = nblk - first
    written, total = int(fresh.sum()), int(nblk.sum())
    pick = np.random.default_rng(int(torch.randint(1 << 30, (1,), generator=gen, **dev)))
    new_ids, old_ids = pick.permutation(written), written + pick.permutation(total - written)
    tables = np.full((S, int(nblk.max())), 0x3FFFFFF, np.int32)
    a = b = 0
    for i in range(S):
        tables[i, first[i]:nblk[i]] = new_ids[a:a + fresh[i]]
        tables[i, :first[i]] = old_ids[b:b + first[i]]
        a, b = a + int(fresh[i]), b + int(first[i])
    row = hkv * d
    if case["turbo3"]:
        pools = torch.empty(L, 2, total, BLOCK, hkv * 56, dtype=torch.uint8, **dev)
        at = torch.arange(total * BLOCK, **dev)
        for layer in pools:
            kv = [torch.empty(total * BLOCK, row, dtype=torch.float16, **dev)
                  .normal_(0, 1, generator=gen) for _ in range(2)]
            kernels.launch_kv_write_turbo3(_ptr(kv[0]), _ptr(kv[1]), _ptr(layer[0]), _ptr(layer[1]),
                                           _ptr(at), total * BLOCK, hkv)
    else:
        pools = torch.empty(L, 2, total, BLOCK, row, dtype=torch.float16, **dev)
        for layer in pools:
            layer.normal_(0, 1, generator=gen)
    s["pools"] = pools

    # ---- weights
    layers = (kernels.DecodeLayer * L)()
    width = (hq + 2 * hkv) * d
    for i in range(L):
        for name, n, k in (("qkv", width, hidden), ("o", hidden, hq * d),
                           ("gate_up", 2 * inter, hidden), ("down", hidden, inter)):
            setattr(layers[i], name, kernels.Q4Weight(*map(hold, _q4_weight(gen, n, k, 128))))
        for name in ("norm1_w_f32", "norm2_w_f32"):
            setattr(layers[i], name, hold(torch.empty(hidden, **dev).normal_(1, 0.02, generator=gen)))
        if g["bias"]:
            layers[i].qkv_bias_f32 = hold(torch.empty(width, **dev).normal_(0, 1, generator=gen))
        layers[i].k_pool_f16, layers[i].v_pool_f16 = _ptr(pools[i, 0]), _ptr(pools[i, 1])
    # embedding and vocabulary projection share their values (tied embeddings), which also gives
    # the choice of the next token the clear margin a trained model has
    *head, codes = _q4_weight(gen, VOCAB, hidden, 128, keep=True)
    table = torch.empty(VOCAB, hidden, dtype=torch.bfloat16, **dev)
    for r0 in range(0, VOCAB, 16384):
        r1 = min(VOCAB, r0 + 16384)
        sc, ze = (t[r0:r1].float().repeat_interleave(128, 1) for t in head[1:])
        table[r0:r1] = (codes[r0:r1].float() - ze) * sc * 100
    del codes
    s["table"] = table
    s["ids"] = torch.randint(VOCAB, (T,), generator=gen, **i32)

    # ---- the batch
    max_blocks = tables.shape[1]
    max_pos = max_blocks * BLOCK
    ang = torch.arange(max_pos, dtype=torch.float64, **dev)[:, None] * \
        1e6 ** (-torch.arange(0, d, 2, dtype=torch.float64, **dev) / d)
    positions = np.concatenate([np.arange(p, c) for p, c in zip(prior, ctx)]).astype(np.int32)
    s["new"] = torch.from_numpy(new.astype(np.int32)).cuda()
    s["prior"] = torch.from_numpy(prior.astype(np.int32)).cuda()
    s["tables"] = torch.from_numpy(tables).cuda()
    s["cu"], s["ctx"] = torch.zeros(S + 1, **i32), torch.zeros(S, **i32)
    s["slots"] = torch.zeros(T, dtype=torch.int64, **dev)
    s["h"] = torch.zeros(T, hidden, **dev)
    splits = kernels.paged_attn_num_splits(S, hkv, BLOCK, max_blocks, d)
    s["cfg"] = kernels.DecodeConfig(
        num_layers=L, hidden=hidden, num_q_heads=hq, num_kv_heads=hkv, head_dim=d,
        intermediate=inter, rms_eps=1e-6, block_size=BLOCK, max_blocks_per_seq=max_blocks,
        max_pos=max_pos, vocab=VOCAB if g["head"] else 0, kv_turbo3=int(case["turbo3"]))
    batch = kernels.DecodeBatch(
        hidden_f32=_ptr(s["h"]), final_norm_w_f32=hold(torch.ones(hidden, **dev)),
        block_tables=_ptr(s["tables"]), cu_seqlens=_ptr(s["cu"]), context_lens=_ptr(s["ctx"]),
        positions=hold(torch.from_numpy(positions).cuda()), slot_mapping=_ptr(s["slots"]),
        rope_cos_f32=hold(ang.cos().float()), rope_sin_f32=hold(ang.sin().float()),
        num_seqs=S, num_splits=splits, total_tokens=T, max_seqlen_q=int(new.max()))
    # the rows appended to the cache are an output; of a 3-bit cache they are codes, of which a
    # last bit in front of the encoder flips whole ones: what they hold shows in the hidden
    # state, whose attention has read them
    s["out"] = dict(hidden=s["h"]) if case["turbo3"] else \
        dict(hidden=s["h"], new_kv=pools[:, :, :written])
    if g["head"]:
        s["head"] = kernels.Q4Weight(*map(hold, head))
        s["out"]["tokens"] = torch.zeros(S, **i32)
        s["out"]["logits"] = torch.zeros(S, VOCAB, **dev)
        batch.token_ids, batch.embed_table_bf16 = _ptr(s["ids"]), _ptr(table)
        batch.lm_head = C.pointer(s["head"])
        batch.out_tokens_u32 = _ptr(s["out"]["tokens"])
        batch.logits_f32 = _ptr(s["out"]["logits"])
        batch.tokens_for_last_rows = int(T > S or S > 32)
    else:
        s["out"]["normed"] = torch.zeros(T, hidden, dtype=torch.bfloat16, **dev)
        batch.out_bf16 = _ptr(s["out"]["normed"])
    need = kernels.decode_step_workspace_bytes_tokens(s["cfg"], S, T, splits)
    s["ws"] = torch.empty(need, dtype=torch.uint8, **dev)
    s.update(batch=batch, layers=layers, S=S, T=T, max_blocks=max_blocks, hidden=hidden)
    return s


def _run_step(s):
    kernels.launch_pack_ragged(_ptr(s["new"]), _ptr(s["prior"]), _ptr(s["tables"]), _ptr(s["cu"]),
                               _ptr(s["slots"]), _ptr(s["ctx"]), s["S"], BLOCK, s["max_blocks"])
    if not s["cfg"].vocab:
        kernels.launch_embed_lookup(_ptr(s["table"]), _ptr(s["ids"]), _ptr(s["h"]), s["T"],
                                    s["hidden"], VOCAB, True)
    kernels.launch_decode_step(s["cfg"], s["layers"], s["batch"], _ptr(s["ws"]))
    return s["out"]


_PREPARE = dict(linear=_prepare_linear, front=_prepare_front, step=_prepare_step)
_RUN = dict(linear=_run_linear, front=_run_front, step=_run_step)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    s = _PREPARE[case["kind"]](case, gen)
    s["run"] = _RUN[case["kind"]]
    return s


def run(state):
    return state["run"](state)


def _q4_bytes(n, k, group):
    return n * k // 2 + n * (k // group) * 4


def work(case):
    if case["kind"] == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        if case["format"] == "q8g32":
            return dict(bytes=n * k + n * (k // 32) * 2 + 4 * (n + k), flops=2 * n * k)
        size = 4 if case["format"] == "q4g32" and m == 1 else 2
        return dict(bytes=_q4_bytes(n, k, 32 if case["format"] == "q4g32" else 128)
                    + size * m * (n + k), flops=2 * m * n * k)
    if case["kind"] == "front":
        m, h, w = case["batch"] * case["seq"], case["hidden"], case["heads"] * case["d"]
        return dict(bytes=2 * (2 * m * h + h + h * w + m * w) + 4 * case["seq"] * case["d"],
                    flops=2 * m * h * w + 4 * m * h + 3 * m * w)
    g = GEOMETRIES[case["geometry"]]
    L, hidden, hq, hkv, d, inter = (g[x] for x in ("layers", "hidden", "hq", "hkv", "d", "inter"))
    new, prior = _batch_shape(case)
    ctx = new + prior
    S, T = len(new), int(new.sum())
    mats = [((hq + 2 * hkv) * d, hidden), (hidden, hq * d), (2 * inter, hidden), (hidden, inter)]
    kv_row = 2 * hkv * (56 if case["turbo3"] else 2 * d)  # K and V of one token, one layer
    pairs = int((new * prior + new * (new + 1) // 2).sum())
    # weights, the visible cache (the new rows are written, not read), ids, tables and rows
    size = L * (sum(_q4_bytes(n, k, 128) for n, k in mats) + 8 * hidden
                + kv_row * int(prior.sum() + T))
    size += T * (4 + 2 * hidden + 4 * hidden) + 4 * int((-(-ctx // BLOCK)).sum())
    flops = L * (2 * T * sum(n * k for n, k in mats) + 4 * pairs * hq * d)
    if g["head"]:
        size += _q4_bytes(VOCAB, hidden, 128) + 4 * S * VOCAB
        flops += 2 * S * VOCAB * hidden
    else:
        size += 2 * T * hidden
    return dict(bytes=size, flops=flops)


def tolerance(case):
    """About four times what was measured of two correct forms of the same arithmetic."""
    if case["kind"] == "linear":
        if case["format"] == "q8g32" or (case["format"] == "q4g32" and case["rows"] == 1):
            return {"rel": 2e-6, "max": 1e-5}  # fp32 out, against 64 bits: 1.2e-7, 4.3e-7
        return {"rel": 1e-3, "max": 0.03}  # bf16 out, against the rounded 64-bit result: 1e-4, 7e-3
    if case["kind"] == "front":
        return {"rel": 1e-3, "max": 7e-3}  # against 64 bits with the same roundings: 2.1e-4, 1.6e-3
    # a step with other numbers of KV partitions, and two halves of a batch (other tiles) against
    # the whole: every bf16 rounding point of a layer turns last bits into flips that the
    # following layers carry on
    return {
        "h896": {"rel": 0.01, "max": 0.04},  # 2.4e-3, 7.8e-3
        "h1536": {"rel": 0.02, "max": 0.1},  # 5.2e-3, 2.2e-2
        "h4096": {"rel": 0.03, "max": 0.5, "differ": 0.01},  # 1.6e-2, 1.2e-1; no token differed
    }[case["geometry"]]
