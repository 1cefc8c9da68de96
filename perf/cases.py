"""The calls this framework is timed on: attention steps over the paged KV cache, the MLP half of
a decode layer, and whole engine steps of a Llama model.

A case is a dict of plain values.  Sequence lengths belong to the case (``lengths`` seeds them);
tensor contents come from the seed given to :func:`prepare`.  Kinds:

``decode``   one new token per sequence as ``PagedAttentionOp`` runs it: ``rope_reshape_and_cache``
             of the new rows, then ``execute`` (v1 up to 4096 tokens of context, v2 beyond).
``step``     the same step through ``launch_rope_reshape_and_cache_v1`` with a workspace that the
             caller keeps, as a serving loop holds it.
``prefill``  packed prompt chunks: ``rope_reshape_and_cache``, then ``prefill_packed``.
``mlp``      the second half of a decode layer: o_proj onto the residual stream, the folded
             RmsNorm with gate/up and SiLU * mul, down_proj onto the residual stream.
``model``    ``RailgunLlama.forward`` of one engine step: prompt chunks first, then decode slots.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from railgun_amd.batch import DecodeSlot, PrefillChunk, pack_step
from railgun_amd.kv_pool import GpuBlockPool
from railgun_amd.llama import DeviceStep, LayerWeights, LlamaConfig, LlamaWeights, RailgunLlama
from railgun_amd.ops import (PagedAttentionKernels, PagedAttentionOp, interleave_gate_up, linear_residual,
                             linear_silu_mul, linear_workspace_bytes, rope_cos_sin_table)

DEVICE = "cuda:0"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
THETA = 500000.0
EPS = 1e-5
# The 1B Llama of the model cases: 16 layers, 32 / 8 heads of 64, tied embedding.
MODEL = dict(hidden_size=2048, intermediate_size=8192, num_hidden_layers=16, num_attention_heads=32,
             num_key_value_heads=8, vocab_size=128256, rms_norm_eps=EPS, rope_theta=THETA)
MODEL_DIM = 64


def listed():
    return [
        # The reference's own CPU-runnable shape and element type: a handful of short chats in fp32.
        # The smallest call: launches and latency count.
        dict(name="decode_f32_small", kind="decode", dtype="f32", heads=32, kv_heads=8, head_dim=64, block_size=16,
             fused=False, batch=4, ctx_lo=17, ctx_hi=255, lengths=1),
        # One interactive user of an 8B-shaped model, a thousand tokens into a chat.
        dict(name="decode_one_user", kind="decode", dtype="bf16", heads=32, kv_heads=8, head_dim=128, block_size=16,
             fused=True, batch=1, ctx_lo=1003, ctx_hi=1003, lengths=2),
        # The headline serving load: one layer of an 8B-shaped model, 64 sequences of 512 to 4096 tokens.
        dict(name="step_b64", kind="step", dtype="bf16", heads=32, kv_heads=8, head_dim=128, block_size=16,
             fused=False, batch=64, ctx_lo=512, ctx_hi=4096, lengths=3),
        # Long documents: 8 sequences of 32k tokens, the v2 split-K branch of the op.
        dict(name="decode_long_b8", kind="decode", dtype="bf16", heads=32, kv_heads=8, head_dim=128, block_size=16,
             fused=False, batch=8, ctx_lo=32768, ctx_hi=32768, lengths=4),
        # An odd-sized batch in fp16 (the reference's default KV type) over a fused pool, seven query
        # heads to a kv-head, blocks of 32.
        dict(name="decode_f16_gqa7", kind="decode", dtype="f16", heads=28, kv_heads=4, head_dim=128, block_size=32,
             fused=True, batch=17, ctx_lo=90, ctx_hi=3900, lengths=5),
        # Continuous batching admits a dozen prompts of mixed length at once.
        dict(name="prefill_packed", kind="prefill", dtype="bf16", heads=32, kv_heads=8, head_dim=128, block_size=16,
             fused=False, batch=12, len_lo=128, len_hi=2048, prior_lo=0, prior_hi=0, lengths=6),
        # Chunked prefill of a 1B-shaped model: chunks of up to 512 tokens behind a cached prefix.
        dict(name="prefill_chunked_d64", kind="prefill", dtype="bf16", heads=32, kv_heads=8, head_dim=64,
             block_size=16, fused=True, batch=16, len_lo=300, len_hi=512, prior_lo=0, prior_hi=4096, lengths=7),
        # A few short questions arriving together, fp16, three query heads to a kv-head.
        dict(name="prefill_short_f16", kind="prefill", dtype="f16", heads=24, kv_heads=8, head_dim=128, block_size=16,
             fused=True, batch=9, len_lo=9, len_hi=150, prior_lo=0, prior_hi=0, lengths=8),
        # Prompts in the reference's element type.
        dict(name="prefill_f32", kind="prefill", dtype="f32", heads=32, kv_heads=8, head_dim=64, block_size=16,
             fused=False, batch=5, len_lo=64, len_hi=1000, prior_lo=0, prior_hi=0, lengths=9),
        # The MLP half of an 8B-shaped layer for an odd decode batch.
        dict(name="mlp_rows27", kind="mlp", dtype="bf16", rows=27, hidden=4096, inter=14336),
        # A decode step of a whole 1B model under continuous batching.
        dict(name="model_decode_b64", kind="model", prompts=0, len_lo=0, len_hi=0, prior_hi=0, decodes=64, ctx_lo=64,
             ctx_hi=8192, lengths=11),
        # An engine step that admits three prompts while twenty sequences decode.
        dict(name="model_mixed", kind="model", prompts=3, len_lo=90, len_hi=400, prior_hi=300, decodes=20, ctx_lo=64,
             ctx_hi=4000, lengths=12),
    ]


# (heads, kv_heads, head_dim) of the attention cases.
HEADS = [(32, 8, 64), (32, 8, 128), (24, 8, 128), (28, 4, 128), (40, 8, 128)]


def _log_int(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "step", "prefill", "prefill", "mlp", "model"])
    lengths = rng.randrange(1 << 30)
    if kind == "mlp":
        hidden, inter = rng.choice([(2048, 8192), (3072, 8192), (4096, 14336)])
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "f16"]), rows=_log_int(rng, 1, 128), hidden=hidden,
                    inter=inter)
    if kind == "model":
        prompts = rng.choice([0, 0, 1, 2, 3])
        hi = _log_int(rng, 20, 400) if prompts else 0
        return dict(kind=kind, prompts=prompts, len_lo=min(hi, rng.randint(1, 90)), len_hi=hi,
                    prior_hi=rng.choice([0, 300]) if prompts else 0, decodes=_log_int(rng, 1, 20 if prompts else 64),
                    ctx_lo=rng.randint(1, 64), ctx_hi=_log_int(rng, 65, 4000 if prompts else 8192), lengths=lengths)
    heads, kv_heads, head_dim = rng.choice(HEADS)
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"] if kind != "step" else ["bf16", "f16"])
    case = dict(kind=kind, dtype=dtype, heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                block_size=rng.choice([16, 16, 32]), fused=rng.random() < 0.5)
    if kind == "prefill":
        batch = _log_int(rng, 1, 16)
        # Rows times cached positions are held to what the listed prompts ask for.
        hi = _log_int(rng, 8, (512 if dtype == "f32" else 2048) if batch <= 12 else 512)
        prior = rng.choice([0, 0, _log_int(rng, 16, 1024 if dtype == "f32" else 4096)]) if hi <= 512 else 0
        return dict(case, batch=batch, len_lo=rng.randint(1, hi), len_hi=hi, prior_lo=0, prior_hi=prior,
                    lengths=lengths)
    batch = _log_int(rng, 1, 64)
    hi = _log_int(rng, 17, min(32768 if kind == "decode" else 4096, (131072 if dtype == "f32" else 262144) // batch))
    return dict(case, batch=batch, ctx_lo=rng.randint(1, hi), ctx_hi=hi, lengths=lengths)


# ---------------------------------------------------------------- inputs ----


def _sizes(case):
    """(new tokens, context length with them) of each sequence, int64."""
    rng = np.random.default_rng(case["lengths"])
    if case["kind"] == "prefill":
        new = rng.integers(case["len_lo"], case["len_hi"], size=case["batch"], endpoint=True)
        return new, new + rng.integers(case["prior_lo"], case["prior_hi"], size=case["batch"], endpoint=True)
    if case["kind"] == "model":
        new = rng.integers(case["len_lo"], case["len_hi"], size=case["prompts"], endpoint=True)
        prior = rng.integers(0, case["prior_hi"], size=case["prompts"], endpoint=True)
        ctx = rng.integers(case["ctx_lo"], case["ctx_hi"], size=case["decodes"], endpoint=True)
        return np.concatenate([new, np.ones(len(ctx), np.int64)]), np.concatenate([new + prior, ctx])
    ctx = rng.integers(case["ctx_lo"], case["ctx_hi"], size=case["batch"], endpoint=True)
    return np.ones(len(ctx), np.int64), ctx


def _tables(ctx, block_size, seed):
    """Block tables [sequences, longest] over a shuffled pool a tenth larger than needed, and its size."""
    need = (ctx + block_size - 1) // block_size
    blocks = int(math.ceil(1.1 * need.sum()))
    order = np.random.default_rng(seed).permutation(blocks).astype(np.int32)
    table = np.zeros((len(ctx), int(need.max())), np.int32)
    at = 0
    for s, n in enumerate(need):
        table[s, :n] = order[at:at + n]
        at += n
    return table, blocks


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(g, shape, dtype, std=1.0):
    return torch.empty(shape, device=DEVICE, dtype=dtype).normal_(0.0, std, generator=g)


def _i32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).to(DEVICE)


def _attention_inputs(case, seed):
    """The tensors of one attention call, from the case and the seed alone."""
    new, ctx = _sizes(case)
    bs, hkv, d = case["block_size"], case["kv_heads"], case["head_dim"]
    table, blocks = _tables(ctx, bs, seed)
    pos = np.concatenate([np.arange(c - n, c) for n, c in zip(new, ctx)])
    seq = np.repeat(np.arange(len(new)), new)
    slots = table[seq, pos // bs].astype(np.int64) * bs + pos % bs
    g, dt, t = _generator(seed), DTYPES[case["dtype"]], len(pos)
    q, k, v = (_normal(g, (t, h, d), dt) for h in (case["heads"], hkv, hkv))
    if case["fused"]:
        pool = _normal(g, (blocks, 2, hkv, bs, d), dt)
        kc, vc = pool[:, 0], pool[:, 1]
    else:
        kc, vc = _normal(g, (blocks, hkv, bs, d), dt), _normal(g, (blocks, hkv, bs, d), dt)
    return dict(q=q, k=k, v=v, kc=kc, vc=vc, table=table, new=new, ctx=ctx, pos=pos, slots=slots)


def _mlp_inputs(case, seed):
    g, dt = _generator(seed), DTYPES[case["dtype"]]
    rows, hidden, inter = case["rows"], case["hidden"], case["inter"]
    return dict(x=_normal(g, (rows, hidden), dt), attn=_normal(g, (rows, hidden), dt),
                wo=_normal(g, (hidden, hidden), dt, 0.02), norm=1 + _normal(g, (hidden,), dt, 0.1),
                w_gate_up=_normal(g, (2 * inter, hidden), dt, 0.02), w_down=_normal(g, (hidden, inter), dt, 0.02))


def _model_inputs(case, seed):
    """Weights (stacked gate/up), the filled pool and the host lists of one engine step.  The
    embedding and the projections back onto the residual stream are scaled (1 and 0.02 / sqrt(2
    layers)) so that, as in a trained model, a layer adds to the stream without drowning it."""
    new, ctx = _sizes(case)
    table, blocks = _tables(ctx, 16, seed)
    g, dt, m = _generator(seed), torch.bfloat16, MODEL
    hd, inter, d = m["hidden_size"], m["intermediate_size"], MODEL_DIM
    qkv = (m["num_attention_heads"] + 2 * m["num_key_value_heads"]) * d
    back = 0.02 / math.sqrt(2 * m["num_hidden_layers"])
    embed = _normal(g, (m["vocab_size"], hd), dt)
    layers = [dict(input_norm=1 + _normal(g, (hd,), dt, 0.1), wqkv=_normal(g, (qkv, hd), dt, 0.02),
                   wo=_normal(g, (hd, m["num_attention_heads"] * d), dt, back),
                   post_norm=1 + _normal(g, (hd,), dt, 0.1), w_gate_up=_normal(g, (2 * inter, hd), dt, 0.02),
                   w_down=_normal(g, (hd, inter), dt, back)) for _ in range(m["num_hidden_layers"])]
    norm = 1 + _normal(g, (hd,), dt, 0.1)
    pool = GpuBlockPool.for_model(LlamaConfig(**m), blocks, 16, DEVICE, dt)
    pool.storage.normal_(generator=g)
    tokens = np.random.default_rng(seed).integers(0, m["vocab_size"], size=int(new.sum()))
    return dict(embed=embed, layers=layers, norm=norm, pool=pool, tokens=tokens, table=table, new=new, ctx=ctx)


# ------------------------------------------------------------- the calls ----


def prepare(case, seed):
    if case["kind"] == "mlp":
        i = _mlp_inputs(case, seed)
        rows, hidden, inter = case["rows"], case["hidden"], case["inter"]
        nbytes = max(linear_workspace_bytes(rows, hidden, hidden), linear_workspace_bytes(rows, hidden, inter))
        return dict(kind="mlp", x=i["x"], attn=i["attn"], wo=i["wo"], norm=i["norm"],
                    w_il=interleave_gate_up(i["w_gate_up"]), w_down=i["w_down"],
                    ws=torch.empty(nbytes, dtype=torch.uint8, device=DEVICE) if nbytes else None)
    if case["kind"] == "model":
        i = _model_inputs(case, seed)
        weights = LlamaWeights(i["embed"], [LayerWeights(**w) for w in i["layers"]], i["norm"], i["embed"])
        # "rg" holds the choice between equivalent forms fixed, so that a step's logits are the same
        # in every process.
        model = RailgunLlama(LlamaConfig(**MODEL), weights, i["pool"], max_position=int(i["ctx"].max()), choices="rg")
        return dict(kind="model", model=model, pool=i["pool"], step=DeviceStep.from_host(_pack(case, i), DEVICE))
    i = _attention_inputs(case, seed)
    h, hkv, d, bs = case["heads"], case["kv_heads"], case["head_dim"], case["block_size"]
    kernels = PagedAttentionKernels(0)
    state = dict(kind=case["kind"], op=PagedAttentionOp(1.0 / math.sqrt(d), h, hkv, d, bs, kernels),
                 q=i["q"], k=i["k"], v=i["v"], kc=i["kc"], vc=i["vc"], bt=_i32(i["table"]), cl=_i32(i["ctx"]),
                 pos=_i32(i["pos"]), slots=_i32(i["slots"]), max_ctx=int(i["ctx"].max()),
                 cos_sin=rope_cos_sin_table(int(i["ctx"].max()), d, THETA, torch.device(DEVICE)))
    if case["kind"] == "prefill":
        state.update(cu=_i32(np.concatenate([[0], np.cumsum(i["new"])])), max_len=int(i["new"].max()))
    if case["kind"] == "step":
        nbytes = kernels.v1_workspace_bytes(case["batch"], h, hkv, d, bs, int(state["bt"].shape[1]))
        state.update(ws=torch.empty(nbytes, dtype=torch.uint8, device=DEVICE), out=torch.empty_like(i["q"]))
    return state


def _pack(case, i):
    """The engine step: prompt chunks, then decode slots."""
    chunks, slots, at = [], [], 0
    for s, (n, c) in enumerate(zip(i["new"], i["ctx"])):
        blocks = [int(b) for b in i["table"][s, :(c + 15) // 16]]
        if s < case["prompts"]:
            chunks.append(PrefillChunk([int(t) for t in i["tokens"][at:at + n]], int(c - n), blocks))
        else:
            slots.append(DecodeSlot(int(i["tokens"][at]), int(c), blocks))
        at += int(n)
    return pack_step(chunks, slots, 16)


def run(state):
    kind, s = state["kind"], state
    if kind == "mlp":
        linear_residual(s["attn"], s["wo"], s["x"], s["ws"])
        act = linear_silu_mul(s["x"], s["w_il"], norm_weight=s["norm"], eps=EPS)
        linear_residual(act, s["w_down"], s["x"], s["ws"])
        return {"residual": s["x"], "act": act}
    if kind == "model":
        return {"logits": s["model"].forward(s["step"]), "pool": s["pool"].storage}
    op = s["op"]
    if kind == "step":
        op.kernels.launch_rope_reshape_and_cache_v1(
            s["q"], s["k"], s["v"], s["kc"], s["vc"], s["cos_sin"], s["pos"], s["slots"], s["bt"], s["cl"], s["out"],
            op.scale, op.num_heads, op.num_kv_heads, op.head_dim, op.block_size, s["bt"].shape[1], s["q"].shape[0],
            s["ws"])
        return {"out": s["out"], "k_cache": s["kc"], "v_cache": s["vc"]}
    op.rope_reshape_and_cache(s["q"], s["k"], s["v"], s["kc"], s["vc"], s["cos_sin"], s["pos"], s["slots"])
    if kind == "prefill":
        out = op.prefill_packed(s["q"], s["kc"], s["vc"], s["bt"], s["cl"], s["cu"], s["max_len"])
    else:
        out = op.execute(s["q"], s["kc"], s["vc"], s["bt"], s["cl"], None, s["max_ctx"])
    return {"out": out, "q": s["q"], "k_cache": s["kc"], "v_cache": s["vc"]}


# ------------------------------------------------- what a pass cannot do without ----


def _attention_work(new, ctx, h, hkv, d, bs, e):
    """Each cached row a sequence attends to read once per kv-head, the new k and v rows read and
    written, q read and the output written, the block-table entries and one cos/sin row per token;
    2 flops per multiply-add of QK^T and PV under the causal limit."""
    t = int(new.sum())
    rows = int((ctx - new).sum()) * hkv * d * 2 * e + t * hkv * d * 4 * e
    small = int(((ctx + bs - 1) // bs).sum()) * 4 + len(ctx) * 4 + t * (8 + 4 * d)
    keys = int((new * (ctx - new) + new * (new + 1) // 2).sum())
    return dict(bytes=rows + t * h * d * 2 * e + small, flops=4 * h * d * keys)


def work(case):
    if case["kind"] == "mlp":
        rows, hidden, inter = case["rows"], case["hidden"], case["inter"]
        weights = hidden * hidden + 3 * hidden * inter
        return dict(bytes=2 * (weights + hidden + rows * (3 * hidden + inter)), flops=2 * rows * weights)
    new, ctx = _sizes(case)
    if case["kind"] == "model":
        m, d = MODEL, MODEL_DIM
        hd, inter, t = m["hidden_size"], m["intermediate_size"], int(new.sum())
        layer = (m["num_attention_heads"] * 2 + 2 * m["num_key_value_heads"]) * d * hd + 3 * hd * inter
        a = _attention_work(new, ctx, m["num_attention_heads"], m["num_key_value_heads"], d, 16, 2)
        head, n = m["vocab_size"] * hd, m["num_hidden_layers"]
        # q and the attention output stay inside a layer: only the cache rows and tables count.
        cache = a["bytes"] - t * m["num_attention_heads"] * d * 4
        return dict(bytes=n * (2 * layer + 4 * hd + cache) + 2 * (head + hd) + 2 * t * hd + 2 * len(new) * m["vocab_size"],
                    flops=n * (2 * t * layer + a["flops"]) + 2 * len(new) * head)
    return _attention_work(new, ctx, case["heads"], case["kv_heads"], case["head_dim"], case["block_size"],
                           4 if case["dtype"] == "f32" else 2)


def tolerance(case):
    """About four times the error against 64 bits that was measured: the rounding of q, k, the
    probabilities and the output (and, in the model, of every layer's activations) to 16 bits;
    fp32 sums otherwise."""
    if case["kind"] == "model":
        return {"rel": 3e-2, "max": 0.3}
    if case["kind"] == "mlp":
        return {"rel": 2e-2, "max": 0.2} if case["dtype"] == "bf16" else {"rel": 3e-3, "max": 0.03}
    if case["dtype"] == "f32":
        return {"rel": 2e-6, "max": 5e-5}
    return {"rel": 1e-2, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 1.5e-3, "max": 0.015}


# ------------------------------------------------------ the same in 64 bits ----


def _rotate(x, pos, d):
    """RoPE of x [T, heads, d] at positions pos, halves rotated against each other."""
    inv = THETA ** (-torch.arange(0, d, 2, device=DEVICE, dtype=torch.float64) / d)
    ang = torch.from_numpy(np.asarray(pos, np.float64)).to(DEVICE)[:, None] * inv
    c, s = ang.cos()[:, None, :], ang.sin()[:, None, :]
    lo, hi = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)


def _attend(q, k, v, first):
    """Causal softmax attention of q [L, H, D] at positions first.. over k, v [n, H_kv, D]."""
    rows, h, d = q.shape
    n, hkv, _ = k.shape
    g = h // hkv
    out = torch.empty_like(q)
    keys = torch.arange(n, device=DEVICE)
    for r0 in range(0, rows, 1024):
        qr = q[r0:r0 + 1024]
        hide = keys[None, :] > (first + r0 + torch.arange(len(qr), device=DEVICE))[:, None]
        for kh in range(hkv):
            x = qr[:, kh * g:(kh + 1) * g].transpose(0, 1).reshape(-1, d) @ k[:, kh].t() / math.sqrt(d)
            p = x.view(g, len(qr), n).masked_fill_(hide, -math.inf).softmax(-1)
            out[r0:r0 + 1024, kh * g:(kh + 1) * g] = (p.view(-1, n) @ v[:, kh]).view(g, len(qr), d).transpose(0, 1)
    return out


def _cached(cache, blocks, n):
    """The first n rows [n, H_kv, D] behind a block-table row, in 64 bits."""
    c = cache[torch.from_numpy(blocks.astype(np.int64)).to(DEVICE)].double()
    return c.transpose(1, 2).reshape(-1, c.shape[1], c.shape[3])[:n]


def _attend_all(q, kn, vn, kc, vc, table, new, ctx, bs):
    """Attention of every sequence: cached rows from kc / vc, the new ones from kn / vn."""
    out, at = torch.empty_like(q), 0
    for s, (n, c) in enumerate(zip(new.tolist(), ctx.tolist())):
        blocks = table[s, :(c + bs - 1) // bs]
        k, v = _cached(kc, blocks, c), _cached(vc, blocks, c)
        k[c - n:], v[c - n:] = kn[at:at + n], vn[at:at + n]
        out[at:at + n] = _attend(q[at:at + n], k, v, c - n)
        at += n
    return out


def _with_rows(cache, rows, slots, bs):
    """The cache in 64 bits after the rows are written to their slots."""
    c = cache.double()
    slots = torch.from_numpy(np.asarray(slots, np.int64)).to(DEVICE)
    c[slots // bs, :, slots % bs] = rows
    return c


def _exact_mlp(case, seed):
    i = {n: t.double() for n, t in _mlp_inputs(case, seed).items()}
    x = i["x"] + i["attn"] @ i["wo"].t()
    act = _silu_mul(_rms(x, i["norm"]) @ i["w_gate_up"].t())
    return {"residual": x + act @ i["w_down"].t(), "act": act}


def _rms(x, w):
    return x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt() * w


def _silu_mul(y):
    gate, up = y.chunk(2, -1)
    return gate * gate.sigmoid() * up


def _exact_model(case, seed):
    i, m, d = _model_inputs(case, seed), MODEL, MODEL_DIM
    h, hkv = m["num_attention_heads"], m["num_key_value_heads"]
    new, ctx, store = i["new"], i["ctx"], i["pool"].storage
    pos = np.concatenate([np.arange(c - n, c) for n, c in zip(new, ctx)])
    slots = i["table"][np.repeat(np.arange(len(new)), new), pos // 16].astype(np.int64) * 16 + pos % 16
    x = i["embed"][torch.from_numpy(i["tokens"]).to(DEVICE)].double()
    pool = torch.empty(store.shape, device=DEVICE, dtype=torch.float64)
    for l, w in enumerate(i["layers"]):
        y = (_rms(x, w["input_norm"].double()) @ w["wqkv"].double().t()).view(len(pos), h + 2 * hkv, d)
        q, k, v = _rotate(y[:, :h], pos, d), _rotate(y[:, h:h + hkv], pos, d), y[:, h + hkv:]
        a = _attend_all(q, k, v, store[l, :, 0], store[l, :, 1], i["table"], new, ctx, 16)
        pool[l, :, 0], pool[l, :, 1] = _with_rows(store[l, :, 0], k, slots, 16), _with_rows(store[l, :, 1], v, slots, 16)
        x = x + a.reshape(len(pos), h * d) @ w["wo"].double().t()
        x = x + _silu_mul(_rms(x, w["post_norm"].double()) @ w["w_gate_up"].double().t()) @ w["w_down"].double().t()
    last = torch.from_numpy(np.cumsum(new) - 1).to(DEVICE)
    return {"logits": _rms(x, i["norm"].double())[last] @ i["embed"].double().t(), "pool": pool}


def exact(case, seed):
    if case["kind"] == "mlp":
        return _exact_mlp(case, seed)
    if case["kind"] == "model":
        return _exact_model(case, seed)
    i, d, bs = _attention_inputs(case, seed), case["head_dim"], case["block_size"]
    q, k, v = _rotate(i["q"].double(), i["pos"], d), _rotate(i["k"].double(), i["pos"], d), i["v"].double()
    out = _attend_all(q, k, v, i["kc"], i["vc"], i["table"], i["new"], i["ctx"], bs)
    found = {"out": out, "k_cache": _with_rows(i["kc"], k, i["slots"], bs),
             "v_cache": _with_rows(i["vc"], v, i["slots"], bs)}
    return found if case["kind"] == "step" else dict(found, q=q)
