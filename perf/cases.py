"""The workloads by which this framework's speed is judged, each run through a public entry point on the GPU.

- listed()            named cases: what a decoding server and a training run of this model ask of the framework
- draw(rng)           one more case of the same ranges (odd sizes, other head shapes, windows, contexts)
- prepare(case, seed) what the caller holds before the call: inputs made from the seed, weights, caches, a decoder
- run(state)          one pass; returns the pass's whole outputs
- work(case)          bytes and flops one pass cannot do without
- tolerance(case)     the largest relative error another correct implementation at the same precision shows
- exact(case, seed)   run's outputs in float64 plain torch (None where there is no such value)

Kinds of case:

  decode    one decode step of a batch of sequences (attention.decode_step): QK norm + RoPE, fp8 append, attention
  prefill   a chunk of prompt tokens per sequence (qk_norm_rope_append, then prefill_attention)
  attention the training block (torch.ops.nanochat_amd.attention), forward and backward
  flash     the training attention alone (flash_attn_fwd, flash_attn_bwd), forward and backward
  rows      the training prologue and value-embedding gate (qk_forward, ve_forward and their backwards)
  steps     a decoder serving full slots: several greedy steps, then the logits
  prompts   a decoder given new prompts: prefill, the first token's step, the logits
"""
import math

import torch

from nanochat_amd import attention, attention_op, flash_attn, qk_prologue, ve_gate
from nanochat_amd.decoder import DecoderRuntime
from nanochat_amd.kv_cache import PagedKVCache, contiguous_block_table, pages_for
from nanochat_amd.rotary import rotary_tables
from nanochat_amd.workloads import model_tensors

DEVICE = "cuda"
D = 128
EPS = torch.finfo(torch.float32).eps
SOFTCAP = 15.0


def listed():
    return [
        # One user generating: a single sequence, the small model's 6 heads, 1,024 cached tokens. Latency is all.
        dict(name="decode_one", kind="decode", batch=1, q_heads=6, kv_heads=6, ctx=1024, ctx_min=1024, paged=False,
             outliers=False, window=-1, ve=False),
        # The headline: a full batch at its longest context, grouped-query heads, a fragmented page pool.
        dict(name="decode_bs64_8k", kind="decode", batch=64, q_heads=16, kv_heads=4, ctx=8192, ctx_min=8192,
             paged=True, outliers=True, window=-1, ve=False),
        # The same server in mid-flight: every sequence at a length of its own, 512 to 8,192 tokens.
        dict(name="decode_ragged", kind="decode", batch=64, q_heads=16, kv_heads=4, ctx=8192, ctx_min=512, paged=True,
             outliers=True, window=-1, ve=False),
        # A d20 model's sliding-window layer with value embeddings: half a batch of 4,096-token contexts, 1,024 seen.
        dict(name="decode_window_ve", kind="decode", batch=32, q_heads=10, kv_heads=10, ctx=4096, ctx_min=4096,
             paged=True, outliers=False, window=1024, ve=True),
        # Chunked prefill beside decoding: 512-token chunks of eight prompts onto 3,584 cached tokens each.
        dict(name="prefill_chunk", kind="prefill", batch=8, q_heads=16, kv_heads=4, ctx=3584, chunk=512, window=-1),
        # New prompts of no round length, nothing cached, on a windowed layer of the 13-head model.
        dict(name="prefill_prompt", kind="prefill", batch=3, q_heads=13, kv_heads=13, ctx=0, chunk=1501, window=700),
        # A training step's attention block at the training shape: 32 x 2,048 tokens, 6 heads, value embeddings.
        dict(name="train_block", kind="attention", batch=32, seqlen=2048, heads=6, window=2048, docs=1, ve=True),
        # Packed documents of mixed lengths, a sliding window, a wider model, no value embeddings.
        dict(name="train_docs", kind="attention", batch=5, seqlen=1999, heads=10, window=512, docs=7, ve=False),
        # Long-context training: the attention alone over two 8,192-token documents.
        dict(name="flash_long", kind="flash", segments=2, seqlen=8192, heads=6, window=-1),
        # The memory-bound rest of a small training step: prologue and value-embedding gate of 4 x 1,024 tokens.
        dict(name="train_rows", kind="rows", batch=4, seqlen=1024, heads=6, vocab=65536),
        # End-to-end decoding at full load: 26 layers, d1664, 128 slots at 2,048-token prompts; eight greedy steps.
        dict(name="decoder_steps", kind="steps", layers=26, hidden=1664, vocab=65536, batch=128, prompt=2048, steps=8,
             ve_every=0, window=-1),
        # Time to first token: six new prompts of mixed lengths on a 12-layer d768 model with value embeddings and
        # windowed layers, half of them sampled.
        dict(name="decoder_prompts", kind="prompts", layers=12, hidden=768, vocab=65536, batch=6, prompt=1100,
             ve_every=2, window=512),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_decode(rng):
    hq, hkv = rng.choice([(6, 6), (10, 10), (13, 13), (16, 4), (8, 1), (12, 4)])
    batch, ctx = _log_int(rng, 1, 64), _log_int(rng, 16, 8192)
    while batch * hkv * ctx > 64 * 4 * 8192:
        ctx = max(16, ctx // 2 + rng.randint(0, 15))
    return dict(kind="decode", batch=batch, q_heads=hq, kv_heads=hkv, ctx=ctx,
                ctx_min=rng.choice([ctx, max(1, ctx // 16)]), paged=rng.random() < 0.7, outliers=rng.random() < 0.5,
                window=rng.choice([-1, -1, 256, 1024]), ve=rng.random() < 0.3)


def _draw_prefill(rng):
    hq, hkv = rng.choice([(6, 6), (10, 10), (13, 13), (16, 4), (8, 2)])
    batch, chunk, ctx = _log_int(rng, 1, 8), _log_int(rng, 24, 2000), rng.choice([0, _log_int(rng, 16, 6000)])
    while batch * hq * chunk * (ctx + chunk) > 8 * 16 * 512 * 4096:
        ctx, chunk = ctx // 2, max(24, chunk * 3 // 4)
    return dict(kind="prefill", batch=batch, q_heads=hq, kv_heads=hkv, ctx=ctx, chunk=chunk,
                window=rng.choice([-1, -1, 300, 1024]))


def _draw_attention(rng):
    batch, seqlen = _log_int(rng, 1, 32), _log_int(rng, 128, 2048)
    return dict(kind="attention", batch=batch, seqlen=seqlen, heads=rng.choice([4, 6, 6]),
                window=rng.choice([seqlen, seqlen, max(16, seqlen // 4)]), docs=rng.choice([1, 1, 5, 12]),
                ve=rng.random() < 0.5)


def _draw_flash(rng):
    segments, seqlen, heads = _log_int(rng, 1, 16), _log_int(rng, 64, 8192), rng.choice([1, 4, 6, 10])
    while segments * heads * seqlen * seqlen > 2 * 6 * 8192 * 8192:
        seqlen = seqlen * 3 // 4
    return dict(kind="flash", segments=segments, seqlen=seqlen, heads=heads,
                window=rng.choice([-1, -1, max(1, seqlen // 8), 512]))


def _draw_rows(rng):
    return dict(kind="rows", batch=_log_int(rng, 1, 32), seqlen=_log_int(rng, 64, 2048), heads=rng.choice([4, 6, 10]),
                vocab=rng.choice([4096, 65536]))


def _draw_decoder(rng):
    hidden = rng.choice([768, 1280, 1664])
    if rng.random() < 0.5:
        return dict(kind="steps", layers=rng.randint(2, 8), hidden=hidden, vocab=rng.choice([32768, 65536]),
                    batch=_log_int(rng, 1, 128), prompt=_log_int(rng, 32, 2048), steps=8,
                    ve_every=rng.choice([0, 2]), window=rng.choice([-1, 512]))
    return dict(kind="prompts", layers=rng.randint(2, 8), hidden=hidden, vocab=rng.choice([32768, 65536]),
                batch=_log_int(rng, 1, 16), prompt=_log_int(rng, 32, 2048), ve_every=rng.choice([0, 2]),
                window=rng.choice([-1, 512]))


def draw(rng):
    kinds = [_draw_decode, _draw_decode, _draw_prefill, _draw_prefill, _draw_attention, _draw_attention, _draw_flash,
             _draw_flash, _draw_rows, _draw_decoder]
    return rng.choice(kinds)(rng)


# --- inputs

def _generator(seed, device=DEVICE):
    return torch.Generator(device=device).manual_seed(seed)


def _randn(gen, *shape, dtype=torch.bfloat16, scale=1.0):
    return (torch.randn(*shape, generator=gen, device=gen.device, dtype=torch.float32) * scale).to(dtype)


def _gain(gen):
    return 1.0 + 0.1 * torch.randn(D, generator=gen, device=gen.device, dtype=torch.float32)


def _with_outliers(gen, x):
    """One value in a hundred replaced by 8 standard deviations, as trained K and V caches show."""
    mask = torch.rand(x.shape, generator=gen, device=x.device) < 0.01
    return torch.where(mask, (8.0 * torch.sign(x.float())).to(x.dtype), x)


def _page_table(gen, batch, max_pages, paged):
    if not paged:
        return contiguous_block_table(batch, max_pages, device=DEVICE)
    return torch.randperm(batch * max_pages, generator=gen, device=DEVICE).to(torch.int32).view(batch, max_pages)


def _decode_inputs(c, seed):
    gen = _generator(seed)
    B, Hq, Hkv, ctx = c["batch"], c["q_heads"], c["kv_heads"], c["ctx"]
    ctx_lens = torch.full((B,), ctx, dtype=torch.int32, device=DEVICE)
    if c["ctx_min"] < ctx:
        ctx_lens = torch.randint(c["ctx_min"], ctx + 1, (B,), generator=gen, device=DEVICE, dtype=torch.int32)
    k, v = _randn(gen, B, ctx, Hkv, D), _randn(gen, B, ctx, Hkv, D)
    if c["outliers"]:
        k, v = _with_outliers(gen, k), _with_outliers(gen, v)
    qkv = _randn(gen, B, (Hq + 2 * Hkv) * D)
    q_gain, k_gain = _gain(gen), _gain(gen)
    table = _page_table(gen, B, pages_for(ctx + 1), c["paged"])
    cos, sin = rotary_tables(ctx + 1, device=DEVICE)
    ve = None
    if c["ve"]:
        C, vocab = Hkv * D, 4096
        ve = (_randn(gen, B, C), _randn(gen, vocab, C), _randn(gen, Hkv, C, dtype=torch.float32, scale=0.05),
              torch.randint(0, vocab, (B,), generator=gen, device=DEVICE, dtype=torch.int32))
    return dict(ctx_lens=ctx_lens, k=k, v=v, qkv=qkv, q_gain=q_gain, k_gain=k_gain, table=table, cos=cos, sin=sin,
                ve=ve)


def _prefill_inputs(c, seed):
    gen = _generator(seed)
    B, Hq, Hkv, ctx, T = c["batch"], c["q_heads"], c["kv_heads"], c["ctx"], c["chunk"]
    k, v = _randn(gen, B, ctx, Hkv, D), _randn(gen, B, ctx, Hkv, D)
    qkv = _randn(gen, B, T, (Hq + 2 * Hkv) * D)
    q_gain, k_gain = _gain(gen), _gain(gen)
    table = _page_table(gen, B, pages_for(ctx + T), True)
    cos, sin = rotary_tables(ctx + T, 10000.0, DEVICE)
    return dict(k=k, v=v, qkv=qkv, q_gain=q_gain, k_gain=k_gain, table=table, cos=cos, sin=sin)


def _documents(c):
    """Token offsets of the packed documents: `docs` a row of the batch (1: the row itself), of unequal lengths, the
    first of them one token long when there are several; a document never crosses a row."""
    B, T, n = c["batch"], c["seqlen"], c["docs"]
    marks = [0] + ([1] if n > 1 else []) + [max(2, T * i * i // (n * n)) for i in range(2, n)]
    marks = sorted(set(m for m in marks if m < T))
    return [b * T + m for b in range(B) for m in marks] + [B * T]


def _attention_inputs(c, seed):
    gen = _generator(seed)
    B, T, H = c["batch"], c["seqlen"], c["heads"]
    C, vocab = H * D, 65536
    cos, sin = rotary_tables(T, device=DEVICE)
    p = dict(qkv=_randn(gen, B, T, 3 * C), q_gain=_gain(gen), k_gain=_gain(gen), cos=cos, sin=sin,
             o_weight=_randn(gen, C, C, scale=C ** -0.5), residual=_randn(gen, B, T, C), dh=_randn(gen, B, T, C))
    bounds = _documents(c)
    p["cu"] = torch.tensor(bounds + [bounds[-1]] * 2, dtype=torch.int32, device=DEVICE)   # a padded buffer
    p["segments"] = torch.tensor(len(bounds) - 1)
    p["bounds"] = bounds
    p["n"] = p["ids"] = p["table"] = p["w_gate"] = None
    if c["ve"]:
        p["n"] = _randn(gen, B, T, C)
        p["ids"] = _tokens(gen, B, T, vocab)
        p["table"] = _randn(gen, vocab, C, dtype=torch.float32)
        p["w_gate"] = _randn(gen, H, C, dtype=torch.float32, scale=0.05)
    return p


def _tokens(gen, B, T, vocab):
    """Token ids with text's skew: a few frequent ones, a long tail."""
    u = torch.rand(B, T, generator=gen, device=DEVICE, dtype=torch.float64)
    return (vocab ** u - 1).clamp(0, vocab - 1).to(torch.int32)


def _flash_inputs(c, seed):
    gen = _generator(seed)
    total, H = c["segments"] * c["seqlen"], c["heads"]
    q, k, v, do = (_randn(gen, total, H, D) for _ in range(4))
    cu = torch.arange(0, total + 1, c["seqlen"], dtype=torch.int32, device=DEVICE)
    return dict(q=q, k=k, v=v, do=do, cu=cu)


def _rows_inputs(c, seed):
    gen = _generator(seed)
    B, T, H, vocab = c["batch"], c["seqlen"], c["heads"], c["vocab"]
    C = H * D
    cos, sin = rotary_tables(T, device=DEVICE)
    p = dict(qkv=_randn(gen, B, T, 3 * C), dqn=_randn(gen, B, T, H, D), dkn=_randn(gen, B, T, H, D),
             dvm=_randn(gen, B, T, H, D), q_gain=_gain(gen), k_gain=_gain(gen), cos=cos, sin=sin,
             n=_randn(gen, B, T, C), ids=_tokens(gen, B, T, vocab), table=_randn(gen, vocab, C, dtype=torch.float32),
             w_gate=_randn(gen, H, C, dtype=torch.float32, scale=0.05))
    return p


def _windows(c, max_length):
    """Three windowed layers, then one that sees everything, and the last always does."""
    L, w = c["layers"], c["window"]
    return [w if w >= 0 and l % 4 != 3 and l != L - 1 else max_length for l in range(L)]


def _model(c, seed, max_length):
    """Random-init layers under an lm_head that predicts, for every token, one definite next token by a clear margin,
    as a trained model's does: row next(t) of the head is t's embedding, scaled to logits of the cap's size."""
    ve_layers = tuple(range(0, c["layers"], c["ve_every"])) if c["ve_every"] else ()
    m = model_tensors(c["layers"], c["hidden"], 4 * c["hidden"], c["vocab"], max_length, seed=seed, softcap=SOFTCAP,
                      ve_layers=ve_layers, windows=_windows(c, max_length), device=DEVICE, generator_device=DEVICE)
    unit = m.wte / m.wte.square().mean(-1, keepdim=True).sqrt()
    follow = torch.randperm(c["vocab"] - 1, generator=_generator(seed + 1), device=DEVICE) + 1   # never BOS
    m.lm_head[follow] = (unit[1:] * (42.0 / c["hidden"])).to(torch.bfloat16)
    m.lm_head[0] = 0
    return m


def _prompt_lengths(c):
    """Mixed lengths around `prompt`, odd ones among them, the longest 1.5 times it."""
    n, p = c["batch"], c["prompt"]
    return [max(2, p // 2 + (p * i) // max(1, n - 1) if n > 1 else p) for i in range(n)]


def _steps_left(c):
    return 512 // c["steps"]


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "decode":
        p = _decode_inputs(c, seed)
        cache = PagedKVCache(p["table"].numel(), c["kv_heads"], DEVICE)
        cache.append(p["k"], p["v"], torch.zeros_like(p["ctx_lens"]), p["table"], num_new=p["ctx_lens"])
        del p["k"], p["v"]
        return dict(p, kind=kind, case=c, cache=cache, seq_lens=p["ctx_lens"] + 1)
    if kind == "prefill":
        p = _prefill_inputs(c, seed)
        cache = PagedKVCache(p["table"].numel(), c["kv_heads"], DEVICE)
        start = torch.full((c["batch"],), c["ctx"], dtype=torch.int32, device=DEVICE)
        if c["ctx"]:
            cache.append(p["k"], p["v"], torch.zeros_like(start), p["table"])
        del p["k"], p["v"]
        return dict(p, kind=kind, case=c, cache=cache, start=start)
    if kind == "attention":
        p = _attention_inputs(c, seed)
        p["leaves"] = [p[k] for k in ("qkv", "q_gain", "k_gain", "residual") + (("n", "w_gate") if c["ve"] else ())]
        for t in p["leaves"]:
            t.requires_grad_(True)
        p["o_grad"] = torch.zeros_like(p["o_weight"], dtype=torch.float32)
        p["sorted_ids"] = p["order"] = None
        if c["ve"]:
            p["table"].grad = torch.zeros_like(p["table"])
            p["sorted_ids"], p["order"] = p["ids"].flatten().sort(stable=True)
        return dict(p, kind=kind, case=c)
    if kind == "flash":
        return dict(_flash_inputs(c, seed), kind=kind, case=c)
    if kind == "rows":
        p = _rows_inputs(c, seed)
        p["table"].grad = torch.zeros_like(p["table"])
        p["sorted_ids"], p["order"] = p["ids"].flatten().sort(stable=True)
        p["dqkv"] = torch.zeros_like(p["qkv"])
        _heads(p["dqkv"], c["heads"])[2].copy_(p["dvm"])   # where the attention's backward leaves v's gradient
        return dict(p, kind=kind, case=c)
    gen = _generator(seed + 2, "cpu")
    if kind == "steps":
        max_length = c["prompt"] + 512
        rt = DecoderRuntime(_model(c, seed, max_length), bos_token_id=0, max_length=max_length, max_slots=c["batch"])
        prompts = torch.randint(1, c["vocab"], (c["batch"], c["prompt"]), generator=gen)
        prompts[:, 0] = 0
        prompts = prompts.tolist()
        for b, ids in enumerate(prompts):
            rt.place(b, ids)
        rt.prefill()
        rt.activate(range(c["batch"]))
        return dict(kind=kind, case=c, rt=rt, prompts=prompts, left=_steps_left(c))
    lengths = _prompt_lengths(c)
    max_length = max(lengths) + 16
    rt = DecoderRuntime(_model(c, seed, max_length), bos_token_id=0, max_length=max_length, max_slots=c["batch"])
    prompts = [[0] + torch.randint(1, c["vocab"], (n - 1,), generator=gen).tolist() for n in lengths]
    return dict(kind=kind, case=c, rt=rt, prompts=prompts)


# --- one pass

def _heads(qkv, H):
    return qkv.unflatten(-1, (3, H, D)).unbind(2)


def run(state):
    s, c = state, state["case"]
    if s["kind"] == "decode":
        out = attention.decode_step(s["qkv"], c["q_heads"], s["cache"], s["table"], s["seq_lens"], s["q_gain"],
                                    s["k_gain"], s["cos"], s["sin"], c["ctx"] + 1, window=c["window"], ve=s["ve"])
        return [out, s["cache"].k_pages, s["cache"].v_pages, s["cache"].kv_scale]
    if s["kind"] == "prefill":
        q = attention.qk_norm_rope_append(s["qkv"], c["q_heads"], s["cache"], s["table"], s["start"], s["q_gain"],
                                          s["k_gain"], s["cos"], s["sin"])
        out = attention.prefill_attention(q, s["cache"], s["table"], s["start"], window=c["window"])
        return [out, q, s["cache"].k_pages, s["cache"].v_pages, s["cache"].kv_scale]
    if s["kind"] == "attention":
        s["o_grad"].zero_()
        if c["ve"]:
            s["table"].grad.zero_()
        h, rstd, *_ = attention_op.attention(
            s["qkv"], s["q_gain"], s["k_gain"], s["cos"], s["sin"], c["window"], s["cu"], s["segments"],
            s["o_weight"], s["o_grad"], s["residual"], s["n"], s["ids"], s["table"], s["w_gate"], s["sorted_ids"],
            s["order"])
        grads = torch.autograd.grad(h, s["leaves"], s["dh"])
        return [h.detach(), rstd, *grads, s["o_grad"]] + ([s["table"].grad] if c["ve"] else [])
    if s["kind"] == "flash":
        window = None if c["window"] < 0 else c["window"]
        out, lse = flash_attn.flash_attn_fwd(s["q"], s["k"], s["v"], s["cu"], c["seqlen"], window_left=window)
        dq, dk, dv = flash_attn.flash_attn_bwd(s["q"], s["k"], s["v"], out, s["do"], lse, s["cu"], c["seqlen"],
                                               window_left=window)
        return [out, lse, dq, dk, dv]
    if s["kind"] == "rows":
        H = c["heads"]
        s["table"].grad.zero_()
        q, k, v = _heads(s["qkv"], H)
        dq, dk, dv = _heads(s["dqkv"], H)
        qn, kn = qk_prologue.qk_forward(q, k, s["q_gain"], s["k_gain"], s["cos"], s["sin"])
        vm, gate = ve_gate.ve_forward(s["n"], v, s["ids"], s["table"], s["w_gate"])
        dqg, dkg = qk_prologue.qk_backward(q, k, s["q_gain"], s["k_gain"], s["dqn"], s["dkn"], s["cos"], s["sin"], dq,
                                           dk)
        dn, dw = ve_gate.ve_backward(dv, s["n"], s["sorted_ids"], s["order"], s["table"], s["w_gate"], gate)
        return [qn, kn, vm, gate, s["dqkv"], dqg, dkg, dn, dw, s["table"].grad]
    rt = s["rt"]
    if s["kind"] == "steps":
        if s["left"] == 0:   # the context is full: the slots go back to the end of their prompts
            for b, ids in enumerate(s["prompts"]):
                rt.lib.dec_set_prompt(rt.handle, b, ids[-1], len(ids) - 1, 0.0, 1.0, 0)
            s["left"] = _steps_left(c)
        s["left"] -= 1
        for _ in range(c["steps"]):
            tokens = rt.step()
        return [tokens.copy(), rt.logits(c["batch"])]
    for b, ids in enumerate(s["prompts"]):
        rt.place(b, ids, temperature=0.8 if b % 2 else 0.0, top_p=0.9 if b % 4 == 3 else 1.0, seed=b)
    rt.prefill()
    rt.activate(range(c["batch"]))
    tokens = rt.step()
    return [tokens.copy(), rt.logits(c["batch"])]


# --- what a pass cannot do without

def _visible(T, window, ctx=0):
    """(query, key) pairs of T rows at positions ctx .. that see every key back to `window` before them."""
    w = window if window >= 0 else ctx + T
    return sum(min(ctx + i, w) + 1 for i in range(T))


def _lengths(c):
    return [c["ctx"]] if c["ctx_min"] == c["ctx"] else [(c["ctx_min"] + c["ctx"]) / 2]


def work(case):
    c, kind = case, case["kind"]
    if kind == "decode":
        B, Hq, Hkv = c["batch"], c["q_heads"], c["kv_heads"]
        n = _lengths(c)[0] + 1
        keys = B * (min(n, c["window"] + 1) if c["window"] >= 0 else n)
        nbytes = keys * Hkv * 264 + B * (2 * Hq * 256 + 2 * Hkv * 256 + Hkv * 264) + keys // 4
        if c["ve"]:
            nbytes += B * Hkv * D * 4 + Hkv * Hkv * D * 4
        return dict(bytes=nbytes, flops=4 * D * keys * Hq)
    if kind == "prefill":
        B, Hq, Hkv, T, ctx = c["batch"], c["q_heads"], c["kv_heads"], c["chunk"], c["ctx"]
        seen = min(ctx, c["window"]) if c["window"] >= 0 else ctx
        nbytes = B * (T * (Hq + 2 * Hkv) * 256 + T * Hq * 512 + (T + seen) * Hkv * 264)
        return dict(bytes=nbytes, flops=4 * D * B * Hq * _visible(T, c["window"], ctx))
    if kind == "attention":
        B, T, H = c["batch"], c["seqlen"], c["heads"]
        C, N = H * D, B * T
        bounds = _documents(c)
        window = -1 if c["window"] >= T else c["window"]
        pairs = sum(_visible(b - a, window) for a, b in zip(bounds, bounds[1:]))
        # forward: qkv, residual in, h, rstd out; backward: dh, qkv in, dqkv out; the weight and its gradient
        nbytes = N * (6 * C + 2 * C + 2 * C + 4 + 2 * C + 6 * C + 6 * C) + C * C * (2 + 2 + 8)
        if c["ve"]:
            rows = min(N, 65536)
            nbytes += N * (2 * C + 2 * C + 2 * C + 16) + rows * 4 * C * 4
        return dict(bytes=nbytes, flops=3.5 * 4 * D * pairs * H + 6 * N * C * C)
    if kind == "flash":
        N, H = c["segments"] * c["seqlen"], c["heads"]
        pairs = c["segments"] * _visible(c["seqlen"], c["window"])
        return dict(bytes=N * H * (4 * 256 + 8 * 256 + 8), flops=3.5 * 4 * D * pairs * H)
    if kind == "rows":
        N, H = c["batch"] * c["seqlen"], c["heads"]
        C, rows = H * D, min(N, c["vocab"])
        forward = N * (6 * C + 2 * C + 6 * C + 4 * H + 4) + rows * 4 * C
        backward = N * (4 * C + 4 * C + 4 * C + 4 * C + 2 * C + 4 * H + 12 + 2 * C) + rows * 12 * C
        return dict(bytes=forward + backward + c["vocab"] * C * 4, flops=12 * N * H * C)
    C, L, V, B = c["hidden"], c["layers"], c["vocab"], c["batch"]
    weights, H = 12 * C * C * L, C // D
    full = [l for l, w in enumerate(_windows(c, 1 << 30)) if w >= 1 << 30]
    if kind == "steps":
        n = c["prompt"] + 256
        seen = B * (len(full) * n + (L - len(full)) * min(n, c["window"] + 1))
        per = 2 * (weights + V * C) + seen * H * 264 + B * V * 4
        return dict(bytes=c["steps"] * per, flops=c["steps"] * (2 * B * (weights + V * C) + 4 * D * seen * H))
    lengths = _prompt_lengths(c)
    rows = sum(lengths)
    pairs = sum(len(full) * _visible(n, -1) + (L - len(full)) * _visible(n, c["window"]) for n in lengths)
    return dict(bytes=2 * (weights + V * C) + rows * L * H * 264 + rows * C * 4 + B * V * 4,
                flops=2 * rows * weights + 2 * B * V * C + 4 * D * pairs * H)


def tolerance(case):
    """About four times what each path's outputs are off from float64 (measured: decode and prefill 0.005, the block
    0.0045, the attention alone 0.0024, the row kernels 0.0017: bf16 results of bf16 products). A whole decoder carries
    each layer's bf16 and fp8 roundings through all that follow. Cache bytes and codes are exact."""
    return {"decode": dict(rel=1.5e-2, max=0.3, differ=0.0), "prefill": dict(rel=1.5e-2, max=0.3, differ=0.0),
            "attention": dict(rel=1.5e-2, max=0.5, differ=0.0), "flash": dict(rel=1e-2, max=0.4, differ=0.0),
            "rows": dict(rel=7e-3, max=0.2, differ=0.0), "steps": dict(rel=3e-2, max=0.95, differ=0.01),
            "prompts": dict(rel=3e-2, max=0.95, differ=0.01)}[case["kind"]]


# --- the same in float64

def _quantized(x):
    """What the cache holds of x [..., 128]: e4m3fn codes of x / scale, scale = max|x| / 448 a row in fp32 (1 for a
    zero row), times the scale; float64."""
    amax = x.float().abs().amax(-1, keepdim=True)
    scale = torch.where(amax > 0, amax / 448.0, torch.ones_like(amax))
    codes = (x.float() / scale).clamp(-448, 448).to(torch.float8_e4m3fn)
    return codes.double() * scale.double()


def _norm_rope(x, gain, cos, sin):
    """x [..., 128] float64, cos and sin broadcastable to [..., 64]."""
    y = x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * gain.double()
    a, b = y[..., :64], y[..., 64:]
    c, s = cos.double(), sin.double()
    return torch.cat([a * c + b * s, b * c - a * s], -1)


def _bf16(x):
    return x.to(torch.bfloat16).double()


def _softmax_av(q, k, v, mask):
    """q [H, T, 128], k and v [H, K, 128], mask [T, K] -> [H, T, 128], all float64."""
    scores = (q @ k.transpose(-1, -2)) * D ** -0.5
    scores = scores.masked_fill(~mask, float("-inf"))
    return torch.softmax(scores, -1) @ v


def _exact_decode(c, seed):
    p = _decode_inputs(c, seed)
    B, Hq, Hkv = c["batch"], c["q_heads"], c["kv_heads"]
    G = Hq // Hkv
    x = p["qkv"].double().view(B, Hq + 2 * Hkv, D)
    out = torch.empty(B, Hq, D, dtype=torch.float64, device=DEVICE)
    for b in range(B):
        n = int(p["ctx_lens"][b])
        cos, sin = p["cos"][n], p["sin"][n]
        q = _bf16(_norm_rope(x[b, :Hq], p["q_gain"], cos, sin))
        k = _bf16(_norm_rope(x[b, Hq:Hq + Hkv], p["k_gain"], cos, sin))
        v = x[b, Hq + Hkv:]
        if p["ve"] is not None:
            h, table, gate, tokens = p["ve"]
            g = 2 * torch.sigmoid(gate.double() @ h[b].double())
            v = v + g[:, None] * table[tokens[b]].double().view(Hkv, D)
        lo = max(n - c["window"], 0) if c["window"] >= 0 else 0
        keys = torch.cat([_quantized(p["k"][b, lo:n]), _quantized(k)[None]]).transpose(0, 1)
        values = torch.cat([_quantized(p["v"][b, lo:n]), _quantized(v)[None]]).transpose(0, 1)
        mask = torch.ones(G, n + 1 - lo, dtype=torch.bool, device=DEVICE)
        out[b] = _softmax_av(q.view(Hkv, G, D), keys, values, mask).reshape(Hq, D)
    return [out, None, None, None]


def _exact_prefill(c, seed):
    p = _prefill_inputs(c, seed)
    B, Hq, Hkv, ctx, T = c["batch"], c["q_heads"], c["kv_heads"], c["ctx"], c["chunk"]
    G = Hq // Hkv
    x = p["qkv"].view(B, T, Hq + 2 * Hkv, D)
    out = torch.empty(B, T, Hq, D, dtype=torch.float64, device=DEVICE)
    qs = torch.empty_like(out)
    cos, sin = p["cos"][ctx:ctx + T, None], p["sin"][ctx:ctx + T, None]
    i = torch.arange(T, device=DEVICE)[:, None] + ctx
    j = torch.arange(ctx + T, device=DEVICE)[None]
    mask = (j <= i) & ((i - j <= c["window"]) if c["window"] >= 0 else (j >= 0))
    for b in range(B):
        row = x[b].double()
        qs[b] = _norm_rope(row[:, :Hq], p["q_gain"], cos, sin)
        k = _bf16(_norm_rope(row[:, Hq:Hq + Hkv], p["k_gain"], cos, sin))
        keys = torch.cat([_quantized(p["k"][b]), _quantized(k)]).transpose(0, 1)
        values = torch.cat([_quantized(p["v"][b]), _quantized(row[:, Hq + Hkv:])]).transpose(0, 1)
        for h in range(Hkv):
            q = _bf16(qs[b, :, h * G:(h + 1) * G]).transpose(0, 1)
            out[b, :, h * G:(h + 1) * G] = _softmax_av(q, keys[h], values[h], mask).transpose(0, 1)
    return [out, qs, None, None, None]


def _attend_documents(q, k, v, bounds, window):
    """q, k, v [N, H, 128] float64 -> (out, lse [H, N]), causal inside each document, keys at distance <= window."""
    outs, lses = [], []
    for a, b in zip(bounds, bounds[1:]):
        i = torch.arange(b - a, device=q.device)
        mask = (i[None] <= i[:, None]) & (i[:, None] - i[None] <= window)
        s = (q[a:b].transpose(0, 1) @ k[a:b].permute(1, 2, 0)) * D ** -0.5
        s = s.masked_fill(~mask, float("-inf"))
        lse = torch.logsumexp(s, -1)
        lses.append(lse)
        outs.append((torch.exp(s - lse[..., None]) @ v[a:b].transpose(0, 1)).transpose(0, 1))
    return torch.cat(outs), torch.cat(lses, 1)


def _exact_attention(c, seed):
    p = _attention_inputs(c, seed)
    B, T, H = c["batch"], c["seqlen"], c["heads"]
    C = H * D
    q_gain, k_gain = p["q_gain"].double().requires_grad_(), p["k_gain"].double().requires_grad_()
    o_weight = p["o_weight"].double().requires_grad_()
    leaves = [q_gain, k_gain, o_weight]
    if c["ve"]:
        w_gate = p["w_gate"].double().requires_grad_()
        table = _bf16(p["table"]).requires_grad_()   # the mix reads the table's bf16 rounding
        leaves += [w_gate, table]
    sums = [torch.zeros_like(t) for t in leaves]
    h_out, rstd, dqkv, dres, dn = [], [], [], [], []
    bounds = p["bounds"]
    for b in range(B):   # one row of the batch at a time: documents never cross a row
        inside = [t - b * T for t in bounds if b * T <= t <= (b + 1) * T]
        qkv, res = p["qkv"][b].double().requires_grad_(), p["residual"][b].double().requires_grad_()
        own = [qkv, res]
        q, k, v = qkv.view(T, 3, H, D).unbind(1)
        cos, sin = p["cos"][:, None], p["sin"][:, None]
        q = _norm_rope(q, q_gain, cos, sin)
        k = _norm_rope(k, k_gain, cos, sin)
        if c["ve"]:
            n = p["n"][b].double().requires_grad_()
            own.append(n)
            g = 2 * torch.sigmoid(n @ w_gate.t())
            v = v + g[..., None] * table[p["ids"][b].long()].view(T, H, D)
        out, _ = _attend_documents(q, k, v, inside, c["window"])
        h = res + out.reshape(T, C) @ o_weight.t()
        grads = torch.autograd.grad(h, leaves + own, p["dh"][b].double())
        for total, g in zip(sums, grads):
            total += g
        h_out.append(h.detach())
        rstd.append(1 / torch.sqrt(h.detach().square().mean(-1) + EPS))
        dqkv.append(grads[len(leaves)])
        dres.append(grads[len(leaves) + 1])
        if c["ve"]:
            dn.append(grads[len(leaves) + 2])
    got = [torch.stack(h_out), torch.cat(rstd), torch.stack(dqkv), sums[0], sums[1], torch.stack(dres)]
    if c["ve"]:
        got += [torch.stack(dn), sums[3]]
    return got + [sums[2]] + ([sums[4]] if c["ve"] else [])


def _exact_flash(c, seed):
    p = _flash_inputs(c, seed)
    S, T, H = c["segments"], c["seqlen"], c["heads"]
    window = T if c["window"] < 0 else c["window"]
    outs, lses, grads = [], [], []
    for s in range(S):
        rows = slice(s * T, (s + 1) * T)
        per_head = []
        for h in range(H):
            q, k, v = (p[n][rows, h:h + 1].double().requires_grad_() for n in ("q", "k", "v"))
            out, lse = _attend_documents(q, k, v, [0, T], window)
            per_head.append((out.detach(), lse.detach(), *torch.autograd.grad(out, (q, k, v), p["do"][rows, h:h + 1].double())))
        outs.append(torch.cat([x[0] for x in per_head], 1))
        lses.append(torch.cat([x[1] for x in per_head], 0))
        grads.append([torch.cat([x[2 + i] for x in per_head], 1) for i in range(3)])
    return [torch.cat(outs), torch.cat(lses, 1)] + [torch.cat([g[i] for g in grads]) for i in range(3)]


def _exact_rows(c, seed):
    p = _rows_inputs(c, seed)
    B, T, H = c["batch"], c["seqlen"], c["heads"]
    C = H * D
    cos, sin = p["cos"][:, None], p["sin"][:, None]
    qkv = p["qkv"].double().requires_grad_()
    q_gain, k_gain = p["q_gain"].double().requires_grad_(), p["k_gain"].double().requires_grad_()
    n, w_gate = p["n"].double().requires_grad_(), p["w_gate"].double().requires_grad_()
    table = _bf16(p["table"]).requires_grad_()
    q, k, v = _heads(qkv, H)
    qn, kn = _norm_rope(q, q_gain, cos, sin), _norm_rope(k, k_gain, cos, sin)
    gate = 2 * torch.sigmoid(n @ w_gate.t())
    vm = v + gate[..., None] * table[p["ids"].long()].view(B, T, H, D)
    leaves = [qkv, q_gain, k_gain, n, w_gate, table]
    dqkv, dqg, dkg, dn, dw, dtable = torch.autograd.grad(
        [qn, kn, vm], leaves, [p["dqn"].double(), p["dkn"].double(), p["dvm"].double()])
    return [qn.detach(), kn.detach(), vm.detach(), gate.detach().view(B * T, H), dqkv, dqg, dkg, dn, dw, dtable]


def exact(case, seed):
    made = {"decode": _exact_decode, "prefill": _exact_prefill, "attention": _exact_attention, "flash": _exact_flash,
            "rows": _exact_rows}.get(case["kind"])
    return made(case, seed) if made else None
