"""Performance cases of the paged-attention path: what a serving program has it do.

Five kinds of case, each through the package's public entry points:

* ``decode``: the attention calls of one decode step, layer after layer,
  replayed from one hipGraph as the decode step module does (a step plan first
  where ``plan`` is set, then one fused launch per layer).
* ``mixed``: the same for a packed step of prefill chunks and decode rows: plan,
  then per layer the QKV split + RoPE + append and the varlen attention.
* ``layer``: one drop-in attention layer (projections included), called eagerly.
* ``model_decode`` / ``model_mixed``: a whole step of a 24-layer model through
  ``DecodeModule`` / ``FullMixedModule``, host side included, up to its logits.

Lengths follow from the case alone, all tensor values from the seed.
"""
from __future__ import annotations

import math
import random
import sys
from types import SimpleNamespace

import numpy as np
import torch

import custom_inference_engine_amd as cie
from custom_inference_engine_amd.attn.core import Qwen2Attention
from custom_inference_engine_amd.graphs import StepGraph
from custom_inference_engine_amd.scheduler import DecodeModule, FullMixedModule

THETA = 1e6
VOCAB, HIDDEN, INTER, EPS = 151936, 896, 4864, 1e-6


def listed():
    return [
        # one user's next token, called layer by layer without a graph: the smallest call
        _decode("layer_decode_1", B=1, lo=128, hi=128, layers=1, kind="layer"),
        # one user's chat, 1,000 tokens in: a step of short launches
        _decode("decode_1x1000", B=1, lo=1000, hi=1000, layers=16),
        # the benchmark's headline: 32 users, 4,096 tokens each, append + attention, no plan
        _decode("decode_32x4096", B=32, lo=4096, hi=4096, layers=8, entry="append", plan=False),
        # an odd number of users, each somewhere else in its conversation
        _decode("decode_43_ragged", B=43, lo=512, hi=4096, layers=8),
        # two users with whole books as context
        _decode("decode_2_long", B=2, lo=65536, hi=131072, layers=4),
        # a full house of short conversations
        _decode("decode_200_short", B=200, lo=32, hi=1024, layers=8),
        # a model with 128-wide heads
        _decode("decode_16_d128", B=16, lo=256, hi=4096, layers=4, h_q=32, h_kv=8, d=128),
        # chunked prefill beside running decodes: the benchmark's mixed step
        _mixed("mixed_4x256_28", pre=4, new_lo=256, new_hi=256, prior_lo=0, prior_hi=2048, dec=28, dec_lo=256,
               dec_hi=3072, layers=8),
        # four new prompts of 2,048 tokens: compute-heavy prefill
        _mixed("prefill_4x2048", pre=4, new_lo=2048, new_hi=2048, prior_lo=0, prior_hi=0, dec=0, dec_lo=0, dec_hi=0,
               layers=4),
        # ragged chunks beside decodes with 128-wide heads
        _mixed("mixed_d128", pre=3, new_lo=300, new_hi=1024, prior_lo=0, prior_hi=4096, dec=13, dec_lo=256,
               dec_hi=4096, layers=2, h_q=32, h_kv=8, d=128),
        # a serving engine's decode step: 32 users, the whole model
        _decode("model_decode_32", B=32, lo=128, hi=2048, layers=24, kind="model_decode"),
        # a serving engine's mixed step: two prompt chunks and 24 running users in a 512-token bucket
        _mixed("model_mixed_512", pre=2, new_lo=200, new_hi=240, prior_lo=0, prior_hi=512, dec=24, dec_lo=128,
               dec_hi=1024, layers=24, kind="model_mixed"),
    ]


def _decode(name, *, B, lo, hi, layers, kind="decode", entry="rope", plan=True, h_q=14, h_kv=2, d=64, page=16):
    return dict(name=name, kind=kind, B=B, lo=lo, hi=hi, layers=layers, entry=entry, plan=plan, h_q=h_q, h_kv=h_kv,
                d=d, page=page)


def _mixed(name, *, pre, new_lo, new_hi, prior_lo, prior_hi, dec, dec_lo, dec_hi, layers, kind="mixed", h_q=14,
           h_kv=2, d=64, page=16):
    return dict(name=name, kind=kind, pre=pre, new_lo=new_lo, new_hi=new_hi, prior_lo=prior_lo, prior_hi=prior_hi,
                dec=dec, dec_lo=dec_lo, dec_hi=dec_hi, layers=layers, h_q=h_q, h_kv=h_kv, d=d, page=page)


# (query heads, kv heads, head dim): the benchmark's, and the geometries the tests cover
_HEADS = ((14, 2, 64), (14, 2, 64), (14, 2, 64), (28, 4, 64), (8, 2, 64), (8, 8, 64), (14, 2, 128), (32, 8, 128))


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _range(rng, lo, hi):
    """A range of lengths inside [lo, hi]: two ends spread over the logarithm."""
    a, b = sorted((_log_int(rng, lo, hi), _log_int(rng, lo, hi)))
    return a, b


def draw(rng):
    most = max(_weight(c) for c in listed() if not c["kind"].startswith("model"))
    while True:
        kind = rng.choice(("decode",) * 9 + ("mixed",) * 9 + ("layer", "model"))
        h_q, h_kv, d = rng.choice(_HEADS)
        page = rng.choice((16, 16, 16, 32))
        if kind == "model":
            lo, hi = _range(rng, 16, 2048)
            if rng.random() < 0.5:
                c = _decode(None, B=_log_int(rng, 1, 32), lo=lo, hi=hi, layers=24, kind="model_decode")
            else:
                c = _mixed(None, pre=rng.randint(1, 3), new_lo=16, new_hi=160, prior_lo=0, prior_hi=512,
                           dec=rng.randint(0, 24), dec_lo=lo, dec_hi=hi, layers=24, kind="model_mixed")
        elif kind == "layer":
            lo, hi = _range(rng, 16, 4096)
            c = _decode(None, B=_log_int(rng, 1, 64), lo=lo, hi=hi, layers=1, kind="layer")
        elif kind == "decode":
            lo, hi = _range(rng, 16, 131072)
            c = _decode(None, B=_log_int(rng, 1, 256), lo=lo, hi=hi, layers=rng.randint(4, 16),
                        entry=rng.choice(("rope", "rope", "append")), plan=rng.random() < 0.7, h_q=h_q, h_kv=h_kv,
                        d=d, page=page)
        else:
            new_lo, new_hi = _range(rng, 16, 4096)
            prior_hi = rng.choice((0, _log_int(rng, 64, 16384), _log_int(rng, 64, 16384)))
            dec_lo, dec_hi = _range(rng, 64, 8192)
            c = _mixed(None, pre=rng.randint(1, 8), new_lo=new_lo, new_hi=new_hi, prior_lo=0, prior_hi=prior_hi,
                       dec=rng.choice((0, rng.randint(1, 48))), dec_lo=dec_lo, dec_hi=dec_hi,
                       layers=rng.randint(2, 8), h_q=h_q, h_kv=h_kv, d=d, page=page)
        c.pop("name")
        if c["kind"].startswith("model") or _weight(c) <= most:
            return c


def _weight(c):
    w = work(c)
    return max(w["bytes"], w["flops"] / 50)


def _lens(c):
    """(prior lengths, new rows) of the case's sequences, in batch order."""
    r = random.Random(",".join("%s=%s" % (k, c[k]) for k in sorted(c) if k != "name"))
    if "B" in c:
        return [r.randint(c["lo"], c["hi"]) for _ in range(c["B"])], [1] * c["B"]
    prior = [r.randint(c["prior_lo"], c["prior_hi"]) for _ in range(c["pre"])]
    prior += [r.randint(c["dec_lo"], c["dec_hi"]) for _ in range(c["dec"])]
    new = [r.randint(c["new_lo"], c["new_hi"]) for _ in range(c["pre"])] + [1] * c["dec"]
    return prior, new


def work(case):
    prior, new = _lens(case)
    h_q, h_kv, d, layers = case["h_q"], case["h_kv"], case["d"], case["layers"]
    T = sum(new)
    keys = sum(p + n for p, n in zip(prior, new))            # K/V rows read once
    pairs = sum(n * p + n * (n + 1) // 2 for p, n in zip(prior, new))  # causal (query row, key) pairs
    # K/V read, new rows read and written, q read, o written, page ids
    by = 4 * h_kv * d * keys + 8 * h_kv * d * T + 4 * h_q * d * T + 8 * sum(-(-(p + n) // case["page"]) for p, n in zip(prior, new))
    fl = 4 * h_q * d * pairs
    if case["kind"] == "layer":
        w = HIDDEN * (h_q + 2 * h_kv) * d + HIDDEN * h_q * d
        by, fl = by + 2 * w + 4 * HIDDEN * T, fl + 2 * w * T
    by, fl = by * layers, fl * layers
    if case["kind"].startswith("model"):
        w = layers * (HIDDEN * (2 * h_q + 2 * h_kv) * d + 3 * HIDDEN * INTER)
        by += 2 * (w + VOCAB * HIDDEN) + 2 * VOCAB * len(new)
        fl += 2 * w * T + 2 * VOCAB * HIDDEN * len(new)
    return {"bytes": by, "flops": fl}


# ---- states ----

def _cos_sin(pos, d, dtype):
    inv = THETA ** (-torch.arange(0, d, 2, dtype=torch.float64, device=pos.device) / d)
    ang = pos.double()[:, None] * inv
    ang = torch.cat((ang, ang), -1)
    return ang.cos().to(dtype), ang.sin().to(dtype)


def _cache(case, gen, dev, batch):
    """A filled KV pool: shuffled pages, slots 1..B, random K/V, prior lengths set."""
    prior, new = _lens(case)
    page = case["page"]
    need = [-(-(p + n) // page) for p, n in zip(prior, new)]
    n_pages = 1 + sum(need)
    cfg = SimpleNamespace(num_hidden_layers=case["layers"], num_attention_heads=case["h_q"],
                          num_key_value_heads=case["h_kv"], head_dim=case["d"], hidden_size=case["h_q"] * case["d"])
    kv = cie.KVStorage(cfg, max_cache_len=n_pages * page, page_size=page, n_slots=batch + 1, device=dev,
                       dtype=torch.float16)
    for pool in kv.keys + kv.values:
        pool.normal_(0.0, 0.5, generator=gen)
    perm = torch.randperm(n_pages - 1, generator=gen, device=dev) + 1
    at = 0
    table = torch.zeros_like(kv.block_table)
    for i, n in enumerate(need):
        table[1 + i, :n] = perm[at:at + n]
        at += n
    kv.block_table.copy_(table)
    kv.lens[1:1 + len(prior)] = torch.tensor(prior, device=dev)
    return kv, prior, new


def _rows(kv, prior, new, dev):
    """Per packed row: position, slot, page, in-page offset."""
    pos = torch.tensor([p + i for p, n in zip(prior, new) for i in range(n)], device=dev)
    slot = torch.tensor([1 + b for b, n in enumerate(new) for _ in range(n)], device=dev)
    return pos, slot, kv.block_table[slot, pos // kv.page_size], pos % kv.page_size


def _cu(new):
    return [sum(new[:i]) for i in range(len(new) + 1)]


def _model_config(layers):
    hf = sys.modules[Qwen2Attention.__module__]  # the library whose attention the drop-in replaces
    cfg = hf.Qwen2Config(hidden_size=HIDDEN, num_attention_heads=14, num_key_value_heads=2, intermediate_size=INTER,
                         num_hidden_layers=layers, vocab_size=VOCAB, max_position_embeddings=32768, rope_theta=THETA,
                         rms_norm_eps=EPS, tie_word_embeddings=True)
    cfg._attn_implementation = "sdpa"
    return hf, cfg


def _build(make, gen, dev):
    """A module in fp16 on the device, its parameters drawn from gen: matrices
    with 0.02, norm weights around 1, biases around 0."""
    was = torch.get_default_dtype()
    torch.set_default_dtype(torch.float16)
    try:
        with torch.device(dev):
            m = make().eval().requires_grad_(False)
    finally:
        torch.set_default_dtype(was)
    for name, p in m.named_parameters():
        if p.dim() == 1:
            p.normal_(1.0 if "norm" in name else 0.0, 0.1, generator=gen)
        else:
            p.normal_(0.0, 0.02, generator=gen)
    return m


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(seed)
    kind, layers = case["kind"], case["layers"]
    h_q, h_kv, d = case["h_q"], case["h_kv"], case["d"]

    def rnd(*shape):
        return torch.empty(shape, dtype=torch.float16, device=dev).normal_(0.0, 0.5, generator=gen)

    with torch.inference_mode():
        kv, prior, new = _cache(case, gen, dev, max(len(_lens(case)[0]), 32 if kind.startswith("model") else 0))
        B, T = len(new), sum(new)
        slots = torch.arange(1, B + 1, device=dev)
        pos, row_slot, pages, offsets = _rows(kv, prior, new, dev)
        s = dict(case=case, kv=kv, prior=prior, new=new, slots=slots, pos=pos, row_slot=row_slot, pages=pages,
                 offsets=offsets)

        if kind.startswith("model"):
            hf, cfg = _model_config(layers)
            model = s["model"] = _build(lambda: hf.Qwen2ForCausalLM(cfg), gen, dev)
            # rotary frequencies are computed in 32 bits, whatever the weights' type
            model.model.rotary_emb = hf.Qwen2RotaryEmbedding(cfg).to(dev)
            cie.use_triton_attention(model)
            s["tokens"] = torch.randint(0, VOCAB, (T,), generator=gen, device=dev)
            s["lens0"] = kv.lens.clone()
            s["ids"] = list(range(1, B + 1))
            if kind == "model_decode":
                bucket = next(b for b in (1, 2, 4, 8, 16, 32) if b >= B)
                s["module"] = DecodeModule(model, kv, bucket, warmup_iters=1)
                s["last0"] = kv.last_generated.clone()
                s["last0"][1:B + 1] = s["tokens"]
            else:
                bucket = next(b for b in [16, 32, 64, 128] + list(range(160, 545, 32)) if b >= T)
                s["module"] = FullMixedModule(model, kv, 32, bucket, warmup_iters=1)
                flat, cu = s["tokens"].tolist(), _cu(new)
                s["prompts"] = [flat[cu[b]:cu[b + 1]] for b in range(B)]
            return s

        cos, sin = _cos_sin(pos, d, torch.float16)
        s["cos"], s["sin"] = cos[None], sin[None]
        if kind == "layer":
            hf, cfg = _model_config(1)
            s["layer"] = cie.TritonQwen2Attention(_build(lambda: hf.Qwen2Attention(cfg, layer_idx=0), gen, dev))
            s["hidden"] = rnd(1, T, HIDDEN)
            s["meta"] = cie.AttentionMetadata(token_count=T, full_decode=True, device=dev)
            s["meta"].slot_ids = slots
            return s

        width = (h_q + 2 * h_kv) * d
        if kind == "decode" and case["entry"] == "append":
            s["q"] = [rnd(1, B, h_q, d) for _ in range(layers)]
            s["k"] = [rnd(1, B, h_kv, d) for _ in range(layers)]
            s["v"] = [rnd(1, B, h_kv, d) for _ in range(layers)]
        else:
            s["qkv"] = [rnd(1, T, width) for _ in range(layers)]
        if kind == "decode":
            def step():
                plan = cie.gqa_decode_plan_op(kv.keys[0], kv.lens, slots, kv.block_table) if case["plan"] else None
                out = []
                for l in range(layers):
                    args = (kv.keys[l], kv.values[l])
                    if case["entry"] == "append":
                        out.append(cie.gqa_decode_append_attention_op(
                            s["q"][l], *args, s["k"][l], s["v"][l], kv.lens, slots, kv.block_table, plan=plan))
                    else:
                        out.append(cie.gqa_decode_qkv_rope_attention_op(
                            s["qkv"][l], s["cos"], s["sin"], *args, kv.lens, slots, kv.block_table, h_q, plan=plan))
                return out
        else:
            cu = torch.tensor(_cu(new), device=dev)
            kv_lens = torch.tensor(prior, device=dev)
            s["cu"], s["kv_lens"] = cu, kv_lens

            def step():
                plan = cie.gqa_mixed_plan_op(kv.keys[0], cu, kv_lens, slots, kv.block_table, T, T, h_q)
                out = []
                for l in range(layers):
                    q = cie.kv_append_tokens_qkv_rope_op(s["qkv"][l], s["cos"], s["sin"], kv.keys[l], kv.values[l],
                                                         pages, offsets, h_q)
                    out.append(cie.gqa_mixed_attention_op(q, kv.keys[l], kv.values[l], max_seqlen=T, cu_seqlens=cu,
                                                          kv_lens=kv_lens, slot_ids=slots,
                                                          block_table=kv.block_table, plan=plan))
                return out
        s["step"] = StepGraph(step, device=dev)
    return s


def run(state):
    kind, kv = state["case"]["kind"], state["kv"]
    if kind in ("decode", "mixed"):  # attention outputs and the appended pools
        return {"o": state["step"].replay(), "k": kv.keys, "v": kv.values}
    with torch.inference_mode():
        if kind == "layer":
            o, _ = state["layer"](state["hidden"], (state["cos"], state["sin"]), kv_manager=kv, metadata=state["meta"])
            return {"o": o, "k": kv.keys, "v": kv.values}
        # a step advances the lengths and takes its token: put both back, so that each pass is the same step
        kv.lens.copy_(state["lens0"])
        if kind == "model_decode":
            kv.last_generated.copy_(state["last0"])
            state["module"].forward(state["ids"])
            return {"logits": state["module"].logits[:len(state["ids"])]}
        state["module"].forward(state["prompts"], state["ids"])
        return {"logits": state["module"].last_logits}


def tolerance(case):
    if case["kind"].startswith("model"):
        # 24 layers of 16-bit activations: 4.6e-3 from the 64-bit step, measured
        return {"rel": 1.8e-2, "max": 0.2}
    # 16-bit outputs of 16-bit probabilities over 32-bit sums: 3e-4 from the 64-bit result, measured
    # (a layer with its projections 3.6e-4); the pools are copies and rotations
    return {"rel": 1.2e-3, "max": 0.02}


# ---- the same in 64 bits ----

def _rope64(x, cos, sin):
    h = x.shape[-1] // 2
    return x * cos[:, None] + torch.cat((-x[..., h:], x[..., :h]), -1) * sin[:, None]


def _attend64(q, kpool, vpool, s, d):
    """q (T, h_q, d) against each sequence's pages, causal from its prior length."""
    kv, out, t = s["kv"], torch.empty_like(q), 0
    for b, (p, n) in enumerate(zip(s["prior"], s["new"])):
        L = p + n
        ids = kv.block_table[1 + b, :-(-L // kv.page_size)]
        rows = [x[ids].permute(1, 0, 2, 3).reshape(x.shape[1], -1, d)[:, :L].double() for x in (kpool, vpool)]
        mask = torch.arange(L, device=q.device)[None] > (p + torch.arange(n, device=q.device))[:, None]
        G = q.shape[1] // kpool.shape[1]
        for g in range(kpool.shape[1]):
            k_t = rows[0][g].t().contiguous()
            for h in range(g * G, (g + 1) * G):
                sc = (q[t:t + n, h] @ k_t) * d ** -0.5
                out[t:t + n, h] = torch.softmax(sc.masked_fill_(mask, -math.inf), -1) @ rows[1][g]
        t += n
    return out


def _append64(s, kpool, vpool, k, v):
    kp, vp = kpool.double(), vpool.double()
    kp[s["pages"], :, s["offsets"]] = k
    vp[s["pages"], :, s["offsets"]] = v
    return kp, vp


def exact(case, seed):
    with torch.inference_mode():
        s = prepare(case, seed)
        h_q, h_kv, d, kv = case["h_q"], case["h_kv"], case["d"], s["kv"]
        if case["kind"].startswith("model"):
            return {"logits": _model64(s)}
        cos, sin = s["cos"][0].double(), s["sin"][0].double()
        o, kps, vps = [], [], []
        for l in range(case["layers"]):
            if "q" in s:
                q, k, v = (s[n][l][0].double() for n in "qkv")
            else:
                if case["kind"] == "layer":
                    at = s["layer"].original
                    qkv = torch.cat([s["hidden"][0].double() @ p.weight.double().t() + p.bias.double()
                                     for p in (at.q_proj, at.k_proj, at.v_proj)], -1)
                else:
                    qkv = s["qkv"][l][0].double()
                q, k, v = qkv.view(-1, h_q + 2 * h_kv, d).split((h_q, h_kv, h_kv), 1)
                q, k = _rope64(q, cos, sin), _rope64(k, cos, sin)
            kp, vp = _append64(s, kv.keys[l], kv.values[l], k, v)
            x = _attend64(q, kp, vp, s, d)
            if case["kind"] == "layer":
                o.append(x.reshape(1, -1, h_q * d) @ s["layer"].original.o_proj.weight.double().t())
            else:
                o.append(x[None])
            kps.append(kp)
            vps.append(vp)
        return {"o": o[0] if case["kind"] == "layer" else o, "k": kps, "v": vps}


def _model64(s):
    model, kv, case = s["model"], s["kv"], s["case"]
    d, h_q, h_kv = case["d"], case["h_q"], case["h_kv"]
    cos, sin = _cos_sin(s["pos"], d, torch.float64)

    def norm(x, m):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * m.weight.double()

    def lin(x, m):
        y = x @ m.weight.double().t()
        return y if m.bias is None else y + m.bias.double()

    x = model.model.embed_tokens.weight[s["tokens"]].double()
    for l, layer in enumerate(model.model.layers):
        at = layer.self_attn.original
        h = norm(x, layer.input_layernorm)
        q, k, v = (lin(h, p).view(-1, n, d) for p, n in ((at.q_proj, h_q), (at.k_proj, h_kv), (at.v_proj, h_kv)))
        q, k = _rope64(q, cos, sin), _rope64(k, cos, sin)
        kp, vp = _append64(s, kv.keys[l], kv.values[l], k, v)
        x = x + lin(_attend64(q, kp, vp, s, d).reshape(-1, h_q * d), at.o_proj)
        h = norm(x, layer.post_attention_layernorm)
        x = x + lin(torch.nn.functional.silu(lin(h, layer.mlp.gate_proj)) * lin(h, layer.mlp.up_proj),
                    layer.mlp.down_proj)
    last = torch.tensor(np.cumsum(s["new"]) - 1, device=x.device)
    return norm(x, model.model.norm)[last] @ model.lm_head.weight.double().t()
