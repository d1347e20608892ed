"""Timed cases of the framework's main paths, through the Python binding of its C ABI.

Two families, as the framework has them:

* the Llama / Mistral decoder (``DeviceModel`` + ``Decoder``): greedy decoding on the device,
  decoding with the logits on the host (a program that samples), a prompt's hydration up to its
  first logits, and the scoring of a text (``-m perplexity``);
* layer-list models (``SeqModel`` + ``SeqDecoder``): a request's prompt portion and its decoding.

A case is a dict of plain values; ``prepare`` makes the weights, the caches' history and the
tokens on the GPU from a seed, ``run`` is one pass, ``exact`` the same in 64-bit torch.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from yalm_amd import layered as Ly
from yalm_amd import models as M
from yalm_amd import runtime

DEV = "cuda:0"
DTYPES = {"fp32": M.F32, "fp16": M.F16, "fp8": M.F8E5M2}
TORCH_DTYPES = {M.F32: torch.float32, M.F16: torch.float16, M.F8E5M2: torch.float8_e5m2, M.BF16: torch.bfloat16}
# sizes of the configurations in yalm_amd/models.py; `small` with the full context of the others
CONFIGS = {"mistral-7b": M.MISTRAL_7B, "llama-3.2-3b": M.LLAMA_32_3B, "small": M.SMALL.with_(max_seq_len=4096)}


# ------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: one forward of a small f32 model, where launches and latency are all there is
        dict(name="small-fp32-step", family="dense", model="small", dtype="fp32", kind="sample", pos=37, n=1),
        # the headline use: greedy text generation after a short prompt (README's prompt is 13 tokens)
        dict(name="mistral-fp16-greedy", family="dense", model="mistral-7b", dtype="fp16", kind="greedy", pos=13, n=16),
        # the same far into a conversation, just under the full window
        dict(name="mistral-fp16-greedy-long", family="dense", model="mistral-7b", dtype="fp16", kind="greedy", pos=4003, n=12),
        # the 8-bit weights, mid-conversation
        dict(name="mistral-fp8-greedy", family="dense", model="mistral-7b", dtype="fp8", kind="greedy", pos=700, n=16),
        # the command line's default temperature: every token's logits go to the host's sampler
        dict(name="llama-fp16-sample", family="dense", model="llama-3.2-3b", dtype="fp16", kind="sample", pos=300, n=8),
        # a short question: 13 tokens to the first logits
        dict(name="mistral-fp16-prompt-13", family="dense", model="mistral-7b", dtype="fp16", kind="prompt", pos=0, n=13),
        # the next turn of a conversation: a ragged prompt behind a history
        dict(name="mistral-fp16-prompt-391", family="dense", model="mistral-7b", dtype="fp16", kind="prompt", pos=600, n=391),
        # a pasted page of text, 8-bit weights
        dict(name="mistral-fp8-prompt-1001", family="dense", model="mistral-7b", dtype="fp8", kind="prompt", pos=0, n=1001),
        # -m perplexity over a full window, in the precision form that it runs
        dict(name="llama-fp16-score-4096", family="dense", model="llama-3.2-3b", dtype="fp16", kind="score", pos=0, n=4096, split=True),
        # layer-list models: an answer to a short prompt (mostly single tokens, greedy on the device) ...
        dict(name="sinulorn-2048-answer", family="layered", design="sinulorn", width=2048, dtype="bf16", n=61, want=1, m=24, decode="greedy"),
        # ... a long prompt with some of its positions scored ...
        dict(name="sinulorn-2048-portion", family="layered", design="sinulorn", width=2048, dtype="bf16", n=2048, want=32, m=0, decode="replay"),
        # ... and a ragged prompt with a few replayed single tokens, a narrower model of another design
        dict(name="lenuzen-1024-request", family="layered", design="lenuzen", width=1024, dtype="bf16", n=777, want=1, m=8, decode="replay"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.65:
        model = rng.choice(["mistral-7b", "mistral-7b", "llama-3.2-3b", "llama-3.2-3b", "small"])
        dtype = rng.choice(["fp16", "fp8", "fp32"] if model == "small" else ["fp16", "fp16", "fp8"])
        kinds = ["greedy", "sample"] if model == "small" else ["greedy", "greedy", "sample", "prompt", "prompt", "score"]
        kind = rng.choice(kinds)
        c = dict(family="dense", model=model, dtype=dtype, kind=kind)
        if kind == "greedy" and model == "llama-3.2-3b":
            kind = c["kind"] = "sample"  # a tied classifier: the greedy loop would repeat one token
        if kind in ("greedy", "sample"):
            n = rng.randint(2, 16 if kind == "greedy" else 10)
            return dict(c, pos=min(_log(rng, 1, 4090), 4095 - n), n=n)
        top = 4000 if model == "llama-3.2-3b" else 1800
        if kind == "prompt":
            n = _log(rng, 4, top)
            return dict(c, pos=rng.choice([0, 0, rng.randint(1, 4090 - n)]), n=n)
        return dict(c, pos=0, n=_log(rng, 64, top), split=rng.random() < 0.7)
    design = rng.choice(["sinulorn", "lenuzen"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
    width = 512 * rng.randint(2, 8 if dtype == "bf16" else 4)
    n = _log(rng, 1, 2048 if dtype == "bf16" else 256)
    m = rng.randint(0, 16)
    decode = "replay" if design == "lenuzen" else rng.choice(["replay", "greedy"])
    return dict(family="layered", design=design, width=width, dtype=dtype, n=n, want=rng.choice([1, 1, min(n, 8)]), m=m, decode=decode)


# ------------------------------------------------------------------------------- inputs
def _gen(seed, *what):
    h = 1469598103934665603
    for ch in ":".join(str(x) for x in (seed,) + what).encode():
        h = ((h ^ ch) * 1099511628211) & 0x7FFFFFFFFFFFFFFF
    return torch.Generator(device=DEV).manual_seed(h)


def _normal(g, shape, std, dtype, mean=0.0):
    if dtype == torch.float8_e5m2:
        return _normal(g, shape, std, torch.float16).to(dtype)
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(mean, std, generator=g)


def _dense_config(case):
    return CONFIGS[case["model"]].with_(weight_dtype=DTYPES[case["dtype"]])


def _dense_weights(cfg, seed):
    """Weights as in a trained model: unit-size queries, keys and hidden units, every sublayer's
    result a 1 / sqrt(2 layers) share of the stream, so that the stream keeps the token's
    embedding; an untied classifier row answers the embedding of the token before it, so the next
    token is decided by a clear margin."""
    dt = TORCH_DTYPES[cfg.weight_dtype]
    emb = 0.25 if cfg.tied else 0.5
    out = {}
    for name, (shape, is_norm) in M.tensor_shapes(cfg).items():
        g = _gen(seed, name)
        leaf = name.split(".")[-2]
        if is_norm:
            mean = 1.0 if name != "model.norm.weight" else (0.02 if cfg.tied else 0.1)
            out[name] = _normal(g, shape, 0.1 * mean, torch.float32, mean)
        elif name == "model.embed.weight":
            out[name] = _normal(g, shape, emb, dt)
        elif name == "model.output.weight":
            out[name] = (torch.roll(out["model.embed.weight"].to(torch.float32), 1, 0) * 0.5).to(dt)
        elif leaf in ("wo", "w2"):
            out[name] = _normal(g, shape, emb / math.sqrt(2 * cfg.n_layers * shape[1]), dt)
        else:
            out[name] = _normal(g, shape, 1.28 / math.sqrt(shape[1]), dt)
    return out


def _dense_inputs(case, seed):
    """(weights, caches [layers, key | value, positions, kv_dim] with `pos` positions of history, tokens)."""
    cfg = _dense_config(case)
    w = _dense_weights(cfg, seed)
    kv = _normal(_gen(seed, "kv"), (cfg.n_layers, 2, cfg.max_seq_len, cfg.kv_dim), 1.28, torch.float16)
    rng = np.random.default_rng([seed & 0x7FFFFFFF, case["n"], case["pos"]])
    tok = rng.integers(3, cfg.vocab_size - 64, case["n"]).astype(np.int32)
    if case["kind"] == "score":  # half of the text is what the model expects
        for i in range(1, len(tok)):
            if rng.random() < 0.5:
                tok[i] = tok[i - 1] if cfg.tied else (tok[i - 1] + 1) % cfg.vocab_size
    return cfg, w, kv, tok


def _layered_config(case):
    width, heads = case["width"], case["width"] // 128
    ff = width * 7 // 2
    most = case["n"] + case["m"] + 1
    L = Ly.LayerSpec
    if case["design"] == "sinulorn":
        dense = dict(ff_kind=Ly.FF_DENSE, ff=ff)
        moe = dict(ff_kind=Ly.FF_MOE, ff=ff // 8, experts=16, top=4, groups=4, groups_keep=2, router_scale=2.5, limit=7.0, shared_ff=ff // 2, shared_limit=7.0)
        lat = dict(heads=heads, dim=128, vdim=128, kv_rank=256, q_rank=max(width // 2, 256), attn_scale=128 ** -0.5)
        dlt = dict(heads=heads, kv_heads=max(heads // 2, 1), dim=128, vdim=128, conv=4)
        rec = dict(rec_width=width, blocks=heads, conv=4)
        layers = [L(Ly.MIX_DELTA, **dlt, **dense), L(Ly.MIX_LATENT, **lat, **moe), L(Ly.MIX_RGLRU, **rec, **dense),
                  L(Ly.MIX_DELTA, **dlt, **moe), L(Ly.MIX_LATENT, kv_from=1, **lat, **dense), L(Ly.MIX_RGLRU, **rec, **dense)]
        return Ly.LayeredConfig("Sinulorn", width, 32000, layers, embed_scale=1.0, norm_eps=1e-5, max_tokens=most,
                                weight_dtype=M.BF16 if case["dtype"] == "bf16" else M.F32)
    common = dict(heads=heads, kv_heads=min(max(heads // 4, 1), 4), dim=128, vdim=128, attn_scale=128 ** -0.5, rot_dims=64, rot_base=500000.0,
                  rot_factor=8.0, rot_orig=8192, rot_fast=16.0, rot_slow=2.0, ff_kind=Ly.FF_PLAIN, ff=ff)
    chunked = dict(mask_kind=Ly.MASK_CHUNK, mask_size=2048, qk_norm=Ly.QK_WHOLE, sink=1, talking=True, **common)
    windowed = dict(mask_kind=Ly.MASK_WINDOW, mask_size=1024, qk_norm=Ly.QK_HEAD_UNIT, v_norm=1, out_gate=1, in_biased=True, head_temps=True, **common)
    layers = [L(Ly.MIX_ATTN, **d) for d in (chunked, chunked, windowed, chunked, chunked, windowed)]
    return Ly.LayeredConfig("Lenuzen", width, 32000, layers, embed_scale=float(width) ** 0.5, norm_eps=1e-5, max_tokens=most,
                            weight_dtype=M.BF16 if case["dtype"] == "bf16" else M.F32, norm_kind=Ly.NORM_LAYER, pre_norm=False, pos_embed=False,
                            logit_scale=0.7, tied_head=True)


def _layered_weights(cfg, seed):
    """{"embed", "final_norm", "head"} and one dict per layer, in the engine's packed layout."""
    dt = TORCH_DTYPES[cfg.weight_dtype]
    tied = cfg.tied_head
    top = {"embed": _normal(_gen(seed, "embed"), (cfg.vocab, cfg.width), cfg.width ** -0.5 if tied else 1.0, dt),
           "final_norm": _normal(_gen(seed, "final"), (cfg.width,), 0.1, torch.float32, 1.0)}
    top["head"] = top["embed"] if tied else (torch.roll(top["embed"].float(), 1, 0) * 0.02).to(dt)
    layers = []
    for i, l in enumerate(cfg.layers):
        d = {}
        for k, (shape, kind) in Ly.packed_shapes(cfg, l).items():
            g = _gen(seed, i, k)
            if kind == "w":
                fan = shape[-2] if k == "w_ukt" else shape[-1]
                d[k] = _normal(g, shape, fan ** -0.5, dt)
            elif k == "router":  # as a trained one: the last of a token's choices carries little
                d[k] = _normal(g, shape, 3.0 * shape[-1] ** -0.5, torch.float32)
            elif k in ("gate_a", "gate_i", "shared_sg"):
                d[k] = _normal(g, shape, shape[-1] ** -0.5, torch.float32)
            elif k in ("norm1b", "norm2b"):
                d[k] = _normal(g, shape, 0.05, torch.float32, 0.5)
            elif k in ("norm1", "norm2", "q_norm", "kv_norm", "out_norm", "head_temp"):
                d[k] = _normal(g, shape, 0.1, torch.float32, 1.0)
            elif k == "talk":
                d[k] = torch.eye(l.heads, device=DEV) + _normal(g, shape, 0.3 * l.heads ** -0.5, torch.float32)
            elif k == "conv_w":
                d[k] = _normal(g, shape, 0.5, torch.float32)
            elif k in ("lam", "a_log", "dt_bias"):
                lo, hi = {"lam": (-4.0, 1.0), "a_log": (-3.0, 0.5), "dt_bias": (-2.0, 1.0)}[k]
                d[k] = torch.empty(shape, device=DEV).uniform_(lo, hi, generator=g)
            else:
                d[k] = _normal(g, shape, 0.1, torch.float32)
            if k == "in_bias" and l.out_gate == Ly.GATE_HEAD:
                d[k][-l.heads:] = 0.0
        layers.append(d)
    return top, layers


def _layered_inputs(case, seed):
    cfg = _layered_config(case)
    top, layers = _layered_weights(cfg, seed)
    rng = np.random.default_rng([seed & 0x7FFFFFFF, case["n"], case["width"]])
    tok = rng.integers(3, cfg.vocab - 64, case["n"] + max(case["m"], 1)).astype(np.int32)
    want = np.unique(np.linspace(0, case["n"] - 1, case["want"] + 1)[1:].round().astype(np.int32))
    return cfg, top, layers, tok, want


def prepare(case, seed):
    if case["family"] == "dense":
        cfg, w, kv, tok = _dense_inputs(case, seed)
        model = runtime.DeviceModel(cfg)
        model.ptrs = {k: t.data_ptr() for k, t in w.items()}
        torch.cuda.synchronize()
        dec = runtime.Decoder(model, kv_caches=[(kv[l, 0].data_ptr(), kv[l, 1].data_ptr()) for l in range(cfg.n_layers)])
        if case["kind"] == "score" and case["split"]:
            dec.set_prefill_precision(runtime.PREFILL_SPLIT)
        return dict(case=case, dec=dec, model=model, w=w, kv=kv, tok=tok)
    cfg, top, layers, tok, want = _layered_inputs(case, seed)
    model = runtime.SeqModel(cfg)
    model.ptrs = {k: t.data_ptr() for k, t in top.items()}
    model.layer_ptrs = [{k: t.data_ptr() for k, t in d.items()} for d in layers]
    torch.cuda.synchronize()
    return dict(case=case, dec=runtime.SeqDecoder(model), model=model, w=(top, layers), tok=tok, want=want)


# ------------------------------------------------------------------------------- one pass
def run(state):
    case, dec, tok = state["case"], state["dec"], state["tok"]
    if case["family"] == "layered":
        n, m = case["n"], case["m"]
        dec.reset()
        out = {"portion": dec.step(tok[:n], state["want"])}
        if m and case["decode"] == "greedy":
            out["tokens"] = np.array(dec.generate_greedy(int(tok[n]), m), np.int32)
            out["last"] = dec.step(out["tokens"][-1:], [0])
        elif m:
            out["steps"] = [dec.step(tok[n + i:n + i + 1], [0]) for i in range(m)]
        return out
    pos, n, kind = case["pos"], case["n"], case["kind"]
    rows = state["kv"][:, :, pos:pos + n]
    if kind == "greedy":
        tokens = dec.generate_greedy(int(tok[0]), pos, n)
        return {"tokens": np.array(tokens, np.int32), "logits": dec.get_logits(), "kv": rows}
    if kind == "sample":
        return {"logits": [dec.forward(int(t), pos + i) for i, t in enumerate(tok)], "kv": rows}
    if kind == "prompt":
        dec.prefill(tok[:-1], pos, logprobs=False)
        return {"logits": dec.forward(int(tok[-1]), pos + n - 1), "kv": rows}
    return {"logprobs": dec.prefill(tok, pos), "kv": rows}


# ------------------------------------------------------------------------------- work
def work(case):
    """Every weight that a pass needs once per pass over the tokens (one pass per token when
    decoding), the cached rows read and written, the logits written; products of matrices only."""
    if case["family"] == "dense":
        cfg = _dense_config(case)
        pos, n, kind = case["pos"], case["n"], case["kind"]
        wb = M.DTYPE_BYTES[cfg.weight_dtype]
        layer = cfg.dim * (2 * cfg.q_dim + 2 * cfg.kv_dim + 3 * cfg.hidden_dim)
        head = cfg.vocab_size * cfg.dim
        kv_row = cfg.n_layers * 4 * cfg.kv_dim
        pairs = n * pos + n * (n + 1) // 2
        att = 4 * cfg.n_layers * cfg.q_dim * pairs
        if kind in ("greedy", "sample"):
            per = cfg.weight_bytes_per_token()
            return {"bytes": n * per + kv_row * pairs + (4 * cfg.vocab_size * (n if kind == "sample" else 1)),
                    "flops": 2 * n * (cfg.n_layers * layer + head) + att}
        heads = n if kind == "score" else 1
        return {"bytes": (cfg.n_layers * layer + head) * wb + n * cfg.dim * wb + kv_row * (pos + 2 * n) + 4 * (n if kind == "score" else cfg.vocab_size),
                "flops": 2 * (n * cfg.n_layers * layer + heads * head) + att}
    cfg = _layered_config(case)
    wb = 2 if case["dtype"] == "bf16" else 4
    n, m = case["n"], case["m"]
    steps = m + (1 if m and case["decode"] == "greedy" else 0)
    head = cfg.vocab * cfg.width
    by, fl = 0, 0
    for tokens, times, logits, first in ((n, 1, case["want"], 0), (1, steps, 1, n)):
        if not times:
            continue
        by += times * (head * wb + 4 * logits * cfg.vocab)
        fl += times * 2 * logits * head
        for l in cfg.layers:
            for k, (shape, kind) in Ly.packed_shapes(cfg, l).items():
                size = int(np.prod(shape))
                b = wb if kind == "w" else 4
                if l.ff_kind == Ly.FF_MOE and k in ("w_gate", "w_up", "w_down"):
                    by += times * size * b * min(l.experts, tokens * l.top) // l.experts
                    fl += times * 2 * tokens * size * l.top // l.experts
                else:
                    by += times * size * b
                    fl += times * 2 * tokens * size if len(shape) > 1 else 0
            keys = l.kv_rank if l.mixer == Ly.MIX_LATENT else l.dim if l.mixer == Ly.MIX_ATTN else 0
            span = min(first + tokens * times, l.mask_size or 1 << 30)
            if keys:
                by += times * span * (l.kv_rank or l.kv_heads * 2 * l.dim) * wb
                fl += times * 4 * l.heads * keys * tokens * (span if tokens == 1 else span // 2 + 1)
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """About four times the largest error against 64 bits over the listed and some drawn cases: the
    dense decoder's caches hold f16 (2.1e-4 to 3.2e-4 off), its logits are nearer; layer-list models
    in f32 are 2e-6 off, in bf16 1e-3 to 8e-3 (routers choose among near ties)."""
    if case["family"] == "dense":
        return {"rel": 1.3e-3, "max": 2e-2, "differ": 0.0}
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.0}
    return {"rel": 3e-2, "max": 0.3, "differ": 0.0}


# ------------------------------------------------------------------------------- 64 bits
def _d(t):
    return t.to(torch.float16).double() if t.dtype == torch.float8_e5m2 else t.double()


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _layer_norm(x, w, eps):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w.double()


def _sigmoid(x):
    return torch.sigmoid(x)


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _rope(x, positions, theta):
    """x [T, heads, D]: interleaved pairs (2i, 2i + 1)."""
    D = x.shape[-1]
    f = theta ** (-torch.arange(0, D, 2, device=DEV, dtype=torch.float64) / D)
    a = positions.double()[:, None] * f
    c, s = a.cos()[:, None], a.sin()[:, None]
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack((u * c - v * s, u * s + v * c), -1).flatten(-2)


def _softmax_causal(s, pos0, mask=None, sink=False):
    """s [heads, T, S], row t at position pos0 + t; sink: one more key of score 0 and no value."""
    T, S = s.shape[-2:]
    i = torch.arange(T, device=DEV)[:, None] + pos0
    j = torch.arange(S, device=DEV)[None, :]
    see = j <= i
    if mask is not None:
        see = see & (i - j < mask[1] if mask[0] == "window" else i // mask[1] == j // mask[1])
    s = s.masked_fill(~see, -math.inf)
    top = s.amax(-1, keepdim=True)
    if sink:
        top = top.clamp(min=0.0)
    e = torch.exp(s - top)
    return e / (e.sum(-1, keepdim=True) + (torch.exp(-top) if sink else 0.0))


def _dense_forward(cfg, w, kv, tok, pos0):
    """Appends the tokens' rows to kv (64 bits) in place; returns the final-normed rows."""
    T = len(tok)
    H, G, D = cfg.n_heads, cfg.n_kv_heads, cfg.head_dim
    p = torch.arange(pos0, pos0 + T, device=DEV)
    theta = float(np.float32(cfg.rope_theta))
    x = _d(w["model.embed.weight"][torch.as_tensor(np.asarray(tok), device=DEV).long()])
    for l in range(cfg.n_layers):
        name = M.layer_names(l)
        h = _rms(x, w[name["rms_att"]], cfg.norm_eps)
        q = _rope((h @ _d(w[name["wq"]]).T).view(T, H, D), p, theta)
        kv[l, 0, pos0:pos0 + T] = _rope((h @ _d(w[name["wk"]]).T).view(T, G, D), p, theta).flatten(1)
        kv[l, 1, pos0:pos0 + T] = h @ _d(w[name["wv"]]).T
        k, v = kv[l, :, :pos0 + T].view(2, pos0 + T, G, D)
        o = torch.empty_like(q)
        r = H // G
        for g in range(G):
            s = torch.matmul(q[:, g * r:(g + 1) * r].transpose(0, 1).contiguous(), k[:, g].T.contiguous()) / math.sqrt(D)
            o[:, g * r:(g + 1) * r] = torch.matmul(_softmax_causal(s, pos0), v[:, g].contiguous()).transpose(0, 1)
        x = x + o.flatten(1) @ _d(w[name["wo"]]).T
        h = _rms(x, w[name["rms_ffn"]], cfg.norm_eps)
        a = h @ _d(w[name["w1"]]).T
        a = a * _sigmoid(a) * (h @ _d(w[name["w3"]]).T)
        x = x + a @ _d(w[name["w2"]]).T
    return _rms(x, w["model.norm.weight"], cfg.norm_eps)


def _dense_exact(case, seed):
    cfg, w, kv, tok = _dense_inputs(case, seed)
    pos, n, kind = case["pos"], case["n"], case["kind"]
    kv = kv[:, :, :pos + n].double()
    head = _d(w["model.embed.weight"] if cfg.tied else w["model.output.weight"])
    if kind == "greedy":
        t, tokens = int(tok[0]), []
        for i in range(n):
            logits = (_dense_forward(cfg, w, kv, [t], pos + i) @ head.T)[0]
            t = int(logits.argmax())
            tokens.append(t)
        return {"tokens": np.array(tokens, np.int32), "logits": logits, "kv": kv[:, :, pos:]}
    x = _dense_forward(cfg, w, kv, tok, pos)
    rows = kv[:, :, pos:]
    if kind == "sample":
        return {"logits": list(x @ head.T), "kv": rows}
    if kind == "prompt":
        return {"logits": x[-1] @ head.T, "kv": rows}
    lp = torch.zeros(n, dtype=torch.float64, device=DEV)
    nxt = torch.as_tensor(tok[1:], device=DEV).long()
    for a in range(0, n - 1, 512):
        z = x[a:min(a + 512, n - 1)] @ head.T
        lp[a:a + len(z)] = z.gather(1, nxt[a:a + len(z), None])[:, 0] - torch.logsumexp(z, 1)
    return {"logprobs": lp, "kv": rows}


def _conv(x, taps):
    K = taps.shape[1]
    xp = torch.cat((torch.zeros(K - 1, x.shape[1], device=DEV, dtype=torch.float64), x))
    return sum(xp[j:j + len(x)] * taps[:, j].double() for j in range(K))


def _latent64(l, d, h, c, eps):
    T, H = len(h), l.heads
    q = _rms(h @ d["w_in"][:l.q_rank].double().T, d["q_norm"], eps) @ d["w_uq"].double().T
    q = q.view(T, H, l.dim).transpose(0, 1).contiguous()
    qc = torch.matmul(q, d["w_ukt"].double().transpose(1, 2).contiguous())
    p = _softmax_causal(torch.matmul(qc, c.T.contiguous()) * l.attn_scale, 0)
    v = (c @ d["w_uv"].double().T).view(T, H, l.vdim).transpose(0, 1).contiguous()
    return torch.matmul(p, v).transpose(0, 1).flatten(1)


def _rglru64(l, d, h):
    T, W, B = len(h), l.rec_width, l.blocks
    z = h @ d["w_in"].double().T + d["in_bias"].double()
    u = _conv(z[:, W:], d["conv_w"]) + d["conv_b"].double()
    ub = u.view(T, B, W // B).transpose(0, 1).contiguous()
    r, i = (_sigmoid(torch.matmul(ub, d[k].double().transpose(1, 2).contiguous()).transpose(0, 1).flatten(1) + d[k + "_b"].double()) for k in ("gate_a", "gate_i"))
    log_a = -8.0 * r * torch.nn.functional.softplus(d["lam"].double())
    a, b = torch.exp(log_a), torch.sqrt(-torch.expm1(2.0 * log_a)) * i * u
    s, out = torch.zeros(W, device=DEV, dtype=torch.float64), torch.empty_like(u)
    for t in range(T):
        s = a[t] * s + b[t]
        out[t] = s
    return out * _gelu(z[:, :W])


def _delta64(l, d, h, eps):
    T, H, K, D, V = len(h), l.heads, l.kv_heads, l.dim, l.vdim
    z = h @ d["w_in"].double().T
    cc = 2 * K * D + H * V
    y = _conv(z[:, :cc], d["conv_w"])
    y = y * _sigmoid(y)
    q, k = y[:, :K * D].view(T, K, D), y[:, K * D:2 * K * D].view(T, K, D)
    v = y[:, 2 * K * D:].view(T, H, V)
    q = (q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * D ** -0.5).repeat_interleave(H // K, 1)
    k = (k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // K, 1)
    gate = z[:, cc:cc + H * V].view(T, H, V)
    beta = _sigmoid(z[:, cc + H * V:cc + H * V + H])
    g = torch.exp(-torch.exp(d["a_log"].double()) * torch.nn.functional.softplus(z[:, cc + H * V + H:] + d["dt_bias"].double()))
    s, o = torch.zeros(H, D, V, device=DEV, dtype=torch.float64), torch.empty(T, H, V, device=DEV, dtype=torch.float64)
    for t in range(T):
        s = s * g[t, :, None, None]
        u = beta[t, :, None] * (v[t] - (s * k[t, :, :, None]).sum(1))
        s = s + k[t, :, :, None] * u[:, None]
        o[t] = (s * q[t, :, :, None]).sum(1)
    o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps) * d["out_norm"].double() * gate * _sigmoid(gate)
    return o.flatten(1)


def _expert64(h, gate, up, down, limit):
    g = (h @ gate.double().T).clamp(max=limit)
    u = (h @ up.double().T).clamp(-limit, limit)
    return (g * _sigmoid(1.702 * g) * (u + 1.0)) @ down.double().T


def _experts64(l, d, h):
    s = torch.softmax(h @ d["router"].double().T, 1)
    E, G = l.experts, l.groups
    keep = s.view(-1, G, E // G).amax(2).topk(l.groups_keep, 1).indices
    allowed = torch.zeros(len(h), G, dtype=torch.bool, device=DEV).scatter_(1, keep, True).repeat_interleave(E // G, 1)
    wt, idx = s.masked_fill(~allowed, -1.0).topk(l.top, 1)
    out = _sigmoid(h @ d["shared_sg"].double())[:, None] * _expert64(h, d["ws_gate"], d["ws_up"], d["ws_down"], l.shared_limit)
    for e in range(E):
        row, slot = (idx == e).nonzero(as_tuple=True)
        if len(row):
            out[row] += wt[row, slot, None] * l.router_scale * _expert64(h[row], d["w_gate"][e], d["w_up"][e], d["w_down"][e], l.limit)
    return out


def _sinulorn64(cfg, top, layers, tok):
    T, W, eps = len(tok), cfg.width, cfg.norm_eps
    ang = torch.arange(T, device=DEV).double()[:, None] * 10000.0 ** (-2.0 * torch.arange(W // 2, device=DEV).double() / W)
    x = top["embed"][tok].double() * cfg.embed_scale + torch.stack((ang.sin(), ang.cos()), -1).flatten(1)
    latents = {}
    for i, (l, d) in enumerate(zip(cfg.layers, layers)):
        h = _rms(x, d["norm1"], eps)
        if l.mixer == Ly.MIX_LATENT:
            if l.kv_from < 0:
                latents[i] = _rms(h @ d["w_in"][l.q_rank:].double().T, d["kv_norm"], eps)
            y = _latent64(l, d, h, latents[i if l.kv_from < 0 else l.kv_from], eps)
        else:
            y = _rglru64(l, d, h) if l.mixer == Ly.MIX_RGLRU else _delta64(l, d, h, eps)
        x = x + _rms(y @ d["w_o"].double().T, d["norm1b"], eps)
        h = _rms(x, d["norm2"], eps)
        if l.ff_kind == Ly.FF_DENSE:
            y = (_gelu(h @ d["w_gate"].double().T) * (h @ d["w_up"].double().T)) @ d["w_down"].double().T
        else:
            y = _experts64(l, d, h)
        x = x + _rms(y, d["norm2b"], eps)
    return _rms(x, top["final_norm"], eps)


def _rotate64(x, l, positions):
    dims, half = l.rot_dims, l.rot_dims // 2
    f = l.rot_base ** (-2.0 * torch.arange(half, device=DEV).double() / dims)

    def turn(t):
        return dims * math.log(l.rot_orig / (2.0 * math.pi * t)) / (2.0 * math.log(l.rot_base))

    lo, hi = max(math.floor(turn(l.rot_fast)), 0), min(math.ceil(turn(l.rot_slow)), dims - 1)
    ramp = ((torch.arange(half, device=DEV).double() - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    f = f / l.rot_factor * ramp + f * (1.0 - ramp)
    mag = 0.1 * math.log(l.rot_factor) + 1.0
    a = positions.double()[:, None] * f
    c, s = (a.cos() * mag)[:, None], (a.sin() * mag)[:, None]
    u, v = x[..., 0:dims:2], x[..., 1:dims:2]
    return torch.cat((torch.stack((u * c - v * s, v * c + u * s), -1).flatten(-2), x[..., dims:]), -1)


def _lenuzen64(cfg, top, layers, tok):
    T, eps = len(tok), cfg.norm_eps
    p = torch.arange(T, device=DEV)
    x = top["embed"][tok].double() * cfg.embed_scale
    for l, d in zip(cfg.layers, layers):
        H, G, D, V = l.heads, l.kv_heads, l.dim, l.vdim
        z = x @ d["w_in"].double().T
        if l.in_biased:
            z = z + d["in_bias"].double()
        q, k, v = z[:, :H * D], z[:, H * D:(H + G) * D], z[:, (H + G) * D:(H + G) * D + G * V].view(T, G, V)
        if l.talking:
            q, k = _rms(q, d["q_norm"], eps), _rms(k, d["kv_norm"], eps)
        q, k = _rotate64(q.view(T, H, D), l, p), _rotate64(k.view(T, G, D), l, p)
        if not l.talking:
            q, k, v = (t / torch.sqrt((t * t).mean(-1, keepdim=True) + eps) for t in (q, k, v))
        k, v = (t.repeat_interleave(H // G, 1).transpose(0, 1).contiguous() for t in (k, v))
        s = torch.matmul(q.transpose(0, 1).contiguous(), k.transpose(1, 2).contiguous()) * l.attn_scale
        if l.talking:
            s = (d["talk"].double() @ s.view(H, T * T)).view(H, T, T)
        else:
            s = s * d["head_temp"].double()[:, None, None]
        o = torch.matmul(_softmax_causal(s, 0, ("chunk" if l.talking else "window", l.mask_size), l.talking), v).transpose(0, 1)
        if l.out_gate:
            o = o * _sigmoid(z[:, -H:])[:, :, None]
        x = x + _layer_norm(o.flatten(1) @ d["w_o"].double().T, d["norm1b"], eps)
        x = x + _layer_norm(_gelu(x @ d["w_up"].double().T) @ d["w_down"].double().T, d["norm2b"], eps)
    return _layer_norm(x, top["final_norm"], eps)


def _layered_exact(case, seed):
    cfg, top, layers, tok, want = _layered_inputs(case, seed)
    forward = _sinulorn64 if case["design"] == "sinulorn" else _lenuzen64
    head = top["head"].double() * cfg.logit_scale
    n, m = case["n"], case["m"]
    greedy = m and case["decode"] == "greedy"
    ids = torch.as_tensor(tok[:n + m], device=DEV).long()
    if greedy:  # token by token over the whole sequence would be slow: take the next one from the classifier's rows and check it
        ids = torch.cat((ids[:n], (ids[n] + torch.arange(m + 1, device=DEV)) % cfg.vocab))
    y = forward(cfg, top, layers, ids)
    out = {"portion": y[torch.as_tensor(want, device=DEV).long()] @ head.T}
    if greedy:
        z = y[n:] @ head.T
        if not torch.equal(z[:m].argmax(1), ids[n + 1:]):
            return None
        out["tokens"], out["last"] = ids[n + 1:].to(torch.int32), z[m:]
    elif m:
        out["steps"] = [(y[n + i:n + i + 1] @ head.T) for i in range(m)]
    return out


def exact(case, seed):
    return _dense_exact(case, seed) if case["family"] == "dense" else _layered_exact(case, seed)
