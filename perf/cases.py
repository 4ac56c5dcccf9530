"""The work that a program using this framework has it do, as cases that can be timed and compared.

Kinds (the sizes are those of the framework's own model configurations and kernel sweep):

  gemv     one Q8_0 row dot product per output row, batch 1 (camelid_hip_q8_0_gemv): what a
           program that drives single kernels calls per projection of a decode step
  gemm     the same projection over a batch of prompt tokens (camelid_hip_q8_0_gemm)
  decode   greedy generation over a filled KV cache: one step that returns its logits
           (forward_token, as the seam samples the first token), then the device-side loop
           (generate) from its greedy token
  prefill  a prompt (or the next turn of a conversation, after `history` positions) through
           prefill, then the step of its last token with the logits: time to first token
  verify   a speculative draft of `tokens` tokens through verify_batch, all of it accepted, and
           the step after it with the logits

Engines hold a stage of each configuration's layers at their real widths (a pipeline stage is the
engine with fewer layers; every layer of one configuration is the same work) and its full
lm_head; TinyLlama is whole.  Weights are N(0, 0.02) in the configuration's GGUF formats, the KV
history is N(0, 1) rows handed over as seed_layer does after a CPU prefill.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from camelid_amd import _native
from camelid_amd.engine import PROJ_NAMES, Q4_K, Q6_K, Q8_0, HipResidentDecode
from camelid_amd.model import CONFIGS, QUANT_BYTES, rope_tables

# layers of the stage an engine case holds
STAGE = {"tinyllama-1.1b": 22, "llama-3.2-3b": 7, "mistral-7b-v0.3": 4, "qwen3-8b": 4}
SWEEP = [(2048, 2048), (5632, 2048), (2048, 5632), (32000, 2048), (128256, 3072)]


def listed():
    return [
        # the smallest call: one projection of a TinyLlama layer at batch 1
        {"name": "gemv 2048x2048", "kind": "gemv", "rows": 2048, "k": 2048},
        # the kernel sweep's prefill projection at its 512 tokens
        {"name": "gemm 5632x2048 x512", "kind": "gemm", "rows": 5632, "k": 2048, "tokens": 512},
        # chat on the smallest model: short context, launches and latency count
        {"name": "decode tinyllama p127", "kind": "decode", "model": "tinyllama-1.1b", "layers": 22, "history": 127,
         "steps": 16},
        # the headline benchmark's decode: 512-token prompt, Q8_0
        {"name": "decode llama3b p511", "kind": "decode", "model": "llama-3.2-3b", "layers": 7, "history": 511,
         "steps": 16},
        # long-context decode: attention over an 8K cache
        {"name": "decode mistral p8191", "kind": "decode", "model": "mistral-7b-v0.3", "layers": 4, "history": 8191,
         "steps": 8},
        # decode of a Q4_K_M model (Q4_K and Q6_K projections, QK-norm)
        {"name": "decode qwen p1023", "kind": "decode", "model": "qwen3-8b", "layers": 4, "history": 1023,
         "steps": 16},
        # a short question: an odd handful of tokens, small grids
        {"name": "prefill tinyllama 37", "kind": "prefill", "model": "tinyllama-1.1b", "layers": 22, "history": 0,
         "tokens": 37},
        # the headline prompt (n - 1 of its 512 tokens)
        {"name": "prefill llama3b 511", "kind": "prefill", "model": "llama-3.2-3b", "layers": 7, "history": 0,
         "tokens": 511},
        # a K-quant prompt of two chunks, the second one token short
        {"name": "prefill qwen 1023", "kind": "prefill", "model": "qwen3-8b", "layers": 4, "history": 0,
         "tokens": 1023},
        # a long document: the largest call, most of it causal attention
        {"name": "prefill mistral 8191", "kind": "prefill", "model": "mistral-7b-v0.3", "layers": 2, "history": 0,
         "tokens": 8191},
        # speculative decoding: the largest draft on the headline model
        {"name": "verify llama3b k8 p511", "kind": "verify", "model": "llama-3.2-3b", "layers": 7, "history": 511,
         "tokens": 8},
        # ... and an odd draft on the K-quant model, past 1024 positions
        {"name": "verify qwen k5 p1100", "kind": "verify", "model": "qwen3-8b", "layers": 4, "history": 1100,
         "tokens": 5},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemm", "decode", "prefill", "verify"])
    if kind in ("gemv", "gemm"):
        k = 32 * _log_int(rng, 32, 256)
        rows = _log_int(rng, 1000, 33000)
        if kind == "gemv":
            return {"kind": kind, "rows": rows, "k": k}
        return {"kind": kind, "rows": rows // 4 * 4, "k": k, "tokens": _log_int(rng, 2, 600)}
    model = rng.choice(sorted(STAGE))
    c = {"kind": kind, "model": model, "layers": STAGE[model]}
    if kind == "decode":
        return dict(c, history=_log_int(rng, 2, 8192), steps=_log_int(rng, 2, 16))
    if kind == "prefill":
        return dict(c, history=rng.choice([0, _log_int(rng, 2, 2048)]), tokens=_log_int(rng, 2, 1024))
    return dict(c, history=_log_int(rng, 16, 8192), tokens=rng.randint(2, 8))


# ------------------------------------------------------------------ weights in their GGUF formats
def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _q8_0(x):
    """Q8_0 blocks of x [n][32] and the values they hold in 64 bits."""
    amax = x.abs().amax(1, keepdim=True)
    d = (amax / 127).half()
    q = torch.round(x * (127 / amax)).clamp(-127, 127).to(torch.int8)
    return torch.cat([_bytes(d), _bytes(q)], 1), lambda: d.double() * q.double()


def _q4_k(x):
    """Q4_K superblocks of x [n][256]: 8 sub-blocks with 6-bit scales and minima."""
    n = x.shape[0]
    s = x.view(n, 8, 32)
    low = (-s.amin(2)).clamp_min(0)
    step = (s.amax(2) + low) / 15
    d, dmin = (step.amax(1) / 63).half(), (low.amax(1) / 63).half()
    sc = torch.round(step / d.float()[:, None]).clamp(0, 63).to(torch.int32)
    mn = torch.round(low / dmin.float()[:, None]).clamp(0, 63).to(torch.int32)
    ds, dm = d.double()[:, None] * sc, dmin.double()[:, None] * mn
    q = torch.round((s + dm.float()[..., None]) / ds.float()[..., None].clamp_min(1e-12)).clamp(0, 15).to(torch.int32)
    packed = torch.cat([sc[:, :4] | (sc[:, 4:] >> 4 << 6), mn[:, :4] | (mn[:, 4:] >> 4 << 6),
                        (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1).to(torch.uint8)
    nib = (q[:, 0::2] | (q[:, 1::2] << 4)).to(torch.uint8).reshape(n, 128)
    wire = torch.cat([_bytes(d[:, None]), _bytes(dmin[:, None]), packed, nib], 1)
    return wire, lambda: (ds[..., None] * q - dm[..., None]).reshape(n, 256)


def _q6_k(x):
    """Q6_K superblocks of x [n][256]: 16 sub-blocks with signed 8-bit scales."""
    n = x.shape[0]
    s = x.view(n, 16, 16)
    step = s.abs().amax(2) / 31
    d = (step.amax(1) / 127).half()
    sc = torch.round(step / d.float()[:, None]).clamp(1, 127).to(torch.int8)
    ds = d.double()[:, None] * sc.double()
    q = torch.round(s / ds.float()[..., None]).clamp(-32, 31).to(torch.int32)
    u = (q + 32).reshape(n, 2, 4, 32)  # half, quarter, value: quarter j holds values 32 j .. 32 j + 31
    lo, hi = u & 15, u >> 4
    ql = torch.cat([lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)], 2)
    qh = hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)
    wire = torch.cat([ql.reshape(n, 128).to(torch.uint8), qh.reshape(n, 64).to(torch.uint8), _bytes(sc),
                      _bytes(d[:, None])], 1)
    return wire, lambda: (ds[..., None] * q).reshape(n, 256)


def _matrix(gen, rows, k, quant):
    """N(0, 0.02) weights [rows][k]: their wire bytes, and their values in 64 bits on request."""
    make, width = {Q8_0: (_q8_0, 32), Q4_K: (_q4_k, 256), Q6_K: (_q6_k, 256)}[quant]
    wire, values = make(0.02 * _normal(gen, rows * k // width, width))
    return wire, lambda: values().view(rows, k)


def _host(t):
    return t.cpu().numpy()


def _model(case, seed):
    """The parts of a model and a conversation, in a fixed order of draws from `seed`: yields
    (name, layer, value) so that a user of them need not hold them all at once."""
    cfg = CONFIGS[case["model"]]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n = case.get("tokens", 0) + 1
    yield "embs", -1, 0.02 * _normal(gen, n, cfg.hidden)
    for i in range(case["layers"]):
        for p, (rows, k) in cfg.proj_shapes().items():
            yield p, i, _matrix(gen, rows, k, cfg.proj_quant(p))
        for p in ("attn_norm", "ffn_norm"):
            yield p, i, 1 + 0.1 * _normal(gen, cfg.hidden)
        if cfg.qk_norm:
            for p in ("q_norm", "k_norm"):
                yield p, i, 1 + 0.1 * _normal(gen, cfg.head_dim)
        for p in ("ck", "cv"):
            yield p, i, _normal(gen, cfg.n_kv_heads, case["history"], cfg.head_dim)
    yield "out_norm", -1, 1 + 0.1 * _normal(gen, cfg.hidden)
    yield "out", -1, _matrix(gen, cfg.vocab, cfg.hidden, cfg.output_quant())
    if case["kind"] == "decode":
        yield "token_embd", -1, _matrix(gen, cfg.vocab, cfg.hidden, cfg.embd_quant())


# ------------------------------------------------------------------ the passes
def _kernel_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rows, k, n = case["rows"], case["k"], case.get("tokens", 1)
    wire, values = _matrix(gen, rows, k, Q8_0)
    x = _normal(gen, n, k)
    resid = _normal(gen, n, rows) if case["kind"] == "gemv" else None
    return wire, values, x, resid


def prepare(case, seed):
    if case["kind"] in ("gemv", "gemm"):
        rows, k, n = case["rows"], case["k"], case.get("tokens", 1)
        wire, _, x, resid = _kernel_inputs(case, seed)
        lib = _native.lib()
        st = {"case": case, "lib": lib, "resid": resid,
              "wq": wire[:, 2:].contiguous(), "wd": wire[:, :2].contiguous(),  # the split layout of the device matrices
              "xq": torch.empty(n, k, dtype=torch.int8, device="cuda"),
              "xs": torch.empty(n, k // 32, dtype=torch.float32, device="cuda"),
              "y": torch.empty(n, rows, dtype=torch.float32, device="cuda")}
        for t in range(n):
            _native.check(lib.camelid_hip_quantize_q8_0(x[t].data_ptr(), k, st["xq"][t].data_ptr(),
                                                        st["xs"][t].data_ptr(), None))
        torch.cuda.synchronize()
        return st
    cfg = CONFIGS[case["model"]].scaled(n_layers=case["layers"])
    n, hist = case.get("tokens", 0), case["history"]
    max_pos = hist + n + 1 + case.get("steps", 0)
    eng = HipResidentDecode(cfg.engine_dims(max_pos))
    layer, st = {}, {"case": case, "eng": eng, "scale": cfg.scale()}
    for name, i, v in _model(case, seed):
        if name == "embs":
            st["embs"] = _host(v)
        elif name == "out":
            eng.set_output(layer["out_norm"], _host(v[0]), quant=cfg.output_quant())
        elif name == "token_embd":
            eng.set_embedding(_host(v[0]), quant=cfg.embd_quant())
        else:
            layer[name] = _host(v[0] if isinstance(v, tuple) else v)
        if name == "cv":
            eng.set_layer(i, layer, layer["attn_norm"], layer["ffn_norm"], layer.get("q_norm"), layer.get("k_norm"),
                          quants=[cfg.proj_quant(p) for p in PROJ_NAMES])
            if hist:
                eng.seed_layer(i, layer["ck"], layer["cv"], hist)
            layer = {}
    st["cos"], st["sin"] = rope_tables(cfg, 0, max_pos)
    if case["kind"] == "decode":
        eng.set_rope_table(st["cos"], st["sin"])
    return st


def run(st):
    case = st["case"]
    if case["kind"] == "gemv":
        _native.check(st["lib"].camelid_hip_q8_0_gemv(
            st["wq"].data_ptr(), st["wd"].data_ptr(), case["rows"], case["k"], st["xq"].data_ptr(),
            st["xs"].data_ptr(), st["y"].data_ptr(), st["resid"].data_ptr(), None))
        return st["y"]
    if case["kind"] == "gemm":
        _native.check(st["lib"].camelid_hip_q8_0_gemm(
            st["wq"].data_ptr(), st["wd"].data_ptr(), case["rows"], case["k"], st["xq"].data_ptr(),
            st["xs"].data_ptr(), case["tokens"], st["y"].data_ptr(), None, None))
        return st["y"]
    eng, embs, cos, sin, scale = st["eng"], st["embs"], st["cos"], st["sin"], st["scale"]
    hist, n = case["history"], case.get("tokens", 0)
    eng.set_filled(hist)
    out = {}
    if case["kind"] == "prefill":
        eng.prefill(embs[:n], cos[hist:hist + n], sin[hist:hist + n], scale)
    elif case["kind"] == "verify":
        out["tokens"] = eng.verify_batch(embs[:n], cos[hist:hist + n], sin[hist:hist + n], hist, scale)
        eng.set_filled(hist + n)
    pos = hist + n
    token = eng.forward_token(embs[n], cos[pos], sin[pos], pos, scale)
    out["logits"] = eng.last_logits
    if case["kind"] == "decode":
        out["tokens"] = eng.generate(token, pos + 1, case["steps"], scale)
    return out


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    if case["kind"] in ("gemv", "gemm"):
        rows, k, n = case["rows"], case["k"], case.get("tokens", 1)
        resid = 4 * rows if case["kind"] == "gemv" else 0
        return {"bytes": rows * k * 34 / 32 + n * (k * 36 / 32 + 4 * rows) + resid, "flops": 2 * rows * k * n}
    cfg = CONFIGS[case["model"]].scaled(n_layers=case["layers"])
    hist, n, steps = case["history"], case.get("tokens", 0), case.get("steps", 0)
    per_layer = sum(r * k for r, k in cfg.proj_shapes().values())
    head = cfg.vocab * cfg.hidden

    def attention(first, count):  # products and sums of `count` tokens from position `first` on
        return 4.0 * cfg.nq * cfg.n_layers * (count * first + count * (count + 1) / 2)

    # every decode step reads the weights and the filled cache once
    nbytes = sum(cfg.decode_bytes(hist + n + s) for s in range(steps + 1)) + 4 * cfg.vocab
    flops = (steps + 1) * 2.0 * (per_layer * cfg.n_layers + head) + attention(hist + n, steps + 1)
    if n:  # the batch reads the layers' weights and the history once and writes its own rows
        nbytes += cfg.weight_bytes() + n * 4 * cfg.hidden + cfg.kv_bytes_per_pos() * (hist + n)
        flops += 2.0 * n * per_layer * cfg.n_layers + attention(hist, n)
        if case["kind"] == "verify":
            flops += 2.0 * n * head
        else:  # (no logits of the prompt's earlier tokens)
            nbytes -= head * QUANT_BYTES[cfg.output_quant()]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # every f32 sum runs in the reference CPU path's order and every 16-bit or integer rounding
    # is its own: the results are its bits, whatever kernel computes them
    return "exact"


# ------------------------------------------------------------------ the same in 64 bits
def _rope64(cfg, pos):
    half = cfg.head_dim // 2
    f = cfg.rope_theta ** (-2.0 * np.arange(half) / cfg.head_dim)
    if cfg.rope_scaling == "llama3":
        turns = cfg.rope_orig_ctx * f / (2 * math.pi)
        s = np.clip((turns - cfg.rope_low) / (cfg.rope_high - cfg.rope_low), 0, 1)
        f = (1 - s) * f / cfg.rope_factor + s * f
    a = torch.from_numpy(np.outer(pos, f)).cuda()
    return a.cos(), a.sin()


def _rms64(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def exact(case, seed):
    if case["kind"] in ("gemv", "gemm"):
        st = prepare(case, seed)  # (its quantized activations are inputs of the pass)
        _, values, _, resid = _kernel_inputs(case, seed)
        n, k = case.get("tokens", 1), case["k"]
        x = (st["xq"].double().view(n, k // 32, 32) * st["xs"].double().view(n, k // 32, 1)).view(n, k)
        y = x @ values().T
        return y + resid.double() if resid is not None else y
    cfg = CONFIGS[case["model"]]
    hist, hd, rep = case["history"], cfg.head_dim, cfg.n_heads // cfg.n_kv_heads
    lay, x = {}, None
    for name, i, v in _model(case, seed):
        if name == "embs":
            x = v.double()
            n = x.shape[0]
            cos, sin = (t[:, None] for t in _rope64(cfg, np.arange(hist, hist + n)))
        elif i >= 0:
            lay[name] = v
        elif name == "out_norm":
            x = _rms64(x[-1:], v, cfg.eps)
        elif name == "out":
            return {"logits": (x @ v[1]().T)[0], "tokens": None} if case["kind"] != "prefill" else \
                {"logits": (x @ v[1]().T)[0]}
        if name != "cv":
            continue

        def rope(t):  # [n][heads][hd]
            a, b = (t[..., :hd // 2], t[..., hd // 2:]) if cfg.split_half else (t[..., 0::2], t[..., 1::2])
            a, b = a * cos - b * sin, a * sin + b * cos
            return torch.cat([a, b], -1) if cfg.split_half else torch.stack([a, b], -1).flatten(-2)

        h = _rms64(x, lay["attn_norm"], cfg.eps)
        q, k, val = ((h @ lay[p][1]().T).view(n, -1, hd) for p in "qkv")
        if cfg.qk_norm:
            q, k = _rms64(q, lay["q_norm"], cfg.eps), _rms64(k, lay["k_norm"], cfg.eps)
        q, k = rope(q), rope(k)
        past = torch.arange(hist + n, device="cuda")[None] <= torch.arange(hist, hist + n, device="cuda")[:, None]
        att = torch.empty(n, cfg.n_heads, hd, dtype=torch.float64, device="cuda")
        for g in range(cfg.n_kv_heads):
            keys = torch.cat([lay["ck"][g].half().double(), k[:, g]])
            vals = torch.cat([lay["cv"][g].half().double(), val[:, g]])
            for j in range(g * rep, (g + 1) * rep):
                s = (q[:, j] @ keys.T) / math.sqrt(hd)
                att[:, j] = torch.softmax(s.masked_fill(~past, -math.inf), -1) @ vals
        x = x + att.view(n, -1) @ lay["o"][1]().T
        h = _rms64(x, lay["ffn_norm"], cfg.eps)
        gate, up = h @ lay["gate"][1]().T, h @ lay["up"][1]().T
        x = x + (gate * torch.sigmoid(gate) * up) @ lay["down"][1]().T
        lay = {}
