"""What this framework is used for, as cases that can be run and timed.

Every case goes through a public entry point (`QuantizedLinear`, `GGMLLinear`, `MoEExperts`,
`gptq_quantize`, `CausalLM.generate`) on inputs made on the GPU from a seed. Weights are Gaussian
matrices quantized as a checkpoint's would be (min-max groups, AutoGPTQ packing; GGUF blocks whose
values are centred on zero); activations are Gaussian with a few large channels, as a decoder's
residual stream has.

`exact(case, seed)` gives the same outputs from the same inputs in float64 with plain torch.
"""
import math

import numpy as np
import torch

from webpytorch_amd import core, llm

DEV = "cuda"

# Decoder shapes of this repository's configurations and benchmark
QWEN2_05B = dict(L=24, H=896, NH=14, NKV=2, HD=64, I=4864, V=151936)
# the Qwen2.5-7B shape cut to four layers (hidden 3584, heads of 128: the launch-sequence decode)
QWEN25_7B_4 = dict(L=4, H=3584, NH=28, NKV=4, HD=128, I=18944, V=152064)
MODELS = {"qwen2_05b": QWEN2_05B, "qwen25_7b_4layers": QWEN25_7B_4}

# (K, N) of decoder projections: the 0.5B shape's q|k|v, o, gate, gate|up and down; the 7B and
# 8B classes' q|k|v, o, up and down
PROJECTIONS = ((896, 1152), (896, 896), (896, 4864), (896, 9728), (4864, 896), (3584, 4608), (3584, 3584),
               (4096, 4096), (4096, 6144), (4096, 11008), (11008, 4096))
GGUF_PROJECTIONS = ((1024, 1024), (2048, 8192), (4096, 1024), (4096, 4096), (4096, 6144), (4096, 14336),
                    (14336, 4096))
GGUF_TYPES = ("Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q4_0", "Q5_0", "IQ4_NL")


# ---- the cases ------------------------------------------------------------------------
def listed():
    return [
        # one decode token through one projection of the smallest decoder: a call is latency
        dict(name="int4_token", kind="linear", K=896, N=4864, M=1, bits=4, gs=128, x="f16", out="f32",
             act_order=False, bias=False),
        # a small batch of sequences decoded together: the weights are read once for six rows
        dict(name="int4_batch6", kind="linear", K=4096, N=11008, M=6, bits=4, gs=128, x="f16", out="f32",
             act_order=False, bias=False),
        # a prompt of 512 tokens through an act-order (desc_act) checkpoint's projection, fp16 in and out
        dict(name="int4_actorder_prompt512", kind="linear", K=4096, N=4096, M=512, bits=4, gs=128, x="f16",
             out="f16", act_order=True, bias=False),
        # a long prompt of fp32 activations (the engine's own) through q|k|v of the 7B class, with bias
        dict(name="int4_f32_prompt1500", kind="linear", K=3584, N=4608, M=1500, bits=4, gs=128, x="f32",
             out="f32", act_order=False, bias=True),
        # int8 with one scale per output channel, a short prompt
        dict(name="int8_channel_prompt128", kind="linear", K=4096, N=4096, M=128, bits=8, gs=4096, x="f16",
             out="f16", act_order=False, bias=False),
        # one decode token through a GGUF layer in the file's own Q4_K blocks
        dict(name="gguf_q4k_token", kind="gguf", type="Q4_K", K=4096, N=14336, M=1, x="f32", out="f32"),
        # a prompt of 512 tokens through the same layer
        dict(name="gguf_q4k_prompt512", kind="gguf", type="Q4_K", K=4096, N=14336, M=512, x="f16", out="f32"),
        # a prompt through a file in an older block type (Q4_0), the engine's fp32 activations
        dict(name="gguf_q4_0_prompt77", kind="gguf", type="Q4_0", K=4096, N=4096, M=77, x="f32", out="f32"),
        # one sparse-MoE block (routing, 128 experts of which 8 per token, combine) for 256 tokens
        dict(name="moe_256", kind="moe", T=256, H=2048, E=128, I=768, top_k=8, x="f16"),
        # quantize-on-load of one fp16 projection as a HuggingFace directory holds it, (out, in)
        dict(name="quantize_on_load", kind="quantize", K=4096, N=14336, bits=4, gs=128, w="f16", from_out_in=True),
        # the prefill of a 700-token prompt: every layer, the KV cache and the first new token
        dict(name="model_prefill700", kind="model", model="qwen2_05b", prompt=700, new=1, lmax=1024),
        # a whole greedy generation: a prompt of 64 tokens and 64 new ones
        dict(name="model_decode64", kind="model", model="qwen2_05b", prompt=64, new=64, lmax=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "gguf", "gguf", "moe", "quantize", "model"])
    if kind == "linear":
        bits = rng.choice([4, 4, 4, 8])
        if rng.random() < 0.6:
            K, N = rng.choice(PROJECTIONS)
        else:  # other widths: K whole groups of 128, N whole packed words
            K, N = 128 * rng.randint(2, 64), 8 * rng.randint(16, 1400)
        gs = rng.choice([128, 128, 128, 64, 32] + ([K] if bits == 8 else []))
        return dict(kind=kind, K=K, N=N, M=_log(rng, 1, 2048), bits=bits, gs=gs, x=rng.choice(["f16", "f32"]),
                    out=rng.choice(["f32", "f32", "f16"]), act_order=gs < K and rng.random() < 0.25,
                    bias=rng.random() < 0.3)
    if kind == "gguf":
        K, N = rng.choice(GGUF_PROJECTIONS)
        if rng.random() < 0.4:
            K, N = 256 * rng.randint(2, 32), rng.randint(130, 9000)
        return dict(kind=kind, type=rng.choice(GGUF_TYPES), K=K, N=N, M=_log(rng, 1, 700), x=rng.choice(["f16", "f32"]),
                    out=rng.choice(["f32", "f32", "f16"]))
    if kind == "moe":
        E, k = rng.choice([(8, 2), (60, 4), (64, 6), (128, 8)])
        return dict(kind=kind, T=_log(rng, 1, 900), H=128 * rng.randint(6, 20), E=E, I=128 * rng.randint(4, 12),
                    top_k=k, x=rng.choice(["f16", "f32"]))
    if kind == "quantize":
        gs = rng.choice([32, 64, 128])
        return dict(kind=kind, K=gs * rng.randint(8, 4096 // gs), N=8 * rng.randint(64, 1800), bits=rng.choice([4, 4, 8]),
                    gs=gs, w=rng.choice(["f16", "f32"]), from_out_in=rng.random() < 0.8)
    model = rng.choice(["qwen2_05b", "qwen2_05b", "qwen25_7b_4layers"])
    if rng.random() < 0.5:
        return dict(kind=kind, model=model, prompt=_log(rng, 9, 1000), new=1, lmax=1024)
    return dict(kind=kind, model=model, prompt=_log(rng, 1, 120), new=rng.randint(5, 60), lmax=rng.choice([200, 256, 512]))


# ---- inputs ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000003 + 17)
    return g


def _dtype(s):
    return torch.float16 if s == "f16" else torch.float32


def _rows(g, M, K, dt):
    """Activations: N(0, 1) with one channel in 64 eight times as large."""
    big = 1.0 + 7.0 * (torch.rand(K, device=DEV, generator=g) < 1 / 64).float()
    return (torch.randn((M, K), device=DEV, generator=g) * big).to(_dtype(dt))


def _weights(g, K, N):
    return torch.randn((K, N), device=DEV, generator=g) / math.sqrt(K)


def _pack(q, bits, dim):
    """Codes packed 32 / bits to a word along `dim` (0: rows of a column, 1: columns of a row)."""
    per = 32 // bits
    q = q.to(torch.int32)
    v = q.reshape(q.shape[0] // per, per, q.shape[1]) if dim == 0 else q.reshape(q.shape[0], q.shape[1] // per, per)
    w = torch.zeros_like(v.select(1 if dim == 0 else 2, 0))
    for j in range(per):
        w |= v.select(1 if dim == 0 else 2, j) << (bits * j)
    return w


def _unpack(w, bits, dim):
    per, mask = 32 // bits, (1 << bits) - 1
    parts = [(w >> (bits * j)) & mask for j in range(per)]
    return (torch.stack(parts, 1).reshape(-1, w.shape[1]) if dim == 0
            else torch.stack(parts, 2).reshape(w.shape[0], -1))


def _autogptq(W, gs, bits):
    """AutoGPTQ tensors of W (K, N): asymmetric min-max groups along K, fp16 scales, zero - 1."""
    K, N = W.shape
    qmax = (1 << bits) - 1
    Wg = W.reshape(K // gs, gs, N)
    lo, hi = Wg.amin(1), Wg.amax(1)
    s = ((hi - lo) / qmax).half()
    s32 = s.float()
    z = (-lo / s32).round_().clamp_(1, qmax)
    q = (Wg / s32[:, None]).round_().add_(z[:, None]).clamp_(0, qmax).reshape(K, N)
    return {"qweight": _pack(q, bits, 0), "qzeros": _pack(z - 1, bits, 1), "scales": s}


def _dense(d, gs, bits, zoff=1):
    """float64 (K, N) of GPTQ tensors whose rows are in group order."""
    q = _unpack(d["qweight"], bits, 0).double()
    z = _unpack(d["qzeros"], bits, 1).double() + zoff
    s = d["scales"].double()
    G = s.shape[0]
    return ((q.reshape(G, gs, -1) - z[:, None]) * s[:, None]).reshape(q.shape)


def _linear_inputs(c, seed):
    g = _gen(seed)
    K, N, gs, bits = c["K"], c["N"], c["gs"], c["bits"]
    d = _autogptq(_weights(g, K, N), gs, bits)  # rows in group order
    d["bias"] = torch.randn(N, device=DEV, generator=g) * 0.02 if c["bias"] else None
    d["x"] = _rows(g, c["M"], K, c["x"])
    d["g_idx"] = None
    if c["act_order"]:  # the checkpoint's rows in shuffled order, row k of group g_idx[k]
        order = torch.randperm(K, device=DEV, generator=g)
        d["rows"] = order
        d["g_idx"] = (order // gs).to(torch.int32)
    return d


def _blocks_f16(v):
    return v.half().contiguous().view(torch.uint8)


def _gguf_raw(g, t, K, N):
    """(blocks, bytes) of N rows of a block type, values centred on zero with sd near 1 / sqrt(K)."""
    rnd = lambda n, w: torch.randint(0, 256, (n, w), dtype=torch.uint8, device=DEV, generator=g)  # noqa: E731
    per_block = 256 if t.endswith("_K") else 32
    n = N * K // per_block
    spread = torch.rand((n, 1), device=DEV, generator=g) * 0.5 + 0.75
    sd = 1.0 / math.sqrt(K)
    if t in ("Q4_K", "Q5_K"):  # d sc c - dmin m with m = sc and dmin the middle code times d
        mid, rms = (7.5, 4.61) if t == "Q4_K" else (15.5, 9.23)
        d = spread * (sd / rms / 48)
        sc = torch.randint(32, 64, (n, 8), dtype=torch.uint8, device=DEV, generator=g)
        pk = torch.empty((n, 12), dtype=torch.uint8, device=DEV)
        pk[:, 0:4] = (sc[:, 0:4] & 63) | ((sc[:, 4:8] >> 4) << 6)
        pk[:, 4:8] = pk[:, 0:4]
        pk[:, 8:12] = (sc[:, 4:8] & 15) | ((sc[:, 4:8] & 15) << 4)
        return torch.cat([_blocks_f16(d), _blocks_f16(d * mid), pk, rnd(n, 128 if t == "Q4_K" else 160)], 1)
    if t == "Q6_K":
        sc = (torch.randint(32, 64, (n, 16), device=DEV, generator=g) *
              (1 - 2 * torch.randint(0, 2, (n, 16), device=DEV, generator=g))).to(torch.int8).view(torch.uint8)
        return torch.cat([rnd(n, 192), sc, _blocks_f16(spread * (sd / 18.5 / 48))], 1)
    rms = {"Q8_0": 73.9, "Q4_0": 4.61, "Q5_0": 9.23, "IQ4_NL": 67.0}[t]
    return torch.cat([_blocks_f16(spread * (sd / rms)), rnd(n, {"Q8_0": 32, "Q4_0": 16, "Q5_0": 20, "IQ4_NL": 16}[t])], 1)


_IQ4_NL = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _gguf_dense(raw, t, K, N):
    """float64 (N, K) of GGUF blocks, value by value as the formats are defined."""
    f16 = lambda b: b.contiguous().view(torch.float16).double()  # noqa: E731
    b = raw
    if t in ("Q4_K", "Q5_K"):
        d, dmin, pk = f16(b[:, 0:2]), f16(b[:, 2:4]), b[:, 4:16].int()
        sc = torch.cat([pk[:, 0:4] & 63, (pk[:, 8:12] & 15) | ((pk[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([pk[:, 4:8] & 63, (pk[:, 8:12] >> 4) | ((pk[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, -128:].int().reshape(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)  # sub-blocks 2g low, 2g + 1 high
        if t == "Q5_K":
            qh = b[:, 16:48].int()[:, None, :]
            q = q + (((qh >> torch.arange(8, device=DEV)[None, :, None]) & 1) << 4)
        v = (d * sc)[:, :, None] * q.double() - (dmin * mn)[:, :, None]
    elif t == "Q6_K":
        ql, qh = b[:, 0:128].int().reshape(-1, 2, 64), b[:, 128:192].int().reshape(-1, 2, 32)
        sc, d = b[:, 192:208].contiguous().view(torch.int8).double(), f16(b[:, 208:210])
        parts = [((ql[:, :, 32 * (j & 1):32 * (j & 1) + 32] >> (4 * (j >> 1))) & 15) | (((qh >> (2 * j)) & 3) << 4)
                 for j in range(4)]
        q = (torch.stack(parts, 2).reshape(-1, 16, 16) - 32).double()
        v = q * (sc * d)[:, :, None]
    elif t == "Q8_0":
        v = f16(b[:, 0:2]) * b[:, 2:34].contiguous().view(torch.int8).double()
    else:
        qs = b[:, -16:].int()
        q = torch.cat([qs & 15, qs >> 4], 1)
        if t == "Q5_0":
            qh = b[:, 2:6].contiguous().view(torch.int32)
            q = (q | (((qh >> torch.arange(32, device=DEV, dtype=torch.int32)) & 1) << 4)) - 16
        elif t == "Q4_0":
            q = q - 8
        else:
            q = torch.tensor(_IQ4_NL, device=DEV)[q.long()]
        v = f16(b[:, 0:2]) * q.double()
    return v.reshape(N, K)


def _moe_inputs(c, seed):
    g = _gen(seed)
    E, H, I = c["E"], c["H"], c["I"]
    experts = [{n: _autogptq(_weights(g, K, N), 128, 4) for n, K, N in (("gate", H, I), ("up", H, I), ("down", I, H))}
               for _ in range(E)]
    return experts, _rows(g, c["T"], H, c["x"]), torch.randn((c["T"], E), device=DEV, generator=g) * 2.0


def _model_inputs(c, seed):
    """Device tensors of a random decoder (as a checkpoint directory holds them) and a prompt."""
    g = _gen(seed)
    s = MODELS[c["model"]]
    H, HD, NH, NKV, I, V = (s[k] for k in ("H", "HD", "NH", "NKV", "I", "V"))

    def lin(K, N, bias=False):
        d = _autogptq(_weights(g, K, N), 128, 4)
        if bias:
            d["bias"] = (torch.randn(N, device=DEV, generator=g) * 0.02).half()
        return d

    def norm():
        return (1.0 + 0.02 * torch.randn(H, device=DEV, generator=g)).float()
    layers = [{"q": lin(H, NH * HD, True), "k": lin(H, NKV * HD, True), "v": lin(H, NKV * HD, True),
               "o": lin(NH * HD, H), "gate": lin(H, I), "up": lin(H, I), "down": lin(I, H), "in_ln": norm(),
               "post_ln": norm()} for _ in range(s["L"])]
    embed = (torch.randn((V, H), device=DEV, generator=g) * 0.02).half()
    w = {"layers": layers, "embed": embed, "final_norm": norm(), "cfg": dict(s, gs=128, bits=4, eps=1e-6, theta=1e6)}
    ids = torch.randint(0, V, (c["prompt"],), device=DEV, generator=g).tolist()
    return w, ids


def prepare(case, seed):
    c = case
    if c["kind"] == "linear":
        d = _linear_inputs(c, seed)
        qw = d["qweight"]
        if c["act_order"]:  # file order: row k holds group-order row rows[k]
            qw = _pack(_unpack(qw, c["bits"], 0)[d["rows"]], c["bits"], 0)
        layer = core.QuantizedLinear.from_autogptq(qw, d["qzeros"], d["scales"], d["bias"], c["gs"], c["bits"],
                                                   g_idx=d["g_idx"])
        return {"kind": "call", "f": layer.forward, "x": d["x"], "out": _dtype(c["out"])}
    if c["kind"] == "gguf":
        g = _gen(seed)
        layer = core.GGMLLinear(_gguf_raw(g, c["type"], c["K"], c["N"]), c["type"], c["K"], c["N"])
        return {"kind": "call", "f": layer.forward, "x": _rows(g, c["M"], c["K"], c["x"]), "out": _dtype(c["out"])}
    if c["kind"] == "moe":
        experts, x, logits = _moe_inputs(c, seed)
        ex = core.MoEExperts([{n: core.QuantizedLinear.from_autogptq(d["qweight"], d["qzeros"], d["scales"], None, 128, 4)
                               for n, d in e.items()} for e in experts])
        return {"kind": "moe", "f": ex, "x": x, "logits": logits, "top_k": c["top_k"]}
    if c["kind"] == "quantize":
        W = _weights(_gen(seed), c["K"], c["N"])
        W = (W.t().contiguous() if c["from_out_in"] else W).to(_dtype(c["w"]))
        return {"kind": "quantize", "W": W, "gs": c["gs"], "bits": c["bits"], "from_out_in": c["from_out_in"]}
    w, ids = _model_inputs(c, seed)
    w["embed"] = w["embed"].cpu().numpy()
    return {"kind": "model", "m": llm.CausalLM.from_weights(w, lmax=c["lmax"]), "ids": ids, "new": c["new"]}


def run(state):
    s = state
    if s["kind"] == "call":
        return s["f"](s["x"], out_dtype=s["out"])
    if s["kind"] == "moe":
        return s["f"](s["x"], s["logits"], s["top_k"])
    if s["kind"] == "quantize":
        return core.gptq_quantize(s["W"], s["gs"], s["bits"], s["from_out_in"])
    m, n = s["m"], len(s["ids"]) + s["new"] - 1
    r = m.generate(s["ids"], s["new"])
    return {"tokens": np.array(r.tokens), "logits": m.buf["logits"], "k": m.kc[:, :, :n], "v": m.vc[:, :, :n]}


# ---- what a pass cannot do without -----------------------------------------------------
def _size(s):
    return 2 if s == "f16" else 4


def _gptq_bytes(K, N, gs, bits, scale=2):
    return K * N * bits / 8 + (K // gs) * N * (bits / 8 + scale)


def work(case):
    c = case
    if c["kind"] == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": _gptq_bytes(K, N, c["gs"], c["bits"]) + M * K * _size(c["x"]) + M * N * _size(c["out"]) +
                (4 * N if c["bias"] else 0) + (4 * K if c["act_order"] else 0), "flops": 2.0 * M * K * N}
    if c["kind"] == "gguf":
        M, K, N = c["M"], c["K"], c["N"]
        vals, blk = {"Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210), "Q8_0": (32, 34), "Q4_0": (32, 18),
                     "Q5_0": (32, 22), "IQ4_NL": (32, 18)}[c["type"]]
        return {"bytes": N * K // vals * blk + M * K * _size(c["x"]) + M * N * _size(c["out"]), "flops": 2.0 * M * K * N}
    if c["kind"] == "moe":
        T, H, E, I, k = (c[n] for n in ("T", "H", "E", "I", "top_k"))
        used = E * (1.0 - (1.0 - k / E) ** T)  # experts that some token picks, on average
        per = 2 * _gptq_bytes(H, I, 128, 4) + _gptq_bytes(I, H, 128, 4)
        return {"bytes": used * per + T * H * (_size(c["x"]) + 4) + T * E * 4, "flops": 6.0 * T * k * H * I}
    if c["kind"] == "quantize":
        K, N = c["K"], c["N"]
        return {"bytes": K * N * _size(c["w"]) + _gptq_bytes(K, N, c["gs"], c["bits"], 4), "flops": 4.0 * K * N}
    s = MODELS[c["model"]]
    H, HD, NH, NKV, I, V, L = (s[k] for k in ("H", "HD", "NH", "NKV", "I", "V", "L"))
    shapes = ((H, (NH + 2 * NKV) * HD), (NH * HD, H), (H, 2 * I), (I, H))
    layer = sum(_gptq_bytes(K, N, 128, 4) for K, N in shapes)
    head = _gptq_bytes(H, V, 128, 4, 4)
    mac = sum(K * N for K, N in shapes)
    T, new = c["prompt"], c["new"]
    n = T + new - 1                                           # positions that are computed
    keys = n * (n + 1) // 2                                   # (query, key) pairs of one head
    dec = sum(range(T, n))                                    # cached positions the decode steps read
    return {"bytes": new * (L * layer + head + 4 * V) + L * NKV * HD * 8 * (n + dec) + n * H * 2,
            "flops": 2.0 * (n * L * mac + new * H * V) + 4.0 * L * NH * HD * keys}


def tolerance(case):
    c = case
    if c["kind"] == "quantize":
        return "exact"
    # about four times the distance from float64 seen over the ranges that `draw` gives
    if c["kind"] == "model":  # fp32 through every layer; a prompt's products carry about 22 bits of each row
        return {"rel": 6e-6, "max": 3e-5, "differ": 0.02}
    if c.get("out") == "f16":  # the output's own rounding
        return {"rel": 8e-4, "max": 2e-3}
    return {"rel": 1.5e-6, "max": 8e-6}


# ---- the same in float64 ---------------------------------------------------------------
def _exact_moe(c, seed):
    experts, x, logits = _moe_inputs(c, seed)
    x = x.double()
    w, e = torch.softmax(logits.double(), 1).topk(c["top_k"], 1)
    w = w / w.sum(1, keepdim=True)
    out = torch.zeros_like(x)
    for i, ex in enumerate(experts):
        t, j = (e == i).nonzero(as_tuple=True)
        if t.numel():
            D = {n: _dense(d, 128, 4) for n, d in ex.items()}
            gate = x[t] @ D["gate"]
            out.index_add_(0, t, (gate * torch.sigmoid(gate) * (x[t] @ D["up"])) @ D["down"] * w[t, j][:, None])
    return out


def _quantize_f32(W, gs, bits):
    """(scales float32, zeros, codes) of W (K, N), the quantizer's float32 arithmetic."""
    K, N = W.shape
    qmax = (1 << bits) - 1
    Wg = W.float().reshape(K // gs, gs, N)
    lo, hi = Wg.amin(1), Wg.amax(1)
    # divided by tensors: torch turns a division by a number into a product with its reciprocal
    s = (hi - lo) / torch.full_like(lo, qmax)
    s = torch.where(s == 0, torch.full_like(s, 1e-8), s)
    z = (-lo / s).round().clamp(0, qmax)
    q = ((Wg / s[:, None]).round() + z[:, None]).clamp(0, qmax)
    return s, z, q.reshape(K, N)


def _exact_model(c, seed):
    w, ids = _model_inputs(c, seed)
    s = MODELS[c["model"]]
    H, HD, NH, NKV, I, L = (s[k] for k in ("H", "HD", "NH", "NKV", "I", "L"))
    lays = [{n: _dense(lay[n], 128, 4) for n in ("q", "k", "v", "o", "gate", "up", "down")} for lay in w["layers"]]
    sc, z, q = _quantize_f32(w["embed"].t(), 128, 4)  # the tied head, quantized on load
    head = ((q.double().reshape(-1, 128, s["V"]) - z.double()[:, None]) * sc.double()[:, None]).reshape(H, -1)
    del q
    rms = lambda x, g: x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * g.double()  # noqa: E731
    n_all = c["prompt"] + c["new"] - 1
    ang = torch.arange(n_all, device=DEV).double()[:, None] / (1e6 ** (torch.arange(0, HD, 2, device=DEV).double() / HD))
    cos, sin = torch.cos(ang).repeat(1, 2), torch.sin(ang).repeat(1, 2)
    kc = torch.zeros((L, NKV, n_all, HD), dtype=torch.float64, device=DEV)
    vc = torch.zeros_like(kc)

    def rope(t, p0):  # (T, heads, HD)
        T = t.shape[0]
        rot = torch.cat([-t[..., HD // 2:], t[..., :HD // 2]], -1)
        return t * cos[p0:p0 + T, None] + rot * sin[p0:p0 + T, None]

    def forward(tok, p0):
        T = len(tok)
        h = w["embed"][torch.tensor(tok, device=DEV)].double()
        mask = torch.arange(p0 + T, device=DEV)[None, :] > torch.arange(p0, p0 + T, device=DEV)[:, None]
        for i, (lay, D) in enumerate(zip(w["layers"], lays)):
            x = rms(h, lay["in_ln"])
            q, k, v = ((x @ D[n] + lay[n]["bias"].double()).reshape(T, -1, HD) for n in ("q", "k", "v"))
            kc[i, :, p0:p0 + T] = rope(k, p0).transpose(0, 1)
            vc[i, :, p0:p0 + T] = v.transpose(0, 1)
            q = rope(q, p0)
            att = torch.empty((T, NH, HD), dtype=torch.float64, device=DEV)
            for hd in range(NH):
                kv = hd // (NH // NKV)
                sc_ = (q[:, hd] @ kc[i, kv, :p0 + T].t().contiguous()) / math.sqrt(HD)
                att[:, hd] = torch.softmax(sc_.masked_fill(mask, -math.inf), -1) @ vc[i, kv, :p0 + T]
            h = h + att.reshape(T, -1) @ D["o"]
            x = rms(h, lay["post_ln"])
            gate = x @ D["gate"]
            h = h + (gate * torch.sigmoid(gate) * (x @ D["up"])) @ D["down"]
        return rms(h[-1:], w["final_norm"]) @ head

    logits = forward(ids, 0)
    tokens = [int(logits.argmax())]
    while len(tokens) < c["new"]:
        logits = forward([tokens[-1]], c["prompt"] + len(tokens) - 1)
        tokens.append(int(logits.argmax()))
    return {"tokens": np.array(tokens), "logits": logits, "k": kc, "v": vc}


def exact(case, seed):
    c = case
    if c["kind"] == "linear":
        d = _linear_inputs(c, seed)
        W = _dense(d, c["gs"], c["bits"])
        if c["act_order"]:
            W = W[d["rows"]]
        y = d["x"].double() @ W
        return y if d["bias"] is None else y + d["bias"].double()
    if c["kind"] == "gguf":
        g = _gen(seed)
        W = _gguf_dense(_gguf_raw(g, c["type"], c["K"], c["N"]), c["type"], c["K"], c["N"])
        return _rows(g, c["M"], c["K"], c["x"]).double() @ W.t().contiguous()
    if c["kind"] == "moe":
        return _exact_moe(c, seed)
    if c["kind"] == "quantize":
        s = prepare(c, seed)
        sc, z, q = _quantize_f32(s["W"].t() if c["from_out_in"] else s["W"], c["gs"], c["bits"])
        return [_pack(q, c["bits"], 0), _pack(z, c["bits"], 1), sc, c["K"], c["N"]]
    return _exact_model(c, seed)
