"""The matmul work a GGUF engine has this library do, as cases that can be
timed: single decode projections, one decoder layer's projections, the
vocabulary head, a few rows at once (speculative verification), prompt
processing in each weight type that models are shipped in, and the
mixture-of-experts feed-forward at decode and prompt sizes.

``listed()`` are the cases, ``draw(rng)`` gives more of the same ranges,
``prepare`` makes a case's inputs on the GPU, ``run`` is one pass through the
package's entry points, ``exact`` the same results in 64 bits.

Weights and activations follow the distributions of the repository's
benchmark: uniform codes and sub-scales, fp16 block scales |N(0, 1)| * 0.01
(Q4_0 0.02), activations N(0, 1), prompt rows with 1 % outliers times 20.
Quantized-activation types multiply the activations as the int8 blocks that
the format defines (32 elements, scale amax / 127), so their exact result is
the 64-bit product of those blocks with the dequantized weights.
"""
import math

import torch

from laplace_amd.matmul import GGMLType, Tensor, matmul_gemm_batch, matmul_lm_head, matmul_rows, row_bytes
from laplace_amd.moe import moe_ffn

T = GGMLType
BLOCK = {T.Q4_0: (18, 32), T.Q5_0: (22, 32), T.Q8_0: (34, 32), T.Q2_K: (84, 256), T.Q3_K: (110, 256),
         T.Q4_K: (144, 256), T.Q5_K: (176, 256), T.Q6_K: (210, 256)}
INT8_ACT = (T.Q4_0, T.Q5_0, T.Q8_0, T.Q4_K, T.Q6_K)      # int8 activation blocks; the others take fp32 x
# byte offsets of the fp16 scale fields of a block
SCALES = {T.Q4_0: [0], T.Q5_0: [0], T.Q8_0: [0], T.Q2_K: [80, 82], T.Q3_K: [108], T.Q4_K: [0, 2],
          T.Q5_K: [0, 2], T.Q6_K: [208]}


def listed():
    return [
        # the smallest call: one token's fp32 router logits
        {"name": "router_f32_1", "kind": "rows", "type": "F32", "M": 1, "K": 2816, "N": 128},
        # every projection of one decoder layer for one token, 8B-class sizes, Q4_K with a Q6_K down
        {"name": "decode_layer_q4k", "kind": "layer", "type": "Q4_K", "down": "Q6_K", "H": 4096, "KV": 1024,
         "I": 14336},
        # one token against a 262144-word vocabulary
        {"name": "lm_head_q6k_1", "kind": "head", "type": "Q6_K", "M": 1, "K": 2816, "N": 262144},
        # 8 rows at once (verification of drafted tokens, or 8 sequences), 7B-class gate/up
        {"name": "verify_q4k_8", "kind": "rows", "type": "Q4_K", "M": 8, "K": 3584, "N": 18944},
        # a short prompt of odd length
        {"name": "prompt_q4_0_37", "kind": "rows", "type": "Q4_0", "M": 37, "K": 14336, "N": 4096},
        # prompt processing, one case for each weight type family
        {"name": "prefill_q4k_2048", "kind": "rows", "type": "Q4_K", "M": 2048, "K": 4096, "N": 14336},
        {"name": "prefill_q6k_509", "kind": "rows", "type": "Q6_K", "M": 509, "K": 18944, "N": 3584},
        {"name": "prefill_q8_0_512", "kind": "rows", "type": "Q8_0", "M": 512, "K": 4096, "N": 4096},
        {"name": "prefill_q5k_200", "kind": "rows", "type": "Q5_K", "M": 200, "K": 4096, "N": 14336},
        {"name": "prefill_bf16_512", "kind": "rows", "type": "BF16", "M": 512, "K": 4096, "N": 4096},
        # mixture of experts: 64 sequences' decode step, and a prompt
        {"name": "moe_q4k_64", "kind": "moe", "type": "Q4_K", "down": "Q4_K", "T": 64, "H": 2048, "E": 128,
         "top_k": 8, "I": 768},
        {"name": "moe_q4k_1000", "kind": "moe", "type": "Q4_K", "down": "Q4_K", "T": 1000, "H": 2048, "E": 128,
         "top_k": 8, "I": 768},
    ]


# no drawn case does more than the largest listed ones
MAX_MACS = 2048 * 4096 * 14336
MAX_WEIGHT_BYTES = 262144 * 2816 // 256 * 210


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["rows"] * 7 + ["layer", "head", "moe", "moe"])
    if kind == "rows":
        while True:
            c = {"kind": kind, "type": rng.choice([t.name for t in BLOCK] + ["F32", "F16", "BF16"]),
                 "M": _log(rng, 1, 2048), "K": 256 * _log(rng, 2, 74), "N": _log(rng, 128, 18944)}
            # fp32 products are the router's and the embedding's: small weights
            if c["M"] * c["K"] * c["N"] <= MAX_MACS // (16 if c["type"] == "F32" else 1):
                return c
    if kind == "layer":
        return {"kind": kind, "type": rng.choice(["Q4_K", "Q4_0", "Q8_0"]), "down": rng.choice(["Q4_K", "Q6_K", "Q8_0"]),
                "H": 256 * _log(rng, 4, 16), "KV": 128 * _log(rng, 2, 8), "I": 256 * _log(rng, 12, 56)}
    if kind == "head":
        while True:
            c = {"kind": kind, "type": rng.choice(["Q4_K", "Q6_K", "Q8_0"]), "M": _log(rng, 1, 4),
                 "K": 256 * _log(rng, 4, 16), "N": _log(rng, 32000, 262144)}
            if row_bytes(T[c["type"]], c["K"]) * c["N"] <= MAX_WEIGHT_BYTES:
                return c
    return {"kind": kind, "type": rng.choice(["Q4_K", "Q4_K", "Q8_0"]), "down": rng.choice(["Q4_K", "Q6_K", "Q8_0"]),
            "T": _log(rng, 1, 1000), "H": 256 * _log(rng, 4, 11), "E": rng.choice([32, 64, 128]),
            "top_k": rng.choice([2, 4, 8]), "I": 256 * rng.randint(1, 4)}


# ---------------------------------------------------------------- inputs

def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * seed + salt)
    return g


def _weights(t, K, N, g):
    """N rows of K elements of type t, as the bytes of a GGUF tensor."""
    if t in (T.F32, T.F16, T.BF16):
        v = torch.randn(N * K, generator=g, device="cuda") * 0.05
        return v.to({T.F32: torch.float32, T.F16: torch.float16, T.BF16: torch.bfloat16}[t]).view(torch.uint8)
    size, elems = BLOCK[t]
    n = N * (K // elems)
    w = torch.randint(0, 256, (n, size), generator=g, device="cuda", dtype=torch.uint8)
    if t == T.Q8_0:
        w[:, 2:] = torch.randint(-127, 128, (n, 32), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
    if t == T.Q6_K:
        w[:, 192:208] = torch.randint(-32, 32, (n, 16), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
    for o in SCALES[t]:
        s = torch.randn(n, generator=g, device="cuda").abs() * (0.02 if t == T.Q4_0 else 0.01)
        w[:, o:o + 2] = s.to(torch.float16).view(torch.uint8).view(n, 2)
    return w.view(-1)


def _tensor(t, K, N, g, mats=1):
    return Tensor(type=t, dims=(K, N, mats) if mats > 1 else (K, N), data=_weights(t, K, N * mats, g))


def _acts(M, K, g, outliers):
    x = torch.randn(M, K, generator=g, device="cuda")
    if outliers:
        x = torch.where(torch.rand(M, K, generator=g, device="cuda") < 0.01, x * 20, x)
    return x


def _empty(*shape):
    return torch.empty(*shape, dtype=torch.float32, device="cuda")


def prepare(case, seed):
    c, g = case, _gen(seed, 17)
    t = T[c["type"]]
    if c["kind"] in ("rows", "head"):
        return {"case": c, "w": _tensor(t, c["K"], c["N"], g), "x": _acts(c["M"], c["K"], g, c["M"] > 8),
                "y": _empty(c["M"], c["N"])}
    if c["kind"] == "layer":
        H, KV, I = c["H"], c["KV"], c["I"]
        w = {n: _tensor(t, H, r, g) for n, r in (("q", H), ("k", KV), ("v", KV), ("o", H), ("gate", I), ("up", I))}
        w["down"] = _tensor(T[c["down"]], I, H, g)
        y = {n: _empty(w[n].dims[1]) for n in w}
        # the activation rows that the norms, the attention and the gate hand to the projections
        x = {"attn": _acts(1, H, g, False), "o": _acts(1, H, g, False), "ffn": _acts(1, H, g, False),
             "down": _acts(1, I, g, False)}
        return {"case": c, "w": w, "x": {n: v.view(-1) for n, v in x.items()}, "y": y}
    H, E, I = c["H"], c["E"], c["I"]
    return {"case": c, "x": _acts(c["T"], H, g, False),
            "router": Tensor(T.F32, (H, E), (torch.randn(E * H, generator=g, device="cuda") * 0.5).view(torch.uint8)),
            "router_scale": 1 + 0.1 * torch.randn(H, generator=g, device="cuda"),
            "pre_norm": 1 + 0.1 * torch.randn(H, generator=g, device="cuda"),
            "gate_up": _tensor(t, H, 2 * I, g, E), "down": _tensor(T[c["down"]], I, H, g, E),
            "down_scale": 0.5 + torch.rand(E, generator=g, device="cuda"), "out": _empty(c["T"], H)}


# ---------------------------------------------------------------- one pass

def run(state):
    s, c = state, state["case"]
    if c["kind"] == "rows":
        matmul_rows(s["x"], s["w"], s["y"], c["M"], c["K"], c["N"])
        return s["y"]
    if c["kind"] == "head":
        matmul_lm_head(s["x"], s["w"], s["y"], c["M"], c["K"], c["N"])
        return s["y"]
    if c["kind"] == "layer":
        w, x, y, H, KV, I = s["w"], s["x"], s["y"], c["H"], c["KV"], c["I"]
        matmul_gemm_batch([(x["attn"], w["q"], y["q"], H, H), (x["attn"], w["k"], y["k"], H, KV),
                           (x["attn"], w["v"], y["v"], H, KV)])
        matmul_rows(x["o"], w["o"], y["o"], 1, H, H)
        matmul_gemm_batch([(x["ffn"], w["gate"], y["gate"], H, I), (x["ffn"], w["up"], y["up"], H, I)])
        matmul_rows(x["down"], w["down"], y["down"], 1, I, H)
        return y
    out, idx, wts = moe_ffn(s["x"], s["router"], s["router_scale"], s["pre_norm"], 1e-6, s["gate_up"], s["down"],
                            s["down_scale"], c["E"], c["top_k"], c["I"], out=s["out"], return_routing=True)
    return {"out": out, "experts": idx, "weights": wts}


def work(case):
    c = case
    if c["kind"] in ("rows", "head"):
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": row_bytes(T[c["type"]], K) * N + 4 * M * (K + N), "flops": 2 * M * K * N}
    if c["kind"] == "layer":
        H, KV, I = c["H"], c["KV"], c["I"]
        rows = 2 * H + 2 * KV + 2 * I
        return {"bytes": row_bytes(T[c["type"]], H) * rows + row_bytes(T[c["down"]], I) * H
                + 4 * (3 * H + I + rows + H), "flops": 2 * (H * rows + I * H)}
    Tk, H, E, I, k = c["T"], c["H"], c["E"], c["I"], c["top_k"]
    used = E * (1 - (1 - k / E) ** Tk)        # experts that some token takes
    expert = row_bytes(T[c["type"]], H) * 2 * I + row_bytes(T[c["down"]], I) * H
    return {"bytes": int(used * expert) + 4 * (E * H + 2 * H + E) + 4 * Tk * (2 * H + 2 * k),
            "flops": 2 * Tk * (E * H + k * 3 * H * I)}


def tolerance(case):
    """About four times the largest error against exact() that was measured
    over the listed and 16 drawn cases. fp32 sums of exact products: 2.4e-7.
    Q4_K beyond 16 rows: 8.4e-6, its matrix products split the activations in
    fp16 and fp8 parts. The mixture of experts quantizes its own intermediate
    rows, where a last-bit difference moves a code by one now and then: 7e-5;
    near-ties of two router logits may name another expert."""
    if case["kind"] == "moe":
        return {"rel": 3e-4, "differ": 1e-3}
    if case["type"] == "Q4_K" and case.get("M", 1) > 16:
        return {"rel": 4e-5}
    return {"rel": 1e-6}


# ---------------------------------------------------------------- 64 bits

def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _scale_min_k4(s):
    """The 8 six-bit (scale, min) pairs of [n, 12] bytes."""
    s = s.int()
    lo, hi = s[:, 0:4], s[:, 8:12]
    mid = s[:, 4:8]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)
    return sc.double(), mn.double()


def _values(t, data, K):
    """The weights as [rows, K] doubles."""
    if t in (T.F32, T.F16, T.BF16):
        return data.view({T.F32: torch.float32, T.F16: torch.float16, T.BF16: torch.bfloat16}[t]).double().view(-1, K)
    size, elems = BLOCK[t]
    b = data.view(-1, size)
    n = b.shape[0]

    def nibbles(q):                      # [n, 32 * j] bytes: low nibbles, then high, per 32 bytes
        q = q.reshape(n, -1, 32)
        return torch.stack([q & 15, q >> 4], 2).reshape(n, -1)

    if t == T.Q8_0:
        v = _f16(b[:, 0:2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif t in (T.Q4_0, T.Q5_0):
        q = b[:, 2:] if t == T.Q4_0 else b[:, 6:]
        v = torch.cat([q & 15, q >> 4], 1).int()
        if t == T.Q5_0:
            bits = torch.arange(8, device=b.device)
            v = v + 16 * ((b[:, 2:6].int()[:, :, None] >> bits) & 1).reshape(n, 32)
        v = _f16(b[:, 0:2]) * (v - (8 if t == T.Q4_0 else 16)).double()
    elif t in (T.Q4_K, T.Q5_K):
        sc, mn = _scale_min_k4(b[:, 4:16])
        q = nibbles(b[:, 16:144] if t == T.Q4_K else b[:, 48:176]).int().view(n, 8, 32)
        if t == T.Q5_K:
            bits = torch.arange(8, device=b.device)
            q = q + 16 * ((b[:, None, 16:48].int() >> bits[None, :, None]) & 1)
        v = (_f16(b[:, 0:2])[:, :, None] * sc[:, :, None] * q.double()
             - _f16(b[:, 2:4])[:, :, None] * mn[:, :, None])
    elif t == T.Q6_K:
        ql, qh = b[:, 0:128].int().view(n, 2, 2, 32), b[:, 128:192].int().view(n, 2, 1, 32)
        lo = torch.stack([ql & 15, ql >> 4], 2).view(n, 2, 4, 32)
        hi = (qh >> (2 * torch.arange(4, device=b.device)).view(1, 1, 4, 1)) & 3
        q = (lo + 16 * hi - 32).double().view(n, 16, 16)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = _f16(b[:, 208:210])[:, :, None] * sc[:, :, None] * q
    elif t == T.Q2_K:
        shift = (2 * torch.arange(4, device=b.device)).view(1, 1, 4, 1)
        q = ((b[:, 16:80].int().view(n, 2, 1, 32) >> shift) & 3).double().view(n, 16, 16)
        sc, mn = (b[:, 0:16] & 15).double(), (b[:, 0:16] >> 4).double()
        v = _f16(b[:, 80:82])[:, :, None] * sc[:, :, None] * q - _f16(b[:, 82:84])[:, :, None] * mn[:, :, None]
    else:                                # Q3_K
        shift = (2 * torch.arange(4, device=b.device)).view(1, 1, 4, 1)
        low = ((b[:, 32:96].int().view(n, 2, 1, 32) >> shift) & 3).view(n, 8, 32)
        bit = (b[:, None, 0:32].int() >> torch.arange(8, device=b.device).view(1, 8, 1)) & 1
        q = (low - 4 + 4 * bit).double().view(n, 16, 16)
        s = b[:, 96:108].int()
        low4 = torch.cat([s[:, 0:8] & 15, s[:, 0:8] >> 4], 1)
        high2 = torch.cat([(s[:, 8:12] >> (2 * j)) & 3 for j in range(4)], 1)
        v = _f16(b[:, 108:110])[:, :, None] * ((low4 | (high2 << 4)) - 32).double()[:, :, None] * q
    return v.reshape(-1, K)


def _int8_blocks(x):
    """Activations as their int8 blocks represent them (scale times code), in 64 bits."""
    b = x.float().cpu().reshape(-1, 32)           # on the CPU: its fp32 division rounds as IEEE asks
    d = b.abs().amax(1, keepdim=True) / 127.0
    inv = torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
    q = torch.round(b * inv).clamp(-128, 127)
    return (d.double() * q.double()).view(x.shape).to(x.device)


def _product(t, x, data, K):
    """x [M, K] times the rows of data, a million weight values at a time."""
    x = _int8_blocks(x) if t in INT8_ACT else x.double()
    nb = row_bytes(t, K)
    step = max(1, (1 << 27) // K)
    rows = data.numel() // nb
    return torch.cat([x @ _values(t, data[r * nb:min(r + step, rows) * nb], K).T for r in range(0, rows, step)], 1)


def exact(case, seed):
    c, s = case, prepare(case, seed)
    t = T[c["type"]]
    if c["kind"] in ("rows", "head"):
        return _product(t, s["x"], s["w"].data, c["K"])
    if c["kind"] == "layer":
        src = {"q": "attn", "k": "attn", "v": "attn", "o": "o", "gate": "ffn", "up": "ffn", "down": "down"}
        return {n: _product(w.type, s["x"][src[n]].view(1, -1), w.data, w.dims[0]).view(-1) for n, w in s["w"].items()}
    Tk, H, E, I, k = c["T"], c["H"], c["E"], c["I"], c["top_k"]
    x = s["x"].double()
    unit = x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-6)
    router = s["router"].data.view(torch.float32).double().view(E, H)
    p = torch.softmax((unit * s["router_scale"].double() / math.sqrt(H)) @ router.T, 1)
    wts, idx = torch.topk(p, k, 1)
    wts = wts / wts.sum(1, keepdim=True)
    e_in = unit * s["pre_norm"].double()
    gu_b, dn_b = row_bytes(t, H) * 2 * I, row_bytes(T[c["down"]], I) * H
    out = torch.zeros(Tk, H, dtype=torch.float64, device="cuda")
    for e in range(E):
        tok, slot = torch.nonzero(idx == e, as_tuple=True)
        if tok.numel() == 0:
            continue
        gu = _product(t, e_in[tok], s["gate_up"].data[e * gu_b:(e + 1) * gu_b], H)
        gate, up = gu[:, :I], gu[:, I:]
        hidden = 0.5 * gate * (1 + torch.tanh(0.7978845608028654 * (gate + 0.044715 * gate ** 3))) * up
        y = _product(T[c["down"]], hidden, s["down"].data[e * dn_b:(e + 1) * dn_b], I)
        out.index_add_(0, tok, y * (wts[tok, slot] * s["down_scale"][e].double())[:, None])
    return {"out": out, "experts": None, "weights": wts}
