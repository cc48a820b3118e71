"""Performance cases of the quantized matmul path and of the inference backend built on it.

A case is one call a program makes: a projection (`hq_gemm`), the SwiGLU FFN input
(`hq_gemm_swiglu`), the option readout (`hq_gather_dot_dev`), or a forward pass of a small model
through the backend's vtable. `listed()` names the fixed ones, `draw()` gives more of the same ranges.
Shapes are those of the repository's workloads (synth.py): FFN 9728 x 2560 and 9216 x 2560, attention
widths 4096 / 1024, the 151936 x 2560 head and the 4-layer, 512-wide Llama-architecture model.

Inputs are made on the GPU by torch from the seed alone; weights reach the library as GGUF blocks in
host memory, as a program holding a model file has them. `exact()` decodes the same blocks in torch
and computes in float64.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hilbert-pruned-8b_amd"))
import hq  # noqa: E402

TYPES = {"Q8_0": hq.Q8_0, "Q2_K": hq.Q2_K, "Q3_K": hq.Q3_K, "Q4_K": hq.Q4_K, "Q5_K": hq.Q5_K, "Q6_K": hq.Q6_K}
DEV = "cuda:0"
EPS, THETA = 1e-5, 10000.0


def gemm(name, type, M, N, K, out="f16", acc=False):
    return dict(name=name, kind="gemm", type=type, M=M, N=N, K=K, out=out, acc=acc)


def model(name, type, T, prefix, layers=4, hidden=512, ffn=1408, heads=8, kv_heads=8, head_dim=64, vocab=32000, ids=32):
    return dict(name=name, kind="model", type=type, T=T, prefix=prefix, layers=layers, hidden=hidden, ffn=ffn, heads=heads,
                kv_heads=kv_heads, head_dim=head_dim, vocab=vocab, ids=ids)


def listed():
    return [
        # one token's gate or up projection: the smallest call, launch and weight stream only
        gemm("decode_q4k_up", "Q4_K", 1, 9728, 2560),
        # sixteen sequences decoded together, Q8_0 file
        gemm("batch16_q8_up", "Q8_0", 16, 9728, 2560),
        # a ragged decode batch through the Q6_K down projection of a Q4_K_M file, added to the residual
        gemm("batch37_q6k_down", "Q6_K", 37, 2560, 9728, "f32", True),
        # a short prompt on a Q8_0 file
        gemm("prompt128_q8_up", "Q8_0", 128, 9728, 2560),
        # a prompt of odd length through the attention query projection of a Q5_K_M file
        gemm("prompt301_q5k_q", "Q5_K", 301, 4096, 2560, "f32"),
        # the 512-token prompt: up projection, and the down projection added to the residual
        gemm("prompt512_q4k_up", "Q4_K", 512, 9728, 2560),
        gemm("prompt512_q4k_down", "Q4_K", 512, 2560, 9728, "f32", True),
        # its FFN input with gate and up as one resident pair
        dict(name="prompt512_q4k_swiglu", kind="swiglu", type="Q4_K", M=512, N=9216, K=2560),
        # 64 sequences of 256 tokens through one FFN projection: the largest
        gemm("batch16384_q4k_up", "Q4_K", 16384, 9216, 2560),
        # option scores of 256 states, 8 options each, from the resident head
        dict(name="readout256x8_q8", kind="readout", type="Q8_0", B=256, k=8, N=151936, K=2560),
        # a whole prompt through the model, scored at the end
        model("model_prompt2048", "Q8_0", 2048, 0),
        # one more token behind a cached context
        model("model_token_at1000", "Q8_0", 1, 1000),
    ]


MOST_FLOPS = 2 * 16384 * 9216 * 2560  # of a drawn case: the largest listed one's


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "gemm", "swiglu", "readout", "model", "model"])
    type = rng.choice(["Q4_K", "Q4_K", "Q4_K", "Q8_0", "Q8_0", "Q6_K", "Q5_K", "Q3_K", "Q2_K"])
    per = 32 if type == "Q8_0" else 256
    if kind in ("gemm", "swiglu"):
        M = 1 if rng.random() < 0.2 else _log_int(rng, 2, 8192)
        # widths of a layer of hidden size 1024 .. 4096: its own, kv, q and FFN ones, now and then a ragged one
        H = 256 * rng.randint(4, 16)
        F = rng.choice([H, H // 4, 2 * H, int(3.8 * H) // 256 * 256, int(3.8 * H) // 256 * 256])
        if kind == "swiglu":
            N = F if rng.random() < 0.7 else F - 8 * rng.randint(1, 15)
            return dict(kind="swiglu", type=type, M=min(M, MOST_FLOPS // (4 * N * H)), N=N, K=H)
        N, K = (F, H) if F % per or rng.random() < 0.6 else (H, F)
        N = N if rng.random() < 0.7 else N - rng.randint(1, 100)
        K = K if rng.random() < 0.7 else max(per, K - per * rng.randint(1, 3))
        M = min(M, MOST_FLOPS // (2 * N * K))
        return dict(kind="gemm", type=type, M=M, N=N, K=K, out=rng.choice(["f16", "f32"]), acc=rng.random() < 0.3)
    if kind == "readout":
        return dict(kind="readout", type=type, B=_log_int(rng, 1, 256), k=rng.randint(2, 32), N=rng.choice([32000, 151936]),
                    K=rng.choice([1024, 2048, 2560]))
    head_dim = rng.choice([64, 64, 128])
    kv_heads = rng.choice([2, 4, 8])
    heads = kv_heads * rng.choice([1, 2, 4])
    hidden = 256 * rng.randint(2, 8)
    prefix = rng.choice([0, _log_int(rng, 64, 2048)])
    T = _log_int(rng, 16, 2048) if not prefix else _log_int(rng, 1, 64)
    c = model("", rng.choice(["Q8_0", "Q4_K"]), T, prefix, rng.randint(1, 4), hidden, 256 * rng.randint(4, 16), heads, kv_heads,
              head_dim, 8192, rng.choice([4, 8, 32]))
    del c["name"]
    return c


# ------------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device=DEV, dtype=torch.uint8)


def _scale(g, n, s):
    return (torch.randn(n, generator=g, device=DEV).abs() * s).half().view(torch.uint8).reshape(n, 2)


def random_blocks(g, type, rows, cols):
    """GGUF blocks [blocks, bytes]: uniform codes, fp16 scales |N(0, 1)| times what gives weights of a few 1e-2."""
    if type == "Q8_0":
        n = rows * cols // 32
        q = torch.randint(-127, 128, (n, 32), generator=g, device=DEV, dtype=torch.int8).view(torch.uint8)
        return torch.cat([_scale(g, n, 2e-4), q], 1)
    n = rows * cols // 256
    b = _bytes(g, n, hq.BLOCK_BYTES[TYPES[type]])
    for at, s in {"Q2_K": ((80, 4e-3), (82, 4e-3)), "Q3_K": ((108, 5e-4),), "Q4_K": ((0, 1e-3), (2, 1e-3)),
                  "Q5_K": ((0, 5e-4), (2, 5e-4)), "Q6_K": ((208, 2e-5),)}[type]:
        b[:, at:at + 2] = _scale(g, n, s)
    return b


def quantize(w, type):
    """GGUF blocks of float weights: Q8_0 by absmax / 127, Q4_K by each 32-value group's range."""
    if type == "Q8_0":
        x = w.reshape(-1, 32)
        d = (x.abs().amax(1) / 127).clamp_min(1e-8)
        q = (x / d[:, None]).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([d.half().view(torch.uint8).reshape(-1, 2), q], 1)
    x = w.reshape(-1, 8, 32)
    lo = (-x.amin(2)).clamp_min(0)
    step = (x.amax(2) + lo) / 15
    d, dm = (step.amax(1) / 63).half(), (lo.amax(1) / 63).half()
    s = (step / d.float()[:, None]).round().clamp(0, 63)
    m = (lo / dm.float()[:, None]).round().clamp(0, 63)
    ds = (d.float()[:, None] * s).clamp_min(1e-12)
    q = ((x + (dm.float()[:, None] * m)[:, :, None]) / ds[:, :, None]).round().clamp(0, 15).to(torch.uint8)
    s, m = s.to(torch.uint8), m.to(torch.uint8)
    qs = (q[:, 0::2] | (q[:, 1::2] << 4)).reshape(-1, 128)
    sc = torch.cat([s[:, :4] | ((s[:, 4:] >> 4) << 6), m[:, :4] | ((m[:, 4:] >> 4) << 6), (s[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)], 1)
    return torch.cat([d.view(torch.uint8).reshape(-1, 2), dm.view(torch.uint8).reshape(-1, 2), sc, qs], 1)


def decode(b, type):
    """Float64 values [blocks, block values] of GGUF blocks."""
    def f16(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    def s8(x):
        return x.contiguous().view(torch.int8).double()

    if type == "Q8_0":
        return f16(0) * s8(b[:, 2:])
    if type == "Q6_K":
        ql, qh, sc = b[:, :128], b[:, 128:192], s8(b[:, 192:208])
        parts = []
        for h in (0, 1):
            lo, hi = ql[:, 64 * h:64 * h + 64], qh[:, 32 * h:32 * h + 32]
            for r in range(4):
                n = (lo[:, 32 * (r & 1):32 * (r & 1) + 32] >> (4 * (r >> 1))) & 15
                parts.append((n | (((hi >> (2 * r)) & 3) << 4)).double() - 32)
        return f16(208) * torch.cat(parts, 1) * sc.repeat_interleave(16, 1)
    if type in ("Q4_K", "Q5_K"):
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, 16:144] if type == "Q4_K" else b[:, 48:176]
        q = torch.stack([qs.reshape(-1, 4, 32) & 15, qs.reshape(-1, 4, 32) >> 4], 2).reshape(-1, 8, 32)
        if type == "Q5_K":
            qh = b[:, 16:48]
            q = q + 16 * torch.stack([(qh >> j) & 1 for j in range(8)], 1)
        v = (f16(0) * sc)[:, :, None] * q.double() - (f16(2) * mn)[:, :, None]
        return v.reshape(-1, 256)
    if type == "Q2_K":
        qs = b[:, 16:80].reshape(-1, 2, 32)
        q = torch.stack([(qs >> (2 * j)) & 3 for j in range(4)], 2).reshape(-1, 16, 16).double()
        v = (f16(80) * (b[:, :16] & 15).double())[:, :, None] * q - (f16(82) * (b[:, :16] >> 4).double())[:, :, None]
        return v.reshape(-1, 256)
    hm, qs, s = b[:, :32], b[:, 32:96].reshape(-1, 2, 32), b[:, 96:108]
    q = torch.stack([(qs >> (2 * j)) & 3 for j in range(4)], 2).reshape(-1, 8, 32).double()
    q = q - 4 * torch.stack([1 - ((hm >> j) & 1).double() for j in range(8)], 1)
    lo = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
    hi = torch.cat([(s[:, 8:] >> (2 * j)) & 3 for j in range(4)], 1)
    return (f16(108) * ((lo | (hi << 4)).double() - 32)).repeat_interleave(16, 1) * q.reshape(-1, 256)


def _mat(blocks, type, rows, cols, perm=0):
    return hq.Mat(blocks.cpu().numpy(), TYPES[type], rows, cols, perm)


def _activations(g, M, K):
    return torch.randn(M, K, generator=g, device=DEV).half()


def _inputs(case, seed):
    """The case's blocks and activations on the GPU."""
    g = _gen(seed)
    N, K = case["N"], case["K"]
    if case["kind"] == "swiglu":
        return random_blocks(g, case["type"], N, K), random_blocks(g, case["type"], N, K), _activations(g, case["M"], K)
    b = random_blocks(g, case["type"], N, K)
    if case["kind"] == "readout":
        H = _activations(g, case["B"], K)
        ids = torch.randint(0, N, (case["B"], case["k"]), generator=g, device=DEV, dtype=torch.int64)
        return b, H, ids.to(torch.int32)
    A = _activations(g, case["M"], K)
    dt = torch.float32 if case["out"] == "f32" else torch.float16
    C = torch.randn(case["M"], N, generator=g, device=DEV).to(dt) if case["acc"] else torch.zeros(case["M"], N, device=DEV, dtype=dt)
    return b, A, C


def _model_parts(case, seed):
    """Weights of the model (float, before quantisation), by layer, and the tokens and ids."""
    g = _gen(seed)
    H, I, V, hd = case["hidden"], case["ffn"], case["vocab"], case["head_dim"]
    qw, kvw = case["heads"] * hd, case["kv_heads"] * hd

    def q(rows, cols):
        return quantize(torch.randn(rows * cols, generator=g, device=DEV) * 0.02, case["type"])

    def norm():
        return 1 + 0.1 * torch.randn(H, generator=g, device=DEV)

    m = {"embed": q(V, H), "lm_head": q(V, H), "final_norm": norm(), "layers": []}
    for _ in range(case["layers"]):
        L = {"in_norm": norm(), "post_norm": norm()}
        for n, (r, c) in {"q": (qw, H), "k": (kvw, H), "v": (kvw, H), "o": (H, qw), "gate": (I, H), "up": (I, H), "down": (H, I)}.items():
            L[n] = q(r, c)
        m["layers"].append(L)
    tokens = torch.randint(0, V, (case["prefix"] + case["T"],), generator=g, device=DEV)
    ids = torch.randperm(V, generator=g, device=DEV)[:case["ids"]]
    return m, tokens.cpu().numpy().astype(np.uint32), ids.cpu().numpy().astype(np.uint32)


def prepare(case, seed):
    if case["kind"] == "model":
        hq.device_init(0)
        m, tokens, ids = _model_parts(case, seed)
        cfg = dict(hidden=case["hidden"], n_layers=case["layers"], intermediate=case["ffn"], vocab=case["vocab"],
                   n_heads=case["heads"], n_kv_heads=case["kv_heads"], head_dim=case["head_dim"], rot_dim=case["head_dim"],
                   eps=EPS, rope_theta=THETA)

        def host(d):
            return {k: [host(x) for x in v] if isinstance(v, list) else v.cpu().numpy() for k, v in d.items()}

        view = hq.RefModelView(dict(host(m), cfg=cfg), TYPES[case["type"]])
        be = _Model(view, case["prefix"] + case["T"])
        if case["prefix"]:
            be.forward(tokens[:case["prefix"]])
        be.snapshot()
        return {"kind": "model", "backend": be, "tokens": tokens[case["prefix"]:], "ids": ids}
    hq.device_init(0)
    lib = hq.load()
    parts = _inputs(case, seed)
    N, K, t = case["N"], case["K"], case["type"]
    if case["kind"] == "swiglu":
        W = hq.PairMat(parts[0].cpu().numpy(), parts[1].cpu().numpy(), TYPES[t], N, K)
        out = torch.empty(case["M"], N, device=DEV, dtype=torch.float16)
        return {"kind": "swiglu", "lib": lib, "W": W, "A": parts[2], "M": case["M"], "out": out}
    W = _mat(parts[0], t, N, K)
    if case["kind"] == "readout":
        out = torch.empty(case["B"], case["k"], device=DEV)
        return {"kind": "readout", "lib": lib, "W": W, "H": parts[1], "ids": parts[2], "out": out}
    return {"kind": "gemm", "W": W, "A": parts[1], "C": parts[2], "M": case["M"], "f32": case["out"] == "f32", "acc": case["acc"]}


class _Model(hq.HipBackend):
    """The backend, given back with the state that holds it."""

    def __del__(self):
        try:
            self.destroy()
        except Exception:
            pass


def run(state):
    if state["kind"] == "gemm":
        hq.gemm(state["W"], state["A"].data_ptr(), state["M"], state["C"].data_ptr(), state["f32"], state["acc"])
        return state["C"]
    if state["kind"] == "swiglu":
        if state["lib"].hq_gemm_swiglu(state["W"].h, state["A"].data_ptr(), state["M"], state["out"].data_ptr(), None):
            raise hq.HQError(hq.last_error())
        return state["out"]
    if state["kind"] == "readout":
        B, k = state["ids"].shape
        if state["lib"].hq_gather_dot_dev(state["W"].h, state["H"].data_ptr(), state["ids"].data_ptr(), B, k, state["out"].data_ptr(), None):
            raise hq.HQError(hq.last_error())
        return state["out"]
    be = state["backend"]
    be.restore()
    logits = be.forward(state["tokens"], state["ids"])
    return {"logits": logits, "hidden": be.last_hidden()}


def work(case):
    bw = hq.BLOCK_BYTES[TYPES[case["type"]]] / hq.BLOCK_VALUES[TYPES[case["type"]]]
    if case["kind"] == "gemm":
        M, N, K, c = case["M"], case["N"], case["K"], 4 if case["out"] == "f32" else 2
        return {"bytes": N * K * bw + 2 * M * K + M * N * c * (2 if case["acc"] else 1), "flops": 2 * M * N * K}
    if case["kind"] == "swiglu":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * N * K * bw + 2 * M * K + 2 * M * N, "flops": 4 * M * N * K}
    if case["kind"] == "readout":
        n = case["B"] * case["k"]
        return {"bytes": n * case["K"] * bw + case["B"] * case["K"] * 2 + n * 8, "flops": 2 * n * case["K"]}
    T, H, I, P, L = case["T"], case["hidden"], case["ffn"], case["prefix"], case["layers"]
    qw, kvw = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    weights = L * (H * (2 * qw + 2 * kvw) + 3 * H * I)
    pairs = T * P + T * (T + 1) // 2
    return {"bytes": (weights + (T + case["ids"]) * H) * bw + L * 2 * (P + T) * kvw * 4 + 4 * (T + H + 2 * case["ids"]),
            "flops": 2 * T * weights + L * pairs * 4 * qw + 2 * case["ids"] * H}


def tolerance(case):
    # against exact(): 2.1e-4 for an output rounded once to fp16, 2.9e-4 to 4.6e-4 with the weights also rounded to fp16
    # (Q8_0; Q6_K, Q3_K and Q2_K for larger M), 1e-7 to 1e-6 for fp32 outputs of exactly decoded weights; models 1.2e-3
    if case["kind"] == "model":
        return {"rel": 4e-3, "max": 4e-2}  # fp16 GEMM operands through every layer
    if case["kind"] == "readout":
        return {"rel": 2e-6, "max": 2e-5}
    if case["kind"] == "gemm" and case["out"] == "f32" and case["type"] in ("Q4_K", "Q5_K"):
        return {"rel": 5e-6, "max": 2e-4}
    return {"rel": 1.2e-3, "max": 1.5e-2}


# ------------------------------------------------------------------------------------ float64
def _weights(blocks, type, rows, cols):
    step = max(1, (1 << 24) // cols)
    b = blocks.reshape(rows, -1, blocks.shape[1])
    return torch.cat([decode(b[r:r + step].reshape(-1, blocks.shape[1]), type).reshape(-1, cols) for r in range(0, rows, step)])


def _exact_model(case, seed):
    m, tokens, ids = _model_parts(case, seed)
    H, hd, nh, nkv = case["hidden"], case["head_dim"], case["heads"], case["kv_heads"]
    n, t = len(tokens), case["type"]

    def norm(x, w):
        return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()

    def mat(b, cols):
        return _weights(b, t, b.numel() // (cols // hq.BLOCK_VALUES[TYPES[t]] * b.shape[1]), cols)

    def rotated(w, heads):
        # the file holds each head's rows as pairs (i, i + hd / 2) side by side
        return w.reshape(heads, hd // 2, 2, H).transpose(1, 2).reshape(heads * hd, H)

    inv = torch.from_numpy(hq.rope_inv_freq(THETA, hd)).to(DEV).double()
    a = torch.arange(n, device=DEV).double()[:, None] * inv
    cs, sn = a.cos()[:, None], a.sin()[:, None]

    def rope(x):
        u, v = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat([u * cs - v * sn, u * sn + v * cs], -1)

    at = torch.from_numpy(tokens.astype(np.int64)).to(DEV)
    rows = m["embed"].reshape(case["vocab"], -1, m["embed"].shape[1])[at]
    x = decode(rows.reshape(-1, rows.shape[2]), t).reshape(n, H)
    mask = torch.full((n, n), -math.inf, device=DEV, dtype=torch.float64).triu(1)
    for L in m["layers"]:
        h = norm(x, L["in_norm"])
        q = rope((h @ rotated(mat(L["q"], H), nh).T).reshape(n, nh, hd))
        k = rope((h @ rotated(mat(L["k"], H), nkv).T).reshape(n, nkv, hd))
        v = (h @ mat(L["v"], H).T).reshape(n, nkv, hd)
        o = torch.empty(n, nh, hd, device=DEV, dtype=torch.float64)
        for j in range(nh):
            g = j // (nh // nkv)
            p = torch.softmax(q[:, j].contiguous() @ k[:, g].T.contiguous() / math.sqrt(hd) + mask, -1)
            o[:, j] = p @ v[:, g].contiguous()
        x = x + o.reshape(n, nh * hd) @ mat(L["o"], nh * hd).T
        h = norm(x, L["post_norm"])
        x = x + (torch.nn.functional.silu(h @ mat(L["gate"], H).T) * (h @ mat(L["up"], H).T)) @ mat(L["down"], case["ffn"]).T
    hidden = norm(x[-1], m["final_norm"])
    head = m["lm_head"].reshape(case["vocab"], -1, m["lm_head"].shape[1])[torch.from_numpy(ids.astype(np.int64)).to(DEV)]
    return {"logits": decode(head.reshape(-1, head.shape[2]), t).reshape(len(ids), H) @ hidden, "hidden": hidden}


def exact(case, seed):
    if case["kind"] == "model":
        return _exact_model(case, seed)
    parts = _inputs(case, seed)
    N, K, t = case["N"], case["K"], case["type"]
    if case["kind"] == "swiglu":
        g, u = (parts[2].double() @ _weights(b, t, N, K).T for b in parts[:2])
        return torch.nn.functional.silu(g) * u
    if case["kind"] == "readout":
        rows = parts[0].reshape(N, -1, parts[0].shape[1])[parts[2].long().reshape(-1)]
        w = decode(rows.reshape(-1, rows.shape[2]), t).reshape(case["B"], case["k"], K)
        return (w * parts[1].double()[:, None]).sum(-1)
    r = parts[1].double() @ _weights(parts[0], t, N, K).T
    return r + parts[2].double() if case["acc"] else r
