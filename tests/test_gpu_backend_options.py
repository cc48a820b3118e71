"""The backend's attention options against a float64 forward of the same blocks: output gate (q rows [q_h | gate_h]),
q/k RMSNorm and a norm offset, with q, k and v of one type (one resident matrix, rows [q | k | v]) and of several, for a
prompt, for the same tokens one at a time at its end (positions split over workgroups), for row counts around 16 and 32,
and for rows enough that a block takes 32.

The tolerance is the logits' bar of every forward test: GEMM operands are rounded to fp16 (2^-11 each, logits of size
~1), the rest is fp32. A gate or a norm read at a wrong offset is a different vector of order 1.
"""
import numpy as np
import pytest

import synth
from conftest import max_abs

pytestmark = pytest.mark.gpu
Q8, MIXED = {}, {"q": synth.Q8_0, "k": synth.Q4_K, "v": synth.Q6_K}
Q4, Q5 = ({n: t for n in ("q", "k", "v")} for t in (synth.Q4_K, synth.Q5_K))


def blocks(gtype, rng, rows, cols):
    """Weights of deviation ~0.02, mean 0."""
    if gtype == synth.Q8_0:
        return synth.quantize_q8_0((rng.normal(rows * cols) * 0.02).astype(np.float32).reshape(rows, cols))
    if gtype == synth.Q6_K:
        return synth.q6_k_blocks(rng, rows, cols)
    b = synth.q4_k_blocks(rng, rows, cols, scale=1e-4) if gtype == synth.Q4_K else synth.q5_k_blocks(rng, rows, cols, scale=5e-5)
    v = b.reshape(-1, synth.BLOCK_BYTES[gtype])
    d = v[:, 0:2].copy().view(np.float16).astype(np.float64)
    v[:, 2:4] = synth.f16_bits((7.5 if gtype == synth.Q4_K else 15.5) * d).view(np.uint8).reshape(-1, 2)
    return b


def make(seed, types, gate, qk_norm, offset, nh, nkv, hd, rot):
    cfg = dict(synth.TINY_LLAMA, n_layers=2, hidden=256, intermediate=256, vocab=512, n_heads=nh, n_kv_heads=nkv, head_dim=hd, rot_dim=rot,
               attn_gate=gate, qk_norm=qk_norm, norm_offset=offset)
    model = synth.tiny_llama(seed, cfg)
    rng = synth.Rng(seed + 1)
    for L in model["layers"]:
        rows = {"q": nh * hd * (2 if gate else 1), "k": nkv * hd, "v": nkv * hd}
        for n in rows:
            L[n] = blocks(types.get(n, synth.Q8_0), rng, rows[n], 256)
        L["q_norm"], L["k_norm"] = ((1 - offset + 0.2 * rng.normal(hd)).astype(np.float32) for _ in (0, 1))
        for n in ("in_norm", "post_norm"):
            L[n] = (L[n] - np.float32(offset)).astype(np.float32)
    model["final_norm"] = (model["final_norm"] - np.float32(offset)).astype(np.float32)
    model["types"] = types
    return model


def forward64(oracle, hqlib, model, tokens, ids):
    c = model["cfg"]
    H, hd, nh, nkv, rot, off = c["hidden"], c["head_dim"], c["n_heads"], c["n_kv_heads"], c["rot_dim"], float(np.float32(c["norm_offset"]))
    n, I = len(tokens), c["intermediate"]

    def w(b, name, rows, cols, perm=0):
        return oracle.dequantize(b, model["types"].get(name, synth.Q8_0), rows, cols, perm).astype(np.float64)

    def norm(x, g):
        return x / np.sqrt((x * x).mean(-1, keepdims=True) + c["eps"]) * (off + g.astype(np.float64))

    a = np.arange(n)[:, None] * hqlib.rope_inv_freq(c["rope_theta"], rot).astype(np.float64)
    cs, sn = np.cos(a)[:, None], np.sin(a)[:, None]

    def rope(x):
        u, v = x[..., :rot // 2], x[..., rot // 2:rot]
        return np.concatenate([u * cs - v * sn, u * sn + v * cs, x[..., rot:]], -1)

    x = oracle.dequantize(np.ascontiguousarray(model["embed"][tokens]), synth.Q8_0, n, H).astype(np.float64)
    mask = np.triu(np.full((n, n), -np.inf), 1)
    for L in model["layers"]:
        h = norm(x, L["in_norm"])
        qr = w(L["q"], "q", nh * hd * (2 if c["attn_gate"] else 1), H, 0 if c["attn_gate"] else nh)
        q = (h @ qr.T).reshape(n, nh, -1)
        gate = q[..., hd:]
        q = q[..., :hd]
        k, v = (h @ w(L["k"], "k", nkv * hd, H, nkv).T).reshape(n, nkv, hd), (h @ w(L["v"], "v", nkv * hd, H).T).reshape(n, nkv, hd)
        if c["qk_norm"]:
            q, k = norm(q, L["q_norm"]), norm(k, L["k_norm"])
        q, k = rope(q), rope(k)
        o = np.empty((n, nh, hd))
        for j in range(nh):
            s = q[:, j] @ k[:, j // (nh // nkv)].T / np.sqrt(hd) + mask
            p = np.exp(s - s.max(-1, keepdims=True))
            o[:, j] = p / p.sum(-1, keepdims=True) @ v[:, j // (nh // nkv)]
        if c["attn_gate"]:
            o = o / (1 + np.exp(-gate))
        x = x + o.reshape(n, nh * hd) @ w(L["o"], "o", H, nh * hd).T
        h = norm(x, L["post_norm"])
        g, u = h @ w(L["gate"], "gate", I, H).T, h @ w(L["up"], "up", I, H).T
        x = x + (g / (1 + np.exp(-g)) * u) @ w(L["down"], "down", H, I).T
    head = oracle.dequantize(np.ascontiguousarray(model["lm_head"][ids]), synth.Q8_0, len(ids), H).astype(np.float64)
    return head @ norm(x[-1], model["final_norm"])


CASES = [  # types, gate, q/k norm, offset, heads, kv heads, head size, rotated dims, tokens before the last pass, its tokens
    (Q8, True, True, 1.0, 4, 2, 64, 32, 0, 33), (Q8, True, False, 0.0, 8, 2, 64, 64, 300, 1), (Q8, False, True, 0.0, 4, 4, 96, 96, 40, 17),
    (Q8, False, False, 1.0, 4, 2, 64, 64, 0, 1), (Q4, True, True, 1.0, 8, 2, 64, 16, 270, 1), (Q4, False, True, 1.0, 4, 1, 128, 64, 15, 16),
    (Q5, True, False, 1.0, 2, 1, 256, 64, 0, 70), (Q4, False, False, 0.0, 4, 2, 64, 64, 129, 1), (Q5, False, False, 0.0, 4, 2, 64, 64, 100, 65),
    (MIXED, True, True, 1.0, 4, 2, 64, 32, 200, 1), (MIXED, True, True, 0.5, 4, 2, 64, 64, 0, 31), (MIXED, False, True, 1.0, 4, 2, 128, 32, 66, 3),
    (Q8, True, True, 1.0, 32, 8, 64, 64, 0, 260), (MIXED, True, False, 0.0, 32, 8, 64, 64, 7, 260)]


@pytest.mark.parametrize("types,gate,qk_norm,offset,nh,nkv,hd,rot,prefix,T", CASES)
def test_attention_options(hqlib, oracle, types, gate, qk_norm, offset, nh, nkv, hd, rot, prefix, T):
    model = make(nh + hd + T + prefix, types, gate, qk_norm, offset, nh, nkv, hd, rot)
    tokens, ids = synth.tiny_llama_prompt(7, T=prefix + T, vocab=512, n_ids=16)
    print(f"[gpu] options gate={gate} qk_norm={qk_norm} offset={offset} {nh}/{nkv} x {hd}, {prefix} + {T}", flush=True)
    be = hqlib.HipBackend(hqlib.RefModelView(model), prefix + T)
    if prefix:
        be.forward(tokens[:prefix])
    got = be.forward(tokens[prefix:], ids)
    be.destroy()
    ref = forward64(oracle, hqlib, model, tokens, ids)
    print(f"[gpu]   max_abs {max_abs(got, ref):.2e} of {np.abs(ref).max():.2f}", flush=True)
    assert np.abs(ref).max() > 0.1 and max_abs(got, ref) <= 1e-2
