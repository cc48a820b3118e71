"""The backend's attention (hq_attention.hip) at the edges of its tiles: head sizes around the 64-wide
padding, grouped heads, row counts around 16 and 32, one and several position ranges per row block,
against the oracle's CPU forward of the same one-layer model.

The tolerance is the logits' bar of every forward test: GEMM operands are rounded to fp16 (2^-11 each,
logits of size ~1), attention itself is fp32 on both sides.
"""
import numpy as np
import pytest

import synth
from conftest import max_abs

pytestmark = pytest.mark.gpu

CASES = [  # heads, kv heads, head_dim, prefix, tokens
    (8, 8, 64, 0, 1), (8, 8, 64, 0, 31), (8, 8, 64, 0, 33), (8, 2, 64, 0, 129), (4, 1, 64, 500, 1), (8, 8, 64, 300, 17),
    (8, 4, 40, 0, 70), (4, 4, 96, 33, 20), (8, 2, 128, 0, 130), (16, 4, 128, 257, 3), (2, 1, 160, 0, 67), (2, 2, 192, 40, 9),
    (2, 1, 256, 0, 50), (4, 2, 256, 190, 1), (40, 8, 64, 0, 270), (48, 16, 128, 0, 250),
]


@pytest.mark.parametrize("nh,nkv,hd,prefix,T", CASES)
def test_attention_edges(hqlib, oracle, nh, nkv, hd, prefix, T):
    cfg = dict(synth.TINY_LLAMA, n_layers=1, hidden=256, intermediate=256, vocab=512, n_heads=nh, n_kv_heads=nkv, head_dim=hd,
               rot_dim=hd)
    model = synth.tiny_llama(nh + hd + T, cfg)
    tokens, ids = synth.tiny_llama_prompt(7, T=prefix + T, vocab=512, n_ids=16)
    be = hqlib.HipBackend(hqlib.RefModelView(model), prefix + T)
    if prefix:
        be.forward(tokens[:prefix])
    got = be.forward(tokens[prefix:], ids)
    again = None
    if prefix:  # the same rows as part of one longer pass
        be.reset()
        again = be.forward(tokens, ids)
    be.destroy()
    ref = oracle.llama_forward(model, tokens, ids)
    print(f"[gpu] attention {nh}/{nkv} x {hd}, {prefix} + {T}: max_abs {max_abs(got, ref):.2e}", flush=True)
    assert max_abs(got, ref) <= 1e-2
    assert again is None or max_abs(again, got) <= 1e-3


def test_many_ids_and_long_prompts(hqlib, oracle):
    """Token and id counts on both sides of what a launch carries as arguments (64): the same logits for the
    same ids, the oracle's within the bar."""
    cfg = dict(synth.TINY_LLAMA, n_layers=1, hidden=256, intermediate=256, vocab=512, n_heads=4, n_kv_heads=2, head_dim=64)
    model = synth.tiny_llama(9, cfg)
    tokens, ids = synth.tiny_llama_prompt(8, T=129, vocab=512, n_ids=65)
    be = hqlib.HipBackend(hqlib.RefModelView(model), 129)
    many = be.forward(tokens, ids)
    be.reset()
    be.forward(tokens[:65])
    few = be.forward(tokens[65:], ids[:64])
    be.destroy()
    ref = oracle.llama_forward(model, tokens, ids)
    assert max_abs(many, ref) <= 1e-2 and max_abs(few, many[:64]) <= 1e-3


@pytest.mark.parametrize("nh,nkv,rot,T", [(3, 1, 64, 2049), (5, 1, 32, 2150), (2, 2, 64, 1537), (3, 3, 16, 3)])
def test_passes_of_a_long_prompt(hqlib, oracle, nh, nkv, rot, T):
    """Prompts around one pass of the layer loop (2048 tokens; 2049 leaves a pass of one token), head counts
    that do not fill the rotary kernel's workgroups, and fewer rotated dims than the head has."""
    cfg = dict(synth.TINY_LLAMA, n_layers=1, hidden=256, intermediate=256, vocab=512, n_heads=nh, n_kv_heads=nkv, head_dim=64,
               rot_dim=rot)
    model = synth.tiny_llama(nh + T, cfg)
    tokens, ids = synth.tiny_llama_prompt(11, T=T, vocab=512, n_ids=16)
    be = hqlib.HipBackend(hqlib.RefModelView(model), T)
    got = be.forward(tokens, ids)
    be.reset()
    be.forward(tokens[: T // 2])
    split = be.forward(tokens[T // 2:], ids)
    be.destroy()
    ref = oracle.llama_forward(model, tokens, ids)
    assert max_abs(got, ref) <= 1e-2 and max_abs(split, got) <= 1e-3


@pytest.mark.parametrize("gtype,hidden,inter", [(synth.Q8_0, 256, 64), (synth.Q8_0, 1024, 288), (synth.Q8_0, 1056, 288), (synth.Q8_0, 2048, 256),
                                                (synth.Q8_0, 2080, 256), (synth.Q8_0, 512, 8224)])
def test_one_token_norm(hqlib, oracle, gtype, hidden, inter):
    """One token's RMSNorm inside the q/k/v and gate/up GEMVs, on both sides of their rule (hidden up to 2048, waves
    x hidden x 8 up to 16 MB) and of a lane's one or two chunks of 16 values, some lanes without one: the logits
    of a one-token pass against the oracle's and against the same tokens in one pass, whose norm is the kernel of
    its own."""
    cfg = dict(synth.TINY_LLAMA, n_layers=2, hidden=hidden, intermediate=inter, vocab=512, n_heads=2, n_kv_heads=1, head_dim=32, rot_dim=32)
    model = synth.tiny_llama(hidden, cfg)
    tokens, ids = synth.tiny_llama_prompt(12, T=4, vocab=512, n_ids=16)
    be = hqlib.HipBackend(hqlib.RefModelView(model), 4)
    for t in range(3):
        be.forward(tokens[t:t + 1])
    one = be.forward(tokens[3:], ids)
    be.reset()
    whole = be.forward(tokens, ids)
    be.destroy()
    ref = oracle.llama_forward(model, tokens, ids)
    print(f"[gpu] one-token norm H={hidden} I={inter}: max_abs {max_abs(one, ref):.2e}", flush=True)
    # one against whole: fp16 roundings (2^-11 / sqrt(3) in the mean) of four GEMM inputs in each of two layers and of the
    # whole pass's Q8_0 weights (the GEMVs' are exact), 24 in all, on logits of deviation 0.02 sqrt(2080) = 0.91:
    # sqrt(24) 2.8e-4 0.91 = 1.3e-3, three of them
    assert max_abs(one, ref) <= 1e-2 and max_abs(one, whole) <= 3.8e-3
