"""Device memory of a backend: the activation buffers that its layers use and no others, and passes of 1024 tokens where
2048 tokens' activations would not leave half of the free memory."""
import ctypes as C

import pytest

import hq
import synth


@pytest.mark.parametrize("max_seq,per_token,free,want", [(4096, 1 << 17, 1 << 40, 2048), (4096, 1 << 17, 1 << 29, 2048), (4096, 1 << 17, (1 << 29) - 1, 1024),
                                                         (1500, 1 << 17, 1 << 40, 1500), (1500, 1 << 17, 1 << 28, 1024), (7, 1 << 17, 1 << 28, 7)])
def test_pass_tokens(max_seq, per_token, free, want):
    f = hq.load().hq_internal_pass_tokens
    f.argtypes = [C.c_size_t] * 3
    assert f(max_seq, per_token, free) == want


def free_bytes():
    a, b = C.c_size_t(), C.c_size_t()
    assert C.CDLL("libamdhip64.so.7").hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


@pytest.mark.gpu
@pytest.mark.parametrize("apart", [False, True])
def test_backend_allocates_what_it_uses(hqlib, apart):
    """One layer of hidden 256, 64 heads of 32 over 32 and ffn 8192: 2048 tokens' q, k, v rows are 33.5 MB in one buffer and
    gate and up products 134 MB, which a layer with one gate/up pair does not need. Slack: 2 MiB rounding of each of 30
    allocations."""
    H, I, nh, nkv, hd = 256, 8192, 64, 32, 32
    cfg = dict(synth.TINY_LLAMA, n_layers=1, hidden=H, intermediate=I, vocab=512, n_heads=nh, n_kv_heads=nkv, head_dim=hd, rot_dim=hd)
    model = synth.tiny_llama(3, cfg)
    qw, kvw = nh * hd, nkv * hd
    if apart:  # a q of another type than k and v, an up of another type than gate
        model["layers"][0].update(q=synth.q4_k_blocks(synth.Rng(1), qw, H), up=synth.q6_k_blocks(synth.Rng(2), I, H))
        model["types"] = {"q": synth.Q4_K, "up": synth.Q6_K}
    tokens, ids = synth.tiny_llama_prompt(2, T=8, vocab=512)
    view = hqlib.RefModelView(model)
    be = hqlib.HipBackend(view, 2048)  # the library's own first allocations (upload staging) lie behind
    be.destroy()
    before = free_bytes()
    be = hqlib.HipBackend(view, 2048)
    took = before - free_bytes()
    be.forward(tokens, ids)
    be.destroy()
    weights = (2 * 512 * H + (2 * qw + 2 * kvw) * H + 3 * I * H) * 1.07
    kv = 2 * 2048 * kvw * 4
    acts = 2048 * (4 * H + 4 * (qw if apart else qw + 2 * kvw) + 4 * qw + 2 * H + 2 * qw + 2 * I + (8 * kvw + 8 * I if apart else 0))
    print(f"[gpu] backend memory apart={apart}: {took / 1e6:.0f} MB, needs {(weights + kv + acts) / 1e6:.0f}", flush=True)
    assert took <= weights + kv + acts + 30 * (2 << 20)
