"""The small-tile GEMM kernels (hq_gemm_sm.hip) at the edges of their tiles and of their K shares: 1 .. 3
super-blocks, a Q8_0 K that ends inside one, rows around 16 / 32 / 64 and several hundred to thousand, columns
around 64, one column tile and more than eight, a K split over workgroups, every output mode, against the oracle.
Each case states whether these kernels run it (SMALL names them; the workspace tells them from the Stream-K
kernels of the same names); the others are their neighbours across the dispatch rule, one super-block mostly.

Bars: those of the parity tests (rel-L2 1e-3, max-abs 1e-2), and where these kernels or Stream-K run the types
whose weights they never round (all but Q8_0) fp32 outputs within 2^-18 |W| @ |a| of the float64 product: products are exact
in fp32, so what is left are fp32 sums of at most 256 terms per super-block in 32-term steps, the
super-blocks' and parts' sums and one product with d each, under 32 roundings of 2^-24 per path.
"""
import numpy as np
import pytest

import synth
from conftest import max_abs, rel_l2
from test_gemm_routes import stream_k

pytestmark = pytest.mark.gpu
TYPES = [synth.Q8_0, synth.Q2_K, synth.Q3_K, synth.Q4_K, synth.Q5_K, synth.Q6_K]
SMALL = ("k_gemm_q8_0<", "k_gemm_q4_k<", "k_gemm_q6_k<", "k_gemm_kq<")
SHAPES = [(2, 16, 256), (16, 63, 512), (17, 65, 768), (32, 520, 256), (33, 100, 512), (64, 129, 2560), (65, 640, 512),
          (130, 250, 768), (200, 64, 4096), (48, 1000, 256), (70, 96, 256), (12, 2560, 2560),
          (65, 640, 256), (15, 63, 2560), (301, 520, 1280), (700, 136, 768), (1024, 512, 512), (2048, 64, 4096)]


def small(gtype, M, N, K):
    """Whether a case is meant to be theirs."""
    if K <= 256:
        return gtype not in (synth.Q8_0, synth.Q4_K) and M > 64 and N > 96
    return gtype != synth.Q8_0 or M > 32 or K > 2048


def f64(oracle, blocks, t, N, K, a):
    x, w = oracle.f16_to_f32(a).astype(np.float64), oracle.dequantize(blocks, t, N, K).astype(np.float64)
    return x @ w.T, np.abs(x) @ np.abs(w.T)


@pytest.mark.parametrize("gtype", TYPES)
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_small_tiles(hqlib, oracle, gtype, M, N, K):
    if gtype == synth.Q8_0 and K > 256:
        K -= 96  # ends inside the last stage
    blocks = synth.random_blocks(gtype, synth.Rng(31 + N + gtype), N, K)
    a = synth.activations_f16(synth.Rng(32 + M), M, K)
    name = hqlib.gemm_kernel(gtype, M, N, K)
    print(f"[gpu] small tiles {synth.TYPE_NAMES[gtype]} M={M} N={N} K={K} {name}", flush=True)
    assert (name.startswith(SMALL) and not stream_k(gtype, M, N, K)) == small(gtype, M, N, K), name
    W = hqlib.Mat(blocks, gtype, N, K)
    got = hqlib.gemm_np(W, a)
    c0 = synth.activations_f16(synth.Rng(33), M, N)
    acc = hqlib.gemm_np(W, a, c_f32=True, c_init=c0.view(np.float16).astype(np.float32))
    half = hqlib.gemm_np(W, a, c_f32=False, c_init=c0).view(np.float16).astype(np.float64)
    again = hqlib.gemm_np(W, a)
    W.free()
    ref, bound = f64(oracle, blocks, gtype, N, K, a)
    c = c0.view(np.float16).astype(np.float64)
    assert rel_l2(got, ref) <= 1e-3 and max_abs(got, ref) <= 1e-2 and max_abs(acc, ref + c) <= 1e-2
    assert np.all(np.abs(half - (ref + c)) <= 1e-2 + 2.0 ** -11 * np.abs(ref + c))
    assert np.array_equal(got, again)
    if gtype != synth.Q8_0 and name.startswith(SMALL):
        assert np.all(np.abs(got - ref) <= 2.0 ** -18 * bound)


@pytest.mark.parametrize("gtype", TYPES)
@pytest.mark.parametrize("M,I,K", [(1, 24, 512), (1, 200, 256), (1, 4104, 1024), (2, 24, 512), (16, 200, 256), (33, 1000, 768), (64, 72, 2560)])
def test_small_tiles_swiglu(hqlib, oracle, gtype, M, I, K):
    g, u = (synth.random_blocks(gtype, synth.Rng(41 + I + i), I, K) for i in (0, 1))
    a = synth.activations_f16(synth.Rng(42 + M), M, K)
    P = hqlib.PairMat(g, u, gtype, I, K)
    print(f"[gpu] small tiles SwiGLU {synth.TYPE_NAMES[gtype]} M={M} I={I} K={K}", flush=True)
    got = hqlib.gemm_swiglu_np(P, a).view(np.float16).astype(np.float64)
    P.free()
    G, U = (f64(oracle, b, gtype, I, K, a)[0] for b in (g, u))
    ref = G / (1 + np.exp(-G)) * U
    assert rel_l2(got, ref) <= 1e-3
