"""The narrow Stream-K GEMM kernels at the edges of their tiles (16 / 32 / 64 / 128 rows by 128 columns) and of their
units of 256 K: one unit, a Q8_0 K that ends inside one, tiles cut between workgroups and tiles whole, every output
mode, against the oracle.

Bars: those of the parity tests (rel-L2 1e-3, max-abs 1e-2), and for the types whose weights these kernels never round
(all but Q8_0) fp32 outputs within 2^-13 |W| @ |a| of the float64 product, the bar of every such kernel.
"""
import numpy as np
import pytest

import synth
from conftest import max_abs, rel_l2
from test_gemm_routes import stream_k

pytestmark = pytest.mark.gpu
KQ = [synth.Q2_K, synth.Q3_K, synth.Q5_K, synth.Q6_K]
CASES = [(synth.Q8_0, *s) for s in [(2, 16, 96), (16, 130, 288), (17, 300, 32), (64, 1000, 160), (65, 520, 224),
                                    (200, 2000, 256), (1100, 520, 800), (2049, 520, 672), (700, 1500, 1056)]] + \
        [(synth.Q4_K, *s) for s in [(2, 16, 256), (17, 65, 256), (33, 100, 256), (64, 129, 256)]] + \
        [(t, *s) for t in KQ for s in [(2, 16, 256), (17, 65, 256), (33, 100, 256), (70, 96, 256), (1085, 576, 2304)]]


@pytest.mark.parametrize("gtype,M,N,K", CASES)
def test_stream_k(hqlib, oracle, gtype, M, N, K):
    assert stream_k(gtype, M, N, K)
    blocks = synth.random_blocks(gtype, synth.Rng(71 + N + gtype), N, K)
    a = synth.activations_f16(synth.Rng(72 + M), M, K)
    print(f"[gpu] Stream-K {synth.TYPE_NAMES[gtype]} M={M} N={N} K={K}", flush=True)
    W = hqlib.Mat(blocks, gtype, N, K)
    got = hqlib.gemm_np(W, a)
    c0 = synth.activations_f16(synth.Rng(73), M, N)
    half = hqlib.gemm_np(W, a, c_f32=False, c_init=c0).view(np.float16).astype(np.float64)
    again = hqlib.gemm_np(W, a)
    W.free()
    x, w = oracle.f16_to_f32(a).astype(np.float64), oracle.dequantize(blocks, gtype, N, K).astype(np.float64)
    ref, c = x @ w.T, c0.view(np.float16).astype(np.float64)
    assert rel_l2(got, ref) <= 1e-3 and max_abs(got, ref) <= 1e-2
    assert np.all(np.abs(half - (ref + c)) <= 1e-2 + 2.0 ** -11 * np.abs(ref + c))
    assert np.array_equal(got, again)
    if gtype != synth.Q8_0:
        assert np.all(np.abs(got - ref) <= 2.0 ** -13 * (np.abs(x) @ np.abs(w.T)))
