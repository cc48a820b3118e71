"""`c_is_f32 != 0` asks for fp32 output, whatever the value: 2 and -1 give what 1 gives, bit for bit, through
hq_gemm and hq_gemm_noalloc on every GEMV and on GEMM kernels of each family. (Inside the library 2 is the SwiGLU
epilogue of a gate/up pair matrix, which an ordinary matrix must not reach; the one-wave GEMV, K = 512 and N >= 8192,
would divide by a wave count of 0 there.)
"""
import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu

CASES = [(synth.Q4_K, 1, 8192, 512), (synth.Q4_K, 1, 9728, 2560), (synth.Q4_K, 1, 9728, 256), (synth.Q4_K, 1, 100, 512),
         (synth.Q8_0, 1, 4096, 512), (synth.Q6_K, 1, 8192, 512), (synth.Q5_K, 1, 8192, 256), (synth.Q3_K, 1, 320, 512),
         (synth.Q2_K, 1, 8192, 512), (synth.Q8_0, 2, 512, 256), (synth.Q4_K, 16, 320, 768), (synth.Q6_K, 17, 320, 512),
         (synth.Q4_K, 64, 8192, 512), (synth.Q8_0, 64, 8192, 512), (synth.Q4_K, 128, 9728, 2048), (synth.Q8_0, 128, 9728, 1024),
         (synth.Q4_K, 512, 9728, 256), (synth.Q8_0, 512, 9728, 256), (synth.Q5_K, 300, 9728, 256), (synth.Q2_K, 300, 9728, 256)]


@pytest.mark.parametrize("gtype,M,N,K", CASES)
def test_any_nonzero_means_fp32(hqlib, gtype, M, N, K):
    W = hqlib.Mat(synth.random_blocks(gtype, synth.Rng(61 + N), N, K), gtype, N, K)
    A = hqlib.DevBuf.from_array(synth.activations_f16(synth.Rng(62 + M), M, K))
    print(f"[gpu] output modes {synth.TYPE_NAMES[gtype]} M={M} N={N} K={K}", flush=True)
    out = {}
    for mode in (1, 2, -1):
        for call in (hqlib.gemm, hqlib.gemm_noalloc):
            C = hqlib.DevBuf.from_array(np.full((M, N), 7, np.float32))
            call(W, A, M, C, c_f32=mode)
            out[mode, call.__name__] = C.download((M, N), np.float32)
            C.free()
    A.free()
    W.free()
    want = out[1, "gemm"]
    assert np.all(np.isfinite(want)) and np.any(want != 7)
    for k, got in out.items():
        assert np.array_equal(got, want), k
