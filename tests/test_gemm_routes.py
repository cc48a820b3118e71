"""Which kernel an hq_gemm call runs, where the choice between small tiles and the kernels beside them was measured both
ways (host only: names and workspace of the launch plan on 256 CUs). Each case lost when the small tiles took it, by the
times beside it in us; the last ones won. The narrow Stream-K kernels and the small-tile ones share names, so the
workspace tells them apart: Stream-K holds two fp32 partial tiles of 16 mb x 128 per workgroup.
"""
import pytest

import hq
import synth
from synth import Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, Q8_0


def stream_k(gtype, M, N, K):
    """Whether the plan is a narrow Stream-K one."""
    mb = 1 if M <= 16 else 2 if M <= 32 else 4 if M <= 64 or gtype not in (Q8_0, Q4_K) else 8
    mb = max(mb, 2) if gtype == Q4_K else mb
    units = -(-M // (16 * mb)) * -(-N // 128) * -(-K // 256)
    G = min(units, 256)
    G -= G % 8 if G >= 8 else 0
    return hq.gemm_workspace_bytes(gtype, M, N, K)[0] == 2 * G * 16 * mb * 128 * 4


STREAM_K = [(Q8_0, 4096, 4096, 2592, 156, 256), (Q8_0, 8192, 9728, 2592, 826, 1150), (Q8_0, 1024, 4096, 9760, 135, 184),
            (Q8_0, 2048, 4096, 96, 18, 28), (Q8_0, 16, 4096, 96, 3.9, 6.1), (Q8_0, 16, 1024, 1024, 6.5, 7.2), (Q8_0, 5, 76, 512, 5.2, 6.4),
            (Q6_K, 1263, 576, 1536, 19.6, 23.9), (Q6_K, 16, 996, 256, 5.1, 6.8), (Q5_K, 1131, 564, 2560, 25.0, 33.9),
            (Q3_K, 1085, 576, 2304, 17.0, 23.9)]
OTHERS = [(Q4_K, 3418, 2048, 512, "k_gemm_q4_k_w<8>", 23.5, 40.6), (Q4_K, 222, 12544, 3328, "k_gemm_q4_k_w<8>", 45.0, 59.6),
          (Q5_K, 776, 2048, 512, "k_gemm_q5_k_ws<2>", 10.3, 12.9), (Q4_K, 40, 7680, 2048, "k_gemm_q4_k_rb<1, 4, 3, 2>", 10.4, 11.7)]
SMALL = [(Q6_K, 37, 2560, 9728), (Q4_K, 16, 2560, 2560), (Q4_K, 256, 1024, 2560), (Q8_0, 1024, 512, 512), (Q8_0, 128, 512, 9760),
         (Q5_K, 3, 2048, 2048), (Q2_K, 65, 640, 256)]


@pytest.mark.parametrize("gtype,M,N,K,us,small_us", STREAM_K)
def test_stream_k_keeps(gtype, M, N, K, us, small_us):
    assert stream_k(gtype, M, N, K), hq.gemm_kernel(gtype, M, N, K)


@pytest.mark.parametrize("gtype,M,N,K,name,us,small_us", OTHERS)
def test_other_kernels_keep(gtype, M, N, K, name, us, small_us):
    assert hq.gemm_kernel(gtype, M, N, K) == name


@pytest.mark.parametrize("gtype,M,N,K", SMALL)
def test_small_tiles_keep(gtype, M, N, K):
    name = hq.gemm_kernel(gtype, M, N, K)
    assert name.startswith(("k_gemm_q8_0<", "k_gemm_q4_k<", "k_gemm_q6_k<", "k_gemm_kq<")) and not stream_k(gtype, M, N, K), name
    assert hq.gemm_workspace_bytes(gtype, M, N, K)[3]


# hq_gemm_swiglu at M <= 64: (type, M, I, K, us of hq_gemm's kernel and the pass, us of one small-tile kernel)
SWIGLU = [(Q8_0, 38, 832, 3328, 11.0, 18.8), (Q8_0, 3, 896, 3584, 9.2, 15.1), (Q8_0, 2, 2560, 2560, 9.6, 12.4), (Q8_0, 23, 3840, 3840, 15.1, 18.6),
          (Q8_0, 17, 9728, 2560, 23.6, 25.9), (Q8_0, 16, 9728, 2560, 19.9, 17.3), (Q8_0, 2, 14336, 4096, 24.4, 23.7), (Q4_K, 16, 9728, 2560, 19.3, 16.4),
          (Q4_K, 64, 9728, 2560, 34.3, 29.2), (Q4_K, 2, 5632, 2048, 14.4, 9.3), (Q5_K, 33, 1024, 512, 0, 0), (Q2_K, 64, 1024, 256, 0, 0)]


@pytest.mark.parametrize("gtype,M,I,K,us,small_us", SWIGLU)
def test_swiglu_route(gtype, M, I, K, us, small_us):
    small = bool(hq.load().hq_internal_swiglu_small(gtype, M, I, K, 256))
    if small_us > 1.04 * us:
        assert not small
    elif small_us <= .86 * us:  # (and the k-quants without a time, which all won)
        assert small


@pytest.mark.parametrize("M,N,K", [(7456384, 4096, 288), (5161984, 5000, 416), (818304, 30000, 1312), (828288, 30000, 2592), (8388608, 9000, 96)])
def test_launches_stay_within_a_grid(M, N, K):
    """The largest calls of a Q8_0 matrix with a ragged K: a launch has fewer than 2^32 threads, so the plan is not the
    small-tile kernels' (768 threads per 64 x 64 or 128 x 128 tile) but the persistent one."""
    assert hq.gemm_kernel(Q8_0, M, N, K) == "k_gemm_q8_0<8, 2>" and stream_k(Q8_0, M, N, K)
    assert -(-M // 64) * -(-N // 64) * 768 >= 1 << 32 or -(-M // 128) * -(-N // 128) * 768 >= 1 << 32
