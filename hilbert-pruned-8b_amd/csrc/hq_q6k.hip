// hq_q6k.hip - GGUF Q6_K matrices on gfx950: decode.
//
// Reference arithmetic (cleanroom-transformer/src/ggml_quant.h:151-169): a super-block of 256 values
// {u8 ql[128], u8 qh[64], int8 scales[16], fp16 d}; value 128h + 32r + l (half h, lane r = 0..3,
// l = 0..31) has q = (ql[64h + 32(r % 2) + l] low nibble for r < 2, high for r >= 2)
// | (bits 2r, 2r + 1 of qh[32h + l]) << 4, minus 32, and y = (d * sc) * q with sc = scales[8h + 2r + l/16]
// (d * sc is exact in fp32; the second product can round).
//
// Device layout (written by hq_mat_upload): each 210-byte super-block is stored in a 224-byte slot
// {ql[128], qh[64], scales[16], d, 14 zero bytes}, so every 16-byte load is aligned; hq_mat_download
// restores the GGUF bytes.
//
// Kernels
//   k_dequant_q6_k  rows -> fp32, bit-identical to the reference decoder ((d * sc) * q in fp32).
//   (M = 1 and the option-row gather: k_gemv_sb in hq_kquant.hip)
//   (M >= 2: hq_gemm_sm.hip, k_gemm_kq_ws in hq_gemm_ws.hip)
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hq_device.h"
#include "hq_kernels.h"

namespace {
constexpr int Q6_SLOT = 224;  // device bytes per super-block

// Values v .. v + 15 (v a multiple of 16) of the super-block at blk as fp32, bit-identical to the
// reference decoder.
DEV void q6k_deq16(const uint8_t *blk, int v, float (&w)[16]) {
    const int h = v >> 7, r = (v >> 5) & 3, l0 = v & 16;
    const u4v ql = *(const u4v *)(blk + 64 * h + 32 * (r & 1) + l0);
    const u4v qh = *(const u4v *)(blk + 128 + 32 * h + l0);
    const float ds = h2f(*(const uint16_t *)(blk + 208)) * (float)(int8_t)blk[192 + 8 * h + 2 * r + (l0 >> 4)];
    const int shl = r >= 2 ? 4 : 0, shh = 2 * r;
    const uint32_t lw[4] = {ql.x, ql.y, ql.z, ql.w}, hw[4] = {qh.x, qh.y, qh.z, qh.w};
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const int lo = (int)((lw[e >> 2] >> (8 * (e & 3) + shl)) & 0xfu);
        const int hb = (int)((hw[e >> 2] >> (8 * (e & 3) + shh)) & 3u);
        w[e] = ds * (float)((lo | (hb << 4)) - 32);
    }
}

// one thread per (row, 16-value chunk); output row r is matrix row ids[r] when ids is given
__global__ void __launch_bounds__(256) k_dequant_q6_k(const uint8_t *__restrict__ W, size_t row_bytes, int K,
                                                      uint32_t row0, const uint32_t *__restrict__ ids, uint32_t nrows,
                                                      float *__restrict__ out) {
    const size_t per_row = (size_t)K / 16, total = (size_t)nrows * per_row;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t r = i / per_row, v0 = (i % per_row) * 16, row = ids ? (size_t)ids[r] : row0 + r;
        float w[16];
        q6k_deq16(W + row * row_bytes + (v0 / 256) * Q6_SLOT, (int)(v0 % 256), w);
        float4 *o = (float4 *)(out + r * (size_t)K + v0);
#pragma unroll
        for (int q = 0; q < 4; q++) o[q] = float4{w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]};
    }
}

unsigned grid_cap(size_t n, unsigned per, unsigned cap) {
    const size_t g = (n + per - 1) / per;
    return (unsigned)(g < cap ? (g ? g : 1) : cap);
}
}  // namespace

hipError_t hq_launch_dequant_q6k(const hq_dev_mat *W, uint32_t row0, const uint32_t *ids, uint32_t nrows, float *out,
                                 hipStream_t st) {
    const size_t n = (size_t)nrows * (W->cols / 16);
    k_dequant_q6_k<<<grid_cap(n, 256, 65536), 256, 0, st>>>(W->qs, W->row_bytes, (int)W->cols, row0, ids, nrows, out);
    return hipGetLastError();
}
