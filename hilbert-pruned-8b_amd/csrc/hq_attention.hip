// hq_attention.hip - causal grouped-query softmax attention on the fp32 matrix cores.
//
// The queries that share a kv head are one matrix: row r = t rep + e of kv head g is token t of query
// head g rep + e (rep = nh / nkv), so grouped heads and neighbouring tokens read each key and value
// once. A workgroup takes 16 QB rows of one kv head; its W waves (and, for few rows, the workgroups of
// `splits` position ranges) take tiles of TP positions in turn, each with an online softmax of its own
// in fp32, and the waves' (max, sum, output) triples are added in wave order at the end.
//
// Everything is transposed so that nothing moves between lanes on the way from scores to outputs:
//   S^T = K Q^T: v_mfma_f32_16x16x4_f32 with A = 16 positions x 4 head dims, B = 4 head dims x 16 rows.
//     Lane (li = lane % 16, lg = lane / 16) holds K[position li][16 j + 4 lg + e] for step (j, e) and
//     Q[row li][the same dims]: one 16-byte load feeds four steps.
//   The result has row li of the block in every lane and positions 4 lg + r in its four registers, which
//   is the B operand (positions lg x row li) of step r of O^T = V^T P^T when A takes V[position 4 lg + r].
//     The 16 A rows of output block 4 c + b are the dims 64 c + 4 li + b, so one 16-byte load of V feeds
//     four blocks, and a lane ends with 16 neighbouring dims of its row.
// Row sums stay per lane until the end; the row maximum takes two lane exchanges per tile.
//
// Masked positions of a tile enter the output product with weight 0, not left out: an infinite or NaN value row of a
// later token of the same pass makes NaN of earlier rows of its block. The pass's last row attends to every one of
// them and is not finite either way.
//
// Bound: the fp32 matrix rate (256 FLOP per clock and CU); keys and values come from L2 straight into
// the operand registers (16 QB rows per read), V a tile's score phase ahead, K a softmax and output
// phase ahead. Measured (8 heads of 64, against one wave per token and head with vector dot products):
// 1024 tokens behind none / behind 1024: 370 / 790 -> 32 / 52 us; one token at position 1000, whose 32
// tiles go to 4 workgroups of 8 waves per head: 207 -> 11 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <math.h>

#include "hq_attention.h"
#include "hq_device.h"

namespace {

DEV f4 mfma4(float a, float b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

typedef float f2 __attribute__((ext_vector_type(2)));
constexpr int ATT_SPLITS = 64;  // most workgroups a row block's positions are split over

struct Args {
    HqAttnArgs a;
    int rep, R, nblk, splits;
};

// maximum over the four lanes that share a row
DEV float max_lg(float v) {
    v = fmaxf(v, __shfl_xor(v, 16, 64));
    return fmaxf(v, __shfl_xor(v, 32, 64));
}
DEV float sum_lg(float v) {
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}
// exp(x - m) of a part's maximum x against the row's m; a part without positions has x = -inf
DEV float part_scale(float x, float m) { return x == -INFINITY ? 0.f : expf(x - m); }

// HDP: head_dim rounded up to 64; EXACT: head_dim == HDP; QB: 16-row blocks per workgroup; TP:
// positions per tile; W: waves.
template <int HDP, bool EXACT, int QB, int TP, int W>
__global__ void __launch_bounds__(64 * W) k_attn(Args g) {
    constexpr int NJ = HDP / 16, NC = HDP / 64, PB = TP / 16, ROWS = 16 * QB, LDO = 68;
    __shared__ __align__(16) float os[W][ROWS][LDO];
    __shared__ float ms[W][ROWS], ls[W][ROWS];
    __shared__ int last;
    const HqAttnArgs &a = g.a;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, lg = lane >> 4;
    const int hd = EXACT ? HDP : a.hd, kvw = a.nkv * hd;
    // kv heads deal over the XCDs (consecutive workgroups), so a head's cache stays in one XCD's L2; the
    // row blocks with the most positions first
    int id = blockIdx.x;
    const int kvh = id % a.nkv;
    id /= a.nkv;
    const int split = id % g.splits, rb = g.nblk - 1 - id / g.splits, row0 = rb * ROWS;
    const int n = a.pos0 + std::min(g.R - 1, row0 + ROWS - 1) / g.rep + 1;  // positions some row sees
    const int n_all = a.pos0 + row0 / g.rep + 1;                            // positions every row sees
    const int ntile = (n + TP - 1) / TP, step = W * g.splits;

    f4 q[QB][NJ];
    int lim[QB];
#pragma unroll
    for (int b = 0; b < QB; b++) {
        const int r = row0 + 16 * b + li, t = r / g.rep, h = kvh * g.rep + r % g.rep;
        lim[b] = a.pos0 + t + 1;  // (rows past the last: any)
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int d = 16 * j + 4 * lg;
            q[b][j] = r < g.R && d < hd ? *(const f4 *)(a.qr + ((size_t)t * a.nh + h) * hd + d) : f4{0.f, 0.f, 0.f, 0.f};
        }
    }
    const float *kh = a.kc + (size_t)kvh * hd, *vh = a.vc + (size_t)kvh * hd;
    f4 kf[PB][NJ], vf[PB][4][NC];
    // positions past the last read it again (their weight is 0); dims past hd re-read the last ones (the
    // queries are 0 there, the outputs dropped)
    auto load_k = [&](int s0) {
#pragma unroll
        for (int b = 0; b < PB; b++) {
            const float *p = kh + (size_t)std::min(s0 + 16 * b + li, n - 1) * kvw;
#pragma unroll
            for (int j = 0; j < NJ; j++) kf[b][j] = *(const f4 *)(p + (EXACT ? 16 * j + 4 * lg : std::min(16 * j + 4 * lg, hd - 4)));
        }
    };
    auto load_v = [&](int s0) {
#pragma unroll
        for (int b = 0; b < PB; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float *p = vh + (size_t)std::min(s0 + 16 * b + 4 * lg + r, n - 1) * kvw;
#pragma unroll
                for (int c = 0; c < NC; c++) vf[b][r][c] = *(const f4 *)(p + (EXACT ? 64 * c + 4 * li : std::min(64 * c + 4 * li, hd - 4)));
            }
    };
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
    float m[QB], l[QB];
    f4 o[QB][4 * NC];
#pragma unroll
    for (int b = 0; b < QB; b++) {
        m[b] = -INFINITY, l[b] = 0.f;
#pragma unroll
        for (int c = 0; c < 4 * NC; c++) o[b][c] = zero;
    }
    int i = split * W + w;
    if (i < ntile) load_k(i * TP);
    for (; i < ntile; i += step) {
        const int s0 = i * TP;
        load_v(s0);
        f4 s[QB][PB];
#pragma unroll
        for (int b = 0; b < QB; b++)
#pragma unroll
            for (int p = 0; p < PB; p++) s[b][p] = zero;
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int p = 0; p < PB; p++)
#pragma unroll
                    for (int b = 0; b < QB; b++) s[b][p] = mfma4(kf[p][j][e], q[b][j][e], s[b][p]);
        if (i + step < ntile) load_k((i + step) * TP);
#pragma unroll
        for (int b = 0; b < QB; b++) {
            float mx = -INFINITY;
#pragma unroll
            for (int p = 0; p < PB; p++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    s[b][p][r] *= a.scale;
                    if (s0 + TP > n_all) s[b][p][r] = s0 + 16 * p + 4 * lg + r < lim[b] ? s[b][p][r] : -INFINITY;
                    mx = fmaxf(mx, s[b][p][r]);
                }
            const float mn = fmaxf(m[b], max_lg(mx)), m0 = mn == -INFINITY ? 0.f : mn;
            float add = 0.f;
#pragma unroll
            for (int p = 0; p < PB; p++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    s[b][p][r] = expf(s[b][p][r] - m0);
                    add += s[b][p][r];
                }
            const float alpha = expf(m[b] - m0);  // (0 before the first visible position)
            l[b] = l[b] * alpha + add;
            m[b] = mn;
#pragma unroll
            for (int c = 0; c < 4 * NC; c++) o[b][c] *= alpha;
        }
#pragma unroll
        for (int p = 0; p < PB; p++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int c = 0; c < NC; c++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int b = 0; b < QB; b++) o[b][4 * c + e] = mfma4(vf[p][r][c][e], s[b][p][r], o[b][4 * c + e]);
    }

    // the waves' parts, in wave order
#pragma unroll
    for (int b = 0; b < QB; b++) {
        const float lt = sum_lg(l[b]);
        if (lg == 0) ms[w][16 * b + li] = m[b], ls[w][16 * b + li] = lt;
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < QB; b++) {
        float mm = ms[0][16 * b + li];
#pragma unroll
        for (int v = 1; v < W; v++) mm = fmaxf(mm, ms[v][16 * b + li]);
        const float f = part_scale(m[b], mm);
#pragma unroll
        for (int c = 0; c < 4 * NC; c++) o[b][c] *= f;
    }
    constexpr int PARTF = HDP + 4;  // a partial row: its sums, then (max, sum)
    const int blk = rb * a.nkv + kvh;
    const rsrc_t rp = make_rsrc(a.part + (size_t)blk * g.splits * ROWS * PARTF, (uint32_t)g.splits * ROWS * PARTF * 4);
    // sums of row `row` at dims d .. d + 3, divided by the row's l and gated
    auto finish = [&](int row, int d, f4 v, float lt) {
        const int r = row0 + row, t = r / g.rep, h = kvh * g.rep + r % g.rep;
        if (r >= g.R || d >= hd) return;
        const float *gate = a.qb + (size_t)t * a.qw + (size_t)h * hd * 2 + hd + d;
        h4 y;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float x = v[e] / lt;
            if (a.gated) x *= 1.0f / (1.0f + expf(-gate[e]));
            y[e] = (_Float16)x;
        }
        *(h4 *)(a.out + ((size_t)t * a.nh + h) * hd + d) = y;
    };
#pragma unroll
    for (int c = 0; c < NC; c++) {
        if (c) __syncthreads();
#pragma unroll
        for (int b = 0; b < QB; b++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                *(f4 *)&os[w][16 * b + li][16 * lg + 4 * r] =
                    f4{o[b][4 * c][r], o[b][4 * c + 1][r], o[b][4 * c + 2][r], o[b][4 * c + 3][r]};
        __syncthreads();
        for (int x = threadIdx.x; x < ROWS * 16; x += 64 * W) {
            const int row = x >> 4, d = 4 * (x & 15);
            f4 v = *(const f4 *)&os[0][row][d];
            float mm = ms[0][row];
#pragma unroll
            for (int u = 1; u < W; u++) {
                v += *(const f4 *)&os[u][row][d];
                mm = fmaxf(mm, ms[u][row]);
            }
            float lt = 0.f;
#pragma unroll
            for (int u = 0; u < W; u++) lt += ls[u][row] * part_scale(ms[u][row], mm);
            if (g.splits == 1) {
                finish(row, 64 * c + d, v, lt);
            } else {
                const uint32_t at = (uint32_t)((split * ROWS + row) * PARTF) * 4u;
                buf_store16(rp, v, at + (uint32_t)(64 * c + d) * 4u);
                if (c == 0 && d == 0) buf_store16(rp, f4{mm, lt, 0.f, 0.f}, at + HDP * 4u);
            }
        }
    }
    if (g.splits == 1) return;
    // the last of the block's workgroups adds the parts in split order
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        last = atomicAdd(&a.counters[blk], 1) == g.splits - 1;
        if (last) atomicExch(&a.counters[blk], 0);
    }
    __syncthreads();
    if (!last) return;
    // each split's (max, sum) per row once into LDS, then its sums four loads at a time
    f2 *const ml = (f2 *)&os[0][0][0];
    static_assert(ATT_SPLITS * ROWS * sizeof(f2) <= sizeof os, "the splits' maxima and sums in the waves' arena");
    for (int x = threadIdx.x; x < g.splits * ROWS; x += 64 * W) {
        const f4 v = buf_load16_sc1(rp, (uint32_t)(x * PARTF + HDP) * 4u, 0);
        ml[x] = f2{v.x, v.y};
    }
    __syncthreads();
    for (int x = threadIdx.x; x < ROWS * (HDP / 4); x += 64 * W) {
        const int row = x / (HDP / 4), d = 4 * (x % (HDP / 4));
        if (row0 + row >= g.R) continue;
        float mm = -INFINITY;
        for (int u = 0; u < g.splits; u++) mm = fmaxf(mm, ml[u * ROWS + row].x);
        f4 v = zero;
        float lt = 0.f;
        for (int u0 = 0; u0 < g.splits; u0 += 4) {
            f4 y[4];
#pragma unroll
            for (int e = 0; e < 4; e++)
                y[e] = buf_load16_sc1(rp, (uint32_t)((std::min(u0 + e, g.splits - 1) * ROWS + row) * PARTF + d) * 4u, 0);
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (u0 + e < g.splits) {
                    const f2 p = ml[(u0 + e) * ROWS + row];
                    const float f = part_scale(p.x, mm);
                    v += y[e] * f;
                    lt += p.y * f;
                }
        }
        finish(row, d, v, lt);
    }
}

template <int HDP, int QB, int TP, int W>
void launch(const Args &g, hipStream_t st) {
    const unsigned grid = (unsigned)(g.nblk * g.a.nkv * g.splits);
    if (g.a.hd == HDP) k_attn<HDP, true, QB, TP, W><<<grid, 64 * W, 0, st>>>(g);
    else k_attn<HDP, false, QB, TP, W><<<grid, 64 * W, 0, st>>>(g);
}

constexpr int waves(int hd) { return hd <= 128 ? 8 : 4; }

}  // namespace

size_t hq_attn_work_bytes(int hd, int n_cu) {
    const size_t hdp = (size_t)(hd + 63) / 64 * 64;
    return (size_t)2 * n_cu * 16 * (hdp + 4) * sizeof(float);  // at most 2 n_cu parts of 16 rows
}

hipError_t hq_launch_attention(const HqAttnArgs &a, int n_cu, hipStream_t st) {
    Args g;
    g.a = a;
    g.rep = a.nh / a.nkv;
    g.R = a.T * g.rep;
    const int W = waves(a.hd), tp = a.hd <= 64 ? 32 : 16;
    // 32 rows per workgroup (half the cache reads) where that still gives every CU one
    const int qb = a.hd <= 128 && (long)((g.R + 31) / 32) * a.nkv >= n_cu ? 2 : 1;
    g.nblk = (g.R + 16 * qb - 1) / (16 * qb);
    // few row blocks: their positions over several workgroups, while every wave still gets a tile
    const long blocks = (long)g.nblk * a.nkv;
    const int tiles = (a.pos0 + a.T + tp - 1) / tp;
    g.splits = 1;
    if (blocks < n_cu && blocks <= HQ_ATTN_MAX_BLOCKS)
        g.splits = (int)std::max(1l, std::min({(long)(n_cu / blocks), (long)((tiles + W - 1) / W), (long)ATT_SPLITS}));
    if (a.hd <= 64) {
        if (qb == 2) launch<64, 2, 32, 8>(g, st);
        else launch<64, 1, 32, 8>(g, st);
    } else if (a.hd <= 128) {
        if (qb == 2) launch<128, 2, 16, 8>(g, st);
        else launch<128, 1, 16, 8>(g, st);
    } else if (a.hd <= 192) {
        launch<192, 1, 16, 4>(g, st);
    } else {
        launch<256, 1, 16, 4>(g, st);
    }
    return hipGetLastError();
}
