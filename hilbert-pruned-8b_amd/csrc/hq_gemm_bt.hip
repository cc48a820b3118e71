// hq_gemm_bt.hip - Q4_K GEMM for large M on gfx950: 256 x 256 output tiles, 8 cooperating waves.
//
// C[M,N] (+)= A[M,K] . W^T with A fp16 and W GGUF Q4_K super-blocks resident in HBM (reference
// arithmetic: cleanroom-transformer/src/ggml_quant.h:51-59, :135-150; matmul src/cpu_backend.c:38-54).
//
// Why this shape. A 256 x 256 tile over the whole of K, 8 waves (two per SIMD, so one wave's LDS waits
// and decode run under the other's MFMAs) of all 256 rows and 32 columns each: every quant is decoded
// by one wave. Decoded weights never pass through LDS: in a 16 x 16 x 32 MFMA the weight operand of
// lane (ln, lg) is column ln, k 8lg .. 8lg + 7, and in a Q4_K quant group byte l holds k = l (low
// nibble) and k = 32 + l (high nibble), so the 8 quant bytes 8lg .. 8lg + 7 of a column's 32-byte group
// decode in registers into that lane's operands of both 32-k steps of a 64-k stage. Per stage LDS
// carries the activation tile (32 KB written, 256 KB read: each wave reads all rows) and the quant
// groups (8 KB written and read).
//
// What bounds it. The matrix cores are busy 61 % of the cycles, and under this load the card holds
// about 1.7 - 1.9 GHz of its 2.4: time goes with the work per product. Measured at M = 16384, K = 2560,
// fp32 output, GEMM with its k_asums pass: N = 9728 908 -> 820 us (895 -> 992 TFLOP/s), N = 9216
// 867 -> 776, M = 4096 259 -> 228, against waves of 128 x 64 that formed the column tables themselves,
// with a barrier at the end of each stage's MFMAs. Of that: tables from upload 2 %, waves of 32 columns
// 3 - 6 %, operands read across the barrier 2 %, pairs of M-tiles 0 - 4 %, whole lines stored 2 - 5 %.
// Slower: 32 x 32 x 16 MFMAs (8 - 15 %), persistent workgroups whose next tile loads under the stores
// (1 - 3 %: 22 registers spilled); no gain: non-temporal stores (-1 to +3 %), a read-ahead of 7.
//
// Pipeline. K is walked in stages of 64 (one 32-byte quant group p of a super-block u: low nibbles
// = sub-block 2p, high = 2p + 1). Activations and quant groups are triple-buffered in LDS. In stage
// s = 4u + p every wave issues the activation DMA of stage s + 2 (4 of the tile's 32 1-KB DMAs) and its
// quant DMA (1 of 8), at p = 1 also its shares of the super-block's activation sums and Bmin and of the
// next one's records; then the stage's two 32-k k-steps (32 MFMAs each), at p = 3 followed by the min
// k-step (below). Every load is issued as assembly, out of the compiler's count: the wait of stage s
// (s_waitcnt vmcnt, then s_barrier, 5 of its 32 MFMA groups before its end) is for everything issued
// before stage s, so each load has between one and two stages to land.
//
// Arithmetic: as hq_gemm_ws.hip (accumulators in units of c_u = d_u, the weight operand the exact
// integer s*q; at a super-block's end times c_u/c_{u+1}, then the min term, one bf16 MFMA per (16 x 16
// block, super-block) with hi/lo splits of the sub-block sums S and of x = -dmin*m/c_{u+1}; behind the
// last super-block, which stays in its own units, times c_{U-1}). Output lane (ln, lg) of a 16 x 16
// block holds row ln, columns 4lg .. 4lg + 3.
//
// LDS (144 KB): A [3][256 rows][64 k] fp16, 128 B per row, 16-byte slot p at p ^ ((row >> 1) & 7)
// (the 16 lanes of an operand read hit 16 distinct 4-bank groups); quant groups [3][256 columns][32
// B], the two 16-byte halves of column c swapped where (c >> 3) & 1 (conflict-free 8-byte reads); S
// [256 rows][16] bf16 (hi[8], lo[8]); from the column tables formed at upload (k_q4k_tables) Bmin
// [256][16] bf16 (Bh[8], Bl[8]) and records [2][256] {scale words of sub-blocks 0-3 and 4-7 (zero where
// d = 0), c_u/c_{u+1}, c_{u+1}} by super-block parity.
#include <type_traits>

#include "hq_device.h"
#include "hq_kernels.h"

namespace {
constexpr int BT_BM = 256, BT_BN = 256, BT_KS = 64, BT_NT = 512;
constexpr int BT_MI = 16, BT_NJ = 2;      // a wave's 16-row and 16-column blocks: all 256 rows, 32 columns
constexpr int BT_GM = 2;                  // M-tiles walked together
constexpr int BT_RING = 8, BT_AHEAD = 5;  // activation operand ring and read-ahead, in row blocks

struct BtArgs {
    const uint8_t *W;  // Q4_K super-blocks, row n at n * row_bytes
    uint32_t row_bytes;
    const uint16_t *A;  // fp16 [M][K]
    const uint16_t *S;  // activation sub-block sums [M][K/256][16] (k_asums, bf16 hi/lo)
    const uint8_t *tab; // per-super-block column tables (hq_launch_q4k_tables)
    int M, N, K;
    void *C;
    int c_f32, accumulate;
    int mt, nt;
};

struct BtLds {
    static constexpr int A = 0, A_BYTES = BT_BM * BT_KS * 2;  // per buffer (3 buffers)
    static constexpr int Q = 3 * A_BYTES, Q_BYTES = BT_BN * 32;  // quant groups, per buffer (3 buffers)
    static constexpr int S = Q + 3 * Q_BYTES;        // [256][16] bf16
    static constexpr int BM = S + BT_BM * 32;        // [256][16] bf16
    static constexpr int REC = BM + BT_BN * 32;      // [2][256][16 B], by super-block parity
    static constexpr int TOTAL = REC + 2 * BT_BN * 16;
    static_assert(TOTAL <= 160 * 1024, "LDS budget");
};

DEV void bt_barrier() { asm volatile("s_barrier" ::: "memory"); }

__global__ void __launch_bounds__(BT_NT) k_gemm_q4_k_bt(BtArgs g) {
    using L = BtLds;
    constexpr int MI = BT_MI, NJ = BT_NJ, RING = BT_RING, AD = BT_AHEAD;
    __shared__ __attribute__((aligned(256))) char lds[L::TOTAL];
    const int M = g.M, N = g.N, K = g.K, U = K / 256, S2 = 4 * U;
    // tile of this workgroup: XCD x = b % 8 runs the x-th eighth of the tile list (pairs of M-tiles, N-tile
    // by N-tile: the workgroups that run together on an XCD share activations and weights in its L2).
    // M = 16384, K = 2560: 836 us at N = 9216 one M-tile at a time, 805 in pairs, 812 in fours, 825 in eights.
    const int T = g.mt * g.nt, per = (T + 7) / 8, b = blockIdx.x, t = (b & 7) * per + (b >> 3);
    if (t >= T) return;
    const int g0 = t / (BT_GM * g.nt) * BT_GM, gm = min(g.mt - g0, BT_GM), tr = t - g0 * g.nt;
    const int m0 = (g0 + tr % gm) * BT_BM, n0 = tr / gm * BT_BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 15, lg = lane >> 4;
    const rsrc_t ra = make_rsrc(g.A, (uint32_t)((size_t)M * K * 2));
    const rsrc_t rw = make_rsrc(g.W, (uint32_t)((size_t)N * g.row_bytes));
    const rsrc_t rs = make_rsrc(g.S, (uint32_t)((size_t)M * U * 32));
    const rsrc_t rt = make_rsrc(g.tab, (uint32_t)((size_t)N * U * HQ_Q4K_TAB_BYTES + HQ_Q4K_TAB_PAD));
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds, tab_step = (uint32_t)N * HQ_Q4K_TAB_BYTES;

    // ---- activation DMA: instruction q (0..3) of wave w fills rows 8(4w + q) .. + 8 of a buffer;
    // lane i: row r = 8(4w + q) + i/8, LDS slot i % 8, global 8-value chunk (i % 8) ^ ((r >> 1) & 7),
    // which is the q = 0 chunk ^ 4 for odd q
    // (the row in the VGPR offset, the one a buffer load range-checks: rows past M read zeros and no
    // load reads past the end of A)
    const int a_row0 = 32 * wave + (lane >> 3);
    const uint32_t a_ch = (uint32_t)((lane & 7) ^ ((a_row0 >> 1) & 7));
    uint32_t a_voff[4];
#pragma unroll
    for (int q = 0; q < 4; q++) a_voff[q] = (uint32_t)(m0 + a_row0 + 8 * q) * (uint32_t)K * 2u + 16u * (q & 1 ? a_ch ^ 4u : a_ch);
    auto dma_a1 = [&](int s, int buf, int q) {
        dma16_so(ra, lds0 + (uint32_t)(L::A + buf * L::A_BYTES + wave * 4096 + q * 1024), a_voff[q], (uint32_t)(s * BT_KS * 2));
    };
    // S of super-block u: wave w moves rows 32w .. + 32 (1 KB); lane i: row 32w + i/2, half i % 2
    const uint32_t s_voff = (uint32_t)(m0 + 32 * wave + (lane >> 1)) * (uint32_t)U * 32u + 16u * (uint32_t)(lane & 1);
    auto dma_s = [&](int u) { dma16_so(rs, lds0 + (uint32_t)(L::S + wave * 1024), s_voff, (uint32_t)(u * 32)); };
    // quant DMA of stage s (group s % 4 of super-block s / 4, 32 bytes per column): wave w moves
    // columns 32w .. + 32; lane i: column c = 32w + i/2, LDS half i % 2 of the column's 32 bytes, which
    // holds the group's half (i % 2) ^ ((c >> 3) & 1) (so that the 8-byte operand reads below hit
    // distinct banks)
    const int q_col = 32 * wave + (lane >> 1);
    const uint32_t q_voff = (uint32_t)(n0 + q_col) * g.row_bytes + 16u * (uint32_t)((lane & 1) ^ ((q_col >> 3) & 1));
    auto dma_q = [&](int s, int buf) {
        dma16_so(rw, lds0 + (uint32_t)(L::Q + buf * L::Q_BYTES + wave * 1024), q_voff,
                 (uint32_t)((s >> 2) * 144 + 16 + 32 * (s & 3)));
    };
    // column tables of super-block u: Bmin (wave w: columns 32w .. + 32), records (64 columns; waves 4 - 7
    // repeat what waves 0 - 3 bring, so that every wave's count of loads is the same). Columns past N read
    // other table bytes (the upload leaves HQ_Q4K_TAB_PAD zero bytes after the last tables); their outputs
    // are not stored.
    const uint32_t bm_voff = (uint32_t)(n0 + 32 * wave) * 32u + 16u * (uint32_t)lane;
    const uint32_t rec_voff = (uint32_t)N * 32u + (uint32_t)(n0 + 64 * (wave & 3) + lane) * 16u;
    auto dma_bm = [&](int u) { dma16_so(rt, lds0 + (uint32_t)(L::BM + wave * 1024), bm_voff, (uint32_t)u * tab_step); };
    auto dma_rec = [&](int u, int par) {
        dma16_so(rt, lds0 + (uint32_t)(L::REC + par * BT_BN * 16 + (wave & 3) * 1024), rec_voff, (uint32_t)u * tab_step);
    };

    // ---- MFMA work of a wave: rows 16 i (i < MI), columns 16 (NJ wave + j)
    const uint32_t xs = 16u * ((uint32_t)lg ^ (uint32_t)((ln >> 1) & 7));  // k-step 0 slot; k-step f: ^ 64 f
    const uint32_t a_lane = lds0 + (uint32_t)(L::A + ln * 128) + xs;
    const uint32_t s_lane = lds0 + (uint32_t)(L::S + ln * 32 + 16 * (lg & 1));
    const uint32_t m_lane = lds0 + (uint32_t)(L::BM + (16 * NJ * wave + ln) * 32 + 16 * (lg >> 1));
    const uint32_t f_lane = lds0 + (uint32_t)(L::REC + (16 * NJ * wave + 4 * lg) * 16 + 8);   // F, c of the lane's output columns
    const uint32_t sw_lane = lds0 + (uint32_t)(L::REC + (16 * NJ * wave + ln) * 16);         // scale words of its operand column
    // quants of column block j for lane (ln, lg): column c = 16 (NJ wave + j) + ln, bytes 8 lg .. + 7 of the
    // group (((c >> 3) & 1) is j-independent)
    const uint32_t q_lane = lds0 + (uint32_t)(L::Q + (16 * NJ * wave + ln) * 32 + 16 * ((lg >> 1) ^ ((ln >> 3) & 1)) + 8 * (lg & 1));
    using lds_h8 = const __attribute__((address_space(3))) h8;
    using lds_f1 = const __attribute__((address_space(3))) float;
    using lds_u1 = const __attribute__((address_space(3))) uint32_t;
    using lds_u2 = const __attribute__((address_space(3))) u2v;
    auto at = [](uint32_t byte) { return *(lds_h8 *)(uintptr_t)byte; };
    auto atf = [](uint32_t byte) { return *(lds_f1 *)(uintptr_t)byte; };
    auto at1 = [](uint32_t byte) { return *(lds_u1 *)(uintptr_t)byte; };
    auto at2 = [](uint32_t byte) { return *(lds_u2 *)(uintptr_t)byte; };
    f4 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    // One stream of MFMA groups (a group: one 16-row block against the wave's NJ column blocks): 2 MI per
    // stage, and behind stage 3 the MI groups of the super-block's min term. The activation operands
    // (and the sums' in the min groups) come through a ring of 8 that reads AD groups ahead, across
    // stages: the stage's wait and barrier stand AD groups before its end, where its own reads are all
    // out, so the next stage's first operands, quants and scale words are read and decoded behind the
    // last AD groups' MFMAs. Groups are held in order by scheduling barriers: left alone, the compiler
    // reads each operand right before its MFMAs.
    static_assert(AD < RING && (2 * MI) % RING == 0 && MI % RING == 0 && NJ < 8, "operand ring");
    static_assert(11 * (MI / 8) < 2 * MI - AD, "a stage's loads are issued before its wait");
    h8 af[RING], b0[NJ], b1[NJ], bm[NJ];
    f4 r[NJ];
    u2v q[NJ];
    uint32_t sw[NJ];
    h2 mu[NJ], ad[NJ];
    auto read_quants = [&](int p, int buf, int u) {
        const uint32_t ql = q_lane + (uint32_t)(buf * L::Q_BYTES), sl = sw_lane + (uint32_t)((u & 1) * BT_BN * 16 + (p >> 1) * 4);
#pragma unroll
        for (int j = 0; j < NJ; j++) q[j] = at2(ql + (uint32_t)(j * 16 * 32)), sw[j] = at1(sl + (uint32_t)(j * 256));
    };
    // scales of column block j's sub-blocks 2p, 2p + 1 (bytes 2(p % 2), 2(p % 2) + 1 of its scale word)
    // and its k-step 0 operand
    auto decode0 = [&](int p, int j) {
        const h2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
        const h2 sp = as_h2(__builtin_amdgcn_perm(0x64646464u, sw[j] >> ((p & 1) * 16), 0x04010400u)) - k1024;  // (s_lo, s_hi)
        mu[j] = sp * h2{(_Float16)1.0f, (_Float16)0.0625f};
        ad[j] = sp * h2{(_Float16)-1024.0f, (_Float16)-64.0f};
        b0[j] = decode8<false>(q[j], h2{mu[j].x, mu[j].x}, h2{ad[j].x, ad[j].x});
    };
    const int u_last = U - 1;
    auto stage = [&](auto P, int u, int ab) {
        constexpr int p = decltype(P)::value, G = p == 3 ? 3 * MI : 2 * MI, pn = (p + 1) & 3;
        const int s = 4 * u + p, an = ab == 2 ? 0 : ab + 1, ab2 = ab == 0 ? 2 : ab - 1;  // buffers s, s + 1, s + 2 (% 3)
        const int s_src = s + 2 < S2 ? s + 2 : S2 - 1;
        const uint32_t al[2] = {a_lane + (uint32_t)(ab * L::A_BYTES), (a_lane ^ 64u) + (uint32_t)(ab * L::A_BYTES)};
        const uint32_t aln = a_lane + (uint32_t)(an * L::A_BYTES);
        auto rd = [&](int g) {
            return g < 2 * MI ? at(al[g / MI] + (uint32_t)((g % MI) * 16 * 128))
                 : g < G      ? at(s_lane + (uint32_t)((g - 2 * MI) * 16 * 32))
                              : at(aln + (uint32_t)((g - G) * 16 * 128));
        };
#pragma unroll
        for (int g = 0; g < G; g++) {
            if (g == G - AD) {
                // every load issued before this stage has landed (the ones of this stage may stay in
                // flight): activations and quants of stage s + 1, at p = 2 the min term's tables
                if (p == 1) asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
                else asm volatile("s_waitcnt vmcnt(5) lgkmcnt(0)" ::: "memory");
                bt_barrier();
                read_quants(pn, an, p == 3 ? u + 1 : u);
            }
            af[(g + AD) % RING] = rd(g + AD);
            if (p == 3 && g == 2 * MI - 4) {
                const uint32_t fl = f_lane + (uint32_t)((u & 1) * BT_BN * 16);
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    bm[j] = at(m_lane + (uint32_t)(j * 16 * 32));
#pragma unroll
                    for (int e = 0; e < 4; e++) r[j][e] = atf(fl + (uint32_t)(j * 256 + e * 16));
                }
            }
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                f4 &c = acc[g % MI][j];
                c = g < MI ? mfma(b0[j], af[g % RING], c) : g < 2 * MI ? mfma(b1[j], af[g % RING], c) : mfma_bf16(bm[j], af[g % RING], c);
            }
            if (g < NJ) b1[g] = decode8<true>(q[g], h2{mu[g].y, mu[g].y}, h2{ad[g].y, ad[g].y});
            if (p == 3 && g >= 2 * MI - 1 && g + 1 < G)  // c_u -> c_{u+1}, one group before the min term
#pragma unroll
                for (int j = 0; j < NJ; j++) acc[(g + 1) % MI][j] *= r[j];
            if (g >= G - NJ) decode0(pn, g - (G - NJ));
            // the stage's loads, spread over its groups (a burst of them would hold up every wave's MFMAs
            // while the address unit works through them)
            constexpr int D = MI / 8;
            if (g % D == 0) {
                const int k = g / D;
                if (k == 1 || k == 3 || k == 5 || k == 7) dma_a1(s_src, ab2, k >> 1);
                if (k == 8) dma_q(s_src, ab2);
                if (p == 1 && k == 9) dma_s(u);  // their last readers are two barriers back
                if (p == 1 && k == 10) dma_bm(u);
                if (p == 1 && k == 11) dma_rec(u < u_last ? u + 1 : u_last, (u + 1) & 1);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // ---- prologue: activations and quants of stages 0 and 1, records of unit 0
#pragma unroll
    for (int s = 0; s < 2; s++) {
#pragma unroll
        for (int i = 0; i < 4; i++) dma_a1(s, s, i);
        dma_q(s, s);
    }
    dma_rec(0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    bt_barrier();
    read_quants(0, 0, 0);
#pragma unroll
    for (int i = 0; i < AD; i++) af[i] = at(a_lane + (uint32_t)(i * 16 * 128));
#pragma unroll
    for (int j = 0; j < NJ; j++) decode0(0, j);

    // ---- main loop: one super-block (4 stages) per iteration; stage s = 4u + p in buffer s % 3. Every
    // stage issues the same loads whatever u is (sources past the end of K are clamped to the last unit
    // or stage; what they bring is never used), so the wait counts are constants.
    int ab = 0;
    auto nxt = [](int b) { return b == 2 ? 0 : b + 1; };
    for (int u = 0; u < U; u++) {
        stage(std::integral_constant<int, 0>{}, u, ab), ab = nxt(ab);
        stage(std::integral_constant<int, 1>{}, u, ab), ab = nxt(ab);
        stage(std::integral_constant<int, 2>{}, u, ab), ab = nxt(ab);
        stage(std::integral_constant<int, 3>{}, u, ab), ab = nxt(ab);
    }
    // the last stages' (clamped, unused) loads still write LDS: land them
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // ---- output: back to true units (the last unit's c), rows 16 i + ln, columns
    // 16 (NJ wave + j) + 4 lg .. + 3
    const uint32_t cl_lane = f_lane + (uint32_t)((u_last & 1) * BT_BN * 16) + 4u;
    f4 cl[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) cl[j][e] = atf(cl_lane + (uint32_t)(j * 256 + e * 16));
#pragma unroll
    for (int i = 0; i < MI; i++) {
        const int m = m0 + 16 * i + ln;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int n = n0 + 16 * (NJ * wave + j) + 4 * lg;
            const f4 v = acc[i][j] * cl[j];
            if (n >= N) continue;
            const size_t idx = (size_t)m * N + n;
            if (n + 4 <= N && (N & 3) == 0) {
                if (g.c_f32) {
                    f4 *c = (f4 *)((float *)g.C + idx);
                    *c = g.accumulate ? *c + v : v;
                } else {
                    typedef _Float16 hh4 __attribute__((ext_vector_type(4)));
                    hh4 *c = (hh4 *)((_Float16 *)g.C + idx);
                    *c = __builtin_convertvector(g.accumulate ? __builtin_convertvector(*c, f4) + v : v, hh4);
                }
            } else {
                for (int e = 0; e < 4 && n + e < N; e++) store_out(g.C, idx + e, v[e], g.c_f32, g.accumulate);
            }
        }
    }
}
}  // namespace

// every byte offset of the kernel (tile rows and columns past the matrix included) fits 32 bits
int hq_bt_fits(const hq_dev_mat *W, int M) {
    const size_t lim = (size_t)1 << 32, mr = (size_t)M + BT_BM;
    return W->type == HQ_TYPE_Q4_K && W->cols % 256 == 0 && M >= 1 && mr * W->cols * 2 < lim &&
           mr * (W->cols / 256) * 32 < lim && ((size_t)W->rows + BT_BN) * W->row_bytes < lim &&
           ((size_t)W->rows + BT_BN) * (W->cols / 256) * HQ_Q4K_TAB_BYTES + HQ_Q4K_TAB_PAD < lim;
}

hipError_t hq_launch_gemm_bt(const hq_dev_mat *W, const uint16_t *A, const uint16_t *S, int M, void *C, int c_f32,
                             int accumulate, hipStream_t st) {
    if (!hq_bt_fits(W, M) || !W->tab) return hipErrorInvalidValue;
    BtArgs g;
    g.W = W->qs, g.row_bytes = (uint32_t)W->row_bytes, g.A = A, g.S = S, g.tab = W->tab;
    g.M = M, g.N = (int)W->rows, g.K = (int)W->cols, g.C = C, g.c_f32 = c_f32, g.accumulate = accumulate;
    g.mt = (M + BT_BM - 1) / BT_BM;
    g.nt = (g.N + BT_BN - 1) / BT_BN;
    const int T = g.mt * g.nt, per = (T + 7) / 8;
    k_gemm_q4_k_bt<<<(unsigned)(8 * per), BT_NT, 0, st>>>(g);
    return hipGetLastError();
}
