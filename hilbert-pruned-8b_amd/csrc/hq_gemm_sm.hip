// hq_gemm_sm.hip - GEMM for few output tiles (2 <= M, small M or small N), all block types: small tiles
// whose K is shared by the waves of a workgroup.
//
// C[M,N] (+)= A[M,K] . W^T, A fp16, W GGUF blocks resident in HBM (block layouts: hq_kquant.h,
// hq_q6k.hip, hq_kernels.hip; reference arithmetic cleanroom-transformer/src/ggml_quant.h:95-169).
//
// A workgroup of eight consumer and four loader waves computes a tile of 16 MB rows x 16 CW columns over K, or over one of
// `parts` ranges of it (tile_finish adds them). K runs in stages of one super-block (256 values) through
// a ring of NST LDS slots: the tile's activations and its columns' super-blocks as they lie in HBM, all
// by LDS DMA with neighbouring lanes on neighbouring bytes (the MFMA operand order, 16 rows by 64 bytes
// per instruction, read from L2 into registers took four times the cycles of a contiguous load). Wave
// (cg, kq) owns all rows of column group cg and the stage's kq-th share of K (8 / CW shares): it decodes
// its columns' bytes straight into MFMA fragments, so nothing decoded is stored. One barrier per stage.
// The K shares' tiles meet in LDS at the end and are added in share order.
//
// Why: a K loop inside one wave set leaves most CUs idle or a long serial chain where tiles are few, and
// cutting K over workgroups costs a round trip through memory per tile; here a tile is small (N = 2560:
// 40 of 64 columns) and its K still goes through 8 waves.
//
// What bounds it: the chain of stages, each a barrier, the decode (Q6_K at M = 37, N = 2560, K = 9728: 6.7 VALU
// instructions per MFMA; Q4_K at M = 256, N = 1024, K = 2560: 10) and few products per decoded operand (2 or 4 row
// blocks). There the matrix cores are busy 18 and 12 % of the cycles; for the first, HBM delivers 1.9 TB/s and L2 3.2,
// both well below what they can. Against the Stream-K kernels: the first shape 27.0 -> 15.5 us, the second 26.1 -> 9, Q4_K M = 16,
// N = K = 2560 11.1 -> 7.4.
//
// Operands of v_mfma_f32_16x16x32_f16 for k-step j of a half super-block: lane (ln, lg) holds row
// (column) ln, values 32 j + 8 lg .. + 7. Weights are never rounded, except Q8_0's (fp16(q d), as in
// every Q8_0 kernel): B is the exact integer of the value times its 6-bit (Q2_K: 4-bit) scale, a
// super-block's sums are multiplied by its fp32 d, and the mins (Q4_K, Q5_K, Q2_K) are a second exact
// product, of the min code with the same activations, times dmin. Q6_K's integer (up to 4096) is the
// exact sum of two fp16 ones, sc (low nibble) and 16 sc (high bits - 2).
#include <algorithm>
#include <type_traits>

#include "hq_device.h"
#include "hq_kernels.h"
#include "hq_kquant.h"

namespace {
struct SmArgs {
    const uint8_t *W;   // k-quants: super-blocks, row n at n * row_bytes; Q8_0: quant plane, row n at n * K
    const uint16_t *D;  // Q8_0 scale plane, row n at n * ldd
    uint32_t row_bytes, ldd;
    const uint16_t *A;
    int M, N, K;
    void *C;
    int c_f32, accumulate;
    int mt, nt, ntiles;
    int parts;
    float *partials;
    int *counters;
};

DEV u4v ld16(const char *p) { return *(const u4v *)p; }
DEV u2v ld8(const char *p) { return *(const u2v *)p; }
DEV uint32_t ld4(const char *p) { return *(const uint32_t *)p; }
DEV h2 splat2h(float x) { return h2{(_Float16)x, (_Float16)x}; }
// byte b of w (0 .. 255) in both halves as fp16, exact
DEV h2 byte_h2(uint32_t w, int b) { return as_h2(__builtin_amdgcn_perm(0x64646464u, w, 0x04000400u | (uint32_t)b | (uint32_t)b << 16)) - splat2h(1024.f); }
DEV h8 splat8h(h2 x) { return h8{x.x, x.x, x.x, x.x, x.x, x.x, x.x, x.x}; }
// (b - bias) * f for the 8 bytes b of w0, w1: exact integers
DEV h8 bytes_times(uint32_t w0, uint32_t w1, float bias, h2 f) {
    const h2 k = splat2h(1024.f + bias);
    const h2 a = (as_h2(perm_lo(w0)) - k) * f, b = (as_h2(perm_hi(w0)) - k) * f;
    const h2 c = (as_h2(perm_lo(w1)) - k) * f, d = (as_h2(perm_hi(w1)) - k) * f;
    return h8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}

// The lane's bytes of one column's half super-block h (b: the column's staged super-block), and the B
// operands of its four k-steps. Two MFMAs per block and k-step with MIN (the min term: its own sums and
// scale) and with TWO (two exact parts of the value).
template <int T>
struct Wb;

template <>
struct Wb<HQ_TYPE_Q4_K> {
    static constexpr bool MIN = true, TWO = false;
    u4v hdr;
    u2v q[2];
    __device__ __forceinline__ void load(const char *b, const char *, int h, int lg) {
        hdr = ld16(b);
#pragma unroll
        for (int i = 0; i < 2; i++) q[i] = ld8(b + 16 + 64 * h + 32 * i + 8 * lg);
    }
    uint32_t sw, mw;
    __device__ __forceinline__ void setup(int h, int) {
        uint32_t s0, s1, m0, m1;
        q4k_scale_words(hdr.y, hdr.z, hdr.w, s0, s1, m0, m1);
        sw = h ? s1 : s0, mw = h ? m1 : m0;
    }
    template <int J>
    __device__ __forceinline__ void frags(int, int, h8 &b1, h8 &b2) const {
        const h2 s = byte_h2(sw, J);
        constexpr float f = J & 1 ? 0.0625f : 1.0f;
        const h2 mul = s * splat2h(f), add = s * splat2h(-1024.f * f);
        b1 = decode8<(J & 1) != 0>(q[J >> 1], mul, add);
        b2 = splat8h(byte_h2(mw, J));
    }
    __device__ __forceinline__ float d() const { return h2f((uint16_t)hdr.x); }
    __device__ __forceinline__ float dmin() const { return h2f((uint16_t)(hdr.x >> 16)); }
};

template <>
struct Wb<HQ_TYPE_Q5_K> {
    static constexpr bool MIN = true, TWO = false;
    u4v hdr;
    u2v q[2], qh;
    __device__ __forceinline__ void load(const char *b, const char *, int h, int lg) {
        hdr = ld16(b);
        qh = ld8(b + 16 + 8 * lg);
#pragma unroll
        for (int i = 0; i < 2; i++) q[i] = ld8(b + 48 + 64 * h + 32 * i + 8 * lg);
    }
    uint32_t sw, mw;
    __device__ __forceinline__ void setup(int h, int) {
        uint32_t s0, s1, m0, m1;
        q4k_scale_words(hdr.y, hdr.z, hdr.w, s0, s1, m0, m1);
        sw = h ? s1 : s0, mw = h ? m1 : m0;
    }
    template <int J>
    __device__ __forceinline__ void frags(int h, int, h8 &b1, h8 &b2) const {
        constexpr int sh = 4 * (J & 1);
        const int sub = 4 * h + J;
        const uint32_t q0 = ((q[J >> 1].x >> sh) & 0x0f0f0f0fu) | (((qh.x >> sub) & 0x01010101u) << 4);
        const uint32_t q1 = ((q[J >> 1].y >> sh) & 0x0f0f0f0fu) | (((qh.y >> sub) & 0x01010101u) << 4);
        b1 = bytes_times(q0, q1, 0.f, byte_h2(sw, J));
        b2 = splat8h(byte_h2(mw, J));
    }
    __device__ __forceinline__ float d() const { return h2f((uint16_t)hdr.x); }
    __device__ __forceinline__ float dmin() const { return h2f((uint16_t)(hdr.x >> 16)); }
};

template <>
struct Wb<HQ_TYPE_Q2_K> {
    static constexpr bool MIN = true, TWO = false;
    u2v sc, q;
    uint32_t dd;
    __device__ __forceinline__ void load(const char *b, const char *, int h, int lg) {
        sc = ld8(b + 8 * h);
        dd = ld4(b + 80);
        q = ld8(b + 16 + 32 * h + 8 * lg);
    }
    __device__ __forceinline__ void setup(int, int lg) {  // bytes of scale 2 j + (lg >> 1) at byte 2 (j % 2)
        if (lg & 2) sc.x >>= 8, sc.y >>= 8;
    }
    template <int J>
    __device__ __forceinline__ void frags(int, int, h8 &b1, h8 &b2) const {
        const uint32_t s = J < 2 ? sc.x : sc.y;
        b1 = bytes_times((q.x >> (2 * J)) & 0x03030303u, (q.y >> (2 * J)) & 0x03030303u, 0.f, byte_h2(s & 0x0f0f0f0fu, 2 * (J & 1)));
        b2 = splat8h(byte_h2((s >> 4) & 0x0f0f0f0fu, 2 * (J & 1)));
    }
    __device__ __forceinline__ float d() const { return h2f((uint16_t)dd); }
    __device__ __forceinline__ float dmin() const { return h2f((uint16_t)(dd >> 16)); }
};

template <>
struct Wb<HQ_TYPE_Q3_K> {
    static constexpr bool MIN = false, TWO = false;
    u4v sc;  // scales[12], d
    u2v q, hm;
    __device__ __forceinline__ void load(const char *b, const char *, int h, int lg) {
        sc = ld16(b + 96);
        hm = ld8(b + 8 * lg);
        q = ld8(b + 32 + 32 * h + 8 * lg);
    }
    uint32_t s0, s1;  // 6-bit codes of scales 8 h + i in byte i of s0 (i < 4) and i - 4 of s1, moved as for Q2_K
    __device__ __forceinline__ void setup(int h, int lg) {
        const uint32_t lo0 = (h ? sc.x >> 4 : sc.x) & 0x0f0f0f0fu, lo1 = (h ? sc.y >> 4 : sc.y) & 0x0f0f0f0fu;
        s0 = lo0 | (((sc.z >> (4 * h)) & 0x03030303u) << 4);
        s1 = lo1 | (((sc.z >> (4 * h + 2)) & 0x03030303u) << 4);
        if (lg & 2) s0 >>= 8, s1 >>= 8;
    }
    template <int J>
    __device__ __forceinline__ void frags(int h, int, h8 &b1, h8 &) const {
        const h2 s = byte_h2(J < 2 ? s0 : s1, 2 * (J & 1)) - splat2h(32.f);
        const uint32_t q0 = ((q.x >> (2 * J)) & 0x03030303u) | (((hm.x >> (4 * h + J)) & 0x01010101u) << 2);
        const uint32_t q1 = ((q.y >> (2 * J)) & 0x03030303u) | (((hm.y >> (4 * h + J)) & 0x01010101u) << 2);
        b1 = bytes_times(q0, q1, 4.f, s);
    }
    __device__ __forceinline__ float d() const { return h2f((uint16_t)sc.w); }
    __device__ __forceinline__ float dmin() const { return 0.f; }
};

template <>
struct Wb<HQ_TYPE_Q6_K> {
    static constexpr bool MIN = false, TWO = true;
    u2v ql[2], qh, sc;
    uint32_t dd;
    __device__ __forceinline__ void load(const char *b, const char *, int h, int lg) {
#pragma unroll
        for (int i = 0; i < 2; i++) ql[i] = ld8(b + 64 * h + 32 * i + 8 * lg);
        qh = ld8(b + 128 + 32 * h + 8 * lg);
        sc = ld8(b + 192 + 8 * h);
        dd = ld4(b + 208);
    }
    __device__ __forceinline__ void setup(int, int lg) {
        if (lg & 2) sc.x >>= 8, sc.y >>= 8;
        sc.x ^= 0x80808080u, sc.y ^= 0x80808080u;  // signed scale + 128
    }
    template <int J>
    __device__ __forceinline__ void frags(int, int, h8 &b1, h8 &b2) const {
        const h2 s = byte_h2(J < 2 ? sc.x : sc.y, 2 * (J & 1)) - splat2h(128.f), s16 = s * splat2h(16.f);
        const u2v l = ql[J & 1];
        constexpr int sh = J < 2 ? 0 : 4;
        b1 = bytes_times((l.x >> sh) & 0x0f0f0f0fu, (l.y >> sh) & 0x0f0f0f0fu, 0.f, s);
        b2 = bytes_times((qh.x >> (2 * J)) & 0x03030303u, (qh.y >> (2 * J)) & 0x03030303u, 2.f, s16);
    }
    __device__ __forceinline__ float d() const { return h2f((uint16_t)dd); }
    __device__ __forceinline__ float dmin() const { return 0.f; }
};

template <>
struct Wb<HQ_TYPE_Q8_0> {
    static constexpr bool MIN = false, TWO = false;
    u2v q[4], dd;
    __device__ __forceinline__ void load(const char *b, const char *ds, int h, int lg) {
        dd = ld8(ds + 8 * h);
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = ld8(b + 128 * h + 32 * i + 8 * lg);
    }
    __device__ __forceinline__ void setup(int, int) {}
    template <int J>
    __device__ __forceinline__ void frags(int, int, h8 &b1, h8 &) const {
        const uint32_t w = J < 2 ? dd.x : dd.y;
        const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t)(J & 1 ? w >> 16 : w));
        b1 = bytes_times(q[J].x, q[J].y, 128.f, h2{d, d});  // stored bytes are q + 128
    }
    __device__ __forceinline__ float d() const { return 1.f; }
    __device__ __forceinline__ float dmin() const { return 0.f; }
};

// 16-byte pieces of a column's super-block, and the pieces its LDS copy takes: an odd number, so that the
// 16 columns of a fragment start in different bank groups
constexpr int sm_pieces(int t) { return t == HQ_TYPE_Q8_0 ? 16 : t == HQ_TYPE_Q4_K ? 9 : kq_slot(t) / 16; }
constexpr int sm_pitch(int t) { return sm_pieces(t) | 1; }
// waves of a workgroup: consumers, and loaders that issue the DMA (an instruction holds its wave at issue
// ~25 clocks per KB moved by the CU, so consumers would spend about half their time there)
constexpr int SM_W = 8, SM_L = 4, SM_NT = 64 * (SM_W + SM_L);
constexpr int SM_PARTS = 8;  // most workgroups a tile's K is split over
constexpr uint32_t SM_OUT = 0xfffffff0u;  // an offset past every buffer (of at most 2^32 - 16 bytes): reads zero

template <int T, int MB, int KW>
struct SmLds {
    static constexpr int CW = SM_W / KW, BM = 16 * MB, BN = 16 * CW, CP = sm_pitch(T);
    // weight DMA instructions of a stage; Q8_0: more for the columns' 8 scales (16 bytes each)
    static constexpr int WN = (BN * CP + 63) / 64, DN = T == HQ_TYPE_Q8_0 ? (BN + 63) / 64 : 0;
    static constexpr int A = BM * 512, D = A + WN * 1024, STAGE = D + DN * 1024;
    // slots: as many as leave room for two workgroups on a CU, at most four; two where one workgroup fills it
    static constexpr int NST = 4 * STAGE <= 80 * 1024 ? 4 : 3 * STAGE <= 160 * 1024 ? 3 : 2 * STAGE <= 160 * 1024 ? 2 : 1;
    static constexpr int RED = KW * BM * (BN + 4) * 4 + 16, RING = NST * STAGE, BYTES = RING > RED ? RING : RED;
    static_assert(BYTES <= 160 * 1024, "LDS budget");
};

// The tile of one workgroup.
template <int T, int MB, int KW>
DEV void sm_tile(const SmArgs &g, char *lds) {
    using B = Wb<T>;
    using L = SmLds<T, MB, KW>;
    constexpr int BM = L::BM, BN = L::BN, CP = L::CP, NST = L::NST, LD = BN + 4, SLOT = BM * LD;
    constexpr int AI = (BM / 2 + SM_L - 1) / SM_L, WN = L::WN, WI = (WN + L::DN + SM_L - 1) / SM_L;
    constexpr bool SB = T != HQ_TYPE_Q8_0;
    // column tiles dealt to the XCDs in turn, a column tile's parts and row tiles on one (its weights
    // come from HBM once); fewer than 8 column tiles: their row tiles and parts in turn
    const int per = g.mt * g.parts, r8 = g.nt < 8 ? blockIdx.x : blockIdx.x >> 3;
    const int nt_i = g.nt < 8 ? r8 / per : (int)(blockIdx.x & 7) + 8 * (r8 / per), part = (r8 % per) / g.mt, mt_i = r8 % g.mt;
    if (nt_i >= g.nt) return;
    const int m0 = mt_i * BM, n0 = nt_i * BN, tile = nt_i * g.mt + mt_i;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), ln = lane & 15, lg = lane >> 4;
    const int cg = w % L::CW, kq = w / L::CW;  // a consumer's column group and K share
    const int M = g.M, N = g.N, K = g.K, U = (K + 255) / 256;
    const int ua = (int)((long)U * part / g.parts), S = (int)((long)U * (part + 1) / g.parts) - ua;
    if (w >= SM_W) {
        const int lw = w - SM_W;
        const rsrc_t ra = make_rsrc(g.A, (uint32_t)((size_t)M * K * 2));
        const rsrc_t rw = make_rsrc(g.W, (uint32_t)((size_t)N * g.row_bytes));
        const rsrc_t rd = make_rsrc(g.D, (uint32_t)((size_t)N * g.ldd * 2));
        const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
        // A loader's DMA instructions of a stage. Activations: instruction q moves rows 2 q, 2 q + 1, slot p
        // of row r taking piece p ^ (r & 15). Weights: instruction t moves pieces 64 t .. 64 t + 63 of the
        // tile's [column][CP] pieces. Rows past M, columns past N and padding lie outside the ranges: their
        // whole offset but the stage's is in the (range-checked) VGPR, and stages stay inside a row.
        uint32_t va[AI], vw[WI];
        int per_stage = 0;
#pragma unroll
        for (int i = 0; i < AI; i++) {
            const int q = lw + SM_L * i, r = 2 * q + (lane >> 5), c = (lane & 31) ^ (r & 15);
            if (q < BM / 2) per_stage++;
            va[i] = m0 + r < M ? (uint32_t)(m0 + r) * (uint32_t)K * 2u + 16u * (uint32_t)c : SM_OUT;
        }
#pragma unroll
        for (int i = 0; i < WI; i++) {
            const int t = lw + SM_L * i, id = 64 * t + lane, col = t < WN ? id / CP : 64 * (t - WN) + lane, p = t < WN ? id % CP : 0;
            if (t < WN + L::DN) per_stage++;
            const bool in = col < BN && n0 + col < N && p < sm_pieces(T);
            vw[i] = !in ? SM_OUT : t < WN ? (uint32_t)(n0 + col) * g.row_bytes + 16u * (uint32_t)p : (uint32_t)(n0 + col) * g.ldd * 2u;
        }
        auto issue = [&](int s) __attribute__((always_inline)) {
            const int u = ua + s;
            const uint32_t at = lds0 + (uint32_t)(s % NST) * L::STAGE;
            // Q8_0: K may end inside the stage; pieces past it read zero
            const bool cut = T == HQ_TYPE_Q8_0 && 256 * u + 256 > K;
#pragma unroll
            for (int i = 0; i < AI; i++)
                if (lw + SM_L * i < BM / 2) {
                    const int q = lw + SM_L * i, c = (lane & 31) ^ ((2 * q + (lane >> 5)) & 15);
                    dma16_so(ra, at + (uint32_t)q * 1024u, cut && 256 * u + 8 * c >= K ? SM_OUT : va[i], (uint32_t)u * 512u);
                }
#pragma unroll
            for (int i = 0; i < WI; i++) {
                const int t = lw + SM_L * i;
                if (t < WN) {
                    const int p = (64 * t + lane) % CP;
                    dma16_so(rw, at + L::A + (uint32_t)t * 1024u, cut && 256 * u + 16 * p >= K ? SM_OUT : vw[i],
                             (uint32_t)u * (uint32_t)(16 * sm_pieces(T)));
                } else if (t < WN + L::DN) {
                    dma16_so(rd, at + L::D + (uint32_t)(t - WN) * 1024u, vw[i], (uint32_t)u * 16u);
                }
            }
        };
        // NST slots: stages up to s + NST - 1 are on their way while stage s is read (one slot: no overlap)
#pragma unroll
        for (int s = 0; s < (NST > 1 ? NST - 1 : 1); s++)
            if (s < S) issue(s);
        for (int s = 0; s < S; s++) {
            wait_vmcnt(per_stage * std::min(NST > 1 ? NST - 2 : 0, S - 1 - s));
            asm volatile("s_barrier" ::: "memory");  // stage s has landed; stage s - 1 is read
            if (NST > 1 && s + NST - 1 < S) issue(s + NST - 1);
            if (NST == 1 && s + 1 < S) {
                asm volatile("s_barrier" ::: "memory");
                issue(s + 1);
            }
        }
        asm volatile("s_barrier" ::: "memory");
    } else {
        const f4 zero = {0.f, 0.f, 0.f, 0.f};
        f4 acc[MB];
#pragma unroll
        for (int i = 0; i < MB; i++) acc[i] = zero;
        for (int s = 0; s < S; s++) {
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            const char *st = lds + (s % NST) * L::STAGE;
            const _Float16 *at = (const _Float16 *)st;
            f4 s1[MB], s2[MB];
#pragma unroll
            for (int i = 0; i < MB; i++) s1[i] = SB ? zero : acc[i], s2[i] = zero;
            float d = 1.f, dm = 0.f;
            auto half = [&](int h) __attribute__((always_inline)) {
                B b;
                b.load(st + L::A + (16 * cg + ln) * (CP * 16), st + L::D + (16 * cg + ln) * 16, h, lg);
                b.setup(h, lg);
                auto step = [&](auto J) __attribute__((always_inline)) {
                    constexpr int j = decltype(J)::value;
                    h8 b1, b2;
                    b.template frags<j>(h, lg, b1, b2);
#pragma unroll
                    for (int i = 0; i < MB; i++) {
                        const int r = 16 * i + ln, c = 16 * h + 4 * j + lg;
                        const h8 a = *(const h8 *)(at + r * 256 + 8 * (c ^ (r & 15)));
                        s1[i] = mfma(a, b1, s1[i]);
                        if constexpr (B::MIN) s2[i] = mfma(a, b2, s2[i]);
                        if constexpr (B::TWO) s1[i] = mfma(a, b2, s1[i]);
                    }
                };
                using std::integral_constant;
                step(integral_constant<int, 0>{});
                step(integral_constant<int, 1>{});
                step(integral_constant<int, 2>{});
                step(integral_constant<int, 3>{});
                d = b.d(), dm = b.dmin();
            };
            half(KW == 2 ? kq : 0);
            if constexpr (KW == 1) half(1);
#pragma unroll
            for (int i = 0; i < MB; i++) {
                if constexpr (SB) acc[i] += s1[i] * d;
                else acc[i] = s1[i];
                if constexpr (B::MIN) acc[i] -= s2[i] * dm;
            }
            if (NST == 1 && s + 1 < S) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        float *const red = (float *)lds;
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) red[kq * SLOT + (16 * i + 4 * lg + r) * LD + 16 * cg + ln] = acc[i][r];
    }
    __syncthreads();
    if constexpr (KW > 1) {
        for (int e = threadIdx.x; e < BM * BN / 4; e += SM_NT) {
            float *p = (float *)lds + e / (BN / 4) * LD + e % (BN / 4) * 4;
            *(f4 *)p += *(const f4 *)(p + SLOT);
        }
        __syncthreads();
    }
    tile_finish<BM, BN, SM_NT, SM_PARTS>(lds, g, m0, n0, tile, part, (int *)(lds + L::RED - 16));
}

#define SM_LDS(T, MB, KW) __shared__ __attribute__((aligned(1024))) char lds[SmLds<T, MB, KW>::BYTES]

}  // namespace

// The kernels: tiles of 16 MB rows x 128 / KW columns, each super-block shared by KW waves per column
template <int MB, int KW>
__global__ void __launch_bounds__(SM_NT) k_gemm_q8_0(SmArgs g) {
    SM_LDS(HQ_TYPE_Q8_0, MB, KW);
    sm_tile<HQ_TYPE_Q8_0, MB, KW>(g, lds);
}
template <int MB, int KW>
__global__ void __launch_bounds__(SM_NT) k_gemm_q4_k(SmArgs g) {
    SM_LDS(HQ_TYPE_Q4_K, MB, KW);
    static_assert(SmLds<HQ_TYPE_Q4_K, 1, KW>::BYTES <= SmLds<HQ_TYPE_Q4_K, 2, KW>::BYTES, "the one-block tile in the same arena");
    if (MB == 2 && g.M <= 16) sm_tile<HQ_TYPE_Q4_K, 1, KW>(g, lds);  // the second row block would be padding
    else sm_tile<HQ_TYPE_Q4_K, MB, KW>(g, lds);
}
template <int MB, int KW>
__global__ void __launch_bounds__(SM_NT) k_gemm_q6_k(SmArgs g) {
    SM_LDS(HQ_TYPE_Q6_K, MB, KW);
    sm_tile<HQ_TYPE_Q6_K, MB, KW>(g, lds);
}
template <int T, int MB, int KW>
__global__ void __launch_bounds__(SM_NT) k_gemm_kq(SmArgs g) {
    SM_LDS(T, MB, KW);
    sm_tile<T, MB, KW>(g, lds);
}

// Workgroups of a launch: column tiles padded to whole turns over the XCDs; 0 where their threads would pass the 2^32 - 1
// that a launch can have (outputs of some 50 GB: no plan then, another kernel runs)
static unsigned sm_grid(long mt, long nt, long parts) {
    const long n = (nt < 8 ? nt : 8 * ((nt + 7) / 8)) * mt * parts;
    return n * SM_NT < 1l << 32 ? (unsigned)n : 0u;
}

hipError_t hq_launch_gemm_sm(const hq_dev_mat *W, const uint16_t *A, int M, void *C, int c_f32, int accumulate, const HqSmPlan &p,
                             float *partials, int *counters, hipStream_t st) {
    if (p.parts < 1 || p.parts > SM_PARTS || (p.parts > 1 && (!partials || !counters))) return hipErrorInvalidValue;
    SmArgs g;
    g.W = W->qs, g.D = W->type == HQ_TYPE_Q8_0 ? W->d : (const uint16_t *)W->qs;
    g.row_bytes = W->type == HQ_TYPE_Q8_0 ? W->cols : (uint32_t)W->row_bytes;
    g.ldd = W->type == HQ_TYPE_Q8_0 ? (uint32_t)W->ldd : 0;
    g.A = A, g.M = M, g.N = (int)W->rows, g.K = (int)W->cols, g.C = C, g.c_f32 = c_f32, g.accumulate = accumulate;
    const int bn = 16 * SM_W / p.kw;
    g.mt = (M + 16 * p.mb - 1) / (16 * p.mb), g.nt = (g.N + bn - 1) / bn, g.ntiles = g.mt * g.nt;
    g.parts = p.parts, g.partials = partials, g.counters = counters;
    const unsigned grid = sm_grid(g.mt, g.nt, g.parts);
    if (!grid) return hipErrorInvalidValue;
#define SM_LAUNCH(k) k<<<grid, SM_NT, 0, st>>>(g); break
#define SM_CASE(mb, kw)                                                             \
    switch (W->type) {                                                              \
    case HQ_TYPE_Q8_0:                                                              \
        if constexpr (kw == 1) return hipErrorInvalidValue;                         \
        else k_gemm_q8_0<mb, kw><<<grid, SM_NT, 0, st>>>(g);                        \
        break;                                                                      \
    case HQ_TYPE_Q4_K: SM_LAUNCH((k_gemm_q4_k<mb == 1 ? 2 : mb, kw>));              \
    case HQ_TYPE_Q6_K: SM_LAUNCH((k_gemm_q6_k<mb, kw>));                            \
    case HQ_TYPE_Q2_K: SM_LAUNCH((k_gemm_kq<HQ_TYPE_Q2_K, mb, kw>));                \
    case HQ_TYPE_Q3_K: SM_LAUNCH((k_gemm_kq<HQ_TYPE_Q3_K, mb, kw>));                \
    case HQ_TYPE_Q5_K: SM_LAUNCH((k_gemm_kq<HQ_TYPE_Q5_K, mb, kw>));                \
    default: return hipErrorInvalidValue;                                           \
    }                                                                               \
    return hipGetLastError()
    switch (10 * p.mb + p.kw) {
    case 12: SM_CASE(1, 2);
    case 22: SM_CASE(2, 2);
    case 42: SM_CASE(4, 2);
    case 11: SM_CASE(1, 1);
    case 21: SM_CASE(2, 1);
    case 41: SM_CASE(4, 1);
    default: return hipErrorInvalidValue;
    }
#undef SM_CASE
#undef SM_LAUNCH
}

// Rows per tile follow M. One super-block (K <= 256) leaves nothing to share: 128-column tiles (not for Q8_0, which other
// kernels serve better there). Above, the row blocks and
// workgroups per tile with the least estimated time. The estimate, in us: launch, prologue and epilogue; what each
// further round of the fullest XCD costs; the stages of its CUs (decode and products, by type and rows); all stages'
// MB through the LDS DMA; millions of outputs, dearer where rows of C are not whole 8-value pieces; and the partial tiles'
// round trip of a K split. (Least squares over 51000 measured calls of every type, N = 1 .. 20000, K = 32 .. 15360,
// M = 2 .. 8192: half within 4 %, nine in ten within 9 %, 18 % for K <= 256.)
HqSmPlan hq_sm_plan(const hq_dev_mat *W, int M, int n_cu, int max_parts) {
    const int type = W->type, N = (int)W->rows, K = (int)W->cols, U = (K + 255) / 256;
    const bool q8 = type == HQ_TYPE_Q8_0, one = U <= 1;
    struct Fit { float base, round, stage, read, out, ragged; };
    static const Fit onek[3] = {{5.15f, 0.f, 0.f, .04f, 0.f, 12.2f}, {5.7f, 0.f, 0.f, 0.f, 0.f, 5.4f}, {7.f, 3.1f, 0.f, .06f, 0.f, 4.6f}},
                     fit8[3] = {{4.65f, 0.f, .63f, .033f, 0.f, 14.3f}, {4.86f, 2.5f, .8f, .013f, 0.f, 3.6f}, {5.6f, 3.5f, .97f, .007f, .4f, 2.f}},
                     fitk[3] = {{4.44f, 0.f, .4f, .033f, 0.f, 15.4f}, {4.84f, .8f, .5f, .022f, 0.f, 3.7f}, {5.47f, 3.8f, .7f, .02f, .53f, 2.7f}};
    const float decode = one || q8 || type == HQ_TYPE_Q3_K ? 0.f : type == HQ_TYPE_Q6_K ? .26f : type == HQ_TYPE_Q5_K ? .155f : .04f;
    const float q6 = one && type == HQ_TYPE_Q6_K ? 1.05f : 0.f, outputs = 1e-6f * (float)M * (float)N;
    const int top = M <= 16 ? 0 : M <= 32 ? 1 : 2, low = !one && M > 64 ? 1 : top, cols = one ? 128 : 64;
    const long nt = (N + cols - 1) / cols, xcd = std::max(1, n_cu / 8);
    HqSmPlan best = {0, 0, 0, 0.f};
    for (int lg = top; lg >= low; lg--) {
        const int mb = 1 << lg;
        const Fit &f = one ? onek[lg] : q8 ? fit8[lg] : fitk[lg];
        const long mt = (M + 16 * mb - 1) / (16 * mb);
        const float bytes = 1e-6f * (float)(16 * mb * 512 + cols * 16 * sm_pitch(type));
        for (int parts = 1; parts <= std::min(max_parts, SM_PARTS) && (parts == 1 || (2 * parts <= U && mt * nt * parts <= n_cu)); parts++) {
            if (!sm_grid(mt, nt, parts)) break;  // (K split or not, the next is larger)
            const long wgs = mt * nt * parts, rounds = nt < 8 ? (wgs + n_cu - 1) / n_cu : ((nt + 7) / 8 * mt * parts + xcd - 1) / xcd;
            const float stages = (float)((U + parts - 1) / parts);
            const float t = f.base + q6 + std::max(f.round, decode > .1f ? 3.f : 0.f) * (float)(rounds - 1) + (float)rounds * stages * (f.stage + decode) +
                            f.read * stages * (float)wgs * bytes + outputs * (f.out + (N % 8 ? f.ragged : 0.f)) +
                            (parts > 1 ? 1.f + .19f * (float)parts + .13f * (float)mb : 0.f);
            if (!best.parts || t < best.us) best = {mb == 1 && type == HQ_TYPE_Q4_K ? 2 : mb, one ? 1 : 2, parts, t};
        }
    }
    return best;
}
