// attn_fwd_f32.hip -- the fp32 mode's flash-attention forward for gfx950.
//
// Same result definition and masks as attn_fwd.hip, on fp32 Q, K and V with
// fp32 accuracy: both products run on the bf16 matrix cores as six products
// of three-piece operands (split3, mfma_split3 in common.h).
//
// A workgroup is NW (4 or 8) wave64s: WQ of them along the queries (32 rows
// each) and WK = NW / WQ along the keys. A stage is WK sub-tiles of 32 keys, one per
// key wave. The threads load a stage's K and V as fp32 one stage ahead, split
// them and store the pieces in LDS (row-major planes in the slab layout of
// common.h). S^T = K Q^T gives every lane the scores of one query; P is split
// in registers and feeds O^T += V^T P^T, whose V^T operand is read from the
// row-major planes with ds_read_b64_tr_b16. Key waves keep their own offset,
// row sum and O and merge through LDS at the end.
//
// Bound: the matrix cores, at 6 bf16 products per fp32 product (2.7 times the
// rate of v_mfma_f32_32x32x2_f32, the earlier form), and beside them the VALU
// (6.5 instructions per MFMA at D = 64: exp2, the splits of P, K and V; the
// matrix pipe is busy 0.53 of the C2 grid's cycles). Large grids reach 207
// TFLOP/s of fp32 work at D = 64 and 215 at D = 128 (192 x 4096 x 4096; 128 and
// 131 before), 70% of what a loop of bf16 MFMAs on random data sustains. The C2
// encoder (B 8, H 12, S 1024, D 64) 248 -> 143 us traced, 217 -> 133 us a call
// in a stream of them; error against 64 bits O 6.5e-7 -> 5.4e-7, LSE 3.6e-8 ->
// 2.1e-8 (fewer roundings per sum).
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace gonn {

// The running offset moves only when a tile's maximum exceeds it by more
// than this (log2 units), so the O rescale is rare and P stays below 2^8.
constexpr float kF32LazyLog2 = 8.0f;

// The wave's 32 rows again on the fp32 matrix cores, reading global memory:
// for rows whose result SplitCheck rejects. An infinite or nearly infinite input
// has no three-piece split (inf - inf), a very small one loses bits in it, so
// such rows take the plain products.
// One wave, 16 bytes a load: 8 x 12 x 1024, D 64 takes 169 us on ordinary data,
// 450 with one infinite V in every slice (one float a load: 1319) and 230 in a
// kernel of nothing but fp32 instructions.
template <int D, bool CAUSAL>
GONN_DEV void fwd_f32_plain(const FwdParams& p, int bh, int qw, int Sk, f32x16* oacc, float& m,
                            float& l) {
    constexpr int HD = D / 2, NDT = D / 32;
    const int lane = threadIdx.x & 63, g = lane >> 5, ln = lane & 31, qi = qw + ln;
    const int Ss = p.Sk;
    const float* qrow = (const float*)p.q + ((size_t)bh * p.Sq + (qi < p.Sq ? qi : 0)) * D + g * HD;
    const float sg = qi < p.Sq ? p.qsign : 0.f, c2 = p.scale_log2;
    const float* Kg = (const float*)p.k + (size_t)bh * Ss * D;
    const float* Vg = (const float*)p.v + (size_t)bh * Ss * D;
    const float* mrow = p.mask ? p.mask + (size_t)(bh / p.H) * p.mask_sb +
                                     (size_t)(bh % p.H) * p.mask_sh +
                                     (size_t)(qi < p.Sq ? qi : 0) * Ss
                               : nullptr;
    int kend = Sk;
    if (CAUSAL && qw + 32 < kend) kend = qw + 32;
    for (int t = 0; t < NDT; t++) oacc[t] = f32x16{};
    m = -INFINITY;
    l = 0.f;
#pragma unroll 1
    for (int kb = 0; kb < kend; kb += 32) {
        const int kr = kb + ln < Sk ? kb + ln : Sk - 1;
        const float* krow = Kg + (size_t)kr * D + g * HD;
        f32x16 s = f32x16{};
#pragma unroll 1
        for (int i0 = 0; i0 < HD; i0 += 32) {
            f32x4 kx[8], qx[8];
            for (int i = 0; i < 8; i++) {
                kx[i] = *(const f32x4*)(krow + i0 + 4 * i);
                qx[i] = *(const f32x4*)(qrow + i0 + 4 * i);
            }
            for (int i = 0; i < 32; i++) s = mfma_f32(kx[i / 4][i % 4], qx[i / 4][i % 4] * sg, s);
        }
        float mx = -INFINITY;
        for (int r = 0; r < 16; r++) {
            const int key = kb + 8 * (r >> 2) + 4 * g + (r & 3);
            if (mrow && key < Sk) s[r] += mrow[key] * p.mask_mul;
            if (key >= Sk || (CAUSAL && key > qi)) s[r] = -INFINITY;
            mx = fmaxf(mx, s[r]);
        }
        mx = pair_max32(mx);
        const float mnew = fmaxf(m, mx);
        const float alpha = (m == -INFINITY) ? 0.f : fast_exp2((m - mnew) * c2);
        const float mref = (mnew == -INFINITY) ? 0.f : mnew;
        float rs = 0.f;
        for (int r = 0; r < 16; r++) {
            s[r] = fast_exp2((s[r] - mref) * c2);
            rs += s[r];
        }
        l = l * alpha + rs;
        m = mnew;
        for (int t = 0; t < NDT; t++) oacc[t] *= alpha;
        for (int r = 0; r < 16; r++) {
            int key = kb + 8 * (r >> 2) + 4 * g + (r & 3);
            key = key < Sk ? key : Sk - 1;
            for (int t = 0; t < NDT; t++)
                oacc[t] = mfma_f32(Vg[(size_t)key * D + t * 32 + ln], s[r], oacc[t]);
        }
    }
    l = pair_sum32(l);
}

template <int D, bool CAUSAL, bool MASK, int NW, int WQ, int NBUF, int OCC>
__global__ __launch_bounds__(NW * 64, OCC) void fwd_f32_kernel(FwdParams p) {
    constexpr int WK = NW / WQ, NT = NW * 64;
    constexpr int BM = WQ * 32, BN = WK * 32;
    constexpr int NKS = D / 16, NDT = D / 32;
    constexpr uint32_t PB = 32 * D * 2;  // bytes of one piece plane of a sub-tile
    constexpr uint32_t SUB = 6 * PB, STAGE = WK * SUB;
    constexpr int NCH = 32 * D / 8;      // 8-element chunks of a sub-tile plane
    constexpr int CH = WK * NCH / NT;    // chunks per thread (each of K, V)
    static_assert(CH * NT == WK * NCH && (NCH % NT == 0 || NT % NCH == 0), "whole chunks");
    __shared__ __attribute__((aligned(16))) char smem[NBUF * STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wq = wave % WQ, wk = wave / WQ;
    const int g = lane >> 5, ln = lane & 31;
    int bh, qb;
    map_block(blockIdx.x, p.nqb, p.BH, CAUSAL, bh, qb, CAUSAL ? p.hgroup : 1,
              deal_slices(p));
    const int q0 = qb * BM, qw = q0 + wq * 32, qi = qw + ln;
    const int Sq = p.Sq, Sk = fwd_keys(p, bh), Ss = p.Sk;  // keys taking part, slice stride
    if (Sk == 0) {  // uniform: the whole slice is padded
        fwd_empty_rows<D>(p, bh, q0, BM);
        return;
    }
    const float c2 = p.scale_log2;
    int kend = Sk;
    if (CAUSAL && q0 + BM < kend) kend = q0 + BM;
    const int nst = (kend + BN - 1) / BN;
    const float* Kg = (const float*)p.k + (size_t)bh * Ss * D;
    const float* Vg = (const float*)p.v + (size_t)bh * Ss * D;

    // Chunk i of this thread: sub-tile csub, row crow, elements ccol .. +7.
    f32x4 kreg[CH][2], vreg[CH][2];
    int crow[CH], ccol[CH];
    for (int i = 0; i < CH; i++) {
        const int pos = i * NT + tid;
        int r, c;
        slab_chunk(pos % NCH, 32, r, c);
        crow[i] = pos / NCH * 32 + r;
        ccol[i] = c * 8;
    }
    // Sub-tiles past the key end are neither loaded nor stored, nor read (by
    // chunk instruction, which fills part of one or whole ones).
    auto live_chunk = [&](int st, int i) { return WK == 1 || st * BN + i * NT / NCH * 32 < kend; };
    auto gload = [&](int st) {
        for (int i = 0; i < CH; i++) {
            if (!live_chunk(st, i)) break;
            int key = st * BN + crow[i];
            key = key < Sk ? key : Sk - 1;  // clamped rows are masked
            const float* kp = Kg + (size_t)key * D + ccol[i];
            const float* vp = Vg + (size_t)key * D + ccol[i];
            kreg[i][0] = *(const f32x4*)kp;
            kreg[i][1] = *(const f32x4*)(kp + 4);
            vreg[i][0] = *(const f32x4*)vp;
            vreg[i][1] = *(const f32x4*)(vp + 4);
        }
    };
    auto sstore = [&](int st, int buf) {
        for (int i = 0; i < CH; i++) {
            if (!live_chunk(st, i)) break;
            const int pos = i * NT + tid;
            char* dst = smem + buf * STAGE + pos / NCH * SUB + pos % NCH * 16;
            for (int w = 0; w < 2; w++) {
                float x[8];
                for (int e = 0; e < 8; e++) x[e] = w ? vreg[i][e >> 2][e & 3] : kreg[i][e >> 2][e & 3];
                const bf16x8x3 t = split3(x);
                *(bf16x8*)(dst + (3 * w + 0) * PB) = t.h;
                *(bf16x8*)(dst + (3 * w + 1) * PB) = t.m;
                *(bf16x8*)(dst + (3 * w + 2) * PB) = t.l;
            }
        }
    };
    gload(0);

    // Q pieces: qf[ks] = Q[qi][16 ks + 8 g .. +7] * sign(scale).
    bf16x8x3 qf[NKS];
    {
        const float* qrow = (const float*)p.q + ((size_t)bh * Sq + (qi < Sq ? qi : 0)) * D + g * 8;
        const float sg = qi < Sq ? p.qsign : 0.f;
        for (int ks = 0; ks < NKS; ks++) {
            const f32x4 a = *(const f32x4*)(qrow + ks * 16), b = *(const f32x4*)(qrow + ks * 16 + 4);
            float x[8];
            for (int e = 0; e < 4; e++) {
                x[e] = a[e] * sg;
                x[4 + e] = b[e] * sg;
            }
            qf[ks] = split3(x);
        }
    }
    // The additive mask's row of this lane's query (rows Ss apart).
    const float* mrow = nullptr;
    if constexpr (MASK)
        mrow = p.mask + (size_t)(bh / p.H) * p.mask_sb + (size_t)(bh % p.H) * p.mask_sh +
               (size_t)(qi < Sq ? qi : 0) * Ss;

    // Operand reads from a sub-tile: K row ln, chunk 2 ks + g (ds_read_b128);
    // V^T (row d = 32 dt + ln, k-slots = keys 16 ks + {4g..4g+3, 8+4g..8+4g+3},
    // the order P holds them) by two ds_read_b64_tr_b16, as the dK/dV kernel
    // reads its Q and dO transposes (attn_bwd.hip).
    const int hs = slab_swz(ln);
    const uint32_t qa0 = (uint32_t)(ln * 64 + ((0 + g) ^ hs) * 16);
    const uint32_t qa1 = (uint32_t)(ln * 64 + ((2 + g) ^ hs) * 16);
    const int s16 = lane & 15, tcx = 2 * ((ln >> 4) & 1) + ((s16 >> 1) & 1);
    const uint32_t ta0 = (uint32_t)((4 * g + (s16 >> 2)) * 64 + (tcx ^ g) * 16 + 8 * (s16 & 1));
    const uint32_t ta1 =
        (uint32_t)((8 + 4 * g + (s16 >> 2)) * 64 + (tcx ^ (2 + g)) * 16 + 8 * (s16 & 1));
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s4 lds_s4;
    typedef __attribute__((address_space(3))) char lds_char;
    lds_char* const tm = (lds_char*)smem;
    auto kfrag = [&](uint32_t base, int piece, int ks) {
        return *(const bf16x8*)(smem + base + piece * PB + (ks >> 1) * 2048 +
                                ((ks & 1) ? qa1 : qa0));
    };
    auto vfrag = [&](uint32_t base, int piece, int ks, int dt) {
        lds_char* const b = tm + base + (3 + piece) * PB + (dt * 32 + 16 * ks) * 64;
        const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(b + ta0));
        const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(b + ta1));
        const s4 b8[2] = {lo, hi};
        return __builtin_bit_cast(bf16x8, b8);
    };

    f32x16 oacc[NDT];
    for (int t = 0; t < NDT; t++) oacc[t] = f32x16{};
    // m: the offset in raw score units, mc = m c2 rounded; P = 2^(s c2 - mc)
    // is exact for any offset while its rounding stays small, so only LSE
    // needs it (dlt below).
    float m = -INFINITY, mc = 0.f, l = 0.f;

    auto compute = [&](int st, int buf) {
        const int kbase = st * BN + wk * 32;
        if (kbase >= kend || (CAUSAL && kbase > qw + 31)) return;  // wave-uniform: no key here
        const uint32_t base = buf * STAGE + wk * SUB;
        f32x16 s = f32x16{};
        for (int ks = 0; ks < NKS; ks++) {
            const bf16x8x3 k = {kfrag(base, 0, ks), kfrag(base, 1, ks), kfrag(base, 2, ks)};
            s = mfma_split3(k, qf[ks], s);
        }
        if constexpr (MASK) {  // scale * s + m = scale_abs * (s + m / scale_abs)
            for (int r = 0; r < 16; r++) {
                const int key = kbase + 8 * (r >> 2) + 4 * g + (r & 3);
                if (key < Sk) s[r] += mrow[key] * p.mask_mul;
            }
        }
        if ((kbase + 32 > Sk) || (CAUSAL && kbase + 31 > qw)) {
            int lim = Sk - 1;
            if (CAUSAL) lim = qi < lim ? qi : lim;
            const int thr = lim - (kbase + 4 * g);
            for (int r = 0; r < 16; r++) s[r] = 8 * (r >> 2) + (r & 3) > thr ? -INFINITY : s[r];
        }
        float mx = fmaxf(s[0], s[1]);
        for (int r = 2; r < 16; r++) mx = fmaxf(mx, s[r]);
        mx = pair_max32(mx);
        const bool need = mx > m && (m == -INFINITY || (mx - m) * c2 > kF32LazyLog2);
        if (__builtin_amdgcn_ballot_w64(need)) {
            const float mn = need ? mx : m;
            const float mcn = (mn == -INFINITY) ? 0.f : mn * c2;
            // The ratio of the two offsets as they were subtracted: without a
            // mask that of the rounded products.
            const float step = MASK ? (m - mn) * c2 : mc - mcn;
            const float alpha = (m == -INFINITY) ? 0.f : fast_exp2(step);
            m = mn;
            mc = mcn;
            l *= alpha;
            for (int t = 0; t < NDT; t++) oacc[t] *= alpha;
        }
        float rs[4] = {0.f, 0.f, 0.f, 0.f};
        const float mref = (m == -INFINITY) ? 0.f : m;
        bf16x8x3 pf[2];
        for (int ks = 0; ks < 2; ks++) {
            float e[8];
            for (int j = 0; j < 8; j++) {
                // With an additive mask the difference is formed before the
                // scaling, so scores equal to the offset give exactly 1 at any
                // magnitude (-1e30 on every key of a row gives ties).
                if constexpr (MASK) e[j] = fast_exp2((s[8 * ks + j] - mref) * c2);
                else e[j] = fast_exp2(__builtin_fmaf(s[8 * ks + j], c2, -mc));
                rs[j & 3] += e[j];
            }
            pf[ks] = split3(e);
        }
        l += (rs[0] + rs[1]) + (rs[2] + rs[3]);
        for (int ks = 0; ks < 2; ks++)
            for (int dt = 0; dt < NDT; dt++) {
                const bf16x8x3 v = {vfrag(base, 0, ks, dt), vfrag(base, 1, ks, dt),
                                    vfrag(base, 2, ks, dt)};
                oacc[dt] = mfma_split3(v, pf[ks], oacc[dt]);
            }
    };

    sstore(0, 0);
    __syncthreads();
    for (int st = 0; st < nst; st++) {
        const int buf = NBUF == 2 ? st & 1 : 0;
        if (st + 1 < nst) gload(st + 1);
        compute(st, buf);
        if (NBUF == 1) __syncthreads();
        if (st + 1 < nst) sstore(st + 1, NBUF == 2 ? buf ^ 1 : 0);
        __syncthreads();
    }

    float lt = pair_sum32(l);
    if constexpr (WK > 1) {
        const int nlive = kend + 31 < WK * 32 ? (kend + 31) / 32 : WK;  // key waves with keys
        // Key wave w > 0 of query wave wq leaves (O, m, mc, l) in LDS, element
        // e of lane at word (e * 64 + lane); key wave 0 merges them in order.
        constexpr int NE = 16 * NDT + 3;
        static_assert((WK - 1) * WQ * NE * 256 <= NBUF * (int)STAGE, "the merge fits in the stages");
        float* red = (float*)smem;
        if (wk > 0 && wk < nlive) {
            float* d = red + ((wk - 1) * WQ + wq) * NE * 64 + lane;
            for (int t = 0; t < NDT; t++)
                for (int r = 0; r < 16; r++) d[(t * 16 + r) * 64] = oacc[t][r];
            d[(NE - 3) * 64] = m;
            d[(NE - 2) * 64] = mc;
            d[(NE - 1) * 64] = lt;
        }
        if (nlive > 1) __syncthreads();  // uniform
        if (wk > 0) return;
        for (int w = 1; w < nlive; w++) {
            const float* d = red + ((w - 1) * WQ + wq) * NE * 64 + lane;
            const float m2 = d[(NE - 3) * 64], mc2 = d[(NE - 2) * 64], l2 = d[(NE - 1) * 64];
            const bool up = m2 > m;
            const float M = up ? m2 : m, MC = up ? mc2 : mc;
            float a, b;
            if constexpr (MASK) {
                a = m == -INFINITY ? 0.f : fast_exp2((m - M) * c2);
                b = m2 == -INFINITY ? 0.f : fast_exp2((m2 - M) * c2);
            } else {
                a = m == -INFINITY ? 0.f : fast_exp2(mc - MC);
                b = m2 == -INFINITY ? 0.f : fast_exp2(mc2 - MC);
            }
            lt = lt * a + l2 * b;
            for (int t = 0; t < NDT; t++)
                for (int r = 0; r < 16; r++) oacc[t][r] = oacc[t][r] * a + d[(t * 16 + r) * 64] * b;
            m = M;
            mc = MC;
        }
    }
    // Rows that are not finite or below the split's range, or whose scores are
    // so large that mc is far from m c2: once more without the split (see above).
    float dlt = (MASK || m == -INFINITY) ? 0.f : __builtin_fmaf(m, c2, -mc);
    {
        // A mask of -inf on every key leaves m = -inf, l = 0: a result.
        bool bad = nonfinite(lt);
        // The rounding of mc scales P by up to 2^16 here, beyond by too much.
        if constexpr (!MASK) bad |= m == -INFINITY || !(__builtin_fabsf(mc) < 0x1p28f);
        SplitCheck chk;
        for (int t = 0; t < NDT; t++)
            for (int r = 0; r < 16; r++) chk.add(oacc[t][r]);
        bad |= chk.plain();
        if (__builtin_amdgcn_ballot_w64(bad && qi < Sq)) {
            fwd_f32_plain<D, CAUSAL>(p, bh, qw, Sk, oacc, m, lt);
            dlt = 0.f;
        }
    }
    if (qi < Sq) {
        const float inv = 1.f / lt;
        float* orow = p.o + ((size_t)bh * Sq + qi) * D;
        for (int t = 0; t < NDT; t++)
            for (int rq = 0; rq < 4; rq++) {
                f32x4 v;
                for (int i = 0; i < 4; i++) v[i] = oacc[t][rq * 4 + i] * inv;
                *(f32x4*)(orow + t * 32 + rq * 8 + g * 4) = v;
            }
        // LSE = (mc + log2 l) ln 2 with mc = m c2 - dlt. l's exponent and the
        // sum are taken in double: log2 l is as large as log2 of the key count
        // (the offset may trail the maximum), where fp32 would lose bits.
        if (p.lse && g == 0) {
            const int ex = __builtin_amdgcn_frexp_expf(lt);
            const float lm = fast_log2(__builtin_amdgcn_frexp_mantf(lt)) - dlt;
            p.lse[(size_t)bh * Sq + qi] = (float)((double)m * p.scale_abs + ((double)ex + lm) * kLn2d);
        }
    }
}

template <int D, bool C, int NW, int WQ, int NBUF, int OCC>
static void launch_f32(FwdParams p, long long cus, hipStream_t s) {
    p.nqb = (p.Sq + WQ * 32 - 1) / (WQ * 32);
    // Causal dispatch groups of about two XCDs' worth of resident workgroups
    // (map_block): 611 -> 530 us at D 64, 48 x 4096 queries, against groups
    // sized for two workgroups per CU where three are resident.
    const int slots = (int)cus / 8 * (OCC * 4 / NW);
    p.hgroup = 2 * slots / p.nqb > 1 ? 2 * slots / p.nqb : 1;
    const dim3 grid(p.nqb * p.BH);
    if (p.mask) fwd_f32_kernel<D, C, true, NW, WQ, NBUF, OCC><<<grid, NW * 64, 0, s>>>(p);
    else fwd_f32_kernel<D, C, false, NW, WQ, NBUF, OCC><<<grid, NW * 64, 0, s>>>(p);
}

// Waves and query rows per workgroup. Four waves of 128 rows split each K/V
// element least often and keep two (D = 128) or three (D = 64) workgroups on a
// CU; a grid too small to fill the chip that way gives waves to the keys
// instead, which shortens each workgroup's chain of key tiles, and takes eight
// of them where one workgroup per CU is all there is. Measured (us, rows x
// waves), heads x length on both sides of each bound:
//   D 64                      128x4  128x8   64x8   64x4
//     full     16 x 1024         56     45     33     38
//              20 x 1024         57     46     60     54
//              64 x 512          32     29     36     32
//              72 x 512          43     51     52     46
//     causal   32 x 512          31     26     19     22
//              64 x 512          32     27     26     24
//              192 x 512         49     64     76     61
//              32 x 1024         58     47     40     42
//              96 x 1024         85    108    114    107
//   D 128      16 x 1024        101     85      -     72
//     full     16 x 2048        211    183      -    282
//              96 x 512          86    100      -    120
//     causal   16 x 2048        199    163      -    158
//              48 x 1024        114     94      -    157
//              96 x 1024        163    197      -    247
// (64 rows and 8 waves would need 196 KB of LDS at D = 128.) A causal grid
// counts twice, since its blocks' lengths differ and the longest start first;
// under 1024 keys at D = 64 its blocks are too short for a second round of
// eight waves to pay and four waves take over. Up to 128 keys there is nothing
// for eight waves to do (D 64: 96 x 16 7.7 with 4, 8.0 with 8), and one
// sub-tile of keys at D = 128 goes to the smallest kernel (96 x 16: 10.0 with
// 128 rows, 10.8 with 64).
template <int D, bool C>
static void launch_f32_rows(const FwdParams& p, hipStream_t s) {
    const long long cus = device_cus();
    const long long b64 = (long long)((p.Sq + 63) / 64) * p.BH;
    const long long b128 = (long long)((p.Sq + 127) / 128) * p.BH;
    const bool uneven = C && p.Sq > 128;
    const long long room = (uneven ? 2 : 1) * cus;
    const bool many = p.Sk > 128;
    if constexpr (D == 64) {
        const bool chopped = uneven && p.Sk < 1024;
        if (many && b64 <= (chopped ? cus : room)) launch_f32<D, C, 8, 2, 1, 2>(p, cus, s);
        else if (many && !chopped && b128 <= room) launch_f32<D, C, 8, 4, 1, 2>(p, cus, s);
        else if (b64 <= (!many ? 2 : chopped ? 4 : 0) * cus) launch_f32<D, C, 4, 2, 1, 2>(p, cus, s);
        else launch_f32<D, C, 4, 4, 2, 3>(p, cus, s);
    } else {
        if (p.Sk > 32 && b64 <= room) launch_f32<D, C, 4, 2, 1, 1>(p, cus, s);
        else if (many && b128 <= room) launch_f32<D, C, 8, 4, 1, 2>(p, cus, s);
        else launch_f32<D, C, 4, 4, 1, 2>(p, cus, s);
    }
}

hipError_t launch_fwd_f32(const FwdParams& p, int D, int causal, hipStream_t s) {
    if (D == 64) {
        if (causal) launch_f32_rows<64, true>(p, s);
        else launch_f32_rows<64, false>(p, s);
    } else if (D == 128) {
        if (causal) launch_f32_rows<128, true>(p, s);
        else launch_f32_rows<128, false>(p, s);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace gonn
