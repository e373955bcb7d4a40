// attn_bwd_f32.hip -- the fp32 mode's backward (dK/dV and dQ) for gfx950.
//
// The identities, masks and padding of attn_bwd.hip on fp32 Q, K, V and dO
// with fp32 accuracy: every product runs on the bf16 matrix cores as six
// products of three-piece operands (split3, mfma_split3 in common.h).
//
//   dK/dV  a workgroup owns WB blocks of 32 keys, one per block wave, whose
//          K and V pieces stay in registers; its 4 / WB stream waves take
//          alternate 32-query tiles. S = Q K^T and dP = dO V^T give each lane
//          one key; P and dS are split in registers and feed
//          dV^T += dO^T P and dK^T += Q^T dS.
//   dQ     the same with the roles exchanged: a wave owns 32 queries (their Q
//          and dO pieces in registers), key tiles stream, S^T = K Q^T and
//          dP^T = V dO^T give each lane one query, dQ^T += K^T dS^T.
// A stage is 4 / WB tiles of 32 streamed rows of both streamed tensors: the
// threads load it as fp32 one stage ahead, split it and store the pieces in
// LDS (row-major planes in the slab layout of common.h); the transposed
// operands are read from the same planes with ds_read_b64_tr_b16. Stream
// waves keep their own sums and add them through LDS in order at the end, so
// results are deterministic.
//
// Bound: the matrix cores (six bf16 products per fp32 product, 2.7 times the
// rate of v_mfma_f32_32x32x2_f32, the earlier form), busy 0.54 of the cycles at
// D = 64, where the VALU of P, dS and the splits takes most of the rest, and 0.64
// (dK/dV) and 0.60 (dQ) at D = 128 (one wave per SIMD: the fragments need more
// than half the registers). Traced on one box, both forms in turn: B 8, H 12, S
// 1024, D 64: dK/dV 545 -> 282 us, dQ 361 -> 213 us; B 4, H 12, S 1024 causal:
// 289 -> 139 and 227 -> 91 us; 32 x 2048, D 128: 1127 -> 652 and 851 -> 511 us.
// Error against 64 bits: dQ 4.9e-7 -> 3.5e-7, dK 8.2e-7 -> 6.3e-7, dV 8.1e-7 ->
// 6.2e-7 (fewer roundings per sum).
#include "attn_f32_split.h"

namespace gonn {

// ---- plain fp32 products from global memory, for blocks whose result
// SplitCheck rejects: an infinite or nearly infinite input has no three-piece
// split, a very small one loses bits in it. 8 x 12 x 1024, D 64 forms dQ, dK and
// dV in 526 us on ordinary data, in 1773 with one infinite dO in every slice,
// which reaches every block (one float a load: 3512), and in 894 with nothing
// but fp32 instructions. ----
template <int D, bool CAUSAL>
GONN_DEV void dkdv_f32_plain(const BwdParams& p, int bh, int kw, f32x16* dvacc, f32x16* dkacc) {
    constexpr int HD = D / 2, NDT = D / 32;
    const int lane = threadIdx.x & 63, g = lane >> 5, ln = lane & 31, kj = kw + ln;
    const int S = p.S, Sk = p.Sk, kr = kj < Sk ? kj : Sk - 1;
    const float* kp = (const float*)p.k + ((size_t)bh * Sk + kr) * D + g * HD;
    const float* vp = (const float*)p.v + ((size_t)bh * Sk + kr) * D + g * HD;
    const float* Qg = (const float*)p.q + (size_t)bh * S * D;
    const float* dOg = (const float*)p.dO + (size_t)bh * S * D;
    const float* lg = p.lse2 + (size_t)bh * p.Sp;
    const float* dg = p.delta + (size_t)bh * p.Sp;
    const float* mcol = p.mask ? mask_slice(p, bh) + kr : nullptr;
    for (int t = 0; t < NDT; t++) dvacc[t] = dkacc[t] = f32x16{};
#pragma unroll 1
    for (int q0 = CAUSAL ? kw : 0; q0 < S; q0 += 32) {
        const int qr = q0 + ln < S ? q0 + ln : S - 1;
        f32x16 s = f32x16{}, dp = f32x16{};
        const float *qp = Qg + (size_t)qr * D + g * HD, *op = dOg + (size_t)qr * D + g * HD;
#pragma unroll 1
        for (int i0 = 0; i0 < HD; i0 += 16) plain_pair16(s, dp, qp + i0, kp + i0, op + i0, vp + i0);
        for (int r = 0; r < 16; r++) {
            const int q = q0 + 8 * (r >> 2) + 4 * g + (r & 3), qc = q < S ? q : S - 1;
            float off = q < S ? -lg[q] : -INFINITY;
            if (mcol) off += mcol[(size_t)qc * Sk] * kLog2e;
            float pv = fast_exp2(__builtin_fmaf(s[r], p.scale_log2, off));
            if (CAUSAL && kj > q) pv = 0.f;
            s[r] = pv;
            dp[r] = pv * (dp[r] - (q < S ? dg[q] : 0.f));
        }
        for (int r = 0; r < 16; r++) {
            const int q = q0 + 8 * (r >> 2) + 4 * g + (r & 3), qc = q < S ? q : S - 1;
            for (int t = 0; t < NDT; t++) {
                dvacc[t] = mfma_f32(dOg[(size_t)qc * D + t * 32 + ln], s[r], dvacc[t]);
                dkacc[t] = mfma_f32(Qg[(size_t)qc * D + t * 32 + ln], dp[r], dkacc[t]);
            }
        }
    }
}

template <int D, bool CAUSAL, bool MASK, int WB, int NBUF, int OCC>
__global__ __launch_bounds__(256, OCC) void bwd_dkdv_f32_kernel(BwdParams p) {
    constexpr int NS = 4 / WB, BK = WB * 32, BQ = NS * 32;  // keys per block, queries per stage
    constexpr int NKS = D / 16, NDT = D / 32;
    constexpr uint32_t STAGE = NS * SplitTile<D>::BYTES;
    __shared__ __attribute__((aligned(16))) char smem[NBUF * STAGE];
    __shared__ __attribute__((aligned(16))) float sld[NBUF][2][BQ];
    // With one wave per SIMD the next stage is split and stored beside the dK
    // products, with two after them (the registers allow no more).
    constexpr bool INNER = NBUF == 2 && OCC == 1;
    static_assert((NS - 1) * WB * 2 * NDT * 4096 <= NBUF * (int)STAGE, "the merge fits");

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wb = wave % WB, ws = wave / WB;
    const int g = lane >> 5, ln = lane & 31;
    const int S = p.S, Sp = p.Sp, Sk = p.Sk;  // S queries, Sk keys
    int bh, kb;
    map_block(blockIdx.x, (Sk + BK - 1) / BK, p.BH, false, bh, kb, 1, deal_slices(p));
    const int k0 = kb * BK, kw = k0 + wb * 32, kj = kw + ln;
    const int Skv = bwd_keys(p, bh);  // keys >= Skv are padded: dK = dV = 0
    const int st0 = CAUSAL ? k0 / BQ : 0, st1 = (S + BQ - 1) / BQ;
    if (k0 >= Skv || st0 >= st1) {
        bwd_zero_rows<D>(p.dk, Sk, bh, k0, BK);
        bwd_zero_rows<D>(p.dv, Sk, bh, k0, BK);
        return;
    }
    const float* Qg = (const float*)p.q + (size_t)bh * S * D;
    const float* dOg = (const float*)p.dO + (size_t)bh * S * D;
    const float* lg = p.lse2 + (size_t)bh * Sp;
    const float* dg = p.delta + (size_t)bh * Sp;

    SplitStage<D, NS> in;
    in.init(tid);
    float rl = 0.f, rd = 0.f;
    auto gload = [&](int st) {
        in.load(Qg, dOg, st * BQ, S);
        if (tid < BQ) {  // rows S .. Sp - 1 hold lse2 = +inf (P = 0)
            const int q = st * BQ + tid < Sp ? st * BQ + tid : Sp - 1;
            rl = lg[q];
            rd = dg[q];
        }
    };
    auto sstore = [&](int st, int buf) {
        in.store(smem + buf * STAGE, tid, st * BQ, S);
        if (tid < BQ) {
            sld[buf][0][tid] = rl;
            sld[buf][1][tid] = rd;
        }
    };
    gload(st0);
    const int kr = kj < Sk ? kj : Sk - 1;  // keys past Sk are computed, never written
    bf16x8x3 kf[NKS], vf[NKS];
    load_row_split<D>((const float*)p.k + ((size_t)bh * Sk + kr) * D, g, kf);
    load_row_split<D>((const float*)p.v + ((size_t)bh * Sk + kr) * D, g, vf);
    // The additive mask's column of this lane's key (rows Sk apart).
    const float* mcol = nullptr;
    if constexpr (MASK) mcol = mask_slice(p, bh) + kr;
    SplitTile<D> tl;
    tl.init(lane);

    f32x16 acc[2 * NDT];  // dV^T tiles, then dK^T tiles
    for (int t = 0; t < 2 * NDT; t++) acc[t] = f32x16{};
    const float c2 = p.scale_log2;

    auto compute = [&](int st, int buf, auto stage) {
        const int q0 = st * BQ + ws * 32;
        if (q0 >= S || (CAUSAL && kw > q0 + 31)) {  // wave-uniform: no pair here
            if constexpr (INNER) stage();
            return;
        }
        char* tile = smem + buf * STAGE + ws * SplitTile<D>::BYTES;
        // Each product beside the VALU work the one before it allows: dP with
        // P, dV with dS, dK with the next stage's splits.
        f32x16 s = f32x16{}, dp = f32x16{};
        for (int ks = 0; ks < NKS; ks++) s = mfma_split3(tl.row(tile, 0, ks), kf[ks], s);
        for (int ks = 0; ks < NKS; ks++) dp = mfma_split3(tl.row(tile, 1, ks), vf[ks], dp);
        const bool need_mask = CAUSAL && q0 < kw + 31;
        const int thr = need_mask ? kj - q0 - 4 * g : -1;  // query 8 (r / 4) + r % 4 < thr is masked
        bf16x8x3 pf[2], df[2];
        for (int ks = 0; ks < 2; ks++) {
            float e[8];
            for (int j4 = 0; j4 < 2; j4++) {
                const int qr = 16 * ks + 8 * j4 + 4 * g;
                const f32x4 L = *(const f32x4*)&sld[buf][0][ws * 32 + qr];
                for (int j = 0; j < 4; j++) {
                    const int r = 8 * ks + 4 * j4 + j;
                    float off = -L[j];
                    if constexpr (MASK) {
                        const int q = q0 + qr + j;
                        off += mcol[(size_t)(q < S ? q : S - 1) * Sk] * kLog2e;
                    }
                    const float pv = fast_exp2(__builtin_fmaf(s[r], c2, off));
                    s[r] = CAUSAL && 8 * (r >> 2) + (r & 3) < thr ? 0.f : pv;
                    e[4 * j4 + j] = s[r];
                }
            }
            pf[ks] = split3(e);
        }
        for (int ks = 0; ks < 2; ks++)
            for (int t = 0; t < NDT; t++) acc[t] = mfma_split3(tl.col(tile, 1, ks, t), pf[ks], acc[t]);
        for (int ks = 0; ks < 2; ks++) {
            float d[8];
            for (int j4 = 0; j4 < 2; j4++) {
                const f32x4 Dl = *(const f32x4*)&sld[buf][1][ws * 32 + 16 * ks + 8 * j4 + 4 * g];
                for (int j = 0; j < 4; j++) {
                    const int r = 8 * ks + 4 * j4 + j;
                    d[4 * j4 + j] = s[r] * (dp[r] - Dl[j]);
                }
            }
            df[ks] = split3(d);
        }
        for (int ks = 0; ks < 2; ks++)
            for (int t = 0; t < NDT; t++)
                acc[NDT + t] = mfma_split3(tl.col(tile, 0, ks, t), df[ks], acc[NDT + t]);
        if constexpr (INNER) stage();
    };
    // The same step with each product's MFMAs and the VALU work that may run
    // beside them interleaved by hand: S with the next stage's splits, dP with
    // P, dV with dS, then dK. For D = 128, where one wave per SIMD has no other
    // to fill its VALU stretches (same box: 32 x 2048 x 2048 768 -> 667 us);
    // at D = 64 the VALU work does not fit beside half as many MFMAs and the
    // compiler's order is faster (96 x 1024 x 1024: 316 against 290 us). One
    // tile per stage (NS = 1).
    auto step_sched = [&](int st, int buf) {
        // Causal: a wave whose keys all lie past the tile works on P = 0; it
        // would wait for the others at the stage's end.
        const int q0 = st * BQ;
        char* tile = smem + buf * STAGE;
        const int thr = CAUSAL && q0 < kw + 31 ? kj - q0 - 4 * g : -1;
        f32x16 s = f32x16{}, dp = f32x16{};
        f32x4 L[4], Dl[4];
        // Operand pieces of a 16-row or 16-element group, two groups in turn.
        bf16x8 opr[2][3];
        constexpr int NR = 6 * NKS, NC = 12 * NDT;  // MFMAs of a row and of a column product
        auto fetch_row = [&](auto W, auto K, auto P) {
            constexpr int ks = decltype(K)::value;
            opr[ks & 1][decltype(P)::value] = tl.rowp(tile, decltype(W)::value, decltype(P)::value, ks);
        };
        auto fetch_col = [&](auto W, auto G, auto P) {
            constexpr int gi = decltype(G)::value;
            opr[gi & 1][decltype(P)::value] =
                tl.colp(tile, decltype(W)::value, decltype(P)::value, gi / NDT, gi % NDT);
        };
        using std::integral_constant;
        // Slot e of a product over groups of six MFMAs: fetches of the next
        // group's pieces l, h, m sit in slots 0, 2, 4 of the group.
        auto fetch_next = [&](auto E, auto NG, auto fetch) {
            constexpr int e = decltype(E)::value, grp = e / 6, c = e % 6;
            if constexpr (c % 2 == 0 && grp + 1 < decltype(NG)::value) {
                constexpr int pc = c == 0 ? 2 : (c == 2 ? 0 : 1);
                fetch(integral_constant<int, grp + 1>{}, integral_constant<int, pc>{});
            }
        };
        auto first = [&](auto fetch) {
            static_for<3>([&](auto P) { fetch(integral_constant<int, 0>{}, P); });
        };
        auto row_q = [&](auto K, auto P) { fetch_row(integral_constant<int, 0>{}, K, P); };
        auto row_o = [&](auto K, auto P) { fetch_row(integral_constant<int, 1>{}, K, P); };
        auto col_o = [&](auto G, auto P) { fetch_col(integral_constant<int, 1>{}, G, P); };
        auto col_q = [&](auto G, auto P) { fetch_col(integral_constant<int, 0>{}, G, P); };

        // ---- S, and the next stage's splits (pair k of the thread's chunks:
        // chunk k / 8, tensor (k / 4) % 2, elements 2 (k % 4) and the next) ----
        constexpr int CH = SplitStage<D, NS>::CH, NP = 8 * CH;
        PairSplit sp[NP];
        auto stage_uop = [&](auto U) {
            constexpr int i = decltype(U)::value / 3, j = decltype(U)::value % 3, k = i - j;
            if constexpr (k >= 0 && k < NP) {
                constexpr int ch = k / 8, w = (k / 4) % 2, pr = k % 4;
                if constexpr (j == 0) {
                    sp[k].a = in.r[ch][w][pr >> 1][(pr & 1) * 2];
                    sp[k].b = in.r[ch][w][pr >> 1][(pr & 1) * 2 + 1];
                }
                sp[k].template step<j>();
                if constexpr (j == 2 && pr == 3) {
                    char* dst = smem + (buf ^ 1) * STAGE + (ch * 256 + tid) * 16;
                    for (int q = 0; q < 3; q++) {
                        const u32x4 v = {sp[k - 3].w[q], sp[k - 2].w[q], sp[k - 1].w[q], sp[k].w[q]};
                        *(u32x4*)(dst + (3 * w + q) * SplitTile<D>::PB) = v;
                    }
                }
            }
        };
        first(row_q);
        mfma_slots<NR, 3 * (NP + 2)>(
            [&](auto E) {
                constexpr int e = decltype(E)::value, ks = e / 6, c = e % 6;
                fetch_next(E, integral_constant<int, NKS>{}, row_q);
                if constexpr (e < 4) L[e] = *(const f32x4*)&sld[buf][0][8 * e + 4 * g];
                s = mfma_bf16(opr[ks & 1][kSplitA[c]], piece(kf[ks], kSplitB[c]), s);
            },
            stage_uop);
        if (tid < BQ) {
            sld[buf ^ 1][0][tid] = rl;
            sld[buf ^ 1][1][tid] = rd;
        }
        gload(st + 2);

        // ---- dP, and P (pair k: registers 2k, 2k + 1) ----
        PairSplit pp[8];
        float e16[16];
        auto p_uop = [&](auto U) {
            constexpr int i = decltype(U)::value / 4, j = decltype(U)::value % 4, k = i - j;
            if constexpr (k >= 0 && k < 8) {
                if constexpr (j == 0) {
                    for (int z = 0; z < 2; z++) {
                        const int r = 2 * k + z;
                        const float pv = fast_exp2(__builtin_fmaf(s[r], c2, -L[r >> 2][r & 3]));
                        e16[r] = CAUSAL && 8 * (r >> 2) + (r & 3) < thr ? 0.f : pv;
                        pin(e16[r]);
                    }
                    pp[k].a = e16[2 * k];
                    pp[k].b = e16[2 * k + 1];
                } else {
                    pp[k].template step<j - 1>();
                }
            }
        };
        first(row_o);
        mfma_slots<NR, 4 * 11>(
            [&](auto E) {
                constexpr int e = decltype(E)::value, ks = e / 6, c = e % 6;
                fetch_next(E, integral_constant<int, NKS>{}, row_o);
                if constexpr (e < 4) Dl[e] = *(const f32x4*)&sld[buf][1][8 * e + 4 * g];
                dp = mfma_bf16(opr[ks & 1][kSplitA[c]], piece(vf[ks], kSplitB[c]), dp);
            },
            p_uop);
        bf16x8x3 pf[2], df[2];
        auto gather = [&](const PairSplit* x, bf16x8x3* f) {
            for (int ks = 0; ks < 2; ks++) {
                u32x4 v[3];
                for (int q = 0; q < 3; q++)
                    for (int z = 0; z < 4; z++) v[q][z] = x[4 * ks + z].w[q];
                f[ks] = {__builtin_bit_cast(bf16x8, v[0]), __builtin_bit_cast(bf16x8, v[1]),
                         __builtin_bit_cast(bf16x8, v[2])};
            }
        };
        gather(pp, pf);

        // ---- dV, and dS ----
        PairSplit ds[8];
        auto d_uop = [&](auto U) {
            constexpr int i = decltype(U)::value / 4, j = decltype(U)::value % 4, k = i - j;
            if constexpr (k >= 0 && k < 8) {
                if constexpr (j == 0) {
                    ds[k].a = e16[2 * k] * (dp[2 * k] - Dl[k >> 1][(2 * k) & 3]);
                    ds[k].b = e16[2 * k + 1] * (dp[2 * k + 1] - Dl[k >> 1][(2 * k + 1) & 3]);
                    pin(ds[k].a);
                    pin(ds[k].b);
                } else {
                    ds[k].template step<j - 1>();
                }
            }
        };
        first(col_o);
        mfma_slots<NC, 4 * 11>(
            [&](auto E) {
                constexpr int e = decltype(E)::value, gi = e / 6, c = e % 6, ks = gi / NDT, t = gi % NDT;
                fetch_next(E, integral_constant<int, 2 * NDT>{}, col_o);
                acc[t] = mfma_bf16(opr[gi & 1][kSplitA[c]], piece(pf[ks], kSplitB[c]), acc[t]);
            },
            d_uop);
        gather(ds, df);

        // ---- dK ----
        first(col_q);
        mfma_slots<NC, 0>(
            [&](auto E) {
                constexpr int e = decltype(E)::value, gi = e / 6, c = e % 6, ks = gi / NDT, t = gi % NDT;
                fetch_next(E, integral_constant<int, 2 * NDT>{}, col_q);
                acc[NDT + t] = mfma_bf16(opr[gi & 1][kSplitA[c]], piece(df[ks], kSplitB[c]), acc[NDT + t]);
            },
            [](auto) {});
    };
    sstore(st0, 0);
    __syncthreads();
    constexpr bool SCHED = INNER && !MASK && D == 128 && NS == 1;
    if constexpr (SCHED) {
        gload(st0 + 1);
        for (int st = st0; st < st1; st++) {
            step_sched(st, (st - st0) & 1);
            __syncthreads();
        }
    }
    for (int st = st0; !SCHED && st < st1; st++) {
        // The stage past the last is loaded (clamped rows) and never read.
        const int buf = NBUF == 2 ? (st - st0) & 1 : 0;
        gload(st + 1);
        compute(st, buf, [&] { sstore(st + 1, buf ^ 1); });
        if constexpr (NBUF == 1) __syncthreads();
        if constexpr (!INNER) sstore(st + 1, NBUF == 2 ? buf ^ 1 : 0);
        __syncthreads();
    }
    const int left = (S - st0 * BQ + 31) / 32;  // tiles of this block
    if (!merge_stream<2 * NDT, WB, NS>(acc, smem, wb, ws, lane, left < NS ? left : NS)) return;

    const bool live = kj < Skv;  // a padded key of a partial block: zeros
    {
        SplitCheck chk;
        for (int t = 0; t < 2 * NDT; t++)
            for (int r = 0; r < 16; r++) chk.add(acc[t][r]);
        if (__builtin_amdgcn_ballot_w64(chk.plain() && live))
            dkdv_f32_plain<D, CAUSAL>(p, bh, kw, acc, acc + NDT);
    }
    if (kj < Sk) {
        const float sc = p.scale;
        float* dkr = p.dk + ((size_t)bh * Sk + kj) * D;
        float* dvr = p.dv + ((size_t)bh * Sk + kj) * D;
        for (int t = 0; t < NDT; t++)
            for (int rq4 = 0; rq4 < 4; rq4++) {
                f32x4 a, b;
                for (int i = 0; i < 4; i++) {
                    a[i] = live ? acc[NDT + t][rq4 * 4 + i] * sc : 0.f;
                    b[i] = live ? acc[t][rq4 * 4 + i] : 0.f;
                }
                *(f32x4*)(dkr + t * 32 + rq4 * 8 + g * 4) = a;
                *(f32x4*)(dvr + t * 32 + rq4 * 8 + g * 4) = b;
            }
    }
}

template <int D, bool C, int WB, int NBUF, int OCC>
static void launch_dkdv(const BwdParams& p, hipStream_t s) {
    const dim3 grid((p.Sk + WB * 32 - 1) / (WB * 32) * p.BH);
    if (p.mask) bwd_dkdv_f32_kernel<D, C, true, WB, NBUF, OCC><<<grid, 256, 0, s>>>(p);
    else bwd_dkdv_f32_kernel<D, C, false, WB, NBUF, OCC><<<grid, 256, 0, s>>>(p);
}
// Keys per workgroup: 128 read and split each Q and dO element least often;
// fewer keys (stream waves instead of block waves) where 128 would leave CUs
// without a workgroup, or a causal grid with few long ones. Measured (us, keys
// per workgroup 128 / 64 / 32, 1024 x 1024 unless noted), one line per side of
// each bound:
//   D 64 full    16 x 512   43 / 38 / 29       16    78 / 67 / 81     48  160 / 190 / 222
//   D 64 causal  16   85 / 67 / 54             48 x 512   49 / 59 / 60
//   D 128 full   16   145 / 121                48 x 512   87 / 131
//   D 128 causal 16   138 / 115                48 x 512   79 / 101
// With 128 keys and D = 64 one wave per SIMD (no spills, the next stage
// split beside the dK products) is as fast as two in full grids and faster in
// small causal ones (16 x 4096: 382 against 539); in large causal ones two
// waves hide the skipped tiles better, 16 to 18 spilled registers included (192
// x 2048: 1306 -> 1159). The masked causal 128-key kernel of D = 128 spills about
// 50 and serves up to 128 keys only (backward of 768 x 128 x 128: 363 us, 415 on
// the fp32 instruction).
template <int D, bool C>
static void launch_dkdv_keys(const BwdParams& p, hipStream_t s) {
    const long long cus = device_cus();
    const long long b32 = (long long)((p.Sk + 31) / 32) * p.BH;
    const long long b64 = (long long)((p.Sk + 63) / 64) * p.BH;
    const long long b128 = (long long)((p.Sk + 127) / 128) * p.BH;
    const bool uneven = C && p.Sk > 128;
    if constexpr (D == 64) {
        if (b32 <= (uneven ? 2 : 1) * cus) launch_dkdv<D, C, 1, 1, 1>(p, s);
        else if (b64 <= cus) launch_dkdv<D, C, 2, 2, 1>(p, s);
        else {
            if constexpr (C)
                if (uneven && b128 > 2 * cus) return launch_dkdv<D, C, 4, 2, 2>(p, s);
            launch_dkdv<D, C, 4, 2, 1>(p, s);
        }
    } else {
        // With an additive mask the 128-key step is the compiler's.
        if (b64 <= cus || (p.mask && uneven)) launch_dkdv<D, C, 2, 1, 1>(p, s);
        else launch_dkdv<D, C, 4, 2, 1>(p, s);
    }
}

hipError_t launch_bwd_dkdv_f32(const BwdParams& p, int D, int causal, hipStream_t s) {
    if (D == 64) {
        if (causal) launch_dkdv_keys<64, true>(p, s);
        else launch_dkdv_keys<64, false>(p, s);
    } else if (D == 128) {
        if (causal) launch_dkdv_keys<128, true>(p, s);
        else launch_dkdv_keys<128, false>(p, s);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace gonn
