// attn_bwd_dq_f32.hip -- the fp32 mode's dQ (see attn_bwd_f32.hip). Its own
// file for its MFMA flag: with VGPR accumulators (which the softmax VALU
// reads) the compiler-ordered step runs 198 against 210 us at 96 x 1024 x
// 1024, D = 64 (the hand-ordered one of D = 128 runs the same either way);
// dK/dV, whose long-lived fragments then leave the AGPRs, 334 against 282 us.
#include "attn_f32_split.h"

namespace gonn {

// Plain fp32 products for blocks outside the split's range (see dkdv_f32_plain).
template <int D, bool CAUSAL>
GONN_DEV void dq_f32_plain(const BwdParams& p, int bh, int qw, int Skv, f32x16* dqacc) {
    constexpr int HD = D / 2, NDT = D / 32;
    const int lane = threadIdx.x & 63, g = lane >> 5, ln = lane & 31, qi = qw + ln;
    const int S = p.S, Sk = p.Sk, qr = qi < S ? qi : S - 1;
    const float* qp = (const float*)p.q + ((size_t)bh * S + qr) * D + g * HD;
    const float* op = (const float*)p.dO + ((size_t)bh * S + qr) * D + g * HD;
    const float* Kg = (const float*)p.k + (size_t)bh * Sk * D;
    const float* Vg = (const float*)p.v + (size_t)bh * Sk * D;
    const float lq = p.lse2[(size_t)bh * p.Sp + qi], dl = p.delta[(size_t)bh * p.Sp + qi];
    const float* mrow = p.mask ? mask_slice(p, bh) + (size_t)qr * Sk : nullptr;
    const int kend = CAUSAL && qw + 32 < Skv ? qw + 32 : Skv;
    for (int t = 0; t < NDT; t++) dqacc[t] = f32x16{};
#pragma unroll 1
    for (int kb = 0; kb < kend; kb += 32) {
        const int kr = kb + ln < Skv ? kb + ln : Skv - 1;
        f32x16 s = f32x16{}, dp = f32x16{};
        const float *kp = Kg + (size_t)kr * D + g * HD, *vp = Vg + (size_t)kr * D + g * HD;
#pragma unroll 1
        for (int i0 = 0; i0 < HD; i0 += 16) plain_pair16(s, dp, kp + i0, qp + i0, vp + i0, op + i0);
        for (int r = 0; r < 16; r++) {
            const int key = kb + 8 * (r >> 2) + 4 * g + (r & 3);
            float off = -lq;
            if (mrow && key < Skv) off += mrow[key] * kLog2e;
            float pv = fast_exp2(__builtin_fmaf(s[r], p.scale_log2, off));
            if (key >= Skv || (CAUSAL && key > qi)) pv = 0.f;
            dp[r] = pv * (dp[r] - dl);
        }
        for (int r = 0; r < 16; r++) {
            int key = kb + 8 * (r >> 2) + 4 * g + (r & 3);
            key = key < Skv ? key : Skv - 1;
            for (int t = 0; t < NDT; t++)
                dqacc[t] = mfma_f32(Kg[(size_t)key * D + t * 32 + ln], dp[r], dqacc[t]);
        }
    }
}

template <int D, bool CAUSAL, bool MASK, int WB, int NBUF, int OCC>
__global__ __launch_bounds__(256, OCC) void bwd_dq_f32_kernel(BwdParams p) {
    constexpr int NS = 4 / WB, BM = WB * 32, BN = NS * 32;  // queries per block, keys per stage
    constexpr int NKS = D / 16, NDT = D / 32;
    constexpr uint32_t STAGE = NS * SplitTile<D>::BYTES;
    __shared__ __attribute__((aligned(16))) char smem[NBUF * STAGE];
    static_assert((NS - 1) * WB * NDT * 4096 <= NBUF * (int)STAGE, "the merge fits");

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wb = wave % WB, ws = wave / WB;
    const int g = lane >> 5, ln = lane & 31;
    const int S = p.S, Sk = p.Sk;  // S queries, Sk keys
    int bh, qb;
    map_block(blockIdx.x, (S + BM - 1) / BM, p.BH, CAUSAL, bh, qb, 1, deal_slices(p));
    const int q0 = qb * BM, qw = q0 + wb * 32, qi = qw + ln;
    const int Skv = bwd_keys(p, bh);  // keys taking part (key padding)
    if (Skv == 0) {
        bwd_zero_rows<D>(p.dq, S, bh, q0, BM);
        return;
    }
    const int kend = CAUSAL && q0 + BM < Skv ? q0 + BM : Skv;
    const int nst = (kend + BN - 1) / BN;
    const float* Kg = (const float*)p.k + (size_t)bh * Sk * D;
    const float* Vg = (const float*)p.v + (size_t)bh * Sk * D;

    SplitStage<D, NS> in;
    in.init(tid);
    in.load(Kg, Vg, 0, kend);
    const int qr = qi < S ? qi : S - 1;  // pad queries have lse2 = +inf: P = 0
    bf16x8x3 qf[NKS], of[NKS];
    load_row_split<D>((const float*)p.q + ((size_t)bh * S + qr) * D, g, qf);
    load_row_split<D>((const float*)p.dO + ((size_t)bh * S + qr) * D, g, of);
    const float lq = p.lse2[(size_t)bh * p.Sp + qi];
    const float dl = p.delta[(size_t)bh * p.Sp + qi];
    const float* mrow = nullptr;  // the additive mask's row of this lane's query
    if constexpr (MASK) mrow = mask_slice(p, bh) + (size_t)qr * Sk;
    SplitTile<D> tl;
    tl.init(lane);

    f32x16 acc[NDT];
    for (int t = 0; t < NDT; t++) acc[t] = f32x16{};
    const float c2 = p.scale_log2;

    auto compute = [&](int st, int buf) {
        const int kbase = st * BN + ws * 32;
        if (kbase >= kend || (CAUSAL && kbase > qw + 31)) return;  // wave-uniform: no pair here
        char* tile = smem + buf * STAGE + ws * SplitTile<D>::BYTES;
        f32x16 s = f32x16{}, dp = f32x16{};
        for (int ks = 0; ks < NKS; ks++) {
            s = mfma_split3(tl.row(tile, 0, ks), qf[ks], s);
            dp = mfma_split3(tl.row(tile, 1, ks), of[ks], dp);
        }
        const bool need_mask = (kbase + 32 > Skv) || (CAUSAL && kbase + 31 > qw);
        bf16x8x3 df[2];
        for (int ks = 0; ks < 2; ks++) {
            float d[8];
            for (int j = 0; j < 8; j++) {
                const int r = 8 * ks + j, key = kbase + 8 * (r >> 2) + 4 * g + (r & 3);
                float off = -lq;  // log2 units: s scale log2e + m log2e - L log2e
                if constexpr (MASK)
                    if (key < Skv) off += mrow[key] * kLog2e;
                float pv = fast_exp2(__builtin_fmaf(s[r], c2, off));
                if (need_mask) pv = key >= Skv || (CAUSAL && key > qi) ? 0.f : pv;
                d[j] = pv * (dp[r] - dl);
            }
            df[ks] = split3(d);
        }
        for (int ks = 0; ks < 2; ks++)
            for (int t = 0; t < NDT; t++)
                acc[t] = mfma_split3(tl.col(tile, 0, ks, t), df[ks], acc[t]);
    };
    // The same step with the MFMAs and the VALU work that may run beside them
    // interleaved by hand (as in bwd_dkdv_f32_kernel): S with the next stage's
    // splits, dP with P, then dS, its second half beside dQ's first (same box:
    // 32 x 2048 x 2048, D 128: 583 -> 516 us).
    auto step_sched = [&](int st, int buf) {
        const int kbase = st * BN;
        char* tile = smem + buf * STAGE;
        int lim = Skv - 1;
        if (CAUSAL) lim = qi < lim ? qi : lim;
        const int thr = lim - kbase - 4 * g;  // key 8 (r / 4) + r % 4 > thr is masked
        f32x16 s = f32x16{}, dp = f32x16{};
        bf16x8 opr[2][3];
        constexpr int NR = 6 * NKS, NC = 12 * NDT;
        using std::integral_constant;
        auto row = [&](auto W, auto K, auto P) {
            constexpr int ks = decltype(K)::value;
            opr[ks & 1][decltype(P)::value] = tl.rowp(tile, decltype(W)::value, decltype(P)::value, ks);
        };
        auto row_k = [&](auto K, auto P) { row(integral_constant<int, 0>{}, K, P); };
        auto row_v = [&](auto K, auto P) { row(integral_constant<int, 1>{}, K, P); };
        auto col_k = [&](auto G, auto P) {
            constexpr int gi = decltype(G)::value;
            opr[gi & 1][decltype(P)::value] = tl.colp(tile, 0, decltype(P)::value, gi / NDT, gi % NDT);
        };
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
        first(row_k);
        mfma_slots<NR, 3 * (NP + 2)>(
            [&](auto E) {
                constexpr int e = decltype(E)::value, ks = e / 6, c = e % 6;
                fetch_next(E, integral_constant<int, NKS>{}, row_k);
                s = mfma_bf16(opr[ks & 1][kSplitA[c]], piece(qf[ks], kSplitB[c]), s);
            },
            stage_uop);
        in.load(Kg, Vg, (st + 2) * BN, kend);

        first(row_v);
        mfma_slots<NR, 16>(
            [&](auto E) {
                constexpr int e = decltype(E)::value, ks = e / 6, c = e % 6;
                fetch_next(E, integral_constant<int, NKS>{}, row_v);
                dp = mfma_bf16(opr[ks & 1][kSplitA[c]], piece(of[ks], kSplitB[c]), dp);
            },
            [&](auto U) {
                constexpr int r = decltype(U)::value;
                const float pv = fast_exp2(__builtin_fmaf(s[r], c2, -lq));
                s[r] = 8 * (r >> 2) + (r & 3) > thr ? 0.f : pv;
                pin(s[r]);
            });

        PairSplit ds[8];
        auto d_step = [&](auto K, auto J) {
            constexpr int k = decltype(K)::value, j = decltype(J)::value;
            if constexpr (j == 0) {
                ds[k].a = s[2 * k] * (dp[2 * k] - dl);
                ds[k].b = s[2 * k + 1] * (dp[2 * k + 1] - dl);
                pin(ds[k].a);
                pin(ds[k].b);
            } else {
                ds[k].template step<j - 1>();
            }
        };
        bf16x8x3 df[2];
        auto gather = [&](auto H) {
            constexpr int h = decltype(H)::value;
            u32x4 v[3];
            for (int q = 0; q < 3; q++)
                for (int z = 0; z < 4; z++) v[q][z] = ds[4 * h + z].w[q];
            df[h] = {__builtin_bit_cast(bf16x8, v[0]), __builtin_bit_cast(bf16x8, v[1]),
                     __builtin_bit_cast(bf16x8, v[2])};
        };
        first(col_k);
        static_for<4>([&](auto J) { static_for<4>([&](auto K) { d_step(K, J); }); });
        gather(integral_constant<int, 0>{});
        auto dq_slot = [&](auto E) {
            constexpr int e = decltype(E)::value, gi = e / 6, c = e % 6, ks = gi / NDT, t = gi % NDT;
            fetch_next(E, integral_constant<int, 2 * NDT>{}, col_k);
            acc[t] = mfma_bf16(opr[gi & 1][kSplitA[c]], piece(df[ks], kSplitB[c]), acc[t]);
        };
        mfma_slots<NC / 2, 16>(dq_slot, [&](auto U) {
            constexpr int u = decltype(U)::value;
            d_step(integral_constant<int, 4 + u % 4>{}, integral_constant<int, u / 4>{});
        });
        gather(integral_constant<int, 1>{});
        mfma_slots<NC / 2, 0>(
            [&](auto E) { dq_slot(integral_constant<int, NC / 2 + decltype(E)::value>{}); }, [](auto) {});
    };
    in.store(smem, tid, 0, kend);
    __syncthreads();
    constexpr bool SCHED = NBUF == 2 && OCC == 1 && !MASK && D == 128 && NS == 1;
    if constexpr (SCHED) {
        in.load(Kg, Vg, BN, kend);
        for (int st = 0; st < nst; st++) {
            step_sched(st, st & 1);
            __syncthreads();
        }
    }
    for (int st = 0; !SCHED && st < nst; st++) {
        const int buf = NBUF == 2 ? st & 1 : 0;
        if (st + 1 < nst) in.load(Kg, Vg, (st + 1) * BN, kend);
        compute(st, buf);
        if (NBUF == 1) __syncthreads();
        if (st + 1 < nst) in.store(smem + (NBUF == 2 ? buf ^ 1 : 0) * STAGE, tid, (st + 1) * BN, kend);
        __syncthreads();
    }
    const int left = (kend + 31) / 32;  // key tiles of this block
    if (!merge_stream<NDT, WB, NS>(acc, smem, wb, ws, lane, left < NS ? left : NS)) return;
    {
        SplitCheck chk;
        for (int t = 0; t < NDT; t++)
            for (int r = 0; r < 16; r++) chk.add(acc[t][r]);
        if (__builtin_amdgcn_ballot_w64(chk.plain() && qi < S)) dq_f32_plain<D, CAUSAL>(p, bh, qw, Skv, acc);
    }
    if (qi < S) {
        const float sc = p.scale;
        float* dqr = p.dq + ((size_t)bh * S + qi) * D;
        for (int t = 0; t < NDT; t++)
            for (int rq4 = 0; rq4 < 4; rq4++) {
                f32x4 a;
                for (int i = 0; i < 4; i++) a[i] = acc[t][rq4 * 4 + i] * sc;
                *(f32x4*)(dqr + t * 32 + rq4 * 8 + g * 4) = a;
            }
    }
}

template <int D, bool C, int WB, int NBUF, int OCC>
static void launch_dq(const BwdParams& p, hipStream_t s) {
    const dim3 grid((p.S + WB * 32 - 1) / (WB * 32) * p.BH);
    if (p.mask) bwd_dq_f32_kernel<D, C, true, WB, NBUF, OCC><<<grid, 256, 0, s>>>(p);
    else bwd_dq_f32_kernel<D, C, false, WB, NBUF, OCC><<<grid, 256, 0, s>>>(p);
}

// Query rows per workgroup, chosen as launch_dkdv_keys chooses keys. Measured
// (us, rows 128 / 64 / 32, 1024 x 1024 unless noted):
//   D 64 full    16 x 512  41 / 32 / 22       16   72 / 47 / 64    48 x 512  44 / 50 / 55
//   D 64 causal  16   77 / 47 / 43            16 x 2048  147 / 100 / 129
//                48  114 / 85 / 114           192 x 2048  891 / 934 / 1559
//   D 128 full   16  112 / 93                 48 x 512   67 / 100
//   D 128 causal 16  107 / 91                 48 x 512   61 / 78
template <int D, bool C>
static void launch_dq_rows(const BwdParams& p, hipStream_t s) {
    const long long cus = device_cus();
    const long long b32 = (long long)((p.S + 31) / 32) * p.BH;
    const long long b64 = (long long)((p.S + 63) / 64) * p.BH;
    const long long b128 = (long long)((p.S + 127) / 128) * p.BH;
    const bool uneven = C && p.S > 128;
    if constexpr (D == 64) {
        if (b32 <= (uneven ? 2 : 1) * cus) launch_dq<D, C, 1, 1, 1>(p, s);
        else if (b64 <= (uneven ? 2 : 1) * cus) launch_dq<D, C, 2, 2, 1>(p, s);
        else {
            if constexpr (C)
                if (uneven && b128 <= 6 * cus) return launch_dq<D, C, 2, 1, 2>(p, s);
            launch_dq<D, C, 4, 2, 2>(p, s);
        }
    } else {
        // With an additive mask the 128-row step is the compiler's.
        if (b64 <= (p.mask && uneven ? 3 : 1) * cus) launch_dq<D, C, 2, 1, 1>(p, s);
        else launch_dq<D, C, 4, 2, 1>(p, s);
    }
}

hipError_t launch_bwd_dq_f32(const BwdParams& p, int D, int causal, hipStream_t s) {
    if (D == 64) {
        if (causal) launch_dq_rows<64, true>(p, s);
        else launch_dq_rows<64, false>(p, s);
    } else if (D == 128) {
        if (causal) launch_dq_rows<128, true>(p, s);
        else launch_dq_rows<128, false>(p, s);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace gonn
