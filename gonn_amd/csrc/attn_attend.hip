// attn_attend.hip -- causal multi-token attend over the bf16 KV cache.
//
// T new queries per (b,h) whose own K/V rows are the last T cached positions
// of their sequence (chunked prefill into a cache, several tokens of one
// decoding step). Query t sees keys [0, lim_t), lim_t = kv_len[b] - (T-1-t):
// the top-left causal mask of nn/attention.go:185-196 aligned at the
// sequence's end, which is what decoding one position at a time computes.
//
// A workgroup is 4 wave64s: WQ along the queries (32 rows each) and WK = 4 /
// WQ along the keys. It takes one split of its rows' key range [0, lim of the
// last row); a stage of WK sub-tiles of 32 keys is loaded straight into LDS
// (buffer_load ... lds, one stage ahead) and shared by the query waves. The
// cache holds bf16, so K and V are exact operands as they lie; the fp32 q and
// P keep their accuracy as three bf16 pieces each (split3): three products per
// term on the bf16 matrix cores. S^T = K q^T gives each lane one query; P
// feeds O^T += V^T P^T from registers, V^T read from the row-major tile with
// ds_read_b64_tr_b16. Key waves merge through LDS; with more than one split
// the partial (m, l, o) go to the combine kernel, otherwise O is written.
//
// Bound: with many queries the matrix cores (three bf16 products per term: 82
// us at the rate they sustain on random data for B 4, H 32, T 256, D 128 over
// 2048 to 4096 cached positions), with up to 32 the cache stream. That chunk
// took 1720 to 2000 us in the split kernel of attn_decode.hip, whose VALU dots
// read the cache once per 4 queries, and takes 140 to 166 us here (the same boxes
// in turn; matrix pipe busy 0.31 of the cycles); T 8 over B 64, H 32, up to 8192
// positions 1855 -> 941 us (5.2 TB/s). Non-temporal loads are slower (1385 against
// 1100 us there, before slices were dealt over the XCDs: a load instruction fills
// 64-byte pieces of 16 rows, so a line is read by two instructions). 128 rows per
// workgroup were as fast as 64 but make longer sums (error 2.7e-7 against 2.2e-7,
// the VALU kernel's 2.4e-7).
#include "attn_f32_split.h"

namespace gonn {

namespace {

// q and o need no alignment beyond a float's (the loads are 16 bytes all the same).
typedef f32x4 f32x4u __attribute__((aligned(4)));

// The wave's 32 rows over keys [k0, k1) on the fp32 matrix cores, for workgroups
// with a result that is not finite (an infinite operand has no three-piece split).
// Tiles that some row does not see in full (keys from lim0, the wave's least
// lim, or from k1) add P V with a select per key: a masked key's weight of 0
// would make NaN of an infinite V. 128 slices of 4096 keys, D 128 with one
// infinite V each take 1112 us with T 256 (215 on ordinary data) and 222 with T 8
// (63); one key wave alone 1811 and 657; the VALU kernel 2277 and 118 on any data.
template <int D>
GONN_DEV void attend_plain(const float* qrow, float sg, const bf16* Kg, const bf16* Vg, int k0,
                           int k1, int lim0, int lim, f32x16* oacc, float& m, float& l) {
    constexpr int HD = D / 2, NDT = D / 32;
    typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63, g = lane >> 5, ln = lane & 31;
    const uint16_t* K = (const uint16_t*)Kg;
    const uint16_t* V = (const uint16_t*)Vg;
    for (int t = 0; t < NDT; t++) oacc[t] = f32x16{};
    m = -INFINITY;
    l = 0.f;
#pragma unroll 1
    for (int kb = k0; kb < k1; kb += 32) {
        const int kr = kb + ln < k1 ? kb + ln : k1 - 1;
        const uint16_t* krow = K + (size_t)kr * D + g * HD;
        f32x16 s = f32x16{};
#pragma unroll 1
        for (int i0 = 0; i0 < HD; i0 += 32) {
            u16x8 kx[4];
            f32x4 qx[8];
            for (int i = 0; i < 4; i++) kx[i] = *(const u16x8*)(krow + i0 + 8 * i);
            for (int i = 0; i < 8; i++) qx[i] = *(const f32x4u*)(qrow + g * HD + i0 + 4 * i);
            for (int i = 0; i < 32; i++)
                s = mfma_f32(bf16_to_f32(kx[i / 8][i % 8]), qx[i / 4][i % 4] * sg, s);
        }
        float mx = -INFINITY;
        for (int r = 0; r < 16; r++) {
            const int key = kb + 8 * (r >> 2) + 4 * g + (r & 3);
            if (key >= k1 || key >= lim) s[r] = -INFINITY;
            mx = fmaxf(mx, s[r]);
        }
        mx = pair_max32(mx);
        const float mnew = fmaxf(m, mx), mref = mnew == -INFINITY ? 0.f : mnew;
        const float alpha = m == -INFINITY ? 0.f : fast_exp2(m - mref);
        float rs = 0.f;
        for (int r = 0; r < 16; r++) {
            s[r] = fast_exp2(s[r] - mref);
            rs += s[r];
        }
        l = l * alpha + rs;
        m = mnew;
        for (int t = 0; t < NDT; t++) oacc[t] *= alpha;
        // s moves down as its weights are used.
        if (kb + 32 <= k1 && kb + 32 <= lim0) {
#pragma unroll 1
            for (int r4 = 0; r4 < 4; r4++) {
                for (int r = 0; r < 4; r++) {
                    const uint16_t* v = V + (size_t)(kb + 8 * r4 + 4 * g + r) * D + ln;
                    for (int t = 0; t < NDT; t++)
                        oacc[t] = mfma_f32(bf16_to_f32(v[t * 32]), s[r], oacc[t]);
                }
                for (int i = 0; i < 12; i++) s[i] = s[i + 4];
            }
            continue;
        }
        // Both halves of the wave hold the same 32 queries, 16 keys each.
#pragma unroll 1
        for (int r = 0; r < 16; r++) {
            const float other = __shfl_xor(s[0], 32);
            for (int h = 0; h < 2; h++) {
                const int key = kb + 8 * (r >> 2) + 4 * h + (r & 3);
                if (key >= k1) continue;  // uniform
                const float pv = h == g ? s[0] : other;
                for (int e = 0; e < 4 * NDT; e++) {
                    const u16x4 v = *(const u16x4*)(V + (size_t)key * D + e * 8 + 4 * g);
                    for (int j = 0; j < 4; j++) {
                        const int i = (e % 4) * 4 + j;
                        const float o = oacc[e / 4][i];
                        oacc[e / 4][i] = key < lim ? __builtin_fmaf(pv, bf16_to_f32(v[j]), o) : o;
                    }
                }
            }
            for (int i = 0; i < 15; i++) s[i] = s[i + 1];
        }
    }
    l = pair_sum32(l);
}

}  // namespace

template <int D, int WQ>
__global__ __launch_bounds__(256, (D == 128 && WQ == 1) ? 1 : 2) void attend_causal_kernel(
    DecodeParams p) {
    constexpr int WK = 4 / WQ, BM = WQ * 32, BN = WK * 32;
    constexpr int NKS = D / 16, NDT = D / 32;
    constexpr uint32_t PB = 32 * D * 2;       // bytes of one sub-tile of K (or V)
    constexpr uint32_t STAGE = 2 * WK * PB;   // K sub-tiles, then V sub-tiles
    constexpr int NLD = WK * PB / 16 / 256;   // load instructions per wave (each of K, V)
    __shared__ __attribute__((aligned(16))) char smem[2 * STAGE];
    __shared__ int again;  // some row's result is not finite

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wq = wave % WQ, wk = wave / WQ;
    const int g = lane >> 5, ln = lane & 31;
    const int T = p.T, nqb = (T + BM - 1) / BM;
    // Slice-splits are dealt over the XCDs, all first splits before the second
    // ones (which short sequences do not have), longest rows of each first.
    int us, qb;
    map_block(blockIdx.x, nqb, p.B * p.H * p.nsplit, true, us, qb, 1, true);
    const int sp = __builtin_amdgcn_readfirstlane(us / (p.B * p.H));
    const int bh = us - sp * (p.B * p.H);
    const int b = bh / p.H;
    int len = p.kv_len[b];
    len = __builtin_amdgcn_readfirstlane(len < 0 ? 0 : (len > p.Lmax ? p.Lmax : len));
    const int t0 = qb * BM, tl0 = t0 + BM < T ? t0 + BM : T;  // rows t0 .. tl0 - 1
    const int kmax = causal_group_keys(len, T, tl0 - 1);
    const int ns = kmax > 0 ? (kmax + p.split_keys - 1) / p.split_keys : 0;
    if (sp >= ns) return;  // uniform for the workgroup
    const int k0 = (int)((long long)sp * kmax / ns);
    const int k1 = (int)((long long)(sp + 1) * kmax / ns);
    const int tw = t0 + wq * 32, ti = tw + ln;  // this wave's first row, this lane's
    const int lim = causal_group_keys(len, T, ti < T ? ti : T - 1);
    const bf16* Kg = (const bf16*)p.kc + (size_t)bh * p.Lmax * D;
    const bf16* Vg = (const bf16*)p.vc + (size_t)bh * p.Lmax * D;
    const int nst = (k1 - k0 + BN - 1) / BN;

    // Loads: 16-byte position i * 256 + tid of the stage's K (V) sub-tiles;
    // rows past k1 - 1 are clamped to it (masked below).
    const uint32_t bytes = (uint32_t)(k1 - k0) * D * 2;
    const brsrc krs = make_rsrc(Kg + (size_t)k0 * D, bytes);
    const brsrc vrs = make_rsrc(Vg + (size_t)k0 * D, bytes);
    int lrow[NLD];
    uint32_t lcol[NLD];
    for (int i = 0; i < NLD; i++) {
        constexpr int NCH = PB / 16;
        const int pos = i * 256 + tid;
        int r, c;
        slab_chunk(pos % NCH, 32, r, c);
        lrow[i] = pos / NCH * 32 + r;
        lcol[i] = (uint32_t)c * 16;
    }
    const uint32_t lb = lds_addr(smem) + wave * 1024;
    auto load = [&](int st, int buf) {
        for (int i = 0; i < NLD; i++) {
            int r = st * BN + lrow[i];
            r = r < k1 - k0 ? r : k1 - k0 - 1;
            const uint32_t vo = (uint32_t)r * (D * 2) + lcol[i];
            const uint32_t dst = lb + buf * STAGE + i * 4096;
            dma16(krs, dst, vo, 0);
            dma16(vrs, dst + WK * PB, vo, 0);
        }
    };
    load(0, 0);
    if (tid == 0) again = 0;

    // q pieces: q[ti][16 ks + 8 g .. +7] * scale log2 e.
    const float* qrow = (const float*)p.q + ((size_t)bh * T + (ti < T ? ti : T - 1)) * D;
    const float sg = ti < T ? p.scale_log2 : 0.f;
    bf16x8x3 qf[NKS];
    for (int ks = 0; ks < NKS; ks++) {
        const f32x4 a = *(const f32x4u*)(qrow + ks * 16 + g * 8);
        const f32x4 c = *(const f32x4u*)(qrow + ks * 16 + g * 8 + 4);
        float x[8];
        for (int e = 0; e < 4; e++) {
            x[e] = a[e] * sg;
            x[4 + e] = c[e] * sg;
        }
        qf[ks] = split3(x);
    }
    SplitTile<D> tl;
    tl.init(lane);

    f32x16 oacc[NDT];
    for (int t = 0; t < NDT; t++) oacc[t] = f32x16{};
    float m = -INFINITY, l = 0.f;
    const int limw0 = causal_group_keys(len, T, tw);                          // of the wave's first row
    const int limw1 = causal_group_keys(len, T, tw + 31 < T ? tw + 31 : T - 1);  // and its last

    auto compute = [&](int st, int buf) {
        const int kbase = k0 + st * BN + wk * 32;
        if (tw >= T || kbase >= k1 || kbase >= limw1) return;  // wave-uniform: no pair here
        char* kt = smem + buf * STAGE + wk * PB;
        char* vt = kt + WK * PB;
        // The small pieces' products in a sum of their own, so that each score
        // takes NKS + 1 roundings of its own size.
        f32x16 s = f32x16{}, s2 = f32x16{};
        for (int ks = 0; ks < NKS; ks++) {
            const bf16x8 k = tl.row1(kt, ks);
            s2 = mfma_bf16(k, qf[ks].l, s2);
            s2 = mfma_bf16(k, qf[ks].m, s2);
            s = mfma_bf16(k, qf[ks].h, s);
        }
        for (int r = 0; r < 16; r++) s[r] += s2[r];
        if (kbase + 32 > k1 || kbase + 32 > limw0) {
            const int thr = (lim < k1 ? lim : k1) - 1 - (kbase + 4 * g);
            for (int r = 0; r < 16; r++) s[r] = 8 * (r >> 2) + (r & 3) > thr ? -INFINITY : s[r];
        }
        float mx = fmaxf(s[0], s[1]);
        for (int r = 2; r < 16; r++) mx = fmaxf(mx, s[r]);
        mx = pair_max32(mx);
        // The offset moves by more than 2^8 at a time (P stays below 2^8).
        const bool need = mx > m && (m == -INFINITY || mx - m > 8.f);
        if (__builtin_amdgcn_ballot_w64(need)) {
            const float mn = need ? mx : m;
            const float alpha = m == -INFINITY ? 0.f : fast_exp2(m - mn);
            m = mn;
            l *= alpha;
            for (int t = 0; t < NDT; t++) oacc[t] *= alpha;
        }
        const float mref = m == -INFINITY ? 0.f : m;
        float rs[4] = {0.f, 0.f, 0.f, 0.f};
        bf16x8x3 pf[2];
        for (int ks = 0; ks < 2; ks++) {
            float e[8];
            for (int j = 0; j < 8; j++) {
                e[j] = fast_exp2(s[8 * ks + j] - mref);
                rs[j & 3] += e[j];
            }
            pf[ks] = split3(e);
        }
        l += (rs[0] + rs[1]) + (rs[2] + rs[3]);
        // Each tile's V^T P^T on its own, added once: one rounding of O's size
        // per 32 keys instead of six.
        for (int t = 0; t < NDT; t++) {
            f32x16 x = f32x16{};
            const bf16x8 v0 = tl.col1(vt, 0, t), v1 = tl.col1(vt, 1, t);
            x = mfma_bf16(v0, pf[0].l, x);
            x = mfma_bf16(v1, pf[1].l, x);
            x = mfma_bf16(v0, pf[0].m, x);
            x = mfma_bf16(v1, pf[1].m, x);
            x = mfma_bf16(v0, pf[0].h, x);
            x = mfma_bf16(v1, pf[1].h, x);
            for (int r = 0; r < 16; r++) oacc[t][r] += x[r];
        }
    };
    for (int st = 0; st < nst; st++) {
        GONN_VMCNT(0);
        __syncthreads();  // stage st has landed, and its buffer's last reader is past it
        if (st + 1 < nst) load(st + 1, (st + 1) & 1);
        compute(st, st & 1);
    }

    // Key waves > 0 leave (o, m, l) in LDS, key wave 0 merges in order.
    auto merge = [&](float& l) {
        constexpr int NE = 16 * NDT + 2;
        static_assert((WK - 1) * WQ * NE * 256 <= 2 * (int)STAGE, "the merge fits in the stages");
        __syncthreads();  // every wave is past its last tile
        float* red = (float*)smem;
        if (wk > 0) {
            float* d = red + ((wk - 1) * WQ + wq) * NE * 64 + lane;
            for (int t = 0; t < NDT; t++)
                for (int r = 0; r < 16; r++) d[(t * 16 + r) * 64] = oacc[t][r];
            d[(NE - 2) * 64] = m;
            d[(NE - 1) * 64] = l;
        }
        __syncthreads();
        if (wk > 0) return;
        for (int w = 1; w < WK; w++) {
            const float* d = red + ((w - 1) * WQ + wq) * NE * 64 + lane;
            const float m2 = d[(NE - 2) * 64], l2 = d[(NE - 1) * 64];
            const float M = fmaxf(m, m2), Mr = M == -INFINITY ? 0.f : M;
            const float a = fast_exp2(m - Mr), c = fast_exp2(m2 - Mr);
            l = l * a + l2 * c;
            for (int t = 0; t < NDT; t++)
                for (int r = 0; r < 16; r++) oacc[t][r] = oacc[t][r] * a + d[(t * 16 + r) * 64] * c;
            m = M;
        }
    };
    float lt = pair_sum32(l);
    merge(lt);
    if (wk == 0) {
        bool bad = nonfinite(lt);
        for (int t = 0; t < NDT; t++)
            for (int r = 0; r < 16; r++) bad |= nonfinite(oacc[t][r]);
        if (__builtin_amdgcn_ballot_w64(bad && ti < T) && lane == 0) again = 1;
    }
    __syncthreads();
    if (again) {  // uniform: all rows once more, a share of the keys to each key wave
        const int share = (k1 - k0 + BN - 1) / BN * 32, ks = k0 + wk * share;
        const int end = k1 < limw1 ? k1 : limw1;
        attend_plain<D>(qrow, sg, Kg, Vg, ks, ks + share < end ? ks + share : end, limw0, lim, oacc,
                        m, lt);
        merge(lt);
    }
    if (wk > 0 || ti >= T) return;
    const size_t row = (size_t)bh * T + ti;
    float* orow = p.nsplit == 1 ? p.o + row * D : p.part_o + (row * p.nsplit + sp) * D;
    // Every query sees at least its own key; one with none in this split
    // leaves (m, l, o) = (-inf, 0, 0). A query whose keys all score -inf
    // has l = 0: O = 0, as the combine kernel writes it.
    const float inv = p.nsplit == 1 ? (lt == 0.f ? 0.f : 1.f / lt) : 1.f;
    for (int t = 0; t < NDT; t++)
        for (int rq = 0; rq < 4; rq++) {
            f32x4 v;
            for (int i = 0; i < 4; i++) v[i] = oacc[t][rq * 4 + i] * inv;
            *(f32x4u*)(orow + t * 32 + rq * 8 + g * 4) = v;
        }
    if (p.nsplit > 1 && g == 0) {
        // A NaN query has no maximum; a finite one keeps its weight non-zero.
        p.part_ml[(row * p.nsplit + sp) * 2 + 0] = lt != lt ? 0.f : m;
        p.part_ml[(row * p.nsplit + sp) * 2 + 1] = lt;
    }
}

hipError_t launch_attend_causal(const DecodeParams& p, int D, hipStream_t s) {
    if (p.T <= 0 || p.nsplit <= 0 || (p.group != 32 && p.group != 64)) return hipErrorInvalidValue;
    const unsigned grid = (unsigned)((p.T + p.group - 1) / p.group) * (unsigned)p.nsplit *
                          (unsigned)(p.B * p.H);
    if (D == 128) {
        if (p.group == 32) attend_causal_kernel<128, 1><<<grid, 256, 0, s>>>(p);
        else attend_causal_kernel<128, 2><<<grid, 256, 0, s>>>(p);
    } else if (D == 64) {
        if (p.group == 32) attend_causal_kernel<64, 1><<<grid, 256, 0, s>>>(p);
        else attend_causal_kernel<64, 2><<<grid, 256, 0, s>>>(p);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace gonn
