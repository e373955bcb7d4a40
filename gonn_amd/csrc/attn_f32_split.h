// attn_f32_split.h -- tiles of three-piece operands in LDS.
//
// A tile is 32 rows of two fp32 tensors as six row-major bf16 planes of 32 x D
// (three pieces each) in the slab layout of common.h: what the fp32 backward
// streams. The causal attend reads its bf16 K and V tiles, one plane each, with
// the same addressing (row1, col1).
#pragma once
#include <utility>

#include "common.h"
#include "kernels.h"

namespace gonn {

// LDS reads of one 32-row tile's planes (three of the first tensor, three of
// the second), byte offsets from the tile's start.
template <int D>
struct SplitTile {
    static constexpr uint32_t PB = 32 * D * 2, BYTES = 6 * PB;
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s4 lds_s4;
    typedef __attribute__((address_space(3))) char lds_char;
    uint32_t qa0, qa1, ta0, ta1;
    GONN_DEV void init(int lane) {
        const int g = lane >> 5, ln = lane & 31, hs = slab_swz(ln);
        qa0 = (uint32_t)(ln * 64 + ((0 + g) ^ hs) * 16);
        qa1 = (uint32_t)(ln * 64 + ((2 + g) ^ hs) * 16);
        const int s16 = lane & 15, tcx = 2 * ((ln >> 4) & 1) + ((s16 >> 1) & 1);
        ta0 = (uint32_t)((4 * g + (s16 >> 2)) * 64 + (tcx ^ g) * 16 + 8 * (s16 & 1));
        ta1 = (uint32_t)((8 + 4 * g + (s16 >> 2)) * 64 + (tcx ^ (2 + g)) * 16 + 8 * (s16 & 1));
    }
    // Row ln, elements 16 ks + 8 g .. +7 of tensor w: an operand whose lanes
    // take one row each (ds_read_b128).
    GONN_DEV bf16x8x3 row(const char* tile, int w, int ks) const {
        const char* b = tile + 3 * w * PB + (ks >> 1) * 2048 + ((ks & 1) ? qa1 : qa0);
        return {*(const bf16x8*)b, *(const bf16x8*)(b + PB), *(const bf16x8*)(b + 2 * PB)};
    }
    // One piece (0 h, 1 m, 2 l) of row() and col().
    GONN_DEV bf16x8 rowp(const char* tile, int w, int piece, int ks) const {
        return row1(tile + (3 * w + piece) * PB, ks);
    }
    GONN_DEV bf16x8 colp(char* tile, int w, int piece, int ks, int t) const {
        return col1(tile + (3 * w + piece) * PB, ks, t);
    }
    // The same from one plane (a tile of a single bf16 tensor).
    GONN_DEV bf16x8 row1(const char* plane, int ks) const {
        return *(const bf16x8*)(plane + (ks >> 1) * 2048 + ((ks & 1) ? qa1 : qa0));
    }
    // Element 32 t + ln of rows 16 ks + {4g..4g+3, 8+4g..8+4g+3}: the
    // transposed operand, in the row order an accumulator holds them.
    GONN_DEV bf16x8x3 col(char* tile, int w, int ks, int t) const {
        char* b = tile + 3 * w * PB;
        return {col1(b, ks, t), col1(b + PB, ks, t), col1(b + 2 * PB, ks, t)};
    }
    GONN_DEV bf16x8 col1(char* plane, int ks, int t) const {
        lds_char* b = (lds_char*)plane + (t * 32 + 16 * ks) * 64;
        const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(b + ta0));
        const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(b + ta1));
        const s4 b8[2] = {lo, hi};
        return __builtin_bit_cast(bf16x8, b8);
    }
};

// split3 of one pair of floats in three steps, for hand-scheduled kernels.
struct PairSplit {
    float a, b;
    uint32_t w[3];  // h, m, l
    template <int J>
    GONN_DEV void step() {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        const bf16x2 c = {to_bf16(a), to_bf16(b)};
        w[J] = __builtin_bit_cast(uint32_t, c);
        if constexpr (J < 2) {
            a -= __uint_as_float(w[J] << 16);
            b -= __uint_as_float(w[J] & 0xffff0000u);
            pin(a);
            pin(b);
        } else {
            pin(w[J]);
        }
    }
};
// The six piece products of mfma_split3 in its order: pieces of a and b.
constexpr int kSplitA[6] = {2, 0, 1, 1, 0, 0}, kSplitB[6] = {0, 2, 1, 0, 1, 0};
GONN_DEV bf16x8 piece(const bf16x8x3& x, int i) { return i == 0 ? x.h : (i == 1 ? x.m : x.l); }

// NM MFMA slots of a hand-scheduled stretch: slot e runs slot(e), then the
// micro-ops u of [0, NU) that fall to it, fenced so the compiler keeps them
// beside that MFMA.
template <int NM, int NU, typename S, typename U>
GONN_DEV void mfma_slots(S&& slot, U&& uop) {
    static_for<NM>([&](auto E) {
        constexpr int e = decltype(E)::value, u0 = e * NU / NM, u1 = (e + 1) * NU / NM;
        slot(E);
        static_for<u1 - u0>([&](auto I) { uop(std::integral_constant<int, u0 + decltype(I)::value>{}); });
        __builtin_amdgcn_sched_barrier(0);
    });
}

// The streamed side of a stage: NT tiles of 32 rows of two fp32 tensors.
template <int D, int NT>
struct SplitStage {
    static constexpr int NCH = 32 * D / 8, CH = NT * NCH / 256;
    f32x4 r[CH][2][2];  // [chunk][tensor][half]
    int row[CH], col[CH];
    GONN_DEV void init(int tid) {
        for (int i = 0; i < CH; i++) {
            int rr, c;
            const int pos = i * 256 + tid;
            slab_chunk(pos % NCH, 32, rr, c);
            row[i] = pos / NCH * 32 + rr;
            col[i] = c * 8;
        }
    }
    // Tiles that start past the last of n rows are neither loaded nor stored
    // (uniform: a chunk instruction fills one tile or part of one).
    static GONN_DEV bool live(int i, int row0, int n) {
        return NT == 1 || row0 + i * 256 / NCH * 32 < n;
    }
    // Rows row0 .. of a and b, clamped to the last of n (clamped rows carry
    // no weight).
    GONN_DEV void load(const float* a, const float* b, int row0, int n) {
        for (int i = 0; i < CH; i++) {
            if (!live(i, row0, n)) break;
            int x = row0 + row[i];
            x = x < n ? x : n - 1;
            const float* pa = a + (size_t)x * D + col[i];
            const float* pb = b + (size_t)x * D + col[i];
            r[i][0][0] = *(const f32x4*)pa;
            r[i][0][1] = *(const f32x4*)(pa + 4);
            r[i][1][0] = *(const f32x4*)pb;
            r[i][1][1] = *(const f32x4*)(pb + 4);
        }
    }
    GONN_DEV void store(char* stage, int tid, int row0, int n) const {
        constexpr uint32_t PB = SplitTile<D>::PB;
        for (int i = 0; i < CH; i++) {
            if (!live(i, row0, n)) break;
            const int pos = i * 256 + tid;
            char* dst = stage + pos / NCH * SplitTile<D>::BYTES + pos % NCH * 16;
            for (int w = 0; w < 2; w++) {
                float x[8];
                for (int e = 0; e < 8; e++) x[e] = r[i][w][e >> 2][e & 3];
                const bf16x8x3 t = split3(x);
                *(bf16x8*)(dst + (3 * w + 0) * PB) = t.h;
                *(bf16x8*)(dst + (3 * w + 1) * PB) = t.m;
                *(bf16x8*)(dst + (3 * w + 2) * PB) = t.l;
            }
        }
    }
};

// Pieces of one row's elements 16 ks + 8 g .. +7.
template <int D>
GONN_DEV void load_row_split(const float* rowp, int g, bf16x8x3* f) {
    for (int ks = 0; ks < D / 16; ks++) {
        const f32x4 a = *(const f32x4*)(rowp + ks * 16 + g * 8);
        const f32x4 b = *(const f32x4*)(rowp + ks * 16 + g * 8 + 4);
        float x[8];
        for (int e = 0; e < 4; e++) {
            x[e] = a[e];
            x[4 + e] = b[e];
        }
        f[ks] = split3(x);
    }
}

// 16 steps of the two D-contractions on the fp32 instruction: s += a b, dp += c d.
GONN_DEV void plain_pair16(f32x16& s, f32x16& dp, const float* a, const float* b, const float* c,
                           const float* d) {
    f32x4 x[4][4];
    for (int i = 0; i < 4; i++) {
        x[0][i] = *(const f32x4*)(a + 4 * i);
        x[1][i] = *(const f32x4*)(b + 4 * i);
        x[2][i] = *(const f32x4*)(c + 4 * i);
        x[3][i] = *(const f32x4*)(d + 4 * i);
    }
    for (int i = 0; i < 16; i++) {
        s = mfma_f32(x[0][i / 4][i % 4], x[1][i / 4][i % 4], s);
        dp = mfma_f32(x[2][i / 4][i % 4], x[3][i / 4][i % 4], dp);
    }
}

GONN_DEV const float* mask_slice(const BwdParams& p, int bh) {
    return p.mask + (size_t)(bh / p.H) * p.mask_sb + (size_t)(bh % p.H) * p.mask_sh;
}

// Adds the accumulators of stream waves 1 .. nlive - 1 (those that had a tile)
// of each block wave to stream wave 0's, in order, through LDS; true in the
// waves that keep them.
template <int NACC, int WB, int NS>
GONN_DEV bool merge_stream(f32x16* acc, char* smem, int wb, int ws, int lane, int nlive) {
    if constexpr (NS > 1) {
        float* red = (float*)smem;
        if (ws > 0 && ws < nlive) {
            float* d = red + ((ws - 1) * WB + wb) * NACC * 1024 + lane;
            for (int t = 0; t < NACC; t++)
                for (int r = 0; r < 16; r++) d[(t * 16 + r) * 64] = acc[t][r];
        }
        if (nlive > 1) __syncthreads();  // uniform
        if (ws > 0) return false;
        for (int w = 1; w < nlive; w++) {
            const float* d = red + ((w - 1) * WB + wb) * NACC * 1024 + lane;
            for (int t = 0; t < NACC; t++)
                for (int r = 0; r < 16; r++) acc[t][r] += d[(t * 16 + r) * 64];
        }
    }
    return true;
}

}  // namespace gonn
