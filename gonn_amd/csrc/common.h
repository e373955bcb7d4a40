// common.h -- shared device helpers for the gfx950 attention kernels.
//
// MFMA operand/result layouts used throughout (wave64, lane l, g = l / 32,
// n = l % 32), for both v_mfma_f32_32x32x16_bf16 and v_mfma_f32_32x32x2_f32:
//   A (32 x K):  lane l holds row m = n, k-slots of lane-group g
//   B (K x 32):  lane l holds column n, the same k-slots of group g
//   C (32 x 32): lane l holds column n; register r holds row
//                8*(r/4) + 4*g + (r%4)
// Only the C layout is relied upon; the assignment of k to (g, item) merely
// has to be the same for A and B, which it is by construction.
// gonn_hip_selftest_mfma() checks this layout on the device.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

typedef __bf16 bf16;
typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

#define GONN_DEV __device__ __forceinline__

namespace gonn {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr double kLn2d = 0.6931471805599453;

GONN_DEV f32x16 mfma_bf16(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

GONN_DEV f32x16 mfma_f32(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Round-to-nearest-even fp32 -> bf16 (v_cvt_pk_bf16_f32 on gfx950).
GONN_DEV bf16 to_bf16(float x) { return (bf16)x; }

GONN_DEV float bf16_to_f32(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }

GONN_DEV bf16x8 pack8(float a0, float a1, float a2, float a3, float a4, float a5, float a6,
                      float a7) {
    bf16x8 r;
    r[0] = to_bf16(a0); r[1] = to_bf16(a1); r[2] = to_bf16(a2); r[3] = to_bf16(a3);
    r[4] = to_bf16(a4); r[5] = to_bf16(a5); r[6] = to_bf16(a6); r[7] = to_bf16(a7);
    return r;
}

// An fp32 value as three bf16 pieces, x = h + m + l to about 2^-26 |x| where
// 2^-110 <= |x| < 2^127.99, to 2^-134 below (each piece rounds the remainder to
// nearest; the differences are exact; SplitCheck finds results that either end
// of the range shows in). The fp32
// kernels form their products on the bf16 matrix cores as the six piece
// products of order 2^-16 and above (hh, hm, mh, hl, lh, mm); the three left
// out are below 2^-25 of the product, half a unit of its fp32 rounding. One
// 32x32x16 MFMA of each piece product takes 6 x 32 cycles against 8 x 64 for
// v_mfma_f32_32x32x2_f32 over the same 16 k.
struct bf16x8x3 {
    bf16x8 h, m, l;
};
GONN_DEV bf16x8x3 split3(const float* x) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    u32x4 r[3];
    for (int i = 0; i < 4; i++) {
        float a = x[2 * i], b = x[2 * i + 1];
        for (int j = 0; j < 3; j++) {
            // One v_cvt_pk_bf16_f32 per pair, and its halves back as floats.
            const bf16x2 c = {to_bf16(a), to_bf16(b)};
            const uint32_t u = __builtin_bit_cast(uint32_t, c);
            r[j][i] = u;
            a -= __uint_as_float(u << 16);
            b -= __uint_as_float(u & 0xffff0000u);
        }
    }
    return {__builtin_bit_cast(bf16x8, r[0]), __builtin_bit_cast(bf16x8, r[1]),
            __builtin_bit_cast(bf16x8, r[2])};
}
// c += a b over 16 k in the six piece products, the small ones first.
GONN_DEV f32x16 mfma_split3(const bf16x8x3& a, const bf16x8x3& b, f32x16 c) {
    c = mfma_bf16(a.l, b.h, c);
    c = mfma_bf16(a.h, b.l, c);
    c = mfma_bf16(a.m, b.m, c);
    c = mfma_bf16(a.m, b.h, c);
    c = mfma_bf16(a.h, b.m, c);
    return mfma_bf16(a.h, b.h, c);
}
// True when x is infinite or NaN. A file that uses it is built with NaNs
// honoured: an infinite operand shows by the NaN that its pieces make. The
// bits pass through an empty asm, without which the test becomes a
// floating-point class test and the D = 128 dK/dV kernel spills (358 -> 437 us
// at 64 x 500 x 2001).
GONN_DEV bool nonfinite(float x) {
    uint32_t u = __float_as_uint(x);
    asm("" : "+v"(u));
    return (u & 0x7f800000u) == 0x7f800000u;
}
// Collects result elements and tells whether one of them needs the plain fp32
// products: it is not finite, or neither zero nor above 2^-96. A bf16 holds
// nothing below 2^-133, so an operand below 2^-110 loses bits of its pieces,
// up to 2^-134 of absolute error; a result above 2^-96 does not show that. (An
// operand below 2^-134 has no pieces left and counts as zero. A score shows the
// loss only beside an operand of 2^100 or more; a forward's P not at all, since
// its row's sum is at least about 1.)
struct SplitCheck {
    uint32_t lo = ~0u, hi = 0;
    GONN_DEV void add(float x) {
        const uint32_t u = __float_as_uint(x) << 1;
        lo = u - 1 < lo ? u - 1 : lo;  // zero: the largest
        hi = u > hi ? u : hi;
    }
    GONN_DEV bool plain() const { return hi >= 0xff000000u || lo < (127u - 96) << 24; }
};

// 2^x on the transcendental unit (v_exp_f32).
GONN_DEV float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
// log2(x) (v_log_f32).
GONN_DEV float fast_log2(float x) { return __builtin_amdgcn_logf(x); }

// Combine a value with the one held by the lane 32 positions away
// (v_permlane32_swap). Both results of the swap are used, so the operation
// is symmetric in the two halves of the wave.
GONN_DEV float pair_max32(float x) {
    const uint32_t u = __float_as_uint(x);
    auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
GONN_DEV float pair_sum32(float x) {
    const uint32_t u = __float_as_uint(x);
    auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The same with the lane 16 positions away (rows 0 and 1, or 2 and 3).
GONN_DEV float pair_sum16(float x) {
    const uint32_t u = __float_as_uint(x);
    auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Rotate within each row of 16 lanes (DPP row_ror:n). n in 1..15.
template <int N>
GONN_DEV float row_ror(float x) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 | N, 0xf, 0xf, false));
}
// Sum over each row of 16 lanes; every lane of the row receives the total.
GONN_DEV float row_sum16(float x) {
    x += row_ror<8>(x);
    x += row_ror<4>(x);
    x += row_ror<2>(x);
    x += row_ror<1>(x);
    return x;
}

// Workgroup -> (bh, block) map for a grid of nblk blocks per (b,h) slice.
// Workgroups are dealt round-robin to the 8 XCDs (L & 7), so XCD x receives a
// contiguous range of slices in dispatch order: the blocks that share one
// slice's K/V (or Q/dO) run on the same XCD and share its L2. Within a slice
// the block order is reversed when `reverse` is set, which puts the longest
// causal blocks first.
//
// hgroup > 1 (causal grids): the blocks of hgroup consecutive slices of an
// XCD are dispatched interleaved, longest first (block nblk-1 of each slice,
// then nblk-2, ...). With hgroup * nblk close to the XCD's workgroup slots,
// each group's long blocks start together and its short blocks fill in
// behind them, so the grid ends without a tail of long blocks, while only
// about one group's K/V is live in the XCD's L2 at a time.
//
// deal: slice j * 8 + x instead of the range goes to XCD x (whole slices per
// XCD only). Where each sequence has its own length, a contiguous range gives
// an XCD the heads of one or two sequences and the whole grid waits for the
// XCD of the longest; dealt out, every XCD has its share of each sequence
// (causal attend, B 4, H 32, T 256, D 128, 2048 to 4096 keys: 193 -> 161 us,
// mean of five draws; B 64, T 8, 512 to 8192 keys: 1109 -> 941 us).
GONN_DEV void map_block(int L, int nblk, int BH, bool reverse, int& bh, int& blk,
                        int hgroup = 1, bool deal = false) {
    const int N = nblk * BH;
    int idx = L;
    if ((N & 7) == 0) {
        const int per = N >> 3;
        idx = (L & 7) * per + (L >> 3);
        if ((hgroup > 1 || deal) && per % nblk == 0) {
            // XCD-local position i among its Hx whole slices.
            const int x = L & 7, i = L >> 3, Hx = per / nblk;
            const int gsz = hgroup * nblk, gi = i / gsz, r = i - gi * gsz;
            const int gh = Hx - gi * hgroup < hgroup ? Hx - gi * hgroup : hgroup;
            const int rank = r / gh, hs = r - rank * gh;
            const int j = gi * hgroup + hs;
            bh = deal ? j * 8 + x : x * Hx + j;
            blk = reverse ? (nblk - 1 - rank) : rank;
            bh = __builtin_amdgcn_readfirstlane(bh);
            blk = __builtin_amdgcn_readfirstlane(blk);
            return;
        }
    }
    bh = idx / nblk;
    const int r = idx - bh * nblk;
    blk = reverse ? (nblk - 1 - r) : r;
    // The integer division runs on the VALU; pin the (uniform) results to
    // SGPRs so buffer resources built from them stay scalar (a resource in
    // VGPRs makes the compiler wrap every buffer load in a readfirstlane loop).
    bh = __builtin_amdgcn_readfirstlane(bh);
    blk = __builtin_amdgcn_readfirstlane(blk);
}

// Key position inside a 16-key group of the transposed-V (Vt) layout. The
// bf16 PV product reads, for lane-group g, keys {4g..4g+3, 8+4g..8+4g+3} as 8
// consecutive elements, which is how the S^T accumulator holds P. The map is
// its own inverse: it swaps the middle two quads.
GONN_DEV int vt_pos(int o) {
    return (o >= 4 && o < 8) ? o + 4 : ((o >= 8 && o < 12) ? o - 4 : o);
}

// ---- HBM -> LDS tile loads (buffer_load_dwordx4 ... lds) ----
// A raw buffer resource over [base, base + bytes): stride 0, reads past the
// end return zero. The fourth descriptor word selects 32-bit raw access.
typedef __amdgpu_buffer_rsrc_t brsrc;
GONN_DEV brsrc make_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
// Every lane reads 16 bytes at voff + soff of the buffer; lane L of the wave
// writes them to LDS byte address lds + 16 L (lds must be wave-uniform). The load counts
// in vmcnt only; callers wait with GONN_VMCNT and publish with a barrier.
//
// Issued from inline asm on purpose: the compiler treats an LDS-DMA load as a
// possible writer of any LDS address it cannot disambiguate, and then waits
// for all of them (vmcnt(0)) before the next ds_read, which turns a load
// meant to run a whole step ahead into a synchronous one. Hidden in asm, the
// load is invisible to the compiler's wait insertion; every buffer read
// after it is ordered by the explicit wait + barrier of the kernel's
// pipeline. M0 is set inside the statement; the compiler sets M0 itself
// before each of its own M0 uses (these kernels make none).
GONN_DEV void dma16(brsrc r, uint32_t lds, uint32_t voff, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(r), "s"(soff)
                 : "memory");
}
// dma16 with the non-temporal hint, for data read exactly once.
GONN_DEV void dma16_nt(brsrc r, uint32_t lds, uint32_t voff, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(r), "s"(soff)
                 : "memory");
}
// dma16 when the wave-uniform `on` is non-zero. The skip is a scalar branch
// inside the asm statement, so the caller's code stays one basic block (an
// exec-masked branch around the load would split the hand-scheduled MFMA
// stream and perturb register allocation).
GONN_DEV void dma16_if(brsrc r, uint32_t lds, uint32_t voff, uint32_t soff, uint32_t on) {
    asm volatile(
        "s_cmp_eq_u32 %4, 0\n\ts_cbranch_scc1 1f\n\t"
        "s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds\n1:"
        :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(r), "s"(soff),
           "s"(__builtin_amdgcn_readfirstlane(on))
        : "memory", "scc");
}
// dma16 split in two, so the M0 write can sit one instruction slot ahead of
// its load (an M0 write needs one wait state before an LDS-DMA load; another
// instruction in between fills it instead of an s_nop). The kernels that use
// these make no M0 use of their own between the two statements.
GONN_DEV void dma_set_m0(uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0" ::"s"(__builtin_amdgcn_readfirstlane(lds)) : "memory");
}
GONN_DEV void dma16_m0(brsrc r, uint32_t voff, uint32_t soff) {
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(r), "s"(soff)
                 : "memory");
}
GONN_DEV void dma16_m0_if(brsrc r, uint32_t voff, uint32_t soff, uint32_t on) {
    asm volatile(
        "s_cmp_eq_u32 %3, 0\n\ts_cbranch_scc1 1f\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds\n1:"
        ::"v"(voff), "s"(r), "s"(soff), "s"(__builtin_amdgcn_readfirstlane(on))
        : "memory", "scc");
}
// LDS byte address of a __shared__ object (apply to the array itself, so the
// address-space cast folds to a constant).
GONN_DEV uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
// s_waitcnt vmcnt(n) (expcnt, lgkmcnt unconstrained), n < 64: the gfx9
// encoding splits vmcnt into bits 3:0 and 15:14.
#define GONN_VMCNT(n) \
    __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | ((((n) >> 4) & 3) << 14))

// Swizzled slab layout of LDS tiles (forward K / Vt tiles, dK/dV Q / dO
// tiles). A tile of `rows` rows of 16-byte chunks is stored in 64-byte
// segments of four chunks: position (16 bytes each)
//   pos(row, chunk) = ((chunk / 4) * rows + row) * 4 + ((chunk % 4) ^ h(row)),
//   h(row) = (row >> 2) & 3.
// A load instruction then fills 16 rows x 64 contiguous bytes (coalesced).
// LDS on gfx950 has 64 banks (256 bytes); a ds_read_b128 serves 16 lanes per
// cycle, but not 16 consecutive ones: a probe of SQ_LDS_BANK_CONFLICT over
// 50 lane patterns fits only groups within one half-wave made of 4-lane
// quads {0, 2, 5, 7} and {1, 3, 4, 6} of that half (or {0, 3, 5, 6} and
// {1, 2, 4, 7}). A read of rows 32m + ln, one chunk, puts quad q of a half
// on banks 4 (ln & 3) + (chunk % 4 ^ (q & 3)): distinct within every such
// group, so the operand reads are conflict-free. (h = ((row >> 1) ^
// (row >> 3)) & 3, distinct over 16 consecutive lanes, measured 2-way.)
// No padding: a tile of 64 rows x 128 bf16 is 16 KB.
GONN_DEV int slab_swz(int row) { return (row >> 2) & 3; }
// Row and chunk held by position `pos` of a tile of `rows` rows.
GONN_DEV void slab_chunk(int pos, int rows, int& row, int& chunk) {
    const int q = pos >> 2;
    row = q % rows;
    chunk = (q / rows) * 4 + ((pos & 3) ^ slab_swz(row));
}

// ---- hand scheduling helpers ----
// Forces x to be computed at this point of the program (an empty asm that
// reads it): keeps hand-scheduled VALU work from being sunk to its uses.
template <typename T>
GONN_DEV void pin(const T& x) {
    asm volatile("" ::"v"(x));
}

// Compile-time loop: f(std::integral_constant<int, i>) for i = 0 .. N-1.
template <typename F, int... I>
GONN_DEV void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
GONN_DEV void static_for(F&& f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

}  // namespace gonn
