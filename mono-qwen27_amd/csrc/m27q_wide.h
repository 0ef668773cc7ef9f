// m27q_wide.h -- products of up to 64 activation rows in one pass over the
// weights: Y[M][N] = X[M][K] W[N][K]^T.
//
// What bounds it.  With 64 tokens a weight byte meets 64 activation rows, so
// the arithmetic on group sums, not HBM, sets the time: every (row, token,
// 32-group) sum has to be scaled by the token's fp32 group scale dx and added
// in fp32.  On exact int8 sums that took about 3.5 VALU operations (int to
// float, two scales, the add), for each of the launches of 16 tokens, and each
// launch unpacked the weights again.  Here:
//   - one launch takes all tokens (NT tiles of 16), so the weights are read
//     and unpacked once;
//   - Q4_K, Q5_K and Q6_K put the block's small integer scales into the weight
//     operand: sc q is an integer that fp16 holds exactly (Q4_K <= 945, Q5_K
//     <= 1953; Q6_K's up to 4096 as an exact sum of two fp16 values), the int8
//     codes are exact in fp16, and the fp32 MFMA accumulator holds the group's
//     integer sum exactly (below 2^24).  What is left per (row, token, group)
//     is one FMA with dx; d (and dmin) follow once per 256 weights.  Q4_K and
//     Q5_K keep all of this 2^-10 down until the final sum, so that dx times a
//     group's sum does not overflow where the result does not (results below
//     2^-116 are sums of multiples of 2^-139 for it);
//   - Q4_K / Q5_K's min term, sum_j m_j (dx_j sum(codes_j)), is one bf16 MFMA
//     per tile and block: m_j is exact in bf16, and the fp32 token factor is
//     split into three bf16 values that add up to it exactly (two of them kept
//     2^7 and 2^14 up against m_j as much down, for the smallest factors);
//   - Q8_0 (a scale per 32 weights and row) and IQ4_XS (12-bit products) stay
//     on int8 MFMA with the scales in fp32 afterwards.
//
// Operands (v_mfma_f32_16x16x32_f16 / _bf16, v_mfma_i32_16x16x32_i8; q = lane
// / 16, c = lane % 16): A = weights, lane holds row c of the set, 8 positions
// of the group; B = activations, token c, the same positions; the result is
// rows 4 q + e (e = 0..3) x token c, so dx is one value per lane and tile.
// Positions may be dealt to lanes and slots in any order that both operands
// share: byte 8 q + {0, 2, 1, 3, 4, 6, 5, 7} of the group for the fp16 types
// (the halves of a dword are taken with one mask), 8 q + 0..7 for Q8_0, and
// 4 q + 0..3 and 16 + 4 q + 0..3 for IQ4_XS (both nibbles of four bytes).
//
// Work.  8 waves, one workgroup per CU: RW row waves x KW slices of K.  A
// workgroup owns a run of 16-row sets (spread evenly over the grid), dealt to
// its row waves, at most RSM each.  The row waves of a K slice share its
// activations, converted and laid out in operand order in LDS four groups at a
// time (a step; double-buffered, one barrier per step; a slice of one wave has
// one buffer and no barrier), while each wave's weights stream from memory
// straight into registers, asked for one 256-weight unit ahead.  The KW partial
// sums are added in LDS in slice order.
//
// What holds it back now, by the compiler's output (VGPRs, spills, instructions
// and waits of the loops):
//   - a step is conditional (slices differ by a unit), so the wait counts merge
//     over both paths and every step waits once for all loads in flight
//     (vmcnt(0)): the weights are not a whole unit ahead in effect.  The next
//     unit's scales, needed by its first group, are asked for last;
//   - Q6_K with four token tiles and three sets per wave (M = 49 to 64 past two
//     sets per CU) does not fit 256 registers and spills 14 to 51 of them: 17408 x
//     5120 42.7 us at M = 48, 84.6 at M = 64 (107.1 in launches of 16 tokens).
//
// What was measured on the way (gate/up, 2 x 17408 x 5120 Q4_K, and down, 5120
// x 17408 Q6_K, at M = 64; replays of a graph; what was slower, on the loop as it
// is, so an unconditional one may decide otherwise):
//   - four launches of 16 tokens of the MFMA kernel: 115 and 103 us; this kernel
//     59 and 65;
//   - the vector and matrix instructions of a wave pair add up (they hardly
//     overlap): down's 543 vector instructions of 4 cycles and 64 MFMAs of 16 per
//     unit (and set, of one per wave) are about 45 of its 65 us.  Dealing MFMAs
//     between vector instructions of other groups (schedule groups, software
//     pipelining over sets) was slower: 75 against 67 us on gate/up (traced);
//   - loads must touch few 128-byte lines: a step of 4 groups reads each
//     token's 128 codes as one line (2 groups, half a line: Q4_K 5120 x 17408
//     87 us against 58), and the weights' 8-byte pieces of a line come in
//     several loads, so they are temporal (non-temporal: down 90 us against 79,
//     Q4_K at M = 17-48 5-11% slower);
//   - 12 or 16 waves per workgroup (2-group steps) were slower at every size, and
//     two units of weights in flight 3-5% slower than one;
//   - offsets kept in registers instead of computed per step: down 90 -> 78 us.
//
// No reference counterpart: the reference runs prefill one token at a time
// (src/mono27b_chat.cpp:399-403).
#pragma once

#include <algorithm>

#include "m27q_internal.h"
#include "m27q_device.h"

namespace m27q {
namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef int i4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));

constexpr int kStepGroups = 4;  // groups of 32 weights per step, half a 256-weight unit
constexpr int kMinStep = 7;  // powers of two between the parts of a min term's token factor
constexpr uint32_t kH1024 = 0x64006400u;  // (1024, 1024) in fp16: or-ing an integer below 1024 in adds it

__device__ __forceinline__ h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ uint32_t as_u32(h2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ h2 splat(float v) { return h2{(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ h2 pk_fma(h2 a, h2 b, h2 c) { return __builtin_elementwise_fma(a, b, c); }
__device__ __forceinline__ float ubyte(uint32_t w, int e) { return (float)((w >> (8 * e)) & 0xffu); }
__device__ __forceinline__ float bperm(int byte_lane, float v) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(byte_lane, __float_as_int(v)));
}
__device__ __forceinline__ uint32_t bperm(int byte_lane, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute(byte_lane, (int)v);
}

// Masks and biases held in vector registers: a three-operand instruction takes
// no literal and one scalar register, so with these (x & mask) | bias is one
// instruction (v_and_or_b32 / v_bitop3_b32) instead of two.
struct Cst {
    uint32_t lo = 0x000f000fu, hi = 0x00f000f0u, h1024 = kH1024;
    uint32_t byte = 0x00ff00ffu, bias = 0x64806480u;
    uint32_t q6l = 0x00300030u, q6h = 0x03000300u;
    __device__ Cst() {
        asm volatile("" : "+v"(lo), "+v"(hi), "+v"(h1024), "+v"(byte), "+v"(bias), "+v"(q6l), "+v"(q6h));
    }
};

// (x & m) | c, written out: the compiler regroups a chain of these into an and
// per term and one three-way or, which is one instruction more per pair.
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t m, uint32_t c) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(m), "v"(c));
    return r;
}

template <int AUX>
__device__ __forceinline__ u4 ld16(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff) {
    return __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, AUX));
}
template <int AUX>
__device__ __forceinline__ u2 ld8(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff) {
    return __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, AUX));
}
// Fields of GGUF Q6_K and Q8_0 blocks, 2-byte aligned: one unaligned global
// load each (the target's unaligned access mode), reading the field alone.
__device__ __forceinline__ u4 ldu16(const uint8_t *p) {
    typedef uint32_t u4u __attribute__((ext_vector_type(4), aligned(2)));
    return *(const u4u *)p;
}
__device__ __forceinline__ u2 ldu8(const uint8_t *p) {
    typedef uint32_t u2u __attribute__((ext_vector_type(2), aligned(2)));
    return *(const u2u *)p;
}

// One weight operand (or two that add up to it).
template <bool TWO>
struct AOp {
    h8 a, b;
};
template <>
struct AOp<false> {
    h8 a;
};

__device__ __forceinline__ h8 make_h8(uint32_t x, uint32_t y, uint32_t z, uint32_t w) {
    return __builtin_bit_cast(h8, u4{x, y, z, w});
}

// ------------------------------------------------------------ Q4_K, Q5_K --
template <bool Q5>
struct WQ4K {
    static constexpr bool kF16 = true, kMin = true, kTwo = false, kInterleave = false, kRagged = false;
    static constexpr int kUnitBytes = Q5 ? kQ5KUnit : kQ4KUnit;  // per 8 rows, TILED
    static constexpr int kBlockBytes = Q5 ? kQ5KBytes : kQ4KBytes;
    struct Reg {
        u2 q[4];         // bytes 8 q .. of the four 32-byte chunk pairs (groups 2 j, 2 j + 1)
        u4 h;            // d | dmin << 16, scales[12]
        u2 qh;           // Q5_K: qh bytes 8 q ..
    };
    template <int LAYOUT, int G0>  // groups G0 .. G0 + 3 of unit u
    __device__ static void load(Reg &r, const uint8_t *wp, __amdgpu_buffer_rsrc_t rs, uint32_t base, int i, int q, int u, int) {
        if constexpr (LAYOUT == M27Q_LAYOUT_TILED) {
            const uint32_t s = (uint32_t)u * (uint32_t)kUnitBytes;
#pragma unroll
            for (int j = G0 / 2; j < G0 / 2 + 2; ++j) r.q[j] = ld8<0>(rs, base + (uint32_t)(q4k_tqs(i, j) + 8 * q), s);
            if constexpr (G0 == 4) {
                r.h = ld16<0>(rs, base + 16u * (uint32_t)i, s);
                if constexpr (Q5) r.qh = ld8<0>(rs, base + (uint32_t)(kQ5KTQh + 32 * i + 8 * q), s);
            }
        } else {
            const uint32_t s = (uint32_t)u * (uint32_t)kBlockBytes;
            constexpr int qs = Q5 ? kQ5KQs : kQ4KHdr;
#pragma unroll
            for (int j = G0 / 2; j < G0 / 2 + 2; ++j) r.q[j] = ld8<0>(rs, base + (uint32_t)(qs + 32 * j + 8 * q), s);
            if constexpr (G0 == 4) {
                r.h = ld16<0>(rs, base, s);
                if constexpr (Q5) r.qh = ld8<0>(rs, base + (uint32_t)(kQ5KQh + 8 * q), s);
            }
        }
    }
    // 2^-10 sc q of group G: 1024 + q (even groups; 1024 + 16 q for the high
    // nibbles of odd ones) from one mask, then one FMA: (1024 + q) s - 1024 s
    // with s = 2^-10 sc, or 2^-14 sc; every intermediate is exact in fp16.  The
    // 2^-10 (kDown; the final sum takes it back) keeps dx times the group's sum
    // within fp32 wherever the 16-token kernel's, which applies sc later, is:
    // without it rows of magnitude 1e34 to 1e36 came out infinite.
    static constexpr int kDown = 10;
    template <int G>
    __device__ static AOp<false> operand(const Reg &r, int, const Cst &cst) {
        constexpr bool odd = G & 1;
        const uint32_t scw = G < 4 ? (r.h.y & 0x3f3f3f3fu) : ((r.h.w & 0x0f0f0f0fu) | ((r.h.y >> 2) & 0x30303030u));
        constexpr uint32_t sel = 0x04000400u | (uint32_t)(G & 3) | ((uint32_t)(G & 3) << 16);
        const h2 t = as_h2(__builtin_amdgcn_perm(0x64646464u, scw, sel));  // 1024 + sc
        const h2 s = odd ? pk_fma(t, splat(0x1p-14f), splat(-0x1p-4f)) : pk_fma(t, splat(0x1p-10f), splat(-1.f));
        const h2 n = s * splat(-1024.f);
        const uint32_t m = odd ? cst.hi : cst.lo;
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint32_t x = k ? r.q[G / 2].y : r.q[G / 2].x;
            uint32_t a = (x & m) | cst.h1024, b = ((x >> 8) & m) | cst.h1024;
            if constexpr (Q5) {  // bit G of the qh bytes at bit 4 (8 for the high nibbles)
                const uint32_t hb = k ? r.qh.y : r.qh.x;
                constexpr uint32_t bm = odd ? 0x01000100u : 0x00100010u;
                constexpr int up = (odd ? 8 : 4) - G;  // even bytes: shift left by this (right if negative)
                a |= (up >= 0 ? hb << (up & 31) : hb >> (-up & 31)) & bm;
                b |= (hb >> (8 - up)) & bm;
            }
            w[2 * k] = as_u32(pk_fma(as_h2(a), s, n));
            w[2 * k + 1] = as_u32(pk_fma(as_h2(b), s, n));
        }
        return {make_h8(w[0], w[1], w[2], w[3])};
    }
    // The min term's weight operand: 2^-(10 + 7 q) m_0 .. m_7 of row c in bf16
    // in lane quarters q = 0-2 (against the three parts of the token factors,
    // the second and third of which are kept 2^7 and 2^14 up), 0 in quarter 3.
    // The power of two is taken off the exponents (m = 0 saturates at 0).
    __device__ static b8 min_operand(const Reg &r, int q) {
        typedef uint16_t s2 __attribute__((ext_vector_type(2)));
        const s2 down = (s2)(uint16_t)((kDown + kMinStep * q) << 7);
        const uint32_t on = q < 3 ? ~0u : 0u;
        const uint32_t m0 = r.h.z & (0x3f3f3f3fu & on);
        const uint32_t m1 = (((r.h.w >> 4) & 0x0f0f0f0fu) | ((r.h.z >> 2) & 0x30303030u)) & on;
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t m = k < 2 ? m0 : m1;
            const int e = 2 * (k & 1);
            const uint32_t b = __builtin_amdgcn_perm(__float_as_uint(ubyte(m, e + 1)), __float_as_uint(ubyte(m, e)), 0x07060302u);
            w[k] = __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(s2, b), down));
        }
        return __builtin_bit_cast(b8, u4{w[0], w[1], w[2], w[3]});
    }
    __device__ static uint32_t dword(const Reg &r) { return r.h.x; }  // d | dmin << 16 of row c
};

// ------------------------------------------------------------------ Q6_K --
// Group 4 h + rr: low (rr < 2) or high nibbles of ql bytes 64 h + 32 (rr & 1)
// .., bits 2 rr of qh bytes 32 h .., scale 8 h + 2 rr + (position / 16).
struct WQ6K {
    static constexpr bool kF16 = true, kMin = false, kTwo = true, kInterleave = false, kRagged = false;
    static constexpr int kDown = 0;
    static constexpr int kUnitBytes = kQ6KUnit, kBlockBytes = kQ6KBytes;
    struct Reg {
        u2 ql[4], qh[2];
        u4 sc;
        uint32_t d;
    };
    template <int LAYOUT, int G0>
    __device__ static void load(Reg &r, const uint8_t *wp, __amdgpu_buffer_rsrc_t rs, uint32_t base, int i, int q, int u, int) {
        constexpr int h = G0 / 4;  // half of the unit
        if constexpr (LAYOUT == M27Q_LAYOUT_TILED) {
            const uint32_t s = (uint32_t)u * (uint32_t)kUnitBytes;
#pragma unroll
            for (int x = 0; x < 2; ++x)
                r.ql[2 * h + x] = ld8<0>(rs, base + (uint32_t)(kQ6KTQl + 128 * i + 64 * h + 32 * x + 8 * q), s);
            r.qh[h] = ld8<0>(rs, base + (uint32_t)(kQ6KTQh + 64 * i + 32 * h + 8 * q), s);
            if constexpr (G0 == 4) {
                r.sc = ld16<0>(rs, base + (uint32_t)(kQ6KTSc + 16 * i), s);
                r.d = bld_u16<0>(rs, base + (uint32_t)(kQ6KTD + 2 * i), s);
            }
        } else {
            const uint8_t *blk = wp + (base + (uint32_t)u * (uint32_t)kBlockBytes);
#pragma unroll
            for (int x = 0; x < 2; ++x) r.ql[2 * h + x] = ldu8(blk + kQ6KQl + 64 * h + 32 * x + 8 * q);
            r.qh[h] = ldu8(blk + kQ6KQh + 32 * h + 8 * q);
            if constexpr (G0 == 4) {
                r.sc = ldu16(blk + kQ6KSc);
                r.d = *(const uint16_t *)(blk + kQ6KD);
            }
        }
    }
    // sc (q - 32) of group G as two fp16 operands: their product rounded to
    // fp16, and the remainder (an FMA; exact).
    template <int G>
    __device__ static AOp<true> operand(const Reg &r, int q, const Cst &cst) {
        constexpr int h = G / 4, rr = G % 4;
        constexpr bool hi = rr >= 2;
        const u2 ql = r.ql[2 * h + (rr & 1)], qh = r.qh[h];
        const uint32_t scw = h ? (rr < 2 ? r.sc.z : r.sc.w) : (rr < 2 ? r.sc.x : r.sc.y);
        // scale byte 2 (rr & 1) + (q / 2), as 1152 + sc
        const uint32_t sub = (uint32_t)(q >> 1) * 0x00010001u;
        const h2 t = as_h2(__builtin_amdgcn_perm(0x64646464u, scw ^ 0x80808080u, (0x04000400u + 0x00020002u * (rr & 1)) + sub));
        // high nibbles stay in place: 16 (q - 32) against sc / 16
        const h2 s = hi ? pk_fma(t, splat(0.0625f), splat(-72.f)) : t - splat(1152.f);
        const uint32_t m = hi ? cst.hi : cst.lo;
        const uint32_t hm = hi ? cst.q6h : cst.q6l;
        constexpr int up = (rr & 1) ? 2 : 4;  // qh's bits to bit 4 (8): left by this, odd bytes right by 8 - this
        uint32_t w[4], e[4];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint32_t l = k ? ql.y : ql.x, hb = k ? qh.y : qh.x;
            const uint32_t a = and_or(hb << up, hm, and_or(l, m, cst.h1024));
            const uint32_t b = and_or(hb >> (8 - up), hm, and_or(l >> 8, m, cst.h1024));
            const h2 o = splat(hi ? 1536.f : 1056.f);
            const h2 va = as_h2(a) - o, vb = as_h2(b) - o;
            const h2 pa = va * s, pb = vb * s;
            w[2 * k] = as_u32(pa);
            w[2 * k + 1] = as_u32(pb);
            e[2 * k] = as_u32(pk_fma(va, s, -pa));
            e[2 * k + 1] = as_u32(pk_fma(vb, s, -pb));
        }
        return {make_h8(w[0], w[1], w[2], w[3]), make_h8(e[0], e[1], e[2], e[3])};
    }
    __device__ static uint32_t dword(const Reg &r) { return r.d; }
};

// ------------------------------------------------------------------ Q8_0 --
// A unit here is 8 blocks (two TILED units).
struct WQ80 {
    static constexpr bool kF16 = false, kMin = false, kTwo = false, kInterleave = false, kRagged = true;
    static constexpr int kDown = 0;
    static constexpr int kUnitBytes = kQ80Unit, kBlockBytes = kQ80Bytes;
    struct Reg {
        u2 q[8];
        uint32_t d[8];  // TILED: words 0, 2, 4, 6 hold two scales each; GGUF: one each
    };
    template <int LAYOUT, int G0>
    __device__ static void load(Reg &r, const uint8_t *wp, __amdgpu_buffer_rsrc_t rs, uint32_t base, int i, int q, int u, int rb) {
        if constexpr (LAYOUT == M27Q_LAYOUT_TILED) {
            const int nu = (rb + kQ80UnitBlocks - 1) / kQ80UnitBlocks;
            const uint32_t s = (uint32_t)min(2 * u + G0 / 4, nu - 1) * (uint32_t)kUnitBytes;
#pragma unroll
            for (int g = G0; g < G0 + 4; ++g) r.q[g] = ld8<0>(rs, base + (uint32_t)(128 * i + 32 * (g & 3) + 8 * q), s);
            r.d[G0] = bld_u32<0>(rs, base + (uint32_t)(kQ80TD + 8 * i), s);
            r.d[G0 + 2] = bld_u32<0>(rs, base + (uint32_t)(kQ80TD + 8 * i + 4), s);
        } else {
#pragma unroll
            for (int g = G0; g < G0 + 4; ++g) {
                const uint8_t *blk = wp + (base + (uint32_t)min(8 * u + g, rb - 1) * (uint32_t)kBlockBytes);
                r.q[g] = ldu8(blk + 2 + 8 * q);
                r.d[g] = *(const uint16_t *)blk;
            }
        }
    }
    template <int G>
    __device__ static long operand(const Reg &r) {
        return __builtin_bit_cast(long, r.q[G]);
    }
    // Group G's scale of row c (0 past the row's blocks).
    template <int G, int LAYOUT>
    __device__ static float factor(const Reg &r, int u, int rb) {
        const uint32_t w = LAYOUT == M27Q_LAYOUT_TILED ? r.d[G / 2 * 2] >> (16 * (G & 1)) : r.d[G];
        return 8 * u + G < rb ? f16_bits_to_f32(w) : 0.f;
    }
};

// ---------------------------------------------------------------- IQ4_XS --
struct WIQ4XS {
    static constexpr bool kF16 = false, kMin = false, kTwo = false, kInterleave = true, kRagged = false;
    static constexpr int kDown = 0;
    static constexpr int kUnitBytes = kIQ4XSUnit, kBlockBytes = kIQ4XSBytes;
    struct Reg {
        uint32_t q[8];  // qs bytes 4 q .. + 4 of each group
        u2 hd;          // d | scales_h << 16, scales_l[4]
    };
    template <int LAYOUT, int G0>
    __device__ static void load(Reg &r, const uint8_t *wp, __amdgpu_buffer_rsrc_t rs, uint32_t base, int i, int q, int u, int) {
        constexpr bool kT = LAYOUT == M27Q_LAYOUT_TILED;
        const uint32_t s = (uint32_t)u * (uint32_t)(kT ? kUnitBytes : kBlockBytes);
        const uint32_t qs = base + (uint32_t)(kT ? 128 * i : kIQ4XSQs) + 4u * (uint32_t)q;
#pragma unroll
        for (int g = G0; g < G0 + 4; ++g) r.q[g] = bld_u32<0>(rs, qs + 16u * (uint32_t)g, s);
        if constexpr (G0 == 4) r.hd = ld8<0>(rs, base + (uint32_t)(kT ? kIQ4XSTHdr + 8 * i : 0), s);
    }
    template <int G>
    __device__ static long operand(const Reg &r) {
        const uint32_t w = r.q[G];
        return __builtin_bit_cast(long, u2{iq4_lut(w & 0x0f0f0f0fu), iq4_lut((w >> 4) & 0x0f0f0f0fu)});
    }
    template <int G, int LAYOUT>
    __device__ static float factor(const Reg &r, int, int) {
        const int ls = (int)(((r.hd.y >> (8 * (G >> 1) + 4 * (G & 1))) & 15u) | (((r.hd.x >> (16 + 2 * G)) & 3u) << 4)) - 32;
        return f16_bits_to_f32(r.hd.x) * (float)ls;
    }
};

// ------------------------------------------------------------ the kernel --

constexpr uint32_t kPast = 0xffffff00u;  // past every activation buffer (below 2^27 bytes)

// Launch shapes: RW row waves x KW slices of K, at most RSM sets per wave.
template <int RW_, int KW_, int RSM_>
struct Shape {
    static constexpr int RW = RW_, KW = KW_, RSM = RSM_, W = RW_ * KW_;
};

template <class T, int NT, class SH>
struct Wide {
    static constexpr int RW = SH::RW, KW = SH::KW, RSM = SH::RSM, GS = kStepGroups, W = SH::W;
    static constexpr int NB = RW == 1 ? 1 : 2;   // step buffers
    // activation loads in flight, in steps: a step of one set is shorter than
    // their latency
    static constexpr int DP = RSM == 1 ? 2 : 1;
    static constexpr int TOK = 16 * NT;
    static constexpr int FB = T::kF16 ? 16 : 8;  // operand bytes per lane
    static constexpr int kCodes = GS * NT * kWave * FB;
    static constexpr int kDx = GS * TOK * 4;
    static constexpr int kAux = T::kMin ? NT * 48 * 16 : 0;  // per unit
    static constexpr int oDx = NB * kCodes, oAux = oDx + NB * kDx, kSlice = oAux + NB * kAux;
    static constexpr int kStage = KW * kSlice;
    static constexpr int NTH = RW * kWave;                // threads staging a slice
    static constexpr int kChunks = TOK * GS * 2;          // 16-code chunks of a step
    static constexpr int NC = (kChunks + NTH - 1) / NTH;  // per thread
    static constexpr int kScales = TOK * GS;
    static constexpr int NSC = (kScales + NTH - 1) / NTH;
    static constexpr int kMaxSets = RW * RSM;
    static constexpr int kRed = KW * kMaxSets * NT * kWave * 16;
    static constexpr int kLds = kStage > kRed ? kStage : kRed;
    static_assert(kLds <= kWideLds, "one workgroup per CU");
};

// 16 int8 codes -> the fp16 operands of two lane quarters (or the int8 ones).
// c is the token's slot in the quarter: its column xor the chunk's place j in
// the step, so that the eight lanes that hold one token's chunks write to
// different banks; the reader (lane q, c) finds group g's operand of its token
// in slot c ^ (2 g + q / 2).
template <class T>
__device__ __forceinline__ void store_codes(uint8_t *dst, const u4 &v, int j, int tok, const Cst &cst) {
    const int hh = j & 1, c = tok ^ j;
    if constexpr (T::kF16) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t x = k == 0 ? (j ? v.y : v.x) : (j ? v.w : v.z);
                // 1024 + (code + 128): the sign bit flipped under fp16's 1024
                w[2 * j] = as_u32(as_h2((x & cst.byte) ^ cst.bias) - splat(1152.f));
                w[2 * j + 1] = as_u32(as_h2(((x >> 8) & cst.byte) ^ cst.bias) - splat(1152.f));
            }
            *(u4 *)(dst + ((2 * hh + k) * 16 + c) * 16) = u4{w[0], w[1], w[2], w[3]};
        }
    } else if constexpr (T::kInterleave) {
#pragma unroll
        for (int k = 0; k < 4; ++k) *(uint32_t *)(dst + (k * 16 + (c ^ hh ^ (k >> 1))) * 8 + 4 * hh) = v[k];
    } else {
        *(u2 *)(dst + ((2 * hh) * 16 + c) * 8) = u2{v.x, v.y};
        *(u2 *)(dst + ((2 * hh + 1) * 16 + c) * 8) = u2{v.z, v.w};
    }
}

// Between a wave's LDS accesses that exchange values between its lanes.  The
// hardware runs a wave's LDS operations in order, so no wait is needed; this
// keeps the compiler, which sees each lane's own addresses, from moving them.
// It also keeps it from scheduling across: over 800 shapes of up to one set per
// CU, M = 17 to 64, 0.1% slower on average and 5% at most (Q6_K 1024 x 5120 at
// M = 32 12.9 us with and without, IQ4_XS 2560 x 5120 at M = 48 17.3 against
// 16.6).  In the loop it stands before the step's loads for IQ4_XS, between them
// for Q8_0 and after them for the others, where each type lost least.
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <int V>
struct Int {
    static constexpr int value = V;
};
template <int N, class F>
__device__ __forceinline__ void unroll(F &&f) {
    if constexpr (N > 0) {
        unroll<N - 1>(f);
        f(Int<N - 1>{});
    }
}

template <class T, int NT, class SH, int LAYOUT>
__global__ __launch_bounds__(kWave *SH::W, SH::W / 4) void k_matmul_wide(MatmulMultiParams p) {
    extern __shared__ __align__(16) uint8_t smem[];
    using C = Wide<T, NT, SH>;
    constexpr int RW = C::RW, KW = C::KW, GS = C::GS, RSM = C::RSM, TOK = C::TOK, NTH = C::NTH;
    constexpr int NST = 8 / GS;  // steps per unit
    constexpr bool kT = LAYOUT == M27Q_LAYOUT_TILED;
    const int lane = (int)(threadIdx.x & 63), q = lane >> 4, c = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // Waves w and w + 4 share a SIMD: waves 4-7 deal the sets from the other
    // end, so the waves with one set more land on different SIMDs.
    const int kw = wave / RW, rw = wave % RW;
    const int deal = wave & 4 ? RW - 1 - rw : rw;
    const int K = p.K, ngk = K / 32, U = (K + 255) / 256;

    // This workgroup's sets and this wave's share.
    const int S = p.wg_start[p.nmat];
    const int s0 = (int)((long long)S * blockIdx.x / gridDim.x);
    const int nsets = (int)((long long)S * (blockIdx.x + 1) / gridDim.x) - s0;
    const int f0 = (nsets * deal + RW - 1) / RW;
    const int ns = (nsets * (deal + 1) + RW - 1) / RW - f0;
    // ... and its slice of K.
    const int ua = U * kw / KW, ub = U * (kw + 1) / KW;
    const int umax = (U + KW - 1) / KW;

    __amdgpu_buffer_rsrc_t rs[RSM];
    const uint8_t *wp[RSM];
    uint32_t base[RSM];
    int ri[RSM];
#pragma unroll
    for (int s = 0; s < RSM; ++s) {
        const int gs = s0 + f0 + (s < ns ? s : 0);
        int mi = 0;
#pragma unroll
        for (int k = 1; k < kMaxMulti; ++k)
            if (k < p.nmat && gs >= p.wg_start[k]) mi = k;
        const int rc = p.rc[mi], row0 = min((gs - p.wg_start[mi]) * 16, (rc - 1) / 16 * 16);
        if constexpr (kT) {
            const int tile0 = row0 / kTileRows, tiles = (rc + kTileRows - 1) / kTileRows;
            const uint32_t tb = (uint32_t)p.upr * (uint32_t)T::kUnitBytes;
            wp[s] = p.W[mi] + (size_t)tile0 * tb;
            rs[s] = buf_rsrc(wp[s], (uint32_t)min(2, tiles - tile0) * tb);
            base[s] = (uint32_t)min(c >> 3, tiles - 1 - tile0) * tb;  // rows past the end reread a tile
            ri[s] = c & 7;
        } else {
            const uint32_t rowb = (uint32_t)p.rb * (uint32_t)T::kBlockBytes;
            wp[s] = p.W[mi] + (size_t)row0 * rowb;
            rs[s] = buf_rsrc(wp[s], (uint32_t)min(16, rc - row0) * rowb);
            base[s] = (uint32_t)min(c, rc - 1 - row0) * rowb;
            ri[s] = 0;
        }
    }

    const Cst cst;
    // Activation staging of this slice, one step at a time.
    uint8_t *sl = smem + kw * C::kSlice;
    const int tid = rw * kWave + lane;
    const __amdgpu_buffer_rsrc_t xr = buf_rsrc(p.xq, (uint32_t)p.M * (uint32_t)K);
    const __amdgpu_buffer_rsrc_t dr = buf_rsrc(p.xd, (uint32_t)p.M * (uint32_t)ngk * 4u);
    const __amdgpu_buffer_rsrc_t sr = buf_rsrc(p.xs, (uint32_t)p.M * (uint32_t)ngk * 4u);
    // Chunk n of this thread: 16 codes j of a token's step; scale n: group g of
    // a token.  Offsets are kept, the step's own comes as a scalar: rows past M
    // repeat the last one and have scale 0; so have the groups past K of a
    // partial last step (Q8_0), whose codes are read as zeros.
    uint32_t aoff[C::NC], soff[C::NSC];
    int adst[C::NC], sdst[C::NSC], xdst[T::kMin ? C::NSC : 1];
#pragma unroll
    for (int n = 0; n < C::NC; ++n) {
        const int id = n * NTH + tid, j = id % (2 * GS), tok = id / (2 * GS);
        aoff[n] = id < C::kChunks ? (uint32_t)min(tok, p.M - 1) * (uint32_t)K + 16u * (uint32_t)j : kPast;
        adst[n] = ((j >> 1) * NT + (tok >> 4)) * (kWave * C::FB);
    }
#pragma unroll
    for (int n = 0; n < C::NSC; ++n) {
        const int id = n * NTH + tid, g = id % GS, tok = id / GS;
        soff[n] = tok < p.M ? ((uint32_t)tok * (uint32_t)ngk + (uint32_t)g) * 4u : kPast;
        sdst[n] = (g * TOK + tok) * 4;
        if constexpr (T::kMin) xdst[n] = ((tok >> 4) * 48 + (tok & 15)) * 16 + 2 * g;
    }
    u4 ra[C::DP][C::NC];
    uint32_t rd[C::DP][C::NSC], rx[C::DP][C::NSC];
    auto issue = [&](int step, auto set) __attribute__((always_inline)) {  // step: GS groups from group step * GS
        constexpr int R = decltype(set)::value % C::DP;
        // steps past the last one (loaded ahead, not used) repeat it
        const uint32_t g0 = (uint32_t)(min(step, (ngk - 1) / GS) * GS);
#pragma unroll
        for (int n = 0; n < C::NC; ++n) {
            uint32_t o = aoff[n];
            if constexpr (T::kRagged) o = 32 * (int)g0 + 16 * ((n * NTH + tid) % (2 * GS)) < K ? o : kPast;
            ra[R][n] = ld16<0>(xr, o, 32u * g0);
        }
#pragma unroll
        for (int n = 0; n < C::NSC; ++n) {
            uint32_t o = soff[n];
            if constexpr (T::kRagged) o = (int)g0 + (n * NTH + tid) % GS < ngk ? o : kPast;
            rd[R][n] = bld_u32<0>(dr, o, 4u * g0);
            if constexpr (T::kMin) rx[R][n] = bld_u32<0>(sr, o, 4u * g0);
        }
    };
    auto commit = [&](int buf, auto st, int ubuf) __attribute__((always_inline)) {
        constexpr int R = decltype(st)::value % C::DP;
        uint8_t *xc = sl + buf * C::kCodes, *dT = sl + C::oDx + buf * C::kDx;
#pragma unroll
        for (int n = 0; n < C::NC; ++n)
            if (C::kChunks % NTH == 0 || n * NTH + tid < C::kChunks)
                store_codes<T>(xc + adst[n], ra[R][n], (n * NTH + tid) % (2 * GS), (n * NTH + tid) / (2 * GS) & 15, cst);
#pragma unroll
        for (int n = 0; n < C::NSC; ++n) {
            if (C::kScales % NTH == 0 || n * NTH + tid < C::kScales) {
                const float d = __uint_as_float(rd[R][n]);
                *(float *)(dT + sdst[n]) = d;
                if constexpr (T::kMin) {
                    // dx sum(codes) as three bf16 values: each the top half of
                    // what is left, and the rest (below 2^-7 of it, exact) moved
                    // 2^7 up, so that the smallest factors keep their last bits
                    const int sum = (int)(int16_t)(rx[R][n] & 0xffffu) + (int)(int16_t)(rx[R][n] >> 16);
                    const float a = d * (float)sum;
                    constexpr float up = (float)(1 << kMinStep);
                    const float r1 = (a - __uint_as_float(__float_as_uint(a) & 0xffff0000u)) * up;
                    const float r2 = (r1 - __uint_as_float(__float_as_uint(r1) & 0xffff0000u)) * up;
                    uint8_t *ax = sl + C::oAux + ubuf * C::kAux + xdst[n] + 2 * decltype(st)::value * GS;
                    *(uint16_t *)ax = (uint16_t)(__float_as_uint(a) >> 16);
                    *(uint16_t *)(ax + 16 * 16) = (uint16_t)(__float_as_uint(r1) >> 16);
                    *(uint16_t *)(ax + 32 * 16) = (uint16_t)(__float_as_uint(r2) >> 16);
                }
            }
        }
    };

    f4 *red = (f4 *)smem;  // [KW][nsets][NT][64]
    // The loop over the slice for a wave of NS sets (a compile-time count: one
    // straight-line step, so that the compiler can move the operand reads of a
    // group ahead of the previous group's arithmetic).
    auto run = [&](auto nsc) __attribute__((always_inline)) {
    constexpr int NS = decltype(nsc)::value;
    typename T::Reg w[NS];
    // Sums by unit (ab), by slice (acc) and, in waves of one set, by runs of 4
    // units (hi): short chains, so that the fp32 sums round no worse than the
    // 16-token kernel's, which splits K over more waves (5120 x 17408 at M = 64
    // against 64 bits, 16-token kernel / without / with: Q8_0 1.6e-7 / 2.2e-7 /
    // 9.5e-8, Q6_K 9.9e-8 / 1.02e-7 / 9.2e-8).
    constexpr bool kHi = RSM == 1 && !T::kMin;
    f4 acc[NS][NT], ab[NS][NT], hi[kHi ? NT : 1];
#pragma unroll
    for (int t = 0; t < (kHi ? NT : 1); ++t) hi[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[s][t] = f4{0.f, 0.f, 0.f, 0.f};
    int xo[GS];  // this lane's operand in a fragment of the step's group g
#pragma unroll
    for (int g = 0; g < GS; ++g) xo[g] = (16 * q + (c ^ (2 * g + (q >> 1)))) * C::FB;
    int el[4];  // byte lane index of row 4 q + e, for ds_bpermute
#pragma unroll
    for (int e = 0; e < 4; ++e) el[e] = 4 * (4 * q + e);

    // One step: GS groups of unit u from buffer `buf`, then the next unit's
    // weights for these groups into the registers just used.
    auto compute = [&](auto st, int u, int buf, int ubuf) __attribute__((always_inline)) {
        constexpr int ST = decltype(st)::value;
        const uint8_t *xc = sl + buf * C::kCodes;
        const float *dT = (const float *)(sl + C::oDx + buf * C::kDx);
        unroll<GS>([&](auto gi) __attribute__((always_inline)) {
            constexpr int GI = decltype(gi)::value, G = ST * GS + GI;
            float dx[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) dx[t] = dT[GI * TOK + 16 * t + c];
            if constexpr (T::kF16) {
                h8 b[NT];
#pragma unroll
                for (int t = 0; t < NT; ++t) b[t] = *(const h8 *)(xc + (GI * NT + t) * (kWave * 16) + xo[GI]);
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                        const auto a = T::template operand<G>(w[s], q, cst);
                        f4 d[NT];
#pragma unroll
                        for (int t = 0; t < NT; ++t)
                            d[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.a, b[t], f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                        if constexpr (T::kTwo) {
#pragma unroll
                            for (int t = 0; t < NT; ++t) d[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.b, b[t], d[t], 0, 0, 0);
                        }
#pragma unroll
                        for (int t = 0; t < NT; ++t)
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                ab[s][t][e] = G == 0 ? dx[t] * d[t][e] : __builtin_fmaf(dx[t], d[t][e], ab[s][t][e]);
                        // kept here: the compiler otherwise sinks these sums to
                        // the unit's end and spills the group sums until then
#pragma unroll
                        for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(ab[s][t]));
                    }
            } else {
                long b[NT];
#pragma unroll
                for (int t = 0; t < NT; ++t) b[t] = __builtin_bit_cast(long, *(const u2 *)(xc + (GI * NT + t) * (kWave * 8) + xo[GI]));
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                        const long a = T::template operand<G>(w[s]);
                        const float f = T::template factor<G, LAYOUT>(w[s], u, p.rb);
                        i4 d[NT];
#pragma unroll
                        for (int t = 0; t < NT; ++t)
                            d[t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b[t], i4{0, 0, 0, 0}, 0, 0, 0);
                        float fe[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) fe[e] = bperm(el[e], f);
#pragma unroll
                        for (int t = 0; t < NT; ++t)
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                ab[s][t][e] = G == 0 ? fe[e] * dx[t] * (float)d[t][e]
                                                     : __builtin_fmaf(fe[e] * dx[t], (float)d[t][e], ab[s][t][e]);
#pragma unroll
                        for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(ab[s][t]));
                    }
            }
        });
        if constexpr (T::kF16) {  // the unit's d (and dmin) terms
            if constexpr (ST == NST - 1) {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                    const uint32_t dw = T::dword(w[s]);
                    float d[4], dm[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t v = bperm(el[e], dw);
                        d[e] = f16_bits_to_f32(v);
                        dm[e] = f16_bits_to_f32(v >> 16);
                    }
                    if constexpr (T::kMin) {
                        const b8 a = T::min_operand(w[s], q);
                        const uint8_t *ax = sl + C::oAux + ubuf * C::kAux + ((q < 3 ? 16 * q : 0) + c) * 16;
                        f4 m[NT];
#pragma unroll
                        for (int t = 0; t < NT; ++t)
                            m[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, *(const b8 *)(ax + t * 48 * 16),
                                                                           f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                        for (int t = 0; t < NT; ++t)
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                acc[s][t][e] = __builtin_fmaf(d[e], ab[s][t][e], acc[s][t][e]);
                                acc[s][t][e] = __builtin_fmaf(-dm[e], m[t][e], acc[s][t][e]);
                            }
                    } else {
#pragma unroll
                        for (int t = 0; t < NT; ++t)
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[s][t][e] = __builtin_fmaf(d[e], ab[s][t][e], acc[s][t][e]);
                    }
                }
            }
        } else {
            if constexpr (ST == NST - 1) {
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[s][t] += ab[s][t];
            }
        }
    };

    // The next unit's weights for the groups just used.
    auto reload = [&](auto st, int u) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < NS; ++s)
            T::template load<LAYOUT, decltype(st)::value * GS>(w[s], wp[s], rs[s], base[s], ri[s], q, min(u + 1, ub - 1), p.rb);
    };

    if (ua < ub) {
        issue(ua * NST, Int<0>{});
        if constexpr (C::DP == 2) issue(ua * NST + 1, Int<1>{});
#pragma unroll
        for (int s = 0; s < NS; ++s)
            unroll<NST>([&](auto st) __attribute__((always_inline)) {
                    T::template load<LAYOUT, decltype(st)::value * GS>(w[s], wp[s], rs[s], base[s], ri[s], q, ua, p.rb);
                });
        commit(0, Int<0>{}, 0);
        issue(ua * NST + C::DP, Int<C::DP>{});
    }
    if constexpr (RW > 1) __syncthreads();
    else wave_order();
    // Step i of the slice computes from buffer i % 2 while step i + 1 is
    // written to the other one (last read a barrier ago); a one-wave slice has
    // one buffer, written after the step that reads it (wave_order).  Every wave
    // passes umax * NST barriers.
    for (int k = 0; k < umax; ++k) {
        const int u = ua + k;
        const bool on = u < ub;
        if constexpr (kHi)
            if (k % 4 == 0) {
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    hi[t] += acc[0][t];
                    acc[0][t] = f4{0.f, 0.f, 0.f, 0.f};
                }
            }
        unroll<NST>([&](auto st) __attribute__((always_inline)) {
            constexpr int ST = decltype(st)::value;
            constexpr int NX = (ST + 1) % NST;
            const int step = u * NST + ST, ubuf = C::NB == 2 ? k & 1 : 0;
            const int nub = C::NB == 2 ? (k + (ST + 1) / NST) & 1 : 0;
            if (on) {
                if constexpr (RW > 1) {
                    commit((ST + 1) & 1, Int<NX>{}, nub);  // NST is even: a step's buffer is its parity in the unit
                    issue(step + 1 + C::DP, Int<ST + 1 + C::DP>{});
                    compute(st, u, ST & 1, ubuf);
                    reload(st, u);
                } else {
                    compute(st, u, 0, ubuf);
                    wave_order();
                    commit(0, Int<NX>{}, nub);
                    if constexpr (T::kInterleave) wave_order();
                    issue(step + 1 + C::DP, Int<ST + 1 + C::DP>{});
                    if constexpr (T::kRagged) wave_order();
                    reload(st, u);
                    if constexpr (T::kF16) wave_order();
                }
            }
            if constexpr (RW > 1) __syncthreads();
        });
    }

    // Partials to LDS by slice and set, then the sum in slice order.
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int t = 0; t < NT; ++t)
            if (s < ns) red[((kw * nsets + f0 + s) * NT + t) * kWave + lane] = kHi ? hi[kHi ? t : 0] + acc[s][t] : acc[s][t];
    };
    // A wave without a set (an odd set count over two row waves) stages and
    // passes the barriers with the others, on a set in range, and drops its sums.
    if (ns <= 1) run(Int<1>{});
    else if constexpr (RSM > 1) {
        if (ns == 2) run(Int<2>{});
        else run(Int<3>{});
    }
    __syncthreads();
    const int per = nsets * NT * kWave;
    for (int idx = (int)threadIdx.x; idx < per; idx += kWave * C::W) {
        f4 v = red[idx];
#pragma unroll
        for (int k = 1; k < KW; ++k) v += red[k * per + idx];
        const int ln = idx % kWave, t = idx / kWave % NT, gs = s0 + idx / (kWave * NT);
        int mi = 0;
#pragma unroll
        for (int k = 1; k < kMaxMulti; ++k)
            if (k < p.nmat && gs >= p.wg_start[k]) mi = k;
        const int rc = p.rc[mi], row = (gs - p.wg_start[mi]) * 16 + 4 * (ln >> 4), tok = 16 * t + (ln & 15);
        if (tok < p.M) {
            const size_t o = (size_t)tok * rc + row;
            float *y = p.Y[mi] + o;
            const float *r = p.res[mi] ? p.res[mi] + o : nullptr;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (row + e < rc) y[e] = v[e] * (float)(1 << T::kDown) + (r ? r[e] : 0.f);
        }
    }
}

template <class T, int NT, class SH, int LAYOUT>
hipError_t launch_wide_t(const MatmulMultiParams &p, int grid, hipStream_t s) {
    hipLaunchKernelGGL((k_matmul_wide<T, NT, SH, LAYOUT>), dim3(grid), dim3(kWave * SH::W), (Wide<T, NT, SH>::kLds), s, p);
    return hipGetLastError();
}

using ShapeFew = Shape<1, 8, 1>;
using ShapePair = Shape<2, 4, 1>;
using ShapeMid = Shape<2, 4, 3>;
using ShapeMany = Shape<4, 2, 3>;

// Grid and split by the number S of 16-row sets per CU.
template <class T, int NT, int LAYOUT>
hipError_t launch_wide_nt(MatmulMultiParams p, hipStream_t s) {
    int S = 0;
    for (int i = 0; i < p.nmat; ++i) {
        p.wg_start[i] = S;
        S += (p.rc[i] + 15) / 16;
    }
    p.wg_start[p.nmat] = S;
    const int cus = cu_count();
    auto grid = [&](int max_sets) {  // whole rounds of one workgroup per CU
        const int r = (S + max_sets * cus - 1) / (max_sets * cus);
        return std::min(S, r * cus);
    };
    if (S <= cus) return launch_wide_t<T, NT, ShapeFew, LAYOUT>(p, S, s);
    if (S <= 2 * cus) return launch_wide_t<T, NT, ShapePair, LAYOUT>(p, (S + 1) / 2, s);
    if (S <= 6 * cus) return launch_wide_t<T, NT, ShapeMid, LAYOUT>(p, grid(Wide<T, NT, ShapeMid>::kMaxSets), s);
    return launch_wide_t<T, NT, ShapeMany, LAYOUT>(p, grid(Wide<T, NT, ShapeMany>::kMaxSets), s);
}

template <class T, int LAYOUT>
hipError_t launch_wide_m(const MatmulMultiParams &p, hipStream_t s) {
    switch ((p.M + 15) / 16) {
        case 1:  // fewer than 17 rows: only for types the 16-token kernel does not take
            if constexpr (!T::kF16 && LAYOUT == M27Q_LAYOUT_GGUF) return launch_wide_nt<T, 1, LAYOUT>(p, s);
            else return hipErrorInvalidValue;
        case 2: return launch_wide_nt<T, 2, LAYOUT>(p, s);
        case 3: return launch_wide_nt<T, 3, LAYOUT>(p, s);
        case 4: return launch_wide_nt<T, 4, LAYOUT>(p, s);
        default: return hipErrorInvalidValue;
    }
}

template <class T>
hipError_t launch_wide_l(int layout, const MatmulMultiParams &p, hipStream_t s) {
    return layout == M27Q_LAYOUT_TILED ? launch_wide_m<T, M27Q_LAYOUT_TILED>(p, s) : launch_wide_m<T, M27Q_LAYOUT_GGUF>(p, s);
}

}  // namespace
}  // namespace m27q
