// mx4_device.h -- device-side building blocks shared by the gfx950 kernels.
//
// MXFP4 storage (engine/src/mxfp4.rs:5-8, :27-33): weight row r of width K is
// K/2 packed bytes (element 2j in the low nibble of byte j, 2j+1 in the high
// nibble) plus K/32 E8M0 scale bytes. One 32-element block is 16 contiguous
// bytes -- exactly one 128-bit load -- and one scale byte.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mx4 {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWave = 64;

// Buffer resource over [base, base + bytes): loads past the end return zero
// without touching memory, so tail loads can be issued unconditionally.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

// Greedy argmax of the logits (engine/src/model.rs:288-296: the first index of
// the maximum under a strict `>` scan from index 0) as one unsigned 64-bit key
// per row, so that the largest key is the answer: the value in an order-
// preserving integer form above the complemented row, so equal values favour
// the lower row. +0 and -0 compare equal in the scan, so both map to +0. A NaN
// is never greater than anything and nothing is greater than a NaN: a NaN at
// row 0 is the answer (key = all ones), a NaN elsewhere never is (key 0).
__device__ __forceinline__ uint64_t argmax_key(float v, uint32_t row) {
    if (v != v) return row == 0 ? ~0ull : 0ull;
    uint32_t b = __float_as_uint(v == 0.0f ? 0.0f : v);
    b = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    return ((uint64_t)b << 32) | (uint32_t)~row;
}

__device__ __forceinline__ uint64_t max_u64(uint64_t a, uint64_t b) { return a > b ? a : b; }

// An f32 activation as three bf16 terms, hi + mid + lo == x, for exact
// products on the bf16 matrix cores. Each term is cut from the bits
// (truncation, never rounding up): hi keeps the top 8 significant bits of x,
// mid the top 8 of the remainder, lo what is left (at most 8 bits, exact),
// so no finite x yields an infinite term (rounding to nearest would turn
// |x| >= 0x7F7F8000 into a bf16 inf and the remainder into inf - inf = NaN).
// A non-finite x stays in hi (a NaN keeps its quiet bit in the upper half)
// with mid = lo = 0, so its products are the f32 products of the reference's
// loop: +-inf, or NaN against a zero weight.
__device__ __forceinline__ void split3_bf16(float v, __bf16& hi, __bf16& mid, __bf16& lo) {
    const uint32_t u = __float_as_uint(v);
    const uint32_t hb = (u & 0xFFFF0000u) | (v != v ? 0x00400000u : 0u);
    float r1 = v - __uint_as_float(hb);  // NaN exactly when x is not finite
    r1 = r1 == r1 ? r1 : 0.0f;
    const uint32_t mb = __float_as_uint(r1) & 0xFFFF0000u;
    const float r2 = r1 - __uint_as_float(mb);
    hi = __builtin_bit_cast(__bf16, (uint16_t)(hb >> 16));
    mid = __builtin_bit_cast(__bf16, (uint16_t)(mb >> 16));
    lo = (__bf16)r2;
}

// The three terms of eight finite values, packed as MFMA operands: 5 operations
// a value where split3_bf16 takes twice that (its care for inf and NaN).
__device__ __forceinline__ void split3_finite(const u32x4 lo4, const u32x4 hi4, bf16x8& hi, bf16x8& mid, bf16x8& lo,
                                              float* bad = nullptr) {
    uint32_t h[4], m[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        uint32_t r[2], d[2];
        float rest[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const uint32_t u = p < 2 ? lo4[2 * p + e] : hi4[2 * p + e - 4];
            const float r1 = __uint_as_float(u) - __uint_as_float(u & 0xFFFF0000u);  // NaN if u is not finite
            r[e] = __float_as_uint(r1);
            rest[e] = r1 - __uint_as_float(r[e] & 0xFFFF0000u);
            d[e] = u;
            lo[2 * p + e] = (__bf16)rest[e];
        }
        if (bad) *bad = __builtin_fmaf(rest[0], rest[1], *bad);
        // the upper halves of a pair: element 2 p below element 2 p + 1
        h[p] = __builtin_amdgcn_perm(d[1], d[0], 0x07060302u);
        m[p] = __builtin_amdgcn_perm(r[1], r[0], 0x07060302u);
    }
    hi = __builtin_bit_cast(bf16x8, u32x4{h[0], h[1], h[2], h[3]});
    mid = __builtin_bit_cast(bf16x8, u32x4{m[0], m[1], m[2], m[3]});
}

// The terms of any eight values, by split3_bf16.
__device__ __forceinline__ void split3_careful(const u32x4 a, const u32x4 b, bf16x8& hi, bf16x8& mid, bf16x8& lo) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        __bf16 h, m, l;
        split3_bf16(__uint_as_float(e < 4 ? a[e] : b[e - 4]), h, m, l);
        hi[e] = h;
        mid[e] = m;
        lo[e] = l;
    }
}

// The terms of eight values, finite or not: the wave takes the short form and,
// where some lane has an inf or a NaN (or the check, a NaN from either on,
// overflows), the careful one.
__device__ __forceinline__ void split3x8(const u32x4 a, const u32x4 b, bf16x8& hi, bf16x8& mid, bf16x8& lo) {
    float bad = 0.0f;
    split3_finite(a, b, hi, mid, lo, &bad);
    if (__any(bad != bad)) split3_careful(a, b, hi, mid, lo);
}

// Eight E2M1 weights of a packed word, the block's scale folded in (bytes 2..252:
// exact in bf16).
__device__ __forceinline__ bf16x8 decode8(uint32_t word, float sc) {
    const bf16x2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, sc, 0);
    const bf16x2 p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, sc, 1);
    const bf16x2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, sc, 2);
    const bf16x2 p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, sc, 3);
    bf16x8 r;
    r[0] = p0[0]; r[1] = p0[1]; r[2] = p1[0]; r[3] = p1[1];
    r[4] = p2[0]; r[5] = p2[1]; r[6] = p3[0]; r[7] = p3[1];
    return r;
}

constexpr uint32_t kPastEnd = 0x80000000u;  // past every buffer resource: a load there returns zeros
typedef double f64x16 __attribute__((ext_vector_type(16)));

// Values below 2^-110 lose bits as three bf16 terms, whose least is 2^-133. The
// kernels for any width and for bf16 weights lose none all the same: where a lane
// holds, in a step of the reduction, only such values (zeros apart), or an inf or
// a NaN, they do their work again with the careful split and two passes a step.
// The first pass has the other lanes' values, the second those tiny ones, 2^64
// times as large (every bit of an f32 then fits, and no product overflows: 2^-36
// times weights below 2^128), and adds 2^-64 of its sum. (Beside a value above
// 2^-100 a tiny one's bits below 2^-133 are 2^-33 of that value.) `most` is the
// largest magnitude of a lane's values in the step, NaN if one of them is.
constexpr double kTinyDown = 0x1p-64;
__device__ __forceinline__ void take_most(const u32x4 v, float& most) {  // two instructions
#pragma unroll
    for (int p = 0; p < 4; p += 2)
        most = __builtin_elementwise_maximum(__builtin_fabsf(__uint_as_float(v[p])),
                                             __builtin_elementwise_maximum(__builtin_fabsf(__uint_as_float(v[p + 1])), most));
}
__device__ __forceinline__ bool all_tiny(float most) { return (most != 0.0f) & (most < 0x1p-100f); }
__device__ __forceinline__ bool plain(float most) {  // the short split has it
    return (most == 0.0f) | ((most >= 0x1p-100f) & (most < __builtin_inff()));
}
// The terms of a pass's share of eight values; `tiny`: the lane's all_tiny.
__device__ __forceinline__ void split3_pass(int pass, bool tiny, u32x4 a, u32x4 b, bf16x8& hi, bf16x8& mid, bf16x8& lo) {
    const float scale = pass ? 0x1p64f : 1.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        a[e] = tiny == (pass != 0) ? __float_as_uint(__uint_as_float(a[e]) * scale) : 0u;
        b[e] = tiny == (pass != 0) ? __float_as_uint(__uint_as_float(b[e]) * scale) : 0u;
    }
    split3_careful(a, b, hi, mid, lo);
}

__device__ __forceinline__ uint64_t wave_max_u64(uint64_t m) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const uint32_t lo = __shfl_xor((uint32_t)m, off, kWave), hi = __shfl_xor((uint32_t)(m >> 32), off, kWave);
        m = max_u64(m, ((uint64_t)hi << 32) | lo);
    }
    return m;
}

// E2M1 magnitude levels (engine/src/mxfp4.rs:3).
__device__ __forceinline__ float level_of(uint32_t code) {
    // Built from bits like gpu.metal's mxfp4_level, independent of a table:
    // m = code & 7; m == 0 -> 0; m == 1 -> 0.5; else 2^(m/2 - 1) * (1 + (m & 1) / 2).
    uint32_t m = code & 7u;
    uint32_t bits = m == 0 ? 0u : (m == 1 ? 0x3f000000u : (((126u + (m >> 1)) << 23) | ((m & 1u) << 22)));
    return __uint_as_float(bits | ((code & 8u) << 28));
}

// 2^(s - 127) for an E8M0 byte s in [0, 254], exact (2^-127 is the subnormal
// 0x00400000; f32 denormals are preserved on gfx950 by default).
__device__ __forceinline__ float e8m0_to_f32(uint32_t s) {
    return __builtin_amdgcn_ldexpf(1.0f, (int)s - 127);
}

// One decoded element, bit-exact with engine/src/mxfp4.rs:27-33:
// LEVELS[c & 7] * 2^(s-127), negated when c & 8.
__device__ __forceinline__ float decode_exact(uint32_t code, uint32_t s) {
    return level_of(code) * e8m0_to_f32(s);
}

// Two E2M1 codes from byte `sel` of `word` -> two f32 levels (scale 1), using
// gfx950's hardware converter. Element order: low nibble -> .x, high -> .y.
template <int SEL>
__device__ __forceinline__ f32x2 cvt_fp4x2_f32(uint32_t word) {
    return __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, SEL);
}
template <int SEL>
__device__ __forceinline__ bf16x2 cvt_fp4x2_bf16(uint32_t word) {
    return __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, 1.0f, SEL);
}

__device__ __forceinline__ uint32_t as_u32(bf16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ bf16x2 as_bf16x2(uint32_t v) { return __builtin_bit_cast(bf16x2, v); }

// Sum of 32 products sum_i x[i] * level(code_i) for one MX block whose 16
// packed bytes are w (4 dwords), x given as 16 bf16 pairs in element order.
__device__ __forceinline__ float block_dot_bf16(const u32x4 w, const uint32_t* xp) {
    float acc = 0.0f;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        acc = __builtin_amdgcn_fdot2_f32_bf16(cvt_fp4x2_bf16<0>(w[d]), as_bf16x2(xp[4 * d + 0]), acc, false);
        acc = __builtin_amdgcn_fdot2_f32_bf16(cvt_fp4x2_bf16<1>(w[d]), as_bf16x2(xp[4 * d + 1]), acc, false);
        acc = __builtin_amdgcn_fdot2_f32_bf16(cvt_fp4x2_bf16<2>(w[d]), as_bf16x2(xp[4 * d + 2]), acc, false);
        acc = __builtin_amdgcn_fdot2_f32_bf16(cvt_fp4x2_bf16<3>(w[d]), as_bf16x2(xp[4 * d + 3]), acc, false);
    }
    return acc;
}

// The same with f32 activations: products x * level are exact in f32 before
// each FMA's single rounding.
__device__ __forceinline__ float block_dot_f32(const u32x4 w, const float* x) {
    float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        f32x2 v0 = cvt_fp4x2_f32<0>(w[d]);
        f32x2 v1 = cvt_fp4x2_f32<1>(w[d]);
        f32x2 v2 = cvt_fp4x2_f32<2>(w[d]);
        f32x2 v3 = cvt_fp4x2_f32<3>(w[d]);
        a0 = __builtin_fmaf(x[8 * d + 0], v0.x, a0);
        a1 = __builtin_fmaf(x[8 * d + 1], v0.y, a1);
        a0 = __builtin_fmaf(x[8 * d + 2], v1.x, a0);
        a1 = __builtin_fmaf(x[8 * d + 3], v1.y, a1);
        a0 = __builtin_fmaf(x[8 * d + 4], v2.x, a0);
        a1 = __builtin_fmaf(x[8 * d + 5], v2.y, a1);
        a0 = __builtin_fmaf(x[8 * d + 6], v3.x, a0);
        a1 = __builtin_fmaf(x[8 * d + 7], v3.y, a1);
    }
    return a0 + a1;
}

// Wave64 sum; every lane receives the total.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}
// Wave64 sums of four values at once: every quarter of 16 lanes receives the sum
// of one, lane/16 its index. Half of what is left goes over with each of the first
// two steps, 7 exchanges for 24.
__device__ __forceinline__ double wave_sum4(const double (&v)[4], uint32_t lane) {
    const bool up = lane & 32u, odd = lane & 16u;
    double t[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) t[i] = (up ? v[2 + i] : v[i]) + __shfl_xor(up ? v[i] : v[2 + i], 32, kWave);
    double r = (odd ? t[1] : t[0]) + __shfl_xor(odd ? t[0] : t[1], 16, kWave);
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) r += __shfl_xor(r, off, kWave);
    return r;
}

__device__ __forceinline__ u32x4 load_u32x4(const uint8_t* p) {
    return *reinterpret_cast<const u32x4*>(p);
}

__device__ __forceinline__ u32x4 load_u32x4_nt(const uint8_t* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}

// bf16 <-> f32 (engine/src/lib.rs:74-76 for the widening direction)
__device__ __forceinline__ float bf16_bits_to_f32(uint32_t bits16) { return __uint_as_float(bits16 << 16); }

__device__ __forceinline__ uint32_t f32_to_bf16_bits(float v) {
    uint32_t u = __float_as_uint(v);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// ---------------------------------------------------------------- wave sums

// Sum R per-lane values over the 64 lanes of a wave in log2(64) exchange
// stages. In the first log2(R) stages each lane keeps half of its values and
// sends the other half to its partner, so the R totals cost 63 + R - 1
// additions instead of R * 63. The exchanges stay in the VALU: DPP
// row_half_mirror (partner l ^ 7), quad permutations (l ^ 1, l ^ 2) and
// row_ror:8 (l ^ 8) within rows of 16 lanes, then v_permlane16_swap (l ^ 16)
// and v_permlane32_swap (l ^ 32). The half-mirror stage goes first: it flips
// lane bits 0-2 together, which is a valid butterfly partner only while no
// earlier stage has made lanes differ in bits 0-1. The halving stages select
// by lane bits 2, 0, 1 in that order, so lane l ends with the total of row
// reduced_row_of_lane<R>(l).
template <int CTRL>
__device__ __forceinline__ float dpp_partner(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

template <int CTRL, int R>
__device__ __forceinline__ void dpp_stage(float (&v)[R], int& n, bool upper) {
    if (n > 1) {
        const int half = n / 2;
#pragma unroll
        for (int i = 0; i < R / 2; ++i) {
            if (i < half) {
                const float send = upper ? v[i] : v[i + half];
                const float keep = upper ? v[i + half] : v[i];
                v[i] = keep + dpp_partner<CTRL>(send);
            }
        }
        n = half;
    } else {
        v[0] += dpp_partner<CTRL>(v[0]);
    }
}

// Exchange across rows (SWAP = 16) or half-waves (SWAP = 32). After
// permlane*_swap(a, b) lane l holds {own a, partner's a} if it is the lower
// partner and {partner's b, own b} if it is the upper one, so the sum of the
// pair is keep + partner's send in both cases.
template <int SWAP>
__device__ __forceinline__ float swap_sum(float lower_keeps, float upper_keeps) {
    const auto p = SWAP == 16
                       ? __builtin_amdgcn_permlane16_swap(__float_as_uint(lower_keeps), __float_as_uint(upper_keeps), false, false)
                       : __builtin_amdgcn_permlane32_swap(__float_as_uint(lower_keeps), __float_as_uint(upper_keeps), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}

template <int SWAP, int R>
__device__ __forceinline__ void swap_stage(float (&v)[R], int& n) {
    if (n > 1) {
        const int half = n / 2;
#pragma unroll
        for (int i = 0; i < R / 2; ++i)
            if (i < half) v[i] = swap_sum<SWAP>(v[i], v[i + half]);
        n = half;
    } else {
        v[0] = swap_sum<SWAP>(v[0], v[0]);
    }
}

constexpr int kDppHalfMirror = 0x141, kDppQuadXor1 = 0xB1, kDppQuadXor2 = 0x4E, kDppRowRor8 = 0x128;

// SUB rows side by side: the sum over each 64 / SUB lanes only (SUB 2 or 4;
// lane l's row is then reduced_row_of_lane<R>(l) of its part of the wave).
template <int R, int SUB = 1>
__device__ __forceinline__ float wave_reduce_rows(float (&v)[R], uint32_t lane) {
    int n = R;
    dpp_stage<kDppHalfMirror, R>(v, n, (lane & 4) != 0);
    dpp_stage<kDppQuadXor1, R>(v, n, (lane & 1) != 0);
    dpp_stage<kDppQuadXor2, R>(v, n, (lane & 2) != 0);
    dpp_stage<kDppRowRor8, R>(v, n, (lane & 8) != 0);
    if constexpr (SUB < 4) swap_stage<16, R>(v, n);
    if constexpr (SUB < 2) swap_stage<32, R>(v, n);
    return v[0];
}

// Row whose total lane `lane` holds after wave_reduce_rows<R> (R <= 8): the
// halving stages take the upper half when lane bit 2, then 0, then 1 is set.
template <int R>
__device__ __forceinline__ uint32_t reduced_row_of_lane(uint32_t lane) {
    static_assert(R == 1 || R == 2 || R == 4 || R == 8, "rows per team");
    uint32_t row = 0;
    if constexpr (R >= 2) row += (lane & 4) ? R / 2 : 0;
    if constexpr (R >= 4) row += (lane & 1) ? R / 4 : 0;
    if constexpr (R >= 8) row += (lane & 2) ? 1 : 0;
    return row;
}

// One lane per row writes its total: lane bits outside the row-select bits are zero.
template <int R>
__device__ __forceinline__ bool row_writer(uint32_t lane) {
    constexpr uint32_t row_bits = R >= 8 ? 7u : R == 4 ? 5u : R == 2 ? 4u : 0u;
    return (lane & ~row_bits) == 0;
}

// ---------------------------------------------------------------- inf weights

// bf16 weights and f32 activations: an inf weight times a zero middle or low term
// is a NaN that the reference's product of the whole value is not. An output that
// came out as NaN is summed again from whole values, but only where that can be
// the reason (its token row has no NaN, and its weight row an inf and no NaN):
// summing every NaN again, one output after the other, made a call whose
// activations held one take a hundred times as long. Rows of whole 16-byte pieces.
__device__ __forceinline__ bool inf_and_no_nan(const uint16_t* w, uint32_t len, uint32_t lane) {
    bool inf = false, nan = false;
#pragma unroll 4
    for (uint32_t e = 8 * lane; e < len; e += 512) {
        const u32x4 v = load_u32x4(reinterpret_cast<const uint8_t*>(w + e));
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const uint32_t a = v[d] & 0x7fffu, b = (v[d] >> 16) & 0x7fffu;
            inf |= (a == 0x7f80u) | (b == 0x7f80u);
            nan |= (a > 0x7f80u) | (b > 0x7f80u);
        }
    }
    return __any(inf) && !__any(nan);
}
__device__ __forceinline__ float dot_whole(const float* x, const uint16_t* w, uint32_t len, uint32_t lane) {
    float p = 0.0f;
#pragma unroll 2
    for (uint32_t e = 8 * lane; e < len; e += 512) {
        const u32x4 v = load_u32x4(reinterpret_cast<const uint8_t*>(w + e));
        const f32x4 x0 = *reinterpret_cast<const f32x4*>(x + e), x1 = *reinterpret_cast<const f32x4*>(x + e + 4);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const float a = d < 2 ? x0[2 * d] : x1[2 * d - 4], b = d < 2 ? x0[2 * d + 1] : x1[2 * d - 3];
            p = __builtin_fmaf(a, bf16_bits_to_f32(v[d] & 0xffffu), p);
            p = __builtin_fmaf(b, bf16_bits_to_f32(v[d] >> 16), p);
        }
    }
    return wave_sum(p);
}

// ---------------------------------------------------------------- LDS pipelines

// Does any of the NW waves of the workgroup say so (each with one wave-wide
// answer)? Over LDS that no wave has a use for any more, by the first barrier.
template <int NW>
__device__ __forceinline__ bool workgroup_any(bool mine, uint32_t* words, uint32_t wave) {
    __syncthreads();
    if (threadIdx.x % 64 == 0) words[wave] = mine;
    __syncthreads();
    uint32_t any = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) any |= words[w];
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(any) != 0;
}

// LDS barrier that does not wait for outstanding global loads (the next
// stage's prefetch stays in flight across it).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

typedef __attribute__((address_space(3))) void* lds_ptr;

// Direct-to-LDS buffer loads of 16 or 4 bytes per lane: lane l's bytes land
// at dst + l * size. (Only the device pass sees the builtin: the host pass
// checks the size against its own target, rejects 16, and would then drop
// the kernels' launch stubs without a word.)
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, lds_ptr dst, uint32_t voffset) {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, voffset, 0, 0, 0);
#else
    (void)r; (void)dst; (void)voffset;
#endif
}
__device__ __forceinline__ void load_lds4(__amdgpu_buffer_rsrc_t r, lds_ptr dst, uint32_t voffset) {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 4, voffset, 0, 0, 0);
#else
    (void)r; (void)dst; (void)voffset;
#endif
}

}  // namespace mx4
