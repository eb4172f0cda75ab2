// Device helpers shared by the row quantisers (quant_rows.hip) and the fused producer +
// quantiser kernels (fused_rows.hip): abs-max reduction, the reference's scale rule and the
// leaf quantisers for int8 / OCP e4m3fn / OCP e5m2.
#pragma once

#include <type_traits>

#include "daxq_common.h"
#include "store_rule.h"

namespace daxq {

typedef unsigned short us2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
    us2 va = __builtin_bit_cast(us2, a), vb = __builtin_bit_cast(us2, b);
    us2 r = __builtin_elementwise_max(va, vb);
    return __builtin_bit_cast(uint32_t, r);
}

// Element type of the tensor being quantised: XT = DAXQ_BF16 / DAXQ_F16 (two per 32-bit word) / DAXQ_F32.
// The bit pattern of a non-negative value orders like the value in all three, NaN above infinity.
template <int XT>
__device__ __forceinline__ float x_bits_to_f32(uint32_t b) {
    if constexpr (XT == DAXQ_BF16) return __uint_as_float(b << 16);
    else if constexpr (XT == DAXQ_F16) return (float)__builtin_bit_cast(_Float16, (uint16_t)b);
    else return __uint_as_float(b);
}

// f32 rounded to the element type (round to nearest even, subnormals of fp16 included), as a float
template <int XT>
__device__ __forceinline__ float round_to_x(float s) {
    if constexpr (XT == DAXQ_BF16) {
        if (s != s) return s;
        return bf16_bits_to_f32(f32_to_bf16_bits(s));
    } else if constexpr (XT == DAXQ_F16) {
        asm volatile("" : "+v"(s));  // keeps the conversion a conversion (no fold with the operation that produced s)
        return (float)(_Float16)s;
    } else {
        return s;
    }
}

// Columns [k, fill_width) of a quantised row are written as zeros: up to the next multiple of the GEMM's K granularity,
// as far as the row reaches.  A row stride beyond that (rows kept apart on purpose, or a column slice of a wider
// buffer) is left alone.
inline int64_t fill_width(int64_t k, int64_t ld_q) {
    const int64_t kp = (k + DAXQ_K_ALIGN - 1) / DAXQ_K_ALIGN * DAXQ_K_ALIGN;
    return kp < ld_q ? kp : ld_q;
}

// abs-max bits (sign cleared) of a block -> fp32 scale, exactly as the reference rounds it: the quotient is
// computed and floored in the tensor's own dtype when ROUND (dynamic activations,
// dax/quant/nn/dynamic/functional.py:124-129), in fp32 otherwise (weight observer).
template <bool ROUND, int XT = DAXQ_BF16>
__device__ __forceinline__ float scale_from_amax_bits(uint32_t amax_bits, float qmax) {
    float a = x_bits_to_f32<XT>(amax_bits);
    float s = a / qmax;  // IEEE binary32 division (hipcc default: correctly rounded)
    if (ROUND) s = round_to_x<XT>(s);
    return max_nan(s, kEps);  // clamp(min=eps): a NaN abs-max (a NaN anywhere in the row) stays NaN
}

// The same rule with the caller's floor and the rounding chosen at run time (uniform over the launch):
// round_x != 0   the eager chain: quotient and floor live in the tensor's own element type, so both are rounded to it
//                (clamp(min=eps) on a bf16 tensor compares with eps rounded to bf16)
// round_x == 0   quotient and floor stay in fp32: what a code generator that fuses the chain leaves of it
//                (the reference's forward carries a torch.compile decorator, dax/quant/nn/dynamic/linear.py:143)
template <int XT>
__device__ __forceinline__ float scale_from_amax_bits_rt(uint32_t amax_bits, float qmax, float eps, int round_x) {
    float a = x_bits_to_f32<XT>(amax_bits);
    float s = a / qmax;
    if (round_x) {
        s = round_to_x<XT>(s);
        eps = round_to_x<XT>(eps);
    }
    return max_nan(s, eps);
}

// Wavefront-wide reductions with DPP (data-parallel primitives: the partner lane's value is an operand
// modifier of the VALU instruction, no trip through the LDS crossbar as with ds_bpermute): four steps
// give every lane the result of its row of 16 lanes, the four row results are then read as scalars.
#define DAXQ_DPP_QUAD_SWAP1 0xB1   /* quad_perm [1,0,3,2] */
#define DAXQ_DPP_QUAD_SWAP2 0x4E   /* quad_perm [2,3,0,1] */
#define DAXQ_DPP_HALF_MIRROR 0x141 /* lane i <-> 7 - i within 8 */
#define DAXQ_DPP_ROW_MIRROR 0x140  /* lane i <-> 15 - i within 16 */

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    uint32_t o;
    o = dpp_u32<DAXQ_DPP_QUAD_SWAP1>(v); v = v > o ? v : o;
    o = dpp_u32<DAXQ_DPP_QUAD_SWAP2>(v); v = v > o ? v : o;
    o = dpp_u32<DAXQ_DPP_HALF_MIRROR>(v); v = v > o ? v : o;
    o = dpp_u32<DAXQ_DPP_ROW_MIRROR>(v); v = v > o ? v : o;
    const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 0), r1 = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
    const uint32_t r2 = (uint32_t)__builtin_amdgcn_readlane((int)v, 32), r3 = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
    const uint32_t a = r0 > r1 ? r0 : r1, b = r2 > r3 ? r2 : r3;
    return a > b ? a : b;
}

// fp32 sum over the wavefront, the same value in every lane (fixed order: deterministic)
__device__ __forceinline__ float wave_sum_f32(float x) {
    uint32_t v = __float_as_uint(x);
    v = __float_as_uint(__uint_as_float(v) + __uint_as_float(dpp_u32<DAXQ_DPP_QUAD_SWAP1>(v)));
    v = __float_as_uint(__uint_as_float(v) + __uint_as_float(dpp_u32<DAXQ_DPP_QUAD_SWAP2>(v)));
    v = __float_as_uint(__uint_as_float(v) + __uint_as_float(dpp_u32<DAXQ_DPP_HALF_MIRROR>(v)));
    v = __float_as_uint(__uint_as_float(v) + __uint_as_float(dpp_u32<DAXQ_DPP_ROW_MIRROR>(v)));
    const float r0 = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)v, 0));
    const float r1 = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)v, 16));
    const float r2 = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)v, 32));
    const float r3 = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)v, 48));
    return (r0 + r1) + (r2 + r3);
}

// clamp(rint(x * inv), -128, 127) as the low byte of a float: the product is clamped first (same result, the
// bounds are integers) and 1.5 * 2^23 is added, which rounds it to an integer, half to even, in the low mantissa
// bits; those bits are the two's-complement value.  Two operations fewer than round + convert.
// CLAMP = false: a row quantised with its own bf16-rounded (or fp32) scale of abs-max / 127 never leaves [-127.4, 127.4]
// (the rounding of the scale moves x * inv at the row maximum by at most 2^-8 of it: checked for every bf16 abs-max), so
// the clamp is dead code there and is left out.  (A NaN product -- an infinite element of a row whose scale is infinite
// -- then gives the byte 0 instead of -128; such a row's output is non-finite through its scale either way.)
template <bool CLAMP = true>
__device__ __forceinline__ uint32_t q_i8_bits(float x, float inv) {
    float r = x * inv;
    if constexpr (CLAMP) r = fminf(fmaxf(r, -128.0f), 127.0f);
    else asm("" : "+v"(r));  // the product is rounded before the addition, as in the reference: no contraction into one fma
    return __float_as_uint(r + 12582912.0f);
}

// FMT: 0 = int8, 1 = OCP e4m3fn (max 448), 2 = OCP e5m2 (max 57344)
// x / s, correctly rounded, from the correctly rounded reciprocal inv = RN(1 / s) of the row: one multiply,
// the exact residual by fma, one correction (Markstein's sequence; it yields RN(x / s) unless the
// significand of s is all ones, which a scale whose low 16 bits are zero never has).  The reference's
// true division costs about ten instructions per element when spelled x / s.
// TRUE_DIV: spell the division out (leaf quantiser with an arbitrary fp32 scale, used once per weight).
// CLAMP = false: with the row's own scale of abs-max / qmax the quotient at the row maximum stays below qmax * (1 + 2^-8)
// (449.5 for e4m3fn, 57530 for e5m2: checked for every bf16 abs-max), which the cast's round-to-nearest-even takes to
// the format's largest finite value by itself (the next step up lies beyond 464 / 61440), so the clamp is left out.
template <int FMT, bool TRUE_DIV, bool CLAMP = true>
__device__ __forceinline__ float q_f8_pre(float x, float s, float inv) {
    constexpr float kMax = FMT == 2 ? 57344.0f : 448.0f;
    float v;
    if constexpr (TRUE_DIV) {
        v = x / s;  // IEEE division
    } else {
        const float q0 = x * inv;
        const float e = __builtin_fmaf(-q0, s, x);
        v = __builtin_copysignf(__builtin_fmaf(e, inv, q0), x);  // s > 0; keeps -0 for x = -0 (0 + -0 is +0 in the fma)
    }
    // With a scale from the caller a NaN element must stay NaN through the clamp, as in the reference, and become
    // the format's NaN byte; with the row's own scale a NaN element has already made that scale NaN.
    if constexpr (!CLAMP) return v;
    if constexpr (TRUE_DIV) return min_nan(max_nan(v, -kMax), kMax);
    return fminf(fmaxf(v, -kMax), kMax);
}

template <int FMT>
__device__ __forceinline__ int cvt_pk_f8(float a, float b, int old, bool hi) {
    if constexpr (FMT == 2)
        return hi ? __builtin_amdgcn_cvt_pk_bf8_f32(a, b, old, true) : __builtin_amdgcn_cvt_pk_bf8_f32(a, b, old, false);
    else
        return hi ? __builtin_amdgcn_cvt_pk_fp8_f32(a, b, old, true) : __builtin_amdgcn_cvt_pk_fp8_f32(a, b, old, false);
}

// 8 bf16 / fp16 values (one 16-byte chunk) -> 8 quantised bytes
template <int FMT, bool TRUE_DIV = false, int XT = DAXQ_BF16, bool CLAMP = true>
__device__ __forceinline__ uint2 quant_chunk(const uint4& v, float s, float inv) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    uint32_t o[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float f0, f1, f2, f3;
        if constexpr (XT == DAXQ_BF16) {
            f0 = __uint_as_float(w[2 * h] << 16);
            f1 = __uint_as_float(w[2 * h] & 0xffff0000u);
            f2 = __uint_as_float(w[2 * h + 1] << 16);
            f3 = __uint_as_float(w[2 * h + 1] & 0xffff0000u);
        } else {
            f0 = x_bits_to_f32<XT>(w[2 * h] & 0xffffu);
            f1 = x_bits_to_f32<XT>(w[2 * h] >> 16);
            f2 = x_bits_to_f32<XT>(w[2 * h + 1] & 0xffffu);
            f3 = x_bits_to_f32<XT>(w[2 * h + 1] >> 16);
        }
        if (FMT != 0) {
            int p = cvt_pk_f8<FMT>(q_f8_pre<FMT, TRUE_DIV, CLAMP>(f0, s, inv), q_f8_pre<FMT, TRUE_DIV, CLAMP>(f1, s, inv), 0, false);
            p = cvt_pk_f8<FMT>(q_f8_pre<FMT, TRUE_DIV, CLAMP>(f2, s, inv), q_f8_pre<FMT, TRUE_DIV, CLAMP>(f3, s, inv), p, true);
            o[h] = (uint32_t)p;
        } else {
            // byte 0 of each of the four words: three v_perm_b32
            const uint32_t p01 = __builtin_amdgcn_perm(q_i8_bits<CLAMP>(f1, inv), q_i8_bits<CLAMP>(f0, inv), 0x0c0c0400u);
            const uint32_t p23 = __builtin_amdgcn_perm(q_i8_bits<CLAMP>(f3, inv), q_i8_bits<CLAMP>(f2, inv), 0x0c0c0400u);
            o[h] = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
        }
    }
    return make_uint2(o[0], o[1]);
}

// packed abs-max (two bf16 magnitudes per word) of 8 bf16 values
__device__ __forceinline__ uint32_t chunk_absmax(uint32_t mx, const uint4& v) {
    mx = pk_max_u16(mx, v.x & 0x7fff7fffu);
    mx = pk_max_u16(mx, v.y & 0x7fff7fffu);
    mx = pk_max_u16(mx, v.z & 0x7fff7fffu);
    mx = pk_max_u16(mx, v.w & 0x7fff7fffu);
    return mx;
}

// Accesses of the kernels that fuse a producer and the quantiser.  The bf16 row is read once, past the caches with the non-temporal
// hint; where the quantised row goes: fused_store_through.
typedef unsigned daxq_v4u __attribute__((ext_vector_type(4)));
typedef unsigned daxq_v2u __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint4 load_stream_16(const uint4* p) {
    const daxq_v4u t = __builtin_nontemporal_load(reinterpret_cast<const daxq_v4u*>(p));
    return make_uint4(t.x, t.y, t.z, t.w);
}
// p is a multiple of 8
template <bool THROUGH>
__device__ __forceinline__ void store_row_8(uint2* p, uint2 v) {
    const daxq_v2u t = {v.x, v.y};
    if constexpr (THROUGH) __hip_atomic_store(reinterpret_cast<uint64_t*>(p), __builtin_bit_cast(uint64_t, t), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else __builtin_nontemporal_store(t, reinterpret_cast<daxq_v2u*>(p));
}

// A row is cut into chunks of 8 elements.  Any alignment is taken: the loads and stores are the same 16- and 8-byte
// instructions whatever the address (gfx950 runs them on any byte address of global memory).
template <int XT>
struct Chunk {
    daxq_v4u w[XT == DAXQ_F32 ? 2 : 1];
};

template <int XT>
__device__ __forceinline__ void load_chunk(Chunk<XT>& v, const char* p) {
    typedef daxq_v4u loose __attribute__((aligned(2)));
#pragma unroll
    for (int h = 0; h < (XT == DAXQ_F32 ? 2 : 1); ++h) v.w[h] = __builtin_nontemporal_load(reinterpret_cast<const loose*>(p) + h);
}

// for what other workgroups of the XCD read, too: the hint above would evict it from the L2 that they share
template <int XT>
__device__ __forceinline__ void load_chunk_shared(Chunk<XT>& v, const char* p) {
    typedef daxq_v4u loose __attribute__((aligned(2)));
#pragma unroll
    for (int h = 0; h < (XT == DAXQ_F32 ? 2 : 1); ++h) v.w[h] = reinterpret_cast<const loose*>(p)[h];
}

// STORE: where the bytes go (store_of; p is a multiple of 8 with kStoreThrough)
template <int STORE>
__device__ __forceinline__ void store_chunk(uint8_t* p, uint2 v) {
    typedef daxq_v2u loose __attribute__((aligned(1)));
    const daxq_v2u t = {v.x, v.y};
    if constexpr (STORE == kStoreThrough) __hip_atomic_store(reinterpret_cast<uint64_t*>(p), __builtin_bit_cast(uint64_t, t), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else if constexpr (STORE == kStoreKeep) *reinterpret_cast<loose*>(p) = t;
    else __builtin_nontemporal_store(t, reinterpret_cast<loose*>(p));
}

// running abs-max of chunks: packed 16-bit magnitudes or 32-bit ones
template <int XT>
__device__ __forceinline__ uint32_t chunk_amax(uint32_t mx, const Chunk<XT>& v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (XT != DAXQ_F32) {
            mx = pk_max_u16(mx, v.w[0][i] & 0x7fff7fffu);
        } else {
            const uint32_t a = v.w[0][i] & 0x7fffffffu, b = v.w[1][i] & 0x7fffffffu;
            mx = a > mx ? a : mx;
            mx = b > mx ? b : mx;
        }
    }
    return mx;
}
template <int XT>
__device__ __forceinline__ uint32_t amax_of_lane(uint32_t mx) {
    if constexpr (XT == DAXQ_F32) return mx;
    return (mx & 0xffffu) > (mx >> 16) ? (mx & 0xffffu) : (mx >> 16);
}

template <int XT>
__device__ __forceinline__ void chunk_values(const Chunk<XT>& v, float (&f)[8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if constexpr (XT == DAXQ_F32) f[i] = __uint_as_float(v.w[i >> 2][i & 3]);
        else if constexpr (XT == DAXQ_BF16) f[i] = __uint_as_float(i & 1 ? v.w[0][i >> 1] & 0xffff0000u : v.w[0][i >> 1] << 16);
        else f[i] = x_bits_to_f32<XT>(i & 1 ? v.w[0][i >> 1] >> 16 : v.w[0][i >> 1] & 0xffffu);
    }
}

// How the elements of a row become bytes, one choice per row:
//   kOwn       a bf16 row under its own scale at no more than the format's maximum: no clamp (dead code there,
//              quant_rows.h), for FP8 the reciprocal sequence verified exhaustively for bf16 elements under bf16 scales
//   kDivide    x / s by IEEE division (int8: x * inv), clamped
//   kNear      FP8 and fp32 elements: x * inv, whose error is at most 1.5 steps of fp32, rounds to the byte of x / s
//              unless it lies that close to a value where the byte changes.  Those values, in the normal and the subnormal
//              range of either format, have at most five significant bits, i.e. zeros in the low 19 bits of the fp32
//              pattern, so a product within three steps of such a pattern sends the wavefront's chunks through the
//              division (seven patterns in 2^19, 13 elements in 10^6 under an arbitrary scale; zeros and infinities
//              too).  A NaN need not be near (some of its payload lies in those 19 bits): the clamp keeps it instead
//              (v_maximum3 / v_minimum3 return a NaN, fmed3 its lower bound; a compare per element beside the fmed3 cost
//              32 rows of 13824 0.2 us).
//   kExact     FP8 under a power of two: x * inv is the quotient
//   kShort     FP8 and 16-bit elements under any other scale: the sequence of kOwn, clamped, and the division for chunks
//              that hold an infinity or a NaN.  Quotients of such elements hit values where the byte changes all the time
//              (an abs-max of 8 bits over 448 = 7 x 64 is the scale of a calibrated or a weight's row: every element with the
//              abs-max's significand does), so that kNear divides nearly every chunk: e4m3 under such a scale, us, kNear ->
//              kShort: 4725 x 5120 17.5 -> 13.6, a weight of 13824 x 5120 47.9 -> 34.8, 9000 x 1536 11.3 -> 9.4; fp16 rows
//              under their own fp16 scale, which divided every element, 4725 x 5120 19.8 -> 14.9.
//              Its bytes are those of the division: with u the step of the quotient, the corrected quotient is x / s,
//              off by less than 6 x 2^-24 u (reciprocal and residual are rounded once each, the first quotient is off
//              by at most 3 u), rounded.  Another byte than that of RN(x / s) needs a midpoint m, half a step from a value of five bits, inside
//              that error.  In units of u / 2, m = +-1 mod 2^20 and x / s = X / S with the significand S of s and X a multiple of 2^36
//              (x has at most 11 bits), so |X - m S| is at least the distance of S from a multiple of 2^20, not zero (m is odd
//              and longer than x), and would have to be below 12: scales that close to a significand of four bits, but not one
//              themselves, divide.
enum { kOwn = 0, kDivide = 1, kNear = 2, kExact = 3, kShort = 4 };

template <int FMT, int XT>
__device__ __forceinline__ int form_of_scale(float s) {
    if constexpr (FMT == 0) return kDivide;
    const uint32_t b = __float_as_uint(s);
    // (NaN too; from 2^-80 on the residual of a quotient that is not rounded to zero is a normal number)
    if (!(s >= (XT == DAXQ_F32 ? 0x1p-100f : 0x1p-80f) && s <= 0x1p100f)) return kDivide;
    if ((b & 0x7fffffu) == 0) return kExact;
    if constexpr (XT == DAXQ_F32) return kNear;
    return ((b + 16u) & 0xfffffu) <= 32u && (b & 0xfffffu) != 0 ? kDivide : kShort;
}

template <int FMT, int FORM, int XT>
__device__ __forceinline__ uint2 quant8(const float (&f)[8], float s, float inv) {
    uint32_t o[2];
    if constexpr (FMT == 0) {
        constexpr bool CLAMP = FORM != kOwn;
#pragma unroll
        for (int h = 0; h < 2; ++h) {  // byte 0 of each of the four words: three v_perm_b32
            const uint32_t p01 = __builtin_amdgcn_perm(q_i8_bits<CLAMP>(f[4 * h + 1], inv), q_i8_bits<CLAMP>(f[4 * h], inv), 0x0c0c0400u);
            const uint32_t p23 = __builtin_amdgcn_perm(q_i8_bits<CLAMP>(f[4 * h + 3], inv), q_i8_bits<CLAMP>(f[4 * h + 2], inv), 0x0c0c0400u);
            o[h] = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
        }
    } else {
        constexpr float kMax = FMT == 2 ? 57344.0f : 448.0f;
        float v[8];
        if constexpr (FORM == kNear || FORM == kExact || FORM == kShort) {
            uint32_t near = 0xffffffffu;
            bool nan = false;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                float q0 = f[i] * inv;
                // (the negated residual: +0 where there is none, so that a -0 stays one; a NaN's sign is the division's)
                if constexpr (FORM == kShort) q0 = __builtin_fmaf(-__builtin_fmaf(q0, s, -f[i]), inv, q0);
                if constexpr (FORM == kNear) {
                    const uint32_t d = (__float_as_uint(q0) << 13) + (3u << 13);
                    near = d < near ? d : near;
                }
                if constexpr (FORM == kNear) {  // a NaN stays one
                    v[i] = __builtin_elementwise_minimum(__builtin_elementwise_maximum(q0, -kMax), kMax);
                } else {
                    nan |= q0 != q0;
                    v[i] = __builtin_amdgcn_fmed3f(q0, -kMax, kMax);
                }
            }
            if (__ballot((FORM == kNear && near <= (6u << 13)) || nan)) {
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = q_f8_pre<FMT, true>(f[i], s, inv);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = q_f8_pre<FMT, FORM != kOwn, FORM != kOwn>(f[i], s, inv);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int p = cvt_pk_f8<FMT>(v[4 * h], v[4 * h + 1], 0, false);
            o[h] = (uint32_t)cvt_pk_f8<FMT>(v[4 * h + 2], v[4 * h + 3], p, true);
        }
    }
    return make_uint2(o[0], o[1]);
}

// Calls f with the form (a compile-time constant) that the elements of a row take under scale s.  scale_in: the scale is the
// caller's; round_x: a dynamic scale was rounded to the element type; leaf: the scale is a tensor's or a weight's, and the leaf
// quantiser's bytes are wanted also where it is not finite (under an infinite scale a finite element is x / inf = 0, which the
// reciprocal sequence gives as NaN, and an infinity is inf / inf, whose int8 byte depends on the clamp; so does that of a NaN)
template <int FMT, int XT, typename F>
__device__ __forceinline__ void with_form(float s, float qmax, bool scale_in, int round_x, int leaf, F&& f) {
    constexpr float kFmtMax = FMT == 0 ? 127.0f : FMT == 1 ? 448.0f : 57344.0f;
    if (XT == DAXQ_BF16 && !scale_in && qmax <= kFmtMax && (FMT == 0 || round_x) && (!leaf || s < __builtin_inff())) {
        f(std::integral_constant<int, kOwn>{});
    } else if constexpr (FMT == 0) {
        f(std::integral_constant<int, kDivide>{});
    } else {
        const int form = form_of_scale<FMT, XT>(s);
        constexpr int kMost = XT == DAXQ_F32 ? kNear : kShort;
        if (form == kMost) f(std::integral_constant<int, kMost>{});
        else if (form == kExact) f(std::integral_constant<int, kExact>{});
        else f(std::integral_constant<int, kDivide>{});
    }
}

}  // namespace daxq
