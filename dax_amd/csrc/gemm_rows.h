// Pieces of the kernels whose wavefronts stream a part of the weight each (gemm_rows.hip, gemm_few.hip): the MFMAs of a step of 128
// K bytes and the epilogue of one 16x16 block.
#pragma once

#include <type_traits>

#include "gemm_tile.h"

namespace daxq {

// FP8 formats as in the tiled kernels: the weight is the MFMA "A" operand (cbsz), the activations the "B" operand (blgp)
template <bool FP8, int F8>
__device__ __forceinline__ typename Acc16<FP8>::type mfma_step(v8i w, v8i x, typename Acc16<FP8>::type c) {
    if constexpr (FP8) {
        return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, x, c, (F8 & kF8WE5) ? 1 : 0, (F8 & kF8XE5) ? 1 : 0, 0, 0, 0, 0);
    } else {
        c = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_shufflevector(w, w, 0, 1, 2, 3), __builtin_shufflevector(x, x, 0, 1, 2, 3), c, 0, 0, 0);
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_shufflevector(w, w, 4, 5, 6, 7), __builtin_shufflevector(x, x, 4, 5, 6, 7), c, 0, 0, 0);
    }
}

template <int T, typename F>
__device__ __forceinline__ void for_down(F&& f) {
    f(Int<T>{});
    if constexpr (T > 0) for_down<T - 1>(f);
}

// Scales and bias elements of the four consecutive columns from nc on (beyond the matrix: its last column, not stored).  Plain loads, the
// conversions are left to the epilogue: nothing waits for them where they are requested.
template <int OUTK>
struct ColumnBits {
    typedef typename std::conditional<OUTK == DAXQ_F32, float, uint16_t>::type elem;
    float sw[4];
    elem b[4];
    bool none;
    __device__ __forceinline__ ColumnBits(const GemmArgs& p, int nc) : none(!p.bias) {
        const elem* bp = p.bias ? reinterpret_cast<const elem*>(p.bias) : reinterpret_cast<const elem*>(p.sw);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = nc + e < p.n ? nc + e : p.n - 1;
            sw[e] = p.sw[c];
            b[e] = bp[c];
        }
    }
    __device__ __forceinline__ float bias(int e) const {
        if (none) return -0.0f;  // x + (-0.0) == x bit for bit
        if constexpr (OUTK == DAXQ_F32) return b[e];
        else if constexpr (OUTK == DAXQ_F16) return f16_bits_to_f32(b[e]);
        else return bf16_bits_to_f32(b[e]);
    }
};

// The epilogue (the arithmetic of tile_epilogue16) of four accumulators: output row m, columns nc .. nc + 3 as far as there are
template <bool FP8, int OUTK>
__device__ __forceinline__ void store_columns(const GemmArgs& p, typename Acc16<FP8>::type acc, float sxv, const ColumnBits<OUTK>& cols, int m, int nc) {
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float y = (float)acc[e];  // (int8: v_cvt_f32_i32, round to nearest even)
        y = y * sxv;
        y = y * cols.sw[e];
        if constexpr (OUTK == DAXQ_F32 || FP8) {
            o[e] = y + cols.bias(e);
            if constexpr (OUTK == DAXQ_F16) asm("" : "+v"(o[e]));  // the sum is rounded to fp32 before the cast to fp16
        } else if constexpr (OUTK == DAXQ_F16) {
            asm("" : "+v"(y));
            float z = (float)(_Float16)y + cols.bias(e);
            asm("" : "+v"(z));
            o[e] = z;
        } else {
            o[e] = bf16_bits_to_f32(pack_bf16_rne(y, 0.0f) & 0xffffu) + cols.bias(e);
        }
    }
    const int64_t at = (int64_t)m * p.ldo + nc;
    if constexpr (OUTK == DAXQ_F32) {
        float* dst = reinterpret_cast<float*>(p.out) + at;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (nc + e < p.n) dst[e] = o[e];
    } else {
        uint32_t lo, hi;
        if constexpr (OUTK == DAXQ_F16) lo = pack_f16_rne(o[0], o[1]), hi = pack_f16_rne(o[2], o[3]);
        else lo = pack_bf16_rne(o[0], o[1]), hi = pack_bf16_rne(o[2], o[3]);
        typedef v2u loose __attribute__((aligned(2)));
        uint16_t* dst = p.out + at;
        if (nc + 4 <= p.n) {
            *reinterpret_cast<loose*>(dst) = v2u{lo, hi};
        } else {
            const uint32_t w[4] = {lo & 0xffffu, lo >> 16, hi & 0xffffu, hi >> 16};
#pragma unroll
            for (int e = 0; e < 3; ++e)
                if (nc + e < p.n) dst[e] = (uint16_t)w[e];
        }
    }
}

}  // namespace daxq
