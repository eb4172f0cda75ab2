// Pieces shared by the tiled W8A8 GEMM kernels (gemm_tile256.hip: INT8; gemm_tile_fp8.hip: FP8): fragment types, the
// tile a workgroup computes, the epilogue for accumulators held as 16x16 blocks, and the cut of a launch's last,
// partial round of workgroups.
#pragma once

#include "gemm_common.h"

namespace daxq {

template <bool FP8>
struct Frag {
    typedef v4i type;
};
template <>
struct Frag<true> {
    typedef v8i type;
};

struct Yes {
    static constexpr bool value = true;
};
struct No {
    static constexpr bool value = false;
};
template <int N>
struct Int {
    static constexpr int value = N;
};

template <int I, int N, typename F>
__device__ __forceinline__ void for_up(F&& f) {
    if constexpr (I < N) {
        f(Int<I>{});
        for_up<I + 1, N>(f);
    }
}

// GemmArgs::lines
constexpr int kLinesNone = 0, kLinesPlain = 1, kLinesThrough = 2;
// GemmArgs::order
constexpr int kOrderRowGroups = 0, kOrderBanded = 1;

// Which BT x BT output tile workgroup `tile_id` computes: its origin (m0, n0), shifted inwards at the M / N edge
// instead of being predicated (the overlap rows are computed twice with identical results).  False: a padding slot of
// the banded order, the workgroup exits at once.  With quad_base > 0, BT = 128 means the four quadrants of the
// 256x256 tiles from id quad_base - 1 on, one workgroup per quadrant (tile_id counts quadrants).
template <int BT>
__device__ __forceinline__ bool tile_origin(const GemmArgs& p, int tile_id, int& m0, int& n0) {
    int tm, tn;
    if (BT == 128 && p.quad_base) {
        tile_of_block(p.gm, p.quad_base - 1 + (tile_id >> 2), p.tiles_m, p.tiles_n, tm, tn);  // the 256x256 tile
        m0 = tm * 256, n0 = tn * 256;
        m0 = (m0 + 256 <= p.m ? m0 : p.m - 256) + ((tile_id >> 1) & 1) * 128;
        n0 = (n0 + 256 <= p.n ? n0 : p.n - 256) + (tile_id & 1) * 128;
        return true;
    }
    if (p.order == kOrderBanded) {
        if (!tile_of_block_banded(tile_id, p.tiles_m, p.tiles_n, 4, tm, tn)) return false;
    } else {
        tile_of_block(p.gm, tile_id, p.tiles_m, p.tiles_n, tm, tn);
    }
    m0 = tm * BT, n0 = tn * BT;
    m0 = m0 + BT <= p.m ? m0 : p.m - BT;
    n0 = n0 + BT <= p.n ? n0 : p.n - BT;
    return true;
}

// workgroups of a launch of 256x256 tiles in the tile order a.order
static inline int64_t grid_of_order(const GemmArgs& a) {
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n;
    if (a.order != kOrderBanded) return tiles;
    // the patch arithmetic of the banded order is 32-bit: beyond 2^30 tiles none of it runs and the caller's check of the
    // grid size refuses the launch
    return tiles <= (1 << 30) ? banded_grid(a.tiles_m, a.tiles_n, 4) : (int64_t)1 << 40;
}

// accumulators of one 16x16 block: int32 (v_mfma_i32_16x16x64_i8) or fp32 (v_mfma_f32_16x16x128_f8f6f4)
template <bool FP8>
struct Acc16 {
    typedef v4i type;
};
template <>
struct Acc16<true> {
    typedef v4f type;
};

// Behind the last MFMA of a path.  The MFMAs are inline asm, so the compiler cannot count the wait states between one of them and
// another instruction that reads its result: idle cycles first.  It stands in front of a join of control flow, not behind it: where
// two paths hold an accumulator in different registers, the compiler copies it at the end of a path, and a copy in front of the idle
// cycles reads a result that is not there yet (found in a kernel with the accumulator dump: the halves' sums were off by 3 %).
__device__ __forceinline__ void mfma_settle() {
    asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 7");
    __builtin_amdgcn_sched_barrier(0);
}

// Four outputs of a row as 16-bit values (OUTK: DAXQ_BF16 / DAXQ_F16)
template <bool FP8, int OUTK>
__device__ __forceinline__ uint2 outputs4(const typename Acc16<FP8>::type& acc, float sx, const v4f& sw, const v4f& bias) {
    uint32_t pk[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int r = 2 * h;
        if constexpr (FP8) {
            float z0 = acc[r] * sx * sw[r] + bias[r], z1 = acc[r + 1] * sx * sw[r + 1] + bias[r + 1];
            if constexpr (OUTK == DAXQ_F16) {  // one rounding, to fp16 (kept apart from the add: no mixed-precision fold)
                asm("" : "+v"(z0), "+v"(z1));
                pk[h] = pack_f16_rne(z0, z1);
            } else {
                pk[h] = pack_bf16_rne(z0, z1);
            }
        } else {
            float y0 = (float)acc[r];  // v_cvt_f32_i32, round to nearest even
            float y1 = (float)acc[r + 1];
            y0 = y0 * sx;
            y1 = y1 * sx;
            y0 = y0 * sw[r];
            y1 = y1 * sw[r + 1];
            if constexpr (OUTK == DAXQ_F16) {  // fp16 module: the same two roundings, to fp16
                // (the products and sums pass through empty asm statements: the compiler otherwise folds
                // a multiply or add and the conversion behind it into one mixed-precision instruction
                // that rounds once, where the reference rounds to fp32 first)
                asm("" : "+v"(y0), "+v"(y1));
                const uint32_t o1 = pack_f16_rne(y0, y1);
                pk[h] = pack_f16_rne(add_f16_half<0>(o1, bias[r]), add_f16_half<1>(o1, bias[r + 1]));
            } else {
                // second rounding: the bias is added to the bf16 value, which the first leaves in the upper half of a word
                const float o0 = __uint_as_float(pack_bf16_rne(0.0f, y0)), o1 = __uint_as_float(pack_bf16_rne(0.0f, y1));
                pk[h] = pack_bf16_rne(o0 + bias[r], o1 + bias[r + 1]);
            }
        }
    }
    return make_uint2(pk[0], pk[1]);
}

// 16 bytes at any address, into the L2 and through it to memory at once (a device-coherent store)
__device__ __forceinline__ void store_through(uint8_t* p, v4u v) {
    __builtin_amdgcn_global_store_b128((DAXQ_GLOBAL v4u*)p, v, "agent");
}

// Accumulators as they are (tests): int32 / fp32 [m, ldacc]
template <int NBJ, int NBI, bool FP8>
__device__ __forceinline__ void dump_tile16(const GemmArgs& p, typename Acc16<FP8>::type (&acc)[NBJ][NBI], int m0, int n0, int l15, int g4) {
#pragma unroll
    for (int j = 0; j < NBJ; ++j)
#pragma unroll
        for (int i = 0; i < NBI; ++i) {
            const int64_t m = m0 + i * 16 + l15;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if constexpr (FP8) static_cast<float*>(p.acc)[m * p.ldacc + n0 + j * 16 + 4 * g4 + v] = acc[j][i][v];
                else static_cast<int32_t*>(p.acc)[m * p.ldacc + n0 + j * 16 + 4 * g4 + v] = acc[j][i][v];
            }
        }
}

// In a 16x16 block a lane owns output row m = l%16 and the columns n = 4*(l/16) + {0..3}.
// The outputs of a wavefront's accumulators held as NBJ x NBI such blocks (v_mfma_i32_16x16x64_i8, v_mfma_f32_16x16x128_f8f6f4), of
// which (m0, n0) is the first: acc[j][i] is weight block j (16 output columns) and activation block i (16 output rows).
// sx, sw, bias: the scales of the lane's output row in each block of rows, scales and bias of its four columns in each block of columns.

// fp32 module: one rounding less and four-byte outputs, a lane's four columns of a block as one store.
template <int NBJ, int NBI, bool FP8>
__device__ __forceinline__ void outputs_f32(const GemmArgs& p, typename Acc16<FP8>::type (&acc)[NBJ][NBI], int m0, int n0, int l15, int g4,
                                            const float (&sx)[NBI], const v4f (&sw)[NBJ], const v4f (&bias)[NBJ]) {
    // a lane's place in the first block of rows; the others lie a uniform step apart, the blocks of columns at constant offsets
    float* row = reinterpret_cast<float*>(p.out) + (int64_t)(m0 + l15) * p.ldo + n0 + 4 * g4;
#pragma unroll
    for (int i = 0; i < NBI; ++i) {
#pragma unroll
        for (int j = 0; j < NBJ; ++j) {
            float o[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float y = (float)acc[j][i][r];  // (int8: v_cvt_f32_i32, round to nearest even)
                y = y * sx[i];
                y = y * sw[j][r];
                o[r] = y + bias[j][r];
            }
            *reinterpret_cast<float4*>(row + j * 16) = make_float4(o[0], o[1], o[2], o[3]);
        }
        row += 16 * p.ldo;
    }
}

// Outputs of 16 bits straight from the registers.  One v_permlane16_swap per word over two neighbouring blocks gives each lane 8
// consecutive columns of one of them: lanes 0-15 block 2jp columns 0-7, lanes 16-31 block 2jp+1 columns 0-7, lanes 32-47 block
// 2jp columns 8-15, lanes 48-63 block 2jp+1 columns 8-15.
template <int NBJ, int NBI, bool FP8, int OUTK>
__device__ __forceinline__ void outputs_straight(const GemmArgs& p, typename Acc16<FP8>::type (&acc)[NBJ][NBI], int m0, int n0, int l15, int g4,
                                                 const float (&sx)[NBI], const v4f (&sw)[NBJ], const v4f (&bias)[NBJ]) {
    static_assert(NBJ % 2 == 0, "blocks in pairs");
    uint16_t* row = p.out + (int64_t)(m0 + l15) * p.ldo + n0 + (g4 & 1) * 16 + (g4 >> 1) * 8;
#pragma unroll
    for (int i = 0; i < NBI; ++i) {
#pragma unroll
        for (int j = 0; j < NBJ; j += 2) {
            const uint2 lo = outputs4<FP8, OUTK>(acc[j][i], sx[i], sw[j], bias[j]), up = outputs4<FP8, OUTK>(acc[j + 1][i], sx[i], sw[j + 1], bias[j + 1]);
            v2u s0 = __builtin_amdgcn_permlane16_swap(lo.x, up.x, false, false);
            v2u s1 = __builtin_amdgcn_permlane16_swap(lo.y, up.y, false, false);
            *reinterpret_cast<uint4*>(row + j * 16) = make_uint4(s0.x, s1.x, s0.y, s1.y);
        }
        row += 16 * p.ldo;
    }
}

// Outputs of 16 bits as whole rows of the wavefront's, through `own`, its part of the LDS: 16 NBI rows of 32 NBJ + 16 bytes.
template <int NBJ, int NBI, bool FP8, int OUTK, bool ALWAYS_THROUGH>
__device__ __forceinline__ void outputs_lines(const GemmArgs& p, typename Acc16<FP8>::type (&acc)[NBJ][NBI], uint8_t* own, int m0, int n0, int lane,
                                              const float (&sx)[NBI], const v4f (&sw)[NBJ], const v4f (&bias)[NBJ]) {
    // groups of G blocks of rows, so that the stores of one run beside the arithmetic of the next
    constexpr int G = 2, ROW = 32 * NBJ + 16, CHUNKS = 2 * NBJ, ROWS = 64 / CHUNKS, STEPS = 16 * G / ROWS;
    static_assert(NBI % G == 0 && 64 % CHUNKS == 0, "whole stores");
    uint8_t* const to = own + (lane & 15) * ROW + (lane >> 4) * 8;
    const uint8_t* const from = own + lane / CHUNKS * ROW + lane % CHUNKS * 16;
    uint8_t* out = reinterpret_cast<uint8_t*>(p.out) + ((int64_t)(m0 + lane / CHUNKS) * p.ldo + n0 + lane % CHUNKS * 8) * 2;
    const int64_t step = ROWS * 2 * p.ldo;
    v4u line[STEPS];
    auto store_group = [&]() __attribute__((always_inline)) {
        typedef v4u loose_v4u __attribute__((aligned(2)));
        if (ALWAYS_THROUGH || p.lines == kLinesThrough) {
#pragma unroll
            for (int s = 0; s < STEPS; ++s) store_through(out + s * step, line[s]);
        } else {
#pragma unroll
            for (int s = 0; s < STEPS; ++s) *reinterpret_cast<loose_v4u*>(out + s * step) = line[s];
        }
        out += STEPS * step;
    };
#pragma unroll
    for (int g = 0; g < NBI / G; ++g) {
#pragma unroll
        for (int ii = 0; ii < G; ++ii) {
            const int i = g * G + ii;
#pragma unroll
            for (int j = 0; j < NBJ; ++j) *reinterpret_cast<uint2*>(to + i * 16 * ROW + j * 32) = outputs4<FP8, OUTK>(acc[j][i], sx[i], sw[j], bias[j]);
            if (g > 0 && ii == 0) store_group();  // the group before: its reads have come back meanwhile
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (the LDS serves a wavefront in order)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s = 0; s < STEPS; ++s) line[s] = *reinterpret_cast<const v4u*>(from + (g * G * 16 + s * ROWS) * ROW);
    }
    store_group();
}

// LDS bytes of the epilogue below: scales and bias of the tile, then (LINES) a part per wavefront
constexpr int epilogue16_scales(int nbj, int nbi) { return (32 * nbi + 2 * 32 * nbj) * 4; }
constexpr int epilogue16_part(int nbj, int nbi) { return 16 * nbi * (32 * nbj + 16); }
constexpr int epilogue16_lds(int nbj, int nbi, bool lines) { return epilogue16_scales(nbj, nbi) + (lines ? 4 * epilogue16_part(nbj, nbi) : 0); }

// The epilogue of kernels that have no registers for the scales beside their main loop: a thread has requested one of each, and they
// pass through the LDS, which it begins to write at once: a barrier lies between the workgroup's last fragment read and this call (the one
// in front of the last MFMAs).
// OUTK: element type of out and bias, DAXQ_BF16 / DAXQ_F16 / DAXQ_F32.  A template argument, i.e. a kernel
// of its own per type: with all three forms inside one kernel behind uniform branches its code grew from 27 to 44 KB
// and the bf16 launches at K = 1536, which change between main loop and epilogue every 24 slices, lost 2.7 %; with
// the choice inside the loops they lost 2 to 11 % everywhere.
// LINES: 16-bit outputs leave as whole rows (lines_of says when).  A template argument for the same reason: as a uniform branch in the
// kernel it cost 1 to 2 % (75600 x 5120 x 5120 e4m3 1564 -> 1592 us, 9830 x 5120, K = 1536 84.6 -> 85.7), and some FP8 forms spilled.
template <bool DUMP, int NBJ, int NBI, bool FP8 = false, int OUTK = DAXQ_BF16, bool LINES = false, bool ALWAYS_THROUGH = false>
__device__ __forceinline__ void tile_epilogue16(const GemmArgs& p, typename Acc16<FP8>::type (&acc)[NBJ][NBI], uint8_t* smem, int m0, int n0, int t,
                                                int wm, int wn, int l15, int g4, float pre_sx, float pre_sw,
                                                float pre_bias) {
    constexpr int WTM = 16 * NBI, WTN = 16 * NBJ, BM = 2 * WTM, BN = 2 * WTN, T = 256;
    float* s_sx = reinterpret_cast<float*>(smem);
    float* s_sw = s_sx + BM;
    float* s_bias = s_sw + BN;
    if (BM == T || t < BM) s_sx[t] = pre_sx;
    if (BN == T || t < BN) {
        s_sw[t] = pre_sw;
        s_bias[t] = pre_bias;
    }
    __syncthreads();
    float sx[NBI];
    v4f sw[NBJ], bias[NBJ];
#pragma unroll
    for (int i = 0; i < NBI; ++i) sx[i] = s_sx[wm * WTM + i * 16 + l15];
#pragma unroll
    for (int j = 0; j < NBJ; ++j) {
        const int nl = wn * WTN + j * 16 + 4 * g4;
        sw[j] = *reinterpret_cast<const v4f*>(s_sw + nl);
        bias[j] = *reinterpret_cast<const v4f*>(s_bias + nl);
    }
    __builtin_amdgcn_sched_barrier(0);
    const int mw = m0 + wm * WTM, nw = n0 + wn * WTN;
    if constexpr (DUMP) dump_tile16<NBJ, NBI, FP8>(p, acc, mw, nw, l15, g4);
    if constexpr (OUTK == DAXQ_F32) {
        outputs_f32<NBJ, NBI, FP8>(p, acc, mw, nw, l15, g4, sx, sw, bias);
    } else if constexpr (LINES) {
        uint8_t* const own = smem + epilogue16_scales(NBJ, NBI) + (t >> 6) * epilogue16_part(NBJ, NBI);
        outputs_lines<NBJ, NBI, FP8, OUTK, ALWAYS_THROUGH>(p, acc, own, mw, nw, t & 63, sx, sw, bias);
    } else {
        outputs_straight<NBJ, NBI, FP8, OUTK>(p, acc, mw, nw, l15, g4, sx, sw, bias);
    }
}

// CUs of the current device (0 if the query fails), asked once per device
static inline int cu_count() {
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (dev >= 0 && dev < 64) {
        if (int c = cached[dev].load(std::memory_order_relaxed)) return c;
    }
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) return 0;
    if (dev >= 0 && dev < 64) cached[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

// Tiles of the last, partial round of a 256x256 launch that run as 128x128 quadrants, in workgroups behind those of
// the whole tiles; 0 = none.
// One workgroup of 256x256 tiles fills a CU, so a launch of R whole rounds and L more tiles takes R + 1 tile times
// however small L is.  As 4 L quadrants with a CU each (L <= a quarter of the CUs) the L tiles take half a tile time
// or less.  Measured as a second launch against the launch of whole tiles (INT8 / e4m3, K = 5120 unless noted; in one
// grid the quadrants start on the first CUs that come free, another +1 to +10 %, most on short launches):
//   4725 x 13824 (4 rounds + 2 tiles) +5.6 / +6.1 %; 8500 x 4096, K = 2048 (2 + 32) +9.9 / +9.9 %;
//   4095 x 4608, K = 1536 (1 + 32) +10.7 / +9.8 %, K = 8960 +24 / +26 %;
//   20000 x 5120 (6 + 44) +3.3 / +2.4 %; 75600 x 5120 in row groups (23 + 32) -0.6 / -0.8 %: over many rounds the CUs
//   drift apart and the early ones pick the last tiles up, so the cut is taken up to kTailMaxRounds whole rounds;
//   with two quadrants per CU (L up to half the CUs: 4725 x 5120, 1 + 124) -5.3 / -5.9 %: a round of 128x128 tiles
//   at two per CU takes as long as a round of 256x256 tiles, so those launches stay whole.
constexpr int kTailMaxRounds = 8;
static inline int tail_tiles(const GemmArgs& a, int tail) {
    if (tail == 1 || a.order != kOrderRowGroups) return 0;  // the banded order deals whole patches: its ids are not tile counts
    const int cus = cu_count();
    if (cus < 8) return 0;
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n, rounds = tiles / cus, left = tiles - rounds * cus;
    if (rounds < 1 || left == 0 || 4 * left > cus) return 0;
    return (tail == 2 || rounds <= kTailMaxRounds) ? (int)left : 0;
}
// The same for a last round of more than a quarter and at most half of the CUs' worth of tiles: those run as halves of
// 256 x 128 with a CU each (gemm_tile_fit.h), about 0.65 of a tile time instead of one.
static inline int tail_half_tiles(const GemmArgs& a, int tail) {
    if (tail == 1 || a.order != kOrderRowGroups) return 0;
    const int cus = cu_count();
    if (cus < 8) return 0;
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n, rounds = tiles / cus, left = tiles - rounds * cus;
    if (rounds < 1 || 4 * left <= cus || 2 * left > cus) return 0;
    return (tail == 2 || rounds <= kTailMaxRounds) ? (int)left : 0;
}

// How the 16-bit outputs of 256x256 tiles leave (GemmArgs::lines).  128x128 and fitted tiles run in one round, or as a launch's last
// one, and always take whole rows through the L2.
// Straight from the registers a store instruction writes 16 rows x 64 bytes.  Whole rows (outputs_lines, 256 bytes each) cost a trip
// through the LDS, which other workgroups' main loops hide as well or better over many rounds; with rows through the L2 less is left to
// write back when the launch ends, which short launches feel.  Rows that start on odd elements are split by the path to the L2.
// GEMM and quantiser, us, straight / whole rows / and through, INT8 unless noted:
//   rounds, K = 1536: 3200 x 5120 (1.02) 36.2 / 35.9 / 35.3   6400 x 5120 (1.95) 53.5 / 54.1 / 51.9   9830 x 5120 (3.05) 84.6 / 85.3 / 83.7
//     13000 x 5120 (4.0) 101.0 / 102.5 / 100.0   19600 x 5120 (6.0) 155.3 / 157.2 / 155.2   26000 x 5120 (8.0) 199.3 / 203.3 / 201.4
//     32760 x 4608 (9) 228.1 / 230.2 / 230.3
//   K = 5120: 4096 x 5120 per-tensor e5m2 (1.25) 99.7 / 99.1 / 96.7   6400 x 5120 (1.95) 132.7 / 132.9 / 132.3   9830 x 5120 (3.05) 213.0 / 213.1 / 211.5
//     13000 x 5120 (4.0) 262.0 / 262.6 / 264.4   75600 x 5120 e4m3 1523 / 1526 / 1530
//   row starts, 6400 rows, K = 1536: N = 5119 73.5 / 54.6 / 54.6   5124 62.6 / 62.2 / 63.3   5136 61.2 / 62.1 / 61.8   5152 61.3 / 62.0 / 60.8
//     20000 rows: N = 5119 219.1 / 162.3 / 167.2   5124 164.7 / 164.7 / 170.3   5152 160.1 / 163.6 / 164.7
static inline int lines_of(const GemmArgs& a) {
    if (a.acc || a.out_kind == DAXQ_F32) return kLinesNone;
    const uint64_t at = (uint64_t)(uintptr_t)a.out | (uint64_t)a.ldo * 2;
    if (at & 2) return kLinesPlain;  // (the last bit of ldo: rows on odd elements)
    const int64_t rounds = a.k < 4096 ? 4 : 2;
    return (at & 63) == 0 && (int64_t)a.m * a.n <= rounds * 65536 * cu_count() ? kLinesThrough : kLinesNone;
}

}  // namespace daxq
