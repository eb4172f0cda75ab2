// W8A8 GEMM tile of BM x BN outputs for INT8 and FP8 operands as a device function: the body of the kernels that fit the tile to
// the launch (gemm_tile_fit.hip) and of the 256 x 128 halves that run behind whole 256x256 tiles (gemm_tile256.hip,
// gemm_tile_fp8.hip).
//
// WM x WN wavefronts, each with NBI x NBJ blocks of 16x16 outputs.  The K loop walks pairs of 64-byte slices:
//   * both operands' fragments of a pair sit in registers twice (8 x (NBI + NBJ) x 2): those of pair q+1 are read during the
//     MFMAs of pair q;
//   * the LDS holds NS pairs of (BM + BN) x 128 bytes: at the barrier of pair q, the only one of a pair, pair q+1 has landed and
//     everyone has read pair q out of its slot, which takes the loads of pair q+NS; every load has NS-1 pairs to land;
//   * a load instruction takes 8 rows x 128 bytes, whole lines (gemm_tile256.hip says what that is worth).
// Same arithmetic as the 256x256 kernels.  INT8 accumulators are exact; an FP8 output element is the same sequence of MFMAs over the
// same K bytes in the same register positions as in gemm_tile_fp8.hip -- one MFMA per pair, a lane's fragments holding chunk
// l/16 of the pair's first slice, then of its second -- so its bits do not depend on which of the kernels computed it.
#pragma once

#include "gemm_tile.h"

namespace daxq {

template <int WM_, int WN_, int NBI_, int NBJ_, int NS_>
struct FitTile {
    static constexpr int WM = WM_, WN = WN_, NBI = NBI_, NBJ = NBJ_, NS = NS_;
    static constexpr int T = 64 * WM * WN, BM = 16 * NBI * WM, BN = 16 * NBJ * WN, BKP = 128;
    static constexpr int SLOT = (BM + BN) * BKP, SMEM = NS * SLOT;
    static constexpr int ROWS = T / 8;  // rows a load instruction of the workgroup takes
    static constexpr int A_LOADS = BM / ROWS, B_LOADS = BN / ROWS, PAIR_LOADS = A_LOADS + B_LOADS;
    // the way of 16-bit outputs to memory (tile_lines): groups of G blocks of rows per wavefront, so that the stores of one run beside
    // the arithmetic of the next (256 rows in two groups of four: 2000 x 4608 22.5 instead of 22.2 us); chunks of 16 bytes
    static constexpr int G = 2, GROUPS = NBI / G, GROUP_ROWS = 16 * G * WM;
    static constexpr int CHUNKS = BN / 8, STEPS = GROUP_ROWS * CHUNKS / T;  // of a row; stores of a group
    static constexpr int PERIOD = CHUNKS % 7 == 0 ? 7 : CHUNKS % 5 == 0 ? 5 : CHUNKS % 3 == 0 ? 3 : 1, PERIOD_ROWS = PERIOD * T / CHUNKS;
    static constexpr int OUT_ROW = 2 * BN + 16;  // bytes: 4 banks times an odd number
    static_assert(NBI % G == 0 && GROUP_ROWS * CHUNKS % T == 0 && PERIOD * T % CHUNKS == 0 && GROUP_ROWS % PERIOD_ROWS == 0, "whole stores");
    static_assert((16 * G) % PERIOD_ROWS == 0 || PERIOD_ROWS % (16 * G) == 0, "a step's rows are a lane's and a constant");
    static_assert(GROUPS * GROUP_ROWS * OUT_ROW <= SMEM, "the outputs fit into the LDS of the pairs");
    static_assert(BM % ROWS == 0 && BN % ROWS == 0, "whole load instructions");
    static_assert(NS >= 3 && SMEM <= 160 * 1024 && NS * PAIR_LOADS < 60, "LDS and load counter");
    static constexpr int SCALE_LOADS = NBI + 2 * NBJ;  // of the epilogue's scales and bias, behind the last tile loads
    static_assert((NS - 2) * PAIR_LOADS + SCALE_LOADS < 64, "the waits of the last pairs fit the load counter");
};
typedef FitTile<2, 2, 8, 4, 3> HalfTile;  // 256 x 128

// fragments of a pair: FP8 one MFMA operand of 8 registers, INT8 two of 4
template <bool FP8>
struct PairFrag {
    v4i h[2];
};
template <>
struct PairFrag<true> {
    v8i v;
};

template <class TILE, bool FP8, int F8, bool DUMP, int OUTK>
__device__ __forceinline__ void gemm_fit_body(const GemmArgs& p, const int m0, const int n0) {
    static_assert(OUTK == DAXQ_BF16 || !DUMP, "the accumulator dump exists with bf16 outputs");
    constexpr int WN = TILE::WN, NBI = TILE::NBI, NBJ = TILE::NBJ, NS = TILE::NS, BM = TILE::BM, BN = TILE::BN, BKP = TILE::BKP;
    constexpr int SLOT = TILE::SLOT, A_PART = BM * BKP, A_LOADS = TILE::A_LOADS, PAIR_LOADS = TILE::PAIR_LOADS, ROWS = TILE::ROWS;
    constexpr int BLOCKS = NBI * NBJ, NREG = FP8 ? BLOCKS : 2 * BLOCKS;           // MFMAs = scheduling regions of a pair
    constexpr int READS = FP8 ? NBI + NBJ : 2 * (NBI + NBJ);                      // fragment reads: whole (FP8) or one slice of one
    constexpr int RSTEP = NREG >= 2 * READS ? 2 : 1;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave / WN, wn = wave % WN;

    // ---- HBM side: lane l of a load instruction takes row l/8 and the 16-byte chunk that is stored at chunk l%8 of the row
    const uint32_t gsw = (uint32_t)(((t & 7) ^ ((t >> 3) & 7)) << 4);
    uint32_t voff_a = (uint32_t)(t >> 3) * (uint32_t)p.lda + gsw;
    uint32_t voff_b = (uint32_t)(t >> 3) * (uint32_t)p.ldb + gsw;
    const uint8_t* abase = p.a + (int64_t)m0 * p.lda;
    const uint8_t* bbase = p.b + (int64_t)n0 * p.ldb;
    const int64_t a_step = ROWS * p.lda, b_step = ROWS * p.ldb;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(DAXQ_LDS uint8_t*)smem;
    const uint32_t wave_lds = lds0 + (uint32_t)__builtin_amdgcn_readfirstlane(wave * 1024);
    // load g of a pair: the activation rows, then the weight rows.  Address = uniform row-block base (SGPR pair) + per-lane 32-bit
    // offset: no VALU work per load.
    auto issue_one = [&](uint32_t slot, int g) __attribute__((always_inline)) {
        const bool w = g >= A_LOADS;
        const int j = w ? g - A_LOADS : g;
        const uint8_t* src = w ? bbase + j * b_step : abase + j * a_step;
        const uint32_t dst = wave_lds + slot + (w ? A_PART : 0) + j * (ROWS * BKP);
        __builtin_amdgcn_global_load_lds((const DAXQ_GLOBAL void*)(src + (w ? voff_b : voff_a)), (DAXQ_LDS void*)(uintptr_t)dst, 16, 0, 0);
    };
    auto advance = [&]() {
        voff_a += BKP;
        voff_b += BKP;
    };

    // ---- LDS side: rows of 128 bytes, chunk c of row r at chunk c ^ (r & 7)
    const int lr = lane & 15, kg = lane >> 4;
    const int xo = (kg ^ (lr & 7)) << 4;
    const uint8_t* a_rd = smem + (wm * 16 * NBI + lr) * BKP + xo;
    const uint8_t* b_rd = smem + A_PART + (wn * 16 * NBJ + lr) * BKP + xo;
    const int to_up = 64 - 2 * (xo & 64);  // from a lane's chunk of the first slice to its chunk of the second
    const uint8_t *a_up = a_rd + to_up, *b_up = b_rd + to_up;
    typedef PairFrag<FP8> frag_t;
    // read r of a pair: the fragments of the activation blocks, then of the weight blocks (INT8: of the first slice, then of the second)
    auto read_frag = [&](uint32_t slot, int r, frag_t (&af)[NBI], frag_t (&bf)[NBJ]) __attribute__((always_inline)) {
        const int h = FP8 ? 0 : r / (NBI + NBJ), f = FP8 ? r : r % (NBI + NBJ);
        const bool w = f >= NBI;
        const int blk = w ? f - NBI : f;
        const uint32_t at = slot + blk * 16 * BKP;
        if constexpr (FP8) {
            const v4i lo = *reinterpret_cast<const v4i*>((w ? b_rd : a_rd) + at);
            const v4i up = *reinterpret_cast<const v4i*>((w ? b_up : a_up) + at);
            (w ? bf[w ? blk : 0] : af[w ? 0 : blk]).v = __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
        } else {
            (w ? bf[w ? blk : 0] : af[w ? 0 : blk]).h[h] = *reinterpret_cast<const v4i*>((h ? (w ? b_up : a_up) : (w ? b_rd : a_rd)) + at);
        }
    };

    typename Acc16<FP8>::type acc[NBJ][NBI];
    frag_t fa0[NBI] = {}, fb0[NBJ] = {}, fa1[NBI] = {}, fb1[NBJ] = {};  // by parity of the pair
    // weights are the MFMA "A" operand (format select cbsz), activations the "B" operand (blgp); accumulators tied in place
    auto mfma = [&](auto PAR, auto FIRST, int g) __attribute__((always_inline)) {
        const int h = g / BLOCKS, j = g % BLOCKS / NBI, i = g % NBI;
        auto& c = acc[j][i];
        if constexpr (!FP8) {
            const v4i bfr = decltype(PAR)::value ? fb1[j].h[h] : fb0[j].h[h];
            const v4i afr = decltype(PAR)::value ? fa1[i].h[h] : fa0[i].h[h];
            if (decltype(FIRST)::value && h == 0) asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, 0" : "=a"(c) : "v"(bfr), "v"(afr));
            else asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(c) : "v"(bfr), "v"(afr));
        } else {
            const v8i bfr = decltype(PAR)::value ? fb1[j].v : fb0[j].v;
            const v8i afr = decltype(PAR)::value ? fa1[i].v : fa0[i].v;
            if constexpr (decltype(FIRST)::value) {
                if constexpr (F8 == 0) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0" : "=a"(c) : "v"(bfr), "v"(afr));
                else if constexpr (F8 == kF8XE5) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0 blgp:1" : "=a"(c) : "v"(bfr), "v"(afr));
                else if constexpr (F8 == kF8WE5) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0 cbsz:1" : "=a"(c) : "v"(bfr), "v"(afr));
                else asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0 cbsz:1 blgp:1" : "=a"(c) : "v"(bfr), "v"(afr));
            } else {
                if constexpr (F8 == 0) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+a"(c) : "v"(bfr), "v"(afr));
                else if constexpr (F8 == kF8XE5) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 blgp:1" : "+a"(c) : "v"(bfr), "v"(afr));
                else if constexpr (F8 == kF8WE5) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 cbsz:1" : "+a"(c) : "v"(bfr), "v"(afr));
                else asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 cbsz:1 blgp:1" : "+a"(c) : "v"(bfr), "v"(afr));
            }
        }
    };

    const int Q = p.k / BKP;  // pairs; K is a multiple of 128
    uint32_t st[NS];          // slots of pairs q, q+1, ...
#pragma unroll
    for (int i = 0; i < NS; ++i) st[i] = i * SLOT;
    // One pair.  PAR: which register set it consumes.  ISSUE: pair q+NS exists, its loads go into the slot of pair q.
    // NEXT: pair q+1 exists, its fragments are read into the other set.  YOUNG: tile loads behind those of pair q+1 that
    // may stay in flight.  EXTRA: younger loads that are not tile loads.  FIRST: the accumulators start from zero.
    auto pair = [&](auto PAR, auto ISSUE, auto NEXT, auto YOUNG, auto EXTRA, auto FIRST) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(YOUNG.value + EXTRA.value) & lgkmcnt0_mask());
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int g = 0; g < NREG; ++g) {
            if constexpr (ISSUE.value) {  // in twos (one by one is as fast to 1 %)
#pragma unroll
                for (int l = 0; l < PAIR_LOADS; ++l)
                    if (l / 2 * 2 * NREG / PAIR_LOADS == g) issue_one(st[0], l);
            }
            if constexpr (NEXT.value) {
                if (g % RSTEP == RSTEP - 1 && g / RSTEP < READS) {
                    if constexpr (PAR.value) read_frag(st[1], g / RSTEP, fa0, fb0);
                    else read_frag(st[1], g / RSTEP, fa1, fb1);
                }
            }
            mfma(PAR, FIRST, g);
            if (g == NREG - 1) {
                if constexpr (ISSUE.value) advance();
                const uint32_t o = st[0];
#pragma unroll
                for (int i = 0; i + 1 < NS; ++i) st[i] = st[i + 1];
                st[NS - 1] = o;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // the epilogue's scales and bias, requested behind the last tile loads, each lane its own outputs': always NBI + 2 NBJ loads (a missing
    // bias reads a scale instead and is replaced by -0.0: x + (-0.0) == x bit for bit), so that the counts of the waits hold
    constexpr int SCALE_LOADS = TILE::SCALE_LOADS;
    typedef v4f loose_v4f __attribute__((aligned(4)));
    typedef v2u loose_v2u __attribute__((aligned(2)));
    const int mw = m0 + wm * 16 * NBI, nw = n0 + wn * 16 * NBJ;
    float sx[NBI];
    v4f sw[NBJ], bias[NBJ];
    v2u bias_bits[NBJ];  // bf16 / fp16
    auto request_scales = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NBI; ++i) sx[i] = p.sx[mw + 16 * i + lr];
#pragma unroll
        for (int j = 0; j < NBJ; ++j) {
            const int n = nw + 16 * j + 4 * kg;
            sw[j] = *reinterpret_cast<const loose_v4f*>(p.sw + n);
            if constexpr (OUTK == DAXQ_F32) bias[j] = *reinterpret_cast<const loose_v4f*>((p.bias ? reinterpret_cast<const float*>(p.bias) : p.sw) + n);
            else bias_bits[j] = *reinterpret_cast<const loose_v2u*>((p.bias ? p.bias : reinterpret_cast<const uint16_t*>(p.sw)) + n);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // Outputs of 16 bits leave by way of the LDS, as rows of the tile, and through the L2 to memory (store_through).  A launch of one
    // round writes all its outputs at its end.  Stored straight from the registers, 16 rows x 64 bytes an instruction, they took a CU 36
    // cycles per KB, and what lay in the L2s was written back behind the kernel, 2.4 us of nothing else at 4096 x 1536; whole rows take 17
    // cycles per KB, and half lines stored through the L2 are slower than ones that stay in it.  us, straight / rows / rows and
    // through, INT8 forwards: 4096 x 1536 x 1536 20.7 / 20.3 / 19.5, 2900 x 3080, K = 1000 fp16 20.0 / 20.2 / 19.1, 2000 x 4608, K = 1536
    // 22.7 / 22.7 / 21.4, 512 x 5120 x 5120 22.7 / 22.6 / 22.0, 4096 x 1537, K = 1536 24.3 / 20.8 / 20.0 (rows that start anywhere);
    // none of 25 launches slower by more than 0.5 %.
    // Chunk s T + t of a group of rows is the thread's at step s: its row and column repeat every PERIOD steps, PERIOD_ROWS rows further.
    // (put together here, where the first loads are waited for, and kept in registers)
    typedef TILE L;
    constexpr bool LINES = OUTK != DAXQ_F32;
    int64_t line_out[L::PERIOD];   // bytes from the tile's first output
    uint32_t line_lds[L::PERIOD];  // bytes from the group's first output in the LDS
    auto tile_lines = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < L::PERIOD; ++s) {
            const int c = s * L::T + t, r = c / L::CHUNKS, col = c - r * L::CHUNKS;  // row r of the group's, wavefront row by wavefront row
            line_out[s] = ((int64_t)(r / (16 * L::G) * (16 * NBI) + r % (16 * L::G)) * p.ldo + col * 8) * 2;
            line_lds[s] = (uint32_t)(r * L::OUT_ROW + col * 16);
            asm volatile("" : "+v"(line_out[s]), "+v"(line_lds[s]));
        }
    };
    auto issue_pair = [&](uint32_t slot) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < PAIR_LOADS; ++g) issue_one(slot, g);
        advance();
    };

    if (Q > NS) {
        // ---- prologue: pairs 0 .. NS-1 in flight, pair 0 landed, its fragments in set 0
#pragma unroll
        for (int s = 0; s < NS; ++s) issue_pair(st[s]);
        if constexpr (LINES) tile_lines();
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 1) * PAIR_LOADS));
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int r = 0; r < READS; ++r) read_frag(st[0], r, fa0, fb0);
        // pair 0, then the steady pairs two at a time; the NS pairs of the tail are code paths with fixed sets (odd, even, ...
        // after an even number of pairs behind pair 0, else the fragments move over to the other set once)
        typedef Int<(NS - 2) * PAIR_LOADS> Steady;
        pair(No{}, Yes{}, Yes{}, Steady{}, Int<0>{}, Yes{});
        int q = 1;
        for (; q + NS + 1 < Q; q += 2) {
            pair(Yes{}, Yes{}, Yes{}, Steady{}, Int<0>{}, No{});
            pair(No{}, Yes{}, Yes{}, Steady{}, Int<0>{}, No{});
        }
        if (q + NS < Q) {
            pair(Yes{}, Yes{}, Yes{}, Steady{}, Int<0>{}, No{});
#pragma unroll
            for (int i = 0; i < NBI; ++i) fa1[i] = fa0[i];
#pragma unroll
            for (int j = 0; j < NBJ; ++j) fb1[j] = fb0[j];
        }
        request_scales();
        auto tail = [&](auto T) __attribute__((always_inline)) {
            constexpr int n = decltype(T)::value;  // of NS
            pair(Int<n % 2 == 0>{}, No{}, Int<(n < NS - 1)>{}, Int<(n < NS - 2 ? NS - 2 - n : 0) * PAIR_LOADS>{}, Int<SCALE_LOADS>{}, No{});
        };
        for_up<0, NS>(tail);
        mfma_settle();
    } else {
        // ---- short K: every pair has a slot
        for (int q = 0; q < Q; ++q) issue_pair(q * SLOT);
        request_scales();
        if constexpr (LINES) tile_lines();
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        __builtin_amdgcn_s_barrier();
        for (int q = 0; q < Q; ++q) {
#pragma unroll
            for (int r = 0; r < READS; ++r) read_frag(q * SLOT, r, fa0, fb0);
            __builtin_amdgcn_s_waitcnt(lgkmcnt0_mask() & vmcnt_imm(63));
            __builtin_amdgcn_sched_barrier(0);
            if (q == 0) {
#pragma unroll
                for (int g = 0; g < NREG; ++g) mfma(No{}, Yes{}, g);
            } else {
#pragma unroll
                for (int g = 0; g < NREG; ++g) mfma(No{}, No{}, g);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();  // (the outputs go where other wavefronts may still read fragments)
        mfma_settle();
    }

    // ... and every accumulator is passed through an empty statement, which no read of it can move above
#pragma unroll
    for (int j = 0; j < NBJ; ++j)
#pragma unroll
        for (int i = 0; i < NBI; ++i) asm volatile("" : "+a"(acc[j][i]));

#pragma unroll
    for (int j = 0; j < NBJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (OUTK != DAXQ_F32) {
                const uint32_t w = bias_bits[j][r >> 1], b = r & 1 ? w >> 16 : w & 0xffffu;
                bias[j][r] = OUTK == DAXQ_F16 ? f16_bits_to_f32((uint16_t)b) : bf16_bits_to_f32(b);
            }
            if (!p.bias) bias[j][r] = -0.0f;
        }
    if constexpr (DUMP) dump_tile16<NBJ, NBI, FP8>(p, acc, mw, nw, lr, kg);
    if constexpr (!LINES) {
        outputs_f32<NBJ, NBI, FP8>(p, acc, mw, nw, lr, kg, sx, sw, bias);
    } else {
        uint8_t* const to = smem + (wm * 16 * L::G + lr) * L::OUT_ROW + (wn * 16 * NBJ + 4 * kg) * 2;
        uint8_t* const out = reinterpret_cast<uint8_t*>(p.out) + ((int64_t)m0 * p.ldo + n0) * 2;
        v4u line[L::STEPS];
        auto store_group = [&](int g) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < L::STEPS; ++s) {
                constexpr int GR = 16 * L::G;
                const int r = s / L::PERIOD * L::PERIOD_ROWS;  // (uniform: whole segments of GR rows, or a part of one)
                store_through(out + (int64_t)(r / GR * (16 * NBI) + r % GR + g * GR) * p.ldo * 2 + line_out[s % L::PERIOD], line[s]);
            }
        };
#pragma unroll
        for (int g = 0; g < L::GROUPS; ++g) {
#pragma unroll
            for (int ii = 0; ii < L::G; ++ii) {
                const int i = g * L::G + ii;
#pragma unroll
                for (int j = 0; j < NBJ; ++j)
                    *reinterpret_cast<uint2*>(to + (g * L::GROUP_ROWS + ii * 16) * L::OUT_ROW + j * 32) = outputs4<FP8, OUTK>(acc[j][i], sx[i], sw[j], bias[j]);
                if (g > 0 && ii == 0) store_group(g - 1);  // their reads have come back meanwhile
            }
            __syncthreads();
#pragma unroll
            for (int s = 0; s < L::STEPS; ++s)
                line[s] = *reinterpret_cast<const v4u*>(smem + (g * L::GROUP_ROWS + s / L::PERIOD * L::PERIOD_ROWS) * L::OUT_ROW + line_lds[s % L::PERIOD]);
        }
        store_group(L::GROUPS - 1);
    }
}

// half `half_id & 1` of the 256x256 tile quad_base - 1 + half_id / 2 of the row-group order (launches that leave tiles over after
// their whole rounds of workgroups: tail_half_tiles)
template <bool FP8, int F8, bool DUMP, int OUTK>
__device__ __forceinline__ void gemm_half_body(const GemmArgs& p, const int half_id) {
    int tm, tn;
    tile_of_block(p.gm, p.quad_base - 1 + (half_id >> 1), p.tiles_m, p.tiles_n, tm, tn);
    int m0 = tm * 256, n0 = tn * 256;
    m0 = m0 + 256 <= p.m ? m0 : p.m - 256;
    n0 = (n0 + 256 <= p.n ? n0 : p.n - 256) + (half_id & 1) * 128;
    gemm_fit_body<HalfTile, FP8, F8, DUMP, OUTK>(p, m0, n0);
}

}  // namespace daxq
