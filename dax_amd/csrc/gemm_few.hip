// The whole forward of a W8A8 linear of at most eight rows (or up to 64 short ones) in one launch: every workgroup quantises the activation
// for itself, in LDS, while its share of the weight arrives, and multiplies (gfx950).
//
// What bounds it: the launches.  The quantiser and the GEMM of such a call take 2 and 3 to 7 us, their launches cost the host 2.8 to
// 3.6 us each (a per-tensor scale is a third one), and the second one starts when the first has ended and drained.  The quantised rows
// are few (40 KB up to eight rows, 64 KB beyond), so that quantising them once per workgroup costs about what waiting for the weight does anyway.
// Forwards back to back, us, separate launches -> this: 1 x 1536 x 1536 8.2 -> 5.5, 4 x 1536 x 1536 e5m2 under a per-tensor scale
// 10.9 -> 5.7, 1 x 5120 x 5120 e4m3 8.2 -> 7.9 (its kernel).
//
// Work decomposition
//   workgroup  8 wavefronts, two groups (CG) of 16 output columns
//   quantiser  the wavefronts are dealt to the rows (more than eight: each takes several); all of the activation is in flight at once,
//              maxima meet in LDS once, and the bytes go to LDS rows of K + 16 bytes (the rows a fragment read touches then lie in different banks)
//   GEMM       as gemm_rows.hip: wavefront w < CG x KS streams K / KS bytes of 16 weight rows through an LDS ring of its own, the
//              first R steps of 128 bytes requested behind the activation's loads and in front of the quantiser's arithmetic.  INT8 cuts
//              K over KS = 4 wavefronts (sums of integers); FP8 runs KS = 1, so that an output element is the sequence of MFMAs over
//              the same K bytes in the same register positions that every other kernel runs.
// Same statistics, scales, bytes and epilogue as quant_rows.hip and gemm_rows.hip, whose helpers it calls: the outputs are their bits.
#include "gemm_rows.h"
#include "quant_rows.h"

namespace daxq {

// a lane's value in every lane
__device__ __forceinline__ float lane_value(float f, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), lane)); }

struct FewArgs {
    GemmArgs g;           // b, sw, bias, out, ldb, ldo, m, n, k (padded); a, sx unused
    const char* x;        // [m, kx] elements
    const float* scale1;  // static: the tensor's scale
    int64_t ld_x;
    int kx;               // columns of x, a multiple of 8
    int round_x, scheme;  // kFewToken ...
};
enum { kFewToken = 0, kFewTensor = 1, kFewStatic = 2 };

constexpr int kFewWaves = 8;
// columns; quantised bytes in LDS, rows counted as they are dealt out.  WIDE: twice as many, in kernels of their own (the longer
// code of more chunks per lane costs the smaller calls 0.25 us)
constexpr int kFewMaxK = 16384, kFewMaxBytes = 20480, kFewWideBytes = 40960;
constexpr int few_rows_bytes(int rows, bool one) { return !one ? 32768 : rows == 16 ? 40960 : rows == 32 ? 49152 : 65536; }  // the same for more than eight rows
constexpr int kFewRingI8 = 2 * 4 * 4 * 2048, kFewRingF8 = 2 * 1 * 10 * 2048;  // LDS of the weight's rings: CG x KS x R steps of 2 KB
// chunks of 8 elements per lane and row: up to eight rows 8 / rows wavefronts share one, of more of them a wavefront takes rows / 8
constexpr int few_chunks(int rows, bool wide, bool one) {
    if (rows > kFewWaves) return (few_rows_bytes(rows, one) / rows + 511) / 512;
    return ((rows == 1 ? kFewMaxK : wide ? kFewWideBytes : kFewMaxBytes) + kFewWaves * 512 - 1) / (kFewWaves * 512);
}

// MR: rows the wavefronts are dealt to (1, 2, 4, 8, 16, 32, 64).  ONE: one scale for the tensor (dynamic or the caller's) instead of one per row
template <bool FP8, int F8, int XT, bool ONE, int MR, bool WIDE, int CG, int KS, int R>
__global__ __launch_bounds__(64 * kFewWaves) void gemm_few_kernel(const FewArgs a) {
    typedef typename Acc16<FP8>::type acc_t;
    constexpr int XB = XT == DAXQ_F32 ? 4 : 2, OUTK = XT, FMT = !FP8 ? 0 : (F8 & kF8XE5) ? 2 : 1;
    constexpr float kMax = FMT == 0 ? 127.0f : FMT == 1 ? 448.0f : 57344.0f;
    constexpr int NCH = few_chunks(MR, WIDE, ONE), WPR = MR < kFewWaves ? kFewWaves / MR : 1;  // wavefronts per row
    constexpr int RW = MR > kFewWaves ? MR / kFewWaves : 1, MB = (MR + 15) / 16;           // rows per wavefront, blocks of 16 rows
    constexpr int STEP = 2048, L = 2;  // LDS of a step: 16 weight rows of 128 bytes, two load instructions
    static_assert(CG * KS <= kFewWaves && R * L < 64, "wavefronts, load counter");
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    const GemmArgs& p = a.g;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l15 = lane & 15, g4 = lane >> 4;
    const int xs = p.k + 16;  // LDS row of quantised bytes
    uint8_t* s_x = smem + CG * KS * R * STEP;
    uint32_t* s_max = reinterpret_cast<uint32_t*>(s_x + MR * xs);  // [8]
    float* s_sx = reinterpret_cast<float*>(s_max + kFewWaves);       // [MR]
    static_assert(CG * KS * R * STEP >= (KS > 1 ? kFewWaves * MB * 1024 : 0), "the partial sums fit the rings");

    // ---- the activation: WPR wavefronts a row, or RW rows a wavefront, all of it requested at once (beyond the row or the rows: the
    //      last chunk or row again)
    const int row = wave / WPR, rpart = wave % WPR, nch = a.kx >> 3;  // a wavefront's first row; the others lie kFewWaves apart
    Chunk<XT> v[RW][NCH];
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const int at = row + r * kFewWaves;
        const char* xrow = a.x + (int64_t)(at < p.m ? at : p.m - 1) * a.ld_x * XB;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            if (i * WPR * 64 < nch && (r == 0 || r * kFewWaves < p.m)) {
                const int c = (i * WPR + rpart) * 64 + lane;
                load_chunk_shared<XT>(v[r][i], xrow + (uint32_t)(c < nch ? c : nch - 1) * (8u * XB));
            }
        }
    }
    // ---- the weight's first steps (gemm_rows.hip)
    const bool works = CG * KS == kFewWaves || wave < CG * KS;
    const int group = wave / KS, part = wave % KS;
    const int n0 = ((int)blockIdx.x * CG + group) * 16;
    const int nc = n0 + 4 * g4;  // a lane owns output row l % 16 of the block and 4 consecutive columns
    const ColumnBits<OUTK> cols(p, nc);
    const float scale1 = ONE && a.scheme == kFewStatic ? a.scale1[0] : 0.0f;
    __builtin_amdgcn_sched_barrier(0);
    const int steps = p.k >> 7;
    const int first = steps * part / KS, cnt = works && n0 < p.n ? steps * (part + 1) / KS - first : 0;
    const int lrow = lane >> 3;
    const uint32_t gsw = (uint32_t)(((lane & 7) ^ lrow) << 4);
    const uint8_t* wbase = p.b + (int64_t)n0 * p.ldb + (int64_t)first * 128;
    uint32_t woff[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) woff[h] = (uint32_t)(n0 + h * 8 + lrow < p.n ? h * 8 + lrow : p.n - 1 - n0) * (uint32_t)p.ldb + gsw;
    const uint32_t ring = (uint32_t)(uintptr_t)(DAXQ_LDS uint8_t*)smem + (uint32_t)wave * (R * STEP);
    auto load = [&](int step, uint32_t slot) __attribute__((always_inline)) {
        const uint8_t* w = wbase + (int64_t)step * 128;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            __builtin_amdgcn_global_load_lds((const DAXQ_GLOBAL void*)(w + woff[h]), (DAXQ_LDS void*)(uintptr_t)(ring + slot + h * 1024), 16, 0, 0);
    };
    const int ahead = cnt < R ? cnt : R;
#pragma unroll
    for (int s = 0; s < R; ++s)
        if (s < ahead) load(s, s * STEP);
    __builtin_amdgcn_sched_barrier(0);

    // ---- scales
    auto sync = [&]() __attribute__((always_inline)) {  // (LDS traffic only: the weight's loads stay in flight)
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(63) & lgkmcnt0_mask());
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    // lane r holds the scale of the wavefront's r-th row (all lanes that of the tensor, or of the only row)
    float s = scale1;
    if (!ONE || a.scheme != kFewStatic) {
        uint32_t mine = 0;
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            uint32_t amax = ONE ? mine : 0;
#pragma unroll
            for (int i = 0; i < NCH; ++i)
                if (i * WPR * 64 < nch && (r == 0 || r * kFewWaves < p.m)) amax = chunk_amax<XT>(amax, v[r][i]);
            if constexpr (ONE) {
                mine = amax;
            } else {
                amax = wave_max_u32(amax_of_lane<XT>(amax));
                mine = r == 0 || lane == r ? amax : mine;
            }
        }
        if constexpr (ONE) mine = wave_max_u32(amax_of_lane<XT>(mine));
        if (ONE || WPR > 1) {  // meets the maxima of the row's other wavefronts, or (rows beyond m repeat the last one) of all
            if (lane == 0) s_max[wave] = mine;
            sync();
#pragma unroll
            for (int w = 0; w < (ONE ? kFewWaves : WPR); ++w) {
                const uint32_t o = s_max[ONE ? w : row * WPR + w];
                mine = o > mine ? o : mine;
            }
        }
        s = scale_from_amax_bits_rt<XT>(mine, kMax, kEps, a.round_x);
    }
    if (rpart == 0 && lane < RW) s_sx[row + lane * kFewWaves] = s;
    // ---- bytes: a row under its own scale takes one form (a bf16 row kOwn; fp16 and fp32 rows, int8 only, kDivide), the one scale of a
    //      tensor picks one
    const float inv = 1.0f / s;  // IEEE division, not v_rcp_f32
    auto store = [&](auto FORM) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            if (r > 0 && r * kFewWaves >= p.m) continue;
            const float sr = RW == 1 ? s : lane_value(s, r), ir = RW == 1 ? inv : lane_value(inv, r);
#pragma unroll
            for (int i = 0; i < NCH; ++i) {
                if (i * WPR * 512 >= p.k) continue;
                const int c = (i * WPR + rpart) * 64 + lane;
                uint2 o = make_uint2(0, 0);
                if (i * WPR * 64 < nch) {
                    float f[8];
                    chunk_values<XT>(v[r][i], f);
                    o = quant8<FMT, decltype(FORM)::value, XT>(f, sr, ir);
                }
                if (c * 8 < p.k) *reinterpret_cast<uint2*>(s_x + (row + r * kFewWaves) * xs + c * 8) = c < nch ? o : make_uint2(0, 0);
            }
        }
    };
    if constexpr (ONE) with_form<FMT, XT>(s, kMax, a.scheme == kFewStatic, a.round_x, a.scheme == kFewTensor, store);
    else store(std::integral_constant<int, XT == DAXQ_BF16 ? kOwn : kDivide>{});
    sync();

    // ---- the GEMM
    const int xo = (g4 ^ (l15 & 7)) << 4;
    const uint8_t *rd = smem + wave * (R * STEP) + l15 * 128 + xo, *rd_up = rd + (64 - 2 * (xo & 64));
    // (rows of a block beyond the ones dealt out repeat the last of them; those beyond m that nobody wrote are multiplied and not stored)
    const uint8_t* xr = s_x + (l15 < MR ? l15 : MR - 1) * xs + (int64_t)first * 128 + g4 * 16;
    acc_t acc[MB] = {};
    auto next_slot = [](uint32_t slot) { return slot == (R - 1) * STEP ? 0 : slot + STEP; };
    auto work = [&](auto STEPS, auto MORE, int step, uint32_t slot) __attribute__((always_inline)) {
        constexpr int U = decltype(STEPS)::value;
        v8i w[U], x[U][MB];
        uint32_t at[U];
        at[0] = slot;
#pragma unroll
        for (int u = 1; u < U; ++u) at[u] = next_slot(at[u - 1]);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const v4i lo = *reinterpret_cast<const v4i*>(rd + at[u]), up = *reinterpret_cast<const v4i*>(rd_up + at[u]);
            w[u] = __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                const uint8_t* xb = xr + i * 16 * xs + (step + u) * 128;
                const v4i xl = *reinterpret_cast<const v4i*>(xb), xu = *reinterpret_cast<const v4i*>(xb + 64);
                x[u][i] = __builtin_shufflevector(xl, xu, 0, 1, 2, 3, 4, 5, 6, 7);
            }
        }
        if constexpr (MORE.value) {
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(63) & lgkmcnt0_mask());  // the reads are over
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; ++u) load(step + u + R, at[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < MB; ++i) acc[i] = mfma_step<FP8, F8>(w[u], x[u][i], acc[i]);
        __builtin_amdgcn_sched_barrier(0);
    };
    int step = 0;
    uint32_t slot = 0;
    for (; step + R + 1 < cnt; step += 2) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((R - 2) * L));
        __builtin_amdgcn_sched_barrier(0);
        work(Int<2>{}, Yes{}, step, slot);
        slot = next_slot(next_slot(slot));
    }
    for (; step + R < cnt; ++step) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((R - 1) * L));
        __builtin_amdgcn_sched_barrier(0);
        work(Int<1>{}, Yes{}, step, slot);
        slot = next_slot(slot);
    }
    auto tail = [&](auto T) __attribute__((always_inline)) {  // T steps behind this one
        constexpr int t = decltype(T)::value;
        if (t >= ahead) return;
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(t * L));
        __builtin_amdgcn_sched_barrier(0);
        work(Int<1>{}, No{}, step, slot);
        slot = next_slot(slot);
        ++step;
    };
    for_down<R - 1>(tail);

    v4i* s_part = reinterpret_cast<v4i*>(smem);  // [wave][block][lane], in the rings, which everyone has left
    if constexpr (KS > 1) {
        sync();
#pragma unroll
        for (int i = 0; i < MB; ++i) s_part[(wave * MB + i) * 64 + lane] = __builtin_bit_cast(v4i, acc[i]);
        sync();
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        if (KS > 1 && i % KS != part) continue;  // the wavefronts of a K range share the row blocks out
        if constexpr (KS > 1) {
            v4i sum = s_part[(group * KS * MB + i) * 64 + lane];
#pragma unroll
            for (int w = 1; w < KS; ++w) sum += s_part[((group * KS + w) * MB + i) * 64 + lane];
            acc[i] = __builtin_bit_cast(acc_t, sum);
        }
        const int m = i * 16 + l15;
        if (!works || m >= p.m || nc >= p.n) continue;
        store_columns<FP8, OUTK>(p, acc[i], s_sx[m], cols, m, nc);
    }
}

// args null: only raises the kernel's LDS limit on the current device
template <bool FP8, int F8, int XT, bool ONE, int MR, bool WIDE = false>
static int launch_few_one(const FewArgs* a, hipStream_t st) {
    constexpr int CG = 2, KS = FP8 ? 1 : 4, R = FP8 ? 10 : 4;  // (rings of 15 and 20 steps: 0 to 3 % slower, a CU then has room for fewer workgroups)
    auto kern = gemm_few_kernel<FP8, F8, XT, ONE, MR, WIDE, CG, KS, R>;
    static_assert(CG * KS * R * 2048 == (FP8 ? kFewRingF8 : kFewRingI8), "rings");
    static std::atomic<uint64_t> lds_set{0};  // per instantiation
    constexpr int ring = FP8 ? kFewRingF8 : kFewRingI8;
    constexpr int most = ring + (MR > kFewWaves ? few_rows_bytes(MR, ONE) : WIDE ? kFewWideBytes : kFewMaxBytes) + MR * 16 + (kFewWaves + MR) * 4;
    static_assert(most <= 160 * 1024, "LDS");
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), most, lds_set)) return rc;
    if (!a) return DAXQ_OK;
    const int lds = ring + MR * (a->g.k + 16) + (kFewWaves + MR) * 4;
    launch_kernel(kern, dim3((unsigned)((a->g.n + 16 * CG - 1) / (16 * CG))), dim3(64 * kFewWaves), lds, st, *a);
    return check_launch("gemm_few");
}

template <bool FP8, int F8, int XT, bool ONE>
static int launch_few_rows(const FewArgs* a, int m, bool wide, hipStream_t st) {
    if constexpr (ONE) {
        if (m > 32) return launch_few_one<FP8, F8, XT, ONE, 64>(a, st);
    }
    if (m > 16) return launch_few_one<FP8, F8, XT, ONE, 32>(a, st);
    if (m > 8) return launch_few_one<FP8, F8, XT, ONE, 16>(a, st);
    if (wide) return m <= 4 ? launch_few_one<FP8, F8, XT, ONE, 4, true>(a, st) : launch_few_one<FP8, F8, XT, ONE, 8, true>(a, st);
    if (m <= 1) return launch_few_one<FP8, F8, XT, ONE, 1>(a, st);
    if (m <= 2) return launch_few_one<FP8, F8, XT, ONE, 2>(a, st);
    if (m <= 4) return launch_few_one<FP8, F8, XT, ONE, 4>(a, st);
    return launch_few_one<FP8, F8, XT, ONE, 8>(a, st);
}

template <bool ONE>
static int launch_few(const FewArgs* a, int m, bool wide, int x_fmt, int x_dtype, hipStream_t st) {
    if (x_fmt == DAXQ_FMT_E4M3) return launch_few_rows<true, 0, DAXQ_BF16, ONE>(a, m, wide, st);
    if (x_fmt == DAXQ_FMT_E5M2) return launch_few_rows<true, kF8XE5, DAXQ_BF16, ONE>(a, m, wide, st);
    if (x_dtype == DAXQ_F16) return launch_few_rows<false, 0, DAXQ_F16, ONE>(a, m, wide, st);
    if (x_dtype == DAXQ_F32) return launch_few_rows<false, 0, DAXQ_F32, ONE>(a, m, wide, st);
    return launch_few_rows<false, 0, DAXQ_BF16, ONE>(a, m, wide, st);
}

int prepare_few_kernels() {
    int rc = 0;
    auto prepare = [&](int m, bool wide, int fmt, int x) {
        if (!rc) rc = launch_few<false>(nullptr, m, wide, fmt, x, nullptr);
        if (!rc) rc = launch_few<true>(nullptr, m, wide, fmt, x, nullptr);
    };
    for (int m : {1, 2, 4, 8, 16, 32, 64})
        for (bool wide : {false, true}) {
            if (wide && (m < 4 || m > 8)) continue;
            for (int x : {DAXQ_BF16, DAXQ_F16, DAXQ_F32}) prepare(m, wide, DAXQ_FMT_I8, x);
            for (int f : {DAXQ_FMT_E4M3, DAXQ_FMT_E5M2}) prepare(m, wide, f, DAXQ_BF16);
        }
    return rc;
}

// More than eight rows: the longest K (padded) whose forward is one launch.  Quantising in every workgroup costs the same at any N, so
// K and the number of rows draw the line (the quantiser's arithmetic: FP8 elements take more of it than int8 ones, fp32 ones more
// loads), up to N = 8192, where a workgroup has a CU to itself; beyond, two share one and quantise one after the other.  A tensor's scale
// saves a third launch or the second reading of the matrix.  us per call on the GPU, separate launches / one; weights near, out of reach
// of the caches.  The lines are drawn for forwards back to back, which besides save the 3.6 us that the host takes for a launch and its
// buffers (every size here 10.5 / 6.9), and for weights out of reach, a model's: what loses is FP8 of 17 to 32 rows beyond K = 512 and
// 16 rows at K = 2048 in a graph that replays one weight, up to 0.9 us (32 x 5120, K = 512 e4m3 4.6 / 4.4; 6.0 / 5.2, K = 640 4.8 / 5.6; 6.6 / 6.2;
// 17 rows, K = 768 4.7 / 5.1; 6.5 / 5.8).
//   own scales        16 x 1536 x 1536 int8 5.1 / 4.7; 7.1 / 5.0    e4m3 5.4 / 5.3; 7.2 / 5.3         16 x 8192, K = 2048 int8 6.2 / 5.7; 8.0 / 7.5   e4m3 6.0 / 6.2; 8.0 / 7.4
//                     16 x 4096, K = 2560 int8 6.3 / 5.8; 7.2 / 7.5  e4m3 6.2 / 7.0; 7.1 / 7.5         16 x 1536, K = 2048 fp32 5.4 / 5.8; 6.9 / 6.2   K = 1536 5.2 / 5.1; 6.8 / 5.3
//                     32 x 1536, K = 512 int8 5.0 / 4.4; 6.9 / 4.6   e4m3 5.2 / 4.9; 6.7 / 4.9         32 x 5120, K = 1024 int8 5.3 / 5.4; 6.5 / 6.3   e4m3 5.3 / 6.3; 7.1 / 6.6
//                     32 x 5120, K = 768 e4m3 5.2 / 6.1; 7.1 / 6.2   fp32 5.4 / 6.2; 7.3 / 6.5         16 x 13824, K = 256 int8 4.8 / 4.4; 8.3 / 4.6   K = 1536 6.2 / 8.2; 8.9 / 10.8
//   one of the tensor 16 x 1536, K = 2560 int8 7.5 / 5.9; 7.8 / 6.3  e5m2 7.9 / 7.4; 8.0 / 7.6         32 x 5120, K = 1536 int8 7.9 / 6.5; 9.4 / 7.7   e5m2 7.8 / 8.0; 9.3 / 9.2
//                     32 x 1536, K = 1024 e5m2 7.0 / 6.6; 7.1 / 6.8  64 x 1536, K = 640 int8 7.5 / 7.4; 7.6 / 7.6   fp16 7.6 / 7.9; 7.6 / 8.1   e5m2 7.2 / 9.1; 7.3 / 9.3
//                     64 x 5120, K = 1024 int8 8.9 / 7.6; 9.9 / 8.5  64 x 5120, K = 256 e5m2 7.2 / 6.6; 7.3 / 6.6   32 x 13824, K = 256 int8 7.2 / 5.7; 7.6 / 5.8   K = 512 7.7 / 8.0; 8.5 / 8.9
static int64_t few_rows_most_k(int x_dtype, bool f8, bool tensor, int64_t m, int64_t n) {
    const bool fp32 = x_dtype == DAXQ_F32;
    if (n > 8192) return (tensor ? m <= 32 : m <= 16) ? 256 : 0;
    if (tensor) {
        if (m <= 16) return fp32 ? 2048 : 2560;
        if (m <= 32) return f8 || fp32 ? 1024 : 1536;
        return f8 || fp32 ? 256 : x_dtype == DAXQ_BF16 && n >= 4096 ? 1024 : 512;
    }
    if (m <= 16) return fp32 ? 1536 : 2048;
    return m > 32 ? 0 : fp32 ? 512 : f8 ? 768 : 1024;
}

// rows as the wavefronts are dealt to them
static inline int64_t few_dealt(int64_t m) { return m <= 2 ? m : m <= 4 ? 4 : m <= 8 ? 8 : m <= 16 ? 16 : m <= 32 ? 32 : 64; }

// formats, element types and sizes that the kernels take at all
static bool few_forms(int x_dtype, int x_fmt, int w_fmt, int out_dtype, int scheme, int act_scale_round, int64_t n, int64_t k) {
    if (scheme < kFewToken || scheme > kFewStatic) return false;
    // (an fp8 row under a scale that is not rounded to bf16 takes another form per row: left to the quantiser)
    if (x_fmt != DAXQ_FMT_I8 && scheme == kFewToken && act_scale_round != DAXQ_SCALE_ROUND_X) return false;
    const bool i8 = x_fmt == DAXQ_FMT_I8 && w_fmt == DAXQ_FMT_I8;
    const bool f8 = (x_fmt == DAXQ_FMT_E4M3 || x_fmt == DAXQ_FMT_E5M2) && w_fmt == DAXQ_FMT_E4M3 && x_dtype == DAXQ_BF16;
    if ((!i8 && !f8) || x_dtype != out_dtype || x_dtype < DAXQ_BF16 || x_dtype > DAXQ_F32) return false;
    return k >= 8 && k % 8 == 0 && k <= kFewMaxK && n >= (f8 ? 128 : 1) && n <= (1 << 20);
}

// a call that the entry point `what` takes
static int few_linear(const char* what, int x_dtype, int x_fmt, int w_fmt, int out_dtype, int scheme, int act_scale_round, const void* x, int64_t ld_x,
                      const float* in_scale, const void* wq, int64_t ld_wq, const float* sw, const void* bias, void* out, int64_t ld_out,
                      int64_t m, int64_t n, int64_t k, daxq_stream_t stream) {
    const int64_t kp = (k + DAXQ_K_ALIGN - 1) / DAXQ_K_ALIGN * DAXQ_K_ALIGN;
    if ((scheme == kFewStatic) != (in_scale != nullptr)) return fail(DAXQ_ERR_ARG, "%s: scheme %d takes in_scale: %d", what, scheme, scheme == kFewStatic);
    if (act_scale_round != DAXQ_SCALE_ROUND_X && act_scale_round != DAXQ_SCALE_ROUND_NONE)
        return fail(DAXQ_ERR_ARG, "%s: unknown scale rounding %d", what, act_scale_round);
    if (!x || !wq || !sw || !out) return fail(DAXQ_ERR_ARG, "%s: null pointer", what);
    if (ld_x < k || ld_wq < kp || ld_out < n || ld_wq >= (1 << 26)) return fail(DAXQ_ERR_ARG, "%s: bad leading dimension", what);
    const uintptr_t xa = x_dtype == DAXQ_F32 ? 3 : 1;
    if (((uintptr_t)x & xa) || ((uintptr_t)out & xa) || ((uintptr_t)bias & xa) || ((uintptr_t)sw & 3) || ((uintptr_t)in_scale & 3) ||
        ((uintptr_t)wq & 15) || (ld_wq & 15))
        return fail(DAXQ_ERR_ALIGN, "%s: misaligned pointer or weight rows", what);
    FewArgs a = {};
    a.g.b = static_cast<const uint8_t*>(wq);
    a.g.sw = sw;
    a.g.bias = static_cast<const uint16_t*>(bias);
    a.g.out = static_cast<uint16_t*>(out);
    a.g.ldb = ld_wq;
    a.g.ldo = ld_out;
    a.g.m = (int)m;
    a.g.n = (int)n;
    a.g.k = (int)kp;
    a.x = static_cast<const char*>(x);
    a.scale1 = in_scale;
    a.ld_x = ld_x;
    a.kx = (int)k;
    a.round_x = act_scale_round == DAXQ_SCALE_ROUND_X;
    a.scheme = scheme;
    const bool wide = m > 2 && m <= 8 && few_dealt(m) * kp > kFewMaxBytes;
    if (scheme == kFewToken) return launch_few<false>(&a, (int)m, wide, x_fmt, x_dtype, (hipStream_t)stream);
    return launch_few<true>(&a, (int)m, wide, x_fmt, x_dtype, (hipStream_t)stream);
}

}  // namespace daxq

extern "C" {

int daxq_linear_few_applies(int x_dtype, int x_fmt, int w_fmt, int out_dtype, int scheme, int act_scale_round, int64_t m, int64_t n, int64_t k) {
    using namespace daxq;
    if (m < 1 || m > 8 || !few_forms(x_dtype, x_fmt, w_fmt, out_dtype, scheme, act_scale_round, n, k)) return 0;
    const bool i8 = x_fmt == DAXQ_FMT_I8, f8 = !i8;
    // What it costs to quantise in every workgroup grows with rows x K, what it saves does not: more of it is taken where a launch
    // has a workgroup for most CUs (N from 4096) and all of them run at once (to 8192; fp8, whose rings are smaller, two to a CU).
    // Below 4096 columns the other kernels cut a long K of int8 over more wavefronts than this one.  us per call on the GPU, weights
    // out of reach of the caches, separate launches / one, INT8; e4m3; e5m2 under a per-tensor scale (two launches or this):
    //   5 x 1536, K = 3072 6.1 / 5.8; 7.0 / 6.1; 8.0 / 6.6      4 x 5120, K = 8960 14.8 / 13.8; 14.9 / 14.0; 16.0 / 13.9   8 x 15360, K = 2048 10.8 / 12.1; 10.8 / 8.7; 11.8 / 9.4
    //   3 x 1536, K = 5120 7.7 / 8.1; 8.4 / 8.2; 9.4 / 8.1      8 x 4096 x 4096 8.8 / 8.4; 8.8 / 8.8; 10.2 / 9.3           3 x 13824, K = 5120 19.0 / 19.4; 19.1 / 16.0; 20.0 / 15.9
    //   2 x 1536, K = 8192 8.8 / 9.3; 10.5 / 9.5; 11.5 / 9.6    8 x 5120 x 5120 11.1 / 10.4; 11.3 / 10.2; 12.4 / 10.9      2 x 13824, K = 8192 27.1 / 25.2; 27.1 / 25.9; 28.0 / 26.2
    //   1 x 1536, K = 13824 11.7 / 13.3; 14.7 / 13.1; 15.1 / 13.2  3 x 8192, K = 5120 12.2 / 11.7; 12.4 / 11.8; 12.3 / 11.8  8 x 13824, K = 5120 19.5 / 21.8; 19.5 / 22.2; 20.7 / 22.9
    //   8 x 1536, K = 5120 8.2 / 9.2; 8.6 / 9.1; 9.9 / 9.6      8 x 8192, K = 4608 12.4 / 11.9; 12.1 / 11.6; 13.3 / 11.9
    // (forwards back to back besides save what the host takes for a launch: 5 x 1536, K = 3072 9.1 -> 6.0, 8 x 5120 x 5120 11.0 -> 10.1.)
    // One row of int8 against fewer than 4096 columns loses to the K ranges from some K on, later where the launches that it saves
    // are dearer (fp32 and fp16 rows, the abs-max of a tensor) or the other kernel gets slower (N from 3328).  us, separate / one, GPU
    // alone; back to back:
    //   1 x 512, K = 6144 7.5 / 7.9; 8.2 / 8.0     1 x 1536, K = 6144 7.7 / 8.1; 8.3 / 8.2     1 x 3328, K = 8192 9.7 / 9.9; 9.8 / 9.7
    //            K = 7168 7.9 / 8.4; 8.2 / 8.3              K = 8192 8.7 / 9.2; 8.9 / 9.1               K = 8960 10.4 / 10.9; 10.4 / 10.7
    //            K = 8960 8.8 / 9.7; 8.6 / 9.7              K = 10240 9.9 / 11.5; 10.0 / 11.4           K = 10240 11.3 / 12.6; 11.2 / 12.3
    //   fp16 1 x 768, K = 8192 8.5 / 9.0; 9.2 / 8.9           K = 8960 9.1 / 9.9; 9.9 / 9.8             K = 10240 9.7 / 11.2; 10.6 / 11.1
    //   fp32 1 x 768, K = 8960 9.7 / 9.8; 10.3 / 9.7          K = 10240 10.4 / 11.1; 11.0 / 11.0
    //   one scale for the tensor, 1 x 768, K = 8960 9.7 / 9.8; 9.7 / 9.7     K = 10240 10.4 / 11.2; 10.3 / 11.1
    // (Weights that the caches hold: one launch is 1 to 30 % faster at all of these; a model's are not there.)
    const int64_t kp = (k + DAXQ_K_ALIGN - 1) / DAXQ_K_ALIGN * DAXQ_K_ALIGN, bytes = few_dealt(m) * kp;
    if (i8 && n < 4096 && kp > (scheme == kFewTensor || x_dtype == DAXQ_F32 ? 8960 : x_dtype == DAXQ_F16 || n >= 3328 ? 8192 : 6144)) return 0;
    // More workgroups than CUs (N from 8193): int8 wants two to a CU, which its LDS holds up to K = 8064 with two rows; one to a CU has a
    // second round, which only pays beyond 12288 columns.  One fp8 row loses a little between 8256 and 11264.  us, separate / one, GPU
    // alone, weights far; near:
    //   int8 2 x 8960, K = 7168 17.9 / 17.1   K = 8064 19.1 / 19.0   K = 8192 20.6 / 22.4   K = 8960 21.1 / 24.5; 20.5 / 20.8
    //        2 x 12288, K = 8960 24.3 / 26.4   2 x 13824, K = 8192 28.3 / 25.4, K = 10240 31.8 / 31.2   1 x 8576, K = 15360 33.4 / 33.5, K = 16384 38.5 / 43.2
    //   e4m3 1 x 8200, K = 8192 (ratio) 0.92   1 x 8960, K = 6912 1.00, K = 8192 1.05; 1.06, K = 13824 1.05; 1.04   1 x 11264 1.00   2 x 8960, K = 8960 1.04; 0.93
    if (i8 && n > 8192 && n <= 12288 && few_dealt(m) * (kp + 16) + (kFewWaves + few_dealt(m)) * 4 > 81920 - kFewRingI8) return 0;
    if (f8 && m == 1 && n > 8256 && n < 11264 && kp > 7168) return 0;
    if (bytes <= 12288) return 1;
    if (n < 4096) return bytes <= (m > 2 ? 24576 : kFewMaxBytes) && (f8 || kp <= 4096);
    if (n <= 8192) return bytes <= (m > 2 ? kFewWideBytes : kFewMaxBytes);
    return bytes <= kFewMaxBytes && (f8 || m <= 2);
}

int daxq_linear_few(int x_dtype, int x_fmt, int w_fmt, int out_dtype, int scheme, int act_scale_round, const void* x, int64_t ld_x,
                    const float* in_scale, const void* wq, int64_t ld_wq, const float* sw, const void* bias, void* out, int64_t ld_out,
                    int64_t m, int64_t n, int64_t k, daxq_stream_t stream) {
    using namespace daxq;
    if (m == 0 || n == 0) return DAXQ_OK;
    if (!daxq_linear_few_applies(x_dtype, x_fmt, w_fmt, out_dtype, scheme, act_scale_round, m, n, k))
        return fail(DAXQ_ERR_ARG, "linear_few: does not take m=%lld n=%lld k=%lld in these formats", (long long)m, (long long)n, (long long)k);
    return few_linear("linear_few", x_dtype, x_fmt, w_fmt, out_dtype, scheme, act_scale_round, x, ld_x, in_scale, wq, ld_wq, sw, bias, out, ld_out, m, n, k, stream);
}

int daxq_linear_short_rows_applies(int x_dtype, int x_fmt, int w_fmt, int out_dtype, int scheme, int act_scale_round, int64_t m, int64_t n, int64_t k) {
    using namespace daxq;
    if (m < 9 || m > 64 || !few_forms(x_dtype, x_fmt, w_fmt, out_dtype, scheme, act_scale_round, n, k)) return 0;
    const int64_t kp = (k + DAXQ_K_ALIGN - 1) / DAXQ_K_ALIGN * DAXQ_K_ALIGN;
    return kp <= few_rows_most_k(x_dtype, x_fmt != DAXQ_FMT_I8, scheme == kFewTensor, m, n);
}

int daxq_linear_short_rows(int x_dtype, int x_fmt, int w_fmt, int out_dtype, int scheme, int act_scale_round, const void* x, int64_t ld_x,
                           const float* in_scale, const void* wq, int64_t ld_wq, const float* sw, const void* bias, void* out, int64_t ld_out,
                           int64_t m, int64_t n, int64_t k, daxq_stream_t stream) {
    using namespace daxq;
    if (m == 0 || n == 0) return DAXQ_OK;
    if (!daxq_linear_short_rows_applies(x_dtype, x_fmt, w_fmt, out_dtype, scheme, act_scale_round, m, n, k))
        return fail(DAXQ_ERR_ARG, "linear_short_rows: does not take m=%lld n=%lld k=%lld in these formats", (long long)m, (long long)n, (long long)k);
    return few_linear("linear_short_rows", x_dtype, x_fmt, w_fmt, out_dtype, scheme, act_scale_round, x, ld_x, in_scale, wq, ld_wq, sw, bias, out, ld_out, m, n, k, stream);
}

}  // extern "C"
