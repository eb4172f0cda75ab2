// The whole forward of a W8A8 linear of at most eight rows in one launch: every workgroup quantises the activation for itself, in
// LDS, while its share of the weight arrives, and multiplies (gfx950).
//
// What bounds it: the launches.  The quantiser and the GEMM of such a call take 2 and 3 to 7 us, their launches cost the host 2.8 to
// 3.6 us each (a per-tensor scale is a third one), and the second one starts when the first has ended and drained.  The quantised rows
// are few (m x K <= 40 KB), so that quantising them once per workgroup costs about what waiting for the weight does anyway.
// Forwards back to back, us, separate launches -> this: 1 x 1536 x 1536 8.2 -> 5.5, 4 x 1536 x 1536 e5m2 under a per-tensor scale
// 10.9 -> 5.7, 1 x 5120 x 5120 e4m3 8.2 -> 7.9 (its kernel).
//
// Work decomposition
//   workgroup  8 wavefronts, two groups (CG) of 16 output columns
//   quantiser  the wavefronts are dealt to the rows; all of the activation is in flight at once, maxima meet in LDS once, and the
//              bytes go to LDS rows of K + 16 bytes (the rows a fragment read touches then lie in different banks)
//   GEMM       as gemm_rows.hip: wavefront w < CG x KS streams K / KS bytes of 16 weight rows through an LDS ring of its own, the
//              first R steps of 128 bytes requested behind the activation's loads and in front of the quantiser's arithmetic.  INT8 cuts
//              K over KS = 4 wavefronts (sums of integers); FP8 runs KS = 1, so that an output element is the sequence of MFMAs over
//              the same K bytes in the same register positions that every other kernel runs.
// Same statistics, scales, bytes and epilogue as quant_rows.hip and gemm_rows.hip, whose helpers it calls: the outputs are their bits.
#include "gemm_rows.h"
#include "quant_rows.h"

namespace daxq {

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
// chunks of 8 elements per lane: 8 / rows wavefronts share a row of what those bytes leave it
constexpr int few_chunks(int rows, bool wide) {
    return ((rows == 1 ? kFewMaxK : wide ? kFewWideBytes : kFewMaxBytes) + kFewWaves * 512 - 1) / (kFewWaves * 512);
}

// MR: rows the wavefronts are dealt to (1, 2, 4, 8).  ONE: one scale for the tensor (dynamic or the caller's) instead of one per row
template <bool FP8, int F8, int XT, bool ONE, int MR, bool WIDE, int CG, int KS, int R>
__global__ __launch_bounds__(64 * kFewWaves) void gemm_few_kernel(const FewArgs a) {
    typedef typename Acc16<FP8>::type acc_t;
    constexpr int XB = XT == DAXQ_F32 ? 4 : 2, OUTK = XT, FMT = !FP8 ? 0 : (F8 & kF8XE5) ? 2 : 1;
    constexpr float kMax = FMT == 0 ? 127.0f : FMT == 1 ? 448.0f : 57344.0f;
    constexpr int NCH = few_chunks(MR, WIDE), WPR = kFewWaves / MR;  // wavefronts per row
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

    // ---- the activation: WPR wavefronts a row, all of it requested at once (beyond the row or the rows: the last chunk or row again)
    const int row = wave / WPR, rpart = wave % WPR, nch = a.kx >> 3;
    Chunk<XT> v[NCH];
    const char* xrow = a.x + (int64_t)(row < p.m ? row : p.m - 1) * a.ld_x * XB;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        if (i * WPR * 64 < nch) {
            const int c = (i * WPR + rpart) * 64 + lane;
            load_chunk_shared<XT>(v[i], xrow + (uint32_t)(c < nch ? c : nch - 1) * (8u * XB));
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
    float s = scale1;
    if (!ONE || a.scheme != kFewStatic) {
        uint32_t amax = 0;
#pragma unroll
        for (int i = 0; i < NCH; ++i)
            if (i * WPR * 64 < nch) amax = chunk_amax<XT>(amax, v[i]);
        amax = wave_max_u32(amax_of_lane<XT>(amax));
        if (ONE || WPR > 1) {  // meets the maxima of the row's other wavefronts, or (rows beyond m repeat the last one) of all
            if (lane == 0) s_max[wave] = amax;
            sync();
#pragma unroll
            for (int w = 0; w < (ONE ? kFewWaves : WPR); ++w) {
                const uint32_t o = s_max[ONE ? w : row * WPR + w];
                amax = o > amax ? o : amax;
            }
        }
        s = scale_from_amax_bits_rt<XT>(amax, kMax, kEps, a.round_x);
    }
    if (rpart == 0 && lane == 0) s_sx[row] = s;
    // ---- bytes: a row under its own scale takes one form (a bf16 row kOwn; fp16 and fp32 rows, int8 only, kDivide), the one scale of a
    //      tensor picks one
    const float inv = 1.0f / s;  // IEEE division, not v_rcp_f32
    auto store = [&](auto FORM) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            if (i * WPR * 512 >= p.k) continue;
            const int c = (i * WPR + rpart) * 64 + lane;
            uint2 o = make_uint2(0, 0);
            if (i * WPR * 64 < nch) {
                float f[8];
                chunk_values<XT>(v[i], f);
                o = quant8<FMT, decltype(FORM)::value, XT>(f, s, inv);
            }
            if (c * 8 < p.k) *reinterpret_cast<uint2*>(s_x + row * xs + c * 8) = c < nch ? o : make_uint2(0, 0);
        }
    };
    if constexpr (ONE) with_form<FMT, XT>(s, kMax, a.scheme == kFewStatic, a.round_x, a.scheme == kFewTensor, store);
    else store(std::integral_constant<int, XT == DAXQ_BF16 ? kOwn : kDivide>{});
    sync();

    // ---- the GEMM
    const int xo = (g4 ^ (l15 & 7)) << 4;
    const uint8_t *rd = smem + wave * (R * STEP) + l15 * 128 + xo, *rd_up = rd + (64 - 2 * (xo & 64));
    const uint8_t* xr = s_x + (l15 < MR ? l15 : MR - 1) * xs + (int64_t)first * 128 + g4 * 16;
    acc_t acc = {};
    auto next_slot = [](uint32_t slot) { return slot == (R - 1) * STEP ? 0 : slot + STEP; };
    auto work = [&](auto STEPS, auto MORE, int step, uint32_t slot) __attribute__((always_inline)) {
        constexpr int U = decltype(STEPS)::value;
        v8i w[U], x[U];
        uint32_t at[U];
        at[0] = slot;
#pragma unroll
        for (int u = 1; u < U; ++u) at[u] = next_slot(at[u - 1]);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const v4i lo = *reinterpret_cast<const v4i*>(rd + at[u]), up = *reinterpret_cast<const v4i*>(rd_up + at[u]);
            w[u] = __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
            const v4i xl = *reinterpret_cast<const v4i*>(xr + (step + u) * 128), xu = *reinterpret_cast<const v4i*>(xr + (step + u) * 128 + 64);
            x[u] = __builtin_shufflevector(xl, xu, 0, 1, 2, 3, 4, 5, 6, 7);
        }
        if constexpr (MORE.value) {
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(63) & lgkmcnt0_mask());  // the reads are over
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; ++u) load(step + u + R, at[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) acc = mfma_step<FP8, F8>(w[u], x[u], acc);
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

    if constexpr (KS > 1) {
        v4i* s_part = reinterpret_cast<v4i*>(smem);  // [wave][lane], in the rings, which everyone has left
        sync();
        s_part[wave * 64 + lane] = __builtin_bit_cast(v4i, acc);
        sync();
        if (part != 0) return;
        v4i sum = s_part[wave * 64 + lane];
#pragma unroll
        for (int i = 1; i < KS; ++i) sum += s_part[(wave + i) * 64 + lane];
        acc = __builtin_bit_cast(acc_t, sum);
    }
    if (!works || l15 >= p.m || nc >= p.n) return;
    store_columns<FP8, OUTK>(p, acc, s_sx[l15], cols, l15, nc);
}

// args null: only raises the kernel's LDS limit on the current device
template <bool FP8, int F8, int XT, bool ONE, int MR, bool WIDE = false>
static int launch_few_one(const FewArgs* a, hipStream_t st) {
    constexpr int CG = 2, KS = FP8 ? 1 : 4, R = FP8 ? 10 : 4;  // (rings of 15 and 20 steps: 0 to 3 % slower, a CU then has room for fewer workgroups)
    auto kern = gemm_few_kernel<FP8, F8, XT, ONE, MR, WIDE, CG, KS, R>;
    static std::atomic<uint64_t> lds_set{0};  // per instantiation
    constexpr int ring = CG * KS * R * 2048, most = ring + (WIDE ? kFewWideBytes : kFewMaxBytes) + MR * 16 + (kFewWaves + MR) * 4;
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), most, lds_set)) return rc;
    if (!a) return DAXQ_OK;
    const int lds = ring + MR * (a->g.k + 16) + (kFewWaves + MR) * 4;
    launch_kernel(kern, dim3((unsigned)((a->g.n + 16 * CG - 1) / (16 * CG))), dim3(64 * kFewWaves), lds, st, *a);
    return check_launch("gemm_few");
}

template <bool FP8, int F8, int XT, bool ONE>
static int launch_few_rows(const FewArgs* a, int m, bool wide, hipStream_t st) {
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
    for (int m : {1, 2, 4, 8})
        for (bool wide : {false, true}) {
            if (wide && m < 4) continue;
            for (int x : {DAXQ_BF16, DAXQ_F16, DAXQ_F32}) prepare(m, wide, DAXQ_FMT_I8, x);
            for (int f : {DAXQ_FMT_E4M3, DAXQ_FMT_E5M2}) prepare(m, wide, f, DAXQ_BF16);
        }
    return rc;
}

// rows as the wavefronts are dealt to them
static inline int64_t few_dealt(int64_t m) { return m <= 2 ? m : m <= 4 ? 4 : 8; }

}  // namespace daxq

extern "C" {

int daxq_linear_few_applies(int x_dtype, int x_fmt, int w_fmt, int out_dtype, int scheme, int act_scale_round, int64_t m, int64_t n, int64_t k) {
    using namespace daxq;
    if (scheme < kFewToken || scheme > kFewStatic) return 0;
    // (an fp8 row under a scale that is not rounded to bf16 takes another form per row: left to the quantiser)
    if (x_fmt != DAXQ_FMT_I8 && scheme == kFewToken && act_scale_round != DAXQ_SCALE_ROUND_X) return 0;
    const bool i8 = x_fmt == DAXQ_FMT_I8 && w_fmt == DAXQ_FMT_I8;
    const bool f8 = (x_fmt == DAXQ_FMT_E4M3 || x_fmt == DAXQ_FMT_E5M2) && w_fmt == DAXQ_FMT_E4M3 && x_dtype == DAXQ_BF16;
    if ((!i8 && !f8) || x_dtype != out_dtype || x_dtype < DAXQ_BF16 || x_dtype > DAXQ_F32) return 0;
    if (m < 1 || m > 8 || k < 8 || k % 8 || k > kFewMaxK || n < (f8 ? 128 : 1) || n > (1 << 20)) return 0;
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
    const int64_t kp = (k + DAXQ_K_ALIGN - 1) / DAXQ_K_ALIGN * DAXQ_K_ALIGN, bytes = few_dealt(m) * kp;
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
    const int64_t kp = (k + DAXQ_K_ALIGN - 1) / DAXQ_K_ALIGN * DAXQ_K_ALIGN;
    if ((scheme == kFewStatic) != (in_scale != nullptr)) return fail(DAXQ_ERR_ARG, "linear_few: scheme %d takes in_scale: %d", scheme, scheme == kFewStatic);
    if (act_scale_round != DAXQ_SCALE_ROUND_X && act_scale_round != DAXQ_SCALE_ROUND_NONE)
        return fail(DAXQ_ERR_ARG, "linear_few: unknown scale rounding %d", act_scale_round);
    if (!x || !wq || !sw || !out) return fail(DAXQ_ERR_ARG, "linear_few: null pointer");
    if (ld_x < k || ld_wq < kp || ld_out < n || ld_wq >= (1 << 26)) return fail(DAXQ_ERR_ARG, "linear_few: bad leading dimension");
    const uintptr_t xa = x_dtype == DAXQ_F32 ? 3 : 1;
    if (((uintptr_t)x & xa) || ((uintptr_t)out & xa) || ((uintptr_t)bias & xa) || ((uintptr_t)sw & 3) || ((uintptr_t)in_scale & 3) ||
        ((uintptr_t)wq & 15) || (ld_wq & 15))
        return fail(DAXQ_ERR_ALIGN, "linear_few: misaligned pointer or weight rows");
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
    const bool wide = m > 2 && few_dealt(m) * kp > kFewMaxBytes;
    if (scheme == kFewToken) return launch_few<false>(&a, (int)m, wide, x_fmt, x_dtype, (hipStream_t)stream);
    return launch_few<true>(&a, (int)m, wide, x_fmt, x_dtype, (hipStream_t)stream);
}

}  // extern "C"
