// Row-wise symmetric quantisation of a bf16 / fp16 / fp32 matrix to int8, OCP e4m3fn or OCP e5m2.
//
// One launch covers both uses on the path:
//   * dynamic per-token activation quantisation (scale rounded to bf16 first, as
//     the eager dtype chain of dax/quant/nn/dynamic/functional.py:124-129 does), and
//   * one-time per-output-channel weight quantisation (scale kept in fp32,
//     dax/quant/quantization/observer.py:97-134).
// The element rule is the leaf quantiser of dax/quant/nn/quantized/functional.py:11-20:
//   int8:  clamp(rint(f32(x) * (1.0f / s)), -128, 127)      reciprocal-multiply
//   e4m3:  e4m3fn_rne(clamp(f32(x) / s, -448, 448))         true division
//   e5m2:  e5m2_rne(clamp(f32(x) / s, -57344, 57344))       true division (activations only)
//
// HBM-bound: 2 B read + 1 B written per element.  The row stays in VGPRs between the abs-max pass and the quantise pass,
// so memory is read once.
#include <type_traits>

#include "quant_rows.h"

namespace daxq {

struct QuantArgs {
    const char* x;
    int64_t m, ld_x;  // ld_x in elements
    int k, kfill;     // columns [k, kfill) of q are written as zeros
    uint8_t* q;
    int64_t ld_q;
    float* scale;             // [m]: the scale of every row, written; null = not wanted
    const float* scale_in;    // SCALE_IN: the caller's scale, of row r at [r * scale_stride]
    int scale_stride;         // 1, or 0: one scale for the tensor
    const uint32_t* partials; // dynamic scale of the whole tensor: kPartials abs-max patterns, their maximum is the tensor's; null = per row
    float* scale1;            // ... and where that one scale goes besides (or null)
    float qmax, eps;          // dynamic scale: divisor and floor,
    int round_x;              // and whether both are rounded to the element type
    int leaf;                 // the scale is a tensor's or a weight's: the leaf quantiser's bytes also where it is not finite
};
constexpr int kPartials = 256;  // workgroups of tensor_amax_kernel, one per CU
constexpr int kTensorQuantPieces = 128;  // pieces of 64 chunks that tensor_quant_kernel has in flight: 8 in each of 16 wavefronts

// Workgroup b of n as its XCD's (b mod 8) next one of a contiguous range
__device__ __forceinline__ uint32_t xcd_range(uint32_t b, uint32_t n) {
    const uint32_t x = b & 7, q = n >> 3, r = n & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// W wavefronts share a row (4 / W rows per workgroup), lane l of wavefront w holding chunks (i W + w) 64 + l.  One
// wavefront per row for short rows, four for long ones: the chunks of a row then arrive in a quarter of the instructions,
// which is what a launch of few rows waits for (512 x 5120: 4.1 -> 3.0 us, 17 x 5120 3.5 -> 2.4 us; a wavefront alone on
// its SIMD issues one instruction in eight cycles), and a launch of many keeps more, smaller pieces of work in flight
// (9450 x 5120: 25.9 -> 23.9 us = 6.1 TB/s, 75600 x 5120 186.2 -> 180.3 us = 6.4 TB/s, x 13824 543.8 -> 529.3 us); at
// K = 1536 the barrier costs more than it returns (6.06 against 4.78 TB/s).  fp32 rows, and rows of any length or
// address, against one workgroup per row that read them twice, element by element: 4096 x 5120 fp32 43.9 -> 19.7 us,
// 2900 x 1001 bf16 6.1 -> 3.7 us.
// SCALE_IN: the per-row scale is an input (leaf quantiser) instead of being derived from the row.
// PLAIN: bf16 rows of whole chunks under their own scales, bytes as kOwn: what the DiT's linears launch.  The loads and the
// stores then sit in one straight piece of code; with the other forms' branches between them a wavefront issues later, which
// short rows feel most.  us, all forms in one / PLAIN, INT8 (e4m3): 32760 x 1536 26.0 / 24.3 (26.2 / 24.5), 4096 x 2048 6.2 / 6.0
// (6.3 / 6.2), 9450 x 5120 24.2 / 23.4 (24.4 / 23.8), 516 x 5120 3.4 / 3.2 (3.6 / 3.4); none of eighteen slower.
// STORE: where the bytes go (store_of)
// Rows of one wavefront whose bytes stay in the caches are dealt out in ranges, an eighth of the matrix to each XCD, as the tiled GEMMs'
// row groups take them: what the consumer's own L2 holds it need not fetch, and no L2 has to give up lines that the next pass rewrites.
// Quantiser + GEMM, us, rows dealt round the XCDs / in ranges, INT8: 11732 x 304, K = 1536 23.0 / 20.4, 4096 x 1536 x 1536 20.0 / 19.2,
// 4412 x 1056, K = 920 14.6 / 13.9, 33629 x 504, K = 552 33.1 / 32.2, 32760 x 2728, K = 1536 152.5 / 150.7.  Longer rows are level (0.2 %).
template <int NCH, int W, int FMT, bool SCALE_IN, int XT, bool PLAIN, int STORE>
__global__ __launch_bounds__(256) void quant_rows_kernel(const QuantArgs a) {
    constexpr int XB = XT == DAXQ_F32 ? 4 : 2;
    __shared__ uint32_t s_max[4];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // behind tensor_amax_kernel: the rows that it read last first, each on the XCD that read it
    const int64_t unit = W > 1 && !PLAIN && !SCALE_IN && a.partials ? (int64_t)((gridDim.x >> 3) - 1 - (blockIdx.x >> 3)) * 8 + (blockIdx.x & 7)
                         : W == 1 && STORE != kStorePast ? xcd_range(blockIdx.x, gridDim.x) : blockIdx.x;
    const int64_t row0 = unit * (4 / W) + wave / W;
    if (W == 1 && row0 >= a.m) return;
    const int64_t row = row0 < a.m ? row0 : a.m - 1;  // (rows beyond the last: the wavefront still reaches the barrier)
    const int part = wave % W, nch = a.k >> 3, npad = a.kfill >> 3;
    const char* xr = a.x + row * a.ld_x * XB;
    // what whole chunks do not cover -- the columns behind the last of them, and a width or fill that is no multiple of
    // 8 -- is one element per lane of the row's first wavefront
    const bool ragged = !PLAIN && ((a.k | a.kfill) & 7) != 0;

    Chunk<XT> v[NCH];
    if (PLAIN || nch > 0) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = (i * W + part) * 64 + lane;
            // (beyond the row: its last chunk once more, which leaves the maximum as it is and is not stored)
            load_chunk<XT>(v[i], xr + (uint32_t)(c < nch ? c : nch - 1) * (8u * XB));
        }
    } else {
#pragma unroll
        for (int i = 0; i < NCH; ++i) v[i] = Chunk<XT>{};
    }
    uint32_t tail = 0;
    if (ragged && part == 0 && lane < (a.k & 7)) {
        if constexpr (XT == DAXQ_F32) tail = reinterpret_cast<const uint32_t*>(xr)[nch * 8 + lane];
        else tail = reinterpret_cast<const uint16_t*>(xr)[nch * 8 + lane];
    }
    float s;
    if constexpr (SCALE_IN) {
        s = a.scale_in[row * a.scale_stride];
        if (a.scale && part == 0 && lane == 0) a.scale[row] = s;
    } else {
        uint32_t mx = 0;
        if (!PLAIN && a.partials) {  // every wavefront finds the tensor's maximum in 1 KB of L2 while its row arrives
            const uint4 p = reinterpret_cast<const uint4*>(a.partials)[lane];
            const uint32_t lo = p.x > p.y ? p.x : p.y, hi = p.z > p.w ? p.z : p.w;
            mx = lo > hi ? lo : hi;
        } else {
#pragma unroll
            for (int i = 0; i < NCH; ++i) mx = chunk_amax<XT>(mx, v[i]);
            mx = amax_of_lane<XT>(mx);
            const uint32_t t = tail & (XT == DAXQ_F32 ? 0x7fffffffu : 0x7fffu);
            mx = t > mx ? t : mx;
        }
        uint32_t amax = wave_max_u32(mx);
        if (W > 1 && (PLAIN || !a.partials)) {
            if (lane == 0) s_max[wave] = amax;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < W; ++i) {
                const uint32_t o = s_max[wave / W * W + i];
                amax = o > amax ? o : amax;
            }
        }
        s = scale_from_amax_bits_rt<XT>(amax, a.qmax, a.eps, a.round_x);
        if (part == 0 && lane == 0) {
            a.scale[row] = s;
            if (!PLAIN && a.scale1 && row == 0) a.scale1[0] = s;
        }
    }
    if (W > 1 && row0 >= a.m) return;
    const float inv = 1.0f / s;  // IEEE division, not v_rcp_f32

    uint8_t* qr = a.q + row * a.ld_q;
    auto store = [&](auto FORM) __attribute__((always_inline)) {
        constexpr int F = decltype(FORM)::value;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = (i * W + part) * 64 + lane;
            float f[8];
            chunk_values<XT>(v[i], f);
            const uint2 o = quant8<FMT, F, XT>(f, s, inv);
            if (c < nch) store_chunk<STORE>(qr + (uint32_t)c * 8u, o);
            else if (!ragged && c < npad) store_chunk<STORE>(qr + (uint32_t)c * 8u, make_uint2(0, 0));
        }
    };
    if constexpr (PLAIN) store(std::integral_constant<int, kOwn>{});
    else with_form<FMT, XT>(s, a.qmax, SCALE_IN, a.round_x, a.leaf, store);
    if (ragged && part == 0) {
        const float f = x_bits_to_f32<XT>(tail);
        uint8_t o;
        if constexpr (FMT == 0) o = (uint8_t)q_i8_bits(f, inv);
        else o = (uint8_t)cvt_pk_f8<FMT>(q_f8_pre<FMT, true>(f, s, inv), 0.0f, 0, false);
        for (int c = nch * 8 + lane; c < a.kfill; c += 64) qr[c] = c < a.k ? o : 0;
    }
}

// Rows too long for the registers of four wavefronts: one 256-thread workgroup per row, two passes over memory.
template <int XT>
struct XWord {
    typedef uint16_t type;
};
template <>
struct XWord<DAXQ_F32> {
    typedef uint32_t type;
};

template <int FMT, bool SCALE_IN, int XT = DAXQ_BF16>
__global__ __launch_bounds__(256) void quant_rows_block(const void* __restrict__ xv, int64_t m, int64_t k,
                                                        int64_t ld_x, uint8_t* __restrict__ q, int64_t ld_q, int64_t kfill,
                                                        float* __restrict__ scale, float qmax, float eps, int round_x) {
    typedef typename XWord<XT>::type word_t;
    constexpr uint32_t kAbs = XT == DAXQ_F32 ? 0x7fffffffu : 0x7fffu;
    __shared__ uint32_t red[4];
    const int64_t row = blockIdx.x;
    const word_t* xr = static_cast<const word_t*>(xv) + row * ld_x;
    float s;
    if constexpr (SCALE_IN) {
        s = scale[row];
    } else {
        uint32_t mx = 0;
        for (int64_t c = threadIdx.x; c < k; c += 256) {
            uint32_t a = xr[c] & kAbs;
            mx = a > mx ? a : mx;
        }
        mx = wave_max_u32(mx);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
        __syncthreads();
        uint32_t amax = red[0];
        amax = red[1] > amax ? red[1] : amax;
        amax = red[2] > amax ? red[2] : amax;
        amax = red[3] > amax ? red[3] : amax;
        s = scale_from_amax_bits_rt<XT>(amax, qmax, eps, round_x);
        if (threadIdx.x == 0) scale[row] = s;
    }
    const float inv = 1.0f / s;
    uint8_t* qr = q + row * ld_q;
    for (int64_t c = threadIdx.x; c < kfill; c += 256) {
        uint8_t o = 0;
        if (c < k) {
            float f = x_bits_to_f32<XT>(xr[c]);
            if (FMT != 0) {
                // the reciprocal sequence is verified exhaustively for bf16 elements only; other types divide
                const float pre = (SCALE_IN || XT != DAXQ_BF16 || round_x) ? q_f8_pre<FMT, SCALE_IN || XT != DAXQ_BF16>(f, s, inv)
                                                                           : q_f8_pre<FMT, true>(f, s, inv);
                o = (uint8_t)(cvt_pk_f8<FMT>(pre, 0.0f, 0, false) & 0xff);
            } else {
                o = (uint8_t)(q_i8_bits(f, inv) & 0xffu);
            }
        }
        qr[c] = o;
    }
}

// Anything but a dynamic scale per token or the caller's per row (QuantArgs)
struct ScaleKind {
    bool one_scale = false;              // the caller's scale is one value; scale_rows: where it goes once per row (or null)
    float* scale_rows = nullptr;
    const uint32_t* partials = nullptr;  // the scale comes from the tensor's abs-max; scale1: where it goes besides (or null)
    float* scale1 = nullptr;
    bool weight = false;                 // rows of a weight: the leaf quantiser's bytes also under a scale that is not finite
};

// Rows that a workgroup of quant_rows_kernel takes where a row has more than one wavefront (the instantiations that
// launch_quant_rows_t goes through), else 0.
static int quant_unit(int x_dtype, int64_t kfill) {
    const int64_t cols = (kfill + 511) / 512;
    if (x_dtype == DAXQ_F32) return cols <= 2 ? 0 : 1;
    return cols <= 4 ? 0 : cols <= 6 ? 2 : 1;
}

// at most `count` rows of `a` from row r on
template <int XB>
static QuantArgs rows_from(const QuantArgs& a, int64_t r, int64_t count) {
    QuantArgs b = a;
    if (b.m - r < count) count = b.m - r;
    b.m = count;
    b.x += r * a.ld_x * XB;
    b.q += r * a.ld_q;
    if (b.scale) b.scale += r;
    b.scale_in += r * a.scale_stride;
    if (r) b.scale1 = nullptr;
    return b;
}

template <int FMT, bool SCALE_IN, int XT>
static int launch_quant_rows_t(const void* x, int64_t m, int64_t k, int64_t ld_x, void* q, int64_t ld_q, float* scale,
                               float qmax, hipStream_t st, float eps, int round_x, const ScaleKind& t) {
    constexpr int XB = XT == DAXQ_F32 ? 4 : 2;
    if (m < 0 || k <= 0 || ld_x < k || ld_q < k) return fail(DAXQ_ERR_ARG, "quant_rows: bad shape m=%lld k=%lld ld_x=%lld ld_q=%lld",
                                                               (long long)m, (long long)k, (long long)ld_x, (long long)ld_q);
    if (m == 0) return DAXQ_OK;
    if (!x || !q || !scale) return fail(DAXQ_ERR_ARG, "quant_rows: null pointer");
    const int64_t kfill = fill_width(k, ld_q);
    if (((uintptr_t)x & (XB - 1)) != 0 || ((uintptr_t)scale & 3) != 0) return fail(DAXQ_ERR_ALIGN, "quant_rows: x must be element aligned and scale 4-byte aligned");
    uint8_t* qp = static_cast<uint8_t*>(q);
    if (kfill <= DAXQ_MAX_TENSOR_K) {
        const QuantArgs a{static_cast<const char*>(x), m, ld_x, (int)k, (int)kfill, qp, ld_q, SCALE_IN ? t.scale_rows : scale, scale,
                    t.one_scale ? 0 : 1, t.partials, t.scale1, qmax, eps, round_x, t.partials || t.weight};
        const int cols = (int)((kfill + 511) / 512);
        constexpr bool kMayBePlain = !SCALE_IN && XT == DAXQ_BF16;
        constexpr float kFmtMax = FMT == 0 ? 127.0f : FMT == 1 ? 448.0f : 57344.0f;
        const bool plain = kMayBePlain && ((k | kfill) & 7) == 0 && !a.leaf && qmax <= kFmtMax && (FMT == 0 || round_x);
        // (the rows of a weight, and those under a scale each from the caller, have no GEMM behind them)
        const int to = t.weight || (SCALE_IN && !t.one_scale) ? kStorePast : store_of(m * kfill, (((uintptr_t)q | (uintptr_t)ld_q) & 7) == 0);
        // A launch holds fewer than 2^32 work items, i.e. 2^24 workgroups: more rows are as many launches as they need
#define DAXQ_Q_CASE(N, W)                                                                                                  \
    if (cols <= N * W) {                                                                                                   \
        constexpr int64_t kRows = 4 / W, kSlab = kRows << 23;                                                              \
        for (int64_t r = 0; r < m; r += kSlab) {                                                                           \
            const QuantArgs b = rows_from<XB>(a, r, kSlab);                                                                \
            const unsigned groups = (unsigned)((b.m + kRows - 1) / kRows);                                                 \
            const dim3 grid(W > 1 && a.partials ? (groups + 7) / 8 * 8 : groups);                                          \
            auto launch = [&](auto STORE) {                                                                                \
                constexpr int S = decltype(STORE)::value;                                                                  \
                if (plain) launch_kernel((quant_rows_kernel<N, W, FMT, SCALE_IN, XT, kMayBePlain, S>), grid, dim3(256), 0, st, b); \
                else launch_kernel((quant_rows_kernel<N, W, FMT, SCALE_IN, XT, false, S>), grid, dim3(256), 0, st, b);     \
            };                                                                                                             \
            if (to == kStoreThrough) launch(std::integral_constant<int, kStoreThrough>{});                                 \
            else if (to == kStoreKeep) launch(std::integral_constant<int, kStoreKeep>{});                                  \
            else launch(std::integral_constant<int, kStorePast>{});                                                        \
        }                                                                                                                  \
        return check_launch("quant_rows");                                                                                 \
    }
        DAXQ_Q_CASE(1, 1)
        DAXQ_Q_CASE(2, 1)
        if constexpr (XT != DAXQ_F32) {
            DAXQ_Q_CASE(3, 1)
            DAXQ_Q_CASE(4, 1)
            DAXQ_Q_CASE(3, 2)
        }
        DAXQ_Q_CASE(2, 4)
        DAXQ_Q_CASE(3, 4)
        if constexpr (XT == DAXQ_BF16) {
            DAXQ_Q_CASE(4, 4)
        }
        DAXQ_Q_CASE(5, 4)
        DAXQ_Q_CASE(7, 4)
        DAXQ_Q_CASE(9, 4)
#undef DAXQ_Q_CASE
    }
    if (t.one_scale || t.partials) return fail(DAXQ_ERR_ARG, "quant_rows: one scale for the tensor is taken for rows of at most %d columns", DAXQ_MAX_TENSOR_K);
    if (m > 0x7fffffff) return fail(DAXQ_ERR_ARG, "quant_rows: too many rows");
    launch_kernel((quant_rows_block<FMT, SCALE_IN, XT>), dim3((unsigned)m), dim3(256), 0, st, x, m, k, ld_x, qp,
                       ld_q, kfill, scale, qmax, eps, round_x);
    return check_launch("quant_rows_block");
}

// eps, round_x: floor and rounding of a dynamic scale (scale_from_amax_bits_rt); unused when the scale is an input
template <int FMT, bool SCALE_IN>
static int launch_quant_rows(const void* x, int64_t m, int64_t k, int64_t ld_x, void* q, int64_t ld_q, float* scale,
                             float qmax, hipStream_t st, int x_dtype = DAXQ_BF16, float eps = kEps, int round_x = 1, const ScaleKind& t = {}) {
    if (!SCALE_IN && (!(qmax > 0.0f) || !(eps >= 0.0f))) return fail(DAXQ_ERR_ARG, "quant_rows: quant_max must be positive and eps not negative");
    switch (x_dtype) {
        case DAXQ_BF16: return launch_quant_rows_t<FMT, SCALE_IN, DAXQ_BF16>(x, m, k, ld_x, q, ld_q, scale, qmax, st, eps, round_x, t);
        case DAXQ_F16: return launch_quant_rows_t<FMT, SCALE_IN, DAXQ_F16>(x, m, k, ld_x, q, ld_q, scale, qmax, st, eps, round_x, t);
        case DAXQ_F32: return launch_quant_rows_t<FMT, SCALE_IN, DAXQ_F32>(x, m, k, ld_x, q, ld_q, scale, qmax, st, eps, round_x, t);
        default: return fail(DAXQ_ERR_ARG, "quant_rows: unknown element type %d", x_dtype);
    }
}

// qmax <= 0: the format's own maximum
template <bool SCALE_IN>
static int launch_quant_rows_fmt(int q_fmt, const void* x, int x_dtype, int64_t m, int64_t k, int64_t ld_x, void* q,
                                 int64_t ld_q, float* scale, hipStream_t st, float qmax = 0.0f, float eps = kEps, int round_x = 1, const ScaleKind& t = {}) {
    switch (q_fmt) {
        case DAXQ_FMT_I8: return launch_quant_rows<0, SCALE_IN>(x, m, k, ld_x, q, ld_q, scale, qmax > 0.0f ? qmax : 127.0f, st, x_dtype, eps, round_x, t);
        case DAXQ_FMT_E4M3: return launch_quant_rows<1, SCALE_IN>(x, m, k, ld_x, q, ld_q, scale, qmax > 0.0f ? qmax : 448.0f, st, x_dtype, eps, round_x, t);
        case DAXQ_FMT_E5M2: return launch_quant_rows<2, SCALE_IN>(x, m, k, ld_x, q, ld_q, scale, qmax > 0.0f ? qmax : 57344.0f, st, x_dtype, eps, round_x, t);
        default: return fail(DAXQ_ERR_ARG, "quant_rows: unknown quantised format %d", q_fmt);
    }
}

// Abs-max of a whole matrix as kPartials bit patterns (sign cleared; their maximum is the abs-max, NaN above infinity):
// one workgroup of sixteen wavefronts per CU, U chunks per lane in flight (2 to 4 of 16 bytes are level, 6 and 8 slower by 1 to 10 %:
// the last turns of the loop are emptier).
// It is bound by memory, and what it reads the quantiser reads again right behind it.  With a row or two to a workgroup of the
// quantiser (unit > 0: the rows of one, K > 2048), workgroup i here takes the rows of the quantiser's workgroups i, i + 256, ...,
// which run on the same XCD, and the quantiser begins with the rows that were read last, out of that XCD's L2.  Both launches, us,
// matrix read as it lies -> this (bf16, e5m2): 4096 x 5120 21.3 -> 19.9, 4725 x 13824 55.2 -> 53.8, 12000 x 4608 46.2 -> 44.6, 1000 x 8960
// 12.2 -> 10.8, 300 x 5120 6.7 -> 6.5; shorter rows lose what they gain to the row arithmetic (16000 x 1536 23.7 -> 24.9).
// The loads carry no hint for data that is read once (load_chunk), which would evict what the quantiser reads next, bf16; fp32:
// 4096 x 5120 20.0 -> 17.2; 36.0 -> 28.6, 4725 x 13824 53.2 -> 48.8; 103.6 -> 86.7, 12000 x 4608 45.6 -> 41.8; 88.5 -> 72.0, 16000 x 1536
// 24.4 -> 22.5; 42.7 -> 35.5, 500 x 1536 6.3 -> 5.8; 6.3 -> 6.3, 4096 x 1536 9.7 -> 9.8; 14.7 -> 13.1, 12000 x 15360 143 -> 140; 283 -> 265.
struct AmaxArgs {
    const char* x;
    int64_t m, ld_x;
    int k;
    int unit;  // rows that a workgroup of the quantiser takes, or 0: the matrix is read as it lies
    uint32_t* partials;
};
template <int XT>
__global__ __launch_bounds__(1024) void tensor_amax_kernel(const AmaxArgs a) {
    constexpr int XB = XT == DAXQ_F32 ? 4 : 2, U = XT == DAXQ_F32 ? 2 : 3;
    constexpr uint32_t kAbs = XT == DAXQ_F32 ? 0x7fffffffu : 0x7fffu;
    __shared__ uint32_t s_max[16];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t mx = 0, tl = 0;
    auto element = [&](const char* xr, int64_t e) __attribute__((always_inline)) {
        const uint32_t t = (XT == DAXQ_F32 ? reinterpret_cast<const uint32_t*>(xr)[e] : reinterpret_cast<const uint16_t*>(xr)[e]) & kAbs;
        tl = t > tl ? t : tl;
    };
    if (a.unit) {
        // a wavefront takes every sixteenth piece (64 chunks of a row) of the workgroup's rows
        const int nch = a.k >> 3, pieces = (nch + 63) >> 6;
        const int64_t rows = a.m;
        int64_t row = (int64_t)blockIdx.x * a.unit;
        int in = 0, c = 0;  // row of the unit, piece of the row
        auto advance = [&](int by) __attribute__((always_inline)) {
            c += by;
            while (c >= pieces) {
                c -= pieces;
                if (++in == a.unit) in = 0, row += (int64_t)kPartials * a.unit;
            }
        };
        advance(wave);
        while (row < rows) {
            Chunk<XT> v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (row + in < rows) {
                    const char* xr = a.x + (row + in) * a.ld_x * XB;
                    const int at = c * 64 + lane;
                    load_chunk_shared<XT>(v[u], xr + (uint32_t)(at < nch ? at : nch - 1) * (8u * XB));
                    if (c == pieces - 1 && lane < (a.k & 7)) element(xr, nch * 8 + lane);
                } else {
                    v[u] = Chunk<XT>{};
                }
                advance(16);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) mx = chunk_amax<XT>(mx, v[u]);
        }
    } else {
        int64_t len = a.k, m = a.m;
        if (a.ld_x == a.k || m == 1) {  // one long row
            len *= m;
            m = 1;
        }
        const int64_t nch = len >> 3;
        // a long row is spread over the grid, rows of a strided matrix are dealt to the workgroups
        const int64_t first = m == 1 ? (int64_t)blockIdx.x * 1024 : 0, step = m == 1 ? (int64_t)kPartials * 1024 : 1024;
        for (int64_t r = m == 1 ? 0 : blockIdx.x; r < m; r += kPartials) {
            const char* xr = a.x + r * a.ld_x * XB;
            for (int64_t c = first + threadIdx.x; c < nch; c += U * step) {
                Chunk<XT> v[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int64_t cu = c + u * step;
                    load_chunk_shared<XT>(v[u], xr + (cu < nch ? cu : c) * (8 * XB));  // (beyond the end: the lane's first chunk again)
                }
#pragma unroll
                for (int u = 0; u < U; ++u) mx = chunk_amax<XT>(mx, v[u]);
            }
            const int64_t e = (nch << 3) + threadIdx.x;
            if (e < len) element(xr, e);
        }
    }
    mx = amax_of_lane<XT>(mx);
    mx = wave_max_u32(tl > mx ? tl : mx);
    if (lane == 0) s_max[wave] = mx;
    __syncthreads();
    if (threadIdx.x < 64) {
        mx = wave_max_u32(threadIdx.x < 16 ? s_max[threadIdx.x] : 0u);
        if (threadIdx.x == 0) a.partials[blockIdx.x] = mx;
    }
}

// Dynamic per-tensor quantisation of a small matrix in one launch: every workgroup finds the abs-max of the whole matrix for
// itself and quantises one row, which it requested first.
// What bounds it: latency.  The abs-max launch that it saves costs the host 2.2 us and the GPU a launch that the next one waits
// for; against that, sixteen wavefronts read the matrix out of their XCD's L2, 64 chunks of a row (a piece) per instruction, all
// of their U pieces in flight at once.  Forwards, us, GPU alone (back to back), two launches and GEMM -> this and GEMM:
//   9 x 1536 x 1536 8.3 -> 6.9 e5m2 (11.7 -> 8.5)    40 x 1536 x 1536 8.6 -> 7.8 int8 (12.0 -> 9.0)     64 x 256, N = 1536 7.6 -> 7.0 (12.3 -> 9.0)
//   12 x 5120 x 5120 10.8 -> 10.3 int8 (12.1 -> 10.4)  21 x 3072 x 3072 9.8 -> 8.8 int8 (12.6 -> 9.1)  40 x 1536 x 1536 fp32 8.2 -> 8.1 (12.5 -> 9.1)
template <int FMT, int XT>
__global__ __launch_bounds__(1024) void tensor_quant_kernel(const QuantArgs a) {
    constexpr int XB = XT == DAXQ_F32 ? 4 : 2, U = kTensorQuantPieces / 16, NCH = (DAXQ_MAX_TENSOR_K / 8 + 1023) / 1024;
    constexpr uint32_t kAbs = XT == DAXQ_F32 ? 0x7fffffffu : 0x7fffu;
    __shared__ uint32_t s_max[16];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nch = a.k >> 3, npad = a.kfill >> 3, rest = a.k & 7, pieces = (nch + 63) >> 6;  // (nch > 0: tensor_quant_applies)
    const bool ragged = ((a.k | a.kfill) & 7) != 0;  // as in quant_rows_kernel
    auto element = [&](const char* xr) __attribute__((always_inline)) -> uint32_t {
        if constexpr (XT == DAXQ_F32) return reinterpret_cast<const uint32_t*>(xr)[nch * 8 + lane];
        else return reinterpret_cast<const uint16_t*>(xr)[nch * 8 + lane];
    };
    const char* xr = a.x + (int64_t)blockIdx.x * a.ld_x * XB;
    Chunk<XT> v[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int c = i * 1024 + t;
        if (i * 1024 < nch) load_chunk<XT>(v[i], xr + (uint32_t)(c < nch ? c : nch - 1) * (8u * XB));
        else v[i] = Chunk<XT>{};
    }
    const uint32_t tail = wave == 0 && lane < rest ? element(xr) : 0;

    // the wavefront's pieces: the first, then every sixteenth (pieces <= 36: products with 2^16 / pieces, rounded up, give whole
    // quotients)
    const int inv_pieces = (65536 + pieces - 1) / pieces, rows16 = (16 * inv_pieces) >> 16, c16 = 16 - rows16 * pieces;
    int row = (wave * inv_pieces) >> 16, c = wave - row * pieces;
    uint32_t mx = 0, tl = 0;
    Chunk<XT> w[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (row < a.m) {
            const char* wr = a.x + row * a.ld_x * XB;
            const int at = c * 64 + lane;
            // (with load_chunk: 12 x 5120 fp32 11.1 -> 15.1 us)
            load_chunk_shared<XT>(w[u], wr + (uint32_t)(at < nch ? at : nch - 1) * (8u * XB));
            if (c == pieces - 1 && lane < rest) {
                const uint32_t e = element(wr) & kAbs;
                tl = e > tl ? e : tl;
            }
        } else {
            w[u] = Chunk<XT>{};
        }
        row += rows16, c += c16;
        if (c >= pieces) c -= pieces, ++row;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) mx = chunk_amax<XT>(mx, w[u]);
    mx = amax_of_lane<XT>(mx);
    mx = wave_max_u32(tl > mx ? tl : mx);
    if (lane == 0) s_max[wave] = mx;
    __syncthreads();
    const uint32_t amax = wave_max_u32(s_max[lane & 15]);
    const float s = scale_from_amax_bits_rt<XT>(amax, a.qmax, a.eps, a.round_x);
    if (t == 0) {
        a.scale[blockIdx.x] = s;
        if (a.scale1 && blockIdx.x == 0) a.scale1[0] = s;
    }
    const float inv = 1.0f / s;  // IEEE division, not v_rcp_f32
    uint8_t* qr = a.q + (int64_t)blockIdx.x * a.ld_q;
    with_form<FMT, XT>(s, a.qmax, false, a.round_x, 1, [&](auto FORM) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            if (i * 1024 >= npad) continue;
            const int at = i * 1024 + t;
            float f[8];
            chunk_values<XT>(v[i], f);
            const uint2 o = quant8<FMT, decltype(FORM)::value, XT>(f, s, inv);
            if (at < nch) store_chunk<kStoreKeep>(qr + (uint32_t)at * 8u, o);
            else if (!ragged && at < npad) store_chunk<kStoreKeep>(qr + (uint32_t)at * 8u, make_uint2(0, 0));
        }
    });
    if (ragged && wave == 0) {
        const float f = x_bits_to_f32<XT>(tail);
        uint8_t o;
        if constexpr (FMT == 0) o = (uint8_t)q_i8_bits(f, inv);
        else o = (uint8_t)cvt_pk_f8<FMT>(q_f8_pre<FMT, true>(f, s, inv), 0.0f, 0, false);
        for (int at = nch * 8 + lane; at < a.kfill; at += 64) qr[at] = at < a.k ? o : 0;
    }
}

// Which matrices: those whose pieces are all in flight at once.  With more of them the loads take turns and the GPU loses what the
// host gains: 17 x 5120 bf16 (170 pieces) 11.7 -> 12.2 us with the GEMM, 64 x 1536 (192) 8.8 -> 9.3, 250 x 256 8.4 -> 9.9.
// Not where the bytes lie over the matrix: a workgroup would store into what another one still reads.
static bool tensor_quant_applies(const void* x, int64_t row_bytes, int64_t m, int64_t k, int64_t x_bytes, const void* q, int64_t ld_q) {
    if (k < 64 || m > kTensorQuantPieces || m * ((k / 8 + 63) / 64) > kTensorQuantPieces) return false;
    const uintptr_t x0 = (uintptr_t)x, x1 = x0 + (uintptr_t)((m - 1) * row_bytes + x_bytes);
    const uintptr_t q0 = (uintptr_t)q, q1 = q0 + (uintptr_t)((m - 1) * ld_q + fill_width(k, ld_q));
    return q1 <= x0 || x1 <= q0;
}

template <int FMT>
static bool launch_tensor_quant(const QuantArgs& a, int x_dtype, hipStream_t st) {
    const dim3 grid((unsigned)a.m), block(1024);
    if (x_dtype == DAXQ_BF16) launch_kernel((tensor_quant_kernel<FMT, DAXQ_BF16>), grid, block, 0, st, a);
    else if (x_dtype == DAXQ_F16) launch_kernel((tensor_quant_kernel<FMT, DAXQ_F16>), grid, block, 0, st, a);
    else if (x_dtype == DAXQ_F32) launch_kernel((tensor_quant_kernel<FMT, DAXQ_F32>), grid, block, 0, st, a);
    else return false;
    return true;
}

// Per-row min and max of a bf16 / fp16 / fp32 matrix in fp32 (observer statistics), one workgroup per row, 16-byte loads.
// The bit patterns are compared as two's-complement integers (magnitude bits of negative values flipped), two 16-bit
// values per instruction; a NaN sorts beyond either infinity and makes both results NaN.  HBM-bound; measured against two-byte
// loads and NaN-aware fp32 comparisons: 13824 x 5120 bf16 56.1 -> 22.9 us, 75600 x 5120 409 -> 118 us = 6.5 TB/s.
typedef short daxq_s2 __attribute__((ext_vector_type(2)));
template <int XT>
__device__ __forceinline__ int order_key(uint32_t w) {  // (a pair of values per word for the 16-bit types)
    if constexpr (XT == DAXQ_F32) return (int)(w ^ (((int)w >> 31) & 0x7fffffff));
    const daxq_s2 v = __builtin_bit_cast(daxq_s2, w);
    return (int)(w ^ (__builtin_bit_cast(uint32_t, (daxq_s2)(v >> 15)) & 0x7fff7fffu));
}
template <int XT>
__device__ __forceinline__ void keys_minmax(int& lo, int& hi, int key) {
    if constexpr (XT == DAXQ_F32) {
        lo = key < lo ? key : lo;
        hi = key > hi ? key : hi;
    } else {
        const daxq_s2 k = __builtin_bit_cast(daxq_s2, key);
        lo = __builtin_bit_cast(int, __builtin_elementwise_min(__builtin_bit_cast(daxq_s2, lo), k));
        hi = __builtin_bit_cast(int, __builtin_elementwise_max(__builtin_bit_cast(daxq_s2, hi), k));
    }
}
template <int XT>
__device__ __forceinline__ float value_of_key(int key) {
    if constexpr (XT == DAXQ_F32) return __uint_as_float((uint32_t)key ^ ((uint32_t)(key >> 31) & 0x7fffffffu));
    const uint32_t w = (uint32_t)key & 0xffffu;
    return x_bits_to_f32<XT>(w & 0x8000u ? w ^ 0x7fffu : w);
}

// U: loads per lane in flight, as many as the row has for 256 lanes, up to four
template <int XT, int U>
__global__ __launch_bounds__(256) void row_minmax_kernel(const char* __restrict__ x, int64_t k, int64_t ld_x, float* __restrict__ mn,
                                                         float* __restrict__ mx) {
    constexpr int XB = XT == DAXQ_F32 ? 4 : 2;
    __shared__ int s_lo[4], s_hi[4];
    const int64_t row = blockIdx.x, nch = k >> 3;
    const char* xr = x + row * ld_x * XB;
    int lo = XT == DAXQ_F32 ? 0x7fffffff : 0x7fff7fff, hi = XT == DAXQ_F32 ? (int)0x80000000 : (int)0x80008000;
    for (int64_t c = threadIdx.x; c < nch; c += U * 256) {
        Chunk<XT> v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) load_chunk<XT>(v[u], xr + (c + u * 256 < nch ? c + u * 256 : c) * (8 * XB));
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < (XT == DAXQ_F32 ? 2 : 1); ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) keys_minmax<XT>(lo, hi, order_key<XT>(v[u].w[h][i]));
    }
    const int64_t e = (nch << 3) + threadIdx.x;
    if (e < k) {
        uint32_t w;
        if constexpr (XT == DAXQ_F32) w = reinterpret_cast<const uint32_t*>(xr)[e];
        else w = reinterpret_cast<const uint16_t*>(xr)[e] * 0x10001u;
        keys_minmax<XT>(lo, hi, order_key<XT>(w));
    }
    if constexpr (XT != DAXQ_F32) {  // the pair's own minimum and maximum, sign-extended
        const int l0 = (int)(short)lo, l1 = lo >> 16, h0 = (int)(short)hi, h1 = hi >> 16;
        lo = l0 < l1 ? l0 : l1;
        hi = h0 > h1 ? h0 : h1;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const int ol = __shfl_xor(lo, off, 64), oh = __shfl_xor(hi, off, 64);
        lo = ol < lo ? ol : lo;
        hi = oh > hi ? oh : hi;
    }
    if ((threadIdx.x & 63) == 0) {
        s_lo[threadIdx.x >> 6] = lo;
        s_hi[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < 4; ++w) {
            lo = s_lo[w] < lo ? s_lo[w] : lo;
            hi = s_hi[w] > hi ? s_hi[w] : hi;
        }
        const float l = value_of_key<XT>(lo), h = value_of_key<XT>(hi);
        mn[row] = h != h ? h : l;
        mx[row] = l != l ? l : h;
    }
}

// scale[i] = max( max(-min[i], max[i]) / qmax, eps ), all in fp32
__global__ void scale_from_minmax_kernel(const float* __restrict__ mn, const float* __restrict__ mx, int64_t n,
                                         float qmax, float eps, float* __restrict__ scale) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const float a = max_nan(-mn[i], mx[i]);
        scale[i] = max_nan(a / qmax, eps);
    }
}

}  // namespace daxq

extern "C" {

int daxq_act_quant_i8(const void* x, int64_t m, int64_t k, int64_t ld_x, int8_t* q, int64_t ld_q, float* scale,
                      daxq_stream_t stream) {
    return daxq::launch_quant_rows<0, false>(x, m, k, ld_x, q, ld_q, scale, 127.0f, (hipStream_t)stream);
}

int daxq_act_quant_e4m3(const void* x, int64_t m, int64_t k, int64_t ld_x, uint8_t* q, int64_t ld_q, float* scale,
                        daxq_stream_t stream) {
    return daxq::launch_quant_rows<1, false>(x, m, k, ld_x, q, ld_q, scale, 448.0f, (hipStream_t)stream);
}

int daxq_act_quant_e5m2(const void* x, int64_t m, int64_t k, int64_t ld_x, uint8_t* q, int64_t ld_q, float* scale,
                        daxq_stream_t stream) {
    return daxq::launch_quant_rows<2, false>(x, m, k, ld_x, q, ld_q, scale, 57344.0f, (hipStream_t)stream);
}

int daxq_quantize_rows_i8(const void* x, int64_t m, int64_t k, int64_t ld_x, const float* scale, int8_t* q,
                          int64_t ld_q, daxq_stream_t stream) {
    return daxq::launch_quant_rows<0, true>(x, m, k, ld_x, q, ld_q, const_cast<float*>(scale), 127.0f,
                                                       (hipStream_t)stream);
}

int daxq_quantize_rows_e4m3(const void* x, int64_t m, int64_t k, int64_t ld_x, const float* scale, uint8_t* q,
                            int64_t ld_q, daxq_stream_t stream) {
    return daxq::launch_quant_rows<1, true>(x, m, k, ld_x, q, ld_q, const_cast<float*>(scale), 448.0f,
                                                      (hipStream_t)stream);
}

int daxq_quantize_rows_e5m2(const void* x, int64_t m, int64_t k, int64_t ld_x, const float* scale, uint8_t* q,
                            int64_t ld_q, daxq_stream_t stream) {
    return daxq::launch_quant_rows<2, true>(x, m, k, ld_x, q, ld_q, const_cast<float*>(scale), 57344.0f,
                                                      (hipStream_t)stream);
}

int daxq_row_minmax_t(const void* x, int x_dtype, int64_t m, int64_t k, int64_t ld_x, float* min_out, float* max_out,
                      daxq_stream_t stream) {
    using namespace daxq;
    if (m < 0 || k <= 0 || ld_x < k || m > 0x7fffffff) return fail(DAXQ_ERR_ARG, "row_minmax: bad shape m=%lld k=%lld", (long long)m, (long long)k);
    if (m == 0) return DAXQ_OK;
    if (!x || !min_out || !max_out) return fail(DAXQ_ERR_ARG, "row_minmax: null pointer");
    const dim3 grid((unsigned)m), block(256);
    hipStream_t st = (hipStream_t)stream;
    const char* xp = static_cast<const char*>(x);
    auto launch = [&](auto XT) {
        constexpr int X = decltype(XT)::value;
        if (k <= 2048) launch_kernel((row_minmax_kernel<X, 1>), grid, block, 0, st, xp, k, ld_x, min_out, max_out);
        else if (k <= 4096 || X == DAXQ_F32) launch_kernel((row_minmax_kernel<X, 2>), grid, block, 0, st, xp, k, ld_x, min_out, max_out);
        else launch_kernel((row_minmax_kernel<X, 4>), grid, block, 0, st, xp, k, ld_x, min_out, max_out);
    };
    switch (x_dtype) {
        case DAXQ_BF16: launch(std::integral_constant<int, DAXQ_BF16>{}); break;
        case DAXQ_F16: launch(std::integral_constant<int, DAXQ_F16>{}); break;
        case DAXQ_F32: launch(std::integral_constant<int, DAXQ_F32>{}); break;
        default: return fail(DAXQ_ERR_ARG, "row_minmax: unknown element type %d", x_dtype);
    }
    return check_launch("row_minmax");
}

int daxq_row_minmax(const void* x, int64_t m, int64_t k, int64_t ld_x, float* min_out, float* max_out,
                    daxq_stream_t stream) {
    return daxq_row_minmax_t(x, DAXQ_BF16, m, k, ld_x, min_out, max_out, stream);
}

int daxq_act_quant_rows(const void* x, int x_dtype, int q_fmt, int64_t m, int64_t k, int64_t ld_x, void* q, int64_t ld_q,
                        float* scale, daxq_stream_t stream) {
    return daxq::launch_quant_rows_fmt<false>(q_fmt, x, x_dtype, m, k, ld_x, q, ld_q, scale, (hipStream_t)stream);
}

int daxq_act_quant_rows_ex(const void* x, int x_dtype, int q_fmt, int64_t m, int64_t k, int64_t ld_x, void* q, int64_t ld_q,
                           float* scale, float quant_max, float eps, int scale_round, daxq_stream_t stream) {
    if (scale_round != DAXQ_SCALE_ROUND_X && scale_round != DAXQ_SCALE_ROUND_NONE)
        return daxq::fail(DAXQ_ERR_ARG, "act_quant_rows_ex: unknown scale rounding %d", scale_round);
    if (!(quant_max > 0.0f)) return daxq::fail(DAXQ_ERR_ARG, "act_quant_rows_ex: quant_max must be positive");
    return daxq::launch_quant_rows_fmt<false>(q_fmt, x, x_dtype, m, k, ld_x, q, ld_q, scale, (hipStream_t)stream, quant_max,
                                                    eps, scale_round == DAXQ_SCALE_ROUND_X);
}

int daxq_weight_quant_rows(const void* w, int w_dtype, int q_fmt, int64_t n, int64_t k, int64_t ld_w, void* q, int64_t ld_q, float* scale,
                           float quant_max, float eps, daxq_stream_t stream) {
    if (!(quant_max > 0.0f)) return daxq::fail(DAXQ_ERR_ARG, "weight_quant_rows: quant_max must be positive");
    daxq::ScaleKind t;
    t.weight = true;
    return daxq::launch_quant_rows_fmt<false>(q_fmt, w, w_dtype, n, k, ld_w, q, ld_q, scale, (hipStream_t)stream, quant_max, eps, 0, t);
}

int daxq_quantize_rows(const void* x, int x_dtype, int q_fmt, int64_t m, int64_t k, int64_t ld_x, const float* scale,
                       void* q, int64_t ld_q, daxq_stream_t stream) {
    return daxq::launch_quant_rows_fmt<true>(q_fmt, x, x_dtype, m, k, ld_x, q, ld_q, const_cast<float*>(scale),
                                                    (hipStream_t)stream);
}

int daxq_act_quant_tensor(const void* x, int x_dtype, int q_fmt, int64_t m, int64_t k, int64_t ld_x, void* q, int64_t ld_q,
                          float* scale_rows, float* scale1, void* scratch, float quant_max, float eps, int scale_round, daxq_stream_t stream) {
    using namespace daxq;
    if (m < 0 || k <= 0 || ld_x < k || ld_q < k || m > 0x7fffffff || k > DAXQ_MAX_TENSOR_K)
        return fail(DAXQ_ERR_ARG, "act_quant_tensor: bad shape m=%lld k=%lld (at most %d columns)", (long long)m, (long long)k, DAXQ_MAX_TENSOR_K);
    if (scale_round != DAXQ_SCALE_ROUND_X && scale_round != DAXQ_SCALE_ROUND_NONE)
        return fail(DAXQ_ERR_ARG, "act_quant_tensor: unknown scale rounding %d", scale_round);
    if (!(quant_max > 0.0f) || !(eps >= 0.0f)) return fail(DAXQ_ERR_ARG, "act_quant_tensor: quant_max must be positive and eps not negative");
    if (m == 0) return DAXQ_OK;
    if (!x || !q || !scale_rows || !scratch) return fail(DAXQ_ERR_ARG, "act_quant_tensor: null pointer");
    if ((uintptr_t)scratch & 15) return fail(DAXQ_ERR_ALIGN, "act_quant_tensor: the scratch must be 16-byte aligned");
    const int xb = x_dtype == DAXQ_F32 ? 4 : 2;
    if ((uintptr_t)x & (xb - 1)) return fail(DAXQ_ERR_ALIGN, "act_quant_tensor: x must be element aligned");
    hipStream_t st = (hipStream_t)stream;
    if (((uintptr_t)scale_rows & 3) == 0 && tensor_quant_applies(x, ld_x * xb, m, k, k * xb, q, ld_q)) {
        const QuantArgs a{static_cast<const char*>(x), m, ld_x, (int)k, (int)fill_width(k, ld_q), static_cast<uint8_t*>(q), ld_q, scale_rows, nullptr,
                          0, nullptr, scale1, quant_max, eps, scale_round == DAXQ_SCALE_ROUND_X, 1};
        if (q_fmt == DAXQ_FMT_I8 ? launch_tensor_quant<0>(a, x_dtype, st)
                                 : q_fmt == DAXQ_FMT_E4M3 ? launch_tensor_quant<1>(a, x_dtype, st)
                                                          : q_fmt == DAXQ_FMT_E5M2 && launch_tensor_quant<2>(a, x_dtype, st))
            return check_launch("tensor_quant");
    }
    uint32_t* part = static_cast<uint32_t*>(scratch);
    const AmaxArgs a{static_cast<const char*>(x), m, ld_x, (int)k, quant_unit(x_dtype, fill_width(k, ld_q)), part};
    const dim3 grid(kPartials), block(1024);
    switch (x_dtype) {
        case DAXQ_BF16: launch_kernel(tensor_amax_kernel<DAXQ_BF16>, grid, block, 0, st, a); break;
        case DAXQ_F16: launch_kernel(tensor_amax_kernel<DAXQ_F16>, grid, block, 0, st, a); break;
        case DAXQ_F32: launch_kernel(tensor_amax_kernel<DAXQ_F32>, grid, block, 0, st, a); break;
        default: return fail(DAXQ_ERR_ARG, "act_quant_tensor: unknown element type %d", x_dtype);
    }
    if (int rc = check_launch("tensor_amax")) return rc;
    ScaleKind t;
    t.partials = part;
    t.scale1 = scale1;
    return launch_quant_rows_fmt<false>(q_fmt, x, x_dtype, m, k, ld_x, q, ld_q, scale_rows, st, quant_max, eps, scale_round == DAXQ_SCALE_ROUND_X, t);
}

int daxq_quantize_tensor(const void* x, int x_dtype, int q_fmt, int64_t m, int64_t k, int64_t ld_x, const float* scale1, void* q,
                         int64_t ld_q, float* scale_rows, daxq_stream_t stream) {
    daxq::ScaleKind t;
    t.one_scale = true;
    t.scale_rows = scale_rows;
    return daxq::launch_quant_rows_fmt<true>(q_fmt, x, x_dtype, m, k, ld_x, q, ld_q, const_cast<float*>(scale1), (hipStream_t)stream, 0.0f,
                                             daxq::kEps, 1, t);
}

int daxq_scale_from_minmax(const float* min_in, const float* max_in, int64_t n, float qmax, float* scale,
                           daxq_stream_t stream) {
    return daxq_scale_from_minmax_eps(min_in, max_in, n, qmax, daxq::kEps, scale, stream);
}

int daxq_scale_from_minmax_eps(const float* min_in, const float* max_in, int64_t n, float qmax, float eps, float* scale,
                               daxq_stream_t stream) {
    using namespace daxq;
    if (n < 0 || !(qmax > 0.0f) || eps != eps) return fail(DAXQ_ERR_ARG, "scale_from_minmax: bad argument");
    if (n == 0) return DAXQ_OK;
    if (!min_in || !max_in || !scale) return fail(DAXQ_ERR_ARG, "scale_from_minmax: null pointer");
    launch_kernel(scale_from_minmax_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       min_in, max_in, n, qmax, eps, scale);
    return check_launch("scale_from_minmax");
}

}  // extern "C"
