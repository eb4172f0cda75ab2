// W8A8 GEMM for a handful of rows, or few outputs at all (gfx950): every wavefront streams its own part of the weight, no barriers in the K loop.
//
// What bounds it: every byte of the weight is needed once and multiplied with a few rows, so the launch is a stream of the
// weight from HBM (26 MB at N = K = 5120: 4.3 us at 6.2 TB/s) and what counts is how many bytes are in flight.  The tiled
// kernels put such a launch on N / 128 workgroups (40 of them at N = 5120).
//
// Work decomposition
//   workgroup  16 output columns x MB blocks of 16 rows, KS wavefronts that share K
//   wavefront  K / KS bytes of the 16 weight rows and of the activation rows, in steps of 128 bytes, through a ring of R
//              steps in an LDS region of its own
// Loads go straight into LDS (global_load_lds_dwordx4, four lanes to 64 consecutive bytes of a row); fragments are read
// back in the MFMA's layout with the chunk swizzle of the tiled kernels.  Loading the fragments directly into registers, lane
// l from row l % 16, was built first: neighbouring lanes then sit in different rows, every lane is a cache line of its own,
// and a CU takes 14 bytes per cycle instead of the 60 that four lanes to a row segment give.
// A wavefront reads only what it loaded itself, so a wait on its own load counter is all the synchronisation there is.
// INT8 runs KS = 4 or 1: sums of integers do not depend on how K is cut; partial sums meet in LDS.  FP8 runs KS = 1: an
// output element is then the same sequence of MFMAs over the same K bytes in the same register positions as in
// gemm_tile_fp8.hip, and an output row does not depend on how many rows the launch has.
// Rows and columns beyond the matrix repeat its last row / column and are not stored.
#include "gemm_rows.h"

namespace daxq {

constexpr int rows_step_bytes(int mb) { return 2048 * (1 + mb); }  // LDS of a step: 16 weight rows, then MB x 16 activation rows

// ACC: the accumulators are written out, too.  A form of its own: the branch in the epilogue alone costs every other launch
// 0.1 to 0.3 us (121 x 384, K = 13824 18.6 -> 18.7, e4m3 512 x 1000, K = 5120 20.2 -> 20.5).
template <bool FP8, int F8, int MB, int R, int KS, int OUTK, bool ACC>
__global__ __launch_bounds__(64 * KS) void gemm_rows_kernel(const GemmArgs p) {
    typedef typename Acc16<FP8>::type acc_t;
    constexpr int STEP = rows_step_bytes(MB), L = 2 * (1 + MB);  // load instructions of a step
    static_assert(R >= 2 && (R - 1) * L < 64, "the load counter holds 63");
    static_assert(KS == 1 || KS * MB * 1024 <= KS * R * STEP, "the partial sums fit the ring");
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l15 = lane & 15, g4 = lane >> 4;
    const int n0 = (int)blockIdx.x * 16, mbase = (int)blockIdx.y * (16 * MB);

    const int steps = p.k >> 7;
    const int first = steps * wave / KS, cnt = steps * (wave + 1) / KS - first;

    // ---- memory side: a load instruction takes 16 rows x 64 bytes, lane l row l / 4 and the 16-byte chunk that the swizzle
    //      stores at chunk l % 4 of the row
    const int lrow = lane >> 2;
    const uint32_t gsw = (uint32_t)(((lane & 3) ^ ((lrow >> 1) & 3)) << 4);
    const uint8_t* wbase = p.b + (int64_t)n0 * p.ldb + (int64_t)first * 128;
    const uint8_t* xbase = p.a + (int64_t)mbase * p.lda + (int64_t)first * 128;  // (32-bit offsets reach 64 rows)
    const uint32_t wcol = n0 + lrow < p.n ? lrow : p.n - 1 - n0;
    uint32_t woff = wcol * (uint32_t)p.ldb + gsw, xoff[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) xoff[i] = (uint32_t)(mbase + i * 16 + lrow < p.m ? i * 16 + lrow : p.m - 1 - mbase) * (uint32_t)p.lda + gsw;
    const uint32_t ring = (uint32_t)(uintptr_t)(DAXQ_LDS uint8_t*)smem + (uint32_t)wave * (R * STEP);
    auto load = [&](int step, uint32_t slot) __attribute__((always_inline)) {
        const uint8_t* w = wbase + (int64_t)step * 128;
        const uint8_t* x = xbase + (int64_t)step * 128;
        const uint32_t dst = ring + slot;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            __builtin_amdgcn_global_load_lds((const DAXQ_GLOBAL void*)(w + h * 64 + woff), (DAXQ_LDS void*)(uintptr_t)(dst + h * 1024), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                __builtin_amdgcn_global_load_lds((const DAXQ_GLOBAL void*)(x + h * 64 + xoff[i]),
                                                 (DAXQ_LDS void*)(uintptr_t)(dst + 2048 * (1 + i) + h * 1024), 16, 0, 0);
    };

    // ---- LDS side: row l % 16, K chunk l / 16 of either half
    const uint8_t* rd = smem + wave * (R * STEP) + l15 * 64 + ((g4 ^ ((l15 >> 1) & 3)) << 4);
    acc_t acc[MB] = {};
    auto fragment = [&](uint32_t at) __attribute__((always_inline)) {
        const v4i lo = *reinterpret_cast<const v4i*>(rd + at), up = *reinterpret_cast<const v4i*>(rd + at + 1024);
        return __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto next_slot = [](uint32_t slot) { return slot == (R - 1) * STEP ? 0 : slot + STEP; };
    // U steps that have landed: their fragments into registers, the steps R later into their places, their MFMAs.  Two at a
    // time with one row block: the wait for the LDS reads is then paid half as often (one row, N = 1536, K = 8960, FP8: 9.0 ->
    // 7.8 us; with two row blocks and more the loads' own issue is what a step takes, and two steps at a time lose 3 %)
    auto work = [&](auto STEPS, auto MORE, int step, uint32_t slot) __attribute__((always_inline)) {
        constexpr int U = decltype(STEPS)::value;
        v8i w[U], x[U][MB];
        uint32_t at[U];
        at[0] = slot;
#pragma unroll
        for (int u = 1; u < U; ++u) at[u] = next_slot(at[u - 1]);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            w[u] = fragment(at[u]);
#pragma unroll
            for (int i = 0; i < MB; ++i) x[u][i] = fragment(at[u] + 2048 * (1 + i));
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
    // (loads retire in order: a step has landed when no more than the loads issued behind it are in flight)
    const int ahead = cnt < R ? cnt : R;
#pragma unroll
    for (int s = 0; s < R; ++s)
        if (s < ahead) load(s, s * STEP);
    __builtin_amdgcn_sched_barrier(0);
    int step = 0;
    uint32_t slot = 0;
    for (; MB == 1 && step + R + 1 < cnt; step += 2) {
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
        work(Int<1>{}, No{}, 0, slot);
        slot = next_slot(slot);
    };
    for_down<R - 1>(tail);

    // ---- epilogue (the arithmetic of tile_epilogue16): a lane owns output row l % 16 of a block and 4 consecutive columns
    const int nc = n0 + 4 * g4;
    const ColumnBits<OUTK> cols(p, nc);
    v4i* s_part = reinterpret_cast<v4i*>(smem);
    if constexpr (KS > 1) {
        __syncthreads();  // every wavefront is done with the ring
#pragma unroll
        for (int i = 0; i < MB; ++i) s_part[(wave * MB + i) * 64 + lane] = __builtin_bit_cast(v4i, acc[i]);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        if (KS > 1 && i % KS != wave) continue;  // the wavefronts share the row blocks out
        if constexpr (KS > 1) {
            v4i sum = s_part[i * 64 + lane];
#pragma unroll
            for (int s = 1; s < KS; ++s) sum += s_part[(s * MB + i) * 64 + lane];
            acc[i] = __builtin_bit_cast(acc_t, sum);
        }
        const int m = mbase + i * 16 + l15;
        if (m >= p.m || nc >= p.n) continue;
        const float sxv = p.sx[m];
        if constexpr (ACC) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (nc + e >= p.n) continue;
                if constexpr (FP8) static_cast<float*>(p.acc)[(int64_t)m * p.ldacc + nc + e] = acc[i][e];
                else static_cast<int32_t*>(p.acc)[(int64_t)m * p.ldacc + nc + e] = acc[i][e];
            }
        }
        store_columns<FP8, OUTK>(p, acc[i], sxv, cols, m, nc);
    }
}

// args null: only raises the kernel's LDS limit on the current device.
template <bool FP8, int F8, int MB, int R, int KS, int OUTK, bool ACC = false>
static int launch_rows_one(const GemmArgs* args, hipStream_t st) {
    constexpr int lds = KS * R * rows_step_bytes(MB);
    auto kern = gemm_rows_kernel<FP8, F8, MB, R, KS, OUTK, ACC>;
    static std::atomic<uint64_t> lds_set{0};  // per instantiation
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), lds, lds_set)) return rc;
    if (!args) return DAXQ_OK;
    const dim3 grid((unsigned)((args->n + 15) / 16), (unsigned)((args->m + 16 * MB - 1) / (16 * MB)));
    launch_kernel(kern, grid, dim3(64 * KS), lds, st, *args);
    return check_launch("gemm_rows");
}

// Which form: the number of workgroups per row block (n / 16) and of rows decide how many bytes are in flight and how often
// the activation is fetched.  Measured, us, weight in the caches / never touched before (INT8; FP8 the same where KS = 1):
//                            MB,R,KS   1,10,1      1,5,1       2,5,1       1,5,4       2,3,4       4,2,4      128x128 tiles
//   m = 16,  5120 x 5120           6.1 / 9.3   6.3 / 9.9   9.4 / 10.2  6.8 / 11.4  7.4 / 11.7  9.1 / 13.3   18.8 / 33.6
//   m = 32,  5120 x 5120           7.4 / 11.9  7.1 / 11.6  9.7 / 11.1  8.2 / 11.9  8.9 / 14.5  10.0 / 15.6  18.7 / 33.5
//   m = 64,  5120 x 5120          16.5 / 21.4 12.4 / 17.9 10.3 / 15.5 14.4 / 17.6 10.9 / 14.7  12.6 / 19.0  20.5 / 33.6
//   m = 128, 5120 x 5120          24.7 / 29.4 24.0 / 29.5 18.0 / 25.2 23.8 / 27.0 20.2 / 23.3  16.5 / 19.8  18.6 / 33.3
//   m = 32,  N = 15360            25.6 / 27.8 23.5 / 26.9 15.0 / 20.1 27.6 / 31.2 18.1 / 26.9  20.2 / 28.3  23.8 / 34.7
//   m = 64,  N = 15360            47.6 / 50.1 44.6 / 48.5 31.2 / 37.7 51.1 / 54.5 33.1 / 39.5  24.5 / 35.8  24.0 / 35.0
//   m = 16,  N = 1536, K = 8960    7.8 / 8.0   7.9 / 9.2  14.5 / 14.5  4.5 / 6.0   5.7 / 6.2    7.7 / 7.9   26.4 / 30.0
//   m = 64,  N = 1536, K = 8960    8.2 / 8.5   8.3 / 9.4  14.8 / 14.7  7.4 / 8.2   5.8 / 7.5    7.8 / 10.3  26.3 / 29.5
//   m = 128, N = 1536, K = 8960   10.5 / 11.7  9.9 / 11.2 14.9 / 15.1 12.6 / 12.9  9.6 / 10.9   8.0 / 10.2  26.3 / 29.4
// Few workgroups (small n): cut K where the sums allow it, one row block per workgroup where they do not; many: two row
// blocks, so that the activation is fetched half as often.  With more than 32 rows and N > 8192 the tiles, which fetch it
// once per 128 columns, are as fast.
// FP8 with more than 64 rows and many columns: four row blocks, 2,5,1 / 4,3,1 beside the tiles on 128 rows, us on weights out of
// reach of the caches: N = 8192, K = 5120, m = 72 22.3 / 17.6, m = 128 30.2 / 22.0, 24.1; K = 13824, m = 128 85.2 / 69.4, 72.8;
// N = 6144, K = 5120, m = 128 27.2 / 19.4, 26.8; at N = 5120 15.1 / 15.6 (m = 72) and 21.5 / 19.5 (128), at N = 3072 9.8 / 12.8 and
// 14.3 / 14.7.
// More than 128 rows (rows_applies says which): `blocks` of 16 x 16 outputs count the work.  us, 1,5,1 / 2,5,1 / 4,3,1 and for
// INT8 2,3,4, beside the tiles (or, n < 128, the generic kernel):
//   INT8  390 x 176, K = 3456 (275 blocks)  4.7 / 7.2 / - / 4.0, 11.9     543 x 254, K = 2688 (544)    4.4 / 6.3 / - / 5.0, 10.4
//         392 x 819, K = 1408 (1300)        5.1 / 5.1 / 6.6 / 5.6, 8.7    242 x 2100, K = 8448 (2112) 32.3 / 26.0 / 23.4 / 26.3, 28.6
//   e4m3  443 x 275, K = 3200 (504)         4.6 / 5.9 / 7.8, 12.0         331 x 644, K = 5888 (861)   11.7 / 10.9 / 12.0, 19.5
//         338 x 1233, K = 6016 (1716)      18.1 / 15.5 / 14.2, 21.7
static int64_t row_blocks(int64_t m, int64_t n) { return ((m + 15) / 16) * ((n + 15) / 16); }

template <bool FP8, int F8, int OUTK>
static int launch_rows_out(const GemmArgs* a, hipStream_t st) {
    if (!a) {
        int rc = launch_rows_one<FP8, F8, 1, 10, 1, OUTK>(a, st);
        if (!rc) rc = launch_rows_one<FP8, F8, 1, 5, 1, OUTK>(a, st);
        if (!rc) rc = launch_rows_one<FP8, F8, 2, 5, 1, OUTK>(a, st);
        if (!rc) rc = launch_rows_one<FP8, F8, 4, 3, 1, OUTK>(a, st);
        if (!rc) rc = launch_rows_one<FP8, F8, 4, 3, 1, OUTK, true>(a, st);
        if constexpr (!FP8) {
            if (!rc) rc = launch_rows_one<FP8, F8, 1, 5, 4, OUTK>(a, st);
            if (!rc) rc = launch_rows_one<FP8, F8, 2, 3, 4, OUTK>(a, st);
            if (!rc) rc = launch_rows_one<FP8, F8, 4, 2, 4, OUTK>(a, st);
        }
        return rc;
    }
    if (a->acc) return launch_rows_one<FP8, F8, 4, 3, 1, OUTK, true>(a, st);  // (tests; every form gives the same bits)
    if (a->m > 128) {
        const int64_t blocks = row_blocks(a->m, a->n);
        if constexpr (!FP8) {
            if (blocks <= 512) return launch_rows_one<FP8, F8, 2, 3, 4, OUTK>(a, st);
        }
        if (blocks <= (FP8 ? 640 : 1024)) return launch_rows_one<FP8, F8, 1, 5, 1, OUTK>(a, st);
        if (blocks <= 1280 || a->k < 2048) return launch_rows_one<FP8, F8, 2, 5, 1, OUTK>(a, st);
        return launch_rows_one<FP8, F8, 4, 3, 1, OUTK>(a, st);
    }
    if constexpr (!FP8) {
        if (a->n < 4096 || a->m > 64) {
            if (a->m <= 32) return launch_rows_one<FP8, F8, 1, 5, 4, OUTK>(a, st);
            if (a->m <= 64) return launch_rows_one<FP8, F8, 2, 3, 4, OUTK>(a, st);
            return launch_rows_one<FP8, F8, 4, 2, 4, OUTK>(a, st);
        }
    }
    if constexpr (FP8) {
        if (a->m > 64 && a->n > 5120) return launch_rows_one<FP8, F8, 4, 3, 1, OUTK>(a, st);
    }
    if (a->m <= 16) return launch_rows_one<FP8, F8, 1, 10, 1, OUTK>(a, st);
    if (a->n <= 2048 || (a->m <= 32 && a->n <= 8192)) return launch_rows_one<FP8, F8, 1, 5, 1, OUTK>(a, st);
    return launch_rows_one<FP8, F8, 2, 5, 1, OUTK>(a, st);
}

template <bool FP8, int F8>
static int launch_rows_fmt(const GemmArgs* a, int out_kind, hipStream_t st) {
    if (out_kind == DAXQ_F16) return launch_rows_out<FP8, F8, DAXQ_F16>(a, st);
    if (out_kind == DAXQ_F32) return launch_rows_out<FP8, F8, DAXQ_F32>(a, st);
    return launch_rows_out<FP8, F8, DAXQ_BF16>(a, st);
}

static int launch_rows_any(const GemmArgs* a, int out_kind, bool fp8, int f8, hipStream_t st) {
    if (!fp8) return launch_rows_fmt<false, 0>(a, out_kind, st);
    switch (f8) {
        case 1: return launch_rows_fmt<true, 1>(a, out_kind, st);
        case 2: return launch_rows_fmt<true, 2>(a, out_kind, st);
        case 3: return launch_rows_fmt<true, 3>(a, out_kind, st);
        default: return launch_rows_fmt<true, 0>(a, out_kind, st);
    }
}

// every instantiation on the current device, so that a first launch may sit inside a stream capture
int prepare_rows_kernels() {
    int rc = 0;
    for (int out_kind : {DAXQ_BF16, DAXQ_F16, DAXQ_F32}) {
        if (!rc) rc = launch_rows_any(nullptr, out_kind, false, 0, nullptr);
        for (int f8 = 0; f8 < 4 && !rc; ++f8) rc = launch_rows_any(nullptr, out_kind, true, f8, nullptr);
    }
    return rc;
}

// Launches this kernel is the library's choice for: those of so few outputs that it has more wavefronts to put on them than fitted
// tiles have workgroups (gemm_tile_fit.hip), and all of fewer rows than such a tile has.  `blocks` of 16 x 16 outputs; us, here /
// 64 x 64 tiles (64 x 96 where marked):
//   INT8  66 x 976, K = 3072 (305) 5.0 / 5.9            179 x 448, K = 7168 (336) 6.8 / 12.0          87 x 1224, K = 4608 (462) 6.7 / 8.1
//         235 x 512, K = 5120 (480) 5.6 / 9.8           99 x 1536, K = 13824 (672) 13.6 / 19.9        106 x 1536, K = 8960 (672) 10.0 / 14.0
//         717 x 296, K = 6272 (855) 12.1 / 10.7         71 x 2928, K = 9856 (915) 17.3 / 15.3         164 x 1536, K = 4608 (1056) 9.6 / 8.7
//         219 x 1536, K = 4096 (1344) 12.6 / 8.1        71 x 4608, K = 7296 (1440) 19.1 / 12.7        111 x 4608 x 4608 (2016) 14.3 / 9.1
//   e4m3  102 x 952, K = 8064 (420) 9.4 / 12.7          107 x 1080, K = 6656 (476) 8.2 / 11.0         66 x 1760, K = 4352 (550) 7.4 / 8.2
//         79 x 1840, K = 13824 (575) 21.9 / 19.7        95 x 1712, K = 6784 (642) 13.2 / 11.1         101 x 4608, K = 1536 (2016) 6.6 / 5.3 *
//         289 x 760, K = 6016 (912) 9.3 / 10.3          224 x 1048, K = 8960 (924) 12.7 / 14.1        158 x 1920, K = 10112 (1200) 14.4 / 15.4
//         198 x 1264, K = 15360 (1027) 27.7 / 22.2      247 x 1536, K = 5120 (1536) 11.5 / 9.7        574 x 1536, K = 3968 (3456) 14.8 / 8.7
// (more than 128 rows against 64 to 128 of them: FP8 runs its wider forms there).  INT8 launches of long K stop at 131072 block-steps
// of 128 K bytes.  Fewer than 64 columns leave only the generic kernel (INT8, 9191 x 79, K = 512: 15.4 -> 6.9 us, 2404 x 74, K = 3072:
// 25.6 -> 8.2), which is as fast from about 4000 blocks at K = 4096 on.
// FP8 with fewer than 128 columns keeps the generic kernel at any number of rows: it adds in another order, and beyond a few
// thousand blocks this kernel is too slow to be the only one (e4m3 75600 x 64, K = 5120: 212 against 125 us), so a
// line between the two would change a row's bits with the rows around it.
// acc: the launch asks for its accumulators, which the fitted tiles do not write (beside 128x128 tiles the line lies at 2048 blocks).
bool rows_applies(int64_t m, int64_t n, int64_t k, bool fp8, bool acc) {
    if (fp8 && n < 128) return false;
    if (m < 64) return m <= (n > 8192 ? 32 : 63);
    if (m > (1 << 20) || n > (1 << 20)) return false;
    const int64_t blocks = row_blocks(m, n), work = blocks * (k / 128);
    if (m <= 128 && (n < 128 || (acc && n <= 8192))) return true;
    if (n < 128) return work <= 65536;
    if (m <= 128) return blocks <= (fp8 ? 600 : 768);
    return blocks <= (acc ? 2048 : fp8 ? 1280 : 768) && (fp8 || work <= 131072);
}

// 32-bit row offsets
int launch_rows(const GemmArgs& a, bool fp8, int f8, hipStream_t st) {
    if (a.lda >= (1 << 26) || a.ldb >= (1 << 26))
        return fail(DAXQ_ERR_ARG, "linear: the kernel for few rows takes row strides below 2^26");
    return launch_rows_any(&a, a.out_kind, fp8, f8, st);
}

}  // namespace daxq
