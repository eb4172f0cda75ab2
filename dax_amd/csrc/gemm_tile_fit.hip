// W8A8 GEMM of one round of workgroups: tiles of 64 x 64 to 256 x 160 outputs, chosen so that the launch's tiles just fill the CUs.
//
// What bounds such a launch (a few hundred to a few thousand rows): a CU's load path.  A tile of BM x BN moves (BM + BN) x 128 bytes
// per pair of K slices, at 95 to 105 KB per us whatever the tile (a probe that only loads: 93), and its MFMAs take less than that up
// to about 256 x 192.  160 tiles of 128 x 128 (512 x 5120) leave 96 CUs idle while each of the others moves 32 KB per pair; 216 of 128 x 96
// move 28.  Beside the loop such a launch spends 1.8 us until the first pair has landed and 1.5 to 3 us on its outputs (a tile's scales go
// straight to the registers that use them, behind the last loads); under the MFMAs the clock falls from 2.3 to 1.7 to 1.9 GHz.  The body is gemm_tile_fit.h; every tile gives the bits of the 256x256 kernels.
// Against what these launches took before (128x128 tiles, halves of 256x256 ones, the kernel for few rows), us, weights of three
// launches in turn, INT8 unless noted:
//   512 x 5120 x 5120   20.2 -> 18.4 (128 x 96)     4096 x 1536 x 1536  15.6 -> 14.4 (256 x 96)     2900 x 3080, K = 1024 fp16  19.0 -> 15.7 (256 x 160)
//   1024 x 5120 x 5120  30.4 -> 26.4 (128 x 160)    343 x 1536, K = 4608 e4m3  16.1 -> 8.8 (64 x 64)  371 x 1536, K = 13824  39.7 -> 21.1 (64 x 64)
//   195 x 5120, K = 1920  10.9 -> 6.8 (64 x 96)      84 x 13824 x 13824  103 -> 56 (64 x 128)        536 x 15360, K = 13824  133 -> 104 (192 x 192)
#include "gemm_tile_fit.h"

namespace daxq {

// The tiles, four wavefronts unless noted; NS as many pairs as the LDS of a CU holds, or of half a CU where two workgroups share it.
typedef FitTile<2, 2, 2, 2, 5> T64x64;    // two per CU
typedef FitTile<2, 2, 2, 3, 4> T64x96;    // two per CU
typedef FitTile<2, 2, 2, 4, 6> T64x128;
typedef FitTile<2, 4, 2, 3, 4> T64x192;   // eight wavefronts
typedef FitTile<2, 2, 4, 3, 5> T128x96;
typedef FitTile<2, 2, 4, 5, 4> T128x160;
typedef FitTile<2, 2, 4, 7, 3> T128x224;
typedef FitTile<2, 2, 6, 6, 3> T192x192;
typedef FitTile<2, 2, 8, 3, 3> T256x96;
typedef FitTile<2, 2, 8, 4, 3> T256x128;
typedef FitTile<2, 2, 8, 5, 3> T256x160;
constexpr int kFitCount = 11;

template <class TILE, bool FP8, int F8, int OUTK>
__global__ __launch_bounds__(TILE::T) void gemm_fit_kernel(const GemmArgs p) {
    int tm, tn;
    tile_of_block(p.gm, (int)blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
    int m0 = tm * TILE::BM, n0 = tn * TILE::BN;  // shifted inwards at the edges, as in tile_origin
    m0 = m0 + TILE::BM <= p.m ? m0 : p.m - TILE::BM;
    n0 = n0 + TILE::BN <= p.n ? n0 : p.n - TILE::BN;
    gemm_fit_body<TILE, FP8, F8, false, OUTK>(p, m0, n0);
}

// args null: only raises the kernel's LDS limit on the current device
template <class TILE, bool FP8, int F8, int OUTK>
static int launch_fit_one(const GemmArgs* args, hipStream_t st) {
    auto kern = gemm_fit_kernel<TILE, FP8, F8, OUTK>;
    static std::atomic<uint64_t> lds_set{0};  // per instantiation
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), TILE::SMEM, lds_set)) return rc;
    if (!args) return DAXQ_OK;
    GemmArgs a = *args;
    if (a.m < TILE::BM || a.n < TILE::BN) return fail(DAXQ_ERR_ARG, "linear: this tile needs m >= %d and n >= %d", TILE::BM, TILE::BN);
    a.tiles_m = (a.m + TILE::BM - 1) / TILE::BM;
    a.tiles_n = (a.n + TILE::BN - 1) / TILE::BN;
    if (a.gm == 0) a.gm = group_depth(TILE::BM, TILE::BN, a.tiles_m, a.tiles_n);
    const int64_t nt = (int64_t)a.tiles_m * a.tiles_n;
    if (nt > 0x7fffffff) return fail(DAXQ_ERR_ARG, "gemm: too many tiles");
    launch_kernel(kern, dim3((unsigned)nt), dim3(TILE::T), TILE::SMEM, st, a);
    return check_launch("gemm_fit");
}

template <class TILE, bool FP8, int F8>
static int launch_fit_out(const GemmArgs* a, int out_kind, hipStream_t st) {
    if (out_kind == DAXQ_F16) return launch_fit_one<TILE, FP8, F8, DAXQ_F16>(a, st);
    if (out_kind == DAXQ_F32) return launch_fit_one<TILE, FP8, F8, DAXQ_F32>(a, st);
    return launch_fit_one<TILE, FP8, F8, DAXQ_BF16>(a, st);
}

#ifdef DAXQ_FIT_FP8
template <class TILE>
static int launch_fit_fmt(const GemmArgs* a, int f8, int out_kind, hipStream_t st) {
    switch (f8) {
        case 1: return launch_fit_out<TILE, true, 1>(a, out_kind, st);
        case 2: return launch_fit_out<TILE, true, 2>(a, out_kind, st);
        case 3: return launch_fit_out<TILE, true, 3>(a, out_kind, st);
        default: return launch_fit_out<TILE, true, 0>(a, out_kind, st);
    }
}
#else
template <class TILE>
static int launch_fit_fmt(const GemmArgs* a, int, int out_kind, hipStream_t st) {
    return launch_fit_out<TILE, false, 0>(a, out_kind, st);
}
#endif

static int launch_fit_tile(const GemmArgs* a, int tile, int f8, int out_kind, hipStream_t st) {
    switch (tile) {  // (the order of kFitTiles)
        case 0: return launch_fit_fmt<T64x64>(a, f8, out_kind, st);
        case 1: return launch_fit_fmt<T64x96>(a, f8, out_kind, st);
        case 2: return launch_fit_fmt<T64x128>(a, f8, out_kind, st);
        case 3: return launch_fit_fmt<T64x192>(a, f8, out_kind, st);
        case 4: return launch_fit_fmt<T128x96>(a, f8, out_kind, st);
        case 5: return launch_fit_fmt<T128x160>(a, f8, out_kind, st);
        case 6: return launch_fit_fmt<T128x224>(a, f8, out_kind, st);
        case 7: return launch_fit_fmt<T192x192>(a, f8, out_kind, st);
        case 8: return launch_fit_fmt<T256x96>(a, f8, out_kind, st);
        case 9: return launch_fit_fmt<T256x128>(a, f8, out_kind, st);
        case 10: return launch_fit_fmt<T256x160>(a, f8, out_kind, st);
        default: return fail(DAXQ_ERR_ARG, "linear: unknown fitted tile %d", tile);
    }
}

// (32-bit row offsets as in the other tiled kernels: the caller has checked the row strides)
#ifdef DAXQ_FIT_FP8
int launch_fit_fp8(const GemmArgs& a, int tile, int f8, hipStream_t st) { return launch_fit_tile(&a, tile, f8, a.out_kind, st); }
#else
int launch_fit_i8(const GemmArgs& a, int tile, hipStream_t st) { return launch_fit_tile(&a, tile, 0, a.out_kind, st); }

struct FitShape {
    int bm, bn, per_cu;
};
template <class TILE>
static constexpr FitShape fit_shape() {
    return {TILE::BM, TILE::BN, 2 * TILE::SMEM <= 160 * 1024 ? 2 : 1};
}
static constexpr FitShape kFitTiles[kFitCount] = {fit_shape<T64x64>(),   fit_shape<T64x96>(),   fit_shape<T64x128>(), fit_shape<T64x192>(),
                                         fit_shape<T128x96>(),  fit_shape<T128x160>(), fit_shape<T128x224>(), fit_shape<T192x192>(),
                                         fit_shape<T256x96>(),  fit_shape<T256x128>(), fit_shape<T256x160>()};

// us that a CU takes for `per_cu` tiles at once: their loads or their MFMAs, whichever are longer, and what does not overlap with
// either (fill, epilogue: in proportion to the outputs of a lane; a second workgroup hides three quarters of its own)
static inline __attribute__((always_inline)) double tile_us(int bm, int bn, double pairs, int64_t per_cu) {
    const double load = (bm + bn) * 128.0 / 1024.0 / 105.0, mfma = (double)bm * bn / (128.0 * 128.0) * 512.0 / 2350.0 / 0.9;
    return (double)per_cu * pairs * (load > mfma ? load : mfma) + (0.3 + 1.4 * bm * bn / 8192.0) * (1.0 + 0.25 * (double)(per_cu - 1));
}

// Which fitted tile a launch takes, or -1: the one with the least estimated time whose tiles run in one round (two workgroups per CU
// where the tile leaves room for them), if that is less than the estimate of what the launch takes otherwise (256x256 tiles with
// their cut last round, 128x128 tiles at two per CU).  The constants of the estimate (105 KB per us, 0.9 of the MFMA rate at 2.35 GHz,
// 0.3 us and 1.4 us per 8192 outputs, a quarter of them for a second workgroup) rank the tiles, they do not give their times (1.05
// to 1.8 of the estimate).  Every kernel timed at 140 shapes of 64 to 9000 rows, INT8 and e4m3: where this choice is a fitted tile it is
// 0.2 % slower than the fastest kernel on (geometric) average and within 5 % of it at all but 4 of 203 launches (weights out of reach of
// the caches: 0.3 %, 6).
// Several rounds of fitted tiles are not asked.  Most lose to 256x256 tiles, full rounds as well; us, 256x256 / 256 x 160 / 256 x 128, INT8:
//   4096 x 5120 x 5120 (2.0 rounds of 256 x 160) 82.6 / 83.3 / 99.5    6144 x 5120 x 5120 (3.0) 115.6 / 122.8 / 135.8
//   8192 x 5120 x 5120 (4.0) 154.1 / 163.4 / 174.2                     2299 x 9056, K = 2048 (2.0) 42.8 / 52.7 / 47.1
//   4725 x 5120 x 5120 (2.4; 3.0 of 256 x 128) 95.0 / 112.6 / 106.0    6144 x 4096, K = 5120 (2.4; 3.0 of 256 x 128) 95.4 / 112.1 / 105.3
// Only at most two rounds of 256 x 160 at long K gain a little: 3584 x 5120 x 5120 (1.75) 80.0 / 78.2, 4096 x 5120, K = 13824 (2.0) 215.7 / 208.8.
// FP8 with fewer than 128 columns keeps the generic kernel, which adds in another order, at any number of rows.
int fit_choice(int64_t m, int64_t n, int64_t k, bool fp8) {
    const int cus = cu_count();
    if (m < 64 || n < (fp8 ? 128 : 64) || cus < 8) return -1;
    if (m > 1 << 20 || n > 1 << 20 || m * n > (int64_t)cus * 256 * 160) return -1;  // more outputs than a round of the largest tile
    const double pairs = (double)(k / 128);
    // (every forward comes by here, some of them twice: constant tile sizes and 32 bits instead of divisions by variables, 73 -> 31 ns)
    const uint32_t mu = (uint32_t)m, nu = (uint32_t)n;
    auto tiles = [&](uint32_t bm, uint32_t bn) __attribute__((always_inline)) { return (int64_t)((mu + bm - 1) / bm) * ((nu + bn - 1) / bn); };
    int best = -1;
    double us = 0.0;
#pragma unroll
    for (int i = 0; i < kFitCount; ++i) {
        constexpr const FitShape(&table)[kFitCount] = kFitTiles;
        const FitShape f = table[i];
        if (m < f.bm || n < f.bn) continue;
        const int64_t count = tiles(f.bm, f.bn);
        if (count > (int64_t)f.per_cu * cus) continue;
        const double t = tile_us(f.bm, f.bn, pairs, count > cus ? 2 : 1);
        if (best < 0 || t < us) best = i, us = t;
    }
    if (best < 0 || m < 128 || n < 128) return best;
    const int64_t t256 = tiles(256, 256), t128 = tiles(128, 128);
    double other;
    if (m >= 256 && n >= 256 && t256 >= cus / 2 && t128 > 2 * cus) {
        const int64_t whole = t256 / cus, left = t256 - whole * cus;
        const double last = left == 0 ? 0.0 : whole && 4 * left <= cus ? 0.5 : whole && 2 * left <= cus ? 0.66 : 1.0;
        other = ((double)whole + last) * tile_us(256, 256, pairs, 1);
    } else {
        const int64_t whole = t128 / (2 * cus), left = t128 - whole * 2 * cus;
        other = (double)whole * tile_us(128, 128, pairs, 2) + (left == 0 ? 0.0 : tile_us(128, 128, pairs, left > cus ? 2 : 1));
    }
    return us < other ? best : -1;
}
#endif

// every instantiation on the current device, so that a first launch may sit inside a stream capture
#ifdef DAXQ_FIT_FP8
int prepare_fit_fp8_kernels() {
    constexpr int kFormats = 4;
#else
int prepare_fit_i8_kernels() {
    constexpr int kFormats = 1;
#endif
    int rc = 0;
    for (int tile = 0; tile < kFitCount && !rc; ++tile)
        for (int f8 = 0; f8 < kFormats && !rc; ++f8)
            for (int out_kind : {DAXQ_BF16, DAXQ_F16, DAXQ_F32})
                if (!rc) rc = launch_fit_tile(nullptr, tile, f8, out_kind, nullptr);
    return rc;
}

}  // namespace daxq
