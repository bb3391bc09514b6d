// DIA SpMV on gfx950: y = A x with A, x, y resident in HBM.
//
// Reference: spmv_single_diag_kernel / spmv_row_kernel / spmv_device (src/spMV_gpu.cu:17-168), spmv_host_vectors
// (:171-183), spMV_ntimes_cuda (src/spMV_ntimes_gpu.cu:61-263).
//
// Two kernels serve every diagonal count (the reference's one-diagonal kernel gives the same values: y is zero except
// on the rows of the lone diagonal): row tiles for large matrices, and the wave form (spmv_wave_kernel) for matrices of
// fewer than 1.8 10^6 rows (2^20 in FP32) and for every product that skips zero blocks (sched_for). In the row tiles a
// workgroup owns a tile of 256*RPT consecutive rows; lane l of the tile
// handles rows tile + l + 256*j. For each diagonal (a uniform loop, metadata through scalar loads) the wave reads 64
// consecutive values of the diagonal (one aligned 512-byte FP64 segment, row-aligned layout) and 64 consecutive
// values of the shifted x window, so every access is a full, coalesced line. Each row sums its diagonals in slot
// order in registers and y is written once: A is read once, y written once, and x is read once per diagonal (the
// compulsory bytes count it once; re-reads hit L2 or the Infinity Cache when the windows are near each other).
//
// Column bands: with n_bands > 1 the kernel runs once per band of columns [c0, c1), each pass adding only the
// elements whose column lies in the band (the first pass writes y, later passes add to it). A pass touches only
// 1/n_bands of x, so its x lines stay in the 256 MB Infinity Cache between the diagonals that share them, at the cost
// of one read and one write of y per extra pass.
//
// LDS x window: with lds on, each workgroup stages x[tile - TILE/2, tile + 3 TILE/2) in LDS and the diagonals with
// |offset| <= TILE/2 read x from there (bands, qubit Hamiltonians); scattered offsets gain nothing from it. The
// per-matrix tuner picks it with the other schedule choices.
//
// FP32: values and vectors are float; each row's diagonal sum is Kahan-compensated in FP32.
#include <algorithm>
#include <cstdlib>
#include <mutex>

#include "dia_rows.hpp"

namespace dq {

// Process-wide tuning knobs (set through dq_set_tuning).
static int g_spmv_rpt = 0;    // rows per lane; 0 = automatic
static int g_spmv_bands = 0;  // column bands; 0 = automatic
static int g_spmv_nt = -1;    // non-temporal matrix loads: -1 = automatic, 0 = off, 1 = on
static int g_spmv_pipe = -1;  // load schedule: -1 = automatic, 0 = per-row predicated, 1 = batched
static int g_spmv_lds = -1;   // LDS x window: -1 = automatic, 0 = off, 1 = on
static int g_spmv_xcd = -1;   // tile order: -1 = automatic, 0 = round-robin over the XCDs, 1 = XCD-contiguous

template <typename T, int RPT, bool NT, bool PIPE, bool LDS>
__global__ __launch_bounds__(256) void spmv_rows_kernel(int64_t rows, int64_t cols, int n,
                                                        const DiagMeta *__restrict__ meta, const T *__restrict__ are,
                                                        const T *__restrict__ aim, const T *__restrict__ xr,
                                                        const T *__restrict__ xi, T *__restrict__ yr,
                                                        T *__restrict__ yi, int64_t col_lo, int64_t col_hi,
                                                        int accumulate, int64_t ntiles, int xcd) {
    constexpr int TILE = 256 * RPT;
    constexpr int HALO = LDS ? TILE / 2 : 0;
    constexpr int W = LDS ? TILE + 2 * HALO : 1;
    __shared__ T sr[W], si[W];
    const int64_t t = tile_of_block(blockIdx.x, ntiles, xcd);
    if (t >= ntiles) return;  // uniform: a surplus workgroup of the XCD-contiguous grid
    const int64_t tile = t * TILE;
    const int64_t tile_end = tile + TILE < rows ? tile + TILE : rows;
    if constexpr (LDS) stage_x_window<T, RPT, HALO>(tile, cols, xr, xi, sr, si);
    Acc<T> ar[RPT], ai[RPT];
    if (accumulate) {
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const int64_t r = tile + threadIdx.x + 256 * j;
            if (r < rows) { ar[j].add(yr[r]); ai[j].add(yi[r]); }
        }
    }
    dia_rows_tile<T, RPT, NT, PIPE, HALO>(tile, tile_end, n, meta, are, aim, xr, xi, col_lo, col_hi, ar, ai, sr, si);
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int64_t r = tile + threadIdx.x + 256 * j;
        if (r < rows) { yr[r] = ar[j].get(); yi[r] = ai[j].get(); }
    }
}

// V rows per lane on dia_rows_wave: waves of 64 V rows, four to a workgroup. ZM: zm is a zero-block map of A whose
// all-zero blocks are skipped: the map dq_spmv_tune keeps in the handle (recomputed when the values are rewritten), a
// product's own, or one that spMV_ntimes makes for a call.
// MK: A has no map, and the product leaves one in `made` (map_by_block_bytes) for the products that follow.
template <typename T, int V, bool NT, bool ZM, bool LDS, bool MK>
__global__ __launch_bounds__(256) void spmv_wave_kernel(int64_t rows, int64_t cols, int n,
                                                        const DiagMeta *__restrict__ meta, const T *__restrict__ are,
                                                        const T *__restrict__ aim, const T *__restrict__ xr,
                                                        const T *__restrict__ xi, T *__restrict__ yr,
                                                        T *__restrict__ yi, int64_t col_lo, int64_t col_hi,
                                                        int accumulate, int64_t ntiles, int xcd, ZeroMap zm,
                                                        ulonglong2 *__restrict__ made) {
    constexpr int H = LDS ? 128 * V : 0;
    __shared__ T sr[LDS ? 256 * V + 2 * H : 1], si[LDS ? 256 * V + 2 * H : 1];
    const int64_t t = tile_of_block(blockIdx.x, ntiles, xcd);
    if (t >= ntiles) return;  // uniform
    if constexpr (LDS) stage_x_window<T, V, H>(t * 256 * V, cols, xr, xi, sr, si);
    const int64_t row0 = wave_row0<V>(t);
    if (row0 >= rows) return;  // uniform
    const int64_t r = row0 + V * (threadIdx.x & 63);
    Acc<T> ar[V], ai[V];
    if (accumulate) {
        T br[V], bi[V];
        ld_rows(yr, r, rows, br);
        ld_rows(yi, r, rows, bi);
#pragma unroll
        for (int v = 0; v < V; ++v) {
            ar[v].add(br[v]);
            ai[v].add(bi[v]);
        }
    }
    dia_rows_wave<T, V, NT, ZM, H, MK>(row0, n, meta, are, aim, xr, xi, col_lo, col_hi, ar, ai, zm, sr, si, made, rows);
    T outr[V], outi[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        outr[v] = ar[v].get();
        outi[v] = ai[v].get();
    }
    st_rows(yr, r, rows, outr);
    st_rows(yi, r, rows, outi);
}

// A complete SpMV schedule: rpt = 1 is the wave form (pipe and lds do not apply to it), 2 to 16 the row tiles.
struct SpmvSched {
    int rpt;
    bool nt, pipe, lds;
    int xcd;
    int v = 1;
};

template <typename T>
static void launch_rows(const dq_devmat &A, const T *xr, const T *xi, T *yr, T *yi, const SpmvSched &c, int64_t c0,
                        int64_t c1, int accumulate, hipStream_t s, const ZeroMap &zm, ulonglong2 *made) {
    const int64_t rows = A.rows, cols = A.cols;
    const DiagMeta *meta = A.d_meta.as<DiagMeta>();
    const T *are = static_cast<const T *>(A.re.p), *aim = static_cast<const T *>(A.im.p);
    const int64_t ntiles = (rows + 256 * c.rpt - 1) / (256 * c.rpt);
    const int64_t grid = grid_for_tiles(ntiles, c.xcd);
    if (grid > 0x7fffffffLL) throw ArgError("spmv: too many rows");
    const dim3 g(static_cast<unsigned>(grid));
    if (c.rpt == 1) {
        const int64_t wtiles = (rows + 256 * c.v - 1) / (256 * c.v);
        const dim3 wg(static_cast<unsigned>(grid_for_tiles(wtiles, c.xcd)));
#define DQ_SPMV_WAVE_V(V, NT, Z, L, MK)                                                                              \
    hipLaunchKernelGGL((spmv_wave_kernel<T, V, NT, Z, L, MK>), wg, dim3(256), 0, s, rows, cols, A.n(), meta, are, aim, \
                       xr, xi, yr, yi, c0, c1, accumulate, wtiles, c.xcd, zm, made)
#define DQ_SPMV_WAVE(NT, Z, MK)                                        \
    do {                                                               \
        if (c.v == 2 && c.lds) DQ_SPMV_WAVE_V(2, NT, Z, true, MK);     \
        else if (c.v == 2) DQ_SPMV_WAVE_V(2, NT, Z, false, MK);        \
        else DQ_SPMV_WAVE_V(1, NT, Z, false, MK);                      \
    } while (0)
        if (made && c.nt) DQ_SPMV_WAVE(true, false, true);
        else if (made) DQ_SPMV_WAVE(false, false, true);
        else if (c.nt && zm.any()) DQ_SPMV_WAVE(true, true, false);
        else if (c.nt) DQ_SPMV_WAVE(true, false, false);
        else if (zm.any()) DQ_SPMV_WAVE(false, true, false);
        else DQ_SPMV_WAVE(false, false, false);
#undef DQ_SPMV_WAVE
#undef DQ_SPMV_WAVE_V
        DQ_LAUNCH_CHECK();
        return;
    }
#define DQ_SPMV_LAUNCH(R, NT, PIPE, LDS)                                                                             \
    hipLaunchKernelGGL((spmv_rows_kernel<T, R, NT, PIPE, LDS>), g, dim3(256), 0, s, rows, cols, A.n(), meta, are, aim, \
                       xr, xi, yr, yi, c0, c1, accumulate, ntiles, c.xcd)
#define DQ_SPMV_SCHED(R, LDS)                                           \
    if (c.nt && c.pipe) DQ_SPMV_LAUNCH(R, true, true, LDS);             \
    else if (c.nt) DQ_SPMV_LAUNCH(R, true, false, LDS);                 \
    else if (c.pipe) DQ_SPMV_LAUNCH(R, false, true, LDS);               \
    else DQ_SPMV_LAUNCH(R, false, false, LDS);
#define DQ_SPMV_CASE(R)                                         \
    case R:                                                     \
        if (c.lds) { DQ_SPMV_SCHED(R, true) }                   \
        else { DQ_SPMV_SCHED(R, false) }                        \
        break;
    switch (c.rpt) {
        DQ_SPMV_CASE(2)
        DQ_SPMV_CASE(4)
        DQ_SPMV_CASE(8)
        DQ_SPMV_CASE(16)
        default: throw ArgError("spmv: rows per lane must be 1, 2, 4, 8 or 16");
    }
#undef DQ_SPMV_LAUNCH
#undef DQ_SPMV_SCHED
#undef DQ_SPMV_CASE
    DQ_LAUNCH_CHECK();
}

template <typename T>
__global__ void zero2_kernel(int64_t n, T *__restrict__ a, T *__restrict__ b) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        a[i] = T(0);
        b[i] = T(0);
    }
}

static int auto_bands(const dq_devmat &A) {
    if (g_spmv_bands > 0) return g_spmv_bands;
    return 1;
}

static int auto_rpt(const dq_devmat &A) {
    if (g_spmv_rpt > 0) return g_spmv_rpt;
    if (A.tuned_rpt > 0) return A.tuned_rpt;
    return 8;
}

static bool auto_nt(const dq_devmat &A) {
    if (g_spmv_nt >= 0) return g_spmv_nt == 1;
    if (A.tuned_nt >= 0) return A.tuned_nt == 1;
    return true;
}

static bool auto_pipe(const dq_devmat &A) {
    if (g_spmv_pipe >= 0) return g_spmv_pipe == 1;
    if (A.tuned_pipe >= 0) return A.tuned_pipe == 1;
    return true;
}

// Untuned default for the LDS window: on when at least two off-diagonals lie within the halo of a tile.
bool lds_window_pays(const dq_devmat &A, int rpt) {
    const int halo = 256 * rpt / 2;
    int near = 0;
    for (int32_t d : A.offs)
        if (d != 0 && d >= -halo && d <= halo) ++near;
    return near >= 2;
}

int xcd_tiles_for(const dq_devmat &A) {
    if (g_spmv_xcd >= 0) return g_spmv_xcd;
    if (A.tuned_xcd >= 0) return A.tuned_xcd;
    // untuned: XCD-contiguous when an XCD's eighth of x fits its 4 MB L2 and some diagonals are near each other
    const int64_t x_bytes = static_cast<int64_t>(A.cols) * 2 * elem_bytes(A.precision);
    return (x_bytes / 8 <= (int64_t(4) << 20) && lds_window_pays(A, 8)) ? 1 : 0;
}

bool lds_window_for(const dq_devmat &A, int rpt) {
    if (g_spmv_lds >= 0) return g_spmv_lds == 1;
    if (A.tuned_lds >= 0) return A.tuned_lds == 1;
    return lds_window_pays(A, rpt);
}

// The untuned schedule for reading A's values from memory once per product. The wave form for matrices of few rows, where
// a 2048-row tile leaves CUs idle or with one wave per SIMD, and each row tile pays a chain of dependent loads per
// diagonal (TFIM-12: 24 -> 6 us; 100003 rows x 33 random diagonals: 46 -> 12 us; 2^18 rows, TFIM: 48 -> 27 us). The line,
// us, tiles / wave form, 33 diagonals side by side and at random: FP64 2^20 rows 89 / 90 and 101 / 97, 1.5 10^6 140 / 135
// and 146 / 143, 2^21 184 / 190 and 196 / 204, 4 10^6 755 / 781 random; FP32 700 000 rows 54 / 31 and 49 / 31, 2^20 50 / 57
// and 55 / 54 (TFIM-20 63 / 69), 1.5 10^6 67 / 85 and 75 / 75, 2^21 96 / 113 and 99 / 99. Two rows per lane
// (16-byte loads) from 2^18 rows in FP64, where bytes count more than latency (2^18: equal; 2^20, TFIM: 151 -> 124 us
// with the LDS window); in FP32 one row per lane (a band of 10^6 rows: 44 us against 55). With a map (fewer values to
// read) the wave form at any size, FP32 with two rows per lane from 2^21 rows (TFIM-22: 2.00 -> 1.75 ms for 8
// products). Non-temporal loads when the values exceed the Infinity Cache's 256 MiB (TFIM-18, 155 MB: 27 us plain, 34
// non-temporal; TFIM-22: 613 and 567); with a map from 640 MiB stored, as about a third of it is live in a real
// Hamiltonian.
constexpr int64_t WAVE_ROWS_F64 = int64_t(7) << 18, WAVE_ROWS_F32 = int64_t(1) << 20;
constexpr int64_t WAVE2_ROWS_F64 = int64_t(1) << 18, WAVE2_ROWS_F32 = int64_t(1) << 21;

static SpmvSched wave_default(const dq_devmat &A, bool map) {
    const bool f64 = A.precision == DQ_F64;
    const int64_t bytes = 2 * A.total * elem_bytes(A.precision);
    SpmvSched c{1, false, false, false, 0};
    c.v = A.rows >= (f64 ? WAVE2_ROWS_F64 : WAVE2_ROWS_F32) ? 2 : 1;
    c.lds = f64 && lds_window_pays(A, 2);
    c.nt = bytes > (int64_t(map ? 640 : 256) << 20);
    return c;
}

static SpmvSched sched_for(const dq_devmat &A, bool map) {
    SpmvSched c{8, true, true, false, 0};
    const dq_devmat::WaveSched &w = map ? A.skip_wave : A.tuned_wave;
    const bool few_rows = A.rows < (A.precision == DQ_F64 ? WAVE_ROWS_F64 : WAVE_ROWS_F32);
    const bool wave = map || (g_spmv_rpt > 0 ? g_spmv_rpt == 1 : A.tuned_rpt > 0 ? w.v > 0 : few_rows);
    if (wave) {
        c = wave_default(A, map);
        if (w.v > 0) {
            c.v = w.v;
            c.nt = w.nt;
            c.lds = w.lds;
        }
        if (g_spmv_nt >= 0) c.nt = g_spmv_nt == 1;
        if (g_spmv_lds >= 0) c.lds = g_spmv_lds == 1;
    } else {
        c.rpt = auto_rpt(A);
        c.nt = auto_nt(A);
        c.pipe = auto_pipe(A);
        c.lds = lds_window_for(A, c.rpt);
    }
    c.xcd = xcd_tiles_for(A);
    return c;
}

// y = A x in n_bands column passes (0: automatic), skipping A's all-zero blocks when zm has a map. The schedule is
// `force` if given, else the process-wide knobs, else A's tuned choice, else the defaults. made: the product, in one
// pass, leaves a map by block there.
void spmv_banded(const dq_devmat &A, const void *xr, const void *xi, void *yr, void *yi, int n_bands,
                 hipStream_t s, const ZeroMap &zm = ZeroMap(), const SpmvSched *force = nullptr,
                 ulonglong2 *made = nullptr) {
    if (A.rows == 0) return;
    if (A.n() == 0) {  // no diagonals: y = 0 (a fill kernel, safe inside graph capture)
        const unsigned g = blocks_for(A.rows, 256, 4096);
        if (A.precision == DQ_F64)
            hipLaunchKernelGGL(zero2_kernel<double>, dim3(g), dim3(256), 0, s, (int64_t)A.rows, (double *)yr,
                               (double *)yi);
        else
            hipLaunchKernelGGL(zero2_kernel<float>, dim3(g), dim3(256), 0, s, (int64_t)A.rows, (float *)yr,
                               (float *)yi);
        DQ_LAUNCH_CHECK();
        return;
    }
    if (n_bands <= 0) n_bands = auto_bands(A);
    if (n_bands > static_cast<int>(A.cols)) n_bands = std::max<int>(1, A.cols);
    const SpmvSched c = force ? *force : sched_for(A, zm.any() || made);
    const int64_t cols = A.cols;
    for (int b = 0; b < n_bands; ++b) {
        const int64_t c0 = cols * b / n_bands, c1 = cols * (b + 1) / n_bands;
        if (A.precision == DQ_F64)
            launch_rows<double>(A, (const double *)xr, (const double *)xi, (double *)yr, (double *)yi, c, c0, c1, b > 0,
                                s, zm, made);
        else
            launch_rows<float>(A, (const float *)xr, (const float *)xi, (float *)yr, (float *)yi, c, c0, c1, b > 0, s,
                               zm, made);
    }
}

constexpr int64_t NOALLOC_SCRATCH_WORDS = int64_t(1) << 22;  // see `scratch` below

static int g_spmv_skip = 1;  // "spmv_skip_zero_blocks"

// Whether a sequence of n SpMVs on A's values should make its own zero-block map: not for a single product (the map
// would cost about as much as the product saves), not below 2^16 rows (a product is then a launch and a few round
// trips, and the map's look-up costs it more than the skipped loads), not when the handle already holds a valid one,
// nor with the skip switched off.
static bool ntimes_uses_map(const dq_devmat &A, int n) {
    return g_spmv_skip && n >= 2 && A.n() > 0 && A.rows >= (1u << 16) && !A.zmap_valid;
}

// The launches of a sequence of n products: several products each for a band matrix (band_powers_launches), else one.
// At 1000 to 6 10^6 rows and 3 to 40 diagonals 2 products take 0.35 to 0.93 and 5 products 0.17 to 0.62 of a launch each.
// Not where the tuner found that skipping A's zero blocks pays, nor under a process-wide schedule, nor for a matrix whose
// map would not fit the allocation-free form's scratch (that form refuses the call).
static int sequence_launches(const dq_devmat &A, int n) {
    const bool forced = g_spmv_rpt > 0 || g_spmv_bands > 0 || g_spmv_nt >= 0 || g_spmv_pipe >= 0 || g_spmv_lds >= 0 ||
                        g_spmv_xcd >= 0 || !g_spmv_skip;
    if (forced || A.zmap_valid || zero_map_bytes(A, 8) > sizeof(uint2) * NOALLOC_SCRATCH_WORDS) return n;
    return band_powers_launches(A, n);
}

// The products of launch i.
static int sequence_products(int n, int launches, int i) {
    return static_cast<int>(int64_t(n) * (i + 1) / launches - int64_t(n) * i / launches);
}

// The map a product with A may use without making one: the handle's, for FP64 matrices. (In FP64 a skipped block
// changes no bit; a compensated FP32 sum would change in its last bits, and a single FP32 SpMV keeps the same bits
// whether or not A was tuned.)
static ZeroMap handle_map(const dq_devmat &A) {
    return g_spmv_skip && A.precision == DQ_F64 ? kept_zero_map(A) : ZeroMap();
}

// The handle's map for a sequence of n products: a single product follows handle_map; two or more use the map in
// any precision (their results are not compared with a single untuned SpMV's).
static ZeroMap sequence_map(const dq_devmat &A, int n) {
    if (n == 1) return handle_map(A);
    ZeroMap z = g_spmv_skip ? kept_zero_map(A) : ZeroMap();
    z.loads_only = 0;
    return z;
}

ZeroMap kept_zero_map(const dq_devmat &A) {
    ZeroMap z;
    if (!A.zmap_valid || !A.zmap.p) return z;
    z.w = A.zmap.as<uint2>();
    z.words = zero_block_words(A.rows, 1 << z.shift);
    z.loads_only = A.zmap_loads_only;
    return z;
}

size_t zero_map_bytes(const dq_devmat &A, int shift) {
    return sizeof(uint2) * static_cast<size_t>(zero_block_words(A.rows, 1 << shift)) * static_cast<size_t>(A.n());
}

// Whether the map z of A shows a block, inside some diagonal's rows, whose real or imaginary values are all zero.
static bool has_zero_blocks(const dq_devmat &A, const ZeroMap &z, hipStream_t s) {
    std::vector<uint2> h(static_cast<size_t>(z.words) * A.n());
    DQ_HIP(hipMemcpyAsync(h.data(), z.w, h.size() * sizeof(uint2), hipMemcpyDeviceToHost, s));
    DQ_HIP(hipStreamSynchronize(s));
    for (int k = 0; k < A.n(); ++k) {
        const DiagMeta &m = A.meta[k];
        if (m.rhi <= m.rlo) continue;
        for (int64_t b = m.rlo >> z.shift; b <= (m.rhi - 1) >> z.shift; ++b) {
            const uint2 w = h[static_cast<size_t>(k) * z.words + (b >> 5)];
            if (!((w.x & w.y) >> (b & 31) & 1u)) return true;
        }
    }
    return false;
}

void make_zero_map(const dq_devmat &A, int shift, uint2 *w, hipStream_t s) {
    make_zero_map(A, A.d_meta.as<DiagMeta>(), shift, w, s);
}

void make_zero_map(const dq_devmat &A, const DiagMeta *meta, int shift, uint2 *w, hipStream_t s) {
    const int64_t words = zero_block_words(A.rows, 1 << shift);
    const dim3 grid(static_cast<unsigned>(words), zero_map_grid_y(A.n()), 1);
#define DQ_ZERO_MAP(T, BR)                                                                                          \
    hipLaunchKernelGGL((zero_blocks_kernel<T, BR>), grid, dim3(256), 0, s, static_cast<int64_t>(A.rows), A.n(), meta, \
                       int64_t(0), A.re.as<T>(), A.im.as<T>(), words, w)
    if (A.precision == DQ_F64 && shift == 6) DQ_ZERO_MAP(double, 64);
    else if (A.precision == DQ_F64) DQ_ZERO_MAP(double, 256);
    else if (shift == 6) DQ_ZERO_MAP(float, 64);
    else DQ_ZERO_MAP(float, 256);
#undef DQ_ZERO_MAP
    DQ_LAUNCH_CHECK();
}

__global__ void fill_map_kernel(int64_t n, uint2 *__restrict__ w) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        w[i] = make_uint2(~0u, ~0u);
}

// After A's values were rewritten on stream s: bring the zero-block map the handle keeps up to date in the same buffer,
// ordered after the rewrite. A graph captured earlier that reads the handle's map then sees the new map on its next
// replay, and later SpMVs skip no block that is nonzero now. The map of a tuning is recomputed; a product's map, which
// the caller did not ask for, is set to "every block nonzero" for those graphs instead of reading all values again, and the
// handle has none from then on: a sequence makes its own.
void refresh_zero_map(dq_devmat &A, hipStream_t s) {
    if (!A.zmap_valid || !A.zmap.p) return;
    if (!A.zmap_loads_only) {
        make_zero_map(A, ZeroMap().shift, A.zmap.as<uint2>(), s);
        return;
    }
    const int64_t n = static_cast<int64_t>(A.zmap.bytes / sizeof(uint2));
    hipLaunchKernelGGL(fill_map_kernel, dim3(blocks_for(n, 256, 2048)), dim3(256), 0, s, n, A.zmap.as<uint2>());
    DQ_LAUNCH_CHECK();
    A.zmap_valid = A.zmap_loads_only = false;
}

// y = A x: the schedule of A, skipping its all-zero blocks when the handle holds their map (see handle_map).
void spmv(const dq_devmat &A, const void *xr, const void *xi, void *yr, void *yi, hipStream_t s) {
    spmv_banded(A, xr, xi, yr, yi, 0, s, handle_map(A));
}

}  // namespace dq

using namespace dq;

extern "C" int dq_set_tuning(const char *key, int value) {
    return guard([&] {
        if (!key) throw ArgError("key is NULL");
        const std::string k(key);
        if (k == "spmv_rows_per_lane") {
            if (value != 0 && value != 1 && value != 2 && value != 4 && value != 8 && value != 16)
                throw ArgError("spmv_rows_per_lane must be 0, 1, 2, 4, 8 or 16");
            g_spmv_rpt = value;
        } else if (k == "spmv_nontemporal") {
            if (value < -1 || value > 1) throw ArgError("spmv_nontemporal must be -1, 0 or 1");
            g_spmv_nt = value;
        } else if (k == "spmv_pipelined") {
            if (value < -1 || value > 1) throw ArgError("spmv_pipelined must be -1, 0 or 1");
            g_spmv_pipe = value;
        } else if (k == "spmv_lds") {
            if (value < -1 || value > 1) throw ArgError("spmv_lds must be -1, 0 or 1");
            g_spmv_lds = value;
        } else if (k == "spmv_xcd") {
            if (value < -1 || value > 1) throw ArgError("spmv_xcd must be -1, 0 or 1");
            g_spmv_xcd = value;
        } else if (k == "spmv_bands") {
            if (value < 0 || value > 4096) throw ArgError("spmv_bands must be in [0, 4096]");
            g_spmv_bands = value;
        } else if (k == "alloc_cache_mb") {
            if (value < -1) throw ArgError("alloc_cache_mb must be -1 (an eighth of the device memory) or >= 0");
            set_alloc_cache_budget(value);
        } else if (k == "spmv_skip_zero_blocks") {
            if (value != 0 && value != 1) throw ArgError("spmv_skip_zero_blocks must be 0 or 1");
            g_spmv_skip = value;
        } else if (!product_set_tuning(k, value) && !evo_set_tuning(k, value) && !spmm_set_tuning(k, value) &&
                   !dense_set_tuning(k, value) && !convert_set_tuning(k, value) && !gates_set_tuning(k, value) &&
                   !hamsim_set_tuning(k, value)) {
            throw ArgError("unknown tuning key: " + k);
        }
    });
}

// Time every (load schedule, rows per lane, non-temporal, LDS window) candidate on scratch vectors and keep the fastest
// in the matrix handle; later SpMVs with this matrix use it (unless a process-wide knob overrides it). The LDS window
// is only tried when some off-diagonal lies within its halo. The candidates are passed to the kernels explicitly, so
// SpMVs of other matrices meanwhile keep their own schedules; calls with this matrix must not overlap its tuning
// (the handle's schedule and zero-block map change during it).
extern "C" int dq_spmv_tune(dq_devmat *A, int repeats, uintptr_t stream, float *best_ms) {
    return guard([&] {
        if (!A) throw ArgError("matrix is NULL");
        if (repeats <= 0) repeats = 3;
        hipStream_t s = as_stream(stream);
        if (A->rows == 0 || A->n() == 0) return;
        const size_t eb = elem_bytes(A->precision);
        DevBuf xr(A->cols * eb), xi(A->cols * eb), yr(A->rows * eb), yi(A->rows * eb);
        zero_bytes(xr.p, xr.bytes, s);
        zero_bytes(xi.p, xi.bytes, s);
        hipEvent_t e0, e1;
        DQ_HIP(hipEventCreate(&e0));
        DQ_HIP(hipEventCreate(&e1));
        struct Events {
            hipEvent_t a, b;
            ~Events() { (void)hipEventDestroy(a); (void)hipEventDestroy(b); }
        } ev{e0, e1};
        ZeroMap tz;  // the zero-block map while the skip schedule is timed
        auto time_it = [&](const SpmvSched &c) {
            spmv_banded(*A, xr.p, xi.p, yr.p, yi.p, 1, s, tz, &c);  // warm
            DQ_HIP(hipEventRecord(e0, s));
            for (int r = 0; r < repeats; ++r) spmv_banded(*A, xr.p, xi.p, yr.p, yi.p, 1, s, tz, &c);
            DQ_HIP(hipEventRecord(e1, s));
            DQ_HIP(hipEventSynchronize(e1));
            float ms = 0.f;
            DQ_HIP(hipEventElapsedTime(&ms, e0, e1));
            return ms / repeats;
        };
        float best = 1e30f;
        SpmvSched win{8, true, true, false, 0};
        for (int lds = 0; lds <= 1; ++lds)
            for (int pipe = 0; pipe <= 1; ++pipe)
                for (int rpt : {2, 4, 8, 16})
                    for (int nt = 0; nt <= 1; ++nt) {
                        if (lds && !lds_window_pays(*A, rpt) && !lds_window_pays(*A, 16)) continue;
                        const SpmvSched c{rpt, nt == 1, pipe == 1, lds == 1, 0};
                        const float ms = time_it(c);
                        if (ms < best) { best = ms; win = c; }
                    }
        // second stage: the winner with the XCD-contiguous tile order
        SpmvSched wx = win;
        wx.xcd = 1;
        const float msx = time_it(wx);
        if (msx < best) { best = msx; win = wx; }
        A->tuned_rpt = win.rpt; A->tuned_nt = win.nt; A->tuned_pipe = win.pipe; A->tuned_lds = win.lds;
        A->tuned_xcd = win.xcd;
        // the wave forms, in the same order of tiles
        auto time_waves = [&](float &limit, dq_devmat::WaveSched &to) {
            to = dq_devmat::WaveSched();
            for (int form = 0; form < 3; ++form) {
                if (form == 2 && !lds_window_pays(*A, 2)) continue;
                for (int nt = 0; nt <= 1; ++nt) {
                    SpmvSched c{1, nt == 1, false, form == 2, win.xcd};
                    c.v = form == 0 ? 1 : 2;
                    const float ms = time_it(c);
                    if (ms < limit) {
                        limit = ms;
                        to.v = c.v;
                        to.nt = c.nt;
                        to.lds = c.lds;
                    }
                }
            }
        };
        A->tuned_wave = dq_devmat::WaveSched();
        if (A->rows < (1u << 22)) time_waves(best, A->tuned_wave);  // beyond, the tiles read every block faster
        // last stage: when A has all-zero blocks or parts and skipping them is faster, keep their map in the handle (used
        // by A's FP64 SpMVs and by spMV_ntimes)
        A->zmap_valid = A->zmap_loads_only = false;
        A->skip_wave = dq_devmat::WaveSched();
        if (g_spmv_skip) {
            const size_t zb = zero_map_bytes(*A, tz.shift);
            if (A->zmap.bytes != zb) A->zmap = DevBuf(zb);
            make_zero_map(*A, tz.shift, A->zmap.as<uint2>(), s);
            tz.w = A->zmap.as<uint2>();
            tz.words = zero_block_words(A->rows, 1 << tz.shift);
            if (has_zero_blocks(*A, tz, s)) {
                float zbest = best;
                time_waves(zbest, A->skip_wave);
                A->zmap_valid = A->skip_wave.v > 0;
            }
        }
        if (best_ms) *best_ms = best;
    });
}

extern "C" int dq_spmv_tuned_config(const dq_devmat *A, int *rows_per_lane, int *nontemporal, int *pipelined,
                                    int *lds_window, int *xcd_tiles) {
    return guard([&] {
        if (!A) throw ArgError("matrix is NULL");
        if (rows_per_lane) *rows_per_lane = auto_rpt(*A);
        if (nontemporal) *nontemporal = auto_nt(*A) ? 1 : 0;
        if (pipelined) *pipelined = auto_pipe(*A) ? 1 : 0;
        if (lds_window) *lds_window = lds_window_for(*A, auto_rpt(*A)) ? 1 : 0;
        if (xcd_tiles) *xcd_tiles = xcd_tiles_for(*A);
    });
}

extern "C" int dq_spmv_device(const dq_devmat *A, const void *xr, const void *xi, void *yr, void *yi,
                              uintptr_t stream) {
    return guard([&] {
        if (!A) throw ArgError("matrix is NULL");
        if (A->rows && (!yr || !yi)) throw ArgError("spmv_device: NULL y");
        if (A->n() && (!xr || !xi)) throw ArgError("spmv_device: NULL x");
        spmv(*A, xr, xi, yr, yi, as_stream(stream));
    });
}

extern "C" int dq_spmv_device_banded(const dq_devmat *A, const void *xr, const void *xi, void *yr, void *yi,
                                     int n_bands, uintptr_t stream) {
    return guard([&] {
        if (!A) throw ArgError("matrix is NULL");
        if (n_bands < 0) throw ArgError("n_bands must be >= 0");
        if (A->rows && (!yr || !yi)) throw ArgError("spmv_device: NULL y");
        if (A->n() && (!xr || !xi)) throw ArgError("spmv_device: NULL x");
        spmv_banded(*A, xr, xi, yr, yi, n_bands, as_stream(stream));
    });
}

// Host vectors of doubles through device buffers of the matrix precision.
namespace {
struct DevVec {
    DevBuf r, i;
    int64_t n;
    int prec;
    DevVec(int64_t n_, int prec_) : r(n_ * elem_bytes(prec_)), i(n_ * elem_bytes(prec_)), n(n_), prec(prec_) {}
    void put(const double *hr, const double *hi) {
        if (!n) return;
        if (prec == DQ_F64) {
            DQ_HIP(hipMemcpy(r.p, hr, n * 8, hipMemcpyHostToDevice));
            DQ_HIP(hipMemcpy(i.p, hi, n * 8, hipMemcpyHostToDevice));
        } else {
            std::vector<float> a(hr, hr + n), b(hi, hi + n);
            DQ_HIP(hipMemcpy(r.p, a.data(), n * 4, hipMemcpyHostToDevice));
            DQ_HIP(hipMemcpy(i.p, b.data(), n * 4, hipMemcpyHostToDevice));
        }
    }
    void get(double *hr, double *hi) const {
        if (!n) return;
        if (prec == DQ_F64) {
            DQ_HIP(hipMemcpy(hr, r.p, n * 8, hipMemcpyDeviceToHost));
            DQ_HIP(hipMemcpy(hi, i.p, n * 8, hipMemcpyDeviceToHost));
        } else {
            std::vector<float> a(n), b(n);
            DQ_HIP(hipMemcpy(a.data(), r.p, n * 4, hipMemcpyDeviceToHost));
            DQ_HIP(hipMemcpy(b.data(), i.p, n * 4, hipMemcpyDeviceToHost));
            std::copy(a.begin(), a.end(), hr);
            std::copy(b.begin(), b.end(), hi);
        }
    }
};
}  // namespace

extern "C" int dq_spmv_host(const dq_devmat *A, const double *xr, const double *xi, double *yr, double *yi) {
    return guard([&] {
        if (!A) throw ArgError("matrix is NULL");
        if ((A->cols && (!xr || !xi)) || (A->rows && (!yr || !yi))) throw ArgError("spmv_cuda: NULL vector");
        DevVec x(A->cols, A->precision), y(A->rows, A->precision);
        x.put(xr, xi);
        spmv(*A, x.r.p, x.i.p, y.r.p, y.i.p, 0);
        DQ_LAUNCH_CHECK();
        y.get(yr, yi);
    });
}

// A product of a sequence: with `made`, the first one leaves A's map by block there and the others skip by it. It reads
// every value anyway, and a map from a pass of its own costs as much as a product (10^6 rows, 33 random diagonals, FP64, two
// products: 274 -> 198 us; TFIM-20, five: 418 -> 373).
static void sequence_product(const dq_devmat &A, const void *xr, const void *xi, void *yr, void *yi, hipStream_t s,
                             const ZeroMap &map, ulonglong2 *made, bool first) {
    ZeroMap z = map;
    if (made && !first) {
        z.by_block = made;
        z.words = A.rows;
    }
    spmv_banded(A, xr, xi, yr, yi, 0, s, z, nullptr, first ? made : nullptr);
}

// y = A^n x on device vectors (src/spMV_ntimes_gpu.cu:61-263 on resident data). `fixed_map` (may be null) is
// device memory of fixed_bytes bytes the call may use for A's zero-block map instead of allocating one: the
// allocation-free entry point passes its static scratch array; then the map is made even while the stream is being
// captured (the array outlives every replay), and a map that would not fit is an error.
static void ntimes_device(const dq_devmat *A, const void *xr, const void *xi, void *yr, void *yi, int n, void *work_r,
                          void *work_i, hipStream_t s, uint2 *fixed_map, size_t fixed_bytes) {
    if (!A) throw ArgError("matrix is NULL");
    if (n < 0) throw ArgError("spmv_ntimes_cuda: num_times must be >= 0");
    if (!xr || !xi || !yr || !yi) throw ArgError("spmv_ntimes_device: NULL vector");
    const int64_t M = A->rows, N = A->cols;
    const size_t eb = elem_bytes(A->precision);
    if (n == 0) {
        if (M != N) throw ArgError("spmv_ntimes_cuda: num_times==0 requires square matrix (M==N) to copy x -> y");
        if (xr != yr) DQ_HIP(hipMemcpyAsync(yr, xr, M * eb, hipMemcpyDeviceToDevice, s));
        if (xi != yi) DQ_HIP(hipMemcpyAsync(yi, xi, M * eb, hipMemcpyDeviceToDevice, s));
        return;
    }
    if (A->n() == 0) {  // no diagonals: y = 0 for any num_times >= 1 (src/spMV_ntimes_gpu.cu:98-105)
        spmv_banded(*A, xr, xi, yr, yi, 0, s);
        return;
    }
    if (n > 1 && M != N)
        throw ArgError("spmv_ntimes_cuda: repeated SpMV requires square matrix (M==N) for num_times > 1");
    const bool in_place = xr == yr || xi == yi;
    if (in_place && (xr != yr || xi != yi)) throw ArgError("spmv_ntimes_device: x and y overlap in one part only");
    if ((n > 1 || in_place) && (!work_r || !work_i))
        throw ArgError("spmv_ntimes_device: work vectors are needed for num_times > 1 or x == y");
    // destinations alternate between y and the work vectors so that the last product lands in y; with x == y and an
    // odd count the first product must not overwrite x, so the order flips and a copy ends the sequence
    int launches = sequence_launches(*A, n);
    // x may be the work vector for an odd n: the first product goes to y, and x is not read again. An even number of
    // launches would write over x while it is read.
    if (launches < n && launches % 2 == 0 && (work_r == xr || work_i == xi)) launches = n;
    const bool flip = in_place && (launches % 2 == 1);
    // the zero blocks of A, skipped by every product of the sequence (A cannot change during the call): the map
    // dq_spmv_tune kept in the handle, or else, for two or more products, one made here -- in the caller's fixed
    // memory, or in stream-ordered memory so the call stays asynchronous. Without fixed memory no map is made while
    // the stream is being captured into a graph (a replay must not read memory this call has given back).
    // (Where a map by block fits, the first product leaves it as it goes; else the map is made by a pass of its own.)
    void *stream_mem = nullptr;
    ulonglong2 *made = nullptr;
    ZeroMap z = sequence_map(*A, n);
    if (launches == n && !z.w && ntimes_uses_map(*A, n)) {
        size_t bytes = map_by_block_bytes(M, A->n());
        bool by_block = g_spmv_bands <= 1;
        void *to = nullptr;
        if (fixed_map) {
            by_block = by_block && bytes <= fixed_bytes;
            if (!by_block) {
                bytes = zero_map_bytes(*A, z.shift);
                if (bytes > fixed_bytes) {  // blocks of 256 rows then
                    z.shift = 8;
                    bytes = zero_map_bytes(*A, z.shift);
                }
                if (bytes > fixed_bytes)
                    throw ArgError("spmv_ntimes_device_noalloc: the zero-block map of this matrix needs " +
                                   std::to_string(bytes) + " bytes, more than the " + std::to_string(fixed_bytes) +
                                   " bytes of the library's static scratch (tune the matrix with dq_spmv_tune to keep "
                                   "its map in the handle, or use dq_spmv_ntimes_device)");
            }
            to = fixed_map;
        } else {
            if (!by_block) bytes = zero_map_bytes(*A, z.shift);
            hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
            DQ_HIP(hipStreamIsCapturing(s, &cap));
            if (cap == hipStreamCaptureStatusNone) {
                if (hipMallocAsync(&stream_mem, bytes, s) != hipSuccess) {
                    (void)hipGetLastError();  // no stream-ordered memory: run without the map
                    stream_mem = nullptr;
                }
                to = stream_mem;
            }
        }
        if (to && by_block) {
            made = static_cast<ulonglong2 *>(to);
        } else if (to) {
            make_zero_map(*A, z.shift, static_cast<uint2 *>(to), s);
            z.w = static_cast<uint2 *>(to);
            z.words = zero_block_words(A->rows, 1 << z.shift);
        }
    }
    const void *sr = xr, *si = xi;
    for (int t = 0; t < launches; ++t) {
        const bool to_y = (((launches - 1 - t) % 2) == 0) != flip;
        void *dr = to_y ? yr : work_r, *di = to_y ? yi : work_i;
        if (launches < n) band_powers(*A, sr, si, dr, di, sequence_products(n, launches, t), s);
        else sequence_product(*A, sr, si, dr, di, s, z, made, t == 0);
        sr = dr;
        si = di;
    }
    if (stream_mem) DQ_HIP(hipFreeAsync(stream_mem, s));
    if (flip) {
        DQ_HIP(hipMemcpyAsync(yr, work_r, M * eb, hipMemcpyDeviceToDevice, s));
        DQ_HIP(hipMemcpyAsync(yi, work_i, M * eb, hipMemcpyDeviceToDevice, s));
    }
}

extern "C" int dq_spmv_ntimes_device(const dq_devmat *A, const void *xr, const void *xi, void *yr, void *yi, int n,
                                     void *work_r, void *work_i, uintptr_t stream) {
    return guard([&] { ntimes_device(A, xr, xi, yr, yi, n, work_r, work_i, as_stream(stream), nullptr, 0); });
}

// The allocation-free form's scratch: room for the zero-block map of a sequence (64-row blocks, or 256-row blocks where
// those would not fit; two bits each, for every diagonal), 32 MiB per GPU, held from the library's load until the
// process ends. In host code `scratch` only stands in for the symbol; its device address comes from
// hipGetSymbolAddress, once per device.
static __device__ __align__(256) uint2 scratch[NOALLOC_SCRATCH_WORDS];

constexpr int NOALLOC_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static uint2 *g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};

// This device's copy of `scratch`, looked up on the first call on the device (with that device current).
static uint2 *noalloc_scratch() {
    int dev = 0;
    DQ_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) throw ArgError("spmv_ntimes_device_noalloc: device index out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        DQ_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_ptr[dev] = static_cast<uint2 *>(p);
    }
    return g_scratch_ptr[dev];
}

extern "C" int dq_spmv_ntimes_device_noalloc(const dq_devmat *A, const void *xr, const void *xi, void *yr, void *yi,
                                             int n, void *work_r, void *work_i, uintptr_t stream) {
    return guard([&] {
        ntimes_device(A, xr, xi, yr, yi, n, work_r, work_i, as_stream(stream), noalloc_scratch(),
                      sizeof(uint2) * NOALLOC_SCRATCH_WORDS);
    });
}

extern "C" int dq_spmv_ntimes_host(const dq_devmat *A, const double *xr, const double *xi, double *yr, double *yi,
                                   int n) {
    return guard([&] {
        if (!A) throw ArgError("matrix is NULL");
        if (n < 0) throw ArgError("spmv_ntimes_cuda: num_times must be >= 0");
        const int64_t M = A->rows, N = A->cols;
        if (n == 0) {
            if (M != N)
                throw ArgError("spmv_ntimes_cuda: num_times==0 requires square matrix (M==N) to copy x -> y");
            std::copy(xr, xr + M, yr);
            std::copy(xi, xi + M, yi);
            return;
        }
        if (A->n() == 0) {
            std::fill(yr, yr + M, 0.0);
            std::fill(yi, yi + M, 0.0);
            return;
        }
        if (n > 1 && M != N)
            throw ArgError("spmv_ntimes_cuda: repeated SpMV requires square matrix (M==N) for num_times > 1");
        DevVec a(N, A->precision), b(M, A->precision);
        a.put(xr, xi);
        DevBuf zmap;
        ulonglong2 *made = nullptr;
        ZeroMap z = sequence_map(*A, n);
        const int launches = sequence_launches(*A, n);
        if (launches == n && !z.w && ntimes_uses_map(*A, n)) {
            const bool by_block = g_spmv_bands <= 1;
            zmap = DevBuf(by_block ? map_by_block_bytes(M, A->n()) : zero_map_bytes(*A, z.shift));
            if (by_block) {
                made = zmap.as<ulonglong2>();
            } else {
                make_zero_map(*A, z.shift, zmap.as<uint2>(), 0);
                z.w = zmap.as<uint2>();
                z.words = zero_block_words(A->rows, 1 << z.shift);
            }
        }
        DevVec *in = &a, *out = &b;
        for (int t = 0; t < launches; ++t) {
            if (launches < n) band_powers(*A, in->r.p, in->i.p, out->r.p, out->i.p, sequence_products(n, launches, t), 0);
            else sequence_product(*A, in->r.p, in->i.p, out->r.p, out->i.p, 0, z, made, t == 0);
            if (t != launches - 1) std::swap(in, out);
        }
        out->get(yr, yi);
    });
}
