// y = A^p x for a band matrix, several products per read of A.
//
// Reference: spMV_ntimes_cuda (src/spMV_ntimes_gpu.cu:61-263), one product per pass over A.
//
// When every offset lies in [-hl, hh], rows [r0, r0 + R) of A^p x depend on x and on rows of A within p - 1 halos of
// them. A workgroup takes L = R + (p - 1)(hl + hh) rows, one per lane, loads their values into registers once, the x
// window into LDS, and computes p products: after product s the rows within p - s halos of its R hold A^s x, the
// others hold values that no kept row reads. Every row sums its diagonals in slot order with the operations of
// dia_rows_tile, so the rows have the bits of products that read every block. (A zero block is read like any other: a
// compensated FP32 sum that skips it, as products with a map do, may differ in its last bits.)
//
// Bound: the values' reads, L / (R p) of a pass each, against the sums: a compensated FP32 sum is 16 vector instructions
// per element, 13 us per product of 33 10^6 elements on the whole chip. 512 lanes and, in FP32, at most 128 registers leave
// two workgroups per CU, one loading while the other adds. 10^6 rows, 33 diagonals, FP32, 4 products: 262 -> 112 us.
#include <algorithm>

#include "dia_rows.hpp"

namespace dq {

constexpr int POW_LANES = 512, POW_ND = 40;

template <typename T>
struct alignas(2 * sizeof(T)) Pair {
    T r, i;
};

template <typename T, int ND>
__global__ __launch_bounds__(POW_LANES, (sizeof(T) == 4 || ND <= 16) ? 4 : 2) void band_powers_kernel(
    int64_t N, int n, const DiagMeta *__restrict__ meta, const T *__restrict__ are, const T *__restrict__ aim,
    const T *__restrict__ xr, const T *__restrict__ xi, T *__restrict__ yr, T *__restrict__ yi, int p, int hl, int hh,
    int R, int64_t ntiles) {
    extern __shared__ __align__(16) char smem[];
    Pair<T> *buf = reinterpret_cast<Pair<T> *>(smem);
    const int64_t t = tile_of_block(blockIdx.x, ntiles, 1);
    if (t >= ntiles) return;  // uniform
    const int width = POW_LANES + hl + hh;
    const int64_t r0 = t * R, base = r0 - static_cast<int64_t>(p - 1) * hl;  // base: lane 0's row
    const int64_t row = base + threadIdx.x;
    const bool mine = row >= 0 && row < N;
    T ar[ND], ai[ND];
    int off[ND];  // uniform
#pragma unroll
    for (int k = 0; k < ND; ++k) {
        ar[k] = ai[k] = T(0);
        off[k] = 0;
        if (k < n) {  // uniform
            const DiagMeta md = meta[k];
            off[k] = md.off;
            if (row >= md.rlo && row < md.rhi) {
                ar[k] = are[md.rowbase + row];
                ai[k] = aim[md.rowbase + row];
            }
        }
    }
    for (int e = threadIdx.x; e < width; e += POW_LANES) {  // place e is row base - hl + e; zero outside the matrix
        const int64_t c = base - hl + e;
        const bool in = c >= 0 && c < N;
        buf[e] = Pair<T>{in ? xr[c] : T(0), in ? xi[c] : T(0)};
        buf[width + e] = Pair<T>{T(0), T(0)};
    }
    __syncthreads();
    const bool inside = base - hl >= 0 && base - hl + width <= N;  // uniform: every lane's row has every diagonal
    const int at = static_cast<int>(threadIdx.x) + hl;
    for (int s = 1;; ++s) {
        const Pair<T> *x = buf + (s & 1 ? 0 : width);
        Acc<T> sr, si;
#pragma unroll
        for (int k = 0; k < ND; k += 4)
            if (k < n) {  // uniform
                Pair<T> v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = x[at + off[k + u]];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (k + u < n) {  // uniform
                        // a row off the diagonal adds nothing (not even a zero: a compensated sum is not inert to it)
                        const int64_t c = row + off[k + u];
                        if (inside || (mine && c >= 0 && c < N)) cmac(sr, si, ar[k + u], ai[k + u], v[u].r, v[u].i);
                    }
            }
        if (s == p) {
            const int64_t i = row - r0;
            if (mine && i >= 0 && i < R) {
                yr[row] = sr.get();
                yi[row] = si.get();
            }
            return;  // uniform
        }
        buf[(s & 1 ? width : 0) + at] = mine ? Pair<T>{sr.get(), si.get()} : Pair<T>{T(0), T(0)};
        __syncthreads();
    }
}

// The launches that a sequence of n products with A takes: launch i runs the products from n i / launches on, or, where
// that is at least as good, there are n of one product each. Per product, and against one pass over A, a launch of p products
// reads L / (R p) of A and spends about a quarter of a pass on the sums, for L / R times the rows (FP32, 33 diagonals);
// the split minimises their sum and pays under 0.85 of a pass. Up to POW_ND diagonals, whose values fit the registers.
int band_powers_launches(const dq_devmat &A, int n) {
    int hl = 0, hh = 0;
    for (int32_t o : A.offs) {
        hl = std::max(hl, -o);
        hh = std::max(hh, o);
    }
    const int64_t w = static_cast<int64_t>(hl) + hh;
    if (n < 2 || A.n() == 0 || A.n() > POW_ND || w > POW_LANES / 2) return n;
    int best = 1;
    double cost = 0.85;
    for (int p = 2; p <= n && POW_LANES - (p - 1) * w >= 64; ++p) {
        const double c = POW_LANES * (1.0 / p + 0.25) / static_cast<double>(POW_LANES - (p - 1) * w);
        if (c < cost) {
            cost = c;
            best = p;
        }
    }
    return n / best + (n % best != 0);
}

template <typename T>
static void launch_powers(const dq_devmat &A, const T *xr, const T *xi, T *yr, T *yi, int p, hipStream_t s) {
    int hl = 0, hh = 0;
    for (int32_t o : A.offs) {
        hl = std::max(hl, -o);
        hh = std::max(hh, o);
    }
    const int64_t N = A.rows;
    const int R = POW_LANES - (p - 1) * (hl + hh);
    const int64_t ntiles = (N + R - 1) / R;
    const int64_t grid = grid_for_tiles(ntiles, 1);
    if (grid > 0x7fffffffLL) throw ArgError("spmv: too many rows");
    const size_t lds = 2 * static_cast<size_t>(POW_LANES + hl + hh) * 2 * sizeof(T);
#define DQ_POWERS(ND)                                                                                                \
    hipLaunchKernelGGL((band_powers_kernel<T, ND>), dim3(static_cast<unsigned>(grid)), dim3(POW_LANES), lds, s, N,   \
                       A.n(), A.d_meta.as<DiagMeta>(), A.re.as<T>(), A.im.as<T>(), xr, xi, yr, yi, p, hl, hh, R, ntiles)
    if (A.n() <= 8) DQ_POWERS(8);
    else if (A.n() <= 16) DQ_POWERS(16);
    else if (A.n() <= 24) DQ_POWERS(24);
    else if (A.n() <= 32) DQ_POWERS(32);
    else DQ_POWERS(POW_ND);
#undef DQ_POWERS
    DQ_LAUNCH_CHECK();
}

// y = A^p x, p as band_powers_launches splits; y is neither x nor A's memory.
void band_powers(const dq_devmat &A, const void *xr, const void *xi, void *yr, void *yi, int p, hipStream_t s) {
    if (A.precision == DQ_F64)
        launch_powers<double>(A, (const double *)xr, (const double *)xi, (double *)yr, (double *)yi, p, s);
    else
        launch_powers<float>(A, (const float *)xr, (const float *)xi, (float *)yr, (float *)yi, p, s);
}

}  // namespace dq
