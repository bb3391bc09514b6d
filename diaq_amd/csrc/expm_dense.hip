// The Taylor series of a matrix exponential, row by row of a dense result: U = I + sum_k X^k / k! for a sparse DIA X.
//
// Term k is T_k = T_{k-1} X / k, and row r of T_k depends on row r of T_{k-1} alone. A workgroup takes RB rows, keeps
// their current term in LDS and their sums in registers, and computes several terms in one launch: X (a few diagonals,
// in the L2) is all it reads per term. The pair product computes one term per launch, over the diagonals that the term
// holds, and re-reads each of them once per diagonal of X (TFIM-12: 14 terms of up to 8191 diagonals x 25, 0.66 ms each,
// and as many union-adds, norms, allocations and host dry-runs).
//
// A column c of a row sums T[c - d] X[c - d, c] over X's diagonals d, taken by descending offset: the term's diagonals
// then ascend, which is the order of the pair product, so each element is the same sum (the diagonals a term does not
// hold contribute exact zeros) and U has the same bits. The offsets of the result are the structural ones of the
// series, kept as bitsets on the host.
//
// The waves walk X's live diagonals as dia_rows_wave does: one diagonal's metadata per lane, a ballot of those that hold
// a nonzero in the 64 rows or so that meet the wave's 64 columns (zero-block map; a part that is all zero is not loaded),
// and the loads of several of them in flight.
//
// The series stops after the first term whose Frobenius norm is below the tolerance. Terms are launched in batches; the
// norms of a batch predict how many more are needed (for a normal X the norms fall no faster than the last ratio says,
// so the prediction does not overshoot), and a batch that did run past the stop is run again with the right count.
//
// Bound: the L2's reads of X, once per RB rows and term, and the latency between them (a workgroup per CU: its rows fill
// the LDS). TFIM-12 (4096 rows, 25 diagonals): 14 terms of the series and 14 of the squaring in 4 launches, 0.25 ms per term
// with the launches' reads and writes of T and U. exp(-iHt) as a whole, ms, before / now: TFIM-8 2.7 / 0.25, TFIM-12 39 / 7.1,
// XXZ-13 212 / 82.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <numeric>
#include <stdexcept>

#include "dia_rows.hpp"
#include "taylor_shape.hpp"

namespace dq {

typedef double c64 __attribute__((ext_vector_type(2)));

struct TaylorSlots {
    const DiagMeta *meta;  // X's diagonals by descending offset
    const uint2 *map;      // their zero-block maps (64-row blocks), `words` words each
    int64_t words;
    int n;
};

// The element at a byte offset from p (uniform).
template <typename T>
__device__ __forceinline__ const T *lane_elem(const T *p, uint32_t bytes) {
    return reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + bytes);
}

// Adds, for the wave's 64 columns of RB rows, the products with the diagonals of todo: lane s holds, for diagonal s, xb
// (element index of its value for column c0), ib (row index of that value, which is the term's column) and rng (dia_rows).
template <typename T, int RB, int NS, typename Row, typename Add>
__device__ __forceinline__ void taylor_columns(uint64_t todo, int lane, int64_t xb, int ib, int rng,
                                               const T *__restrict__ xre, const T *__restrict__ xim,
                                               const Row (&row)[RB][NS], Add &&add) {
#pragma clang fp contract(off)
    constexpr int DB = 4;
    while (todo) {  // uniform
        T vr[DB], vi[DB];
        int at[DB], all = 0;
        const int cnt = __popcll(todo);
        int k = 0;
#pragma unroll
        for (int u = 0; u < DB; ++u) {  // past the last diagonal: that one again, as zeros
            if (u < cnt) {
                k = __builtin_ctzll(todo);
                todo &= todo - 1;
            }
            const int64_t b = readlane64(xb, k);
            const int r = __builtin_amdgcn_readlane(rng, k);
            const int l = r & RNG_MASK, h = (r >> RNG_HI) & RNG_MASK;
            const int e = min(max(lane, l), h - 1);
            at[u] = __builtin_amdgcn_readlane(ib, k) + e;
            vr[u] = T(0);
            vi[u] = T(0);
            if (u < cnt) {  // uniform, as the parts
                all |= r;
                if (r & RNG_RE) vr[u] = *lane_elem(xre + b, e * static_cast<uint32_t>(sizeof(T)));
                if (r & RNG_IM) vi[u] = *lane_elem(xim + b, e * static_cast<uint32_t>(sizeof(T)));
                if (l != 0 || h != 64) {  // uniform
                    const bool in = e == lane;
                    vr[u] = in ? vr[u] : T(0);
                    vi[u] = in ? vi[u] : T(0);
                }
            }
        }
        // a part that is zero in all of them leaves products that are zeros of either sign, which no sum keeps; the other
        // products are rounded before they are added, as cmul's are
        if (!(all & RNG_RE)) {
#pragma unroll
            for (int u = 0; u < DB; ++u)
#pragma unroll
                for (int b = 0; b < RB; ++b) {
                    const Row t = row[b][at[u]];
                    add(b, -(t.y * vi[u]), t.x * vi[u]);
                }
        } else if (!(all & RNG_IM)) {
#pragma unroll
            for (int u = 0; u < DB; ++u)
#pragma unroll
                for (int b = 0; b < RB; ++b) {
                    const Row t = row[b][at[u]];
                    add(b, t.x * vr[u], t.y * vr[u]);
                }
        } else {
#pragma unroll
            for (int u = 0; u < DB; ++u)
#pragma unroll
                for (int b = 0; b < RB; ++b) {
                    const Row t = row[b][at[u]];
                    T re, im;
                    cmul(t.x, t.y, vr[u], vi[u], re, im);
                    add(b, re, im);
                }
        }
    }
}

// Terms k0 + 1 .. k0 + terms of rows blockIdx.x * RB ..; Tin / Uin (null: T_0 = U_0 = I), Tout (may be null) / Uout
// row-major complex N x N. part[j * gridDim.x + block]: the block's share of the squared Frobenius norm of term k0 + 1 + j
// (null: no norms, for any number of terms).
template <typename T, int THREADS, int CPT, int RB>
__global__ __launch_bounds__(THREADS) void taylor_rows_kernel(int N, TaylorSlots X, const T *__restrict__ xre,
                                                              const T *__restrict__ xim, int k0, int terms,
                                                              const c64 *__restrict__ Tin, const c64 *__restrict__ Uin,
                                                              c64 *__restrict__ Tout, c64 *__restrict__ Uout,
                                                              double *__restrict__ part) {
    typedef T T2 __attribute__((ext_vector_type(2)));
    constexpr int NS = THREADS * CPT;
    __shared__ T2 row[RB][NS];
    __shared__ double red[THREADS / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r0 = blockIdx.x * RB;
    T ur[RB][CPT], ui[RB][CPT];
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            const int c = tid + THREADS * q, r = r0 + b;
            T2 t{T(0), T(0)};
            ur[b][q] = T(0);
            ui[b][q] = T(0);
            if (r < N && c < N) {
                if (Tin) {
                    const c64 v = Tin[static_cast<int64_t>(r) * N + c], u = Uin[static_cast<int64_t>(r) * N + c];
                    t = T2{static_cast<T>(v.x), static_cast<T>(v.y)};
                    ur[b][q] = static_cast<T>(u.x);
                    ui[b][q] = static_cast<T>(u.y);
                } else if (r == c) {
                    t.x = T(1);
                    ur[b][q] = T(1);
                }
            }
            row[b][c] = t;
        }
    __syncthreads();
    for (int j = 0; j < terms; ++j) {
        T ar[RB][CPT] = {}, ai[RB][CPT] = {};
        for (int s0 = 0; s0 < X.n; s0 += 64) {
            const int s = s0 + lane;
            DiagMeta m{0, 0, 0, 0, 0};
            if (s < X.n) m = X.meta[s];
#pragma unroll
            for (int q = 0; q < CPT; ++q) {
                const int c0 = wave * 64 + THREADS * q;  // the wave's columns c0 .. c0 + 63
                if (c0 >= N) continue;                   // uniform
                // lane s: the rows c0 - off + [lo, hi) of its diagonal that meet the columns, in blocks b0 and b1
                const int ib = c0 - m.off;
                const int lo = max(static_cast<int>(m.rlo) - ib, 0), hi = min(static_cast<int>(m.rhi) - ib, 64);
                int rng = 0;
                if (lo < hi) {
                    const int b0 = (ib + lo) >> 6, b1 = (ib + hi - 1) >> 6;
                    const uint2 w0 = X.map[s * X.words + (b0 >> 5)], w1 = X.map[s * X.words + (b1 >> 5)];
                    const int parts = ((((w0.x >> (b0 & 31)) | (w1.x >> (b1 & 31))) & 1u) ? RNG_RE : 0) |
                                      ((((w0.y >> (b0 & 31)) | (w1.y >> (b1 & 31))) & 1u) ? RNG_IM : 0);
                    rng = parts ? lo | hi << RNG_HI | parts : 0;
                }
                uint64_t todo = __ballot(rng != 0);
                taylor_columns<T, RB, NS>(todo, lane, m.rowbase + ib, ib, rng, xre, xim, row, [&](int b, T re, T im) {
                    ar[b][q] += re;
                    ai[b][q] += im;
                });
            }
        }
        __syncthreads();  // every wave is done with the old term
        const double div = static_cast<double>(k0 + 1 + j);
        double sq = 0.0;
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int q = 0; q < CPT; ++q) {
                const int c = tid + THREADS * q;
                T2 t{ar[b][q], ai[b][q]};
                if (div != 1.0) t = T2{static_cast<T>(ar[b][q] / div), static_cast<T>(ai[b][q] / div)};
                row[b][c] = t;
                ur[b][q] += t.x;
                ui[b][q] += t.y;
                const double x = static_cast<double>(t.x), y = static_cast<double>(t.y);
                if (c < N && r0 + b < N) sq += x * x + y * y;
            }
        if (part) {  // uniform
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o, 64);
            if (lane == 0) red[wave] = sq;
        }
        __syncthreads();  // the new term and the waves' sums
        if (part && tid == 0) {
            double v = 0.0;
            for (int w = 0; w < THREADS / 64; ++w) v += red[w];
            part[static_cast<int64_t>(j) * gridDim.x + blockIdx.x] = v;
        }
    }
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            const int c = tid + THREADS * q, r = r0 + b;
            if (r < N && c < N) {
                const T2 t = row[b][c];
                if (Tout)
                    Tout[static_cast<int64_t>(r) * N + c] = c64{static_cast<double>(t.x), static_cast<double>(t.y)};
                Uout[static_cast<int64_t>(r) * N + c] =
                    c64{static_cast<double>(ur[b][q]), static_cast<double>(ui[b][q])};
            }
        }
}

// out[j] = sum of part[j * n ..], one workgroup per j.
__global__ __launch_bounds__(256) void fold_parts_kernel(int n, const double *__restrict__ part,
                                                         double *__restrict__ out) {
    __shared__ double red[4];
    double v = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) v += part[static_cast<int64_t>(blockIdx.x) * n + i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

namespace {
// Ascending offsets of a bitset over [-(N - 1), N - 1].
struct OffsetSet {
    int64_t N;
    std::vector<uint64_t> w;
    explicit OffsetSet(int64_t n) : N(n), w(static_cast<size_t>((2 * n - 1 + 63) / 64), 0) {}
    void add(int64_t d) { w[(d + N - 1) / 64] |= uint64_t(1) << ((d + N - 1) % 64); }
    // this |= o shifted by d, what leaves the range dropped
    void add_shifted(const OffsetSet &o, int64_t d) {
        const int64_t n = static_cast<int64_t>(w.size());
        const int64_t ws = d >= 0 ? d / 64 : -((-d + 63) / 64);
        const int sh = static_cast<int>(d - ws * 64);
        for (int64_t i = std::max<int64_t>(0, -ws - 1); i < n && i + ws < n; ++i) {
            if (i + ws >= 0) w[i + ws] |= o.w[i] << sh;
            if (sh && i + ws + 1 >= 0 && i + ws + 1 < n) w[i + ws + 1] |= o.w[i] >> (64 - sh);
        }
        const int64_t tail = (2 * N - 1) % 64;
        if (tail) w.back() &= (uint64_t(1) << tail) - 1;
    }
    std::vector<int32_t> list() const {
        std::vector<int32_t> out;
        for (size_t i = 0; i < w.size(); ++i)
            for (uint64_t x = w[i]; x; x &= x - 1)
                out.push_back(static_cast<int32_t>(static_cast<int64_t>(i) * 64 + __builtin_ctzll(x) - (N - 1)));
        return out;
    }
};

// The structural offsets of I + X + .. + X^terms.
std::vector<int32_t> series_offsets(const dq_devmat &X, int terms) {
    OffsetSet sum(X.rows), term(X.rows);
    sum.add(0);
    term.add(0);
    for (int k = 0; k < terms; ++k) {
        OffsetSet next(X.rows);
        for (int32_t d : X.offs) next.add_shifted(term, d);
        const bool same = next.w == term.w;
        term = std::move(next);
        for (size_t i = 0; i < sum.w.size(); ++i) sum.w[i] |= term.w[i];
        if (same) break;  // every later term has these offsets too
    }
    return sum.list();
}

template <typename T>
void launch_rows(int N, const TaylorSlots &S, const dq_devmat &X, int k0, int terms, const c64 *Tin, const c64 *Uin,
                 c64 *Tout, c64 *Uout, double *part, hipStream_t s) {
    const T *xre = X.re.as<T>(), *xim = X.im.as<T>();
    const dim3 grid(static_cast<unsigned>(taylor_grid(N)));
#define DQ_TAYLOR(I)                                                                                               \
    case I:                                                                                                        \
        hipLaunchKernelGGL(                                                                                        \
            (taylor_rows_kernel<T, TAYLOR_SHAPES[I].threads, TAYLOR_SHAPES[I].cols, TAYLOR_SHAPES[I].rows>), grid, \
            dim3(TAYLOR_SHAPES[I].threads), 0, s, N, S, xre, xim, k0, terms, Tin, Uin, Tout, Uout, part);          \
        break;
    switch (taylor_shape(N)) {
        DQ_TAYLOR(0)
        DQ_TAYLOR(1)
        DQ_TAYLOR(2)
        DQ_TAYLOR(3)
        DQ_TAYLOR(4)
        DQ_TAYLOR(5)
    }
#undef DQ_TAYLOR
    DQ_LAUNCH_CHECK();
}

constexpr int FIRST_TERMS = 6;
constexpr double ACTION_COST = 5.0;
}  // namespace

// Up to 1024 rows always: few launches and host steps, whatever X (ms, rows over dense rows / pair products: 1024 rows, 3
// diagonals 0.32 / 1.59; 1024 rows, 2047 diagonals 4.6 / 8.1). Above that while X has at most N / 4 diagonals (a term
// costs as many passes over the rows; 2048 rows, 512 diagonals 4.2 / 10.6, 4095 diagonals 30 / 13.9; 4096 rows, 1024
// diagonals 46 / 52), and above 2048 rows where the result fills enough of the dense matrix (4096 rows: TFIM-12 7.1 / 39,
// a tridiagonal X 1.79 / 1.93).
bool dense_taylor_pays(const dq_devmat &X) {
    const int64_t N = X.rows;
    if (!dense_enabled() || N < 1 || N > TAYLOR_MAX_N || X.n() == 0) return false;
    if (N <= 1024) return true;
    if (4 * static_cast<int64_t>(X.n()) > N) return false;
    if (N <= 2048) return true;
    // the pair products' share of the dense work, for the offsets that about ten terms reach
    const std::vector<int32_t> offs = series_offsets(X, 10);
    double stored = 0.0;
    for (int32_t d : offs) stored += static_cast<double>(N - std::abs(d));
    return stored >= 0.25 * static_cast<double>(N) * N;
}

TaylorRows::TaylorRows(const dq_devmat &X_, hipStream_t s_) : X(X_), s(s_) {
    const int64_t N = X.rows;
    std::vector<int> order(X.n());
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return X.offs[a] > X.offs[b]; });
    for (int k : order) meta.push_back(X.meta[k]);
    words = zero_block_words(N, 64);
    dmeta = DevBuf(sizeof(DiagMeta) * meta.size());
    map = DevBuf(sizeof(uint2) * static_cast<size_t>(words) * X.n());
    DQ_HIP(hipMemcpyAsync(dmeta.p, meta.data(), dmeta.bytes, hipMemcpyHostToDevice, s));
    make_zero_map(X, dmeta.as<DiagMeta>(), 6, map.as<uint2>(), s);
    part = DevBuf(sizeof(double) * static_cast<size_t>(taylor_parts_room(N)));
    folded = DevBuf(sizeof(double) * TAYLOR_BATCH);
}

void TaylorRows::run(int k0, int n, const void *tin, const void *uin, void *tout, void *uout, bool norms) {
    const TaylorSlots S{dmeta.as<DiagMeta>(), map.as<uint2>(), words, X.n()};
    const int N = static_cast<int>(X.rows);
    if (n < 1) return;
    if (N > TAYLOR_MAX_N || taylor_parts(N, n, norms) > static_cast<int64_t>(part.bytes / sizeof(double)))
        throw std::logic_error("expm: a launch of the series outgrows its workspace");
    double *const parts = norms ? part.as<double>() : nullptr;
    if (X.precision == DQ_F64)
        launch_rows<double>(N, S, X, k0, n, static_cast<const c64 *>(tin), static_cast<const c64 *>(uin),
                            static_cast<c64 *>(tout), static_cast<c64 *>(uout), parts, s);
    else
        launch_rows<float>(N, S, X, k0, n, static_cast<const c64 *>(tin), static_cast<const c64 *>(uin),
                           static_cast<c64 *>(tout), static_cast<c64 *>(uout), parts, s);
}

bool TaylorRows::series(int max_iterations, double tol, const char *who, DevBuf &dense, std::vector<int32_t> &offs) {
    const size_t bytes = static_cast<size_t>(X.rows) * X.rows * sizeof(c64);
    DevBuf Tb[2] = {DevBuf(bytes), DevBuf(bytes)}, Ub[2] = {DevBuf(bytes), DevBuf(bytes)};
    int cur = 0;  // which buffers hold the state (none before the first batch)
    double last = 0.0, before = 0.0;
    bool stop = false;
    done = 0;
    while (done < max_iterations && !stop) {
        int want = FIRST_TERMS;
        if (done > 0) {  // the last ratio of norms, times k, is how fast the terms of X^k / k! still grow
            const double rho = before > 0.0 ? last / before * done : 0.0;
            double p = last;
            want = 0;
            do {
                ++want;
                p *= rho / (done + want);
            } while (p >= tol && want < TAYLOR_BATCH);
        }
        want = std::min(want, max_iterations - done);
        double sq[TAYLOR_BATCH];
        for (;;) {
            run(done, want, done ? Tb[cur].p : nullptr, done ? Ub[cur].p : nullptr, Tb[cur ^ 1].p, Ub[cur ^ 1].p, true);
            hipLaunchKernelGGL(fold_parts_kernel, dim3(static_cast<unsigned>(want)), dim3(256), 0, s,
                               static_cast<int>(taylor_grid(X.rows)), part.as<double>(), folded.as<double>());
            DQ_LAUNCH_CHECK();
            DQ_HIP(hipMemcpyAsync(sq, folded.p, sizeof(double) * want, hipMemcpyDeviceToHost, s));
            DQ_HIP(hipStreamSynchronize(s));
            for (int j = 0; j < want; ++j)
                if (!std::isfinite(sq[j])) return false;
            int first = 0;  // the first term of the batch below the tolerance
            while (first < want && !(std::sqrt(sq[first]) < tol)) ++first;
            if (first + 1 < want) {  // past the stop: the batch again, up to that term
                want = first + 1;
                continue;
            }
            stop = first < want;
            break;
        }
        before = want > 1 ? std::sqrt(sq[want - 2]) : last;
        last = std::sqrt(sq[want - 1]);
        done += want;
        cur ^= 1;
    }
    const int i = stop ? done : max_iterations + 1;  // the loop counter of the series, as the pair path leaves it
    if (i == max_iterations)
        std::printf("Warning: %s reached max iterations (%d) without convergence.\n", who, max_iterations);
    dense = std::move(Ub[cur]);
    offs = series_offsets(X, done);
    return true;
}

bool dense_square_pays(int64_t N, size_t n_offsets) {
    return N <= 512 || static_cast<double>(n_offsets) * static_cast<double>(n_offsets) >= 0.25 * static_cast<double>(N) * N;
}

// U holds p(X)^(2^j) for the series' polynomial p: its square is p(X) applied to it 2^j times, at `done` terms of X's
// diagonals each, or one dense product. Measured, ms: TFIM-12 (14 terms of 25
// diagonals) 3.3 by terms, 9.4 by the product; a term and diagonal costs as much as ACTION_COST rows of the product where
// X's values are complex, less where a part is zero.
std::vector<int32_t> TaylorRows::square(const std::vector<int32_t> &offs, DevBuf &U, int j) {
    const int64_t N = X.rows;
    DevBuf P(U.bytes);
    const double action = std::ldexp(static_cast<double>(done) * X.n(), j);
    if (X.precision == DQ_F64 && ACTION_COST * action < static_cast<double>(N)) {
        for (int64_t i = 0; i < (int64_t(1) << j); ++i) {
            run(0, done, U.p, U.p, nullptr, P.p, false);  // `done` may exceed TAYLOR_BATCH; no norms are needed
            std::swap(U, P);
        }
    } else {
        zgemm_dense(N, N, N, U.as<double>(), U.as<double>(), P.as<double>(), 1.0, s);
        std::swap(U, P);
    }
    DQ_HIP(hipStreamSynchronize(s));  // the other buffer goes back to the cache
    if (static_cast<int64_t>(offs.size()) == 2 * N - 1) return offs;  // every diagonal stays
    OffsetSet a(N), r(N);
    for (int32_t d : offs) a.add(d);
    for (int32_t d : offs) r.add_shifted(a, d);
    return r.list();
}

}  // namespace dq
