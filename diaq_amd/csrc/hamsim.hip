// Fused time evolution on gfx950: psi(t) = prod_r exp(-i H t/r) psi0 with a fixed-m Taylor action per step, all on
// the device.
//
// Reference: spmv_row_diag_sparse_kernel, vec_copy / vec_axpy / vec_mul_minus_i_scale, expm_action_taylor_device
// and hamiltonian_simulation_cuda (src/spHamSim_gpu_all_fused.cu:117-376).
//
// The reference runs, per Taylor term, an SpMV (tmp = H term), a scaling pass (term = (-i dt/k) tmp) and an axpy
// (out += term), plus two copies per step and a device synchronisation. Here one kernel does all three: it forms
// h = H term_{k-1} row by row in registers (the shared row-tile core), writes term_k = (-i dt/k) h, i.e.
// (Im h * s, -Re h * s) with s = dt/k, and adds term_k to the step's output; the first term reads psi directly and
// writes out = psi + term_1, so the copies disappear. Per term: H read once, term_{k-1} read, term_k written and the
// output read and written once (b*S + 4*b*N bytes). The same operation order as the reference per element:
// row sums in slot order, then the scaling, then the add. The row sums are dia_rows_wave's; the term kernel may stage
// the x window of each row tile in LDS: the +-2^k offsets of a qubit Hamiltonian then share one copy of the term vector
// per tile. Its schedule is timed on the first evolution of a matrix and kept in its handle.
//
// Each call on a large matrix first maps, per 64-row block of every diagonal, whether its real and its imaginary
// values are all zero (one read of H), and every term skips what is: a zero block adds nothing to a row sum (the
// products it would add are zeros, exact in FP64 for finite inputs), a zero part is the constant 0. A qubit
// Hamiltonian's flip diagonals are zero on alternate runs of 2^k rows (three runs in four for a flip-flop term) and
// its imaginary part often everywhere. H cannot change during the call, so the map stays valid for all of its terms.
//
// Bound: reads of the live values. XXZ-20 (156 MB of nonzero real parts of 637 MB stored, and 67 MB of vectors per
// term): 90.7 us per term with 256-row blocks, both parts read and a metadata chain per diagonal; 45 us now, 4.9 TB/s.
// A launch per term for XXZ-10: 12.9 -> 5.8 us, the launch and three dependent round trips; such small matrices take all
// terms in one workgroup instead, 1.5 us each (taylor_resident_kernel).
#include <algorithm>
#include <type_traits>

#include "dia_rows.hpp"

namespace dq {

static int g_hamsim_skip = 1;  // "hamsim_skip_zero_blocks"
static int g_hamsim_rpt = 0;   // "hamsim_rows_per_lane": 0 = the matrix's choice; 2, 4 or 8: two adjacent rows per lane
static int g_hamsim_lds = -1;  // "hamsim_lds": -1 = the matrix's choice, else 0 or 1 (with two rows per lane)

bool hamsim_set_tuning(const std::string &key, int value) {
    if (key == "hamsim_skip_zero_blocks") {
        if (value != 0 && value != 1) throw ArgError("hamsim_skip_zero_blocks must be 0 or 1");
        g_hamsim_skip = value;
        return true;
    }
    if (key == "hamsim_rows_per_lane") {
        if (value != 0 && value != 2 && value != 4 && value != 8)
            throw ArgError("hamsim_rows_per_lane must be 0, 2, 4 or 8");
        g_hamsim_rpt = value;
        return true;
    }
    if (key == "hamsim_lds") {
        if (value < -1 || value > 1) throw ArgError("hamsim_lds must be -1, 0 or 1");
        g_hamsim_lds = value;
        return true;
    }
    return false;
}

// TO: the precision of the step output (and of psi, read by the first term). TO = T for an FP64 Hamiltonian. An FP32
// Hamiltonian (the precision form) runs its terms in FP32 but adds them into an FP64 output; the step's last term
// also writes the output rounded to FP32 (o32), the next step's FP32 input.
template <typename T, typename TO, int V, bool NT, bool ZM, bool LDS>
__global__ __launch_bounds__(256) void taylor_term_kernel(int64_t rows, int n, const DiagMeta *__restrict__ meta,
                                                          const T *__restrict__ are, const T *__restrict__ aim,
                                                          const T *__restrict__ tr, const T *__restrict__ ti,
                                                          T *__restrict__ nr, T *__restrict__ ni,
                                                          TO *__restrict__ outr, TO *__restrict__ outi,
                                                          const TO *__restrict__ p0r, const TO *__restrict__ p0i,
                                                          T *__restrict__ o32r, T *__restrict__ o32i, double scale,
                                                          int first, int64_t ntiles, int xcd, ZeroMap zm) {
    constexpr int H = LDS ? 128 * V : 0;
    __shared__ T sr[LDS ? 256 * V + 2 * H : 1], si[LDS ? 256 * V + 2 * H : 1];
    const int64_t t = tile_of_block(blockIdx.x, ntiles, xcd);
    if (t >= ntiles) return;  // uniform
    if constexpr (LDS) stage_x_window<T, V, H>(t * 256 * V, rows, tr, ti, sr, si);
    const int64_t row0 = wave_row0<V>(t);
    if (row0 >= rows) return;  // uniform
    const int64_t r = row0 + V * (threadIdx.x & 63);
    // out = psi + term_1 at the first term (psi is the term_0 input), out += term_k after
    TO orr[V], oii[V];
    ld_rows(first ? p0r : outr, r, rows, orr);
    ld_rows(first ? p0i : outi, r, rows, oii);
    Acc<T> hr[V], hi[V];
    dia_rows_wave<T, V, NT, ZM, H>(row0, n, meta, are, aim, tr, ti, 0, rows, hr, hi, zm, sr, si);
    const T s = static_cast<T>(scale);
    T vr[V], vi[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        vr[v] = hi[v].get() * s;  // (-i s)(a + ib)
        vi[v] = -hr[v].get() * s;
        if constexpr (std::is_same<T, TO>::value) {  // one rounding, spelled out so that every schedule has it
            orr[v] = __builtin_fma(s, hi[v].get(), orr[v]);
            oii[v] = __builtin_fma(s, -hr[v].get(), oii[v]);
        } else {
            orr[v] += static_cast<TO>(vr[v]);
            oii[v] += static_cast<TO>(vi[v]);
        }
    }
    st_rows(nr, r, rows, vr);
    st_rows(ni, r, rows, vi);
    st_rows(outr, r, rows, orr);
    st_rows(outi, r, rows, oii);
    if (o32r) {
        T fr[V], fi[V];
#pragma unroll
        for (int v = 0; v < V; ++v) {
            fr[v] = static_cast<T>(orr[v]);
            fi[v] = static_cast<T>(oii[v]);
        }
        st_rows(o32r, r, rows, fr);
        st_rows(o32i, r, rows, fi);
    }
}

template <typename T>
__global__ void copy2_kernel(int64_t n, const T *__restrict__ ar, const T *__restrict__ ai, T *__restrict__ br,
                             T *__restrict__ bi) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        br[i] = ar[i];
        bi[i] = ai[i];
    }
}

template <typename TD, typename TS>
__global__ void convert2_kernel(int64_t n, const TS *__restrict__ ar, const TS *__restrict__ ai, TD *__restrict__ br,
                                TD *__restrict__ bi) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        br[i] = static_cast<TD>(ar[i]);
        bi[i] = static_cast<TD>(ai[i]);
    }
}

template <typename TD, typename TS>
static void convert2(int64_t n, const TS *ar, const TS *ai, TD *br, TD *bi, hipStream_t s) {
    hipLaunchKernelGGL((convert2_kernel<TD, TS>), dim3(blocks_for(n, 256, 8192)), dim3(256), 0, s, n, ar, ai, br, bi);
    DQ_LAUNCH_CHECK();
}

// The term kernel's schedule: rows per lane (1 or 2) and non-temporal loads of H's values.
struct TermSched {
    int v = 1;
    bool nt = true, lds = false;
};

// One term: term_k = (-i scale) H in, out (+)= term_k.
template <typename T, typename TO>
static void launch_term(const dq_devmat &H, const TermSched &c, const T *inr, const T *ini, T *nr, T *ni, TO *outr,
                        TO *outi, const TO *p0r, const TO *p0i, T *o32r, T *o32i, double scale, int first,
                        const ZeroMap &zm, hipStream_t s) {
    const int64_t N = H.rows;
    const int64_t ntiles = (N + 256 * c.v - 1) / (256 * c.v);
    const int xcd = xcd_tiles_for(H);
    const dim3 grid(static_cast<unsigned>(grid_for_tiles(ntiles, xcd)));
    const DiagMeta *meta = H.d_meta.as<DiagMeta>();
    const T *are = static_cast<const T *>(H.re.p), *aim = static_cast<const T *>(H.im.p);
#define DQ_TERM(V, NT, Z, L)                                                                                          \
    hipLaunchKernelGGL((taylor_term_kernel<T, TO, V, NT, Z, L>), grid, dim3(256), 0, s, N, H.n(), meta, are, aim, inr, \
                       ini, nr, ni, outr, outi, p0r, p0i, o32r, o32i, scale, first, ntiles, xcd, zm)
#define DQ_TERM_V(NT, Z)                                   \
    do {                                                   \
        if (c.v == 2 && c.lds) DQ_TERM(2, NT, Z, true);    \
        else if (c.v == 2) DQ_TERM(2, NT, Z, false);       \
        else DQ_TERM(1, NT, Z, false);                     \
    } while (0)
    if (c.nt && zm.w) DQ_TERM_V(true, true);
    else if (c.nt) DQ_TERM_V(true, false);
    else if (zm.w) DQ_TERM_V(false, true);
    else DQ_TERM_V(false, false);
#undef DQ_TERM_V
#undef DQ_TERM
    DQ_LAUNCH_CHECK();
}

// The term kernel's schedule for H: rows per lane, LDS window (where some off-diagonal lies within half a tile) and
// non-temporal loads. Below EVO_SMALL rows it is one row per lane with plain loads: the matrix is small, the launch
// is what a term costs, and more and shorter waves shorten it (10 qubits: 5.8 us per term against 7.3 with two rows
// per lane). Larger matrices time the candidates on two first terms (psi in, scratch out) the first time they are
// evolved, and keep the choice in the handle: it depends on whether the live values stay in the 256 MB Infinity Cache
// from term to term (XXZ-20, 156 MB of nonzero real parts: 45 us per term with plain loads, 53 non-temporal; XXZ-22:
// 235 and 216). Every schedule adds the same products in the same order, so the choice changes the speed only.
constexpr int64_t EVO_SMALL = int64_t(1) << 16;

template <typename T, typename TO>
static TermSched term_schedule(const dq_devmat &H, const T *pr, const T *pi, const TO *p0r, const TO *p0i, TO *outr,
                               TO *outi, T *tr, T *ti, const ZeroMap &zm, hipStream_t s) {
    if (H.rows < EVO_SMALL) {
        H.term_nt = 0;
        H.term_lds = 0;
        H.term_rpt = 1;
    }
    if (H.term_rpt == 0) {
        hipEvent_t e0, e1;
        DQ_HIP(hipEventCreate(&e0));
        DQ_HIP(hipEventCreate(&e1));
        float best = 1e30f;
        TermSched win;
        for (int form = 0; form < 3; ++form) {
            if (form == 2 && !lds_window_pays(H, 2)) continue;
            for (int nt = 0; nt < 2; ++nt) {
                const TermSched c{form == 0 ? 1 : 2, nt == 1, form == 2};
                auto one = [&] {
                    launch_term<T, TO>(H, c, pr, pi, tr, ti, outr, outi, p0r, p0i, nullptr, nullptr, 0.1, 1, zm, s);
                };
                one();  // warm
                DQ_HIP(hipEventRecord(e0, s));
                for (int q = 0; q < 2; ++q) one();
                DQ_HIP(hipEventRecord(e1, s));
                DQ_HIP(hipEventSynchronize(e1));
                float ms = 0.f;
                DQ_HIP(hipEventElapsedTime(&ms, e0, e1));
                if (ms < best) { best = ms; win = c; }
            }
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        H.term_nt = win.nt ? 1 : 0;  // before term_rpt, which marks the choice as made
        H.term_lds = win.lds ? 1 : 0;
        H.term_rpt = win.v;
    }
    TermSched c;
    c.v = g_hamsim_rpt ? 2 : H.term_rpt.load();
    c.lds = g_hamsim_lds >= 0 ? g_hamsim_lds == 1 : H.term_lds.load() == 1;
    c.nt = H.term_nt.load() == 1;
    return c;
}

// One step out = sum_{k=0}^{m} (-i dt H)^k psi / k! (src/spHamSim_gpu_all_fused.cu:235-277). (pr, pi): psi in the
// term precision, the first term's input; (p0r, p0i): psi in the output precision (the same arrays when T = TO).
// t0/t1: scratch terms. (o32r, o32i), for T != TO: receives the output rounded to T.
template <typename T, typename TO>
static void taylor_step(const dq_devmat &H, const T *pr, const T *pi, const TO *p0r, const TO *p0i, TO *outr,
                        TO *outi, T *o32r, T *o32i, T *t0r, T *t0i, T *t1r, T *t1i, double dt, int m,
                        const TermSched &sched, const ZeroMap &zm, hipStream_t s) {
    const int64_t N = H.rows;
    if (m <= 0 || H.n() == 0) {  // out = psi (+ zero terms)
        hipLaunchKernelGGL(copy2_kernel<TO>, dim3(blocks_for(N, 256, 8192)), dim3(256), 0, s, N, p0r, p0i, outr,
                           outi);
        DQ_LAUNCH_CHECK();
        if (o32r) {
            hipLaunchKernelGGL(copy2_kernel<T>, dim3(blocks_for(N, 256, 8192)), dim3(256), 0, s, N, pr, pi, o32r,
                               o32i);
            DQ_LAUNCH_CHECK();
        }
        return;
    }
    const T *inr = pr, *ini = pi;
    T *bufr[2] = {t0r, t1r}, *bufi[2] = {t0i, t1i};
    for (int k = 1; k <= m; ++k) {
        T *nr = bufr[k & 1], *ni = bufi[k & 1];
        launch_term<T, TO>(H, sched, inr, ini, nr, ni, outr, outi, p0r, p0i, k == m ? o32r : nullptr,
                           k == m ? o32i : nullptr, dt / static_cast<double>(k), k == 1 ? 1 : 0, zm, s);
        inr = nr;
        ini = ni;
    }
}

// Many steps of a small matrix in one workgroup: V rows per lane (row = lane + 1024 v), the rows' values of up to ND
// diagonals in registers, the term vector in LDS (two buffers, a barrier per term), the step's output in registers.
// Each buffer has `pad` zeros on either side, pad the largest |offset|, so that a row reads every diagonal at lane +
// offset: one off a diagonal multiplies a zero by a zero, which leaves an FP64 sum that starts at +0 as it is (an FP32
// sum is compensated and takes only the rows on the diagonal). Products, order and roundings are those of
// taylor_term_kernel, so the result has the same bits.
//
// Bound: the LDS reads of x, 16 bytes per row, diagonal and term (10 qubits, 19 diagonals: 311 KB, 1.0 us at 128 bytes a
// clock), where a launch per term costs its launch and the round trips to the L2. 10-qubit XXZ, 20 steps of 18 terms:
// 2013 -> 553 us (1.5 us a term).
constexpr int RES_LANES = 1024, RES_ND = 24;
constexpr int RES_TERMS = 4096;  // terms of a launch: a few milliseconds

template <typename T, typename TO, int V>
__global__ __launch_bounds__(RES_LANES) void taylor_resident_kernel(int rows, int n, const DiagMeta *__restrict__ meta,
                                                                    const T *__restrict__ are,
                                                                    const T *__restrict__ aim, TO *__restrict__ pr,
                                                                    TO *__restrict__ pi, double dt, int m, int steps,
                                                                    int pad) {
    struct alignas(2 * sizeof(T)) Cx {
        T r, i;
    };
    extern __shared__ __align__(16) char smem[];
    Cx *buf = reinterpret_cast<Cx *>(smem);
    constexpr int G = sizeof(T) == 8 ? 3 : 2;  // diagonals whose x is read together: what the registers leave
    static_assert(RES_ND % G == 0 && RES_ND <= 32, "whole groups, one bit per diagonal");
    const int width = rows + 2 * pad;
    T ar[V][RES_ND], ai[V][RES_ND];
    uint32_t on[V];
    int off[RES_ND];  // uniform
#pragma unroll
    for (int k = 0; k < RES_ND; ++k) off[k] = __builtin_amdgcn_readfirstlane(k < n ? meta[k].off : 0);
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int r = static_cast<int>(threadIdx.x) + RES_LANES * v;
        on[v] = 0;
#pragma unroll
        for (int k = 0; k < RES_ND; ++k) {
            ar[v][k] = T(0);
            ai[v][k] = T(0);
            if (k < n) {  // uniform
                const DiagMeta md = meta[k];
                if (r >= md.rlo && r < md.rhi) {
                    ar[v][k] = are[md.rowbase + r];
                    ai[v][k] = aim[md.rowbase + r];
                    on[v] |= 1u << k;
                }
            }
        }
    }
    for (int e = threadIdx.x; e < 2 * width; e += blockDim.x) buf[e] = Cx{T(0), T(0)};
    __syncthreads();
    TO outr[V], outi[V];
    int at[V];  // the row's place in a buffer; rows past the last one write nothing and read zeros or finite terms
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int r = static_cast<int>(threadIdx.x) + RES_LANES * v;
        at[v] = pad + min(r, rows - 1);
        outr[v] = TO(0);
        outi[v] = TO(0);
        if (r < rows) {
            outr[v] = pr[r];
            outi[v] = pi[r];
            buf[at[v]] = Cx{static_cast<T>(outr[v]), static_cast<T>(outi[v])};
        }
    }
    __syncthreads();
    int cur = 0;
    for (int step = 0; step < steps; ++step) {
        for (int k = 1; k <= m; ++k) {
            const Cx *x = buf + cur * width;
            Acc<T> hr[V], hi[V];
#pragma unroll
            for (int g = 0; g < RES_ND; g += G) {
                if (g >= n) continue;  // uniform
                Cx xv[V][G];
#pragma unroll
                for (int u = 0; u < G; ++u)
#pragma unroll
                    for (int v = 0; v < V; ++v) xv[v][u] = x[at[v] + off[g + u]];
#pragma unroll
                for (int u = 0; u < G; ++u)
#pragma unroll
                    for (int v = 0; v < V; ++v)
                        if constexpr (sizeof(T) == 8) {
                            if (g + u < n) cmac(hr[v], hi[v], ar[v][g + u], ai[v][g + u], xv[v][u].r, xv[v][u].i);
                        } else if (on[v] >> (g + u) & 1u) {
                            cmac(hr[v], hi[v], ar[v][g + u], ai[v][g + u], xv[v][u].r, xv[v][u].i);
                        }
            }
            const T s = static_cast<T>(dt / static_cast<double>(k));
            Cx *y = buf + (cur ^ 1) * width;
#pragma unroll
            for (int v = 0; v < V; ++v) {
                Cx t{hi[v].get() * s, -hr[v].get() * s};  // (-i s)(a + ib)
                if constexpr (std::is_same<T, TO>::value) {
                    outr[v] = __builtin_fma(s, hi[v].get(), outr[v]);
                    outi[v] = __builtin_fma(s, -hr[v].get(), outi[v]);
                } else {
                    outr[v] += static_cast<TO>(t.r);
                    outi[v] += static_cast<TO>(t.i);
                }
                if (k == m) t = Cx{static_cast<T>(outr[v]), static_cast<T>(outi[v])};  // the next step's input
                if (static_cast<int>(threadIdx.x) + RES_LANES * v < rows) y[at[v]] = t;
            }
            cur ^= 1;
            __syncthreads();
        }
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int r = static_cast<int>(threadIdx.x) + RES_LANES * v;
        if (r < rows) {
            pr[r] = outr[v];
            pi[r] = outi[v];
        }
    }
}

// Whether H's evolution runs in taylor_resident_kernel: rows and diagonals whose values fit a workgroup's registers (96
// of a lane's 128; FP32 values two rows per lane), and the two term buffers in 64 KB of LDS. A term then takes 0.7 us (6
// qubits) to 1.6 us (10 qubits; FP32 10 qubits 1.9, 11 qubits 4.6), a launch of taylor_term_kernel 4.6 to 6.1 us at these
// sizes. An override of the terms' schedule asks for those launches.
static bool resident_fits(const dq_devmat &H, int m, int *pad, size_t *lds) {
    if (g_hamsim_rpt > 0 || g_hamsim_lds >= 0 || !g_hamsim_skip) return false;
    const int V = H.precision == DQ_F64 ? 1 : 2;
    if (H.rows > static_cast<uint32_t>(RES_LANES * V) || H.n() > RES_ND || H.n() == 0 || m <= 0 || m > RES_TERMS)
        return false;
    int p = 0;
    for (int32_t o : H.offs) p = std::max(p, o < 0 ? -o : o);
    *pad = p;
    *lds = 2 * (H.rows + 2 * static_cast<size_t>(p)) * 2 * elem_bytes(H.precision);
    return *lds <= (size_t(64) << 10);
}

// r steps of dt on the state (pr, pi), in place.
template <typename T, typename TO, int V>
static void launch_resident(const dq_devmat &H, TO *pr, TO *pi, double dt, uint64_t r, int m, int pad, size_t lds,
                            hipStream_t s) {
    const unsigned lanes = std::min<unsigned>(RES_LANES, (H.rows + 63) / 64 * 64);
    const uint64_t per = std::max<uint64_t>(1, RES_TERMS / m);
    for (uint64_t done = 0; done < r; done += per) {
        hipLaunchKernelGGL((taylor_resident_kernel<T, TO, V>), dim3(1), dim3(lanes), lds, s, static_cast<int>(H.rows),
                           H.n(), H.d_meta.as<DiagMeta>(), H.re.as<T>(), H.im.as<T>(), pr, pi, dt, m,
                           static_cast<int>(std::min(per, r - done)), pad);
        DQ_LAUNCH_CHECK();
    }
}

// ||v||^2 of an FP64 complex vector as RENORM_PARTS block partials (each block sums a fixed, grid-strided share of
// the elements in a fixed order, so the partials -- and the fold of them -- have the same bits on every run).
constexpr int RENORM_PARTS = 512;

__device__ inline double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ inline double block_sum256(double v) {
    __shared__ double part[4];
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    const double r = (part[0] + part[1]) + (part[2] + part[3]);
    __syncthreads();
    return r;
}

__global__ __launch_bounds__(256) void sumsq_parts_kernel(int64_t n, const double *__restrict__ re,
                                                          const double *__restrict__ im, double *__restrict__ part) {
    double acc = 0.0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        acc += re[i] * re[i] + im[i] * im[i];
    acc = block_sum256(acc);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// psi *= ||psi0|| / ||psi||, both squared norms folded from their partials by every block in the same order.
__global__ __launch_bounds__(256) void renorm_kernel(int64_t n, double *__restrict__ re, double *__restrict__ im,
                                                     const double *__restrict__ part0,
                                                     const double *__restrict__ part1) {
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < RENORM_PARTS; i += 256) {
        a += part0[i];
        b += part1[i];
    }
    a = block_sum256(a);
    b = block_sum256(b);
    const double f = b > 0.0 ? sqrt(a / b) : 1.0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        re[i] *= f;
        im[i] *= f;
    }
}

static void sumsq_parts(int64_t n, const double *re, const double *im, double *part, hipStream_t s) {
    hipLaunchKernelGGL(sumsq_parts_kernel, dim3(RENORM_PARTS), dim3(256), 0, s, n, re, im, part);
    DQ_LAUNCH_CHECK();
}

// The state back to the norm that part0 holds.
static void renormalise(int64_t N, double *pr, double *pi, const double *part0, double *part1, hipStream_t s) {
    sumsq_parts(N, pr, pi, part1, s);
    hipLaunchKernelGGL(renorm_kernel, dim3(blocks_for(N, 256, 8192)), dim3(256), 0, s, N, pr, pi, part0,
                       (const double *)part1);
    DQ_LAUNCH_CHECK();
}

// The zero-block map of H, read by every term of one evolution; `buf` keeps it. Below EVO_SMALL rows the look-up costs
// a term more than the skipped loads (8 to 13 qubits: 0.9 to 1.5 us of 5 to 7), so none is made.
static ZeroMap zero_map(const dq_devmat &H, int m, DevBuf &buf, hipStream_t s) {
    ZeroMap z;
    if (g_hamsim_skip && H.n() > 0 && m > 0 && H.rows >= EVO_SMALL) {
        buf = DevBuf(zero_map_bytes(H, z.shift));
        make_zero_map(H, z.shift, buf.as<uint2>(), s);
        z.w = buf.as<uint2>();
        z.words = zero_block_words(H.rows, 1 << z.shift);
    }
    return z;
}

// Evolve the device state (pr, pi) in place over r steps of dt = t / r, all in H's precision.
template <typename T>
static void evolve(const dq_devmat &H, T *pr, T *pi, double t, uint64_t r, int m, hipStream_t s) {
    const int64_t N = H.rows;
    if (r == 0 || N == 0) return;
    const double dt = t / static_cast<double>(r);
    int pad = 0;
    size_t lds = 0;
    if (std::is_same<T, double>::value && resident_fits(H, m, &pad, &lds)) {
        launch_resident<double, double, 1>(H, reinterpret_cast<double *>(pr), reinterpret_cast<double *>(pi), dt, r, m,
                                           pad, lds, s);
        DQ_HIP(hipStreamSynchronize(s));
        return;
    }
    DevBuf br(N * sizeof(T)), bi(N * sizeof(T)), t0r(N * sizeof(T)), t0i(N * sizeof(T)), t1r(N * sizeof(T)),
        t1i(N * sizeof(T));
    DevBuf zmap;
    const ZeroMap zm = zero_map(H, m, zmap, s);
    T *ar = pr, *ai = pi, *xr = br.as<T>(), *xi = bi.as<T>();
    TermSched sched;
    if (m > 0 && H.n() > 0)
        sched = term_schedule<T, T>(H, pr, pi, pr, pi, xr, xi, t0r.as<T>(), t0i.as<T>(), zm, s);
    for (uint64_t step = 0; step < r; ++step) {
        taylor_step<T, T>(H, ar, ai, ar, ai, xr, xi, nullptr, nullptr, t0r.as<T>(), t0i.as<T>(), t1r.as<T>(),
                          t1i.as<T>(), dt, m, sched, zm, s);
        std::swap(ar, xr);
        std::swap(ai, xi);
    }
    if (ar != pr) {  // odd number of steps: the result sits in the scratch pair
        hipLaunchKernelGGL(copy2_kernel<T>, dim3(blocks_for(N, 256, 8192)), dim3(256), 0, s, N, (const T *)ar,
                           (const T *)ai, pr, pi);
        DQ_LAUNCH_CHECK();
    }
    DQ_HIP(hipStreamSynchronize(s));  // scratch buffers are freed on return
}

// The precision form for an FP32 H: the state (pr, pi) stays FP64. Each step's terms run in FP32 from an FP32 copy
// of the state; they are added into an FP64 output, which the step's last term also rounds to FP32 for the next
// step. At the end the state is renormalised in FP64 to the norm it started with (the exact evolution is unitary).
static void evolve_mixed(const dq_devmat &H, double *pr, double *pi, double t, uint64_t r, int m, hipStream_t s) {
    const int64_t N = H.rows;
    if (r == 0 || N == 0) return;
    const double dt = t / static_cast<double>(r);
    const size_t b32 = N * sizeof(float), b64 = N * sizeof(double);
    int pad = 0;
    size_t lds = 0;
    if (resident_fits(H, m, &pad, &lds)) {
        DevBuf parts(2 * RENORM_PARTS * sizeof(double));
        double *part0 = parts.as<double>(), *part1 = part0 + RENORM_PARTS;
        sumsq_parts(N, pr, pi, part0, s);
        if (N <= RES_LANES) launch_resident<float, double, 1>(H, pr, pi, dt, r, m, pad, lds, s);
        else launch_resident<float, double, 2>(H, pr, pi, dt, r, m, pad, lds, s);
        renormalise(N, pr, pi, part0, part1, s);
        DQ_HIP(hipStreamSynchronize(s));
        return;
    }
    DevBuf xr(b64), xi(b64), p32r(b32), p32i(b32), q32r(b32), q32i(b32), t0r(b32), t0i(b32), t1r(b32), t1i(b32);
    DevBuf parts(2 * RENORM_PARTS * sizeof(double));
    double *part0 = parts.as<double>(), *part1 = part0 + RENORM_PARTS;
    sumsq_parts(N, pr, pi, part0, s);
    convert2<float, double>(N, pr, pi, p32r.as<float>(), p32i.as<float>(), s);
    DevBuf zmap;
    const ZeroMap zm = zero_map(H, m, zmap, s);
    double *ar = pr, *ai = pi, *or_ = xr.as<double>(), *oi = xi.as<double>();
    float *in_r = p32r.as<float>(), *in_i = p32i.as<float>(), *nx_r = q32r.as<float>(), *nx_i = q32i.as<float>();
    TermSched sched;
    if (m > 0 && H.n() > 0)
        sched = term_schedule<float, double>(H, in_r, in_i, pr, pi, or_, oi, t0r.as<float>(), t0i.as<float>(), zm, s);
    for (uint64_t step = 0; step < r; ++step) {
        taylor_step<float, double>(H, in_r, in_i, ar, ai, or_, oi, nx_r, nx_i, t0r.as<float>(), t0i.as<float>(),
                                   t1r.as<float>(), t1i.as<float>(), dt, m, sched, zm, s);
        std::swap(ar, or_);
        std::swap(ai, oi);
        std::swap(in_r, nx_r);
        std::swap(in_i, nx_i);
    }
    if (ar != pr) {
        hipLaunchKernelGGL(copy2_kernel<double>, dim3(blocks_for(N, 256, 8192)), dim3(256), 0, s, N,
                           (const double *)ar, (const double *)ai, pr, pi);
        DQ_LAUNCH_CHECK();
    }
    renormalise(N, pr, pi, part0, part1, s);
    DQ_HIP(hipStreamSynchronize(s));  // scratch buffers are freed on return
}

// An FP32 H on an FP32 state: the state is widened to FP64 for the evolution and rounded back once at the end.
static void evolve_fp32_state(const dq_devmat &H, float *pr, float *pi, double t, uint64_t r, int m, hipStream_t s) {
    const int64_t N = H.rows;
    if (r == 0 || N == 0) return;
    DevBuf wr(N * sizeof(double)), wi(N * sizeof(double));
    convert2<double, float>(N, pr, pi, wr.as<double>(), wi.as<double>(), s);
    evolve_mixed(H, wr.as<double>(), wi.as<double>(), t, r, m, s);
    convert2<float, double>(N, wr.as<double>(), wi.as<double>(), pr, pi, s);
    DQ_HIP(hipStreamSynchronize(s));
}

void hamsim_device(const dq_devmat &H, void *pr, void *pi, double t, uint64_t r, int m, hipStream_t s) {
    if (H.rows != H.cols) throw ArgError("hamiltonian_simulation_cuda: H must be square");
    if (H.precision == DQ_F64)
        evolve<double>(H, static_cast<double *>(pr), static_cast<double *>(pi), t, r, m, s);
    else
        evolve_fp32_state(H, static_cast<float *>(pr), static_cast<float *>(pi), t, r, m, s);
}

void hamsim_device_f64(const dq_devmat &H, double *pr, double *pi, double t, uint64_t r, int m, hipStream_t s) {
    if (H.rows != H.cols) throw ArgError("hamiltonian_simulation_cuda: H must be square");
    if (H.precision == DQ_F64)
        evolve<double>(H, pr, pi, t, r, m, s);
    else
        evolve_mixed(H, pr, pi, t, r, m, s);
}

}  // namespace dq

using namespace dq;

extern "C" int dq_hamsim_device(const dq_devmat *H, void *pr, void *pi, double t, uint64_t r, int m,
                                uintptr_t stream) {
    return guard([&] {
        if (!H) throw ArgError("hamiltonian_simulation_cuda: H is null");
        if (H->rows && (!pr || !pi)) throw ArgError("hamiltonian_simulation_cuda: psi0 is null");
        hamsim_device(*H, pr, pi, t, r, m, as_stream(stream));
    });
}

extern "C" int dq_hamsim_device_f64state(const dq_devmat *H, double *pr, double *pi, double t, uint64_t r, int m,
                                         uintptr_t stream) {
    return guard([&] {
        if (!H) throw ArgError("hamiltonian_simulation_cuda: H is null");
        if (H->rows && (!pr || !pi)) throw ArgError("hamiltonian_simulation_cuda: psi0 is null");
        hamsim_device_f64(*H, pr, pi, t, r, m, as_stream(stream));
    });
}

extern "C" int dq_hamsim_host(const dq_devmat *H, const double *psi_r, const double *psi_i, double t, uint64_t r,
                              int max_iterations, double *out_r, double *out_i) {
    return guard([&] {
        if (!H) throw ArgError("hamiltonian_simulation_cuda: H is null");
        if (H->rows != H->cols) throw ArgError("hamiltonian_simulation_cuda: H must be square");
        const int64_t N = H->rows;
        if (N == 0) return;
        if (!psi_r || !psi_i || !out_r || !out_i) throw ArgError("hamiltonian_simulation_cuda: psi0 is null");
        DevBuf dr(N * 8), di(N * 8);
        DQ_HIP(hipMemcpy(dr.p, psi_r, N * 8, hipMemcpyHostToDevice));
        DQ_HIP(hipMemcpy(di.p, psi_i, N * 8, hipMemcpyHostToDevice));
        hamsim_device_f64(*H, dr.as<double>(), di.as<double>(), t, r, max_iterations, 0);
        DQ_HIP(hipMemcpy(out_r, dr.p, N * 8, hipMemcpyDeviceToHost));
        DQ_HIP(hipMemcpy(out_i, di.p, N * 8, hipMemcpyDeviceToHost));
    });
}
