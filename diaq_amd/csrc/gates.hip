// Sequences of gates on a state vector (a Trotter step is one), applied in fused passes over HBM.
//
// Applying the gates one at a time (dq_kron_apply_device) streams the whole state through HBM once per gate. Here the
// sequence is cut into passes. A pass loads tiles of 2^L amplitudes into registers, applies every gate of its stretch
// of the sequence to the tile in order, and writes the tile back: one HBM round trip for the whole stretch.
//
// A tile is the set of amplitudes that agree on every qubit outside the pass's tile qubits T (|T| = L). T holds the
// qubits of the stretch's non-diagonal gates, filled up with the lowest remaining qubits; the planner keeps qubits
// 0..low-1 in T, so each tile is made of runs of at least 2^low contiguous amplitudes. A gate whose only diagonal is
// the main one joins any pass: it multiplies each amplitude by the entry that the amplitude's own index selects,
// wherever its qubits lie.
//
// Layout. A workgroup of 256 lanes holds a tile, 2^R amplitudes per lane (R = L - 8), with a window of R consecutive
// tile bits [a, a + R) in the register index and the other 8 bits in the lane index. A gate inside the window works on
// the lane's own registers, with its entries in scalar registers; when the next gate lies outside, the planner puts a
// step that moves the tile to another window through LDS (real parts, then imaginary parts, through one padded buffer
// of 2^L values, 34 KB in FP64). A diagonal gate runs in any window: the lane's part of
// its index is the same for all the lane's amplitudes, so it looks up one entry per value of the gate's qubits that lie
// in the window (1, 2 or 4 for a two-qubit gate) and not one per amplitude.
//
// What bounds it: HBM for passes of few gates (28 qubits: 1.69 ms for 8 one-qubit gates, 5.1 TB/s; 2.24 ms when the tile's
// runs lie 8 MB and more apart), vector issue for full ones (27 diagonal gates and 12 rotations about X: 2.74 ms, with 12
// general one-qubit gates 3.07). A first-order TFIM-28 step: 3 passes, 6.8 ms; 15.4 ms in 4 passes when the tiles lived in
// LDS and every gate read and wrote them there.
//
// Each gate's arithmetic on each amplitude is the single-gate kernel's (each row adds its terms in the order of the
// gate's diagonal slots, with the rounding sequence of dia_rows.hpp), and the order of the gates is kept, so the
// result is bitwise equal to applying the gates one by one with dq_kron_apply_device (accumulate = 0, in place). The
// plan copies the gates' values: the gates may be freed after planning.
#include <algorithm>
#include <cmath>
#include <limits>
#include <utility>
#include <vector>

#include "dia_rows.hpp"
#include "dq_common.hpp"

namespace dq {

constexpr int GATES_MAX_K = 4;      // gates on up to four qubits (16 x 16)
constexpr int PASS_MAX_GATES = 64;  // gates per pass
constexpr int PASS_MAX_DIAG = 512;  // entries of a pass's diagonal gates, staged in LDS
constexpr int GATE_MAX_TERMS = 512; // nonzero terms of one gate

// One step of a pass. Non-diagonal gates on three or four qubits are no steps: they get a pass of their own, run by
// the single-gate kernel.
// Two kinds take several gates: where the code of different kinds meets the compiler copies every amplitude, so a stretch
// of gates without a meeting point costs less than its steps one by one.
enum { STEP_MOVE = 0, STEP_DIAG = 1, STEP_FULL2 = 2, STEP_ROWS2 = 3, STEP_ROWS4 = 4, STEP_RUN = 5, STEP_LAYER = 6,
       STEP_FULL4 = 7, STEP_MASK2 = 8, STEP_MASK4 = 9 };
struct GateStep {
    int kind;
    int a;     // STEP_MOVE: the new window; STEP_DIAG: which register bits the gate's qubits are (see diag_step)
    int q, k;  // STEP_DIAG: first qubit, qubits; STEP_LAYER: k = 1 where all are cross gates
    int j;     // the gate's first register bit; STEP_DIAG: the gate bit of register bit `a`
    int at;    // STEP_DIAG: its first entry in the pass's LDS table; STEP_FULL*, STEP_MASK*: its entries (row-major,
               // absent ones too) in terms;
               // STEP_LAYER: the entries of full one-qubit gates on register bits 0 .. R - 1, one after the other
    int end;   // STEP_ROWS*: its terms of a row, from `at` on; STEP_MASK*: bit r * rows + c: entry (r, c) is a term;
               // STEP_RUN: this and the next end - 1 steps are diagonal gates on no register bit
    int pad_;
};

struct PassHdr {
    int n_steps, n_diag, nc, a0;  // steps; entries of the LDS table; qubits outside the tile; the first window
    int single, single_q;      // single >= 0: this pass is gate `single` of the plan's own copies, on qubits from single_q
    int tpos[16];              // tile bit i -> global qubit (ascending)
    int cpos[48];              // tile index bit m -> global qubit, for the qubits outside the tile (ascending)
    int64_t step, diag;        // first step / diagonal entry of this pass in the plan's arrays
    // Where a wave's amplitudes may leave the finite ones (stay_finite) it takes the "wild" steps, n_steps further on: every
    // gate by itself, by its terms (STEP_ROWS*). check = 0: no step needs finite amplitudes, there are no others.
    int check, pad_;
    double limit;              // the bound of stay_finite
};

template <typename T>
struct GateTerm {
    T re, im;
    int rc, pad_;  // the column, -1: no term (STEP_ROWS*)
};
template <typename T>
struct GateVal {
    T re, im;
};

// f(0), .., f(N - 1) with constant arguments: the amplitude arrays stay in registers only if every index is a constant.
template <typename F, int... I>
__device__ __forceinline__ void static_for_seq(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_seq(f, std::make_integer_sequence<int, N>{});
}

// Ends the code of one of several window variants: the variants' stores would otherwise be merged into one sequence
// over a choice of addresses, which puts the amplitudes into memory.
#define DQ_VARIANT_END(id) asm volatile("; variant %0" ::"n"(id))

// LDS place of tile element e: one value of padding per 16, so that every window's lanes hit different banks. The
// register and lane parts of e have no bit in common, so their places add up.
__device__ inline int tile_place(int e) { return e + (e >> 4); }

// Tile element of lane t with register index 0 in window a.
template <int R>
__device__ inline int lane_elem_of(int t, int a) {
    return (t & ((1 << a) - 1)) | ((t >> a) << (a + R));
}

// Global index bits of lane t's part of the tile in window a.
template <int R>
__device__ inline int64_t lane_index(const PassHdr &P, int t, int a) {
    int64_t v = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) v |= static_cast<int64_t>((t >> i) & 1) << P.tpos[i < a ? i : i + R];
    return v;
}

// Global index bits of register index m in window a (uniform).
template <int R>
__device__ inline int64_t reg_index(const PassHdr &P, int m, int a) {
    int64_t v = 0;
#pragma unroll
    for (int b = 0; b < R; ++b) v |= static_cast<int64_t>((m >> b) & 1) << P.tpos[a + b];
    return v;
}

// x = v x with the single-gate kernel's rounding, but for the sign of a zero: its sums start at +0, so its zeros are +0.
// Signs of zeros change no other value, so one plus_zero before the store gives its bits.
// The fmas write over x: left to itself the compiler accumulates into the product and copies the result back, two moves
// per amplitude and gate.
__device__ __forceinline__ void fma_over(double &x, double a, double c) {  // x = a x + c
    asm("v_fma_f64 %0, %1, %0, %2" : "+v"(x) : "v"(a), "v"(c));
}
__device__ __forceinline__ void fma_over(float &x, float a, float c) {
    asm("v_fma_f32 %0, %1, %0, %2" : "+v"(x) : "v"(a), "v"(c));
}
template <typename T>
__device__ __forceinline__ void scale_amp(const GateVal<T> &v, T &xr, T &xi) {
    const T nr = -(v.im * xi), ni = v.im * xr;
    fma_over(xr, v.re, nr);
    fma_over(xi, v.re, ni);
}
template <typename T>
__device__ __forceinline__ T plus_zero(T v) {
    return v + T(0);
}

// A diagonal gate. ct: the lane's part of the gate's index. S.a = 0: no register bit is one of its qubits; 1 + b:
// register bit b alone is (its gate bit S.j); 1 + R + b: register bits b and b + 1 are gate bits 0 and 1; else
// (a gate on three or four qubits) S.j holds, per register bit, 1 + its gate bit in 4 bits.
template <typename T, int R, int B>
__device__ __forceinline__ void diag_step(const GateStep &S, const GateVal<T> *tab, int ct, T (&xr)[1 << R],
                                          T (&xi)[1 << R]) {
    constexpr int E = 1 << R;
    if constexpr (B < R) {
        if (S.a == 1 + B) {
            const GateVal<T> v0 = tab[ct], v1 = tab[ct | (1 << S.j)];
            static_for<E>([&](auto m) { scale_amp((m >> B) & 1 ? v1 : v0, xr[m], xi[m]); });
            DQ_VARIANT_END(B);
        } else if (B + 1 < R && S.a == 1 + R + B) {
            const GateVal<T> v0 = tab[ct], v1 = tab[ct | 1], v2 = tab[ct | 2], v3 = tab[ct | 3];
            static_for<E>([&](auto m) {
                constexpr int c = (m >> B) & 3;
                scale_amp(c == 0 ? v0 : c == 1 ? v1 : c == 2 ? v2 : v3, xr[m], xi[m]);
            });
            DQ_VARIANT_END(16 + B);
        } else {
            diag_step<T, R, B + 1>(S, tab, ct, xr, xi);
        }
    } else if (S.a == 0) {
        const GateVal<T> v = tab[ct];
        static_for<E>([&](auto m) { scale_amp(v, xr[m], xi[m]); });
        DQ_VARIANT_END(32);
    } else {
        static_for<E>([&](auto m) {
            int c = ct;
            for (int b = 0; b < R; ++b) {
                const int g = (S.j >> (4 * b)) & 15;
                if (((m >> b) & 1) && g) c |= 1 << (g - 1);
            }
            scale_amp(tab[c], xr[m], xi[m]);
        });
        DQ_VARIANT_END(33);
    }
}

// A one-qubit gate with all four entries g (row-major) on register bit B.
template <typename T, int R, int B>
__device__ __forceinline__ void full2_gate(const GateTerm<T> *__restrict__ g, T (&xr)[1 << R], T (&xi)[1 << R]) {
    const T g0r = g[0].re, g0i = g[0].im, g1r = g[1].re, g1i = g[1].im;
    const T g2r = g[2].re, g2i = g[2].im, g3r = g[3].re, g3i = g[3].im;
    static_for<(1 << R) / 2>([&](auto c) {
        constexpr int m = (c & ((1 << B) - 1)) | ((c >> B) << (B + 1)), n = m | (1 << B);
        // a compensated FP32 sum of two finite terms is their plain sum
        T ar, ai, br, bi, cr, ci, dr, di;
        cmul(g0r, g0i, xr[m], xi[m], ar, ai);
        cmul(g1r, g1i, xr[n], xi[n], br, bi);
        cmul(g2r, g2i, xr[m], xi[m], cr, ci);
        cmul(g3r, g3i, xr[n], xi[n], dr, di);
        xr[m] = ar + br;
        xi[m] = ai + bi;
        xr[n] = cr + dr;
        xi[n] = ci + di;
    });
}

// A cross gate: real diagonal entries, imaginary others (a rotation about X). The products with the zero parts, which
// full2_gate adds as zeros, are left out: 12 instructions for a pair of amplitudes against 20, with the same roundings and,
// while every amplitude is finite, the same values (a TFIM step of 28 qubits 7.13 -> 6.81 ms, of 25 789 -> 744 us).
template <typename T, int R, int B>
__device__ __forceinline__ void cross_gate(const GateTerm<T> *__restrict__ g, T (&xr)[1 << R], T (&xi)[1 << R]) {
#pragma clang fp contract(off)
    const T c0 = g[0].re, s1 = g[1].im, s2 = g[2].im, c3 = g[3].re;
    static_for<(1 << R) / 2>([&](auto c) {
#pragma clang fp contract(off)
        constexpr int m = (c & ((1 << B) - 1)) | ((c >> B) << (B + 1)), n = m | (1 << B);
        const T ar = c0 * xr[m], ai = c0 * xi[m], br = s1 * xi[n], bi = s1 * xr[n];
        const T cr = s2 * xi[m], ci = s2 * xr[m], dr = c3 * xr[n], di = c3 * xi[n];
        xr[m] = ar - br;
        xi[m] = ai + bi;
        xr[n] = dr - cr;
        xi[n] = ci + di;
    });
}

// Whether a lane's amplitudes and all that a pass makes of them stay finite: then zeros may be left out of a sum, and
// a compensated sum of two terms is their plain sum (it is NaN where the first one is infinite). A gate makes the largest
// real or imaginary part at most as many times larger as the entries of a row add up to (absolute real and imaginary
// parts); `limit` is the largest finite value over the product of these factors, with room for the roundings. False for a
// NaN. A wave looks when it has loaded a tile and after each move: FP64 2^(R+1) additions, FP32 half as many maxima. It
// replaces a look per cross layer (FP32, 28 qubits: a TFIM step 4.79 -> 4.72 ms) and is new to passes of general gates in
// FP32 (14 gates on every other qubit in 2 passes 2.01 -> 2.09 ms).
template <typename T, int E>
__device__ __forceinline__ bool stay_finite(const T (&xr)[E], const T (&xi)[E], T limit) {
    T a = T(0), b = T(0);
    static_for<E / 2>([&](auto h) {
        constexpr int m = 2 * h;
        const T w = __builtin_elementwise_abs(xr[m]), x = __builtin_elementwise_abs(xi[m]);
        const T y = __builtin_elementwise_abs(xr[m + 1]), z = __builtin_elementwise_abs(xi[m + 1]);
        if constexpr (sizeof(T) == 4) {  // the largest (NaN if one is), two values an instruction
            a = __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, w), x);
            b = __builtin_elementwise_maximum(__builtin_elementwise_maximum(b, y), z);
        } else {
            a += w;
            b += x;
            a += y;
            b += z;
        }
    });
    return a + b < limit;
}

// The same on register bit j.
template <typename T, int R, int B>
__device__ __forceinline__ void full2_step(int j, const GateTerm<T> *__restrict__ g, T (&xr)[1 << R],
                                           T (&xi)[1 << R]) {
    if constexpr (B < R) {
        if (j != B) {
            full2_step<T, R, B + 1>(j, g, xr, xi);
            return;
        }
        full2_gate<T, R, B>(g, xr, xi);
        DQ_VARIANT_END(48 + B);
    }
}

// A gate of 2^K rows on register bits [j, j + K) whose rows take their terms in ascending column order: the entries g
// are row-major, entry (r, c) is a term where bit r * rows + c of mask is set (FULL: all are). The lane's columns are
// taken in two halves, whose sums fit beside the amplitudes.
template <typename T, int R, int K, bool FULL, int B>
__device__ __forceinline__ void grid_step(int j, int mask, const GateTerm<T> *__restrict__ g, T (&xr)[1 << R],
                                          T (&xi)[1 << R]) {
    if constexpr (B + K <= R) {
        if (j != B) {
            grid_step<T, R, K, FULL, B + 1>(j, mask, g, xr, xi);
            return;
        }
        constexpr int G = 1 << K, NC = 1 << (R - K), H = NC < 2 ? NC : NC / 2;
        static_for<NC / H>([&](auto half) {
            Acc<T> ar[H][G], ai[H][G];
            static_for<G>([&](auto r) {
                static_for<G>([&](auto c) {
                    if (FULL || ((mask >> (r * G + c)) & 1)) {  // uniform
                        const T wr = g[r * G + c].re, wi = g[r * G + c].im;
                        static_for<H>([&](auto u) {
                            constexpr int col = half * H + u;
                            constexpr int at = (col & ((1 << B) - 1)) | ((col >> B) << (B + K)) | (c << B);
                            if constexpr (FULL && c == 0) {  // the first term: adding it to 0 changes a zero's sign only
                                cmul(wr, wi, xr[at], xi[at], ar[u][r].s, ai[u][r].s);
                            } else {
                                cmac(ar[u][r], ai[u][r], wr, wi, xr[at], xi[at]);
                            }
                        });
                        if constexpr (!FULL) DQ_VARIANT_END(4096 + 64 * half + r * G + c);
                    }
                });
            });
            static_for<H>([&](auto u) {
                constexpr int col = half * H + u;
                static_for<G>([&](auto r) {
                    constexpr int at = (col & ((1 << B) - 1)) | ((col >> B) << (B + K)) | (r << B);
                    xr[at] = ar[u][r].get();
                    xi[at] = ai[u][r].get();
                });
            });
        });
        DQ_VARIANT_END(128 + 32 * K + 16 * (FULL ? 1 : 0) + B);
    }
}

// A gate of 2^K rows on register bits [j, j + K), its terms listed row by row in slot order, `per` of them to a row (a
// multiple of 2^K; column rc, -1: none). 2^K terms are read at once, and each is matched against 2^K columns. One by one and
// against every entry of the gate, two-qubit gates in descending slot order took, FP64 / FP32, on 18 qubits 46 / 48 us, on 20
// 102 / 94, on 22 211 / 152, on 25 1188 / 977; so 36 / 38, 81 / 71, 158 / 119 and 901 / 691. (Reading a row ahead spills.) The
// lane's columns are taken in two halves, whose sums fit beside the amplitudes.
template <typename T, int R, int K, int B>
__device__ __forceinline__ void rows_step(int j, int t0, int per, const GateTerm<T> *__restrict__ terms,
                                          T (&xr)[1 << R], T (&xi)[1 << R]) {
    if constexpr (B + K <= R) {
        if (j != B) {
            rows_step<T, R, K, B + 1>(j, t0, per, terms, xr, xi);
            return;
        }
        constexpr int G = 1 << K, NC = 1 << (R - K), H = NC < 2 ? NC : NC / 2;  // H columns per half
        static_for<NC / H>([&](auto half) {
            Acc<T> ar[H][G], ai[H][G];
            static_for<G>([&](auto r) {
                for (int t = t0 + r * per; t < t0 + (r + 1) * per; t += G) {  // uniform
                    GateTerm<T> w[G];
                    static_for<G>([&](auto i) { w[i] = terms[t + i]; });
                    static_for<G>([&](auto i) {
                        static_for<G>([&](auto c) {
                            if (w[i].rc == c) {  // uniform
                                static_for<H>([&](auto u) {
                                    constexpr int col = half * H + u;
                                    constexpr int at = (col & ((1 << B) - 1)) | ((col >> B) << (B + K)) | (c << B);
                                    cmac(ar[u][r], ai[u][r], w[i].re, w[i].im, xr[at], xi[at]);
                                });
                                DQ_VARIANT_END(1024 + 256 * half + 64 * r + 8 * i + c);
                            }
                        });
                    });
                }
            });
            static_for<H>([&](auto u) {
                constexpr int col = half * H + u;
                static_for<G>([&](auto r) {
                    constexpr int at = (col & ((1 << B) - 1)) | ((col >> B) << (B + K)) | (r << B);
                    xr[at] = ar[u][r].get();
                    xi[at] = ai[u][r].get();
                });
            });
        });
        DQ_VARIANT_END(64 + 16 * K + B);
    }
}

// At least three waves per SIMD: 12-qubit tiles at 172 VGPRs had two, and the passes above took 3.69 and 2.62 ms.
template <typename T, int L>
__global__ __launch_bounds__(256, 3) void gates_pass_kernel(const PassHdr *__restrict__ hdr,
                                                         const GateStep *__restrict__ steps,
                                                         const GateTerm<T> *__restrict__ terms,
                                                         const GateVal<T> *__restrict__ diag, T *re, T *im,
                                                         int64_t ntiles) {
    constexpr int R = L - 8, E = 1 << R;
    __shared__ T buf[(1 << L) + (1 << L) / 16];
    __shared__ GateVal<T> tab[PASS_MAX_DIAG];
    const PassHdr &P = *hdr;
    const int tid = threadIdx.x;
    for (int i = tid; i < P.n_diag; i += 256) tab[i] = diag[P.diag + i];
    const GateStep *__restrict__ st = steps + P.step;
    const T limit = static_cast<T>(P.limit);
    __syncthreads();
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        int64_t base = 0;
        for (int i = 0; i < P.nc; ++i) base |= ((t >> i) & 1) << P.cpos[i];
        int a = P.a0;
        asm volatile("" : "+s"(a));  // 2^R register offsets per window: made again per tile, not kept from tile to tile
        int64_t idx = base | lane_index<R>(P, tid, a);
        T xr[E], xi[E];
        static_for<E>([&](auto m) {
            const int64_t om = reg_index<R>(P, m, a);
            xr[m] = (re + om)[idx];
            xi[m] = (im + om)[idx];
        });
        // 0, or n_steps: the wave takes the wild steps, until a move brings it other amplitudes
        int wild = P.check && __any(!stay_finite(xr, xi, limit)) ? P.n_steps : 0;
        for (int s = 0; s < P.n_steps; ++s) {  // uniform
            const GateStep S = st[s + wild];
            if (S.kind == STEP_RUN) {
                for (int i = 0; i < S.end; ++i) {  // uniform
                    const GateStep D = st[s + i];
                    const int ct = static_cast<int>(idx >> D.q) & ((1 << D.k) - 1);
                    const GateVal<T> v = tab[D.at + ct];
                    static_for<E>([&](auto m) { scale_amp(v, xr[m], xi[m]); });
                }
                s += S.end - 1;
                DQ_VARIANT_END(40);
            } else if (S.kind == STEP_LAYER) {
                if (S.k) {
                    static_for<R>([&](auto b) { cross_gate<T, R, b>(terms + S.at + 4 * b, xr, xi); });
                    DQ_VARIANT_END(42);
                } else {
                    static_for<R>([&](auto b) { full2_gate<T, R, b>(terms + S.at + 4 * b, xr, xi); });
                    DQ_VARIANT_END(41);
                }
                s += R - 1;
            } else if (S.kind == STEP_DIAG) {
                const int ct = static_cast<int>(idx >> S.q) & ((1 << S.k) - 1);
                diag_step<T, R, 0>(S, tab + S.at, ct, xr, xi);
            } else if (S.kind == STEP_FULL2) {
                full2_step<T, R, 0>(S.j, terms + S.at, xr, xi);
            } else if (S.kind == STEP_FULL4) {
                grid_step<T, R, 2, true, 0>(S.j, 0, terms + S.at, xr, xi);
            } else if (S.kind == STEP_MASK2) {
                grid_step<T, R, 1, false, 0>(S.j, S.end, terms + S.at, xr, xi);
            } else if (S.kind == STEP_MASK4) {
                grid_step<T, R, 2, false, 0>(S.j, S.end, terms + S.at, xr, xi);
            } else if (S.kind == STEP_MOVE) {
                const int to = S.a;
                const int w = tile_place(lane_elem_of<R>(tid, a)), r = tile_place(lane_elem_of<R>(tid, to));
                static_for<E>([&](auto m) { buf[w + tile_place(m << a)] = xr[m]; });
                __syncthreads();
                static_for<E>([&](auto m) { xr[m] = buf[r + tile_place(m << to)]; });
                __syncthreads();
                static_for<E>([&](auto m) { buf[w + tile_place(m << a)] = xi[m]; });
                __syncthreads();
                static_for<E>([&](auto m) { xi[m] = buf[r + tile_place(m << to)]; });
                __syncthreads();  // the next move, of this tile or the next, writes the buffer again
                a = to;
                idx = base | lane_index<R>(P, tid, a);
                wild = P.check && __any(!stay_finite(xr, xi, limit)) ? P.n_steps : 0;
            } else if (S.kind == STEP_ROWS2) {
                rows_step<T, R, 1, 0>(S.j, S.at, S.end, terms, xr, xi);
            } else {
                rows_step<T, R, 2, 0>(S.j, S.at, S.end, terms, xr, xi);
            }
        }
        static_for<E>([&](auto m) {
            const int64_t om = reg_index<R>(P, m, a);
            (re + om)[idx] = plus_zero(xr[m]);
            (im + om)[idx] = plus_zero(xi[m]);
        });
    }
}

}  // namespace dq

// A planned gate sequence: passes, steps, terms and diagonal entries (copies of the gates' values), built
// once and run any number of times.
struct dq_gate_plan {
    int n_qubits = 0, precision = DQ_F64, L = 11;
    std::vector<dq::PassHdr> passes;
    std::vector<std::unique_ptr<dq_devmat>> big;  // copies of the non-diagonal gates on three or four qubits
    dq::DevBuf d_passes, d_steps, d_terms, d_diag;
};

namespace dq {

static int g_gates_tile_qubits = 0;  // dq_set_tuning "gates_tile_qubits": 10, 11 or 12; 0 = automatic
static int g_gates_low_qubits = 0;   // dq_set_tuning "gates_low_qubits": 4, 5 or 6 (qubits always in a tile); 0 = automatic

bool gates_set_tuning(const std::string &key, int value) {
    if (key == "gates_kernel") {  // kept for callers: there is one pass kernel
        if (value != 0 && value != 1) throw ArgError("gates_kernel must be 0 or 1");
        return true;
    }
    if (key == "gates_low_qubits") {
        if (value != 0 && (value < 4 || value > 6)) throw ArgError("gates_low_qubits must be 0 (automatic), 4, 5 or 6");
        g_gates_low_qubits = value;
        return true;
    }
    if (key != "gates_tile_qubits") return false;
    if (value != 0 && (value < 10 || value > 12))
        throw ArgError("gates_tile_qubits must be 0 (automatic), 10, 11 or 12");
    g_gates_tile_qubits = value;
    return true;
}

static int gate_qubits(const dq_devmat &G) {
    if (G.rows != G.cols) throw ArgError("gates: every gate must be square");
    int k = 0;
    while ((1u << k) < G.rows) ++k;
    if ((1u << k) != G.rows || k < 1 || k > GATES_MAX_K)
        throw ArgError("gates: a gate must be 2^k x 2^k with 1 <= k <= 4");
    return k;
}

// One gate on the host: qubits, and its terms row by row in slot order.
struct HostGate {
    int k = 0, q = 0;
    bool diag = false;
    std::vector<int> rowptr;                // g + 1
    std::vector<int> col;                   // per term
    std::vector<double> vre, vim;           // per term (exact copies of the gate's FP64 or FP32 values)
};

static HostGate host_gate(const dq_devmat &G, int k, int q) {
    HostGate H;
    H.k = k;
    H.q = q;
    H.diag = G.n() == 1 && G.offs[0] == 0;
    const int g = 1 << k;
    const size_t eb = elem_bytes(G.precision);
    std::vector<char> re(G.total * eb), im(G.total * eb);
    if (G.total) {
        DQ_HIP(hipMemcpy(re.data(), G.re.p, re.size(), hipMemcpyDeviceToHost));
        DQ_HIP(hipMemcpy(im.data(), G.im.p, im.size(), hipMemcpyDeviceToHost));
    }
    auto val = [&](const std::vector<char> &v, int64_t i) {
        return G.precision == DQ_F64 ? reinterpret_cast<const double *>(v.data())[i]
                                     : static_cast<double>(reinterpret_cast<const float *>(v.data())[i]);
    };
    H.rowptr.push_back(0);
    for (int r = 0; r < g; ++r) {
        for (int s = 0; s < G.n(); ++s) {
            const DiagMeta &m = G.meta[s];
            if (r >= m.rlo && r < m.rhi) {
                H.col.push_back(r + m.off);
                H.vre.push_back(val(re, m.rowbase + r));
                H.vim.push_back(val(im, m.rowbase + r));
            }
        }
        H.rowptr.push_back(static_cast<int>(H.col.size()));
    }
    return H;
}

// Where window [a, a + R) starts for a gate on tile bits [p, p + k), given the non-diagonal gates that follow it in the
// pass (first tile bit, qubits): the place that holds the most of them, the highest of those (windows from bit 4 up
// keep runs of 16 amplitudes in the lanes, so the pass can store from them).
static int best_window(const std::vector<std::pair<int, int>> &gates, size_t i, int L, int R) {
    const int p = gates[i].first, k = gates[i].second;
    int best = -1, held = -1;
    for (int a = std::max(0, p + k - R); a <= std::min(p, L - R); ++a) {
        int n = 0;
        for (size_t j = i; j < gates.size() && gates[j].first >= a && gates[j].first + gates[j].second <= a + R; ++j) ++n;
        if (n >= held) {
            held = n;
            best = a;
        }
    }
    return best;
}

// Makes stretches of the steps from `from` on one step of several gates, which the pass skips to the end of: diagonal gates
// on no register bit a STEP_RUN, full one-qubit gates on register bits 0, 1, .. R - 1 in turn (whose entries follow each
// other) a STEP_LAYER. A layer of cross gates alone (cross_gate) has k = 1.
template <typename T>
static void merge_steps(std::vector<GateStep> &steps, size_t from, int R, const std::vector<GateTerm<T>> &terms) {
    auto cross = [&](int at) {
        const GateTerm<T> *g = terms.data() + at;
        return g[0].im == T(0) && g[3].im == T(0) && g[1].re == T(0) && g[2].re == T(0);
    };
    for (size_t i = from; i < steps.size();) {
        GateStep &first = steps[i];
        size_t e = i;
        while (e < steps.size() && steps[e].kind == STEP_DIAG && steps[e].a == 0) ++e;
        if (e > i) {
            first.kind = STEP_RUN;
            first.end = static_cast<int>(e - i);
            i = e;
            continue;
        }
        while (e < steps.size() && e - i < static_cast<size_t>(R) && steps[e].kind == STEP_FULL2 &&
               steps[e].j == static_cast<int>(e - i) && steps[e].at == first.at + 4 * static_cast<int>(e - i))
            ++e;
        if (e - i == static_cast<size_t>(R)) {
            first.kind = STEP_LAYER;
            first.k = 1;
            for (int b = 0; b < R; ++b)
                if (!cross(first.at + 4 * b)) first.k = 0;
            i = e;
        } else {
            ++i;
        }
    }
}

// Greedy cut of the sequence into passes: a non-diagonal gate joins the current pass while the qubits of the pass's
// non-diagonal gates, together with qubits 0..low-1, number at most L, and while the pass's diagonal entries fit in LDS.
template <typename T>
static void plan_passes(dq_gate_plan &P, int low_qubits, const std::vector<HostGate> &gates,
                        const std::vector<const dq_devmat *> &devgates) {
    const int n = P.n_qubits, L = P.L, R = L - 8;
    std::vector<GateStep> steps;
    std::vector<GateTerm<T>> terms;
    std::vector<GateVal<T>> diag;
    // the most by which the largest real or imaginary part can grow
    auto growth = [](const HostGate &H) {
        double most = 1.0;
        for (size_t r = 0; r + 1 < H.rowptr.size(); ++r) {
            double row = 0.0;
            for (int t = H.rowptr[r]; t < H.rowptr[r + 1]; ++t) row += std::fabs(H.vre[t]) + std::fabs(H.vim[t]);
            if (!(row <= most)) most = row;  // a NaN stays
        }
        return most;
    };
    auto close = [&](int g0, int g1, uint64_t S) {
        if (g1 <= g0) return;
        uint64_t Tm = S;
        for (int b = 0; b < n && __builtin_popcountll(Tm) < L; ++b) Tm |= uint64_t(1) << b;
        PassHdr D{};
        D.single = -1;
        int i = 0, c = 0;
        for (int b = 0; b < n; ++b) {
            if ((Tm >> b) & 1) D.tpos[i++] = b;
            else D.cpos[c++] = b;
        }
        D.nc = c;
        D.step = static_cast<int64_t>(steps.size());
        D.diag = static_cast<int64_t>(diag.size());
        std::vector<std::pair<int, int>> moving;  // the non-diagonal gates' tile bits (consecutive, as their qubits are)
        for (int j = g0; j < g1; ++j) {
            if (gates[j].diag) continue;
            int pos = 0;
            while (D.tpos[pos] != gates[j].q) ++pos;
            moving.push_back({pos, gates[j].k});
        }
        const int stored = L - R;  // the last window
        int a = stored;
        if (!moving.empty()) {
            const int w = best_window(moving, 0, L, R);
            if (w >= 4) a = w;
        }
        D.a0 = a;
        std::vector<GateStep> wild;          // the pass's steps for tiles that may leave the finite amplitudes
        std::vector<GateTerm<T>> listed;     // and their terms, in slot order
        bool needs_finite = false;
        size_t im = 0;
        for (int j = g0; j < g1; ++j) {
            const HostGate &H = gates[j];
            GateStep st{};
            if (H.diag) {
                st.kind = STEP_DIAG;
                st.q = H.q;
                st.k = H.k;
                st.at = static_cast<int>(static_cast<int64_t>(diag.size()) - D.diag);
                int bits = 0, first = -1, packed = 0;
                for (int b = 0; b < R; ++b) {
                    const int g = D.tpos[a + b] - H.q;  // gate bit of register bit b
                    if (g < 0 || g >= H.k) continue;
                    ++bits;
                    if (first < 0) first = b;
                    packed |= (g + 1) << (4 * b);
                }
                if (bits == 0) {
                    st.a = 0;
                } else if (bits == 1) {
                    st.a = 1 + first;
                    st.j = D.tpos[a + first] - H.q;
                } else if (bits == 2 && H.k == 2) {  // tile bits ascend with the qubits: gate bits 0 and 1
                    st.a = 1 + R + first;
                } else {
                    st.a = 1 + 2 * R;
                    st.j = packed;
                }
                for (size_t t = 0; t < H.col.size(); ++t)
                    diag.push_back(GateVal<T>{static_cast<T>(H.vre[t]), static_cast<T>(H.vim[t])});
            } else {
                const auto [p, k] = moving[im];
                if (p < a || p + k > a + R) {
                    GateStep mv{};
                    mv.kind = STEP_MOVE;
                    mv.a = a = best_window(moving, im, L, R);
                    steps.push_back(mv);
                    wild.push_back(mv);
                }
                ++im;
                st.j = p - a;
                const int t0 = static_cast<int>(terms.size()), l0 = static_cast<int>(listed.size());
                // rows whose terms ascend in column order (finite sums of two terms have the same bits in either order)
                // need no list of terms, only which entries they are
                const int g = 1 << k;
                bool distinct = true, ascending = true;
                int most = g;
                for (int r = 0; r < g; ++r) {
                    most = std::max(most, H.rowptr[r + 1] - H.rowptr[r]);
                    for (int t = H.rowptr[r] + 1; t < H.rowptr[r + 1]; ++t) {
                        distinct = distinct && H.col[t] != H.col[t - 1];
                        ascending = ascending && H.col[t] > H.col[t - 1];
                    }
                }
                distinct = distinct && most == g;
                const int per = (most + g - 1) / g * g;
                for (int r = 0; r < g; ++r) {
                    for (int t = H.rowptr[r]; t < H.rowptr[r + 1]; ++t)
                        listed.push_back(
                            GateTerm<T>{static_cast<T>(H.vre[t]), static_cast<T>(H.vim[t]), H.col[t], 0});
                    listed.resize(static_cast<size_t>(l0) + (r + 1) * per, GateTerm<T>{T(0), T(0), -1, 0});
                }
                GateStep by_terms = st;
                by_terms.kind = k == 1 ? STEP_ROWS2 : STEP_ROWS4;
                by_terms.at = l0;
                by_terms.end = per;
                if (distinct && (k == 1 || ascending)) {
                    terms.resize(terms.size() + static_cast<size_t>(g) * g, GateTerm<T>{T(0), T(0), 0, 0});
                    int mask = 0;
                    for (int r = 0; r < g; ++r)
                        for (int t = H.rowptr[r]; t < H.rowptr[r + 1]; ++t) {
                            mask |= 1 << (r * g + H.col[t]);
                            terms[t0 + r * g + H.col[t]].re = static_cast<T>(H.vre[t]);
                            terms[t0 + r * g + H.col[t]].im = static_cast<T>(H.vim[t]);
                        }
                    const bool full = mask == (1 << (g * g)) - 1;
                    st.kind = k == 1 ? (full ? STEP_FULL2 : STEP_MASK2) : (full ? STEP_FULL4 : STEP_MASK4);
                    st.at = t0;
                    st.end = mask;
                    needs_finite = needs_finite || (sizeof(T) == 4 && (full || !ascending));
                } else {
                    st = by_terms;
                    st.at = t0;
                    terms.insert(terms.end(), listed.begin() + l0, listed.end());
                }
                wild.push_back(by_terms);
            }
            if (H.diag) wild.push_back(st);
            steps.push_back(st);
        }
        merge_steps(steps, static_cast<size_t>(D.step), R, terms);
        if (a < 4 && a != stored) {  // back to a window whose lanes hold runs of 16 amplitudes
            GateStep mv{};
            mv.kind = STEP_MOVE;
            mv.a = stored;
            steps.push_back(mv);
            wild.push_back(mv);
        }
        D.n_steps = static_cast<int>(static_cast<int64_t>(steps.size()) - D.step);
        D.n_diag = static_cast<int>(static_cast<int64_t>(diag.size()) - D.diag);
        for (size_t i = D.step; i < steps.size(); ++i)
            needs_finite = needs_finite || (steps[i].kind == STEP_LAYER && steps[i].k);
        if (needs_finite) {
            for (GateStep &w : wild)
                if (w.kind == STEP_ROWS2 || w.kind == STEP_ROWS4) w.at += static_cast<int>(terms.size());
            terms.insert(terms.end(), listed.begin(), listed.end());
            D.check = 1;
            steps.insert(steps.end(), wild.begin(), wild.end());
            double grows = 32.0;
            for (int j = g0; j < g1; ++j) grows *= growth(gates[j]);
            const bool finite = grows < std::numeric_limits<double>::infinity();  // false for a NaN
            D.limit = finite ? static_cast<double>(std::numeric_limits<T>::max()) / grows : 0.0;
        }
        P.passes.push_back(D);
    };
    const uint64_t low = (uint64_t(1) << low_qubits) - 1;
    uint64_t S = 0;
    int g0 = 0, nd = 0;
    for (int j = 0; j < static_cast<int>(gates.size()); ++j) {
        const HostGate &H = gates[j];
        if (!H.diag && H.k > 2) {  // a pass of its own: the single-gate kernel, on a copy the plan keeps
            if (devgates[j]->n() > 64) throw ArgError("gates: a gate has more than 64 diagonals");
            close(g0, j, S);
            PassHdr D{};
            D.single = static_cast<int>(P.big.size());
            D.single_q = H.q;
            P.big.push_back(copy_devmat(*devgates[j], nullptr));
            P.passes.push_back(D);
            g0 = j + 1;
            S = 0;
            nd = 0;
            continue;
        }
        const uint64_t Q = H.diag ? 0 : ((uint64_t(1) << H.k) - 1) << H.q;
        const int ht = static_cast<int>(H.col.size()), hd = H.diag ? ht : 0;
        if (ht > GATE_MAX_TERMS) throw ArgError("gates: a gate has more than 512 nonzero terms");
        if (j > g0 && (__builtin_popcountll(S | Q | low) > L || j - g0 >= PASS_MAX_GATES || nd + hd > PASS_MAX_DIAG)) {
            close(g0, j, S);
            g0 = j;
            S = 0;
            nd = 0;
        }
        S |= Q;
        nd += hd;
    }
    close(g0, static_cast<int>(gates.size()), S);
    DQ_HIP(hipDeviceSynchronize());  // the copies of the large gates are complete
    auto upload = [](DevBuf &buf, const auto &v) {
        using E = typename std::decay_t<decltype(v)>::value_type;
        buf = DevBuf(sizeof(E) * std::max<size_t>(1, v.size()));
        if (!v.empty()) DQ_HIP(hipMemcpy(buf.p, v.data(), sizeof(E) * v.size(), hipMemcpyHostToDevice));
    };
    upload(P.d_passes, P.passes);
    upload(P.d_steps, steps);
    upload(P.d_terms, terms);
    upload(P.d_diag, diag);
}

template <typename T>
static void run_passes(const dq_gate_plan &P, void *re, void *im, hipStream_t s) {
    const int64_t ntiles = int64_t(1) << (P.n_qubits - P.L);
    // four tiles or more per workgroup of a large state: with sixteen the last workgroups left a tenth of the chip idle
    // (28 qubits 7.15 -> 7.07 ms, FP32 4.91 -> 4.79, 25 qubits 804 -> 781 us)
    const unsigned grid = blocks_for(ntiles, 1, 16384);
    for (size_t i = 0; i < P.passes.size(); ++i) {
        if (P.passes[i].single >= 0) {
            const dq_devmat &G = *P.big[P.passes[i].single];
            int k = 0;
            while ((1u << k) < G.rows) ++k;
            const int q = P.passes[i].single_q;
            kron_apply(G, P.n_qubits - q - k, q, re, im, re, im, false, s);
            continue;
        }
#define DQ_GATES_PASS(LL)                                                                                           \
    hipLaunchKernelGGL((gates_pass_kernel<T, LL>), dim3(grid), dim3(256), 0, s, P.d_passes.as<PassHdr>() + i,        \
                       P.d_steps.as<GateStep>(), P.d_terms.as<GateTerm<T>>(),                                       \
                       P.d_diag.as<GateVal<T>>(), static_cast<T *>(re), static_cast<T *>(im), ntiles)
        if (P.L == 10) DQ_GATES_PASS(10);
        else if (P.L == 12) DQ_GATES_PASS(12);
        else DQ_GATES_PASS(11);
#undef DQ_GATES_PASS
        DQ_LAUNCH_CHECK();
    }
}

}  // namespace dq

using namespace dq;

extern "C" int dq_gate_plan_create(int n_qubits, int n_gates, const dq_devmat *const *gates,
                                   const uint32_t *first_qubit, dq_gate_plan **out) {
    return guard([&] {
        if (!out) throw ArgError("out is NULL");
        if (n_gates < 1 || !gates || !first_qubit) throw ArgError("gates: need at least one gate");
        // Small states want many small tiles (a TFIM step on 14 qubits: 18, 20, 24 us with 10, 11, 12 tile qubits; 19
        // two-qubit gates on 20 qubits: 65, 68, 80 us), large ones few passes (TFIM on 20: 58, 58, 46 us; on 22: 120,
        // 121, 104; on 28: 9.7, 8.8, 6.8 ms). Four low qubits make runs of 16 amplitudes, whole 128-byte
        // lines in FP64; a fifth costs tile qubits (28 qubits: 4 passes for 3, 8.0 ms; FP32 4.6 against 4.7 ms).
        const int L = g_gates_tile_qubits ? g_gates_tile_qubits : n_qubits >= 21 ? 12 : n_qubits >= 19 ? 11 : 10;
        const int low = g_gates_low_qubits ? g_gates_low_qubits : 4;
        const int least = g_gates_tile_qubits ? g_gates_tile_qubits : 11;
        if (n_qubits < least || n_qubits > 40)
            throw ArgError("gates: n_qubits must be in [" + std::to_string(least) + ", 40] (smaller states: "
                           "dq_kron_apply_device per gate)");
        auto P = std::make_unique<dq_gate_plan>();
        P->n_qubits = n_qubits;
        P->L = L;
        std::vector<HostGate> hg;
        for (int j = 0; j < n_gates; ++j) {
            const dq_devmat *G = gates[j];
            if (!G) throw ArgError("gates: NULL gate");
            const int k = gate_qubits(*G);
            if (j == 0) P->precision = G->precision;
            else if (G->precision != P->precision) throw ArgError("gates: all gates need one precision");
            if (first_qubit[j] + k > static_cast<uint32_t>(n_qubits)) throw ArgError("gates: gate beyond n_qubits");
            hg.push_back(host_gate(*G, k, static_cast<int>(first_qubit[j])));
        }
        std::vector<const dq_devmat *> dg(gates, gates + n_gates);
        if (P->precision == DQ_F64) plan_passes<double>(*P, low, hg, dg);
        else plan_passes<float>(*P, low, hg, dg);
        *out = P.release();
    });
}

extern "C" int dq_gate_plan_passes(const dq_gate_plan *plan, int *n_passes) {
    return guard([&] {
        if (!plan || !n_passes) throw ArgError("NULL argument");
        *n_passes = static_cast<int>(plan->passes.size());
    });
}

extern "C" int dq_gate_plan_run(const dq_gate_plan *plan, void *re, void *im, int repetitions, uintptr_t stream) {
    return guard([&] {
        if (!plan) throw ArgError("plan is NULL");
        if (!re || !im) throw ArgError("gates: NULL state");
        if (repetitions < 0) throw ArgError("gates: repetitions must be >= 0");
        hipStream_t s = as_stream(stream);
        for (int r = 0; r < repetitions; ++r) {
            if (plan->precision == DQ_F64) run_passes<double>(*plan, re, im, s);
            else run_passes<float>(*plan, re, im, s);
        }
    });
}

extern "C" void dq_gate_plan_destroy(dq_gate_plan *plan) { delete plan; }
