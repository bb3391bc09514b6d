// The row-tile core shared by SpMV, the fused Taylor-action terms and the batched evolution.
//
// A workgroup of 256 lanes owns the rows [tile, tile + 256*RPT); lane l holds rows tile + l + 256*j, j < RPT, so each
// of the RPT loads of a wave covers 64 consecutive rows: one aligned line per diagonal and one contiguous window of x.
// The diagonal loop is uniform across the workgroup; metadata reads are scalar loads. A diagonal that misses the tile
// (or the column band [col_lo, col_hi)) is skipped by the whole workgroup.
//
// LDS x window (HALO > 0): the workgroup first copies x[tile - HALO, tile + TILE + HALO) into LDS (zero outside the
// matrix columns); every diagonal with |offset| <= HALO then reads its shifted x slice from LDS instead of memory.
// Neighbouring diagonals (a band, or the +-2^k offsets of a qubit Hamiltonian) share that window, so x crosses the
// memory hierarchy once per tile instead of once per near diagonal.
#pragma once

#include "dq_common.hpp"

namespace dq {

template <typename T>
struct Acc {
    T s = T(0);
    __device__ inline void add(T v) { s += v; }
    __device__ inline T get() const { return s; }
};

template <>
struct Acc<float> {  // Kahan-compensated FP32 sum
    float s = 0.0f, c = 0.0f;
    __device__ inline void add(float v) {
        const float y = v - c;
        const float t = s + y;
        c = (t - s) - y;
        s = t;
    }
    __device__ inline float get() const { return s; }
};

// Complex product (a_r + i a_i)(x_r + i x_i) with one fixed rounding sequence -- re = fma(a_r, x_r, -(a_i x_i)),
// im = fma(a_r, x_i, a_i x_r) -- so every kernel instantiation and schedule (tile size, load order) rounds each term
// identically; left to itself the compiler may contract a*b - c*d either way round.
template <typename T>
__device__ inline void cmul(T a_r, T a_i, T x_r, T x_i, T &re, T &im) {
    re = __builtin_fma(a_r, x_r, -(a_i * x_i));
    im = __builtin_fma(a_r, x_i, a_i * x_r);
}
template <>
__device__ inline void cmul<float>(float a_r, float a_i, float x_r, float x_i, float &re, float &im) {
    re = __builtin_fmaf(a_r, x_r, -(a_i * x_i));
    im = __builtin_fmaf(a_r, x_i, a_i * x_r);
}

// Accumulate the complex product into a row's (real, imaginary) sums.
template <typename T>
__device__ inline void cmac(Acc<T> &sr, Acc<T> &si, T a_r, T a_i, T x_r, T x_i) {
    T re, im;
    cmul(a_r, a_i, x_r, x_i, re, im);
    sr.add(re);
    si.add(im);
}

// Loads of the matrix values: plain, or non-temporal (the values are streamed once, so they need not displace x from
// L2 and the Infinity Cache).
template <typename T, bool NT>
__device__ inline T ld_val(const T *p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}

// Row tile of workgroup b. xcd = 0: tile b. xcd = 1: the workgroups of one XCD (b mod 8: the hardware hands
// consecutive workgroups to the 8 XCDs in turn) take one contiguous eighth of the tiles, [x*per, (x+1)*per), so an
// XCD's L2 serves the x rows its neighbouring diagonals share; the grid is then 8*per workgroups and the surplus ones
// (tile >= ntiles) have no work.
__device__ inline int64_t tile_of_block(int64_t b, int64_t ntiles, int xcd) {
    if (!xcd) return b;
    const int64_t per = (ntiles + 7) >> 3;
    return (b & 7) * per + (b >> 3);
}

inline int64_t grid_for_tiles(int64_t ntiles, int xcd) { return xcd ? 8 * ((ntiles + 7) >> 3) : ntiles; }

// Copy x[tile - HALO, tile + TILE + HALO) into LDS (sr, si), zero outside [0, cols), then synchronise the workgroup.
template <typename T, int RPT, int HALO>
__device__ inline void stage_x_window(int64_t tile, int64_t cols, const T *__restrict__ xr, const T *__restrict__ xi,
                                      T *__restrict__ sr, T *__restrict__ si) {
    constexpr int W = 256 * RPT + 2 * HALO;
    const int64_t ws = tile - HALO;
    for (int e = threadIdx.x; e < W; e += 256) {
        const int64_t c = ws + e;
        T a = T(0), b = T(0);
        if (c >= 0 && c < cols) {
            a = xr[c];
            b = xi[c];
        }
        sr[e] = a;
        si[e] = b;
    }
    __syncthreads();
}

// Zero-block map of a DIA layout: word [job][diagonal][b / 32] holds, for the blocks of BR rows b * BR .. b * BR +
// BR - 1, a bit of x when some real part of the diagonal in those rows is nonzero and a bit of y when some imaginary
// part is (a NaN counts as nonzero). A block whose bits are both clear adds nothing to any row sum, so the row loops
// skip its value loads and x gathers: a qubit Hamiltonian's +-2^k flip diagonals are zero on alternate runs of 2^k
// rows (three runs in four for a flip-flop term). Where one part alone is zero -- a real Hamiltonian's imaginary part,
// the real part of -i t H -- its loads are replaced by the constant 0: the products are the same bits but for the
// sign of a zero, which no sum that starts at +0 keeps.
// A workgroup reads 32 blocks of one diagonal, a wave 8 of them, 64 rows at a time as one ballot per part, and each
// wave writes its byte of the two words: one streaming read of the values with 8 or more loads in flight per wave and
// no LDS. Blocks of 64 rows or more are looked at in their first 8 rows first, all of a wave's in one load a part, and read
// only where those are zero (9 dense diagonals of 2^23 rows 216 -> 63 us, TFIM-20 126 -> 110). The diagonals are strided
// over gridDim.y (at most 65535); the values of job j start at j * total.
template <typename T, int BR>
__global__ __launch_bounds__(256) void zero_blocks_kernel(int64_t rows, int n, const DiagMeta *__restrict__ meta,
                                                          int64_t total, const T *__restrict__ are,
                                                          const T *__restrict__ aim, int64_t zwords,
                                                          uint2 *__restrict__ zmask) {
    constexpr int CHUNK = 8 * BR;                     // rows of a wave
    constexpr int STEPS = (CHUNK + 63) / 64;          // ballots of a wave (CHUNK >= 128)
    constexpr int U = STEPS < 4 ? STEPS : 4;          // ballots whose loads are issued together
    const int64_t w = blockIdx.x;
    const int j = blockIdx.z;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t r0 = (w * 4 + wave) * CHUNK;
    for (int d = blockIdx.y; d < n; d += gridDim.y) {  // uniform
        const DiagMeta md = meta[d];
        const T *pr = are + static_cast<int64_t>(j) * total + md.rowbase;
        const T *pi = aim + static_cast<int64_t>(j) * total + md.rowbase;
        const int64_t lo = md.rlo, hi = min(md.rhi, rows);
        uint32_t br = 0, bi = 0;  // the wave's 8 blocks
        if (r0 < hi && r0 + CHUNK > lo) {  // uniform
            if constexpr (BR >= 64) {  // the first 8 rows of each block
                const int64_t r = r0 + BR * (lane >> 3) + (lane & 7);
                const bool in = r >= lo && r < hi;
                const T vr = in ? pr[r] : T(0), vi = in ? pi[r] : T(0);
                const uint64_t nr = __ballot(!(vr == T(0))), ni = __ballot(!(vi == T(0)));
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    if ((nr >> (8 * b)) & 0xff) br |= 1u << b;
                    if ((ni >> (8 * b)) & 0xff) bi |= 1u << b;
                }
            }
            for (int s = 0; s < STEPS; s += U) {
                constexpr int PER = BR >= 64 ? BR / 64 : 1;  // ballots of a block
                uint32_t need_r = ((1u << U) - 1) << s, need_i = need_r;  // ballots that may find a block's first nonzero
                if constexpr (BR >= 64) {
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int b = (s + u) / PER;
                        if (br >> b & 1u) need_r &= ~(1u << (s + u));
                        if (bi >> b & 1u) need_i &= ~(1u << (s + u));
                    }
                    if (!(need_r | need_i)) continue;  // uniform, as all of these
                }
                T vr[U], vi[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int64_t r = r0 + 64 * (s + u) + lane;
                    const bool in = r >= lo && r < hi;
                    vr[u] = in && (need_r >> (s + u) & 1u) ? pr[r] : T(0);
                    vi[u] = in && (need_i >> (s + u) & 1u) ? pi[r] : T(0);
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const uint64_t nr = __ballot(!(vr[u] == T(0))), ni = __ballot(!(vi[u] == T(0)));
                    if constexpr (BR >= 64) {
                        const int b = (s + u) / PER;
                        if (nr) br |= 1u << b;
                        if (ni) bi |= 1u << b;
                    } else {
#pragma unroll
                        for (int q = 0; q < 64 / BR; ++q) {
                            const int b = (s + u) * (64 / BR) + q;
                            constexpr uint64_t M = (uint64_t(1) << (BR % 64)) - 1;
                            if ((nr >> (q * BR)) & M) br |= 1u << b;
                            if ((ni >> (q * BR)) & M) bi |= 1u << b;
                        }
                    }
                }
            }
        }
        if (lane == 0) {
            unsigned char *z = reinterpret_cast<unsigned char *>(zmask + (static_cast<int64_t>(j) * n + d) * zwords + w);
            z[wave] = static_cast<unsigned char>(br);
            z[4 + wave] = static_cast<unsigned char>(bi);
        }
    }
}

// Grid rows for a zero-block map over n diagonals.
inline unsigned zero_map_grid_y(int n) { return static_cast<unsigned>(n < 65535 ? n : 65535); }

inline int64_t zero_block_words(int64_t rows, int block_rows) {
    return ((rows + block_rows - 1) / block_rows + 31) / 32;
}

// A matrix's zero-block map as the kernels take it (w null: none): `words` words per diagonal, blocks of 2^shift rows.
// 64-row blocks are a wave's rows: against 256-row blocks they drop two more pairs of a qubit Hamiltonian's diagonals.
struct ZeroMap {
    const uint2 *w = nullptr;
    int64_t words = 0;
    int shift = 6;
    int loads_only = 0;  // spare the loads of zeros, but add their products too (dia_rows_wave)
    // Or, in place of w, the map that the first product of a sequence leaves (dia_rows_wave, MK): per 64-row block and 64
    // diagonals a word of real and one of imaginary bits (`words` then holds the rows).
    const ulonglong2 *by_block = nullptr;
    __host__ __device__ bool any() const { return w || by_block; }
};

inline int64_t map_by_block_bytes(int64_t rows, int n) { return ((rows + 63) / 64) * ((n + 63) / 64) * 16; }

// Map A's values into w (zero_block_words(A.rows, 2^shift) words per diagonal; shift 6 or 8) on stream s.
void make_zero_map(const dq_devmat &A, int shift, uint2 *w, hipStream_t s);
// The same for A's diagonals in the order of `meta` (A.n() entries, on the device).
void make_zero_map(const dq_devmat &A, const DiagMeta *meta, int shift, uint2 *w, hipStream_t s);
size_t zero_map_bytes(const dq_devmat &A, int shift);
// The map dq_spmv_tune keeps in A's handle (none if it keeps none).
ZeroMap kept_zero_map(const dq_devmat &A);

// Several products with a band matrix per read of it (powers.hip): the launches for a sequence of n, n where one per
// product is at least as good; and one launch, y = A^p x.
int band_powers_launches(const dq_devmat &A, int n);
void band_powers(const dq_devmat &A, const void *xr, const void *xi, void *yr, void *yi, int p, hipStream_t s);

// PIPE = true: each diagonal's 4*RPT loads are issued together (full tiles unconditionally, boundary tiles with
// clamped addresses), the schedule that keeps the most bytes in flight. Every schedule adds exactly the products of
// the rows on the diagonal, in slot order, so a row's sum has the same bits whatever the schedule (a compensated
// FP32 sum is not left unchanged by adding a zero). PIPE = false: per-row predicated loads, which
// the compiler issues row after row -- fewer loads in flight per wave but half the registers, so twice the waves;
// with scattered offsets (no x reuse between diagonals) that variant can fill L2 faster.
//
// With HALO > 0 the caller has staged the x window in (sr, si) with stage_x_window; diagonals with |offset| <= HALO
// read x from there (row r of the tile at LDS index r - tile + HALO + offset), the others from memory.
template <typename T, int RPT, bool NT = false, bool PIPE = true, int HALO = 0>
__device__ inline void dia_rows_tile(int64_t tile, int64_t tile_end, int n, const DiagMeta *__restrict__ meta,
                                     const T *__restrict__ are, const T *__restrict__ aim, const T *__restrict__ xr,
                                     const T *__restrict__ xi, int64_t col_lo, int64_t col_hi, Acc<T> (&ar)[RPT],
                                     Acc<T> (&ai)[RPT], const T *__restrict__ sr = nullptr,
                                     const T *__restrict__ si = nullptr) {
    constexpr int TILE = 256 * RPT;
    for (int k = 0; k < n; ++k) {
        const DiagMeta m = meta[k];
        const int64_t lo = max(m.rlo, col_lo - m.off);
        const int64_t hi = min(m.rhi, col_hi - m.off);
        if (hi <= tile || lo >= tile_end) continue;  // uniform: the diagonal misses this tile
        const T *pr = are + m.rowbase;
        const T *pi = aim + m.rowbase;
        if (HALO > 0 && m.off >= -HALO && m.off <= HALO) {  // uniform: x from the LDS window
            const int base = HALO + m.off;
            T va_r[RPT], va_i[RPT], vx_r[RPT], vx_i[RPT];
            if (lo <= tile && hi >= tile + TILE) {
#pragma unroll
                for (int j = 0; j < RPT; ++j) {
                    const int64_t r = tile + threadIdx.x + 256 * j;
                    va_r[j] = ld_val<T, NT>(pr + r);
                    va_i[j] = ld_val<T, NT>(pi + r);
                    vx_r[j] = sr[threadIdx.x + 256 * j + base];
                    vx_i[j] = si[threadIdx.x + 256 * j + base];
                }
#pragma unroll
                for (int j = 0; j < RPT; ++j)
                    cmac(ar[j], ai[j], va_r[j], va_i[j], vx_r[j], vx_i[j]);
            } else {  // boundary tile: clamped rows stay inside the tile, so their LDS index stays in the window
#pragma unroll
                for (int j = 0; j < RPT; ++j) {
                    const int64_t r = tile + threadIdx.x + 256 * j;
                    const int64_t rc = r < lo ? lo : (r >= hi ? hi - 1 : r);
                    va_r[j] = ld_val<T, NT>(pr + rc);
                    va_i[j] = ld_val<T, NT>(pi + rc);
                    const int e = static_cast<int>(rc - tile) + base;
                    vx_r[j] = sr[e];
                    vx_i[j] = si[e];
                }
#pragma unroll
                for (int j = 0; j < RPT; ++j) {  // rows off the diagonal add nothing (not even a zero)
                    const int64_t r = tile + threadIdx.x + 256 * j;
                    if (r >= lo && r < hi)
                        cmac(ar[j], ai[j], va_r[j], va_i[j], vx_r[j], vx_i[j]);
                }
            }
            continue;
        }
        const T *qr = xr + m.off;
        const T *qi = xi + m.off;
        if constexpr (!PIPE) {
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const int64_t r = tile + threadIdx.x + 256 * j;
                if (r >= lo && r < hi) {
                    const T a_r = ld_val<T, NT>(pr + r), a_i = ld_val<T, NT>(pi + r), x_r = qr[r], x_i = qi[r];
                    cmac(ar[j], ai[j], a_r, a_i, x_r, x_i);
                }
            }
            continue;
        }
        // All 4*RPT loads of this diagonal are issued before the first use, so a wave keeps them in flight together.
        T va_r[RPT], va_i[RPT], vx_r[RPT], vx_i[RPT];
        if (lo <= tile && hi >= tile + TILE) {  // uniform: every row of the tile is on the diagonal
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const int64_t r = tile + threadIdx.x + 256 * j;
                va_r[j] = ld_val<T, NT>(pr + r);
                va_i[j] = ld_val<T, NT>(pi + r);
                vx_r[j] = qr[r];
                vx_i[j] = qi[r];
            }
#pragma unroll
            for (int j = 0; j < RPT; ++j)
                cmac(ar[j], ai[j], va_r[j], va_i[j], vx_r[j], vx_i[j]);
        } else {  // boundary tile: clamp the loads to a valid row; rows off the diagonal add nothing (not even a zero)
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const int64_t r = tile + threadIdx.x + 256 * j;
                const int64_t rc = r < lo ? lo : (r >= hi ? hi - 1 : r);
                va_r[j] = ld_val<T, NT>(pr + rc);
                va_i[j] = ld_val<T, NT>(pi + rc);
                vx_r[j] = qr[rc];
                vx_i[j] = qi[rc];
            }
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const int64_t r = tile + threadIdx.x + 256 * j;
                if (r >= lo && r < hi)
                    cmac(ar[j], ai[j], va_r[j], va_i[j], vx_r[j], vx_i[j]);
            }
        }
    }
}

// A wave's 64 V rows, V adjacent rows per lane. The lanes first read 64 diagonals' metadata (and map words) at once,
// one diagonal each, and keep the diagonals that meet the wave's rows (ZM: and hold a nonzero in their block of the
// map) as a ballot; the wave then walks the set bits up to DB at a time, broadcasting each diagonal's entry with
// readlane and issuing the loads of all of them before the first product is added. A row therefore costs one metadata
// round trip per 64 diagonals and one load round trip per DB live ones, where dia_rows_tile pays a dependent metadata
// -> value chain for every diagonal: that chain is what bounds a matrix too small to hide it behind other waves. The
// products are added in slot order with the operations of dia_rows_tile, so a row's sum has the same bits.
__device__ inline int64_t readlane64(int64_t v, int l) {
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(static_cast<uint64_t>(v)), l);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<int>(static_cast<uint64_t>(v) >> 32), l);
    return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

// V consecutive values at byte offset `bytes` from p (uniform): one access; x windows are aligned to one value only.
template <typename T, int V>
struct Vec {
    typedef T type __attribute__((ext_vector_type(V), aligned(sizeof(T))));
};
template <typename T, int V, bool NT>
__device__ inline void ld_vec(const T *p, uint32_t bytes, T (&out)[V]) {
    const char *q = reinterpret_cast<const char *>(p) + bytes;
    if constexpr (V == 1) {
        out[0] = ld_val<T, NT>(reinterpret_cast<const T *>(q));
    } else {
        typedef typename Vec<T, V>::type W;
        W w;
        if constexpr (NT) w = __builtin_nontemporal_load(reinterpret_cast<const W *>(q));
        else w = *reinterpret_cast<const W *>(q);
#pragma unroll
        for (int v = 0; v < V; ++v) out[v] = w[v];
    }
}

// A diagonal's rng word: its rows in the wave's 64 V as lo | hi << 10, and its nonzero parts.
constexpr int RNG_HI = 10, RNG_MASK = (1 << RNG_HI) - 1, RNG_RE = 1 << 20, RNG_IM = 1 << 21;

// The next DB set bits of todo (PART: the last cnt < DB of them; the slots beyond repeat the last diagonal's loads
// and add nothing). Lane s holds diagonal s: vb (element index of its value in the wave's first row), off and rng.
// ZM: a part whose rng bit is clear is zero in these rows and is not loaded. H > 0: (sr, si) is the workgroup's x
// window at the wave's first row, and the diagonals with |off| <= H read x from there.
// MK: the values' nonzero parts go to `bits` of the diagonal's lane, one bit per 64-row block and part (block q of the
// wave: real 1 << 2 q, imaginary 2 << 2 q), and a diagonal that is zero in all of the wave's rows adds nothing, as with a map.
template <typename T, int V, int DB, bool NT, bool ZM, int H, bool PART, bool MK>
__device__ inline void wave_batch(uint64_t &todo, int cnt, int lane, int64_t vb, int off, int rng,
                                  const T *__restrict__ are, const T *__restrict__ aim, const T *__restrict__ xr,
                                  const T *__restrict__ xi, Acc<T> (&ar)[V], Acc<T> (&ai)[V], const T *sr,
                                  const T *si, int &bits) {
    int from[DB];
    T va_r[DB][V], va_i[DB][V], vx_r[DB][V], vx_i[DB][V];
    int lo[DB], hi[DB];
    bool full = true;  // every row of the wave lies on every diagonal of the batch
    int s = 0;
#pragma unroll
    for (int u = 0; u < DB; ++u) {
        if (!PART || u < cnt) {
            s = __builtin_ctzll(todo);
            todo &= todo - 1;
        }
        from[u] = s;
        const int64_t b = readlane64(vb, s);
        const int x = __builtin_amdgcn_readlane(off, s);
        const bool near = H > 0 && x >= -H && x <= H;  // uniform
        const int r = __builtin_amdgcn_readlane(rng, s);
        lo[u] = r & RNG_MASK;
        hi[u] = (r >> RNG_HI) & RNG_MASK;
        const bool whole = lo[u] == 0 && hi[u] == 64 * V;  // uniform
        full = full && whole;
        if (V == 1 || whole) {
            // V == 1: clamped to the diagonal's rows; otherwise every row is on it
            const int row = V == 1 ? min(max(lane, lo[u]), hi[u] - 1) : V * lane;
            const uint32_t e = static_cast<uint32_t>(row) * static_cast<uint32_t>(sizeof(T));
#pragma unroll
            for (int v = 0; v < V; ++v) {
                va_r[u][v] = T(0);
                va_i[u][v] = T(0);
            }
            if (!ZM || (r & RNG_RE)) ld_vec<T, V, NT>(are + b, e, va_r[u]);  // uniform
            if (!ZM || (r & RNG_IM)) ld_vec<T, V, NT>(aim + b, e, va_i[u]);
            if (near) {
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    vx_r[u][v] = sr[x + row + v];
                    vx_i[u][v] = si[x + row + v];
                }
            } else {
                ld_vec<T, V, false>(xr + x, e, vx_r[u]);
                ld_vec<T, V, false>(xi + x, e, vx_i[u]);
            }
        } else {  // row by row, clamped
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const int row = min(max(V * lane + v, lo[u]), hi[u] - 1);
                va_r[u][v] = (are + b)[row];
                va_i[u][v] = (aim + b)[row];
                vx_r[u][v] = (xr + x)[row];
                vx_i[u][v] = (xi + x)[row];
            }
        }
    }
    bool live[DB];  // uniform
#pragma unroll
    for (int u = 0; u < DB; ++u) live[u] = !PART || u < cnt;
    if constexpr (MK) {
#pragma unroll
        for (int u = 0; u < DB; ++u) {
            bool r = false, i = false;  // a lane's V rows lie in one block
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const bool in = live[u] && V * lane + v >= lo[u] && V * lane + v < hi[u];
                r = r || (in && !(va_r[u][v] == T(0)));
                i = i || (in && !(va_i[u][v] == T(0)));
            }
            const uint64_t nr = __ballot(r), ni = __ballot(i);
            live[u] = nr || ni;
            int found = 0;
#pragma unroll
            for (int q = 0; q < V; ++q) {
                constexpr uint64_t BLOCK = V == 1 ? ~uint64_t(0) : (uint64_t(1) << (64 / V)) - 1;
                if ((nr >> (q * (64 / V) % 64)) & BLOCK) found |= 1 << (2 * q);
                if ((ni >> (q * (64 / V) % 64)) & BLOCK) found |= 2 << (2 * q);
            }
            if (found && lane == from[u]) bits = found;
        }
    }
    if (full) {  // uniform
#pragma unroll
        for (int u = 0; u < DB; ++u)
            if (live[u]) {
#pragma unroll
                for (int v = 0; v < V; ++v) cmac(ar[v], ai[v], va_r[u][v], va_i[u][v], vx_r[u][v], vx_i[u][v]);
            }
        return;
    }
#pragma unroll
    for (int u = 0; u < DB; ++u)  // rows off the diagonal add nothing (not even a zero)
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (live[u] && V * lane + v >= lo[u] && V * lane + v < hi[u])
                cmac(ar[v], ai[v], va_r[u][v], va_i[u][v], vx_r[u][v], vx_i[u][v]);
}

// The sums of rows row0 + V lane + v (row0 a multiple of 64 V, below the matrix's rows). With a map its blocks are at
// least a wave's rows or whole parts of them. H > 0: the caller has staged the x window of the workgroup's 256 V rows
// with stage_x_window (halo H on both sides) in (sr, si).
// MK: no map yet; the wave writes its blocks' words of zm.by_block (passed as `made`) from what it reads.
template <typename T, int V, bool NT, bool ZM, int H = 0, bool MK = false>
__device__ inline void dia_rows_wave(int64_t row0, int n, const DiagMeta *__restrict__ meta,
                                     const T *__restrict__ are, const T *__restrict__ aim, const T *__restrict__ xr,
                                     const T *__restrict__ xi, int64_t col_lo, int64_t col_hi, Acc<T> (&ar)[V],
                                     Acc<T> (&ai)[V], const ZeroMap &zm, const T *sr = nullptr,
                                     const T *si = nullptr, ulonglong2 *made = nullptr, int64_t rows = 0) {
    constexpr int DB = 8 / V;
    const int lane = threadIdx.x & 63;
    xr += row0;
    xi += row0;
    if (H > 0) {  // to the wave's first row
        sr += H + static_cast<int>(row0 % (256 * V));
        si += H + static_cast<int>(row0 % (256 * V));
    }
    for (int k0 = 0; k0 < n; k0 += 64) {
        const int k = k0 + lane;
        int64_t vb = 0;
        int off = 0, rng = 0;
        bool live = false;
        if (k < n) {
            const DiagMeta m = meta[k];
            const int64_t lo = max(max(m.rlo, col_lo - m.off) - row0, int64_t(0));
            const int64_t hi = min(min(m.rhi, col_hi - m.off) - row0, int64_t(64 * V));
            live = lo < hi;
            int parts = RNG_RE | RNG_IM;
            if (ZM && zm.by_block) {  // the wave's blocks (the last ones may lie past the rows: live is false there)
                const int64_t words = (n + 63) >> 6;
                const int64_t blk = (row0 >> 6) * words + (k0 >> 6);
                ulonglong2 w = zm.by_block[blk];
#pragma unroll
                for (int q = 1; q < V; ++q)
                    if (row0 + 64 * q < zm.words) {  // words: the rows of a map by block
                        const ulonglong2 o = zm.by_block[blk + q * words];
                        w.x |= o.x;
                        w.y |= o.y;
                    }
                parts = ((w.x >> lane) & 1 ? RNG_RE : 0) | ((w.y >> lane) & 1 ? RNG_IM : 0);
                live = live && parts;
            } else if constexpr (ZM) {  // the 2^shift-row block that holds the wave's rows, or the blocks that they are
                const uint2 w = zm.w[static_cast<int64_t>(k) * zm.words + (row0 >> (zm.shift + 5))];
                const int b = static_cast<int>((row0 >> zm.shift) & 31);
                uint32_t m2 = 1u;
#pragma unroll
                for (int q = 1; q < V; ++q)
                    if ((64 * q) >> zm.shift) m2 |= 1u << ((64 * q) >> zm.shift);
                parts = (((w.x >> b) & m2) ? RNG_RE : 0) | (((w.y >> b) & m2) ? RNG_IM : 0);
                live = live && (parts || zm.loads_only);
            }
            vb = m.rowbase + row0;
            off = m.off;
            rng = live ? static_cast<int>(lo) | static_cast<int>(hi) << RNG_HI | parts : 0;
        }
        uint64_t todo = __ballot(live);
        int cnt = __popcll(todo), bits = 0;
        for (; cnt >= DB; cnt -= DB)
            wave_batch<T, V, DB, NT, ZM, H, false, MK>(todo, DB, lane, vb, off, rng, are, aim, xr, xi, ar, ai, sr, si, bits);
        if (cnt >= DB / 2) {
            wave_batch<T, V, DB / 2, NT, ZM, H, false, MK>(todo, DB / 2, lane, vb, off, rng, are, aim, xr, xi, ar, ai, sr,
                                                           si, bits);
            cnt -= DB / 2;
        }
        if (cnt)
            wave_batch<T, V, DB / 2, NT, ZM, H, true, MK>(todo, cnt, lane, vb, off, rng, are, aim, xr, xi, ar, ai, sr, si,
                                                          bits);
        if constexpr (MK) {
#pragma unroll
            for (int q = 0; q < V; ++q) {
                const uint64_t re = __ballot((bits >> (2 * q)) & 1), im = __ballot((bits >> (2 * q)) & 2);
                if (lane == 0 && row0 + 64 * q < rows)
                    made[((row0 >> 6) + q) * ((n + 63) >> 6) + (k0 >> 6)] = make_ulonglong2(re, im);
            }
        }
    }
}

// The wave's first row in a workgroup of four waves on row tile t.
template <int V>
__device__ inline int64_t wave_row0(int64_t t) {
    return t * (256 * V) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * (64 * V);
}

// V results of a lane to out + row (rows below `rows` only).
template <typename T, int V>
__device__ inline void st_rows(T *out, int64_t row, int64_t rows, const T (&v)[V]) {
    if (V > 1 && row + V <= rows) {
        typename Vec<T, V>::type w;
#pragma unroll
        for (int q = 0; q < V; ++q) w[q] = v[q];
        *reinterpret_cast<typename Vec<T, V>::type *>(out + row) = w;
        return;
    }
#pragma unroll
    for (int q = 0; q < V; ++q)
        if (row + q < rows) out[row + q] = v[q];
}

// V values of a lane from in + row (zero beyond `rows`).
template <typename T, int V>
__device__ inline void ld_rows(const T *in, int64_t row, int64_t rows, T (&v)[V]) {
    if (V > 1 && row + V <= rows) {
        ld_vec<T, V, false>(in + row, 0, v);
        return;
    }
#pragma unroll
    for (int q = 0; q < V; ++q) v[q] = row + q < rows ? in[row + q] : T(0);
}

}  // namespace dq
