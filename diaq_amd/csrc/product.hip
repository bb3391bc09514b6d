// DIA SpGEMM on gfx950: C = A B by diagonal-pair enumeration, with the structural dry-run that sizes C up front.
//
// Reference: product_kernel / product_device / product_cuda (src/spGEMM_gpu.cu:25-161), pow_cuda
// (src/spPow_gpu.cu:21-56).
//
// Dry-run (host, integer only): every pair (slot a, slot b) with dC = dA + dB in [-(rows-1), cols-1] contributes to
// result diagonal dC; result offsets ascend and each dC keeps its pairs in A-slot order (then B-slot order), so the
// sums run in the reference's order. The pairs are bucketed by dC with a counting sort (two passes over the slot
// pairs, in slot order, so each bucket keeps the enumeration order) when the offset range is at most four times the
// pairs; fewer pairs over a wider range take a stable sort.
//
// Kernel: in row space the pair (a, b) adds A_a[i] * B_b[i + dA] to C_c[i] (row i of A, row i + dA of B), where a
// diagonal's element for row r sits at rowbase + r; rows outside a diagonal's range contribute nothing, exactly the
// reference's position bounds. The work is cut into items of (row chunk of 256*RPT rows, result diagonal) --
// fixed-size items, so result diagonals of length 1 and of length N balance. Items are ordered by row chunk: the
// result diagonals meeting a chunk form a contiguous range of the ascending result offsets, so the host only sizes
// each chunk's range and a device kernel writes the item list. The item index is remapped so the workgroups of one
// row chunk, which read the same rows of A's diagonals, land on the same XCD (workgroup b runs on XCD b mod 8) and
// share its L2. A workgroup walks its diagonal's pairs in batches of 256: the lanes load the batch's pair metadata
// in parallel and leave each pair's row range and base pointers in LDS, then the pair loop reads them from there
// (no chain of dependent metadata loads per pair).
//
// Zero blocks: for large operands the product first maps which 64-row blocks of each diagonal of A and B hold a
// nonzero real or imaginary value (zero_blocks_kernel). A pair whose A rows, or whose B rows, in the item are all zero is
// dropped when its metadata is staged: its products are all +-0, and a sum that starts at +0 is left unchanged by
// adding +-0, so the result has the same bits; only a NaN or Inf facing such rows is not propagated. Of the pairs that
// stay, each wave loads only the blocks and parts that hold a nonzero and multiplies zeros for the others, which gives
// the same sums, NaN and Inf among them. A qubit Hamiltonian's +-2^k flip diagonals are zero on alternate runs of 2^k
// rows, and its imaginary part often everywhere.
//
// Bound: the L2's and the memory's reads of A and B per pair against the stores of C (TFIM-20 H*H: 1681 pairs, 727
// diagonals, 11 GB stored). Reading every part of a live pair: 4.00 ms; only the live blocks and parts: 3.03 ms; eight
// items of a workgroup together: 2.23 ms.
//
// The items also write C's own zero-block map, by ballots on what they store; a large result keeps it (map_blocks).
#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <numeric>

#include "dia_rows.hpp"

namespace dq {

struct DryRun {
    std::vector<int32_t> res;        // ascending result offsets
    std::vector<int64_t> pair_start; // res.size() + 1
    std::vector<int32_t> sa, sb;     // pairs, grouped by result diagonal, A-slot order
};

static DryRun dryrun(uint32_t rows, uint32_t cols, const std::vector<int32_t> &oa, const std::vector<int32_t> &ob) {
    const int64_t lo = -static_cast<int64_t>(rows) + 1, hi = static_cast<int64_t>(cols) - 1;
    DryRun r;
    const int64_t range = hi - lo + 1;
    const int64_t n_ab = static_cast<int64_t>(oa.size()) * static_cast<int64_t>(ob.size());
    if (range <= 0 || n_ab == 0) {
        r.pair_start.push_back(0);
        return r;
    }
    // counting sort by dC when the offset range is at most a few times the pairs (a Taylor term's 8191 x 25 offsets,
    // range 8191); a few pairs over a wide range (TFIM-20 H.H: 1681 pairs, range 2^21) sort faster than they count
    if (range <= 4 * n_ab) {
        std::vector<int64_t> cnt(static_cast<size_t>(range), 0);
        for (size_t a = 0; a < oa.size(); ++a)
            for (size_t b = 0; b < ob.size(); ++b) {
                const int64_t dc = static_cast<int64_t>(oa[a]) + ob[b];
                if (dc >= lo && dc <= hi) ++cnt[static_cast<size_t>(dc - lo)];
            }
        int64_t total = 0;
        for (int64_t i = 0; i < range; ++i) {
            if (!cnt[i]) continue;
            r.res.push_back(static_cast<int32_t>(i + lo));
            r.pair_start.push_back(total);
            const int64_t c = cnt[i];
            cnt[i] = total;  // becomes the bucket's fill position
            total += c;
        }
        r.pair_start.push_back(total);
        r.sa.resize(static_cast<size_t>(total));
        r.sb.resize(static_cast<size_t>(total));
        for (size_t a = 0; a < oa.size(); ++a)
            for (size_t b = 0; b < ob.size(); ++b) {
                const int64_t dc = static_cast<int64_t>(oa[a]) + ob[b];
                if (dc < lo || dc > hi) continue;
                const int64_t at = cnt[static_cast<size_t>(dc - lo)]++;
                r.sa[at] = static_cast<int32_t>(a);
                r.sb[at] = static_cast<int32_t>(b);
            }
        return r;
    }
    struct P {
        int64_t dc;
        int32_t a, b;
    };
    std::vector<P> pairs;
    pairs.reserve(static_cast<size_t>(n_ab));
    for (size_t a = 0; a < oa.size(); ++a)
        for (size_t b = 0; b < ob.size(); ++b) {
            const int64_t dc = static_cast<int64_t>(oa[a]) + ob[b];
            if (dc < lo || dc > hi) continue;
            pairs.push_back(P{dc, static_cast<int32_t>(a), static_cast<int32_t>(b)});
        }
    // stable by construction order (a, then b): sort by dc only
    std::stable_sort(pairs.begin(), pairs.end(), [](const P &x, const P &y) { return x.dc < y.dc; });
    r.sa.reserve(pairs.size());
    r.sb.reserve(pairs.size());
    for (size_t p = 0; p < pairs.size(); ++p) {
        if (p == 0 || pairs[p].dc != pairs[p - 1].dc) {
            r.res.push_back(static_cast<int32_t>(pairs[p].dc));
            r.pair_start.push_back(static_cast<int64_t>(p));
        }
        r.sa.push_back(pairs[p].a);
        r.sb.push_back(pairs[p].b);
    }
    r.pair_start.push_back(static_cast<int64_t>(pairs.size()));
    return r;
}

// The dry-run depends only on the shape and the two offset lists. A Taylor series multiplies operands with the same
// offsets term after term once the terms reach every diagonal they can (TFIM-12: terms 8 to 14, 8191 x 25 offsets,
// ~1.2 ms of host time each), so each thread keeps its last dry-run and reuses it when the inputs are equal. Only
// dry-runs of at most DRYRUN_CACHE_PAIRS slot pairs are kept (their lists take ~16 B per pair), and
// dq_release_cached_memory drops the kept ones: the calling thread's at once, other threads' at their next product.
constexpr int64_t DRYRUN_CACHE_PAIRS = int64_t(1) << 22;
static std::atomic<uint64_t> g_dryrun_generation{0};

struct DryRunCache {
    uint64_t generation = 0;
    uint32_t rows = 0, cols = 0;
    std::vector<int32_t> oa, ob;
    std::shared_ptr<const DryRun> d;
};

static DryRunCache &dryrun_cache() {
    thread_local DryRunCache c;
    return c;
}

void release_dryrun_cache() {
    g_dryrun_generation.fetch_add(1);
    DryRunCache &c = dryrun_cache();
    c.d.reset();
    c.oa = std::vector<int32_t>();
    c.ob = std::vector<int32_t>();
}

static std::shared_ptr<const DryRun> dryrun_reused(uint32_t rows, uint32_t cols, const std::vector<int32_t> &oa,
                                                   const std::vector<int32_t> &ob) {
    DryRunCache &c = dryrun_cache();
    const uint64_t gen = g_dryrun_generation.load();
    if (c.d && c.generation == gen && c.rows == rows && c.cols == cols && c.oa == oa && c.ob == ob) return c.d;
    auto d = std::make_shared<const DryRun>(dryrun(rows, cols, oa, ob));
    const bool keep = static_cast<int64_t>(oa.size()) * static_cast<int64_t>(ob.size()) <= DRYRUN_CACHE_PAIRS;
    c.d = keep ? d : nullptr;
    c.generation = gen;
    c.rows = rows;
    c.cols = cols;
    c.oa = keep ? oa : std::vector<int32_t>();
    c.ob = keep ? ob : std::vector<int32_t>();
    return d;
}

constexpr int PROD_BATCH = 256;
constexpr int PROD_GROUP = 8;  // at most as many items of a workgroup

// Process-wide knobs (dq_set_tuning): chunk order across XCDs and non-temporal stores of C.
static int g_prod_interleave = 1;
static int g_prod_nt_store = 1;
// rows per lane: row chunks of 256 * rpt rows; 0 = automatic: 4 below 2^16 rows, where more and shorter items ran a
// TFIM-12 expm's 4096-row Taylor products faster (DeviceMatrix expm_negative 31.1 -> 28.8 ms), else 8 (TFIM-20 H.H:
// 3.96 ms against 4.02 ms at 4 and 4.16 ms at 16)
static int g_prod_rpt = 0;
static int g_prod_skip = 1; // drop pairs whose rows in a chunk are all zero, for operands of >= 2^16 rows

// Item list: the i-th chunk in processing order (row chunk q_of[i]) owns items [first[i], first[i + 1]), result
// diagonals c_lo[i], c_lo[i] + 1, ...
__global__ void product_items_kernel(int64_t n_chunks, const int64_t *__restrict__ first,
                                     const int32_t *__restrict__ c_lo, const int32_t *__restrict__ q_of,
                                     int2 *__restrict__ items) {
    for (int64_t i = blockIdx.x; i < n_chunks; i += gridDim.x) {
        const int64_t f = first[i], n = first[i + 1] - f;
        const int32_t c0 = c_lo[i], q = q_of[i];
        for (int64_t j = threadIdx.x; j < n; j += blockDim.x) items[f + j] = make_int2(q, c0 + static_cast<int>(j));
    }
}

// Zero the storage outside every diagonal's rows: the alignment gaps between diagonals and the tail.
template <typename T>
__global__ void zero_gaps_kernel(int n, const DiagMeta *__restrict__ meta, int64_t total, T *__restrict__ re,
                                 T *__restrict__ im) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k > n) return;
    const int64_t b = k == 0 ? 0 : meta[k - 1].rowbase + meta[k - 1].rhi;
    const int64_t e = k == n ? total : meta[k].rowbase + meta[k].rlo;
    for (int64_t i = b; i < e; ++i) {
        re[i] = T(0);
        im[i] = T(0);
    }
}

void zero_gaps(dq_devmat &M, hipStream_t s) {
    const int n = M.n();
    if (n == 0 || M.total == 0) return;
    const unsigned g = blocks_for(n + 1, 256, 1 << 20);
    if (M.precision == DQ_F64)
        hipLaunchKernelGGL(zero_gaps_kernel<double>, dim3(g), dim3(256), 0, s, n, M.d_meta.as<DiagMeta>(), M.total,
                           M.re.as<double>(), M.im.as<double>());
    else
        hipLaunchKernelGGL(zero_gaps_kernel<float>, dim3(g), dim3(256), 0, s, n, M.d_meta.as<DiagMeta>(), M.total,
                           M.re.as<float>(), M.im.as<float>());
    DQ_LAUNCH_CHECK();
}

__device__ inline int64_t uniform64(int64_t v) {
    const int lo = __builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint64_t>(v) & 0xffffffffu));
    const int hi = __builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint64_t>(v) >> 32));
    return static_cast<int64_t>((static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) | static_cast<uint32_t>(lo));
}

// The bits of 32 consecutive blocks from block b0 (which may lie outside the map) of diagonal k: x real, y imaginary.
__device__ inline uint2 map_window(const ZeroMap &z, int64_t k, int64_t b0) {
    const uint2 *row = z.w + k * z.words;
    const int64_t w = b0 >> 5;
    const int sh = static_cast<int>(b0 & 31);
    const uint2 a = w >= 0 && w < z.words ? row[w] : make_uint2(0, 0);
    if (sh == 0) return a;
    const uint2 b = w + 1 >= 0 && w + 1 < z.words ? row[w + 1] : make_uint2(0, 0);
    return make_uint2(a.x >> sh | b.x << (32 - sh), a.y >> sh | b.y << (32 - sh));
}

// The same for the 32 blocks of 64 rows that start at row r0, which need not be a block's first row: a bit is set where
// either block that holds some of the rows has it.
__device__ inline uint2 map_rows(const ZeroMap &z, int64_t k, int64_t r0) {
    uint2 m = map_window(z, k, r0 >> 6);
    if (r0 & 63) {
        const uint2 n = map_window(z, k, (r0 >> 6) + 1);
        m.x |= n.x;
        m.y |= n.y;
    }
    return m;
}

// Rows r + 256 j of p into v, R of them: a wave's 64 rows of pass j are block 4 j + wave of the item, and `live` has bit
// 4 j set when they hold a nonzero. The others are zeros and are not loaded (uniform in the wave).
template <typename T, int R>
__device__ inline void ld_blocks(const T *p, uint32_t live, const uint32_t (&r)[R], T (&v)[R]) {
    constexpr uint32_t ALL = R >= 8 ? 0x11111111u : 0x1111u;
    if ((live & ALL) == ALL || (R > 8 && live)) {
#pragma unroll
        for (int j = 0; j < R; ++j) v[j] = p[r[j]];
        return;
    }
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = T(0);
    if (R > 8 || (live & ALL) == 0) return;
#pragma unroll
    for (int j = 0; j < R; ++j)
        if (live >> (4 * (j & 7)) & 1u) v[j] = p[r[j]];
}

// MAP: the operands have zero-block maps (za, zb).
template <typename T, bool NTS, int PROD_RPT, bool MAP>
__global__ __launch_bounds__(256) void product_kernel(const int2 *__restrict__ items, const int64_t *__restrict__ xcd_first,
                                                      const int64_t *__restrict__ pair_start,
                                                      const int32_t *__restrict__ pa, const int32_t *__restrict__ pb,
                                                      const DiagMeta *__restrict__ ma, const DiagMeta *__restrict__ mb,
                                                      const DiagMeta *__restrict__ mc, const T *__restrict__ are,
                                                      const T *__restrict__ aim, const T *__restrict__ bre,
                                                      const T *__restrict__ bim, T *__restrict__ cre,
                                                      T *__restrict__ cim, double divisor,
                                                      ZeroMap za, ZeroMap zb, uint2 *__restrict__ zc,
                                                      int64_t zc_words, int group,
                                                      const unsigned long long *__restrict__ live,
                                                      unsigned long long sparse, int sparse_group) {
    constexpr int PROD_CHUNK = 256 * PROD_RPT;
    __shared__ int64_t s_abase[PROD_BATCH], s_bbase[PROD_BATCH];
    __shared__ int32_t s_lo[PROD_BATCH], s_hi[PROD_BATCH];
    __shared__ uint4 s_live[MAP ? PROD_BATCH : 1];  // the item's blocks that hold a nonzero: A real, A imaginary, B real,
                                                    // B imaginary
    constexpr int ZW = (PROD_RPT + 7) / 8;  // map words of an item's rows
    __shared__ uint32_t s_zr[2][4][ZW], s_zi[2][4][ZW];  // by parity of the item and wave
    // the workgroup's items: result diagonal, first row, its rows [r0, r1) as offsets from that, its pairs
    __shared__ int64_t s_q0[PROD_GROUP], s_cbase[PROD_GROUP], s_p0[PROD_GROUP];
    __shared__ int32_t s_c[PROD_GROUP], s_r0[PROD_GROUP], s_r1[PROD_GROUP], s_cnt[PROD_GROUP];
    // XCD-aware remap: the workgroups of XCD x (x = b mod 8) take the item range [xcd_first[x], xcd_first[x + 1]).
    const int64_t b = blockIdx.x;
    if (MAP && live && *live <= sparse) group = sparse_group;  // uniform; the last workgroups then find nothing to do
    const int64_t w = xcd_first[b & 7] + (b >> 3) * group, w_end = xcd_first[(b & 7) + 1];
    if (w >= w_end) return;  // uniform
    const int ng = MAP ? static_cast<int>(min<int64_t>(group, w_end - w)) : 1;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    struct Item {
        int64_t q0, cbase, p0;
        int32_t c, r0, r1, cnt;
    };
    auto load_item = [&](int64_t i) {
        const int2 it = items[i];
        const DiagMeta m_c = mc[it.y];
        const int64_t q0 = static_cast<int64_t>(it.x) * PROD_CHUNK, p0 = pair_start[it.y];
        return Item{q0, m_c.rowbase, p0, it.y, static_cast<int32_t>(max(m_c.rlo, q0) - q0),
                    static_cast<int32_t>(min(m_c.rhi, q0 + PROD_CHUNK) - q0),
                    static_cast<int32_t>(pair_start[it.y + 1] - p0)};
    };
    Item only{};  // without maps: the one item, uniform
    if constexpr (MAP) {
        if (static_cast<int>(threadIdx.x) < ng) {
            const Item it = load_item(w + threadIdx.x);
            s_q0[threadIdx.x] = it.q0;
            s_cbase[threadIdx.x] = it.cbase;
            s_p0[threadIdx.x] = it.p0;
            s_c[threadIdx.x] = it.c;
            s_r0[threadIdx.x] = it.r0;
            s_r1[threadIdx.x] = it.r1;
            s_cnt[threadIdx.x] = it.cnt;
        }
        __syncthreads();
    } else {
        only = load_item(w);
    }
    int base = 0, staged = 0, first = 0;  // the staged pairs [base, staged) of the workgroup's, and the item's first one
    for (int g = 0; g < ng; ++g) {  // uniform
        const int64_t q0 = MAP ? uniform64(s_q0[g]) : only.q0;
        const int cnt = MAP ? __builtin_amdgcn_readfirstlane(s_cnt[g]) : only.cnt;
        T acc_r[PROD_RPT], acc_i[PROD_RPT];
#pragma unroll
        for (int j = 0; j < PROD_RPT; ++j) { acc_r[j] = T(0); acc_i[j] = T(0); }
        for (int pk = first; pk < first + cnt; ++pk) {
            if (pk == staged) {  // uniform: the next batch of pairs
                __syncthreads();  // the last one is done with
                int of = 0, at = staged + static_cast<int>(threadIdx.x);  // the lane's pair: number `at` of item `of`
                if constexpr (MAP) {
                    while (of < ng && at >= s_cnt[of]) at -= s_cnt[of++];
                } else {
                    of = at >= only.cnt;
                }
                if (of < ng) {
                    const int64_t p = (MAP ? s_p0[of] : only.p0) + at, q0 = MAP ? s_q0[of] : only.q0;
                    const int32_t sa = pa[p], sb = pb[p];
                    const DiagMeta ta = ma[sa];
                    const DiagMeta tb = mb[sb];
                    // rows r of the item with r on A's diagonal and r + dA on B's: [lo, hi), as offsets from q0
                    const int64_t lo = max(max(ta.rlo, tb.rlo - ta.off), q0 + (MAP ? s_r0[of] : only.r0));
                    const int64_t hi = min(min(ta.rhi, tb.rhi - ta.off), q0 + (MAP ? s_r1[of] : only.r1));
                    bool live = hi > lo;
                    uint4 m = make_uint4(~0u, ~0u, ~0u, ~0u);
                    if (MAP && live) {  // rows that a diagonal does not have are clear bits of its map
                        m = make_uint4(0, 0, 0, 0);
#pragma unroll
                        for (int w8 = 0; w8 < ZW; ++w8) {
                            const int64_t q = q0 + 2048 * w8;
                            const uint2 a2 = map_rows(za, sa, q), b2 = map_rows(zb, sb, q + ta.off);
                            m.x |= a2.x; m.y |= a2.y; m.z |= b2.x; m.w |= b2.y;
                        }
                        constexpr uint32_t IN = PROD_RPT < 8 ? 0xffffu : ~0u;  // the item's rows
                        live = ((m.x | m.y) & IN) && ((m.z | m.w) & IN);
                    }
                    if (MAP) s_live[threadIdx.x] = m;
                    s_abase[threadIdx.x] = ta.rowbase;
                    s_bbase[threadIdx.x] = tb.rowbase + ta.off;
                    s_lo[threadIdx.x] = live ? static_cast<int32_t>(lo - q0) : 0;
                    s_hi[threadIdx.x] = live ? static_cast<int32_t>(hi - q0) : 0;
                }
                base = staged;
                staged += PROD_BATCH;
                __syncthreads();
            }
            const int k = pk - base;
            const int64_t lo = q0 + __builtin_amdgcn_readfirstlane(s_lo[k]);
            const int64_t hi = q0 + __builtin_amdgcn_readfirstlane(s_hi[k]);
            if (hi <= lo) continue;  // uniform
            const int64_t abase = uniform64(s_abase[k]), bbase = uniform64(s_bbase[k]);
            const T *apr = are + (abase + q0), *api = aim + (abase + q0);  // the item's first row
            const T *bpr = bre + (bbase + q0), *bpi = bim + (bbase + q0);
            uint32_t l_ar = ~0u, l_ai = ~0u, l_br = ~0u, l_bi = ~0u;
            if constexpr (MAP) {
                const uint4 m = s_live[k];
                l_ar = __builtin_amdgcn_readfirstlane(m.x) >> wave;
                l_ai = __builtin_amdgcn_readfirstlane(m.y) >> wave;
                l_br = __builtin_amdgcn_readfirstlane(m.z) >> wave;
                l_bi = __builtin_amdgcn_readfirstlane(m.w) >> wave;
            }
            const bool whole = lo == q0 && hi == q0 + PROD_CHUNK;  // uniform: the whole chunk, no per-row checks
            T va_r[PROD_RPT], va_i[PROD_RPT], vb_r[PROD_RPT], vb_i[PROD_RPT];
            uint32_t at[PROD_RPT];
            const int32_t l0 = static_cast<int32_t>(lo - q0), h0 = static_cast<int32_t>(hi - q0);
#pragma unroll
            for (int j = 0; j < PROD_RPT; ++j) {
                const int32_t r = static_cast<int32_t>(threadIdx.x) + 256 * j;
                at[j] = whole ? r : (r < l0 ? l0 : (r >= h0 ? h0 - 1 : r));  // clamped to a valid row
            }
            ld_blocks(apr, l_ar, at, va_r);
            ld_blocks(api, l_ai, at, va_i);
            ld_blocks(bpr, l_br, at, vb_r);
            ld_blocks(bpi, l_bi, at, vb_i);
            if (!whole) {  // zero both operands of the rows outside [lo, hi)
#pragma unroll
                for (int j = 0; j < PROD_RPT; ++j) {
                    const int32_t r = static_cast<int32_t>(threadIdx.x) + 256 * j;
                    if (r < l0 || r >= h0) { va_r[j] = T(0); va_i[j] = T(0); vb_r[j] = T(0); vb_i[j] = T(0); }
                }
            }
#pragma unroll
            for (int j = 0; j < PROD_RPT; ++j) {
                T re, im;
                cmul(va_r[j], va_i[j], vb_r[j], vb_i[j], re, im);
                acc_r[j] += re;
                acc_i[j] += im;
            }
        }
        first += cnt;
        const int32_t r0 = MAP ? s_r0[g] : only.r0, r1 = MAP ? s_r1[g] : only.r1;
        const int64_t cbase = (MAP ? uniform64(s_cbase[g]) : only.cbase) + q0;
        uint32_t zr[ZW] = {}, zi[ZW] = {};
#pragma unroll
        for (int j = 0; j < PROD_RPT; ++j) {
            const int32_t r = static_cast<int32_t>(threadIdx.x) + 256 * j;
            const bool in = r >= r0 && r < r1;
            T vr = acc_r[j], vi = acc_i[j];
            if (divisor != 1.0) {
                vr = static_cast<T>(acc_r[j] / divisor);
                vi = static_cast<T>(acc_i[j] / divisor);
            }
            if (in) {
                if constexpr (NTS) {  // C is written once and not read here: keep it out of the caches
                    __builtin_nontemporal_store(vr, cre + cbase + r);
                    __builtin_nontemporal_store(vi, cim + cbase + r);
                } else {
                    cre[cbase + r] = vr;
                    cim[cbase + r] = vi;
                }
            }
            if (MAP && zc) {  // uniform; the wave's 64 rows of pass j are block 4 j + wave of the item
                if (__ballot(in && !(vr == T(0)))) zr[j >> 3] |= 1u << (4 * (j & 7));
                if (__ballot(in && !(vi == T(0)))) zi[j >> 3] |= 1u << (4 * (j & 7));
            }
        }
        if (MAP && zc) {
            uint32_t (&gr)[4][ZW] = s_zr[g & 1], (&gi)[4][ZW] = s_zi[g & 1];
            if ((threadIdx.x & 63) == 0) {
#pragma unroll
                for (int w8 = 0; w8 < ZW; ++w8) {
                    gr[wave][w8] = zr[w8] << wave;
                    gi[wave][w8] = zi[w8] << wave;
                }
            }
            __syncthreads();  // the item after the next writes here again, behind the next item's barrier
            if (threadIdx.x < ZW) {
                const uint32_t br = gr[0][threadIdx.x] | gr[1][threadIdx.x] | gr[2][threadIdx.x] | gr[3][threadIdx.x];
                const uint32_t bi = gi[0][threadIdx.x] | gi[1][threadIdx.x] | gi[2][threadIdx.x] | gi[3][threadIdx.x];
                uint2 *to = zc + s_c[g] * zc_words + (q0 >> 11) + threadIdx.x;
                if constexpr (PROD_RPT == 4) {  // half a word
                    uint16_t *h = reinterpret_cast<uint16_t *>(to) + ((q0 >> 10) & 1);
                    h[0] = static_cast<uint16_t>(br);
                    h[2] = static_cast<uint16_t>(bi);
                } else if ((q0 >> 11) + threadIdx.x < zc_words) {
                    *to = make_uint2(br, bi);
                }
            }
        }
    }
}

// The set bits of a zero-block map, added to *out.
__global__ __launch_bounds__(256) void map_bits_kernel(int64_t n, const uint2 *__restrict__ w,
                                                       unsigned long long *__restrict__ out) {
    unsigned c = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        c += __popc(w[i].x) + __popc(w[i].y);
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    __shared__ unsigned part[4];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(out, static_cast<unsigned long long>(part[0]) + part[1] + part[2] + part[3]);
}

// The blocks of a zero-block map that hold a nonzero, added to *out.
__global__ __launch_bounds__(256) void live_blocks_kernel(int64_t n, const uint2 *__restrict__ w,
                                                          unsigned long long *__restrict__ out) {
    unsigned c = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        c += __popc(w[i].x | w[i].y);
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    __shared__ unsigned part[4];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(out, static_cast<unsigned long long>(part[0]) + part[1] + part[2] + part[3]);
}

// Items of a workgroup, for operands with maps: they share the round trips of their metadata, but take turns where workgroups
// of one item run side by side and find each other's operands in the L2. Where most pairs are dead, as in a qubit
// Hamiltonian, the metadata is a good part of an item; where all are live, sharing costs up to half of the speed. us for
// 1 / 2 / 4 / 8 items:
//   TFIM-20 squared, 372 000 items            3080 / 2680 / 2490 / 2430
//   TFIM-16 squared times itself, 503 000     9690 / 8160 / 7650 / 7930;  times the TFIM, 110 000: 1090 / 975 / 925 / 967
//   33 diagonals side by side, 133 000        8740 / 8900 / 13230 / 17460;  24 far apart, 253 000: 3700 / 3590 / 3650 / 3940
// So from MANY_ITEMS on the product counts the live blocks of its operands' maps (two launches, 10 us) and its workgroups
// read the count: 4 items, from 4 MANY_ITEMS on 8, where a quarter of the blocks is zero or more. The grid is made for the
// other case; the workgroups that have nothing to do then are its last ones. There and from SOME_ITEMS on it is two items
// where a result diagonal has fewer than FEW_PAIRS pairs (TFIM-17, 33 000 items: 318 / 300; 16 diagonals far apart, 53 000:
// 739 / 731; 5 side by side, 9 200: 241 / 244), else one (9 side by side, 8 700: 283 / 293). Smaller products have few
// workgroups: 16 diagonals, 3 360 items 90 / 99, 9 diagonals, 544 items 53 / 57.
constexpr int64_t SOME_ITEMS = int64_t(1) << 12, MANY_ITEMS = int64_t(1) << 16, FEW_PAIRS = 3;

// Pair lists up to this size join the other work lists in one upload; longer ones are copied from where they are, as
// gathering them first would take about as long as a copy of their own.
constexpr size_t UPLOAD_PAIR_BYTES = size_t(1) << 18;

// The 64-row blocks of C's diagonals, when the product is to map them for the result's own products, else 0: FP64 values
// of 1 GiB or more, far beyond the Infinity Cache, where a product is bound by reading them. One SpMV with H*H, us, without
// and with the map: TFIM-20 (10.2 GiB) 1904 / 946, XXZ-18 (1.9 GiB) 392 / 260, TFIM-17 (0.9 GiB) 211 / 246, XXZ-16 (0.4 GiB)
// 99 / 119: there the look-ups cost more than the loads that they spare, and the product itself pays for the map's fill,
// stores, count and read-back (3 diagonals, 2^21 rows: 139 -> 119 without).
constexpr int64_t MAP_RESULT_BYTES = int64_t(1) << 30;

static int64_t blocks_of(const dq_devmat &M) {
    int64_t n = 0;
    for (const DiagMeta &m : M.meta)
        if (m.rhi > m.rlo) n += ((m.rhi - 1) >> 6) - (m.rlo >> 6) + 1;
    return n;
}

static int64_t map_blocks(const dq_devmat &C) {
    if (C.precision != DQ_F64 || C.rows < (1u << 16) || 16 * C.total <= MAP_RESULT_BYTES) return 0;
    return blocks_of(C);
}

std::unique_ptr<dq_devmat> product(const dq_devmat &A, const dq_devmat &B, double divisor, hipStream_t s,
                                   bool allow_dense, bool keep_map) {
    if (A.cols != B.rows) throw ArgError("diaQMatrix product_cuda: dimension mismatch.");
    if (A.precision != B.precision) throw ArgError("product: operands have different precisions");
    if (allow_dense && dense_product_pays(A, B)) return product_dense(A, B, divisor, s);
    const std::shared_ptr<const DryRun> dp = dryrun_reused(A.rows, B.cols, A.offs, B.offs);
    const DryRun &d = *dp;
    // every stored element of C is written by the kernel; only the gaps between diagonals are zeroed
    auto C = make_devmat(A.rows, B.cols, d.res.data(), static_cast<int>(d.res.size()), A.precision, s, false);
    const int nc = C->n();
    if (nc == 0) return C;
    zero_gaps(*C, s);
    // per row chunk, the contiguous range of result diagonals that meet it (rlo and rhi do not increase with c).
    // Chunk order: the chunks q with q mod 8 == 0 first, then those with q mod 8 == 1, ... (interleave: the XCDs work
    // on neighbouring chunks at the same time, so a far pair's B rows, which are another chunk's near rows, are read
    // from the Infinity Cache), or plain ascending order.
    int64_t max_rhi = 0;
    for (int c = 0; c < nc; ++c) max_rhi = std::max(max_rhi, C->meta[c].rhi);
    const int prod_rpt = g_prod_rpt > 0 ? g_prod_rpt : (A.rows < (1u << 16) ? 4 : 8);
    const int64_t PROD_CHUNK = 256 * static_cast<int64_t>(prod_rpt);
    const int64_t n_chunks = (max_rhi + PROD_CHUNK - 1) / PROD_CHUNK;
    std::vector<int64_t> order;
    order.reserve(static_cast<size_t>(n_chunks));
    std::vector<int64_t> xcd_first(9, 0);
    for (int x = 0; x < 8; ++x) {
        if (g_prod_interleave)
            for (int64_t q = x; q < n_chunks; q += 8) order.push_back(q);
        else
            for (int64_t q = n_chunks * x / 8; q < n_chunks * (x + 1) / 8; ++q) order.push_back(q);
    }
    std::vector<int64_t> first(static_cast<size_t>(n_chunks) + 1, 0);
    std::vector<int32_t> c_lo(static_cast<size_t>(std::max<int64_t>(1, n_chunks)), 0), q_of(c_lo.size(), 0);
    for (int64_t i = 0; i < n_chunks; ++i) {
        const int64_t q = order[i];
        const int64_t Q0 = q * PROD_CHUNK, Q1 = Q0 + PROD_CHUNK;
        int lo = 0, hi = nc;  // first c with rlo < Q1
        while (lo < hi) {
            const int mid = (lo + hi) / 2;
            if (C->meta[mid].rlo >= Q1) lo = mid + 1; else hi = mid;
        }
        const int c1 = lo;
        lo = c1; hi = nc;     // first c (from c1) with rhi <= Q0
        while (lo < hi) {
            const int mid = (lo + hi) / 2;
            if (C->meta[mid].rhi > Q0) lo = mid + 1; else hi = mid;
        }
        const int c2 = lo;
        c_lo[i] = c1;
        q_of[i] = static_cast<int32_t>(q);
        first[i + 1] = first[i] + std::max(0, c2 - c1);
    }
    const int64_t n_work = first[n_chunks];
    if (n_work == 0) return C;
    // the item list (in chunk order) is split evenly over the XCDs: with many chunks each XCD works through whole
    // chunks in the order above; with fewer chunks than XCDs a chunk's items spread over several
    for (int x = 0; x <= 8; ++x) xcd_first[x] = n_work * x / 8;
    int64_t per_xcd = 0;
    const bool maps = g_prod_skip && A.rows >= (uint32_t(1) << 16) && A.n() > 0 && B.n() > 0;
    const bool few_pairs = static_cast<int64_t>(d.sa.size()) < FEW_PAIRS * nc;
    const bool by_zeros = maps && n_work >= MANY_ITEMS;
    const int group = maps && n_work >= SOME_ITEMS && few_pairs ? 2 : 1;
    const int sparse_group = n_work >= 4 * MANY_ITEMS ? PROD_GROUP : 4;
    for (int x = 0; x < 8; ++x) per_xcd = std::max(per_xcd, (xcd_first[x + 1] - xcd_first[x] + group - 1) / group);
    const int64_t grid = per_xcd * 8;
    if (grid > 0x7fffffffLL) throw ArgError("product: too many work items");
    // one block for the work lists and, but for long pair lists, one copy: seven of each cost a small product more than
    // its kernel (1024 rows, TFIM-10 squared and applied: 113 -> 81 us; 2048 rows, 11-qubit Pauli sum squared, with the
    // conversion to dense: 172 -> 158)
    size_t lists = 0;
    auto place = [&](size_t bytes) {
        const size_t at = lists;
        lists += (bytes + 15) / 16 * 16;
        return at;
    };
    const size_t at_first = place(sizeof(int64_t) * first.size()), at_clo = place(sizeof(int32_t) * c_lo.size()),
                 at_qof = place(sizeof(int32_t) * q_of.size()), at_xcd = place(sizeof(int64_t) * xcd_first.size()),
                 at_ps = place(sizeof(int64_t) * d.pair_start.size()), small = lists,
                 at_sa = place(sizeof(int32_t) * d.sa.size()), at_sb = place(sizeof(int32_t) * d.sb.size()),
                 whole = lists, at_items = place(sizeof(int2) * static_cast<size_t>(n_work));
    DevBuf work(lists);
    char *const dev = work.as<char>();
    const bool pairs_too = whole - small <= UPLOAD_PAIR_BYTES;
    std::vector<char> host(pairs_too ? whole : small);
    auto put = [&](size_t at, const auto &v) {
        if (!v.empty()) std::memcpy(host.data() + at, v.data(), sizeof(v[0]) * v.size());
    };
    put(at_first, first);
    put(at_clo, c_lo);
    put(at_qof, q_of);
    put(at_xcd, xcd_first);
    put(at_ps, d.pair_start);
    if (pairs_too) {
        put(at_sa, d.sa);
        put(at_sb, d.sb);
    } else {
        DQ_HIP(hipMemcpyAsync(dev + at_sa, d.sa.data(), sizeof(int32_t) * d.sa.size(), hipMemcpyHostToDevice, s));
        DQ_HIP(hipMemcpyAsync(dev + at_sb, d.sb.data(), sizeof(int32_t) * d.sb.size(), hipMemcpyHostToDevice, s));
    }
    DQ_HIP(hipMemcpyAsync(dev, host.data(), host.size(), hipMemcpyHostToDevice, s));
    const auto *dfirst = reinterpret_cast<const int64_t *>(dev + at_first), *dxcd = reinterpret_cast<const int64_t *>(dev + at_xcd),
               *dps = reinterpret_cast<const int64_t *>(dev + at_ps);
    const auto *dclo = reinterpret_cast<const int32_t *>(dev + at_clo), *dqof = reinterpret_cast<const int32_t *>(dev + at_qof),
               *dsa = reinterpret_cast<const int32_t *>(dev + at_sa), *dsb = reinterpret_cast<const int32_t *>(dev + at_sb);
    auto *ditems = reinterpret_cast<int2 *>(dev + at_items);
    // zero-block maps of A and B (a squaring maps its operand once; a map the handle keeps is used as it is)
    DevBuf zab, zbb;
    ZeroMap za, zb;
    if (maps) {
        auto map_of = [&](const dq_devmat &M, DevBuf &buf) {
            ZeroMap z = kept_zero_map(M);
            if (z.w) return z;
            buf = DevBuf(zero_map_bytes(M, z.shift));
            make_zero_map(M, z.shift, buf.as<uint2>(), s);
            z.w = buf.as<uint2>();
            z.words = zero_block_words(M.rows, 1 << z.shift);
            return z;
        };
        za = map_of(A, zab);
        zb = (&A == &B) ? za : map_of(B, zbb);
    }
    DevBuf dlive;
    unsigned long long sparse = 0;
    if (by_zeros) {
        dlive = DevBuf(16);
        zero_bytes(dlive.p, 8, s);
        int64_t blocks = 0;
        auto count = [&](const dq_devmat &M, const ZeroMap &z) {
            const int64_t words = z.words * M.n();
            hipLaunchKernelGGL(live_blocks_kernel, dim3(blocks_for(words, 1024, 128)), dim3(256), 0, s, words, z.w,
                               dlive.as<unsigned long long>());
            DQ_LAUNCH_CHECK();
            blocks += blocks_of(M);
        };
        count(A, za);
        if (&A != &B) count(B, zb);
        sparse = static_cast<unsigned long long>(blocks - blocks / 4);
    }
    // the result's own map, where a product with it may use one: kept when at least an eighth of its blocks are zero
    const int64_t c_blocks = keep_map && za.w ? map_blocks(*C) : 0;
    DevBuf zcb, dbits;
    unsigned long long bits = 0;
    if (c_blocks) {
        zcb = DevBuf(zero_map_bytes(*C, ZeroMap().shift));
        dbits = DevBuf(16);
        zero_bytes(zcb.p, zcb.bytes, s);
        zero_bytes(dbits.p, 8, s);
    }
    const int64_t zc_words = zero_block_words(C->rows, 64);
    hipLaunchKernelGGL(product_items_kernel, dim3(static_cast<unsigned>(std::min<int64_t>(n_chunks, 65536))),
                       dim3(256), 0, s, n_chunks, dfirst, dclo, dqof, ditems);
    DQ_LAUNCH_CHECK();
#define DQ_PROD_LAUNCH_M(T, NTS, R, M)                                                                             \
    hipLaunchKernelGGL((product_kernel<T, NTS, R, M>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, s,        \
                       ditems, dxcd, dps, dsa, dsb, A.d_meta.as<DiagMeta>(), B.d_meta.as<DiagMeta>(), C->d_meta.as<DiagMeta>(), \
                       A.re.as<T>(), A.im.as<T>(), B.re.as<T>(), B.im.as<T>(), C->re.as<T>(), C->im.as<T>(), divisor, \
                       za, zb, zcb.as<uint2>(), zc_words, group, dlive.as<unsigned long long>(), sparse, sparse_group)
#define DQ_PROD_LAUNCH_R(T, NTS, R)                          \
    do {                                                     \
        if (za.w) DQ_PROD_LAUNCH_M(T, NTS, R, true);         \
        else DQ_PROD_LAUNCH_M(T, NTS, R, false);             \
    } while (0)
#define DQ_PROD_LAUNCH(T, NTS)                                     \
    do {                                                           \
        if (prod_rpt == 4) DQ_PROD_LAUNCH_R(T, NTS, 4);            \
        else if (prod_rpt == 16) DQ_PROD_LAUNCH_R(T, NTS, 16);     \
        else DQ_PROD_LAUNCH_R(T, NTS, 8);                          \
    } while (0)
    if (A.precision == DQ_F64) {
        if (g_prod_nt_store) DQ_PROD_LAUNCH(double, true);
        else DQ_PROD_LAUNCH(double, false);
    } else {
        if (g_prod_nt_store) DQ_PROD_LAUNCH(float, true);
        else DQ_PROD_LAUNCH(float, false);
    }
#undef DQ_PROD_LAUNCH
#undef DQ_PROD_LAUNCH_R
#undef DQ_PROD_LAUNCH_M
    DQ_LAUNCH_CHECK();
    if (c_blocks) {
        const int64_t words = static_cast<int64_t>(zcb.bytes / sizeof(uint2));
        hipLaunchKernelGGL(map_bits_kernel, dim3(blocks_for(words, 1024, 128)), dim3(256), 0, s, words, zcb.as<uint2>(),
                           dbits.as<unsigned long long>());
        DQ_LAUNCH_CHECK();
        DQ_HIP(hipMemcpyAsync(&bits, dbits.p, sizeof(bits), hipMemcpyDeviceToHost, s));
    }
    DQ_HIP(hipStreamSynchronize(s));  // before the work list is freed
    if (c_blocks && static_cast<int64_t>(bits) <= 2 * c_blocks - c_blocks / 4) {
        C->zmap = std::move(zcb);
        C->zmap_valid = C->zmap_loads_only = true;
    }
    return C;
}

// A^n as pow_cuda (src/spPow_gpu.cu:21-56): n = 0 gives I, n = 1 a copy, 2^s by s squarings, otherwise binary
// exponentiation starting from the first odd power.
std::unique_ptr<dq_devmat> matrix_pow(const dq_devmat &A, int64_t n, hipStream_t s) {
    if (n < 0) throw ArgError("pow_cuda: negative exponent not supported");
    if (n == 0) {
        const int32_t zero = 0;
        auto I = make_devmat(A.rows, A.rows, &zero, 1, A.precision, s);
        fill_identity(*I, s);
        return I;
    }
    if (n == 1) return copy_devmat(A, s);
    uint64_t e = static_cast<uint64_t>(n);
    std::unique_ptr<dq_devmat> base = copy_devmat(A, s);
    if ((e & (e - 1)) == 0) {
        while (e > 1) {
            base = product(*base, *base, 1.0, s, true);
            e >>= 1;
        }
        return base;
    }
    std::unique_ptr<dq_devmat> result;
    while (e > 0) {
        if (e & 1ULL) result = result ? product(*result, *base, 1.0, s, true) : copy_devmat(*base, s);
        e >>= 1ULL;
        if (e) base = product(*base, *base, 1.0, s, true);
    }
    return result;
}

}  // namespace dq

using namespace dq;

extern "C" int dq_product_dryrun(uint32_t rows, uint32_t cols, int32_t n_a, const int32_t *offs_a, int32_t n_b,
                                 const int32_t *offs_b, int32_t *n_res, int64_t *n_pairs, int32_t *res_offsets,
                                 int64_t *res_pair_start, int32_t *pair_slot_a, int32_t *pair_slot_b) {
    return guard([&] {
        if (n_a < 0 || n_b < 0) throw ArgError("negative diagonal count");
        if ((n_a && !offs_a) || (n_b && !offs_b)) throw ArgError("NULL offsets");
        const DryRun d = dryrun(rows, cols, std::vector<int32_t>(offs_a, offs_a + n_a),
                                std::vector<int32_t>(offs_b, offs_b + n_b));
        if (n_res) *n_res = static_cast<int32_t>(d.res.size());
        if (n_pairs) *n_pairs = static_cast<int64_t>(d.sa.size());
        if (res_offsets) {
            std::copy(d.res.begin(), d.res.end(), res_offsets);
            if (res_pair_start) std::copy(d.pair_start.begin(), d.pair_start.end(), res_pair_start);
            if (pair_slot_a) std::copy(d.sa.begin(), d.sa.end(), pair_slot_a);
            if (pair_slot_b) std::copy(d.sb.begin(), d.sb.end(), pair_slot_b);
        }
    });
}

namespace dq {
// Called by dq_set_tuning for the "product_*" keys.
bool product_set_tuning(const std::string &key, int value) {
    if (key == "product_interleave") {
        if (value < 0 || value > 1) throw ArgError("product_interleave must be 0 or 1");
        g_prod_interleave = value;
        return true;
    }
    if (key == "product_rows_per_lane") {
        if (value != 0 && value != 4 && value != 8 && value != 16)
            throw ArgError("product_rows_per_lane must be 0 (automatic), 4, 8 or 16");
        g_prod_rpt = value;
        return true;
    }
    if (key == "product_skip_zero_blocks") {
        if (value < 0 || value > 1) throw ArgError("product_skip_zero_blocks must be 0 or 1");
        g_prod_skip = value;
        return true;
    }
    if (key == "product_nt_store") {
        if (value < 0 || value > 1) throw ArgError("product_nt_store must be 0 or 1");
        g_prod_nt_store = value;
        return true;
    }
    return false;
}
}  // namespace dq

extern "C" int dq_product_device(const dq_devmat *A, const dq_devmat *B, dq_devmat **out) {
    return guard([&] {
        if (!A || !B || !out) throw ArgError("NULL argument");
        *out = product(*A, *B, 1.0, 0, false, true).release();
    });
}

extern "C" int dq_pow(const dq_devmat *A, int64_t n, dq_devmat **out) {
    return guard([&] {
        if (!A || !out) throw ArgError("NULL argument");
        *out = matrix_pow(*A, n, 0).release();
        DQ_HIP(hipStreamSynchronize(0));
    });
}
