// grid.hip -- counting sort into cells, scans, permutations and the
// 27-cell neighbour sweep (see grid.hpp).
#include <algorithm>
#include <cmath>

#include "grid.hpp"

namespace sph {

GridDesc make_grid(const double lo[3], const double hi[3], double radius, size_t max_cells, int sub) {
    SPH_REQUIRE(sub >= 1 && sub <= 16, SPH_ERR_INVALID, "grid: x subdivision out of range");
    double cs = radius * (1.0 + 1e-4);
    GridDesc g{};
    for (int it = 0; it < 64; it++) {
        size_t total = 1;
        int n[3];
        for (int c = 0; c < 3; c++) {
            const double ext = (hi[c] - lo[c]) + 2.0 * cs;
            n[c] = std::max(1, (int)std::ceil(ext / cs)) * (c == 0 ? sub : 1);
            total *= (size_t)n[c];
        }
        if (total <= max_cells) {
            g.ox = (float)(lo[0] - cs);
            g.oy = (float)(lo[1] - cs);
            g.oz = (float)(lo[2] - cs);
            g.inv = (float)(1.0 / cs);
            g.invx = (float)(sub / cs);
            g.edge = (float)(cs * (1.0 - 1e-6));
            g.nx = n[0];
            g.ny = n[1];
            g.nz = n[2];
            g.sub = sub;
            // An FP32 cell coordinate t = (x - o) / edge is within 2^-23 |t|
            // of the exact one, so two of them differ from the exact
            // difference by at most 2.4e-7 times the grid extent in cells.
            g.teps = (float)(3e-7 * std::max(n[1], n[2]) + 1e-5);
            g.tepsx = (float)(3e-7 * n[0] + 1e-5);
            g.ncells = (unsigned)total;
            return g;
        }
        cs *= 1.26;
    }
    throw Error(SPH_ERR_INVALID, "grid: domain too large");
}

// ------------------------------------------------------------------ kernels
__global__ void k_fill_u32(unsigned *p, size_t n, unsigned v) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

constexpr int SCAN_ITEMS = 4;
constexpr int SCAN_TILE = BLOCK * SCAN_ITEMS;

__device__ __forceinline__ unsigned wave_incl_scan(unsigned v) {
    const int lane = threadIdx.x & 63;
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

// Exclusive scan of a tile of SCAN_TILE values held SCAN_ITEMS per thread;
// returns the thread's exclusive offset within the tile, and the tile total.
__device__ __forceinline__ unsigned block_excl_scan(unsigned tsum, unsigned &total) {
    __shared__ unsigned wsum[BLOCK / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const unsigned incl = wave_incl_scan(tsum);
    if (lane == 63) wsum[wid] = incl;
    __syncthreads();
    unsigned before = 0, tot = 0;
    for (int w = 0; w < BLOCK / 64; w++) {
        if (w < wid) before += wsum[w];
        tot += wsum[w];
    }
    __syncthreads();
    total = tot;
    return before + incl - tsum;
}

__global__ __launch_bounds__(BLOCK) void k_scan_local(const unsigned *__restrict__ in, unsigned *__restrict__ out,
                                                      unsigned n, unsigned *__restrict__ bsum) {
    const size_t base = (size_t)blockIdx.x * SCAN_TILE + (size_t)threadIdx.x * SCAN_ITEMS;
    unsigned v[SCAN_ITEMS], s = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) {
        v[k] = (base + k < n) ? in[base + k] : 0u;
        s += v[k];
    }
    unsigned total;
    unsigned off = block_excl_scan(s, total);
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) {
        if (base + k < n) out[base + k] = off;
        off += v[k];
    }
    if (threadIdx.x == 0) bsum[blockIdx.x] = total;
}

// One block scans nb values (exclusive; out may be in) and writes their total
// to *total_out.
__global__ __launch_bounds__(BLOCK) void k_scan_one(const unsigned *in, unsigned *out, unsigned nb,
                                                    unsigned *__restrict__ total_out) {
    unsigned carry = 0;
    for (unsigned t0 = 0; t0 < nb; t0 += SCAN_TILE) {
        const unsigned base = t0 + threadIdx.x * SCAN_ITEMS;
        unsigned v[SCAN_ITEMS], s = 0;
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; k++) {
            v[k] = (base + k < nb) ? in[base + k] : 0u;
            s += v[k];
        }
        unsigned total;
        unsigned off = block_excl_scan(s, total) + carry;
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; k++) {
            if (base + k < nb) out[base + k] = off;
            off += v[k];
        }
        carry += total;
        __syncthreads();
    }
    if (threadIdx.x == 0) *total_out = carry;
}

__global__ __launch_bounds__(BLOCK) void k_scan_add(unsigned *__restrict__ out, unsigned n,
                                                    const unsigned *__restrict__ bsum) {
    const size_t base = (size_t)blockIdx.x * SCAN_TILE + (size_t)threadIdx.x * SCAN_ITEMS;
    const unsigned add = bsum[blockIdx.x];
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++)
        if (base + k < n) out[base + k] += add;
}

// k_scan_add on the unscanned totals: each block sums those before its own,
// and the last one writes the grand total.
__global__ __launch_bounds__(BLOCK) void k_scan_finish(unsigned *__restrict__ out, unsigned n,
                                                       const unsigned *__restrict__ bsum) {
    unsigned before = 0, add;
    for (unsigned b = threadIdx.x; b < blockIdx.x; b += BLOCK) before += bsum[b];
    (void)block_excl_scan(before, add);
    const size_t base = (size_t)blockIdx.x * SCAN_TILE + (size_t)threadIdx.x * SCAN_ITEMS;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++)
        if (base + k < n) out[base + k] += add;
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = add + bsum[blockIdx.x];
}

// Launches are what a small scan costs, about 4 us each (a search among 1,000
// points 130 -> 117 us, among 512k 431 -> 422 us, without them): up to SCAN_ONE
// values one block scans them all, and up to SCAN_SUMS tiles the blocks of
// the second launch sum the totals before their own, which reads at most 16
// a thread; only beyond that do the totals get a scan of their own.
constexpr unsigned SCAN_ONE = 4 * SCAN_TILE, SCAN_SUMS = 16 * BLOCK;

// ---------------------------------------------------------- radix sort
// Stable LSD radix sort of the cell keys, 8 bits per pass, 1024 keys per
// block. Points start in index order and every pass is stable, so each cell
// ends up ordered by point index whatever the cell sizes (a dense cluster
// costs no more than a uniform cloud) and no atomic order leaks into it.
constexpr int RADIX = 256;
constexpr int RROUNDS = 4;
constexpr unsigned RTILE = BLOCK * RROUNDS;
static_assert(BLOCK == RADIX, "one thread per digit");

__global__ __launch_bounds__(BLOCK) void k_cell_keys(const float4 *__restrict__ x, unsigned n, GridDesc g,
                                                     unsigned *__restrict__ key) {
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) key[i] = cell_id(cell_of(x[i], g), g);
}

// hist[d * nb + b] = keys of block b with digit d.
__global__ __launch_bounds__(BLOCK) void k_radix_hist(const unsigned *__restrict__ key, unsigned n, int shift,
                                                      unsigned nb, unsigned *__restrict__ hist) {
    __shared__ unsigned h[RADIX];
    const unsigned t = threadIdx.x;
    h[t] = 0u;
    __syncthreads();
    const size_t base = (size_t)blockIdx.x * RTILE;
#pragma unroll
    for (int r = 0; r < RROUNDS; r++) {
        const size_t idx = base + (size_t)r * BLOCK + t;
        if (idx < n) atomicAdd(&h[(key[idx] >> shift) & (RADIX - 1)], 1u);
    }
    __syncthreads();
    hist[(size_t)t * nb + blockIdx.x] = h[t];
}

// Stable scatter of one pass: an element's slot is its digit's offset for
// the block plus the number of same-digit elements before it in the block
// (earlier rounds, earlier waves, lower lanes). Lanes with the same digit
// are found with eight ballots.
__global__ __launch_bounds__(BLOCK) void k_radix_scatter(const unsigned *__restrict__ kin,
                                                         const unsigned *__restrict__ vin, unsigned n, int shift,
                                                         unsigned nb, const unsigned *__restrict__ hoff,
                                                         unsigned *__restrict__ kout, unsigned *__restrict__ vout) {
    __shared__ unsigned run[RADIX];
    __shared__ unsigned wc[BLOCK / 64][RADIX];
    const unsigned t = threadIdx.x, w = t >> 6, lane = t & 63u;
    run[t] = hoff[(size_t)t * nb + blockIdx.x];
    const size_t base = (size_t)blockIdx.x * RTILE;
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64u - lane));
    for (int r = 0; r < RROUNDS; r++) {
#pragma unroll
        for (int q = 0; q < BLOCK / 64; q++) wc[q][t] = 0u;
        __syncthreads();
        const size_t idx = base + (size_t)r * BLOCK + t;
        const bool valid = idx < n;
        const unsigned k = valid ? kin[idx] : 0u;
        const unsigned d = (k >> shift) & (RADIX - 1);
        unsigned long long m = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (d >> b) & 1u;
            const unsigned long long bb = __ballot(bit);
            m &= bit ? bb : ~bb;
        }
        const unsigned long long lower = m & below;
        const unsigned rank = (unsigned)__popcll(lower);
        if (valid && lower == 0ull) wc[w][d] = (unsigned)__popcll(m);
        __syncthreads();
        {
            unsigned acc = run[t];
#pragma unroll
            for (int q = 0; q < BLOCK / 64; q++) {
                const unsigned c = wc[q][t];
                wc[q][t] = acc;
                acc += c;
            }
            run[t] = acc;
        }
        __syncthreads();
        if (valid) {
            const unsigned pos = wc[w][d] + rank;
            kout[pos] = k;
            vout[pos] = vin ? vin[idx] : (unsigned)idx;
        }
        __syncthreads();
    }
}

// start[c] = first slot whose key is >= c, c = 0 .. ncells; start[ncells] =
// n. A thread covers START_CELLS consecutive cells: one binary search in the
// sorted keys for the first, then a walk over the few points of the others.
constexpr unsigned START_CELLS = 4;
__global__ __launch_bounds__(BLOCK) void k_cell_start(const unsigned *__restrict__ key, unsigned n, unsigned ncells,
                                                      unsigned *__restrict__ start) {
    const unsigned c0 = (blockIdx.x * blockDim.x + threadIdx.x) * START_CELLS;
    if (c0 > ncells) return;
    unsigned lo = 0, hi = n;
    while (lo < hi) {
        const unsigned mid = (lo + hi) >> 1;
        if (key[mid] < c0)
            lo = mid + 1;
        else
            hi = mid;
    }
    start[c0] = lo;
    for (unsigned c = c0 + 1; c < c0 + START_CELLS && c <= ncells; c++) {
        while (lo < n && key[lo] < c) lo++;
        start[c] = lo;
    }
}

template <class T>
__global__ __launch_bounds__(BLOCK) void k_permute(const unsigned *__restrict__ perm, unsigned n,
                                                   const T *__restrict__ src, T *__restrict__ dst) {
    const unsigned k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) dst[k] = src[perm[k]];
}

// Neighbour sweep, one thread per query, column-major output (neighbour k
// of query i at nbr[k * stride + i]). A query visits the 9 (dy, dz) rows of
// its neighbourhood; each row is one contiguous slot range, trimmed in x to
// the sub-cells the query can reach (row_ranges). A lane records its hits as
// one 64-bit mask per row -- bit b set = the row's b-th candidate slot is a
// neighbour -- and the wave then emits the lists row by row: at output row k
// every lane writes its k-th neighbour, so each store is 64 consecutive
// words (one coalesced 256-B write) rather than scattered 4-byte appends
// that leave partial cache lines behind. Masks and row bases sit in LDS
// (6.75 KiB per wave, independent of the list capacity), so the LDS never
// limits the resident waves. The order of a list is row by row, ascending
// slot within a row.
//
// When no row of the wave holds more than 64 candidates, the wave walks
// each row in lockstep: candidate b of every lane is tested at the same
// step, so the mask bit is a shift-and-add of the test, the four loads of a
// step share one address computation, and a lane's own slot is cleared from
// its mask once at the end. A wave with a longer row walks its rows in the
// same lockstep, 32 steps to a hit word, and each lane stores the entries of
// a word directly as it finds them (the lists of dense clusters outgrow the
// LDS masks); such a build writes no packed copy (it reports the overflow
// flag instead).
constexpr unsigned LIST_ROWS = 9;

// Slot range [s, e) of the (dy, dz) row around xi. A point of row
// (cy + dy, cz + dz) lies at least the y-z distance of that row's cells from
// xi (d_yz), hence within x half-width sqrt(r^2 - d_yz^2) of xi if it is a
// neighbour; the row is cut to the x sub-cells that half-width reaches, and
// dropped when d_yz > r. Distances are taken from the FP32 cell coordinates
// the sort used, narrowed by their rounding margin, and r2t sits above the
// FP64 inclusion radius, so no point within the radius is ever cut.
struct RowQuery {
    float tx, dyl, dyh, dzl, dzh, xlo, xhi;
    int cy, cz;
};
__device__ __forceinline__ RowQuery row_query(const float4 &xi, const GridDesc &g) {
    RowQuery q;
    const float ty = (xi.y - g.oy) * g.inv, tz = (xi.z - g.oz) * g.inv;
    q.tx = (xi.x - g.ox) * g.invx;
    const int cx = clampi((int)floorf(q.tx), 0, g.nx - 1);
    q.cy = clampi((int)floorf(ty), 0, g.ny - 1);
    q.cz = clampi((int)floorf(tz), 0, g.nz - 1);
    const float fy = ty - (float)q.cy, fz = tz - (float)q.cz;
    // distance in cells from xi to the row below / above, lower bounds
    q.dyl = fmaxf(fy - g.teps, 0.0f), q.dyh = fmaxf(1.0f - fy - g.teps, 0.0f);
    q.dzl = fmaxf(fz - g.teps, 0.0f), q.dzh = fmaxf(1.0f - fz - g.teps, 0.0f);
    q.xlo = (float)(cx > g.sub ? cx - g.sub : 0);
    q.xhi = (float)(cx < g.nx - 1 - g.sub ? cx + g.sub : g.nx - 1);
    return q;
}
__device__ __forceinline__ void row_range(const RowQuery &q, const GridDesc &g, float r2t, int dy, int dz,
                                          const unsigned *__restrict__ start, unsigned &s_r, unsigned &e_r) {
    const int z = q.cz + dz, y = q.cy + dy;
    const float a = dy < 0 ? q.dyl : (dy > 0 ? q.dyh : 0.0f), b = dz < 0 ? q.dzl : (dz > 0 ? q.dzh : 0.0f);
    const float w2 = r2t - (a * a + b * b) * (g.edge * g.edge);
    const bool ok = z >= 0 && z < g.nz && y >= 0 && y < g.ny && w2 >= 0.0f;
    const float wx = sqrtf(fmaxf(w2, 0.0f)) * g.invx + g.tepsx;
    // both ends clamped into the stencil: points outside the grid sit in its
    // border sub-cells, so a query beyond the border still reaches them;
    // xlo <= x0 <= x1 <= xhi
    const int x0 = (int)floorf(fminf(fmaxf(q.tx - wx, q.xlo), q.xhi));
    const int x1 = (int)floorf(fminf(fmaxf(q.tx + wx, q.xlo), q.xhi));
    // rows outside the grid read a clamped row and come out empty (no
    // branch: a stored-through select would put the caller's arrays in
    // scratch memory)
    const unsigned row =
        ((unsigned)clampi(z, 0, g.nz - 1) * (unsigned)g.ny + (unsigned)clampi(y, 0, g.ny - 1)) * (unsigned)g.nx;
    const unsigned s = start[row + x0], e = start[row + x1 + 1];
    s_r = ok ? s : 0u;
    e_r = ok ? e : 0u;
}
// All 9 rows, dz slowest.
__device__ __forceinline__ void row_ranges(const float4 &xi, const GridDesc &g, float r2t,
                                           const unsigned *__restrict__ start, unsigned s_r[LIST_ROWS],
                                           unsigned e_r[LIST_ROWS]) {
    const RowQuery q = row_query(xi, g);
    unsigned rr = 0;
#pragma unroll
    for (int dz = -1; dz <= 1; dz++)
#pragma unroll
        for (int dy = -1; dy <= 1; dy++, rr++) row_range(q, g, r2t, dy, dz, start, s_r[rr], e_r[rr]);
}

// Inclusion is decided exactly for the FP32 coordinates: a squared distance
// within FP32 rounding of r^2 (between r2lo and r2hi) is recomputed in FP64
// from the same coordinates, as an FP64 search computes it.
__device__ __forceinline__ bool inside_d(const float4 &xi, const float4 &xj, double r2d) {
    const double ex = (double)xi.x - (double)xj.x, ey = (double)xi.y - (double)xj.y,
                 ez = (double)xi.z - (double)xj.z;
    return (ex * ex + ey * ey) + ez * ez < r2d;
}

template <bool SAME>
__global__ __launch_bounds__(BLOCK) void k_lists_cm(const float4 *__restrict__ q, unsigned nq,
                                                    const float4 *__restrict__ src,
                                                    const unsigned *__restrict__ start, GridDesc g, float r2lo,
                                                    float r2hi, float r2t, double r2d, unsigned *__restrict__ nbr,
                                                    unsigned stride, unsigned cap, unsigned *__restrict__ cnt,
                                                    unsigned *__restrict__ maxcnt, unsigned *__restrict__ nbr16,
                                                    unsigned *__restrict__ ovf16) {
    __shared__ unsigned rowbase[BLOCK / 64][LIST_ROWS][64];
    __shared__ unsigned long long masks[BLOCK / 64][LIST_ROWS][64];
    const unsigned lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    const unsigned i = xcd_block() * blockDim.x + threadIdx.x;
    const bool act = i < nq;
    unsigned k = 0;
    bool wide = false;
    // packed copy: entry t of the list as the 16-bit difference j - i, two
    // per word (word t / 2, entry t in the low half when t is even)
    unsigned plo = 0;
    bool far = false;
    auto pack = [&](unsigned t, unsigned j) {
        const int d = (int)j - (int)i;
        far |= (unsigned)(d + 32768) > 65535u;
        const unsigned h16 = (unsigned)d & 0xffffu;
        if (t & 1u)
            nbr16[(size_t)(t >> 1) * stride + i] = plo | (h16 << 16);
        else
            plo = h16;
    };
    const float4 xi = act ? q[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    unsigned s_r[LIST_ROWS], e_r[LIST_ROWS];
    if (act) {
        row_ranges(xi, g, r2t, start, s_r, e_r);
    } else {
#pragma unroll
        for (unsigned r = 0; r < LIST_ROWS; r++) s_r[r] = e_r[r] = 0u;
    }
#pragma unroll
    for (unsigned r = 0; r < LIST_ROWS; r++)
        if (e_r[r] - s_r[r] > 64u) wide = true;

    const bool wwide = __ballot(wide) != 0ull;
    if (!wwide) {
        // ---- lockstep rows (every row of the wave within 64 candidates)
        const unsigned nsrc = start[g.ncells];
        const __amdgpu_buffer_rsrc_t X = __builtin_amdgcn_make_buffer_rsrc(const_cast<float4 *>(src), (short)0,
                                                                           (int)(nsrc * 16u), 0x00020000);
        unsigned bandrows = 0;
#pragma unroll
        for (unsigned r = 0; r < LIST_ROWS; r++) {
            const unsigned s0 = s_r[r], len = e_r[r] - s0;
            const unsigned T = __builtin_amdgcn_readfirstlane(wave_max_u(len));
            const unsigned vb = s0 << 4;
            unsigned wd[2] = {0u, 0u};
            bool band = false;
            // m = 2 m + hit: after the word's c steps, step b sits at bit c - 1 - b
            auto test = [&](unsigned &m, const sph_v3u v) {
                const float dx = xi.x - __uint_as_float(v.x), dy = xi.y - __uint_as_float(v.y),
                            dz = xi.z - __uint_as_float(v.z);
                const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                const bool in = d2 < r2lo;
                band |= (d2 < r2hi) & !in;
                m = m + m + (unsigned)in;
            };
#pragma unroll
            for (unsigned wv = 0; wv < 2; wv++) {
                const unsigned tb = 32u * wv;
                if (tb >= T) break;
                // steps in chunks of eight loads in flight together; the
                // steps past T read slots whose bits are dropped below
                const unsigned T8 = (T + 7u) & ~7u, te = T8 < tb + 32u ? T8 : tb + 32u;
                unsigned m = 0u;
                for (unsigned t = tb; t < te; t += 8u) {
                    const unsigned o = vb + (t << 4);
                    const sph_v3u c0 = __builtin_amdgcn_raw_buffer_load_b96(X, o, 0, 0);
                    const sph_v3u c1 = __builtin_amdgcn_raw_buffer_load_b96(X, o + 16u, 0, 0);
                    const sph_v3u c2 = __builtin_amdgcn_raw_buffer_load_b96(X, o + 32u, 0, 0);
                    const sph_v3u c3 = __builtin_amdgcn_raw_buffer_load_b96(X, o + 48u, 0, 0);
                    const sph_v3u c4 = __builtin_amdgcn_raw_buffer_load_b96(X, o + 64u, 0, 0);
                    const sph_v3u c5 = __builtin_amdgcn_raw_buffer_load_b96(X, o + 80u, 0, 0);
                    const sph_v3u c6 = __builtin_amdgcn_raw_buffer_load_b96(X, o + 96u, 0, 0);
                    const sph_v3u c7 = __builtin_amdgcn_raw_buffer_load_b96(X, o + 112u, 0, 0);
                    test(m, c0);
                    test(m, c1);
                    test(m, c2);
                    test(m, c3);
                    test(m, c4);
                    test(m, c5);
                    test(m, c6);
                    test(m, c7);
                }
                // step b to bit b, then keep the lane's own candidates
                m = __builtin_bitreverse32(m << (32u - (te - tb)));
                const unsigned nb = len > tb ? len - tb : 0u;
                wd[wv] = nb >= 32u ? m : (m & ((1u << nb) - 1u));
            }
            unsigned long long mk = (unsigned long long)wd[0] | ((unsigned long long)wd[1] << 32);
            if (SAME && r == LIST_ROWS / 2 && act) mk &= ~(1ull << (i - s0));
            if (band) bandrows |= 1u << r;
            rowbase[wid][r][lane] = s0;
            masks[wid][r][lane] = mk;
        }
        if (bandrows != 0u) {
            // candidates within rounding of the radius: decide in FP64
#pragma unroll
            for (unsigned r = 0; r < LIST_ROWS; r++) {
                if (!((bandrows >> r) & 1u)) continue;
                const unsigned s0 = s_r[r], len = e_r[r] - s0;
                unsigned long long mk = masks[wid][r][lane];
                for (unsigned b = 0; b < len; b++) {
                    const float4 xj = src[s0 + b];
                    const float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
                    const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                    if (d2 < r2hi && !(d2 < r2lo) && inside_d(xi, xj, r2d)) mk |= 1ull << b;
                }
                masks[wid][r][lane] = mk;
            }
        }
#pragma unroll
        for (unsigned r = 0; r < LIST_ROWS; r++) k += (unsigned)__popcll(masks[wid][r][lane]);
        if (act) cnt[i] = k;
    } else {
        // ---- lockstep rows of any length, entries stored as found
        const unsigned nsrc = start[g.ncells];
        const __amdgpu_buffer_rsrc_t X = __builtin_amdgcn_make_buffer_rsrc(const_cast<float4 *>(src), (short)0,
                                                                           (int)(nsrc * 16u), 0x00020000);
#pragma unroll
        for (unsigned r = 0; r < LIST_ROWS; r++) {
            const unsigned s0 = s_r[r], len = e_r[r] - s0;
            const unsigned T = __builtin_amdgcn_readfirstlane(wave_max_u(len));
            const unsigned T8 = (T + 7u) & ~7u;
            for (unsigned tb = 0; tb < T; tb += 32u) {
                const unsigned te = T8 < tb + 32u ? T8 : tb + 32u;
                unsigned m = 0u;
                bool band = false;
                for (unsigned t = tb; t < te; t += 8u) {
                    const unsigned o = (s0 + t) << 4;
                    sph_v3u c[8];
#pragma unroll
                    for (unsigned u = 0; u < 8u; u++) c[u] = __builtin_amdgcn_raw_buffer_load_b96(X, o + 16u * u, 0, 0);
#pragma unroll
                    for (unsigned u = 0; u < 8u; u++) {
                        const float dx = xi.x - __uint_as_float(c[u].x), dy = xi.y - __uint_as_float(c[u].y),
                                    dz = xi.z - __uint_as_float(c[u].z);
                        const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                        const bool in = d2 < r2lo;
                        band |= (d2 < r2hi) & !in;
                        m = m + m + (unsigned)in;
                    }
                }
                m = __builtin_bitreverse32(m << (32u - (te - tb)));
                const unsigned nb = len > tb ? (len - tb < 32u ? len - tb : 32u) : 0u;
                m = nb >= 32u ? m : (m & ((1u << nb) - 1u));
                if (SAME && r == LIST_ROWS / 2 && act && i - s0 - tb < 32u) m &= ~(1u << (i - s0 - tb));
                if (band) {
                    // candidates within rounding of the radius: decide in FP64
                    for (unsigned b = 0; b < nb; b++) {
                        const float4 xj = src[s0 + tb + b];
                        const float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
                        const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                        if (d2 < r2hi && !(d2 < r2lo) && inside_d(xi, xj, r2d)) m |= 1u << b;
                    }
                }
                while (m != 0u) {
                    const unsigned j = s0 + tb + (unsigned)__builtin_ctz(m);
                    m &= m - 1u;
                    if (k < cap) nbr[(size_t)k * stride + i] = j;
                    k++;
                }
            }
        }
        if (act) cnt[i] = k;
        // no packed copy for dense waves: their scattered stores bound the
        // build, and the sweeps read the 32-bit lists instead
        far = true;
    }
    const unsigned kk = (act && !wwide) ? (k < cap ? k : cap) : 0u;
    const unsigned mx = wave_max_u(kk);
    unsigned r = 0;
    unsigned long long cur = kk ? masks[wid][0][lane] : 0ull;
    for (unsigned t = 0; t < mx; t++) {
        if (t < kk) {
            while (cur == 0ull) {
                r++;
                cur = masks[wid][r][lane];
            }
            const unsigned b = (unsigned)__builtin_ctzll(cur);
            cur &= cur - 1ull;
            const unsigned j = rowbase[wid][r][lane] + b;
            nbr[(size_t)t * stride + i] = j;
            if (nbr16) pack(t, j);
        }
    }
    if (nbr16) {
        if (kk & 1u) nbr16[(size_t)(kk >> 1) * stride + i] = plo;
        if (__ballot(far) != 0ull && lane == 0) atomicOr(ovf16, 1u);
    }
    const unsigned mk = wave_max_u(act ? k : 0u);
    if (lane == 0 && mk > 0) atomicMax(maxcnt, mk);
}

// ------------------------------------------------- CSR lists (drop-in search)
// The inclusion test of the drop-in search: FP32, every operation rounded.
__device__ __forceinline__ bool csr_inside(const float4 &xi, float x, float y, float z, float r2) {
    const float dx = xi.x - x, dy = xi.y - y, dz = xi.z - z;
    return (dx * dx + dy * dy) + dz * dz < r2;
}

// One wave per query: the lanes test 64 consecutive candidates of a row at
// once, and the ballot of the hits gives each its place in the list, so the
// stores are contiguous and in slot order. The first 64 candidates of all 9
// rows are loaded together (one memory latency for the usual query); longer
// rows follow in windows of 256. Bound by latency for small clouds and by
// instruction issue (about 200 per query at 35 neighbours) for large ones.
// A lane per query that walked its 27 cells alone took 80-99 us a pass for
// 1,000 points and 0.8-0.9 ms for 50k clustered ones (K = 225).
template <bool SAME, bool FILL>
__global__ __launch_bounds__(BLOCK) void k_csr_wave(const float4 *__restrict__ q, const unsigned *__restrict__ qmap,
                                                    unsigned nq, const float4 *__restrict__ src, unsigned nsrc,
                                                    const unsigned *__restrict__ srcmap,
                                                    const unsigned *__restrict__ start, GridDesc g, float r2,
                                                    float r2t, const unsigned *__restrict__ rowoff,
                                                    unsigned *__restrict__ out, unsigned *__restrict__ cnt, unsigned w0) {
    const unsigned lane = threadIdx.x & 63u;
    const unsigned wl = __builtin_amdgcn_readfirstlane(xcd_block() * (BLOCK / 64) + (threadIdx.x >> 6));
    if (wl >= nq - w0) return;
    const unsigned w = w0 + wl;
    const float4 xi = q[w];
    const unsigned i = qmap ? qmap[w] : w;
    unsigned sv = 0u, ev = 0u;
    if (lane < LIST_ROWS) {
        const RowQuery rq = row_query(xi, g);
        row_range(rq, g, r2t, (int)(lane % 3u) - 1, (int)(lane / 3u) - 1, start, sv, ev);
    }
    unsigned s_r[LIST_ROWS], e_r[LIST_ROWS];
    float4 c[LIST_ROWS];
#pragma unroll
    for (unsigned r = 0; r < LIST_ROWS; r++) {
        s_r[r] = __builtin_amdgcn_readlane(sv, r);
        e_r[r] = __builtin_amdgcn_readlane(ev, r);
        if (s_r[r] + lane < e_r[r]) c[r] = src[s_r[r] + lane];
    }
    unsigned k = 0;
    const unsigned o = FILL ? rowoff[i] : 0u;
    const unsigned long long below = (1ull << lane) - 1ull;
    auto window = [&](unsigned j, unsigned e, const float4 &xj) {
        const bool hit = j < e && !(SAME && j == w) && csr_inside(xi, xj.x, xj.y, xj.z, r2);
        const unsigned long long m = __ballot(hit);
        if (FILL && hit) out[o + k + (unsigned)__popcll(m & below)] = srcmap[j];
        k += (unsigned)__popcll(m);
    };
#pragma unroll
    for (unsigned r = 0; r < LIST_ROWS; r++) {
        window(s_r[r] + lane, e_r[r], c[r]);
        for (unsigned t = s_r[r] + 64u; t < e_r[r]; t += 256u) {
            float4 d[4];
#pragma unroll
            for (unsigned u = 0; u < 4u; u++)
                if (t + 64u * u + lane < e_r[r]) d[u] = src[t + 64u * u + lane];
#pragma unroll
            for (unsigned u = 0; u < 4u; u++) window(t + 64u * u + lane, e_r[r], d[u]);
        }
    }
    if (!FILL && lane == 0) cnt[i] = k;
}

// One lane per query, the rows of a wave walked in lockstep as in
// k_lists_cm: eight candidate loads in flight and a hit word of up to 32
// steps, whose entries are stored right away. A lane keeps the last (up to
// four) entries in registers and writes them as one 16-byte store once they
// fill an aligned group: single 4-byte stores of 64 lanes go to 64 lines
// each, and those write requests would bound the pass. 524k uniform points
// (K = 34): the search went from 3.61 to 0.44 ms with it.
template <bool SAME, bool FILL>
__global__ __launch_bounds__(BLOCK) void k_csr_lanes(const float4 *__restrict__ q, const unsigned *__restrict__ qmap,
                                                     unsigned nq, const float4 *__restrict__ src, unsigned nsrc,
                                                     const unsigned *__restrict__ srcmap,
                                                     const unsigned *__restrict__ start, GridDesc g, float r2,
                                                     float r2t, const unsigned *__restrict__ rowoff,
                                                     unsigned *__restrict__ out, unsigned *__restrict__ cnt) {
    const unsigned w = xcd_block() * blockDim.x + threadIdx.x;
    const bool act = w < nq;
    const float4 xi = act ? q[w] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const unsigned i = act ? (qmap ? qmap[w] : w) : 0u;
    unsigned s_r[LIST_ROWS], e_r[LIST_ROWS];
    if (act) {
        row_ranges(xi, g, r2t, start, s_r, e_r);
    } else {
#pragma unroll
        for (unsigned r = 0; r < LIST_ROWS; r++) s_r[r] = e_r[r] = 0u;
    }
    const __amdgpu_buffer_rsrc_t X = __builtin_amdgcn_make_buffer_rsrc(const_cast<float4 *>(src), (short)0,
                                                                       (int)(nsrc * 16u), 0x00020000);
    // positions count from the 16-byte group that holds out[0]
    const unsigned phase = FILL ? ((unsigned)(reinterpret_cast<size_t>(out) >> 2) & 3u) : 0u;
    unsigned *const base = FILL ? out - phase : nullptr;
    unsigned pos = (FILL && act) ? rowoff[i] + phase : 0u, fl = pos, k = 0;
    unsigned b[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (unsigned r = 0; r < LIST_ROWS; r++) {
        const unsigned s0 = s_r[r], len = e_r[r] - s0;
        const unsigned T = __builtin_amdgcn_readfirstlane(wave_max_u(len));
        const unsigned T8 = (T + 7u) & ~7u;
        for (unsigned tb = 0; tb < T; tb += 32u) {
            const unsigned te = T8 < tb + 32u ? T8 : tb + 32u;
            unsigned m = 0u;
            for (unsigned t = tb; t < te; t += 8u) {
                const unsigned at = (s0 + t) << 4;
                sph_v3u c[8];
#pragma unroll
                for (unsigned u = 0; u < 8u; u++) c[u] = __builtin_amdgcn_raw_buffer_load_b96(X, at + 16u * u, 0, 0);
#pragma unroll
                for (unsigned u = 0; u < 8u; u++)
                    m = m + m + (unsigned)csr_inside(xi, __uint_as_float(c[u].x), __uint_as_float(c[u].y),
                                                     __uint_as_float(c[u].z), r2);
            }
            // step b to bit b, then keep the lane's own candidates
            m = __builtin_bitreverse32(m << (32u - (te - tb)));
            const unsigned nb = len > tb ? len - tb : 0u;
            m = nb >= 32u ? m : (m & ((1u << nb) - 1u));
            if (SAME && r == LIST_ROWS / 2 && act && w - s0 - tb < 32u) m &= ~(1u << (w - s0 - tb));
            if (!FILL) {
                k += (unsigned)__popc(m);
                continue;
            }
            while (__ballot(m != 0u) != 0ull) {
#pragma unroll
                for (unsigned u = 0; u < 4u; u++)
                    if (m != 0u && (pos & 3u) == u) {
                        b[u] = srcmap[s0 + tb + (unsigned)__builtin_ctz(m)];
                        m &= m - 1u;
                        pos++;
                    }
                if ((pos & 3u) == 0u && pos != fl) {
                    if (pos - fl == 4u) {
                        *reinterpret_cast<uint4 *>(base + fl) = make_uint4(b[0], b[1], b[2], b[3]);
                    } else {  // the head of the list, before the first whole group
                        if (pos - fl == 3u) base[fl] = b[1];
                        if (pos - fl >= 2u) base[pos - 2u] = b[2];
                        base[pos - 1u] = b[3];
                    }
                    fl = pos;
                }
            }
        }
    }
    if (FILL) {
        // the tail: positions fl .. pos - 1 of one group
#pragma unroll
        for (unsigned u = 0; u < 4u; u++) {
            const unsigned p = (pos & ~3u) + u;
            if (p >= fl && p < pos) base[p] = b[u];
        }
    } else if (act) {
        cnt[i] = k;
    }
}

// -------------------------------------------------------------------- host
void fill_u32(hipStream_t s, unsigned *p, size_t n, unsigned v) {
    if (n == 0) return;
    k_fill_u32<<<(unsigned)((n + BLOCK - 1) / BLOCK), BLOCK, 0, s>>>(p, n, v);
    SPH_HIP(hipGetLastError());
}

size_t scan_bsum_len(size_t n) { return std::max<size_t>((n + SCAN_TILE - 1) / SCAN_TILE, 1); }
size_t radix_hist_len(size_t n) { return (size_t)RADIX * std::max<size_t>((n + RTILE - 1) / RTILE, 1); }

void exclusive_scan_raw(hipStream_t s, const unsigned *in, unsigned *out, unsigned n, unsigned *bsum,
                        KernelTimer &T) {
    TimedScope ts(T, s, "scan");
    if (n == 0) {
        fill_u32(s, out, 1, 0u);
        return;
    }
    const unsigned nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    if (n <= SCAN_ONE) {
        k_scan_one<<<1, BLOCK, 0, s>>>(in, out, n, out + n);
    } else if (nb <= SCAN_SUMS) {
        k_scan_local<<<nb, BLOCK, 0, s>>>(in, out, n, bsum);
        k_scan_finish<<<nb, BLOCK, 0, s>>>(out, n, bsum);
    } else {
        k_scan_local<<<nb, BLOCK, 0, s>>>(in, out, n, bsum);
        k_scan_one<<<1, BLOCK, 0, s>>>(bsum, bsum, nb, out + n);
        k_scan_add<<<nb, BLOCK, 0, s>>>(out, n, bsum);
    }
    SPH_HIP(hipGetLastError());
}

void exclusive_scan(hipStream_t s, const unsigned *in, unsigned *out, unsigned n, DBuf<unsigned> &bsum,
                    KernelTimer &T) {
    bsum.reserve(scan_bsum_len(n));
    exclusive_scan_raw(s, in, out, n, bsum.get(), T);
}

void cell_sort_raw(hipStream_t s, const float4 *x, unsigned n, const GridDesc &g, const CellSortBufs &b,
                   KernelTimer &T) {
    if (!n) {
        fill_u32(s, b.start, (size_t)g.ncells + 1, 0u);
        return;
    }
    int bits = 1;
    while (bits < 32 && ((g.ncells - 1u) >> bits) != 0u) bits++;
    const int passes = (bits + 7) / 8;
    const unsigned nb = (n + RTILE - 1) / RTILE;
    // Pass p writes buffer set (passes - 1 - p) % 2 and reads the other one,
    // so the last pass lands in set 0 = (pcell, perm).
    unsigned *K[2] = {b.pcell, b.keys2};
    unsigned *V[2] = {b.perm, b.vals2};
    {
        TimedScope ts(T, s, "cell_keys");
        k_cell_keys<<<nblocks(n), BLOCK, 0, s>>>(x, n, g, K[passes % 2]);
        SPH_HIP(hipGetLastError());
    }
    for (int p = 0; p < passes; p++) {
        TimedScope ts(T, s, "cell_radix");
        const int out = (passes - 1 - p) % 2, in = 1 - out;
        k_radix_hist<<<nb, BLOCK, 0, s>>>(K[in], n, 8 * p, nb, b.hist);
        SPH_HIP(hipGetLastError());
        exclusive_scan_raw(s, b.hist, b.hoff, RADIX * nb, b.bsum, T);
        k_radix_scatter<<<nb, BLOCK, 0, s>>>(K[in], p == 0 ? nullptr : V[in], n, 8 * p, nb, b.hoff, K[out],
                                             V[out]);
        SPH_HIP(hipGetLastError());
    }
    {
        TimedScope ts(T, s, "cell_start");
        k_cell_start<<<nblocks(((size_t)g.ncells + START_CELLS) / START_CELLS), BLOCK, 0, s>>>(b.pcell, n, g.ncells,
                                                                                            b.start);
        SPH_HIP(hipGetLastError());
    }
}

void CellSorter::sort(hipStream_t s, const float4 *x, unsigned nn, const GridDesc &g, KernelTimer &T) {
    n = nn;
    grid = g;
    start.reserve((size_t)g.ncells + 1);
    const size_t cap = std::max(n, 1u);
    pcell.reserve(cap);
    keys2.reserve(cap);
    vals2.reserve(cap);
    perm.reserve(cap);
    const size_t hl = radix_hist_len(n);
    hist.reserve(hl);
    hoff.reserve(hl + 1);
    bsum.reserve(scan_bsum_len(hl));
    const CellSortBufs b{start.get(), pcell.get(), perm.get(), keys2.get(), vals2.get(),
                         hist.get(), hoff.get(), bsum.get()};
    cell_sort_raw(s, x, n, g, b, T);
}

void permute_f4(hipStream_t s, const unsigned *perm, unsigned n, const float4 *src, float4 *dst) {
    if (!n) return;
    k_permute<float4><<<nblocks(n), BLOCK, 0, s>>>(perm, n, src, dst);
    SPH_HIP(hipGetLastError());
}
void permute_u1(hipStream_t s, const unsigned *perm, unsigned n, const unsigned *src, unsigned *dst) {
    if (!n) return;
    k_permute<unsigned><<<nblocks(n), BLOCK, 0, s>>>(perm, n, src, dst);
    SPH_HIP(hipGetLastError());
}

void build_lists_colmajor(hipStream_t s, const float4 *q, unsigned nq, const float4 *src, const unsigned *start,
                          const GridDesc &g, double radius, bool same_set, unsigned *nbr, unsigned stride, unsigned cap,
                          unsigned *cnt, unsigned *maxcnt, KernelTimer &T, const char *name, unsigned *nbr16,
                          unsigned *ovf16) {
    if (!nq) return;
    SPH_REQUIRE(cap >= 1, SPH_ERR_INVALID, "neighbour capacity out of range");
    TimedScope ts(T, s, name);
    const double r2d = radius * radius;
    // FP32 evaluation error of d^2 stays below 5 units of 2^-24 (rounded
    // coordinate differences, one rounded product, two fused multiply-adds)
    const float r2lo = (float)(r2d * (1.0 - 1e-6)), r2hi = (float)(r2d * (1.0 + 1e-6));
    // row trimming reach: above r^2 by far more than the FP32 rounding of
    // the trimming arithmetic
    const float r2t = (float)(r2d * (1.0 + 1e-5));
    if (same_set)
        k_lists_cm<true><<<nblocks(nq), BLOCK, 0, s>>>(q, nq, src, start, g, r2lo, r2hi, r2t, r2d, nbr, stride, cap,
                                                       cnt, maxcnt, nbr16, ovf16);
    else
        k_lists_cm<false><<<nblocks(nq), BLOCK, 0, s>>>(q, nq, src, start, g, r2lo, r2hi, r2t, r2d, nbr, stride, cap,
                                                        cnt, maxcnt, nbr16, ovf16);
    SPH_HIP(hipGetLastError());
}

// Below this many queries a wave per query, above it a lane per query. Whole
// searches of both, wave / lane: 1k points 133 / 183 us, 50k clustered
// (K = 225) 290 / 522 us, 100k uniform (K = 33) 235 / 212 us and clustered
// (K = 260) 434 / 778 us, 131k uniform (K = 12) 258 / 181 us, 524k uniform
// (K = 34) 698 / 438 us: few lanes per SIMD leave the memory latency open,
// and a wave per query issues about four times the instructions. The line is
// that of even clouds. Long lists would keep the wave ahead beyond it (150k
// clustered, K = 168: 484 / 780 us; 500k, K = 181: 1288 / 1600), but before
// the first pass nothing tells them.
constexpr unsigned CSR_WAVE_MAX = 1u << 17;
// Queries of one launch with a wave each, of the `left` that remain: a launch
// holds fewer than 2^32 threads. (Waves that take several queries in turn are
// slower: 100k uniform points 235 -> 285 us.)
unsigned csr_wave_slice(unsigned left) { return std::min(left, 1u << 25); }

void build_lists_csr(hipStream_t s, const float4 *q, const unsigned *qmap, unsigned nq, const float4 *src,
                     unsigned nsrc, const unsigned *srcmap, const unsigned *start, const GridDesc &g, double radius, bool same_set,
                     const unsigned *rowoff, unsigned *out, unsigned *cnt) {
    if (!nq) return;
    const float r2 = (float)radius * (float)radius;
    const float r2t = (float)(radius * radius * (1.0 + 1e-5));  // row trimming reach, as in build_lists_colmajor
    // (the lanes' buffer loads address 2^28 sources)
    const bool wave = nq < CSR_WAVE_MAX || nsrc >= GATHER_MAX;
#define CSR(K, nb, SAME, FILL, ...) \
    K<SAME, FILL><<<nb, BLOCK, 0, s>>>(q, qmap, nq, src, nsrc, srcmap, start, g, r2, r2t, rowoff, out, cnt, ##__VA_ARGS__)
#define CSR_SF(K, nb, ...)                                                             \
    do {                                                                               \
        if (same_set && rowoff) CSR(K, nb, true, true, ##__VA_ARGS__);                 \
        if (same_set && !rowoff) CSR(K, nb, true, false, ##__VA_ARGS__);               \
        if (!same_set && rowoff) CSR(K, nb, false, true, ##__VA_ARGS__);               \
        if (!same_set && !rowoff) CSR(K, nb, false, false, ##__VA_ARGS__);             \
    } while (0)
    if (wave)
        for (unsigned w0 = 0, n; w0 < nq; w0 += n) {
            n = csr_wave_slice(nq - w0);
            CSR_SF(k_csr_wave, nblocks((size_t)n * 64), w0);
        }
    else
        CSR_SF(k_csr_lanes, nblocks(nq));
#undef CSR_SF
#undef CSR
    SPH_HIP(hipGetLastError());
}

}  // namespace sph
