// grid.hpp -- uniform cell grid, counting sort of points into cells and the
// neighbour-list sweep over the 27 surrounding cells.
#pragma once
#include "common.hpp"

namespace sph {

// Dense grid of cells of edge >= search radius in y and z, split into `sub`
// sub-cells along x. Cells are numbered x-fastest, so the x sub-cells
// (cx-sub..cx+sub, cy, cz) of one row are consecutive and a cell-sorted point
// array holds each row of the neighbourhood as one contiguous slot range: 9
// ranges per query. With sub > 1 a query can trim each row to the sub-cells
// within reach of its own position.
struct GridDesc {
    float ox, oy, oz;  // origin
    float inv;         // 1 / cell edge (y, z)
    float invx;        // sub / cell edge (x)
    float edge;        // cell edge, rounded down
    float teps, tepsx;  // rounding margins of FP32 cell coordinates (cells; x sub-cells)
    int nx, ny, nz;    // nx counts x sub-cells
    int sub;
    unsigned ncells;
};

// Grid covering [lo, hi] (plus one cell of margin) with cell edge
// radius * (1 + 1e-4) and `sub` sub-cells per edge along x; points outside
// are clamped to the border cells, which keeps the search exact (clamping
// never separates two points by more than one cell) at some cost in
// efficiency. The edge grows when the box would need more than max_cells
// cells.
GridDesc make_grid(const double lo[3], const double hi[3], double radius, size_t max_cells = (size_t)1 << 27,
                   int sub = 1);

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

__device__ __forceinline__ int3 cell_of(const float4 &p, const GridDesc &g) {
    return make_int3(clampi((int)floorf((p.x - g.ox) * g.invx), 0, g.nx - 1),
                     clampi((int)floorf((p.y - g.oy) * g.inv), 0, g.ny - 1),
                     clampi((int)floorf((p.z - g.oz) * g.inv), 0, g.nz - 1));
}
__device__ __forceinline__ unsigned cell_id(const int3 &c, const GridDesc &g) {
    return ((unsigned)c.z * (unsigned)g.ny + (unsigned)c.y) * (unsigned)g.nx + (unsigned)c.x;
}

// Counting sort of n points into the grid:
//   perm[slot]  = index of the point placed at `slot`
//   start[c]    = first slot of cell c, start[ncells] = n
// Points of one cell are ordered by ascending index, so the result depends
// only on the input order (no atomics order leaks into it).
class CellSorter {
public:
    DBuf<unsigned> start, pcell, perm, keys2, vals2, hist, hoff, bsum;  // pcell: sorted cell keys after sort()
    unsigned n = 0;
    GridDesc grid{};
    void sort(hipStream_t s, const float4 *x, unsigned n, const GridDesc &g, KernelTimer &T);
};

// Exclusive scan of n unsigned values into out (out[n] = total); uses bsum
// as scratch.
void exclusive_scan(hipStream_t s, const unsigned *in, unsigned *out, unsigned n, DBuf<unsigned> &bsum, KernelTimer &T);

// The same scan and cell sort on memory the caller provides (they allocate
// nothing). scan_bsum_len(n): words of bsum a scan of n values needs;
// radix_hist_len(n): words of hist (and, plus one, of hoff) a cell sort of n
// points needs.
size_t scan_bsum_len(size_t n);
size_t radix_hist_len(size_t n);
void exclusive_scan_raw(hipStream_t s, const unsigned *in, unsigned *out, unsigned n, unsigned *bsum,
                        KernelTimer &T);
struct CellSortBufs {
    unsigned *start;         // ncells + 1
    unsigned *pcell, *perm;  // n each: sorted cell keys, slot -> point
    unsigned *keys2, *vals2; // n each (ping-pong)
    unsigned *hist, *hoff;   // radix_hist_len(n), radix_hist_len(n) + 1
    unsigned *bsum;          // scan_bsum_len(radix_hist_len(n))
};
void cell_sort_raw(hipStream_t s, const float4 *x, unsigned n, const GridDesc &g, const CellSortBufs &b,
                   KernelTimer &T);

// Gathers dst[k] = src[perm[k]] for k < n.
void permute_f4(hipStream_t s, const unsigned *perm, unsigned n, const float4 *src, float4 *dst);
void permute_u1(hipStream_t s, const unsigned *perm, unsigned n, const unsigned *src, unsigned *dst);
void fill_u32(hipStream_t s, unsigned *p, size_t n, unsigned v);

// Neighbour lists of every query point among the cell-sorted source points.
// Column-major output: neighbour k of query i at nbr[k * stride + i] (so a
// wavefront of consecutive queries reads 64 consecutive words per k), the
// source slot as value; cnt[i] = number found (may exceed cap: then the
// entries beyond cap are dropped and *maxcnt reports the true maximum).
// same_set excludes slot == i. A pair is in when its distance is below
// `radius`, decided in FP64 when the FP32 distance is within rounding of it.
// With nbr16 the lists are also written packed: entry k as the 16-bit
// difference (slot - i) in half (k & 1) of word nbr16[(k / 2) * stride + i]
// (an odd count leaves the high half of its last word 0); *ovf16 is set
// nonzero when a difference does not fit or when a wave meets a row of more
// than 64 candidates (dense waves write no packed copy), and the packed copy
// is then unusable.
void build_lists_colmajor(hipStream_t s, const float4 *q, unsigned nq, const float4 *src, const unsigned *start,
                          const GridDesc &g, double radius, bool same_set, unsigned *nbr, unsigned stride, unsigned cap,
                          unsigned *cnt, unsigned *maxcnt, KernelTimer &T, const char *name,
                          unsigned *nbr16 = nullptr, unsigned *ovf16 = nullptr);

// Queries that one launch with a wave per query takes of `left`.
unsigned csr_wave_slice(unsigned left);

// CSR variant for the drop-in search: sources cell-sorted with srcmap[slot] =
// caller index of the source point, queries q with qmap[k] = caller index of
// query k (null: k itself), best in cell order too. With rowoff == nullptr
// only counts are written (pass 1, cnt[caller index]); with rowoff the lists
// are written at out[rowoff[caller index] ...] (pass 2), row by row and in
// slot order, whatever the order of the queries. same_set: q is the source
// array itself (query k in slot k), and a point is not its own neighbour.
void build_lists_csr(hipStream_t s, const float4 *q, const unsigned *qmap, unsigned nq, const float4 *src,
                     unsigned nsrc, const unsigned *srcmap, const unsigned *start, const GridDesc &g, double radius, bool same_set,
                     const unsigned *rowoff, unsigned *out, unsigned *cnt);

}  // namespace sph
