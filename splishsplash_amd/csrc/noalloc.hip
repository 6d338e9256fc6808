// noalloc.hip -- sph_ns_find_neighbors_noalloc: the neighbour search of one
// point set against itself on device-resident positions, writing a CSR into
// caller-provided device buffers, with every intermediate (the float4 copy of
// the positions, the cell keys, the radix-sort ping-pong buffers and
// histograms, the cell table, the cell-sorted copy, the per-point counts and
// the bounding-box partials) carved out of one fixed device array,
// `scratch`. Nothing is allocated on the device: no hipMalloc, no hipFree,
// no library routine that allocates.
//
// The kernels are the ones sph_ns_find_neighbors runs for a set searching
// itself (cell sort, permute, the two CSR passes and the scan of grid.hip),
// on the grid that entry point derives from the same bounding box, so the
// lists are identical: same sets, same order, same caller indices.
#include <mutex>

#include "grid.hpp"

namespace sph {
namespace {

// The whole working memory of the entry point, one copy per GPU (a module
// global lives once in every device that loads the code object, until the
// process ends).
constexpr size_t SCRATCH_BYTES = (size_t)48 << 20;
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

// Largest point count accepted; the cell table takes what the per-point
// buffers leave of the scratch array.
constexpr size_t MAX_POINTS = (size_t)1 << 19;

constexpr int MAX_DEVICES = 64;
struct DeviceScratch {
    std::once_flag once;
    hipError_t status = hipSuccess;
    unsigned char *ptr = nullptr;  // device address of this GPU's `scratch`
    std::mutex lock;               // one call at a time per GPU
};
DeviceScratch g_dev[MAX_DEVICES];

// The device address of `scratch` on the current device, looked up once per
// device with that device current. In host code the array's name is only a
// host-side stand-in for the symbol, so every use below goes through this
// pointer.
DeviceScratch &device_scratch() {
    int dev = 0;
    SPH_HIP(hipGetDevice(&dev));
    SPH_REQUIRE(dev >= 0 && dev < MAX_DEVICES, SPH_ERR_DEVICE, "sph_ns_find_neighbors_noalloc: device index out of range");
    DeviceScratch &d = g_dev[dev];
    std::call_once(d.once, [&] {
        void *p = nullptr;
        d.status = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        d.ptr = static_cast<unsigned char *>(p);
    });
    if (d.status != hipSuccess || d.ptr == nullptr)
        throw Error(SPH_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(d.status));
    return d;
}

// Bump allocator over the scratch array: 256-byte aligned sub-buffers.
struct Carve {
    unsigned char *base;
    size_t used = 0;
    template <class T> T *take(size_t count) {
        T *p = reinterpret_cast<T *>(base + used);
        used += (count * sizeof(T) + 255) & ~(size_t)255;
        return p;
    }
};

// Positions (x, y, z per point, caller order) to float4, with per-block
// minima and maxima of each coordinate in part[6 * block + c].
__global__ __launch_bounds__(BLOCK) void k_pack_bounds(const float *__restrict__ x, unsigned n,
                                                       float4 *__restrict__ x4, float *__restrict__ part) {
    __shared__ float red[6][BLOCK / 64];
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    float v[3] = {0.f, 0.f, 0.f};
    const bool ok = i < n;
    if (ok) {
        v[0] = x[3 * (size_t)i];
        v[1] = x[3 * (size_t)i + 1];
        v[2] = x[3 * (size_t)i + 2];
        x4[i] = make_float4(v[0], v[1], v[2], 0.f);
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int c = 0; c < 3; c++) {
        float lo = ok ? v[c] : INFINITY, hi = ok ? v[c] : -INFINITY;
        for (int o = 32; o > 0; o >>= 1) {
            lo = fminf(lo, __shfl_xor(lo, o, 64));
            hi = fmaxf(hi, __shfl_xor(hi, o, 64));
        }
        if (lane == 0) {
            red[c][wid] = lo;
            red[3 + c][wid] = hi;
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int c = threadIdx.x;
        float r = red[c][0];
        for (int w = 1; w < BLOCK / 64; w++) r = c < 3 ? fminf(r, red[c][w]) : fmaxf(r, red[c][w]);
        part[6 * (size_t)blockIdx.x + c] = r;
    }
}

// One block: the minima and maxima over nb block partials into out[0..6).
__global__ __launch_bounds__(BLOCK) void k_bounds_final(const float *__restrict__ part, unsigned nb,
                                                        float *__restrict__ out) {
    __shared__ float red[6][BLOCK / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int c = 0; c < 6; c++) {
        float r = c < 3 ? INFINITY : -INFINITY;
        for (unsigned b = threadIdx.x; b < nb; b += BLOCK) {
            const float p = part[6 * (size_t)b + c];
            r = c < 3 ? fminf(r, p) : fmaxf(r, p);
        }
        for (int o = 32; o > 0; o >>= 1) {
            const float t = __shfl_xor(r, o, 64);
            r = c < 3 ? fminf(r, t) : fmaxf(r, t);
        }
        if (lane == 0) red[c][wid] = r;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int c = threadIdx.x;
        float r = red[c][0];
        for (int w = 1; w < BLOCK / 64; w++) r = c < 3 ? fminf(r, red[c][w]) : fmaxf(r, red[c][w]);
        out[c] = r;
    }
}

}  // namespace
}  // namespace sph

using namespace sph;

extern "C" int sph_ns_find_neighbors_noalloc(const float *x, size_t n, double radius, unsigned *offsets,
                                             unsigned *neighbors, size_t capacity, size_t *total, void *stream) {
    return guarded([&] {
        SPH_REQUIRE(n <= MAX_POINTS, SPH_ERR_RANGE,
                    "sph_ns_find_neighbors_noalloc: " + std::to_string(n) + " points exceed the maximum of " +
                        std::to_string(MAX_POINTS));
        SPH_REQUIRE(radius > 0 && offsets && total && (x || n == 0), SPH_ERR_INVALID,
                    "sph_ns_find_neighbors_noalloc: bad arguments");
        require_device();
        hipStream_t s = static_cast<hipStream_t>(stream);
        DeviceScratch &dev = device_scratch();
        std::lock_guard<std::mutex> guard(dev.lock);
        KernelTimer T;  // disabled: records nothing
        *total = 0;
        if (n == 0) {
            fill_u32(s, offsets, 1, 0u);
            SPH_HIP(hipStreamSynchronize(s));
            return;
        }
        const unsigned nn = (unsigned)n;
        const size_t hl = radix_hist_len(n);
        const unsigned npart = nblocks(n);
        Carve cv{dev.ptr};
        float4 *x4 = cv.take<float4>(n);
        float4 *srt = cv.take<float4>(n);
        unsigned *pcell = cv.take<unsigned>(n), *perm = cv.take<unsigned>(n);
        unsigned *keys2 = cv.take<unsigned>(n), *vals2 = cv.take<unsigned>(n);
        unsigned *cnt = cv.take<unsigned>(n);
        unsigned *hist = cv.take<unsigned>(hl), *hoff = cv.take<unsigned>(hl + 1);
        unsigned *bsum = cv.take<unsigned>(std::max(scan_bsum_len(hl), scan_bsum_len(n)));
        float *part = cv.take<float>(6 * (size_t)npart);
        float *bounds = cv.take<float>(8);
        unsigned *start = cv.take<unsigned>(0);  // the cell table takes the rest
        SPH_REQUIRE(cv.used < SCRATCH_BYTES, SPH_ERR_RANGE, "sph_ns_find_neighbors_noalloc: scratch exhausted");
        const size_t max_cells = (SCRATCH_BYTES - cv.used) / sizeof(unsigned) - 1;

        // bounding box (the same min/max the host-side search takes)
        k_pack_bounds<<<npart, BLOCK, 0, s>>>(x, nn, x4, part);
        k_bounds_final<<<1, BLOCK, 0, s>>>(part, npart, bounds);
        SPH_HIP(hipGetLastError());
        float hb[6];
        SPH_HIP(hipMemcpyAsync(hb, bounds, sizeof(hb), hipMemcpyDeviceToHost, s));
        SPH_HIP(hipStreamSynchronize(s));
        const double lo[3] = {hb[0], hb[1], hb[2]}, hi[3] = {hb[3], hb[4], hb[5]};
        const GridDesc g = make_grid(lo, hi, radius);
        SPH_REQUIRE((size_t)g.ncells <= max_cells, SPH_ERR_RANGE,
                    "sph_ns_find_neighbors_noalloc: the grid of this point cloud needs " + std::to_string(g.ncells) +
                        " cells; the scratch array holds at most " + std::to_string(max_cells) + " for " +
                        std::to_string(n) + " points");

        const CellSortBufs b{start, pcell, perm, keys2, vals2, hist, hoff, bsum};
        cell_sort_raw(s, x4, nn, g, b, T);
        permute_f4(s, perm, nn, x4, srt);
        build_lists_csr(s, srt, perm, nn, srt, nn, perm, start, g, radius, true, nullptr, nullptr, cnt);
        exclusive_scan_raw(s, cnt, offsets, nn, bsum, T);
        unsigned tot = 0;
        SPH_HIP(hipMemcpyAsync(&tot, offsets + n, sizeof(unsigned), hipMemcpyDeviceToHost, s));
        SPH_HIP(hipStreamSynchronize(s));
        *total = tot;
        SPH_REQUIRE(tot <= capacity, SPH_ERR_RANGE,
                    "sph_ns_find_neighbors_noalloc: " + std::to_string(tot) + " neighbour entries exceed the capacity of " +
                        std::to_string(capacity) + " (offsets are written; *total holds the size needed)");
        SPH_REQUIRE(neighbors || tot == 0, SPH_ERR_INVALID, "sph_ns_find_neighbors_noalloc: null neighbour buffer");
        if (tot) build_lists_csr(s, srt, perm, nn, srt, nn, perm, start, g, radius, true, offsets, neighbors, nullptr);
        SPH_HIP(hipStreamSynchronize(s));
    });
}
