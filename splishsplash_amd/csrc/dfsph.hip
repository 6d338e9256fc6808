// dfsph.hip -- device-resident DFSPH time step.
//
// One thread per particle, particles kept in cell order (re-sorted every
// step by a counting sort; the caller-visible order is the particle id).
// The reference's sweeps (TimeStepDFSPH.cpp, scalar branch) are fused where
// no global dependency separates them:
//   sweep_init   densities + DFSPH factor + divergence set-up (1 sweep)
//   accel/jacobi the two sweeps of every Jacobi iteration; the FP64 error
//                sum is finished by the last block, which also decides
//                convergence on the device
//   post         clear accelerations + Weiler2018 apply + XSPH + CFL
//                + v += h a + p_v scaling (1 sweep)
//   finish/final pressure accelerations + v update, then p scaling and the
//                compensated position update
#include <algorithm>
#include <atomic>
#include <cfloat>
#include <cmath>
#include <cstring>

#include "dfsph.hpp"
#include "mlp.hpp"

namespace sph {


__device__ __forceinline__ unsigned gtid() { return xcd_block() * blockDim.x + threadIdx.x; }

__device__ __forceinline__ float3 f3(const float4 &a) { return make_float3(a.x, a.y, a.z); }

// ------------------------------------------------------------------ small
// The fluid's arrays of a step in cell order, dst[k] = src[perm[k]], in one
// launch instead of seven (2.3 us each at 2,000 particles, more with the gaps
// between them), and what the step and its list build start from. With the
// shorter scans of the cell sort a step of 2,000 particles takes 351 us
// instead of 392, one of 51k IISPH particles 516 instead of 537.
struct FluidArrays {
    float4 *x, *v, *xc, *vdiff;
    float *p, *pv;
    unsigned *id;
};
__global__ __launch_bounds__(BLOCK) void k_permute_fluid(const unsigned *__restrict__ perm, unsigned n, FluidArrays src,
                                                         FluidArrays dst, Ctl *C) {
    const unsigned k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k == 0) {
        C->h_step = C->h;
        C->maxcnt_f = 0;
        C->maxcnt_b = 0;
        C->ovf16 = 0;
        C->tiles_over = 0;
    }
    if (k >= n) return;
    const unsigned j = perm[k];
    const float4 x = src.x[j], v = src.v[j], xc = src.xc[j], vd = src.vdiff[j];
    const float p = src.p[j], pv = src.pv[j];
    const unsigned id = src.id[j];
    dst.x[k] = x;
    dst.v[k] = v;
    dst.xc[k] = xc;
    dst.vdiff[k] = vd;
    dst.p[k] = p;
    dst.pv[k] = pv;
    dst.id[k] = id;
}
__global__ void k_reset(Ctl *C, int which) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    if (which == 0) {
        C->it = 0;
        C->done = 0;
        C->nlearn = 0;
    } else if (which == 1) {
        C->it_v = 0;
        C->done_v = 0;
        C->nlearn_v = 0;
    } else if (which == 2) {
        C->maxcnt_f = 0;
        C->maxcnt_b = 0;
        C->ovf16 = 0;
    } else if (which == 3) {
        C->cg_it = 0;
        C->cg_done = 0;
    }
}

// --------------------------------------------------- densities/factor/div
// TimeStep::computeDensities (TimeStep.cpp:116-169), computeDFSPHFactor
// (TimeStepDFSPH.cpp:1106-1186), computeDensityChange + divergence warm start
// (TimeStepDFSPH.cpp:398-463, 1247-1295).
__device__ __forceinline__ unsigned nb_lo(unsigned i, unsigned w) { return i + (unsigned)(int)(short)(w & 0xffffu); }
__device__ __forceinline__ unsigned nb_hi(unsigned i, unsigned w) { return i + (unsigned)((int)w >> 16); }

// What a sweep loads per neighbour: up to three arrays (a, b, c of the
// result). Groups of neighbours are loaded array by array: the gathers of
// one array together measured 2-5 % faster than neighbour by neighbour
// (k_jacobi, k_jacobi2, k_features at 1M particles).
struct NoLoad {
    __device__ int operator()(unsigned) const { return 0; }
};
template <class A, class B, class C> struct Neighbour {
    A a;
    B b;
    C c;
};
template <class A, class B, class C> struct Loads {
    A a;
    B b;
    C c;
    __device__ __forceinline__ auto operator()(unsigned j) const {
        return Neighbour<decltype(a(j)), decltype(b(j)), decltype(c(j))>{a(j), b(j), c(j)};
    }
    // q[k] = the neighbour j[k], k < 4
    template <class Q> __device__ __forceinline__ void four(const unsigned *j, Q *q) const {
#pragma unroll
        for (int k = 0; k < 4; k++) q[k].a = a(j[k]);
#pragma unroll
        for (int k = 0; k < 4; k++) q[k].b = b(j[k]);
#pragma unroll
        for (int k = 0; k < 4; k++) q[k].c = c(j[k]);
    }
};
template <class A, class B = NoLoad, class C = NoLoad>
__device__ __forceinline__ Loads<A, B, C> loads(A a, B b = B{}, C c = C{}) {
    return {a, b, c};
}

// Calls f(j, ld(j)) for the fluid neighbours of particle i taken by lane hl
// of the particle's LPP lanes, the loads of four neighbours issued before
// the first f. From the packed lists lane hl takes words hl, hl + LPP, ...
// (two neighbours each); from nf neighbours hl, hl + LPP, .... The split is
// fixed by (cnt, LPP, which list), so sums stay deterministic.
template <int LPP, class LD, class F>
__device__ __forceinline__ void fluid_pairs(const Dev &D, unsigned i, unsigned hl, unsigned cnt, LD &&ld, F &&f) {
    const size_t S = D.stride;
    auto four = [&](unsigned j0, unsigned j1, unsigned j2, unsigned j3) {
        const unsigned j[4] = {j0, j1, j2, j3};
        decltype(ld(0u)) q[4];
        ld.four(j, q);
        f(j0, q[0]);
        f(j1, q[1]);
        f(j2, q[2]);
        f(j3, q[3]);
    };
    if (D.nf16) {
        const unsigned *__restrict__ P = D.nf16 + i;
        const unsigned full = cnt >> 1;  // words holding two neighbours
        unsigned w = hl;
        for (; w + LPP < full; w += 2 * LPP) {
            const unsigned a = P[w * S], b = P[(w + LPP) * S];
            four(nb_lo(i, a), nb_hi(i, a), nb_lo(i, b), nb_hi(i, b));
        }
        for (; w < full; w += LPP) {
            const unsigned a = P[w * S];
            f(nb_lo(i, a), ld(nb_lo(i, a)));
            f(nb_hi(i, a), ld(nb_hi(i, a)));
        }
        if ((cnt & 1u) && w == full) {
            const unsigned j = nb_lo(i, P[w * S]);
            f(j, ld(j));
        }
    } else {
        const unsigned *__restrict__ L = D.nf + i;
        unsigned k = hl;
        for (; k + 3 * LPP < cnt; k += 4 * LPP)
            four(L[k * S], L[(k + LPP) * S], L[(k + 2 * LPP) * S], L[(k + 3 * LPP) * S]);
        for (; k < cnt; k += LPP) f(L[k * S], ld(L[k * S]));
    }
}

// ---------------------------------------------------------------- tiles
// The sweeps of the solver iterations visit the same lists some forty times a
// step, and the gathers bound them: a wave's 64 neighbours lie in 42-46
// cache lines, which the vector cache looks up one per cycle (texture data
// path 75 % busy in k_accel, 90 % in k_jacobi at 1M particles, whatever the
// arithmetic between: 12 % fewer vector instructions left the times as they
// were). Consecutive particles share most of their neighbours, so a tile of
// 256 needs about 8 slots a particle instead of 30: a tiled sweep copies
// those to LDS once, coalesced, and its pairs read LDS. At 1M particles
// (pressure / divergence iterations) k_accel 44 / 48 -> 28 / 35 us, k_jacobi
// 69 / 73 -> 50 / 53 us; at 176k 15 / 14 -> 12 / 14 and 20 / 18 -> 17 / 15 us.
// They are now bound by the vector instructions, 45 a pair, some 12 % of them
// in the FP64 band of table_step. Tiles of 128 particles
// take as long in the sweeps and half as long again to build.
//
// k_tile_lists, once a step: marks the tile's neighbour slots in a bitmap of
// the 65536 slots around the tile, numbers the marked ones in slot order and
// rewrites the packed lists with these numbers, entries in the same order
// (85 us at 1M particles, 33 us at 111k; bound by LDS: a marked slot is an
// atomic, a rewritten one two reads).
// A tile with more than TILE_CAP slots, or slots outside the window, keeps a
// count of zero, its sweeps read memory as before, and the control block
// counts it.
constexpr unsigned TILE_WORDS = 65536 / 32;
__global__ __launch_bounds__(TILE) void k_tile_lists(Dev D, uint4 *__restrict__ nt16,
                                                     unsigned *__restrict__ tslot, unsigned *__restrict__ tcount) {
    __shared__ __align__(16) unsigned bits[TILE_WORDS], first[TILE_WORDS];
    __shared__ unsigned wtot[TILE / 64], bad;
    constexpr unsigned PER = TILE_WORDS / TILE;
    const unsigned t = threadIdx.x, lane = t & 63u, blk = xcd_block();
    const unsigned i0 = blk * TILE, i = i0 + t;
#pragma unroll
    for (unsigned q = 0; q < PER; q++) bits[q * TILE + t] = 0u;
    if (t == 0) bad = 0u;
    __syncthreads();
    const unsigned cnt = i < D.n ? D.cf[i] : 0u, nw = (cnt + 1u) >> 1;
    const unsigned *__restrict__ P = D.nf16 + i;
    const size_t S = D.stride;
    // place of entry d (a slot less i) in the window
    auto place = [&](int d) { return (unsigned)(d + (int)t + 32768); };
    bool far = false;
    auto mark = [&](unsigned p) {
        if (p < 65536u)
            atomicOr(&bits[p >> 5], 1u << (p & 31u));
        else
            far = true;
    };
    auto quad = [&](unsigned w, unsigned *a) {
#pragma unroll
        for (unsigned q = 0; q < 4u; q++) a[q] = P[(w + q < nw ? w + q : w) * S];
    };
    for (unsigned w = 0; w < nw; w += 4u) {
        unsigned a[4];
        quad(w, a);
#pragma unroll
        for (unsigned q = 0; q < 4u; q++) {
            if (2u * (w + q) < cnt) mark(place((int)(short)(a[q] & 0xffffu)));
            if (2u * (w + q) + 1u < cnt) mark(place((int)a[q] >> 16));
        }
    }
    if (far) bad = 1u;
    __syncthreads();
    // thread t numbers words t PER .. t PER + PER - 1
    unsigned b[PER], sum = 0;
#pragma unroll
    for (unsigned q = 0; q < PER; q++) {
        b[q] = bits[t * PER + q];
        sum += (unsigned)__popc(b[q]);
    }
    unsigned inc = sum;
    for (unsigned o = 1; o < 64u; o <<= 1) {
        const unsigned v = __shfl_up(inc, o, 64);
        if (lane >= o) inc += v;
    }
    if (lane == 63u) wtot[t >> 6] = inc;
    __syncthreads();
    unsigned base = inc - sum, total = 0;
#pragma unroll
    for (unsigned q = 0; q < TILE / 64; q++) {
        if (q < (t >> 6)) base += wtot[q];
        total += wtot[q];
    }
    const bool fits = total <= TILE_CAP && bad == 0u;
    if (t == 0) tcount[blk] = fits ? total : 0u;
    if (t == 0 && !fits) atomicAdd(&D.ctl->tiles_over, 1u);
    if (!fits) return;
    short *const out = reinterpret_cast<short *>(tslot + (size_t)blk * (TILE_CAP / 2));
#pragma unroll
    for (unsigned q = 0; q < PER; q++) {
        first[t * PER + q] = base;
        for (unsigned m = b[q]; m != 0u; m &= m - 1u) {
            const short d = (short)((int)(t * PER + q) * 32 + __ffs(m) - 1 - 32768);
            out[base] = d;
            // an odd count fills its last word with the same slot
            if (++base == total && (total & 1u)) out[base] = d;
        }
    }
    __syncthreads();
    auto number = [&](unsigned p) {
        return first[p >> 5] + (unsigned)__popc(bits[p >> 5] & ((1u << (p & 31u)) - 1u));
    };
    for (unsigned w = 0; w < nw; w += 4u) {
        unsigned a[4];
        quad(w, a);
#pragma unroll
        for (unsigned q = 0; q < 4u; q++) {
            const unsigned lo = 2u * (w + q) < cnt ? number(place((int)(short)(a[q] & 0xffffu))) : 0u;
            const unsigned hi = 2u * (w + q) + 1u < cnt ? number(place((int)a[q] >> 16)) : 0u;
            a[q] = lo | (hi << 16);
        }
        nt16[(w >> 2) * S + i] = make_uint4(a[0], a[2], a[1], a[3]);
    }
}

// Copies the `cnt` slots of tile blk to LDS: put(k, load(slot)) for the k-th
// slot, by a block of NT threads, the loads of all its slots in flight.
template <unsigned NT, class LD, class PUT>
__device__ __forceinline__ void tile_stage(const Dev &D, unsigned blk, unsigned cnt, LD &&load, PUT &&put) {
    constexpr unsigned R = (TILE_CAP / 2 + NT - 1) / NT;
    const unsigned *__restrict__ W = D.tslot + (size_t)blk * (TILE_CAP / 2);
    const unsigned words = (cnt + 1u) >> 1, i0 = blk * TILE;
    unsigned w[R];
    decltype(load(0u)) lo[R], hi[R];
#pragma unroll
    for (unsigned r = 0; r < R; r++) {
        const unsigned k = r * NT + threadIdx.x;
        w[r] = W[k < words ? k : words - 1u];
    }
#pragma unroll
    for (unsigned r = 0; r < R; r++) {
        if (r * NT >= words) break;
        lo[r] = load(nb_lo(i0, w[r]));
        hi[r] = load(nb_hi(i0, w[r]));
    }
#pragma unroll
    for (unsigned r = 0; r < R; r++) {
        if (r * NT >= words) break;
        const unsigned k = r * NT + threadIdx.x;
        if (k < words) {
            put(2u * k, lo[r]);
            put(2u * k + 1u, hi[r]);
        }
    }
}

// fluid_pairs of a tile: the same split and order, f(LDS places...) for four,
// two or one neighbours. A sweep from LDS would wait for its list words
// (each a trip to HBM) instead of its gathers, so the lane loads them by the
// quad (its 4 / LPP words) and holds two or three quads in registers: the
// first are loaded before the tile is staged. (Words loaded where they are
// used: k_accel 43 / 51 us, k_jacobi 61 / 58 us at 1M particles.)
template <int LPP> struct TileWords {
    static constexpr int W = 4 / LPP;  // words of a quad per lane: 4 or 2
    typedef unsigned Quad __attribute__((ext_vector_type(W)));
    Quad c, n, m;
    const unsigned *P;
    __device__ __forceinline__ static Quad load(const unsigned *p) { return *reinterpret_cast<const Quad *>(p); }
    __device__ __forceinline__ TileWords(const Dev &D, unsigned i, unsigned hl) : P(D.nt16 + 4 * (size_t)i + W * hl) {
        const size_t S = 4 * (size_t)D.stride;
        const unsigned last = D.quads16 - 1u;
        const bool act = i < D.n;
        c = act ? load(P) : Quad{};
        n = act ? load(P + (last < 1u ? last : 1u) * S) : Quad{};
        m = act && W == 2 ? load(P + (last < 2u ? last : 2u) * S) : Quad{};
    }
    template <class F> __device__ __forceinline__ void pairs(const Dev &D, unsigned hl, unsigned cnt, F &&f) {
        constexpr unsigned AHEAD = W == 2 ? 3 : 2;
        const size_t S = 4 * (size_t)D.stride;
        const unsigned full = cnt >> 1, quads = (cnt + 7u) >> 3;  // words of two neighbours; quads
        const unsigned *p = P + AHEAD * S;
        unsigned w = hl, k = AHEAD;
        auto four = [&](unsigned a, unsigned b) { f(a & 0xffffu, a >> 16, b & 0xffffu, b >> 16); };
        for (; w + (W - 1) * LPP < full; w += 4, k++, p += S) {
            const Quad q = c;
            c = n;
            if (W == 2) n = m;
            if (k < quads) (W == 2 ? m : n) = load(p);
            if constexpr (W == 4) {
                four(q.x, q[2]);
                four(q.y, q[3]);
            } else {
                four(q.x, q.y);
            }
        }
        // the lane's rest of c: fewer than W full words, and the odd entry
        unsigned a = c.x;
        if constexpr (W == 4)
            if (w + 1 < full) {
                four(c.x, c[2]);
                a = c.y;
                c[2] = c[3];
                w += 2;
            }
        if (w < full) {
            f(a & 0xffffu, a >> 16);
            a = c[W / 2];
            w += LPP;
        }
        if ((cnt & 1u) && w == full) f(a & 0xffffu);
    }
};

// Calls f(xb) for the Akinci boundary neighbours of particle i in order.
template <class F>
__device__ __forceinline__ void akinci_pairs(const Dev &D, unsigned i, unsigned cb, F &&f) {
    for (unsigned k = 0; k < cb; k++) f(D.bx[D.nb[(size_t)k * D.stride + i]]);
}
// Neighbour sums may be split over LPP = 2 or 4 adjacent lanes: lane h of a
// particle takes words (or neighbours) h, h + LPP, ..., and the partial sums
// are combined by butterfly shuffles in a fixed order (results are
// deterministic; LPP = 1 is the plain sequential sum). Shorter per-lane
// chains of dependent gathers keep more loads in flight per wave.
template <int LPP>
__device__ __forceinline__ float lane_sum(float v) {
    if (LPP >= 2) v += __shfl_xor(v, 1, 64);
    if (LPP >= 4) v += __shfl_xor(v, 2, 64);
    return v;
}

// LPP = ORDERED_LANES shares a particle's pairs over 16 lanes without
// changing the sum: the lanes evaluate up to 64 pairs at once (all their
// index loads, then all their gathers in flight), leave the terms in LDS, and
// one lane per accumulator then adds them in list order, exactly as one lane
// per particle would. For counts that leave the GPU mostly idle: a sweep
// there takes as long as its chain of dependent loads, which this cuts from
// about one per four neighbours to two, and the ordered adds from LDS take a
// few hundred cycles.
constexpr int ORDERED_LANES = 16;
constexpr int ORDERED_SLOTS = 64;

// What a sweep sums per pair: NT terms t and NACC accumulators,
// acc[c] = fma(t[a(c)], t[b(c)], acc[c]), or acc[c] += t[c] with ADD.
template <int N> struct SumAdd {
    static constexpr int NT = N, NACC = N;
    static constexpr bool ADD = true;
    static constexpr int a(int c) { return c; }
    static constexpr int b(int) { return 0; }
};
struct SumVec {  // t = (c, x, y, z): acc += c (x, y, z)
    static constexpr int NT = 4, NACC = 3;
    static constexpr bool ADD = false;
    static constexpr int a(int) { return 0; }
    static constexpr int b(int c) { return 1 + c; }
};
struct SumDot {  // t = (g, d): acc += g d
    static constexpr int NT = 2, NACC = 1;
    static constexpr bool ADD = false;
    static constexpr int a(int) { return 0; }
    static constexpr int b(int) { return 1; }
};
struct SumSym {  // t = (u, r): acc += the upper triangle of u r^T
    static constexpr int NT = 6, NACC = 6;
    static constexpr bool ADD = false;
    static constexpr int a(int c) { return c < 3 ? 0 : (c < 5 ? 1 : 2); }
    static constexpr int b(int c) { return c < 3 ? 3 + c : (c < 5 ? 1 + c : 5); }
};
struct SumVecAdd {  // t = (x, y, z | c, u, v, w): acc += (x, y, z), c (u, v, w)
    static constexpr int NT = 8, NACC = 6;  // t[7] = 1
    static constexpr bool ADD = false;
    static constexpr int a(int c) { return c < 3 ? c : 3; }
    static constexpr int b(int c) { return c < 3 ? 7 : 1 + c; }
};

template <class S> __device__ __forceinline__ void sum_terms(const float *t, float *acc) {
#pragma unroll
    for (int c = 0; c < S::NACC; c++)
        acc[c] = S::ADD ? acc[c] + t[c] : fmaf(t[S::a(c)], t[S::b(c)], acc[c]);
}

// Floats of LDS per particle for up to NT terms per pair (a multiple of four
// off the banks' period, so the four particles of a wave read different
// banks), per block, and a particle's own part. Every sum of a kernel uses
// the same part: the waves of a block are not in step.
template <int NT> constexpr int PAIR_PITCH = ORDERED_SLOTS * NT + 4;
template <int LPP, int NT>
constexpr int PAIR_LDS = LPP == ORDERED_LANES ? (BLOCK / ORDERED_LANES) * PAIR_PITCH<NT> : 1;
template <int LPP, int NT> __device__ __forceinline__ float *pair_part(float *lds) {
    return LPP == ORDERED_LANES ? lds + (threadIdx.x / ORDERED_LANES) * PAIR_PITCH<NT> : nullptr;
}

// A particle's LDS accesses stay within its wave, which executes them in
// program order: only the compiler must keep that order.
__device__ __forceinline__ void pair_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Adds the terms of slots 0 .. m - 1 in order; lane c < NACC of the particle
// holds accumulator c, in and out.
template <class S>
__device__ __forceinline__ void ordered_add(const float *__restrict__ T, unsigned hl, unsigned m, float &my) {
    pair_sync();
    if (hl < (unsigned)S::NACC) {
        int oa = 0, ob = 0;
#pragma unroll
        for (int c = 0; c < S::NACC; c++)
            if (hl == (unsigned)c) {
                oa = S::a(c);
                ob = S::b(c);
            }
#pragma unroll 8
        for (unsigned k = 0; k < m; k++)
            my = S::ADD ? my + T[k * S::NT + oa] : fmaf(T[k * S::NT + oa], T[k * S::NT + ob], my);
    }
    pair_sync();
}
template <class S, class V> __device__ __forceinline__ void ordered_put(float *__restrict__ T, unsigned slot, V &&term) {
    float t[S::NT];
    if (!term(t))
#pragma unroll
        for (int q = 0; q < S::NT; q++) t[q] = 0.f;
#pragma unroll
    for (int q = 0; q < S::NT; q++) T[slot * S::NT + q] = t[q];
}
template <class S> __device__ __forceinline__ float ordered_mine(unsigned hl, const float *acc) {
    float my = 0.f;
#pragma unroll
    for (int c = 0; c < S::NACC; c++)
        if (hl == (unsigned)c) my = acc[c];
    return my;
}
template <class S> __device__ __forceinline__ void ordered_share(float my, float *acc) {
#pragma unroll
    for (int c = 0; c < S::NACC; c++) acc[c] = __shfl(my, c, ORDERED_LANES);
}

// Sums over the cnt fluid neighbours of particle i: ld(j) loads a
// neighbour's data, term(j, data, t) writes its terms and returns whether
// they count; T is the particle's part of LDS. Every lane of the particle
// calls this; acc is the starting value and, after lanes_join, the result in
// each lane of it.
template <int LPP, class S, class LD, class TERM>
__device__ __forceinline__ void fluid_sums(const Dev &D, unsigned i, unsigned hl, unsigned cnt, float *__restrict__ T,
                                           float *acc, LD &&ld, TERM &&term) {
    if constexpr (LPP != ORDERED_LANES) {
        fluid_pairs<LPP>(D, i, hl, cnt, ld, [&](unsigned j, const auto &q) {
            float t[S::NT];
            if (term(j, q, t)) sum_terms<S>(t, acc);
        });
    } else {
        float my = ordered_mine<S>(hl, acc);
        const size_t N = D.stride;
        for (unsigned k0 = 0; k0 < cnt; k0 += ORDERED_SLOTS) {
            // slots of this lane: 2 hl, 2 hl + 1 (one packed word) and the
            // same in the second half; the missing ones read slot 0's
            // neighbour
            unsigned j[4], sl[4];
#pragma unroll
            for (unsigned u = 0; u < 2; u++) {
                sl[2 * u] = 32 * u + 2 * hl;
                sl[2 * u + 1] = sl[2 * u] + 1;
                const unsigned a = k0 + sl[2 * u], b = a + 1;
                if (D.nf16) {
                    const unsigned w = D.nf16[(size_t)((a < cnt ? a : k0) >> 1) * N + i];
                    j[2 * u] = nb_lo(i, w);
                    j[2 * u + 1] = nb_hi(i, w);
                } else {
                    j[2 * u] = D.nf[(size_t)(a < cnt ? a : k0) * N + i];
                    j[2 * u + 1] = D.nf[(size_t)(b < cnt ? b : k0) * N + i];
                }
            }
            decltype(ld(0u)) q[4];
            ld.four(j, q);
#pragma unroll
            for (unsigned u = 0; u < 4; u++)
                if (k0 + sl[u] < cnt) ordered_put<S>(T, sl[u], [&](float *t) { return term(j[u], q[u], t); });
            ordered_add<S>(T, hl, cnt - k0 < ORDERED_SLOTS ? cnt - k0 : ORDERED_SLOTS, my);
        }
        ordered_share<S>(my, acc);
    }
}

// Combines the lanes' sums; every lane of the wave calls this.
template <int LPP, class S> __device__ __forceinline__ void lanes_join(float *acc) {
    if (LPP > 1 && LPP != ORDERED_LANES)
#pragma unroll
        for (int c = 0; c < S::NACC; c++) acc[c] = lane_sum<LPP>(acc[c]);
}

// The same over the Akinci boundary neighbours (cb of them), in list order
// by one lane of the particle (acc valid in lane hl == 0), or shared as
// above.
template <int LPP, class S, class TERM>
__device__ __forceinline__ void akinci_sums(const Dev &D, unsigned i, unsigned hl, unsigned cb,
                                            float *__restrict__ T, float *acc, TERM &&term) {
    if constexpr (LPP != ORDERED_LANES) {
        if (hl == 0)
            akinci_pairs(D, i, cb, [&](const float4 &xb) {
                float t[S::NT];
                if (term(xb, t)) sum_terms<S>(t, acc);
            });
    } else {
        float my = ordered_mine<S>(hl, acc);
        for (unsigned k0 = 0; k0 < cb; k0 += ORDERED_SLOTS) {
            unsigned j[4];
#pragma unroll
            for (unsigned u = 0; u < 4; u++) {
                const unsigned k = k0 + 16 * u + hl;
                j[u] = D.nb[(size_t)(k < cb ? k : k0) * D.stride + i];
            }
            float4 q[4];
#pragma unroll
            for (unsigned u = 0; u < 4; u++) q[u] = D.bx[j[u]];
#pragma unroll
            for (unsigned u = 0; u < 4; u++)
                if (k0 + 16 * u + hl < cb) ordered_put<S>(T, 16 * u + hl, [&](float *t) { return term(q[u], t); });
            ordered_add<S>(T, hl, cb - k0 < ORDERED_SLOTS ? cb - k0 : ORDERED_SLOTS, my);
        }
        ordered_share<S>(my, acc);
    }
}

// ParticleState::Active (FluidModel.h:75) unless the state array says
// otherwise; without states every particle is active.
__device__ __forceinline__ bool is_active(const Dev &D, unsigned i) { return D.state == nullptr || D.state[i] == 0u; }

// Rest density and mass of particle i's fluid model.
__device__ __forceinline__ float rho0_of(const Dev &D, unsigned i) { return D.model ? D.rho0m[D.model[i]] : D.rho0; }
__device__ __forceinline__ float mass_of(const Dev &D, unsigned i) { return D.model ? D.massm[D.model[i]] : D.mass; }
// Whether particle i belongs to the model the solver sweeps work on.
__device__ __forceinline__ bool in_solve(const Dev &D, unsigned i) {
    return D.model == nullptr || D.solveModel < 0 || D.model[i] == (unsigned)D.solveModel;
}
// The stiffness copy in w: p/rho^2 itself, or rho0_i p/rho^2 with several
// models (the acceleration sweeps then form (rho0_j / rho0_i) p_j,
// TimeStepDFSPH.cpp:1321).
__device__ __forceinline__ float stiff_w(const Dev &D, unsigned i, float k) { return D.model ? k * rho0_of(D, i) : k; }
// The non-pressure force coefficients of particle i's model.
__device__ __forceinline__ float svisc_of(const Dev &D, unsigned i) { return D.model ? D.svm[D.model[i]] : D.svisc; }
__device__ __forceinline__ float sviscB_of(const Dev &D, unsigned i) { return D.model ? D.svbm[D.model[i]] : D.sviscB; }
__device__ __forceinline__ float xsph_of(const Dev &D, unsigned i) { return D.model ? D.xsm[D.model[i]] : D.xsph; }
__device__ __forceinline__ float xsphB_of(const Dev &D, unsigned i) { return D.model ? D.xsbm[D.model[i]] : D.xsphB; }

template <bool DENS, bool FACT, bool DIV, int LPP>
__global__ __launch_bounds__(BLOCK) void k_sweep_init(Dev D) {
    constexpr int NF = (DENS ? 1 : 0) + (FACT ? 4 : 0) + (DIV ? 1 : 0);
    constexpr int NB = (DENS ? 1 : 0) + (FACT ? 3 : 0) + (DIV ? 1 : 0);
    __shared__ float plds[PAIR_LDS<LPP, NF>];
    float *const T = pair_part<LPP, NF>(plds);
    const unsigned t = gtid();
    const unsigned i = t / LPP, hl = t % LPP;
    const bool act = i < D.n;
    float4 xi = make_float4(0.f, 0.f, 0.f, 0.f), vi = xi;
    unsigned cnt = 0, cb = 0;
    // the density's own share opens the sequential sum; split sums add it
    // to their total
    float f[NF];
#pragma unroll
    for (int q = 0; q < NF; q++) f[q] = 0.f;
    if (DENS && (LPP == 1 || LPP == ORDERED_LANES)) f[0] = D.V * D.K.W0;
    if (act) {
        xi = D.x[i];
        if (DIV) vi = D.v[i];
        cnt = D.cf[i];
        const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
        const F4Gather X(D.x, D.n), V(D.v, D.n);
        fluid_sums<LPP, SumAdd<NF>>(
            D, i, hl, cnt, T, f, loads([&](unsigned j) { return X.xyz(j); }, [&](unsigned j) { return DIV ? V.xyz(j) : z4; }),
            [&](unsigned, const auto &p, float *u) {
                const float4 &vj = p.b;
                float3 r;
                float w, g;
                kernel_WG(xi, p.a, D.K, r, w, g);
                int q = 0;
                if (DENS) u[q++] = D.V * w;
                const float gx = g * r.x, gy = g * r.y, gz = g * r.z;
                if (FACT) {
                    const float qx = -D.V * gx, qy = -D.V * gy, qz = -D.V * gz;
                    u[q++] = sqn(qx, qy, qz);
                    u[q++] = -qx;
                    u[q++] = -qy;
                    u[q++] = -qz;
                }
                if (DIV) u[q++] = ((vi.x - vj.x) * gx + (vi.y - vj.y) * gy) + (vi.z - vj.z) * gz;
                return true;
            });
    }
    lanes_join<LPP, SumAdd<NF>>(f);
    if (act && D.bmode == 1) cb = D.cb[i];
    float dens = 0.f, sgk = 0.f, gpx = 0.f, gpy = 0.f, gpz = 0.f, div = 0.f, divb = 0.f;
    if (DENS) dens = (LPP == 1 || LPP == ORDERED_LANES) ? f[0] : D.V * D.K.W0 + f[0];
    if (FACT) {
        constexpr int q = DENS ? 1 : 0;
        sgk = f[q];
        gpx = f[q + 1];
        gpy = f[q + 2];
        gpz = f[q + 3];
    }
    if (DIV) div = f[NF - 1];
    if (D.bmode == 1) {
        float b[NB];
        int q = 0;
        if (DENS) b[q++] = dens;
        if (FACT) {
            b[q++] = gpx;
            b[q++] = gpy;
            b[q++] = gpz;
        }
        if (DIV) b[q++] = 0.f;
        akinci_sums<LPP, SumAdd<NB>>(D, i, hl, cb, T, b, [&](const float4 &xb, float *u) {
            float3 r;
            float w, g;
            kernel_WG(xi, xb, D.K, r, w, g);
            int q = 0;
            if (DENS) u[q++] = xb.w * w;
            const float gx = g * r.x, gy = g * r.y, gz = g * r.z;
            if (FACT) {
                u[q++] = xb.w * gx;
                u[q++] = xb.w * gy;
                u[q++] = xb.w * gz;
            }
            if (DIV) u[q++] = xb.w * ((vi.x * gx + vi.y * gy) + vi.z * gz);
            return true;
        });
        q = 0;
        if (DENS) dens = b[q++];
        if (FACT) {
            gpx = b[q++];
            gpy = b[q++];
            gpz = b[q++];
        }
        if (DIV) divb = b[q++];
    }
    if (!act || hl != 0) return;
    const unsigned nnb = cnt + cb;
    if (D.bmode == 2) {
        for (unsigned o = 0; o < D.nvm; o++) {
            const float4 xb = D.vmb[(size_t)o * D.stride + i];
            if (!(xb.w > 0.f)) break;
            float3 r;
            float w, g;
            kernel_WG(xi, xb, D.K, r, w, g);
            if (DENS) dens += xb.w * w;
            const float gx = g * r.x, gy = g * r.y, gz = g * r.z;
            if (FACT) {
                gpx -= -xb.w * gx;
                gpy -= -xb.w * gy;
                gpz -= -xb.w * gz;
            }
            if (DIV) {
                if (D.vmv) {  // v_i - v_b, v_b = getPointVelocity(x_b) (TimeStepDFSPH.cpp:1291)
                    const float4 vb = D.vmv[(size_t)o * D.stride + i];
                    divb += xb.w * ((((vi.x - vb.x) * gx + (vi.y - vb.y) * gy) + (vi.z - vb.z) * gz));
                } else {
                    divb += xb.w * (((vi.x * gx + vi.y * gy) + vi.z * gz));
                }
            }
        }
    } else if (D.bmode == 3) {
        // density maps: rho_b adds to the density, grad rho_b to the factor's
        // gradient sum and the density change (TimeStep.cpp:153-158,
        // TimeStepDFSPH.cpp:1158-1163, 1224-1231)
        for (unsigned o = 0; o < D.nvm; o++) {
            const float4 xb = D.vmb[(size_t)o * D.stride + i];
            if (!(xb.w > 0.f)) break;
            const float4 gb = D.dmg[(size_t)o * D.stride + i];
            if (DENS) dens += xb.w;
            if (FACT) {
                gpx -= gb.x;
                gpy -= gb.y;
                gpz -= gb.z;
            }
            if (DIV) divb -= ((vi.x * gb.x + vi.y * gb.y) + vi.z * gb.z);
        }
    }
    if (DENS) D.rho[i] = dens * rho0_of(D, i);
    if (FACT || DIV) {
        const float invH = (float)(1.0 / D.ctl->h);
        float a;
        if (FACT) {
            sgk += sqn(gpx, gpy, gpz);
            a = (sgk > D.eps) ? 1.0f / sgk : 0.0f;
        } else {
            a = D.alpha[i];
        }
        if (DIV) a *= invH;
        D.alpha[i] = a;
        if (DIV) {
            const float rd = div * D.V + divb;
            D.radv[i] = rd;
            float dAdv = fmaxf(rd, 0.0f);
            if (nnb < 20u) dAdv = 0.0f;
            const float pv0 = D.pv[i];
            if (D.kprev) D.kprev[i] = pv0;
            const float pv1 = (dAdv > 0.0f) ? 0.5f * fminf(pv0, 0.5f) * invH : 0.0f;
            D.pv[i] = pv1;
            reinterpret_cast<float *>(D.x + i)[3] = stiff_w(D, i, pv1);  // the solve's stiffness copy
        }
    }
}

// ------------------------------------------------- pressure accelerations
// computePressureAccel (TimeStepDFSPH.cpp:1299-1367) for particle i. During
// a solve the w component of every fluid position holds the solver's current
// stiffness (p / rho^2 or p_v / rho^2, kept equal to the stiffness array by
// k_stiff_to_w and the Jacobi update), so one 16-byte load per neighbour
// gives both the position and the stiffness.
// t = (c, r) with a_i += c r; false where the pair carries no pressure.
__device__ __forceinline__ bool accel_term(const Dev &D, const float4 &xi, float pi, const float4 &xj, float inv_rho0i,
                                           float *t) {
    const float ps = pi + xj.w * inv_rho0i;  // (times 1 with a single model)
    if (!(fabsf(ps) > D.eps)) return false;
    float3 r;
    const float g = kernel_G(xi, xj, D.K, r);
    t[0] = ps * (-D.V * g);  // a_i += -V (p_i + p_j) gradW_ij
    t[1] = r.x;
    t[2] = r.y;
    t[3] = r.z;
    return true;
}

// Map records of computePressureAccel for particle i (TimeStepDFSPH.cpp:
// 1330-1365).
__device__ __forceinline__ void accel_maps(const Dev &D, unsigned i, const float4 &xi, float pi, float3 &acc) {
    float ax = acc.x, ay = acc.y, az = acc.z;
    if (fabsf(pi) > D.eps) {
        if (D.bmode == 2) {
            for (unsigned o = 0; o < D.nvm; o++) {
                const float4 xb = D.vmb[(size_t)o * D.stride + i];
                if (!(xb.w > 0.f)) break;
                float3 r;
                const float g = kernel_G(xi, xb, D.K, r);
                ax += pi * (-xb.w * (g * r.x));
                ay += pi * (-xb.w * (g * r.y));
                az += pi * (-xb.w * (g * r.z));
            }
        } else if (D.bmode == 3) {  // p_i grad rho_b (TimeStepDFSPH.cpp:1346-1353)
            for (unsigned o = 0; o < D.nvm; o++) {
                if (!(D.vmb[(size_t)o * D.stride + i].w > 0.f)) break;
                const float4 gb = D.dmg[(size_t)o * D.stride + i];
                ax += pi * gb.x;
                ay += pi * gb.y;
                az += pi * gb.z;
            }
        }
    }
    acc = make_float3(ax, ay, az);
}

// Pressure acceleration of particle i from its lanes' fluid sums acc,
// complete in lane hl == 0. The lanes of a particle call this together.
template <int LPP>
__device__ __forceinline__ float3 accel_total(const Dev &D, unsigned i, unsigned hl, bool live, const float4 &xi,
                                              float pi, float *acc, float *__restrict__ T) {
    lanes_join<LPP, SumVec>(acc);
    if (D.bmode == 1)
        akinci_sums<LPP, SumAdd<3>>(D, i, hl, live && fabsf(pi) > D.eps ? D.cb[i] : 0u, T, acc,
                                    [&](const float4 &xb, float *t) {
                                        float3 r;
                                        const float g = kernel_G(xi, xb, D.K, r);
                                        t[0] = pi * (-xb.w * (g * r.x));
                                        t[1] = pi * (-xb.w * (g * r.y));
                                        t[2] = pi * (-xb.w * (g * r.z));
                                        return true;
                                    });
    float3 a = make_float3(acc[0], acc[1], acc[2]);
    if (live && hl == 0) accel_maps(D, i, xi, pi, a);
    return a;
}

// The same with the fluid sums: zero unless live.
template <int LPP>
__device__ __forceinline__ float3 particle_accel(const Dev &D, unsigned i, unsigned hl, bool live,
                                                 const float *__restrict__ P, float *__restrict__ T) {
    float4 xi = make_float4(0.f, 0.f, 0.f, 0.f);
    float pi = 0.f, ir = 1.f;
    float acc[3] = {0.f, 0.f, 0.f};
    if (live) {
        xi = D.x[i];
        pi = P[i];
        if (D.model) ir = 1.0f / rho0_of(D, i);
        const F4Gather X(D.x, D.n);
        fluid_sums<LPP, SumVec>(
            D, i, hl, D.cf[i], T, acc, loads([&](unsigned j) { return X.all(j); }),
            [&](unsigned, const auto &q, float *t) { return accel_term(D, xi, pi, q.a, ir, t); });
    }
    return accel_total<LPP>(D, i, hl, live, xi, pi, acc, T);
}

// The acceleration sweep of block `blk` of a particle range; the single
// scene's kernel passes its XCD-mapped block id, the batched one the
// scene-local block of its block map.
template <bool PRESSURE, int LPP>
__device__ __forceinline__ void accel_sweep(const Dev &D, unsigned blk, int check_done) {
    if (check_done && (PRESSURE ? D.ctl->done : D.ctl->done_v)) return;
    const unsigned t = blk * blockDim.x + threadIdx.x;
    const unsigned i = t / LPP, h = t % LPP;
    // with several models only the current model's particles (the others
    // keep their accelerations, TimeStepDFSPH.cpp:564-569)
    if (i < D.n && !in_solve(D, i)) return;
    const bool act = i < D.n;
    // computePressureAccel leaves a_p = 0 for particles that are not active
    // (TimeStepDFSPH.cpp:1303-1310)
    const bool live = act && is_active(D, i);
    __shared__ float plds[PAIR_LDS<LPP, SumVec::NT>];
    float *const T = pair_part<LPP, SumVec::NT>(plds);
    const float3 acc = particle_accel<LPP>(D, i, h, live, PRESSURE ? D.p : D.pv, T);
    if (act && h == 0) D.ap[i] = make_float4(acc.x, acc.y, acc.z, 0.f);
}

template <bool PRESSURE, int LPP>
__global__ __launch_bounds__(BLOCK) void k_accel(Dev D, int check_done) {
    accel_sweep<PRESSURE, LPP>(D, xcd_block(), check_done);
}

// The same for a tile of one model's particles (TILE LPP threads).
template <bool PRESSURE, int LPP>
__global__ __launch_bounds__(TILE *LPP) void k_accel_tile(Dev D, int check_done) {
    __shared__ float4 tile[TILE_CAP];
    if (check_done && (PRESSURE ? D.ctl->done : D.ctl->done_v)) return;
    const unsigned blk = xcd_block(), i = blk * TILE + threadIdx.x / LPP, h = threadIdx.x % LPP;
    const unsigned m = D.tcount[blk];
    const bool act = i < D.n;
    const bool live = act && is_active(D, i);
    const float4 xi = live ? D.x[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float pi = live ? (PRESSURE ? D.p : D.pv)[i] : 0.f;
    const unsigned cnt = live ? D.cf[i] : 0u;
    float acc[3] = {0.f, 0.f, 0.f};
    const F4Gather X(D.x, D.n);
    if (m != 0u) {
        TileWords<LPP> words(D, i, h);
        tile_stage<TILE * LPP>(
            D, blk, m, [&](unsigned j) { return X.all(j); }, [&](unsigned k, const float4 &v) { tile[k] = v; });
        __syncthreads();
        words.pairs(D, h, cnt, [&](auto... k) {
            const float4 xj[] = {tile[k]...};
            float t[SumVec::NT];
#pragma unroll
            for (unsigned q = 0; q < sizeof...(k); q++)
                if (accel_term(D, xi, pi, xj[q], 1.f, t)) sum_terms<SumVec>(t, acc);
        });
    } else {
        fluid_sums<LPP, SumVec>(
            D, i, h, cnt, nullptr, acc, loads([&](unsigned j) { return X.all(j); }),
            [&](unsigned, const auto &q, float *t) { return accel_term(D, xi, pi, q.a, 1.f, t); });
    }
    const float3 a = accel_total<LPP>(D, i, h, live, xi, pi, acc, nullptr);
    if (act && h == 0) D.ap[i] = make_float4(a.x, a.y, a.z, 0.f);
}

// Many scenes in one launch: block b works on particle block bmap[b].y of
// scene bmap[b].x, whose state Ds[bmap[b].x] describes; bmap[b].z is the
// partial-sum slot the same particles take in the scene's own launch.
template <bool PRESSURE, int LPP>
__global__ __launch_bounds__(BLOCK) void kb_accel(const Dev *__restrict__ Ds, const uint4 *__restrict__ bmap,
                                                  int check_done) {
    const uint4 m = bmap[blockIdx.x];
    accel_sweep<PRESSURE, LPP>(Ds[m.x], m.y, check_done);
}

// t = (g, d) with s += g d: (a_i - a_j) . gradW_ij = g_ij ((a_i - a_j) . r_ij)
__device__ __forceinline__ float aij_dot(const float4 &ai, const float4 &aj, const float3 &r) {
    return fmaf(ai.z - aj.z, r.z, fmaf(ai.y - aj.y, r.y, (ai.x - aj.x) * r.x));
}
__device__ __forceinline__ bool aij_term(const float4 &xi, const float4 &ai, const float4 &xj, const float4 &aj,
                                         const KernelConst &K, float *t) {
    float3 r;
    t[0] = kernel_G(xi, xj, K, r);
    t[1] = aij_dot(ai, aj, r);
    return true;
}

// compute_aij_pj (TimeStepDFSPH.cpp:1370-1420) and the Jacobi update of
// pressureSolveIteration / divergenceSolveIteration (:544-706), FP64 error
// sum finished in the last block.
// A particle's own values in the update.
struct JacobiOwn {
    float alpha, radv, p;
};
template <bool PRESSURE> __device__ __forceinline__ JacobiOwn jacobi_own(const Dev &D, unsigned i) {
    return {D.alpha[i], D.radv[i], (PRESSURE ? D.p : D.pv)[i]};
}
// The pressure update skips particles that are not active
// (TimeStepDFSPH.cpp:578-579); the divergence update takes every particle.
template <bool PRESSURE> __device__ __forceinline__ bool jacobi_takes(const Dev &D, unsigned i) {
    return i < D.n && (!PRESSURE || is_active(D, i)) && in_solve(D, i);
}

// The update of particle i (if act) from its lanes' fluid sums s; own()
// gives its JacobiOwn; err and over are its shares of the error sums.
template <bool PRESSURE, int LPP, class OWN>
__device__ __forceinline__ void jacobi_particle(const Dev &D, unsigned i, unsigned hl, bool act, unsigned cnt,
                                                const float4 &xi, const float4 &ai, float s, float *__restrict__ T,
                                                OWN &&own, double &err, double &over) {
    const double h = D.ctl->h;
    err = over = 0.0;
    lanes_join<LPP, SumDot>(&s);
    s *= D.V;
    unsigned cb = 0;
    if (act && D.bmode == 1) cb = D.cb[i];
    if (D.bmode == 1)
        akinci_sums<LPP, SumAdd<1>>(D, i, hl, cb, T, &s, [&](const float4 &xb, float *u) {
            float3 r;
            const float g = kernel_G(xi, xb, D.K, r);
            u[0] = xb.w * ((ai.x * (g * r.x) + ai.y * (g * r.y)) + ai.z * (g * r.z));
            return true;
        });
    if (act && hl == 0) {
        const unsigned nnb = cnt + cb;
        if (D.bmode == 2) {
            for (unsigned o = 0; o < D.nvm; o++) {
                const float4 xb = D.vmb[(size_t)o * D.stride + i];
                if (!(xb.w > 0.f)) break;
                float3 r;
                const float g = kernel_G(xi, xb, D.K, r);
                s += xb.w * (((ai.x * (g * r.x) + ai.y * (g * r.y)) + ai.z * (g * r.z)));
            }
        } else if (D.bmode == 3) {  // aij_pj -= a_i . grad rho_b (TimeStepDFSPH.cpp:1407-1412)
            for (unsigned o = 0; o < D.nvm; o++) {
                if (!(D.vmb[(size_t)o * D.stride + i].w > 0.f)) break;
                const float4 gb = D.dmg[(size_t)o * D.stride + i];
                s -= (ai.x * gb.x + ai.y * gb.y) + ai.z * gb.z;
            }
        }
        const JacobiOwn o = own();
        if (PRESSURE) {
            const float aij = s * (float)(h * h);
            const float si = 1.0f - o.radv;
            const float res = fminf(si - aij, 0.0f);
            const float pn = fmaxf(o.p - 0.5f * (si - aij) * o.alpha, 0.0f);
            D.p[i] = pn;
            reinterpret_cast<float *>(D.x + i)[3] = stiff_w(D, i, pn);
            const double r0 = rho0_of(D, i);
            err = -r0 * (double)res;
            if (pn > 0.0f && si - aij > 0.0f) over = r0 * (double)(si - aij);
        } else {
            const float aij = s * (float)h;
            const float si = -o.radv;
            float res = fminf(si - aij, 0.0f);
            if (nnb < 20u) res = 0.0f;
            const float pn = fmaxf(o.p - 0.5f * (si - aij) * o.alpha, 0.0f);
            D.pv[i] = pn;
            reinterpret_cast<float *>(D.x + i)[3] = stiff_w(D, i, pn);
            const double r0 = rho0_of(D, i);
            err = -r0 * (double)res;
            if (pn > 0.0f && si - aij > 0.0f && nnb >= 20u) over = r0 * (double)(si - aij);
        }
    }
}

// The lane's share of the fluid sum, neighbours read from memory.
template <int LPP>
__device__ __forceinline__ void aij_sums(const Dev &D, unsigned i, unsigned hl, unsigned cnt, float *__restrict__ T,
                                         const float4 &xi, const float4 &ai, float *s) {
    const F4Gather X(D.x, D.n), A(D.ap, D.n);
    fluid_sums<LPP, SumDot>(
        D, i, hl, cnt, T, s, loads([&](unsigned j) { return X.xyz(j); }, [&](unsigned j) { return A.xyz(j); }),
        [&](unsigned, const auto &q, float *u) { return aij_term(xi, ai, q.a, q.b, D.K, u); });
}

template <bool PRESSURE, int LPP>
__device__ __forceinline__ void jacobi_sweep(const Dev &D, unsigned blk, unsigned part, int check_done) {
    __shared__ double lds[BLOCK / 64];
    __shared__ float plds[PAIR_LDS<LPP, SumDot::NT>];
    float *const T = pair_part<LPP, SumDot::NT>(plds);
    if (check_done && (PRESSURE ? D.ctl->done : D.ctl->done_v)) return;
    const unsigned t = blk * blockDim.x + threadIdx.x;
    const unsigned i = t / LPP, hl = t % LPP;
    const bool act = jacobi_takes<PRESSURE>(D, i);
    float4 xi = make_float4(0.f, 0.f, 0.f, 0.f), ai = xi;
    unsigned cnt = 0;
    float s = 0.f;
    if (act) {
        xi = D.x[i];
        ai = D.ap[i];
        cnt = D.cf[i];
        aij_sums<LPP>(D, i, hl, cnt, T, xi, ai, &s);
    }
    double err, over;
    jacobi_particle<PRESSURE, LPP>(
        D, i, hl, act, cnt, xi, ai, s, T, [&] { return jacobi_own<PRESSURE>(D, i); }, err, over);
    const double bs = block_sum(err, lds);
    const double bo = block_sum(over, lds);
    if (threadIdx.x == 0) {
        D.partial[2 * part] = bs;
        D.partial[2 * part + 1] = bo;
    }
}

// The same for a tile of one model's particles (TILE LPP threads). The error
// partials are those of the blocks of k_jacobi, in the same places.
template <bool PRESSURE, int LPP>
__global__ __launch_bounds__(TILE *LPP) void k_jacobi_tile(Dev D, int check_done) {
    __shared__ float4 tx[TILE_CAP];  // x, y, z, a.x
    __shared__ float2 ta[TILE_CAP];  // a.y, a.z
    __shared__ double lds[2][TILE * LPP / 64];
    if (check_done && (PRESSURE ? D.ctl->done : D.ctl->done_v)) return;
    const unsigned blk = xcd_block(), i = blk * TILE + threadIdx.x / LPP, hl = threadIdx.x % LPP;
    const unsigned m = D.tcount[blk];
    const bool act = jacobi_takes<PRESSURE>(D, i);
    const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 xi = act ? D.x[i] : z4, ai = act ? D.ap[i] : z4;
    const unsigned cnt = act ? D.cf[i] : 0u;
    const JacobiOwn own = act && hl == 0 ? jacobi_own<PRESSURE>(D, i) : JacobiOwn{0.f, 0.f, 0.f};
    float s = 0.f;
    if (m != 0u) {
        struct XA {
            float4 x, a;
        };
        const F4Gather X(D.x, D.n), A(D.ap, D.n);
        TileWords<LPP> words(D, i, hl);
        tile_stage<TILE * LPP>(
            D, blk, m, [&](unsigned j) { return XA{X.xyz(j), A.xyz(j)}; },
            [&](unsigned k, const XA &v) {
                tx[k] = make_float4(v.x.x, v.x.y, v.x.z, v.a.x);
                ta[k] = make_float2(v.a.y, v.a.z);
            });
        __syncthreads();
        words.pairs(D, hl, cnt, [&](auto... k) {
            constexpr unsigned N = sizeof...(k);
            const float4 xj[N] = {tx[k]...};
            const float2 aj[N] = {ta[k]...};
            float3 r[N];
            float g[N];
            kernel_Gs<N>(xi, xj, D.K, r, g);
#pragma unroll
            for (unsigned q = 0; q < N; q++) {
                const float u[SumDot::NT] = {
                    g[q], aij_dot(ai, make_float4(xj[q].w, aj[q].x, aj[q].y, 0.f), r[q])};
                sum_terms<SumDot>(u, &s);
            }
        });
    } else {
        aij_sums<LPP>(D, i, hl, cnt, nullptr, xi, ai, &s);
    }
    double err, over;
    jacobi_particle<PRESSURE, LPP>(
        D, i, hl, act, cnt, xi, ai, s, nullptr, [&] { return own; }, err, over);
    err = wave_sum(err);
    over = wave_sum(over);
    const unsigned wid = threadIdx.x >> 6;
    if ((threadIdx.x & 63u) == 0u) {
        lds[0][wid] = err;
        lds[1][wid] = over;
    }
    __syncthreads();
    const unsigned B = (D.n * LPP + BLOCK - 1) / BLOCK, q = (blk * TILE * LPP + threadIdx.x) / BLOCK;
    if (threadIdx.x % BLOCK == 0 && q < B) {
        double bs = 0.0, bo = 0.0;
        for (int w = 0; w < BLOCK / 64; w++) {
            bs += lds[0][wid + w];
            bo += lds[1][wid + w];
        }
        const unsigned part = xcd_slot(q, B);
        D.partial[2 * part] = bs;
        D.partial[2 * part + 1] = bo;
    }
}

template <bool PRESSURE, int LPP>
__global__ __launch_bounds__(BLOCK) void k_jacobi(Dev D, int check_done) {
    jacobi_sweep<PRESSURE, LPP>(D, xcd_block(), blockIdx.x, check_done);
}

template <bool PRESSURE, int LPP>
__global__ __launch_bounds__(BLOCK) void kb_jacobi(const Dev *__restrict__ Ds, const uint4 *__restrict__ bmap,
                                                   int check_done) {
    const uint4 m = bmap[blockIdx.x];
    jacobi_sweep<PRESSURE, LPP>(Ds[m.x], m.y, m.z, check_done);
}

// Sums the per-block error partials of k_jacobi in a fixed order (one block)
// and decides convergence (TimeStepDFSPH.cpp:324-341, 477-495). The kernel
// boundary makes every partial visible without device-scope fences.
template <bool PRESSURE, bool LEARNED>
__device__ __forceinline__ void jacobi_reduce(const Dev &D, unsigned nparts, int check_done) {
    __shared__ double lds[RBLOCK / 64];
    Ctl *C = D.ctl;
    if (check_done && (PRESSURE ? C->done : C->done_v)) return;
    double t = 0.0, u = 0.0, l = 0.0;
    // eight partials per trip: their loads are issued together (the sums
    // are taken in the same fixed order as one at a time)
    const unsigned stride = blockDim.x;
    unsigned b = threadIdx.x;
    for (; b + 7 * stride < nparts; b += 8 * stride) {
        double2 e[8];
#pragma unroll
        for (int q = 0; q < 8; q++) e[q] = reinterpret_cast<const double2 *>(D.partial)[b + q * stride];
#pragma unroll
        for (int q = 0; q < 8; q++) {
            t += e[q].x;
            u += e[q].y;
        }
        if (LEARNED) {
            double f[8];
#pragma unroll
            for (int q = 0; q < 8; q++) f[q] = D.partial[2 * nparts + b + q * stride];
#pragma unroll
            for (int q = 0; q < 8; q++) l += f[q];
        }
    }
    for (; b < nparts; b += stride) {
        t += D.partial[2 * b];
        u += D.partial[2 * b + 1];
        if (LEARNED) l += D.partial[2 * nparts + b];
    }
    t = block_sum(t, lds);
    u = block_sum(u, lds);
    if (LEARNED) l = block_sum(l, lds);
    if (threadIdx.x == 0) {
        if (LEARNED) (PRESSURE ? C->nlearn : C->nlearn_v) = (unsigned)l;
        const double h = C->h;
        if (D.model) {
            // several models: this is model m's sweep; the iteration counts
            // and convergence is decided after the last model, every model
            // against its own tolerance (TimeStepDFSPH.cpp:324-341, 477-495)
            const int m = D.solveModel;
            const double cnt = (double)D.countm[m];
            const double avg = cnt > 0.0 ? t / cnt : 0.0, avo = cnt > 0.0 ? u / cnt : 0.0;
            const bool finite = isfinite(avg) && isfinite(avo);
            if (!finite) C->flags |= 1;
            const double eta = PRESSURE ? D.maxError * 0.01 * (double)D.rho0m[m]
                                        : (1.0 / h) * D.maxErrorV * 0.01 * (double)D.rho0m[m];
            const int chk = (avg <= eta && finite) ? 1 : 0;
            int &acc = PRESSURE ? C->chk_acc : C->chk_acc_v;
            acc = (m == 0) ? chk : (acc & chk);
            if (PRESSURE) {
                C->avg_err = avg;
                C->avg_over = avo;
            } else {
                C->avg_err_v = avg;
                C->avg_over_v = avo;
            }
            if (m + 1 == (int)D.nmodel) {
                if (PRESSURE) {
                    C->it += 1;
                    C->done = ((acc && C->it >= D.minIt) || C->it >= D.maxIt || !finite) ? 1 : 0;
                } else {
                    C->it_v += 1;
                    C->done_v = ((acc && C->it_v >= 1) || C->it_v >= D.maxItV || !finite) ? 1 : 0;
                }
            }
            return;
        }
        const double avg = D.n ? t / (double)D.n : 0.0;
        const double avo = D.n ? u / (double)D.n : 0.0;
        const bool finite = isfinite(avg) && isfinite(avo);
        if (!finite) C->flags |= 1;
        // The reference's criterion counts remaining compression only. A
        // learned start can also overshoot, which that criterion never
        // sees, so a solve started from it must also bring the excess
        // (positive residual at particles that keep pressure) below eta.
        if (PRESSURE) {
            C->avg_err = avg;
            C->avg_over = avo;
            C->it += 1;
            const double eta = D.maxError * 0.01 * (double)D.rho0;
            const bool chk = avg <= eta && (!D.strictP || avo <= eta);
            C->done = ((chk && C->it >= D.minIt) || C->it >= D.maxIt || !finite) ? 1 : 0;
        } else {
            C->avg_err_v = avg;
            C->avg_over_v = avo;
            C->it_v += 1;
            const double eta = (1.0 / h) * D.maxErrorV * 0.01 * (double)D.rho0;
            const bool chk = avg <= eta && (!D.strictV || avo <= eta);
            C->done_v = ((chk && C->it_v >= 1) || C->it_v >= D.maxItV || !finite) ? 1 : 0;
        }
    }
}

template <bool PRESSURE, bool LEARNED = false>
__global__ __launch_bounds__(RBLOCK) void k_jacobi_reduce(Dev D, unsigned nparts, int check_done) {
    jacobi_reduce<PRESSURE, LEARNED>(D, nparts, check_done);
}

// One block per scene: block s reduces scene s, whose Jacobi sweep ran with
// `lanes` lanes per particle.
template <bool PRESSURE>
__global__ __launch_bounds__(RBLOCK) void kb_jacobi_reduce(const Dev *__restrict__ Ds, int lanes, int check_done) {
    const Dev &D = Ds[blockIdx.x];
    jacobi_reduce<PRESSURE, false>(D, (D.n * (unsigned)lanes + BLOCK - 1) / BLOCK, check_done);
}

// done[s] = the solver's convergence flag of scene s (one thread per scene).
template <bool PRESSURE>
__global__ void kb_done(const Dev *__restrict__ Ds, unsigned nscenes, int *__restrict__ done) {
    const unsigned s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < nscenes) done[s] = PRESSURE ? Ds[s].ctl->done : Ds[s].ctl->done_v;
}

// Copies the solver's stiffness into the w component of the fluid positions
// (read by the acceleration sweeps with the neighbour's position). Launched
// at the start of a solve and before a stand-alone iteration or
// finalisation; the Jacobi update keeps the copy current.
template <bool PRESSURE>
__global__ __launch_bounds__(BLOCK) void k_stiff_to_w(Dev D) {
    const unsigned i = gtid();
    if (i >= D.n) return;
    reinterpret_cast<float *>(D.x + i)[3] = stiff_w(D, i, PRESSURE ? D.p[i] : D.pv[i]);
}

// Outside the pressure solves the viscosity and XSPH sweeps read m_j / rho_j
// from the w component of the fluid positions (the same FP32 quotient as
// computed in place), so one 16-byte load per neighbour gives both.
__global__ __launch_bounds__(BLOCK) void k_mrho_to_w(Dev D) {
    const unsigned i = gtid();
    if (i >= D.n) return;
    reinterpret_cast<float *>(D.x + i)[3] = mass_of(D, i) / D.rho[i];
}

// Field access in particle-id order: out[id[k]] = component values of slot k
// (COMPS 3: x, y, z; 1: component w of a float4), and back. The scattered
// side stays on the device, where a particle's slot and id are close to each
// other in cache; the host moves one contiguous block.
template <int COMPS>
__global__ __launch_bounds__(BLOCK) void k_field_out4(const float4 *__restrict__ f, const unsigned *__restrict__ id,
                                                      unsigned n, float *__restrict__ out) {
    const unsigned k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const float4 v = f[k];
    const size_t o = id[k];
    if (COMPS == 3) {
        out[3 * o] = v.x;
        out[3 * o + 1] = v.y;
        out[3 * o + 2] = v.z;
    } else {
        out[o] = v.w;
    }
}
__global__ __launch_bounds__(BLOCK) void k_field_out1(const unsigned *__restrict__ f, const unsigned *__restrict__ id,
                                                      unsigned n, unsigned *__restrict__ out) {
    const unsigned k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) out[id[k]] = f[k];
}
// f[k] = (in[id[k]], 0); zero (may be null) is cleared beside it.
__global__ __launch_bounds__(BLOCK) void k_field_in4(const float *__restrict__ in, const unsigned *__restrict__ id,
                                                     unsigned n, float4 *__restrict__ f, float4 *__restrict__ zero) {
    const unsigned k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const size_t o = id[k];
    f[k] = make_float4(in[3 * o], in[3 * o + 1], in[3 * o + 2], 0.f);
    if (zero) zero[k] = make_float4(0.f, 0.f, 0.f, 0.f);
}
__global__ __launch_bounds__(BLOCK) void k_field_in1(const unsigned *__restrict__ in, const unsigned *__restrict__ id,
                                                     unsigned n, unsigned *__restrict__ f) {
    const unsigned k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) f[k] = in[id[k]];
}

__global__ void k_set_time(Ctl *C, double t, double h) {
    C->time = t;
    C->h = h;
}

// divergenceSolve / pressureSolve finalisation (TimeStepDFSPH.cpp:345-383,
// 500-540): v += h a_p; the divergence solve also restores alpha *= h.
template <bool PRESSURE, int LPP>
__global__ __launch_bounds__(BLOCK) void k_finish(Dev D) {
    const unsigned t = gtid();
    const unsigned i = t / LPP, hl = t % LPP;
    const bool act = i < D.n;
    const bool live = act && is_active(D, i);  // a_p = 0 otherwise (TimeStepDFSPH.cpp:1309)
    __shared__ float plds[PAIR_LDS<LPP, SumVec::NT>];
    float *const T = pair_part<LPP, SumVec::NT>(plds);
    const float3 a = particle_accel<LPP>(D, i, hl, live, PRESSURE ? D.p : D.pv, T);
    if (!act || hl != 0) return;
    const float h = (float)D.ctl->h;
    D.ap[i] = make_float4(a.x, a.y, a.z, 0.f);
    float4 v = D.v[i];
    v.x += h * a.x;
    v.y += h * a.y;
    v.z += h * a.z;
    D.v[i] = v;
    if (!PRESSURE) D.alpha[i] *= h;
}

// p *= h^2 (which 0) or p_v *= h (which 1).
__global__ __launch_bounds__(BLOCK) void k_scale(Dev D, float *q, int which) {
    const unsigned i = gtid();
    if (i >= D.n) return;
    const double h = D.ctl->h;
    q[i] *= (which == 0) ? (float)(h * h) : (float)h;
}

// ----------------------------------------------------- non-pressure forces
// clearAccelerations (TimeStep.cpp:35-50), Viscosity_Weiler2018::applyForces
// (:928-940), XSPH::step (XSPH.cpp:138-216), updateTimeStepSizeCFL
// (Simulation.cpp:415-493) and v += h a (TimeStepDFSPH.cpp:192-208).
// Tangent frame of MathFunctions::getOrthogonalVectors (MathFunctions.cpp:234-247).
__device__ __forceinline__ void ortho(const float3 &n, float3 &t1, float3 &t2) {
    float3 v = make_float3(1.f, 0.f, 0.f);
    if (fabsf(n.x) > 0.999f) v = make_float3(0.f, 1.f, 0.f);
    t1 = make_float3(n.y * v.z - n.z * v.y, n.z * v.x - n.x * v.z, n.x * v.y - n.y * v.x);
    t2 = make_float3(n.y * t1.z - n.z * t1.y, n.z * t1.x - n.x * t1.z, n.x * t1.y - n.y * t1.x);
    const float l1 = sqrtf(sqn(t1.x, t1.y, t1.z)), l2 = sqrtf(sqn(t2.x, t2.y, t2.z));
    t1 = make_float3(t1.x / l1, t1.y / l1, t1.z / l1);
    t2 = make_float3(t2.x / l2, t2.y / l2, t2.z / l2);
}

// Boundary part of Viscosity_Standard for static boundaries
// (Viscosity_Standard.cpp:293-380): Akinci particles with
// d nu_b rho0 V_b / rho_i, volume maps through four samples of V_b / 4 on
// the tangent plane at (1 - |x_b - x_i| / h) h from the boundary point.
// Velocity of a moving body at sample point xs near boundary point xb, from
// the record's velocity at xb: v(xb) + omega x (xs - xb).
__device__ __forceinline__ float3 body_velocity_at(const Dev &D, const float4 &vrec, const float4 &xb,
                                                   const float4 &xs) {
    const float4 w = D.body[(unsigned)vrec.w];
    const float ex = xs.x - xb.x, ey = xs.y - xb.y, ez = xs.z - xb.z;
    return make_float3(vrec.x + (w.y * ez - w.z * ey), vrec.y + (w.z * ex - w.x * ez), vrec.z + (w.x * ey - w.y * ex));
}

// Volume-map boundary viscosity of slot o of particle i
// (Viscosity_Standard.cpp:355-403): four samples of V_b / 4 on the tangent
// plane at (1 - |x_b - x_i| / h) h from the boundary point, each with the
// body's velocity there (zero at rest). Writes the sample points and the
// acceleration each contributes; false for an empty or degenerate record.
__device__ __forceinline__ bool visc_map_samples(const Dev &D, unsigned i, unsigned o, const float4 &xi,
                                                 const float4 &vi, float4 *xs, float3 *as) {
    const float4 xb = D.vmb[(size_t)o * D.stride + i];
    if (!(xb.w > 0.f)) return false;
    float3 nrm = make_float3(xb.x - xi.x, xb.y - xi.y, xb.z - xi.z);
    const float nl = sqrtf(sqn(nrm.x, nrm.y, nrm.z));
    if (!(nl > 0.0001f)) return false;
    nrm = make_float3(nrm.x / nl, nrm.y / nl, nrm.z / nl);
    float3 t1, t2;
    ortho(nrm, t1, t2);
    const float h = D.K.h;
    const float vb = D.bmode == 3 ? xb.w * D.sphereVol : xb.w;
    const float dist = (1.0f - nl / h) * h, c = sviscB_of(D, i) * (0.25f * vb);
    const float4 vr = D.vmv ? D.vmv[(size_t)o * D.stride + i] : make_float4(0.f, 0.f, 0.f, 0.f);
    for (int q = 0; q < 4; q++) {
        const float3 t = q < 2 ? t1 : t2;
        const float sg = (q % 2 == 0) ? -1.f : 1.f;
        xs[q] = make_float4(xb.x + sg * t.x * dist, xb.y + sg * t.y * dist, xb.z + sg * t.z * dist, 0.f);
        float3 r;
        const float g = kernel_G(xi, xs[q], D.K, r);
        float dot;
        if (D.vmv) {
            const float3 u = body_velocity_at(D, vr, xb, xs[q]);
            dot = ((vi.x - u.x) * r.x + (vi.y - u.y) * r.y) + (vi.z - u.z) * r.z;
        } else {
            dot = (vi.x * r.x + vi.y * r.y) + vi.z * r.z;
        }
        const float s = c * dot / (sqn(r.x, r.y, r.z) + 0.01f * D.hs2);
        as[q] = make_float3(s * (g * r.x), s * (g * r.y), s * (g * r.z));
    }
    return true;
}

__device__ __forceinline__ void std_visc_boundary(const Dev &D, unsigned i, const float4 &xi, const float4 &vi,
                                                  float4 &ai) {
    auto term = [&](const float4 &xs, float c, float &bx, float &by, float &bz) {
        float3 r;
        const float g = kernel_G(xi, xs, D.K, r);
        const float dot = (vi.x * r.x + vi.y * r.y) + vi.z * r.z;
        const float s = c * dot / (sqn(r.x, r.y, r.z) + 0.01f * D.hs2);
        bx += s * (g * r.x);
        by += s * (g * r.y);
        bz += s * (g * r.z);
    };
    if (D.bmode == 1) {
        const float rhoi = D.rho[i];
        const unsigned cb = D.cb[i];
        for (unsigned k = 0; k < cb; k++) {
            const float4 xb = D.bx[D.nb[(size_t)k * D.stride + i]];
            term(xb, sviscB_of(D, i) * (rho0_of(D, i) * xb.w / rhoi), ai.x, ai.y, ai.z);
        }
    } else if (D.bmode == 2 || D.bmode == 3) {
        // Koschier2017: the samples stand for rho_b times the support's
        // volume 4/3 pi h^3 (Viscosity_Standard.cpp:295-340)
        for (unsigned o = 0; o < D.nvm; o++) {
            if (!(D.vmb[(size_t)o * D.stride + i].w > 0.f)) break;
            float4 xs[4];
            float3 as[4];
            if (!visc_map_samples(D, i, o, xi, vi, xs, as)) continue;
            float bx = 0.f, by = 0.f, bz = 0.f;  // a1 + a2 + a3 + a4
            for (int q = 0; q < 4; q++) {
                bx += as[q].x;
                by += as[q].y;
                bz += as[q].z;
            }
            ai.x += bx;
            ai.y += by;
            ai.z += bz;
        }
    }
}

// ------------------------------------------------------ dynamic bodies
// Force and torque partials of one block for body b: thread values summed
// in a fixed order (block_sum), written to bpart[block][b][0..6).
__device__ __forceinline__ void body_partial(const Dev &D, unsigned b, const double *ft, double *lds) {
    for (int c = 0; c < 6; c++) {
        const double v = block_sum(ft[c], lds);
        if (threadIdx.x == 0) D.bpart[((size_t)blockIdx.x * D.nbody + b) * 6 + c] = v;
    }
}

// f at point xs on body b: force += f, torque += (xs - reference point) x f.
__device__ __forceinline__ void body_add(const Dev &D, unsigned b, const float4 &xs, double fx, double fy, double fz,
                                         double *ft) {
    const float4 c = D.body[D.nbody + b];
    const double ex = (double)xs.x - (double)c.x, ey = (double)xs.y - (double)c.y, ez = (double)xs.z - (double)c.z;
    ft[0] += fx;
    ft[1] += fy;
    ft[2] += fz;
    ft[3] += ey * fz - ez * fy;
    ft[4] += ez * fx - ex * fz;
    ft[5] += ex * fy - ey * fx;
}

// BoundaryModel::addForce of computePressureAccel's volume-map terms in the
// solves' finalisation (applyBoundaryForces, TimeStepDFSPH.cpp:1357-1364):
// f = -m_i a with a = p_i (-V_b gradW(x_i - x_b)), acting at x_b.
template <bool PRESSURE>
__global__ __launch_bounds__(BLOCK) void k_body_force_p(Dev D) {
    __shared__ double lds[BLOCK / 64];
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < D.n && is_active(D, i);
    const float pi = live ? (PRESSURE ? D.p[i] : D.pv[i]) : 0.f;
    const float4 xi = live ? D.x[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    for (unsigned b = 0; b < D.nbody; b++) {
        double ft[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        if (live && D.body[b].w != 0.f && fabsf(pi) > D.eps) {
            for (unsigned o = 0; o < D.nvm; o++) {
                const float4 xb = D.vmb[(size_t)o * D.stride + i];
                if (!(xb.w > 0.f)) break;
                if ((unsigned)D.vmv[(size_t)o * D.stride + i].w != b) continue;
                float3 r;
                const float g = kernel_G(xi, xb, D.K, r);
                const float ax = pi * (-xb.w * (g * r.x)), ay = pi * (-xb.w * (g * r.y)),
                            az = pi * (-xb.w * (g * r.z));
                const double m = mass_of(D, i);
                body_add(D, b, xb, -m * ax, -m * ay, -m * az, ft);
            }
        }
        body_partial(D, b, ft, lds);
    }
}

// BoundaryModel::addForce of the non-pressure forces' volume-map terms:
// standard viscosity at its four sample points (Viscosity_Standard.cpp:
// 400-403) and XSPH at the boundary point (XSPH.cpp:203), from the
// velocities before the force sweep applies them.
__global__ __launch_bounds__(BLOCK) void k_body_force_np(Dev D) {
    __shared__ double lds[BLOCK / 64];
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool act = i < D.n;
    const float4 xi = act ? D.x[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 vi = act ? D.v[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float rhoi = act ? D.rho[i] : 1.f;
    const float invH = (float)(1.0 / D.ctl->h);
    const double m = act ? mass_of(D, i) : 0.0;
    for (unsigned b = 0; b < D.nbody; b++) {
        double ft[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        if (act && D.body[b].w != 0.f) {
            for (unsigned o = 0; o < D.nvm; o++) {
                const float4 xb = D.vmb[(size_t)o * D.stride + i];
                if (!(xb.w > 0.f)) break;
                const float4 vb = D.vmv[(size_t)o * D.stride + i];
                if ((unsigned)vb.w != b) continue;
                if (sviscB_of(D, i) != 0.f) {
                    float4 xs[4];
                    float3 as[4];
                    if (visc_map_samples(D, i, o, xi, vi, xs, as))
                        for (int q = 0; q < 4; q++) body_add(D, b, xs[q], -m * as[q].x, -m * as[q].y, -m * as[q].z, ft);
                }
                if (xsphB_of(D, i) != 0.f) {
                    const float w = kernel_W(xi, xb, D.K);
                    const float s = -invH * xsphB_of(D, i) * (rho0_of(D, i) * xb.w / rhoi);
                    body_add(D, b, xb, -m * (s * (vi.x - vb.x) * w), -m * (s * (vi.y - vb.y) * w),
                             -m * (s * (vi.z - vb.z) * w), ft);
                }
            }
        }
        body_partial(D, b, ft, lds);
    }
}

// Adds the per-block partials of every body, in block order, to its force
// and torque (one block).
__global__ __launch_bounds__(RBLOCK) void k_body_reduce(Dev D, unsigned nparts) {
    __shared__ double lds[RBLOCK / 64];
    for (unsigned b = 0; b < D.nbody; b++)
        for (int c = 0; c < 6; c++) {
            double t = 0.0;
            for (unsigned k = threadIdx.x; k < nparts; k += blockDim.x) t += D.bpart[((size_t)k * D.nbody + b) * 6 + c];
            t = block_sum(t, lds);
            if (threadIdx.x == 0) D.bforce[b * 6 + c] += t;
        }
}

template <bool CLEAR, bool APPLY, bool XSPH, bool CFL, bool VUPD, bool SCALEPV, int LPP>
__global__ __launch_bounds__(BLOCK) void k_post(Dev D) {
    __shared__ double lds[BLOCK / 64];
    __shared__ float plds[XSPH ? PAIR_LDS<LPP, SumVecAdd::NT> : 1];
    float *const T = pair_part<LPP, SumVecAdd::NT>(plds);
    Ctl *C = D.ctl;
    const unsigned t = gtid();
    const unsigned i = t / LPP, hl = t % LPP;
    const bool act = i < D.n;
    const double h = C->h;
    const float hf = (float)h;
    const float invH = (float)(1.0 / h);
    double vm = 0.0;
    float4 vi = make_float4(0.f, 0.f, 0.f, 0.f), xi = vi;
    float sx = 0.f, sy = 0.f, sz = 0.f;  // XSPH fluid sum
    float ux = 0.f, uy = 0.f, uz = 0.f;  // standard viscosity fluid sum
    float acc[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (act) {
        vi = D.v[i];
        if (XSPH) {
            xi = D.x[i];
            const float cxs = xsph_of(D, i), csv = svisc_of(D, i);
            const bool xs = cxs != 0.f, sv = csv != 0.f;
            const unsigned mi = D.model ? D.model[i] : 0u;
            const F4Gather X(D.x, D.n), V(D.v, D.n);
            // Viscosity_Standard (Viscosity_Standard.cpp:281-289), within the
            // model (forall_fluid_neighbors_in_same_phase, :271):
            // d nu m_j/rho_j (v_ij . x_ij) / (|x_ij|^2 + 0.01 h^2) gradW
            auto visc = [&](unsigned j, const auto &q, float *u) {
                if (!(sv && (!D.model || D.model[j] == mi))) return false;
                const float4 &xj = q.a, &vj = q.b;  // xj.w: m_j / rho_j
                float3 r;
                const float g = kernel_G(xi, xj, D.K, r);
                const float dot = fmaf(vi.z - vj.z, r.z, fmaf(vi.y - vj.y, r.y, (vi.x - vj.x) * r.x));
                u[0] = csv * xj.w * dot * g * __builtin_amdgcn_rcpf(fmaf(0.01f, D.hs2, sqn_fma(r.x, r.y, r.z)));
                u[1] = r.x;
                u[2] = r.y;
                u[3] = r.z;
                return true;
            };
            auto xsph = [&](const auto &q, float *u) {
                if (!xs) return false;
                const float4 &xj = q.a, &vj = q.b;
                const float w = kernel_W(xi, xj, D.K);
                const float s = invH * cxs * xj.w;
                u[0] = -(s * (vi.x - vj.x) * w);
                u[1] = -(s * (vi.y - vj.y) * w);
                u[2] = -(s * (vi.z - vj.z) * w);
                return true;
            };
            const auto ld = loads([&](unsigned j) { return X.all(j); }, [&](unsigned j) { return V.xyz(j); });
            const unsigned cnt = (xs || sv) ? D.cf[i] : 0u;
            if constexpr (LPP != ORDERED_LANES)
                fluid_pairs<LPP>(D, i, hl, cnt, ld, [&](unsigned j, const auto &q) {
                    float u[4];
                    if (visc(j, q, u)) sum_terms<SumVec>(u, acc + 3);
                    if (xsph(q, u)) sum_terms<SumAdd<3>>(u, acc);
                });
            else
                fluid_sums<LPP, SumVecAdd>(D, i, hl, cnt, T, acc, ld, [&](unsigned j, const auto &q, float *u) {
#pragma unroll
                    for (int c = 0; c < 7; c++) u[c] = 0.f;
                    u[7] = 1.f;
                    visc(j, q, u + 3);
                    xsph(q, u);
                    return true;
                });
        }
    }
    if (XSPH) {
        lanes_join<LPP, SumVecAdd>(acc);
        sx = acc[0];
        sy = acc[1];
        sz = acc[2];
        ux = acc[3];
        uy = acc[4];
        uz = acc[5];
    }
    if (act && hl == 0) {
        float4 ai = CLEAR ? make_float4(D.grav.x, D.grav.y, D.grav.z, 0.f) : D.a[i];
        if (APPLY) {
            float4 xs = D.cgx[i];
            if (C->cg_done == 2) xs = make_float4(0.f, 0.f, 0.f, 0.f);
            const float dx = xs.x - vi.x, dy = xs.y - vi.y, dz = xs.z - vi.z;
            ai.x += invH * dx;
            ai.y += invH * dy;
            ai.z += invH * dz;
            D.vdiff[i] = make_float4(dx, dy, dz, 0.f);
        }
        if (XSPH) {
            // computeViscosity before computeXSPH (Simulation.cpp:495-507)
            if (svisc_of(D, i) != 0.f) {
                ai.x += ux;
                ai.y += uy;
                ai.z += uz;
                if (sviscB_of(D, i) != 0.f) std_visc_boundary(D, i, xi, vi, ai);
            }
            ai.x += sx;
            ai.y += sy;
            ai.z += sz;
            const float cxb = xsphB_of(D, i), r0i = rho0_of(D, i);
            if (cxb != 0.f) {
                const float rhoi = D.rho[i];
                auto bterm = [&](const float4 &xb) {
                    const float w = kernel_W(xi, xb, D.K);
                    const float s = -invH * cxb * (r0i * xb.w / rhoi);
                    ai.x += s * vi.x * w;
                    ai.y += s * vi.y * w;
                    ai.z += s * vi.z * w;
                };
                if (D.bmode == 1) {
                    const unsigned cb = D.cb[i];
                    for (unsigned k = 0; k < cb; k++) bterm(D.bx[D.nb[(size_t)k * D.stride + i]]);
                } else if (D.bmode == 2) {
                    for (unsigned o = 0; o < D.nvm; o++) {
                        const float4 xb = D.vmb[(size_t)o * D.stride + i];
                        if (!(xb.w > 0.f)) break;
                        if (D.vmv) {  // (v_i - v_b) with v_b = getPointVelocity(x_b) (XSPH.cpp:198-203)
                            const float4 vb = D.vmv[(size_t)o * D.stride + i];
                            const float w = kernel_W(xi, xb, D.K);
                            const float s = -invH * cxb * (r0i * xb.w / rhoi);
                            ai.x += s * (vi.x - vb.x) * w;
                            ai.y += s * (vi.y - vb.y) * w;
                            ai.z += s * (vi.z - vb.z) * w;
                        } else {
                            bterm(xb);
                        }
                    }
                } else if (D.bmode == 3) {  // -(1/h) c_b (rho0 / rho_i) v_i rho_b (XSPH.cpp:111-120)
                    for (unsigned o = 0; o < D.nvm; o++) {
                        const float4 xb = D.vmb[(size_t)o * D.stride + i];
                        if (!(xb.w > 0.f)) break;
                        const float s = -invH * cxb * (r0i / rhoi) * xb.w;
                        ai.x += s * vi.x;
                        ai.y += s * vi.y;
                        ai.z += s * vi.z;
                    }
                }
            }
        }
        if (CLEAR || APPLY || XSPH) D.a[i] = ai;
        if (CFL) {
            const double wx = (double)vi.x + (double)ai.x * h, wy = (double)vi.y + (double)ai.y * h,
                         wz = (double)vi.z + (double)ai.z * h;
            vm = (wx * wx + wy * wy) + wz * wz;
        }
        if (VUPD) {
            // active particles only (TimeStepDFSPH.cpp:201)
            const float hs = (float)C->h_step;
            D.v2[i] = is_active(D, i) ? make_float4(vi.x + hs * ai.x, vi.y + hs * ai.y, vi.z + hs * ai.z, 0.f)
                                      : make_float4(vi.x, vi.y, vi.z, 0.f);
        }
        if (SCALEPV) D.pv[i] *= hf;
    }
    if (CFL) {
        const double bm = block_max(vm, lds);
        if (threadIdx.x == 0) D.partial[blockIdx.x] = bm;
    }
}

// CFL time step from the per-block maxima of |v + a h|^2
// (Simulation.cpp:415-493, cflMethod 2 at :399-412).
__global__ __launch_bounds__(RBLOCK) void k_cfl_reduce(Dev D, unsigned nparts) {
    __shared__ double lds[RBLOCK / 64];
    Ctl *C = D.ctl;
    double t = 0.0;
    for (unsigned b = threadIdx.x; b < nparts; b += blockDim.x) t = fmax(t, D.partial[b]);
    t = block_max(t, lds);
    if (threadIdx.x == 0) {
        const double h = C->h;
        double maxVel = t;
        if (!isfinite(maxVel)) C->flags |= 1;
        // animated and dynamic volume maps (Simulation.cpp:470-479): the
        // bodies' speed enters beside the particles' squared speeds, as there
        maxVel = fmax(maxVel, D.bodyMaxVel);
        if (maxVel < 1.0e-9) maxVel = 1.0e-9;
        const double diameter = 2.0 * D.radius;
        double hn = D.cflFactor * 0.4 * (diameter / sqrt(maxVel));
        hn = fmin(hn, D.cflMax);
        hn = fmax(hn, D.cflMin);
        if (D.cflMethod == 2 && C->it != 0) {
            double hh = h;
            if (C->it > 10)
                hh *= 0.9;
            else if (C->it < 5)
                hh *= 1.1;
            hn = fmin(hh, hn);
        }
        C->h = hn;
    }
}

// ------------------------------------------------------- pressure set-up
// computeDensityAdv + warm start (TimeStepDFSPH.cpp:264-309, 1191-1242).
template <int LPP>
__global__ __launch_bounds__(BLOCK) void k_psetup(Dev D) {
    const unsigned t = gtid();
    const unsigned i = t / LPP, hl = t % LPP;
    const bool act = i < D.n;
    __shared__ float plds[PAIR_LDS<LPP, SumDot::NT>];
    float *const T = pair_part<LPP, SumDot::NT>(plds);
    float4 xi = make_float4(0.f, 0.f, 0.f, 0.f), vi = xi;
    float delta = 0.f;
    if (act) {
        xi = D.x[i];
        vi = D.v[i];
        const F4Gather X(D.x, D.n), V(D.v, D.n);
        fluid_sums<LPP, SumDot>(
            D, i, hl, D.cf[i], T, &delta, loads([&](unsigned j) { return X.xyz(j); }, [&](unsigned j) { return V.xyz(j); }),
            [&](unsigned, const auto &q, float *u) { return aij_term(xi, vi, q.a, q.b, D.K, u); });
    }
    lanes_join<LPP, SumDot>(&delta);
    delta *= D.V;
    if (D.bmode == 1)
        akinci_sums<LPP, SumAdd<1>>(D, i, hl, act ? D.cb[i] : 0u, T, &delta, [&](const float4 &xb, float *u) {
            float3 r;
            const float g = kernel_G(xi, xb, D.K, r);
            u[0] = xb.w * ((vi.x * (g * r.x) + vi.y * (g * r.y)) + vi.z * (g * r.z));
            return true;
        });
    if (!act || hl != 0) return;
    const double h = D.ctl->h;
    if (D.bmode == 2) {
        for (unsigned o = 0; o < D.nvm; o++) {
            const float4 xb = D.vmb[(size_t)o * D.stride + i];
            if (!(xb.w > 0.f)) break;
            float3 r;
            const float g = kernel_G(xi, xb, D.K, r);
            if (D.vmv) {  // v_i - v_b, v_b = getPointVelocity(x_b) (TimeStepDFSPH.cpp:1236)
                const float4 vb = D.vmv[(size_t)o * D.stride + i];
                delta += xb.w * (((vi.x - vb.x) * (g * r.x) + (vi.y - vb.y) * (g * r.y)) + (vi.z - vb.z) * (g * r.z));
            } else {
                delta += xb.w * ((vi.x * (g * r.x) + vi.y * (g * r.y)) + vi.z * (g * r.z));
            }
        }
    } else if (D.bmode == 3) {  // TimeStepDFSPH.cpp:1224-1231
        for (unsigned o = 0; o < D.nvm; o++) {
            if (!(D.vmb[(size_t)o * D.stride + i].w > 0.f)) break;
            const float4 gb = D.dmg[(size_t)o * D.stride + i];
            delta -= (vi.x * gb.x + vi.y * gb.y) + vi.z * gb.z;
        }
    }
    const float radv = D.rho[i] / rho0_of(D, i) + (float)h * delta;
    D.radv[i] = radv;
    const float invH2 = (float)(1.0 / (h * h));
    D.alpha[i] *= invH2;
    const float p0 = D.p[i];
    if (D.kprev) D.kprev[i] = p0;
    const float p1 = (radv > 1.0f) ? 0.5f * fminf(p0, 0.00025f) * invH2 : 0.0f;
    D.p[i] = p1;
    reinterpret_cast<float *>(D.x + i)[3] = stiff_w(D, i, p1);  // the solve's stiffness copy
}

// p *= h^2 and the compensated position update x += h_step v (Kahan), then
// t += h_step (TimeStepDFSPH.cpp:220-248, 369-383).
template <bool SCALEP, bool UPDX>
__global__ __launch_bounds__(BLOCK) void k_final(Dev D) {
    const unsigned i = gtid();
    Ctl *C = D.ctl;
    if (UPDX && blockIdx.x == 0 && threadIdx.x == 0) {
        // the time advances once per launch; every block reads h_step only
        C->t_prev = C->time;
        C->time += C->h_step;
    }
    if (i >= D.n) return;
    if (SCALEP) {
        const double h = C->h;
        D.p[i] *= (float)(h * h);
    }
    if (UPDX && is_active(D, i)) {  // TimeStepDFSPH.cpp:229
        const float hs = (float)C->h_step;
        const float4 v = D.v[i];
        float4 x = D.x[i], c = D.xc[i];
        const float yx = hs * v.x - c.x, yy = hs * v.y - c.y, yz = hs * v.z - c.z;
        const float tx = x.x + yx, ty = x.y + yy, tz = x.z + yz;
        c.x = (tx - x.x) - yx;
        c.y = (ty - x.y) - yy;
        c.z = (tz - x.z) - yz;
        x.x = tx;
        x.y = ty;
        x.z = tz;
        D.x[i] = x;
        D.xc[i] = c;
    }
}

// ------------------------------------------------------------ Weiler2018
// diagonalMatrixElement, block form (Viscosity_Weiler2018.cpp:605-742),
// inverted for the block-Jacobi preconditioner (MatrixFreeSolver.h:231-245),
// and the warm start g = v + vDiff (:1244-1251).
__device__ __forceinline__ void sym_inverse(const double m[6], double inv[6]) {
    // m = (xx, xy, xz, yy, yz, zz)
    const double a = m[0], b = m[1], c = m[2], d = m[3], e = m[4], f = m[5];
    const double c00 = d * f - e * e, c01 = c * e - b * f, c02 = b * e - c * d;
    const double det = a * c00 + b * c01 + c * c02;
    const double id = 1.0 / det;
    inv[0] = c00 * id;
    inv[1] = c01 * id;
    inv[2] = c02 * id;
    inv[3] = (a * f - c * c) * id;
    inv[4] = (b * c - a * e) * id;
    inv[5] = (a * d - b * b) * id;
}


// Boundary samples of the Weiler2018 operator for particle i: calls
// f(xs, c) for every boundary sample position xs with its coefficient
// c = d mu_b V_b (Akinci particles: V_b = rho0 V_b / rho_i, as the reference
// weighs them; volume maps: four samples of V_b / 4 on the tangent plane at
// h / 2 from the boundary point, Viscosity_Weiler2018.cpp:327-438, 672-740).
template <class F>
__device__ __forceinline__ void weiler_boundary(const Dev &D, unsigned i, const float4 &xi, float rhoi, F &&f) {
    const float dd = 10.0f;
    if (D.mub == 0.f) return;
    if (D.bmode == 1) {
        const unsigned cb = D.cb[i];
        for (unsigned k = 0; k < cb; k++) {
            const float4 xb = D.bx[D.nb[(size_t)k * D.stride + i]];
            f(xb, dd * D.mub * (D.rho0 * xb.w / rhoi));
        }
    } else if (D.bmode == 2 || D.bmode == 3) {
        // Koschier2017: rho_b times 4/3 pi h^3 (Viscosity_Weiler2018.cpp:154-200)
        for (unsigned o = 0; o < D.nvm; o++) {
            const float4 xb = D.vmb[(size_t)o * D.stride + i];
            if (!(xb.w > 0.f)) break;
            float3 nrm = make_float3(xb.x - xi.x, xb.y - xi.y, xb.z - xi.z);
            const float nl = sqrtf(sqn(nrm.x, nrm.y, nrm.z));
            if (nl > 0.0001f) {
                nrm = make_float3(nrm.x / nl, nrm.y / nl, nrm.z / nl);
                float3 t1, t2;
                ortho(nrm, t1, t2);
                const float dist = 0.5f * D.K.h, vol = 0.25f * (D.bmode == 3 ? xb.w * D.sphereVol : xb.w);
                for (int q = 0; q < 4; q++) {
                    const float3 t = q < 2 ? t1 : t2;
                    const float sg = (q % 2 == 0) ? -1.f : 1.f;
                    const float4 xs = make_float4(xb.x + sg * t.x * dist, xb.y + sg * t.y * dist,
                                                  xb.z + sg * t.z * dist, 0.f);
                    f(xs, dd * D.mub * vol);
                }
            }
        }
    }
}

// Terms of one pair of the operator: with c the pair's coefficient (fluid:
// d mu m_j / rho_j), weiler_av gives t = (s, r) with s r = c (dv . r) /
// (|r|^2 + 0.01 h^2) g_ij r, its part of the product, and weiler_diag
// t = (u, r) with u r^T = c g_ij (r r^T) / (|r|^2 + 0.01 h^2), its part of
// the block diagonal (xx xy xz yy yz zz).
// The quotients use the hardware reciprocal (1 ulp) in place of a
// correctly rounded division: a per-pair term carries rounding at the
// 1e-7 level either way.
__device__ __forceinline__ bool weiler_av(const Dev &D, const float4 &xi, const float4 &xj, float c, const float4 &vi,
                                          const float4 &vj, float *t) {
    float3 r;
    const float g = kernel_G(xi, xj, D.K, r);
    const float iden = __builtin_amdgcn_rcpf(fmaf(0.01f, D.hs2, sqn_fma(r.x, r.y, r.z)));
    const float dot = fmaf(vi.z - vj.z, r.z, fmaf(vi.y - vj.y, r.y, (vi.x - vj.x) * r.x));
    t[0] = c * dot * iden * g;
    t[1] = r.x;
    t[2] = r.y;
    t[3] = r.z;
    return true;
}
__device__ __forceinline__ bool weiler_diag(const Dev &D, const float4 &xi, const float4 &xj, float c, float *t) {
    float3 r;
    const float g = kernel_G(xi, xj, D.K, r);
    const float iden = __builtin_amdgcn_rcpf(fmaf(0.01f, D.hs2, sqn_fma(r.x, r.y, r.z)));
    const float s = c * iden * g;  // c g / den
    t[0] = s * r.x;
    t[1] = s * r.y;
    t[2] = s * r.z;
    t[3] = r.x;
    t[4] = r.y;
    t[5] = r.z;
    return true;
}
__device__ __forceinline__ float3 minv_apply(const Dev &D, unsigned i, const float3 &r) {
    const float4 a = D.minv[2 * i], b = D.minv[2 * i + 1];
    return make_float3((a.x * r.x + a.y * r.y) + a.z * r.z, (a.y * r.x + a.w * r.y) + b.x * r.z,
                       (a.z * r.x + b.x * r.y) + b.y * r.z);
}

// matrixVecProd (Viscosity_Weiler2018.cpp:271-441): (A vec)_i.
// For LPP > 1 every lane of the particle calls this (the fluid sum is split
// over them); the result is valid in lane hl == 0 only. The fluid
// positions' w holds m_j / rho_j.
template <int LPP>
__device__ __forceinline__ float3 weiler_Av(const Dev &D, unsigned i, unsigned hl, bool act,
                                            const float4 *__restrict__ vec, float *__restrict__ T) {
    const float dd = 10.0f;
    float4 xi = make_float4(0.f, 0.f, 0.f, 0.f), vi = xi;
    float a[3] = {0.f, 0.f, 0.f};
    if (act) {
        xi = D.x[i];
        vi = vec[i];
        const F4Gather X(D.x, D.n), Vc(vec, D.n);
        fluid_sums<LPP, SumVec>(
            D, i, hl, D.cf[i], T, a, loads([&](unsigned j) { return X.all(j); }, [&](unsigned j) { return Vc.xyz(j); }),
            [&](unsigned, const auto &q, float *t) { return weiler_av(D, xi, q.a, dd * D.mu * q.a.w, vi, q.b, t); });
    }
    lanes_join<LPP, SumVec>(a);
    if (!act || hl != 0) return make_float3(0.f, 0.f, 0.f);
    const float rhoi = D.rho[i];
    const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
    weiler_boundary(D, i, xi, rhoi, [&](const float4 &xs, float c) {
        float t[4];
        weiler_av(D, xi, xs, c, vi, z4, t);
        sum_terms<SumVec>(t, a);
    });
    const float f = (float)D.ctl->h / rhoi;
    return make_float3(vi.x - f * a[0], vi.y - f * a[1], vi.z - f * a[2]);
}

// Set-up of the Weiler2018 solve, in Eigen's order (ConjugateGradient.h:43-70):
// first the residual of the warm start, and only if it does not meet the
// tolerance the preconditioner. k_weiler_x0 writes x0 = v + vDiff
// (Viscosity_Weiler2018.cpp:1244-1251); k_weiler_r0 forms r = b - A x0
// (b = v for static boundaries) and the sums |b|^2, |r|^2; k_cg_init_reduce
// decides whether the CG iterates.
// x0 = v + vDiff of every particle into the CG solution vector (the warm
// start, Viscosity_Weiler2018.cpp:1244-1251), so that k_weiler_r0 gathers
// one vector per neighbour.
__global__ __launch_bounds__(BLOCK) void k_weiler_x0(Dev D) {
    const unsigned i = gtid();
    if (i >= D.n) return;
    const float4 v = D.v[i], vd = D.vdiff[i];
    D.cgx[i] = make_float4(v.x + vd.x, v.y + vd.y, v.z + vd.z, 0.f);
}

template <int LPP>
__global__ __launch_bounds__(BLOCK) void k_weiler_r0(Dev D) {
    __shared__ double lds[BLOCK / 64];
    const unsigned t = gtid();
    const unsigned i = t / LPP, hl = t % LPP;
    const bool act = i < D.n;
    __shared__ float plds[PAIR_LDS<LPP, SumVec::NT>];
    float *const T = pair_part<LPP, SumVec::NT>(plds);
    const float dd = 10.0f;
    float4 xi = make_float4(0.f, 0.f, 0.f, 0.f), x0i = xi, vi = xi;
    float a[3] = {0.f, 0.f, 0.f};
    if (act) {
        xi = D.x[i];
        vi = D.v[i];
        const float4 vd = D.vdiff[i];
        x0i = make_float4(vi.x + vd.x, vi.y + vd.y, vi.z + vd.z, 0.f);
        const F4Gather X(D.x, D.n), X0(D.cgx, D.n);
        fluid_sums<LPP, SumVec>(
            D, i, hl, D.cf[i], T, a, loads([&](unsigned j) { return X.all(j); }, [&](unsigned j) { return X0.xyz(j); }),
            [&](unsigned, const auto &q, float *u) { return weiler_av(D, xi, q.a, dd * D.mu * q.a.w, x0i, q.b, u); });
    }
    lanes_join<LPP, SumVec>(a);
    double b2 = 0.0, r2 = 0.0;
    if (act && hl == 0) {
        const float rhoi = D.rho[i];
        const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
        weiler_boundary(D, i, xi, rhoi, [&](const float4 &xs, float c) {
            float u[4];
            weiler_av(D, xi, xs, c, x0i, z4, u);
            sum_terms<SumVec>(u, a);
        });
        const float fa = (float)D.ctl->h / rhoi;
        const float3 Ax = make_float3(x0i.x - fa * a[0], x0i.y - fa * a[1], x0i.z - fa * a[2]);
        const float3 r = make_float3(vi.x - Ax.x, vi.y - Ax.y, vi.z - Ax.z);
        D.cgr[i] = make_float4(r.x, r.y, r.z, 0.f);
        b2 = ((double)vi.x * vi.x + (double)vi.y * vi.y) + (double)vi.z * vi.z;
        r2 = ((double)r.x * r.x + (double)r.y * r.y) + (double)r.z * r.z;
    }
    const double s0 = block_sum(b2, lds), s1 = block_sum(r2, lds);
    if (threadIdx.x == 0) {
        D.partial[2 * blockIdx.x] = s0;
        D.partial[2 * blockIdx.x + 1] = s1;
    }
}

__global__ __launch_bounds__(RBLOCK) void k_cg_init_reduce(Dev D, unsigned nparts) {
    __shared__ double lds[RBLOCK / 64];
    Ctl *C = D.ctl;
    double t0 = 0.0, t1 = 0.0;
    for (unsigned b = threadIdx.x; b < nparts; b += blockDim.x) {
        t0 += D.partial[2 * b];
        t1 += D.partial[2 * b + 1];
    }
    t0 = block_sum(t0, lds);
    t1 = block_sum(t1, lds);
    if (threadIdx.x == 0) {
        C->cg_rhs2 = t0;
        C->cg_r2 = t1;
        C->cg_it = 0;
        if (t0 == 0.0) {
            C->cg_done = 2;  // x = 0, no iteration
        } else {
            const double thr = fmax(D.viscoTol * D.viscoTol * t0, DBL_MIN);
            C->cg_thresh = thr;
            C->cg_done = (t1 < thr || D.viscoMaxIt <= 0) ? 1 : 0;
        }
    }
}

// The preconditioner, only when the CG iterates: the block diagonal
// (diagonalMatrixElement, Viscosity_Weiler2018.cpp:605-742) inverted for the
// block-Jacobi preconditioner (MatrixFreeSolver.h:231-245), z = M^-1 r,
// p = z and the sum r . z, which k_cg_rz_reduce turns into Eigen's absNew.
template <int LPP>
__global__ __launch_bounds__(BLOCK) void k_weiler_precond(Dev D) {
    __shared__ double lds[BLOCK / 64];
    if (D.ctl->cg_done) return;
    const unsigned t = gtid();
    const unsigned i = t / LPP, hl = t % LPP;
    const bool act = i < D.n;
    const float dd = 10.0f;
    __shared__ float plds[PAIR_LDS<LPP, SumSym::NT>];
    float *const T = pair_part<LPP, SumSym::NT>(plds);
    float m[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float4 xi = make_float4(0.f, 0.f, 0.f, 0.f);
    if (act) {
        xi = D.x[i];
        const F4Gather X(D.x, D.n);
        fluid_sums<LPP, SumSym>(
            D, i, hl, D.cf[i], T, m, loads([&](unsigned j) { return X.all(j); }),
            [&](unsigned, const auto &q, float *u) { return weiler_diag(D, xi, q.a, dd * D.mu * q.a.w, u); });
    }
    lanes_join<LPP, SumSym>(m);
    double rz = 0.0;
    if (act && hl == 0) {
        const float rhoi = D.rho[i];
        weiler_boundary(D, i, xi, rhoi, [&](const float4 &xs, float c) {
            float u[6];
            weiler_diag(D, xi, xs, c, u);
            sum_terms<SumSym>(u, m);
        });
        const double f = (double)D.ctl->h / (double)rhoi;
        double md[6] = {1.0 - f * m[0], -f * m[1], -f * m[2], 1.0 - f * m[3], -f * m[4], 1.0 - f * m[5]};
        double inv[6];
        sym_inverse(md, inv);
        const float4 ma = make_float4((float)inv[0], (float)inv[1], (float)inv[2], (float)inv[3]);
        const float4 mb = make_float4((float)inv[4], (float)inv[5], 0.f, 0.f);
        D.minv[2 * i] = ma;
        D.minv[2 * i + 1] = mb;
        const float4 r = D.cgr[i];
        const float3 z = make_float3((ma.x * r.x + ma.y * r.y) + ma.z * r.z, (ma.y * r.x + ma.w * r.y) + mb.x * r.z,
                                     (ma.z * r.x + mb.x * r.y) + mb.y * r.z);
        D.cgz[i] = make_float4(z.x, z.y, z.z, 0.f);
        D.cgp[i] = make_float4(z.x, z.y, z.z, 0.f);
        rz = ((double)r.x * z.x + (double)r.y * z.y) + (double)r.z * z.z;
    }
    const double s = block_sum(rz, lds);
    if (threadIdx.x == 0) D.partial[blockIdx.x] = s;
}

__global__ __launch_bounds__(RBLOCK) void k_cg_rz_reduce(Dev D, unsigned nparts) {
    __shared__ double lds[RBLOCK / 64];
    Ctl *C = D.ctl;
    if (C->cg_done) return;
    double t = 0.0;
    for (unsigned b = threadIdx.x; b < nparts; b += blockDim.x) t += D.partial[b];
    t = block_sum(t, lds);
    if (threadIdx.x == 0) C->cg_absNew = t;
}

// tmp = A p and alpha = absNew / (p . tmp).
template <int LPP>
__global__ __launch_bounds__(BLOCK) void k_cg_matvec(Dev D) {
    __shared__ double lds[BLOCK / 64];
    Ctl *C = D.ctl;
    if (C->cg_done) return;
    const unsigned tid = gtid();
    const unsigned i = tid / LPP, hl = tid % LPP;
    const bool act = i < D.n;
    __shared__ float plds[PAIR_LDS<LPP, SumVec::NT>];
    float *const T = pair_part<LPP, SumVec::NT>(plds);
    double pt = 0.0;
    const float3 t = weiler_Av<LPP>(D, i, hl, act, D.cgp, T);
    if (act && hl == 0) {
        D.cgt[i] = make_float4(t.x, t.y, t.z, 0.f);
        const float4 p = D.cgp[i];
        pt = ((double)p.x * t.x + (double)p.y * t.y) + (double)p.z * t.z;
    }
    const double bs = block_sum(pt, lds);
    if (threadIdx.x == 0) D.partial[blockIdx.x] = bs;
}

__global__ __launch_bounds__(RBLOCK) void k_cg_alpha(Dev D, unsigned nparts) {
    __shared__ double lds[RBLOCK / 64];
    Ctl *C = D.ctl;
    if (C->cg_done) return;
    double t = 0.0;
    for (unsigned b = threadIdx.x; b < nparts; b += blockDim.x) t += D.partial[b];
    t = block_sum(t, lds);
    if (threadIdx.x == 0) C->cg_alpha = C->cg_absNew / t;
}

// x += alpha p, r -= alpha tmp, z = M^-1 r; convergence test on |r|^2 and
// beta = (r.z)_new / (r.z)_old (ConjugateGradient.h:71-88).
__global__ __launch_bounds__(BLOCK) void k_cg_update(Dev D) {
    __shared__ double lds[BLOCK / 64];
    Ctl *C = D.ctl;
    if (C->cg_done) return;
    const unsigned i = gtid();
    const float alpha = (float)C->cg_alpha;
    double r2 = 0.0, rz = 0.0;
    if (i < D.n) {
        const float4 p = D.cgp[i], t = D.cgt[i];
        float4 x = D.cgx[i], r = D.cgr[i];
        x.x += alpha * p.x;
        x.y += alpha * p.y;
        x.z += alpha * p.z;
        r.x -= alpha * t.x;
        r.y -= alpha * t.y;
        r.z -= alpha * t.z;
        D.cgx[i] = x;
        D.cgr[i] = r;
        const float3 z = minv_apply(D, i, make_float3(r.x, r.y, r.z));
        D.cgz[i] = make_float4(z.x, z.y, z.z, 0.f);
        r2 = ((double)r.x * r.x + (double)r.y * r.y) + (double)r.z * r.z;
        rz = ((double)r.x * z.x + (double)r.y * z.y) + (double)r.z * z.z;
    }
    const double s1 = block_sum(r2, lds), s2 = block_sum(rz, lds);
    if (threadIdx.x == 0) {
        D.partial[2 * blockIdx.x] = s1;
        D.partial[2 * blockIdx.x + 1] = s2;
    }
}

__global__ __launch_bounds__(RBLOCK) void k_cg_update_reduce(Dev D, unsigned nparts) {
    __shared__ double lds[RBLOCK / 64];
    Ctl *C = D.ctl;
    if (C->cg_done) return;
    double t1 = 0.0, t2 = 0.0;
    for (unsigned b = threadIdx.x; b < nparts; b += blockDim.x) {
        t1 += D.partial[2 * b];
        t2 += D.partial[2 * b + 1];
    }
    t1 = block_sum(t1, lds);
    t2 = block_sum(t2, lds);
    if (threadIdx.x == 0) {
        C->cg_r2 = t1;
        if (!isfinite(t1)) C->flags |= 1;
        if (t1 < C->cg_thresh || !isfinite(t1)) {
            C->cg_done = 1;
        } else {
            const double absOld = C->cg_absNew;
            C->cg_absNew = t2;
            C->cg_beta = t2 / absOld;
            C->cg_it += 1;
            if (C->cg_it >= D.viscoMaxIt) C->cg_done = 3;  // p no longer needed
        }
    }
}

__global__ __launch_bounds__(BLOCK) void k_cg_pupdate(Dev D) {
    Ctl *C = D.ctl;
    if (C->cg_done) return;
    const unsigned i = gtid();
    if (i >= D.n) return;
    const float beta = (float)C->cg_beta;
    const float4 z = D.cgz[i];
    float4 p = D.cgp[i];
    p.x = z.x + beta * p.x;
    p.y = z.y + beta * p.y;
    p.z = z.z + beta * p.z;
    D.cgp[i] = p;
}

// Akinci2012 boundary volume V_b = 1 / (W0 + sum_b' W) (BoundaryModel_Akinci2012.cpp:48-75).
__global__ __launch_bounds__(BLOCK) void k_boundary_volume(float4 *bx, unsigned nb, const unsigned *nbr,
                                                           const unsigned *cnt, unsigned stride, KernelConst K) {
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nb) return;
    const float4 xi = bx[i];
    float delta = K.W0;
    const unsigned c = cnt[i];
    for (unsigned k = 0; k < c; k++) delta += kernel_W(xi, bx[nbr[(size_t)k * stride + i]], K);
    bx[i].w = 1.0f / delta;
}

// ----------------------------------------------------- learned warm start
// Block maxima of the previous-step stiffness, then the step's scale.
__global__ __launch_bounds__(BLOCK) void k_max_partial(Dev D, const float *__restrict__ q) {
    __shared__ double lds[BLOCK / 64];
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    const double v = (i < D.n) ? (double)fmaxf(q[i], 0.0f) : 0.0;
    const double m = block_max(v, lds);
    if (threadIdx.x == 0) D.partial[blockIdx.x] = m;
}
template <bool PRESSURE>
__global__ __launch_bounds__(RBLOCK) void k_kref_reduce(Dev D, unsigned nparts) {
    __shared__ double lds[RBLOCK / 64];
    double t = 0.0;
    for (unsigned b = threadIdx.x; b < nparts; b += blockDim.x) t = fmax(t, D.partial[b]);
    t = block_max(t, lds);
    if (threadIdx.x == 0) {
        if (PRESSURE)
            D.ctl->kref = t;
        else
            D.ctl->kref_v = t;
    }
}

// Per-particle inputs of the warm-start network: the solve's source term
// (density deviation 1 - rho_adv, or the divergence rho_dot h), its kernel-
// weighted neighbourhood mean, the previous-step stiffness and its mean (both
// relative to the step's largest), the boundary volume (relative to V) and
// the neighbour count / 40.
template <bool PRESSURE, int LPP>
__global__ __launch_bounds__(BLOCK) void k_features(Dev D) {
    const unsigned t = gtid();
    const unsigned i = t / LPP, hl = t % LPP;
    if (i >= D.n) return;
    const double h = D.ctl->h;
    const float sh = PRESSURE ? 1.0f : (float)h;
    const float off = PRESSURE ? 1.0f : 0.0f;
    const float kref = (float)(PRESSURE ? D.ctl->kref : D.ctl->kref_v);
    const float ik = kref > 0.f ? 1.0f / kref : 0.0f;
    const float4 xi = D.x[i];
    const float src_i = (D.radv[i] - off) * sh;
    __shared__ float plds[PAIR_LDS<LPP, 3>];
    float *const T = pair_part<LPP, 3>(plds);
    const float w0 = D.V * D.K.W0;
    float acc[3] = {w0, w0 * src_i, w0 * D.kprev[i]};
    const unsigned cnt = D.cf[i], cb = D.bmode == 1 ? D.cb[i] : 0u;
    const F4Gather X(D.x, D.n);
    fluid_sums<LPP, SumAdd<3>>(
        D, i, hl, cnt, T, acc,
        loads([&](unsigned j) { return X.xyz(j); }, [&](unsigned j) { return D.radv[j]; },
              [&](unsigned j) { return D.kprev[j]; }),
        [&](unsigned, const auto &q, float *u) {
            const float w = D.V * kernel_W(xi, q.a, D.K);
            u[0] = w;
            u[1] = w * ((q.b - off) * sh);
            u[2] = w * q.c;
            return true;
        });
    const float wsum = acc[0], ssrc = acc[1], sk = acc[2];
    float bvol = 0.f;
    const unsigned nnb = cnt + cb;
    if (D.bmode == 1)
        akinci_sums<LPP, SumAdd<1>>(D, i, hl, cb, T, &bvol, [&](const float4 &xb, float *u) {
            u[0] = xb.w;
            return true;
        });
    if (hl != 0) return;
    if (D.bmode == 2 || D.bmode == 3) {
        for (unsigned o = 0; o < D.nvm; o++) {
            const float w = D.vmb[(size_t)o * D.stride + i].w;
            if (!(w > 0.f)) break;
            bvol += w;
        }
    }
    float *F = (PRESSURE ? D.feats : D.feats_v) + (size_t)i * 8;
    reinterpret_cast<float4 *>(F)[0] =
        make_float4(100.0f * src_i, 100.0f * ssrc / wsum, D.kprev[i] * ik, (sk / wsum) * ik);
    reinterpret_cast<float4 *>(F)[1] = make_float4(bvol / D.V, (float)nnb * (1.0f / 40.0f), 0.f, 0.f);
}

// The two candidate starts of a learned solve. Fallback (into p / p_v): the
// previous step's full stiffness wherever the reference starts from it
// (rho_adv > 1; rho_dot > 0 with at least 20 neighbours,
// TimeStepDFSPH.cpp:292-296, 418-453), i.e. the reference's start without
// its factor 1/2 and clamp. Candidate (into pred): the previous stiffness
// everywhere (NET = false), or plus the network's predicted change,
// p = max(kappa_prev / kref + y, 0) kref / h^2 (NET = true; p_v: / h).
template <bool PRESSURE, bool NET>
__global__ __launch_bounds__(BLOCK) void k_pred_start(Dev D) {
    const unsigned i = gtid();
    if (i >= D.n) return;
    const double h = D.ctl->h;
    const float c = PRESSURE ? (float)(1.0 / (h * h)) : (float)(1.0 / h);
    const float kp = fmaxf(D.kprev[i], 0.0f);
    float q;
    if (NET) {
        const float kref = (float)(PRESSURE ? D.ctl->kref : D.ctl->kref_v);
        const float *F = (PRESSURE ? D.feats : D.feats_v) + (size_t)i * 8;
        q = fmaxf(F[2] + D.pred[i], 0.0f) * (kref * c);
    } else {
        q = kp * c;
    }
    float b = kp * c;
    if (PRESSURE) {
        if (!(D.radv[i] > 1.0f)) b = 0.0f;
        D.p[i] = b;
    } else {
        const unsigned nnb = D.cf[i] + (D.bmode == 1 ? D.cb[i] : 0u);
        if (!(D.radv[i] > 0.0f) || nnb < 20u) b = q = 0.0f;
        D.pv[i] = b;
    }
    reinterpret_cast<float *>(D.x + i)[3] = b;
    D.pred[i] = q;
}

// Pressure accelerations of both candidate starts (plain P, predicted Q).
template <bool PRESSURE, int LPP>
__global__ __launch_bounds__(BLOCK) void k_accel2(Dev D) {
    const unsigned t = gtid();
    const unsigned i = t / LPP, hl = t % LPP;
    if (i >= D.n) return;
    if (!is_active(D, i)) {
        if (hl == 0) D.ap[i] = D.ap2[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        return;
    }
    const float *__restrict__ P = PRESSURE ? D.p : D.pv;
    const float *__restrict__ Q = D.pred;
    const float4 xi = D.x[i];
    const float pi = P[i], qi = Q[i];
    __shared__ float plds[PAIR_LDS<LPP, 6>];
    float *const T = pair_part<LPP, 6>(plds);
    // the fallback start P of a neighbour comes with its position: k_pred_start
    // wrote it into the w component as well
    const F4Gather X(D.x, D.n);
    float acc[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    fluid_sums<LPP, SumAdd<6>>(
        D, i, hl, D.cf[i], T, acc, loads([&](unsigned j) { return X.all(j); }, [&](unsigned j) { return Q[j]; }),
        [&](unsigned, const auto &n, float *u) {
            const float ps = pi + n.a.w, qs = qi + n.b;
            const bool a = fabsf(ps) > D.eps, b = fabsf(qs) > D.eps;
            if (!(a || b)) return false;
            float3 r;
            const float g = kernel_G(xi, n.a, D.K, r);
            const float gx = -D.V * (g * r.x), gy = -D.V * (g * r.y), gz = -D.V * (g * r.z);
            u[0] = a ? ps * gx : 0.f;
            u[1] = a ? ps * gy : 0.f;
            u[2] = a ? ps * gz : 0.f;
            u[3] = b ? qs * gx : 0.f;
            u[4] = b ? qs * gy : 0.f;
            u[5] = b ? qs * gz : 0.f;
            return true;
        });
    const bool bp = fabsf(pi) > D.eps, bq = fabsf(qi) > D.eps;
    auto bterm = [&](const float4 &xb, float *u) {
        float3 r;
        const float g = kernel_G(xi, xb, D.K, r);
        const float gx = -xb.w * (g * r.x), gy = -xb.w * (g * r.y), gz = -xb.w * (g * r.z);
        u[0] = bp ? pi * gx : 0.f;
        u[1] = bp ? pi * gy : 0.f;
        u[2] = bp ? pi * gz : 0.f;
        u[3] = bq ? qi * gx : 0.f;
        u[4] = bq ? qi * gy : 0.f;
        u[5] = bq ? qi * gz : 0.f;
        return true;
    };
    if (D.bmode == 1) {
        akinci_sums<LPP, SumAdd<6>>(D, i, hl, (bp || bq) ? D.cb[i] : 0u, T, acc, bterm);
    } else if (D.bmode == 2 && (bp || bq) && hl == 0) {
        for (unsigned o = 0; o < D.nvm; o++) {
            const float4 xb = D.vmb[(size_t)o * D.stride + i];
            if (!(xb.w > 0.f)) break;
            float u[6];
            bterm(xb, u);
            sum_terms<SumAdd<6>>(u, acc);
        }
    } else if (D.bmode == 3 && (bp || bq) && hl == 0) {
        for (unsigned o = 0; o < D.nvm; o++) {
            if (!(D.vmb[(size_t)o * D.stride + i].w > 0.f)) break;
            const float4 gb = D.dmg[(size_t)o * D.stride + i];
            if (bp) {
                acc[0] += pi * gb.x;
                acc[1] += pi * gb.y;
                acc[2] += pi * gb.z;
            }
            if (bq) {
                acc[3] += qi * gb.x;
                acc[4] += qi * gb.y;
                acc[5] += qi * gb.z;
            }
        }
    }
    if (hl != 0) return;
    D.ap[i] = make_float4(acc[0], acc[1], acc[2], 0.f);
    D.ap2[i] = make_float4(acc[3], acc[4], acc[5], 0.f);
}

// First Jacobi iteration from the per-particle better of the two starts: the
// one with the smaller initial residual |s - (A p)_i| is kept and updated as
// in pressureSolveIteration / divergenceSolveIteration.
template <bool PRESSURE, int LPP>
__global__ __launch_bounds__(BLOCK) void k_jacobi2(Dev D) {
    __shared__ double lds[BLOCK / 64];
    __shared__ float plds[PAIR_LDS<LPP, 2>];
    float *const T = pair_part<LPP, 2>(plds);
    Ctl *C = D.ctl;
    const unsigned t = gtid();
    const unsigned i = t / LPP, hl = t % LPP;
    const double h = C->h;
    double err = 0.0, over = 0.0;
    bool took = false;
    // the lanes of a particle take this branch together
    if (i < D.n && (!PRESSURE || is_active(D, i))) {
        const float4 xi = D.x[i], ai = D.ap[i], bi = D.ap2[i];
        float s[2] = {0.f, 0.f};
        const unsigned cnt = D.cf[i], cb = D.bmode == 1 ? D.cb[i] : 0u;
        const F4Gather X(D.x, D.n), A(D.ap, D.n), A2(D.ap2, D.n);
        fluid_sums<LPP, SumAdd<2>>(
            D, i, hl, cnt, T, s,
            loads([&](unsigned j) { return X.xyz(j); }, [&](unsigned j) { return A.xyz(j); },
                  [&](unsigned j) { return A2.xyz(j); }),
            [&](unsigned, const auto &q, float *u) {
                float3 r;
                const float g = kernel_G(xi, q.a, D.K, r);
                const float gx = g * r.x, gy = g * r.y, gz = g * r.z;
                u[0] = ((ai.x - q.b.x) * gx + (ai.y - q.b.y) * gy) + (ai.z - q.b.z) * gz;
                u[1] = ((bi.x - q.c.x) * gx + (bi.y - q.c.y) * gy) + (bi.z - q.c.z) * gz;
                return true;
            });
        s[0] *= D.V;
        s[1] *= D.V;
        const unsigned nnb = cnt + cb;
        auto bterm = [&](const float4 &xb, float *u) {
            float3 r;
            const float g = kernel_G(xi, xb, D.K, r);
            const float gx = g * r.x, gy = g * r.y, gz = g * r.z;
            u[0] = xb.w * ((ai.x * gx + ai.y * gy) + ai.z * gz);
            u[1] = xb.w * ((bi.x * gx + bi.y * gy) + bi.z * gz);
            return true;
        };
        if (D.bmode == 1) {
            akinci_sums<LPP, SumAdd<2>>(D, i, hl, cb, T, s, bterm);
        } else if (D.bmode == 2 && hl == 0) {
            for (unsigned o = 0; o < D.nvm; o++) {
                const float4 xb = D.vmb[(size_t)o * D.stride + i];
                if (!(xb.w > 0.f)) break;
                float u[2];
                bterm(xb, u);
                sum_terms<SumAdd<2>>(u, s);
            }
        } else if (D.bmode == 3 && hl == 0) {
            for (unsigned o = 0; o < D.nvm; o++) {
                if (!(D.vmb[(size_t)o * D.stride + i].w > 0.f)) break;
                const float4 gb = D.dmg[(size_t)o * D.stride + i];
                s[0] -= (ai.x * gb.x + ai.y * gb.y) + ai.z * gb.z;
                s[1] -= (bi.x * gb.x + bi.y * gb.y) + bi.z * gb.z;
            }
        }
        if (hl == 0) {
            const float sc = PRESSURE ? (float)(h * h) : (float)h;
            const float si = PRESSURE ? 1.0f - D.radv[i] : -D.radv[i];
            const float r1 = si - s[0] * sc, r2 = si - s[1] * sc;
            took = fabsf(r2) < fabsf(r1);
            const float start = took ? D.pred[i] : (PRESSURE ? D.p[i] : D.pv[i]);
            const float rr = took ? r2 : r1;
            float res = fminf(rr, 0.0f);
            if (!PRESSURE && nnb < 20u) res = 0.0f;
            const float pn = fmaxf(start - 0.5f * rr * D.alpha[i], 0.0f);
            if (PRESSURE)
                D.p[i] = pn;
            else
                D.pv[i] = pn;
            reinterpret_cast<float *>(D.x + i)[3] = pn;
            err = -(double)D.rho0 * (double)res;
            if (pn > 0.0f && rr > 0.0f && (PRESSURE || nnb >= 20u)) over = (double)D.rho0 * (double)rr;
        }
    }
    const double bs = block_sum(err, lds);
    const double bo = block_sum(over, lds);
    const double bl = block_sum(took ? 1.0 : 0.0, lds);
    if (threadIdx.x == 0) {
        D.partial[2 * blockIdx.x] = bs;
        D.partial[2 * blockIdx.x + 1] = bo;
        D.partial[2 * gridDim.x + blockIdx.x] = bl;  // particles that kept the network's start
    }
}

// Training samples: features of every stride-th particle and its converged
// stiffness (the stored p h^2 or p_v h) relative to the step's scale.
template <bool PRESSURE>
__global__ __launch_bounds__(BLOCK) void k_collect(Dev D) {
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    Ctl *C = D.ctl;
    const unsigned stride = PRESSURE ? D.sstride : D.sstride_v;
    const double kref = PRESSURE ? C->kref : C->kref_v;
    const bool take = (i < D.n) && stride && (i % stride) == (D.soff % stride) && kref > 0.0;
    const unsigned long long m = __ballot(take);
    if (!m) return;
    const unsigned lane = threadIdx.x & 63u;
    unsigned base = 0;
    if (lane == (unsigned)__ffsll((long long)m) - 1u)
        base = atomicAdd(PRESSURE ? &C->nsamp : &C->nsamp_v, (unsigned)__popcll(m));
    base = __shfl(base, __ffsll((long long)m) - 1, 64);
    if (!take) return;
    const unsigned slot = base + (unsigned)__popcll(m & ((1ull << lane) - 1ull));
    const unsigned cap = PRESSURE ? D.scap : D.scap_v;
    if (slot >= cap) return;
    const float *F = (PRESSURE ? D.feats : D.feats_v) + (size_t)i * 8;
    float *X = (PRESSURE ? D.sx : D.sx_v) + (size_t)slot * 8;
    reinterpret_cast<float4 *>(X)[0] = reinterpret_cast<const float4 *>(F)[0];
    reinterpret_cast<float4 *>(X)[1] = reinterpret_cast<const float4 *>(F)[1];
    const float kf = PRESSURE ? D.p[i] : D.pv[i];
    (PRESSURE ? D.st : D.st_v)[slot] = (float)(kf / kref);
}

// ==================================================================== host
DFSPH::DFSPH(const sph_dfsph_params_t &p) : P(p) {
    require_device();
    static std::atomic<unsigned long long> next_serial{1};
    serial_ = next_serial.fetch_add(1);
    SPH_REQUIRE(P.particle_radius > 0 && P.density0 > 0, SPH_ERR_INVALID, "particle_radius and density0 must be > 0");
    SPH_REQUIRE(P.viscosity_method == SPH_VISCOSITY_NONE || P.viscosity_method == SPH_VISCOSITY_STANDARD ||
                    P.viscosity_method == SPH_VISCOSITY_WEILER2018,
                SPH_ERR_INVALID, "viscosity_method: only none (0), standard (1) and Weiler2018 (6) are implemented");
    SPH_REQUIRE(P.boundary_handling_method == SPH_BOUNDARY_NONE || P.boundary_handling_method == SPH_BOUNDARY_AKINCI2012 ||
                    P.boundary_handling_method == SPH_BOUNDARY_KOSCHIER2017 ||
                    P.boundary_handling_method == SPH_BOUNDARY_BENDER2019,
                SPH_ERR_INVALID,
                "boundary_handling_method: only none (-1), Akinci2012 (0), Koschier2017 (1) and Bender2019 (2)");
    r = P.particle_radius;
    hs = 4.0 * r;
    const double diam = 2.0 * r;
    V = 0.8 * diam * diam * diam;
    mass = V * P.density0;
    K = make_kernel_const(hs);
    pci_factor_ = pcisph_factor(r, V);
    SPH_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    SPH_HIP(hipHostMalloc((void **)&hctl_, sizeof(Ctl), hipHostMallocDefault));
    std::memset(hctl_, 0, sizeof(Ctl));
    hctl_->h = P.time_step_size;
    hctl_->h_step = P.time_step_size;
    ctl_.reserve(1);
    SPH_HIP(hipMemcpyAsync(ctl_.get(), hctl_, sizeof(Ctl), hipMemcpyHostToDevice, stream));
    SPH_HIP(hipStreamSynchronize(stream));
}

DFSPH::~DFSPH() {
    if (stream) (void)hipStreamSynchronize(stream);
    if (hctl_) (void)hipHostFree(hctl_);
    if (stream) (void)hipStreamDestroy(stream);
}

void DFSPH::set_fluid(const float *x, const float *v, size_t n) {
    SPH_REQUIRE(n < (size_t)0x7fffffff, SPH_ERR_INVALID, "too many particles");
    hx_.assign(x, x + 3 * n);
    if (v)
        hv_.assign(v, v + 3 * n);
    else
        hv_.assign(3 * n, 0.f);
    n_ = n;
    initialized_ = false;
}

void DFSPH::add_boundary(const float *x, size_t n) {
    hbx_.insert(hbx_.end(), x, x + 3 * n);
    nb_ += n;
    initialized_ = false;
}

void DFSPH::set_volume_map_box(const double lo[3], const double hi[3], int invert, double thickness,
                               const unsigned res[3]) {
    Shape sh;
    sh.kind = SHAPE_BOX;
    for (int c = 0; c < 3; c++) {
        sh.box_lo[c] = lo[c];
        sh.box_hi[c] = hi[c];
    }
    sh.invert = invert;
    sh.thickness = thickness;
    add_volume_map(sh, res);
}

void DFSPH::add_volume_map_mesh(const double *vertices, size_t nv, const unsigned *faces, size_t nf, int invert,
                                double thickness, const unsigned res[3]) {
    SPH_REQUIRE(vertices && faces && nv >= 4 && nf >= 4, SPH_ERR_INVALID, "volume map: a closed mesh needs faces");
    Shape sh;
    sh.kind = SHAPE_MESH;
    for (int c = 0; c < 3; c++) {
        sh.box_lo[c] = 1e300;
        sh.box_hi[c] = -1e300;
    }
    for (size_t v = 0; v < nv; v++)
        for (int c = 0; c < 3; c++) {
            sh.box_lo[c] = std::min(sh.box_lo[c], vertices[3 * v + c]);
            sh.box_hi[c] = std::max(sh.box_hi[c], vertices[3 * v + c]);
        }
    sh.tri.reserve(9 * nf);
    for (size_t f = 0; f < 3 * nf; f++) {
        SPH_REQUIRE(faces[f] < nv, SPH_ERR_INVALID, "volume map: face index out of range");
        for (int c = 0; c < 3; c++) sh.tri.push_back(vertices[3 * (size_t)faces[f] + c]);
    }
    sh.invert = invert;
    sh.thickness = thickness;
    add_volume_map(sh, res);
}

void DFSPH::add_volume_map(const Shape &shape, const unsigned res[3]) {
    SPH_REQUIRE(res[0] > 0 && res[1] > 0 && res[2] > 0, SPH_ERR_INVALID, "volume map: resolution must be > 0");
    SPH_REQUIRE(vm_shapes_.size() < 64, SPH_ERR_INVALID, "volume map: at most 64 objects");
    vm_shapes_.push_back(shape);
    vm_res_.push_back({res[0], res[1], res[2]});
    initialized_ = false;
}

Dev DFSPH::dev() const {
    Dev D{};
    D.n = (unsigned)n_;
    D.stride = stride_;
    D.x = x_.get();
    D.v = v_.get();
    D.v2 = v2_.get();
    D.a = a_.get();
    D.ap = ap_.get();
    D.vdiff = vdiff_.get();
    D.xc = xc_.get();
    D.vmb = vmb_.get();
    D.state = states_ ? pst_.get() : nullptr;
    D.nvm = nvm_;
    D.rho = rho_.get();
    D.alpha = alpha_.get();
    D.radv = radv_.get();
    D.p = p_.get();
    D.pv = pv_.get();
    D.nf = nf_.get();
    D.nf16 = use16_ ? nf16_.get() : nullptr;
    const bool tiled = tiled_ && lists_n_ == n_;
    D.nt16 = tiled ? nt16_.get() : nullptr;
    D.tslot = tiled ? tslot_.get() : nullptr;
    D.tcount = tiled ? tcount_.get() : nullptr;
    D.quads16 = (capF_ + 7) / 8;
    D.cf = cf_.get();
    D.nb = nb_l_.get();
    D.cb = cb_.get();
    D.bx = bx_.get();
    const int bm = P.boundary_handling_method;
    D.bmode = (bm == SPH_BOUNDARY_AKINCI2012 && nb_ > 0)       ? 1
              : (bm == SPH_BOUNDARY_BENDER2019 && nvm_ > 0)   ? 2
              : (bm == SPH_BOUNDARY_KOSCHIER2017 && nvm_ > 0) ? 3
                                                              : 0;
    D.dmg = dmg_.get();
    D.vmv = (moving_ && D.bmode == 2) ? vmv_.get() : nullptr;
    D.body = body_.get();
    D.nbody = (moving_ && D.bmode == 2) ? nvm_ : 0u;
    D.bodyMaxVel = (D.bmode == 2) ? body_max_vel_ : 0.0;
    D.bpart = bpart_.get();
    D.bforce = bforce_.get();
    D.sphereVol = (float)(4.0 / 3.0 * 3.14159265358979323846 * hs * hs * hs);
    D.V = (float)V;
    D.rho0 = (float)P.density0;
    D.eps = 1.0e-5f;
    D.mass = (float)mass;
    D.grav = make_float3((float)P.gravity[0], (float)P.gravity[1], (float)P.gravity[2]);
    D.K = K;
    D.ctl = ctl_.get();
    D.partial = partial_.get();
    D.minIt = P.min_iterations;
    D.maxIt = P.max_iterations;
    D.maxItV = P.max_iterations_v;
    D.maxError = P.max_error;
    D.maxErrorV = P.max_error_v;
    D.xsph = (float)P.xsph;
    D.xsphB = (float)P.xsph_boundary;
    const bool stdv = P.viscosity_method == SPH_VISCOSITY_STANDARD;
    D.svisc = stdv ? (float)(10.0 * P.viscosity) : 0.f;
    D.sviscB = stdv ? (float)(10.0 * P.viscosity_boundary) : 0.f;
    D.model = models_ ? model_.get() : nullptr;
    D.solveModel = -1;
    D.nmodel = models_ ? (unsigned)materials_.size() : 1u;
    for (unsigned m = 0; m < 8; m++) {
        const bool ok = models_ && m < materials_.size();
        const double r0 = ok ? materials_[m][0] : P.density0;
        D.rho0m[m] = (float)r0;
        D.massm[m] = (float)(V * r0);
        D.svm[m] = (ok && stdv) ? (float)(10.0 * materials_[m][1]) : 0.f;
        D.svbm[m] = (ok && stdv) ? (float)(10.0 * materials_[m][2]) : 0.f;
        D.xsm[m] = ok ? (float)materials_[m][3] : 0.f;
        D.xsbm[m] = ok ? (float)materials_[m][4] : 0.f;
        D.countm[m] = (ok && m < model_count_.size()) ? model_count_[m] : 0u;
        if (ok) {  // the kernels' gates: on when any model uses the term
            D.svisc = std::max(D.svisc, D.svm[m]);
            D.sviscB = std::max(D.sviscB, D.svbm[m]);
            D.xsph = std::max(D.xsph, D.xsm[m]);
            D.xsphB = std::max(D.xsphB, D.xsbm[m]);
        }
    }
    D.cflMethod = P.cfl_method;
    D.cflFactor = P.cfl_factor;
    D.cflMin = P.cfl_min_time_step_size;
    D.cflMax = P.cfl_max_time_step_size;
    D.radius = r;
    D.minv = minv_.get();
    D.cgx = cgx_.get();
    D.cgr = cgr_.get();
    D.cgp = cgp_.get();
    D.cgz = cgz_.get();
    D.cgt = cgt_.get();
    D.mu = (float)(P.viscosity * P.density0);
    D.mub = (float)(P.viscosity_boundary * P.density0);
    D.hs2 = (float)(hs * hs);
    D.viscoMaxIt = P.visco_max_iter;
    D.viscoTol = P.visco_max_error;
    D.strictP = engaged_[0] ? 1 : 0;
    D.strictV = engaged_[1] ? 1 : 0;
    D.feats = feats_[0].get();
    D.feats_v = feats_[1].get();
    D.pred = pred_.get();
    D.kprev = nullptr;  // set per solve by the callers that save it
    D.ap2 = ap2_.get();
    D.sx = sx_[0].get();
    D.st = st_[0].get();
    D.sx_v = sx_[1].get();
    D.st_v = st_[1].get();
    D.scap = (unsigned)cap_s_[0];
    D.scap_v = (unsigned)cap_s_[1];
    D.sstride = stride_s_[0];
    D.sstride_v = stride_s_[1];
    D.soff = soff_;
    return D;
}

void DFSPH::read_ctl() {
    syncs_++;
    SPH_HIP(hipMemcpyAsync(hctl_, ctl_.get(), sizeof(Ctl), hipMemcpyDeviceToHost, stream));
    SPH_HIP(hipStreamSynchronize(stream));
}

void DFSPH::upload_ctl_field(size_t off, const void *src, size_t bytes) {
    SPH_HIP(hipStreamSynchronize(stream));
    std::memcpy(reinterpret_cast<char *>(hctl_) + off, src, bytes);
    SPH_HIP(hipMemcpyAsync(reinterpret_cast<char *>(ctl_.get()) + off, reinterpret_cast<char *>(hctl_) + off, bytes,
                           hipMemcpyHostToDevice, stream));
    SPH_HIP(hipStreamSynchronize(stream));
}

// Per-particle device buffers for stride_ slots (contents not preserved).
void DFSPH::alloc_particles() {
    const size_t S = stride_;
    no_tile_room_ = false;
    SPH_REQUIRE(S <= GATHER_MAX, SPH_ERR_RANGE, "at most 2^28 particle slots per time step");
    for (DBuf<float4> *b : {&x_, &v_, &v2_, &a_, &ap_, &vdiff_, &xc_, &x2_, &vdiff2_, &xc2_}) b->reserve(S);
    const size_t nobj = maps() ? vm_shapes_.size() : 0;
    vmb_.reserve(std::max<size_t>(nobj, 1) * S);
    if (nobj > 1) vmraw_.reserve(nobj * S);
    if (moving_) {
        vmv_.reserve(std::max<size_t>(nobj, 1) * S);
        if (nobj > 1) vmvraw_.reserve(nobj * S);
    }
    if (P.boundary_handling_method == SPH_BOUNDARY_KOSCHIER2017) {
        dmg_.reserve(std::max<size_t>(nobj, 1) * S);
        if (nobj > 1) dmgraw_.reserve(nobj * S);
    }
    for (DBuf<float> *b : {&rho_, &alpha_, &radv_, &p_, &pv_, &p2_, &pv2_}) b->reserve(S);
    id_.reserve(S);
    id2_.reserve(S);
    if (states_) {
        pst_.reserve(S);
        pst2_.reserve(S);
    }
    if (method_ == SPH_METHOD_PCISPH) {
        predx_.reserve(S);
        predx2_.reserve(S);
    }
    cf_.reserve(S);
    cb_.reserve(S);
    // up to three values per block of the sweeps, which have up to 4 lanes
    // per particle, 16 for small counts (small_lanes)
    partial_.reserve(std::max(12 * (size_t)nblocks(S), 48 * (size_t)nblocks(SMALL_PARTICLES)) + 64);
    if (initialized_ && (mode_[0] || mode_[1] || stride_s_[0] || stride_s_[1])) ensure_learn_buffers();
    if (P.viscosity_method == SPH_VISCOSITY_WEILER2018) {
        minv_.reserve(2 * S);
        for (DBuf<float4> *b : {&cgx_, &cgr_, &cgp_, &cgz_, &cgt_}) b->reserve(S);
    }
}

// Uploads n particles in id order (ids 0..n-1): positions and velocities
// (3 floats each) and the persistent per-particle state (null: zero); the
// other fields start at zero.
void DFSPH::upload_particles(size_t n, const float *x, const float *v, const float4 *xc, const float4 *vdiff,
                             const float *p, const float *pv) {
    const size_t S = stride_;
    const size_t nobj = maps() ? vm_shapes_.size() : 0;
    std::vector<float4> hx(n), hv(n), zero(n, make_float4(0.f, 0.f, 0.f, 0.f));
    std::vector<unsigned> ids(n);
    for (size_t i = 0; i < n; i++) {
        hx[i] = make_float4(x[3 * i], x[3 * i + 1], x[3 * i + 2], 0.f);
        hv[i] = make_float4(v[3 * i], v[3 * i + 1], v[3 * i + 2], 0.f);
        ids[i] = (unsigned)i;
    }
    std::vector<float> zf(n, 0.f);
    SPH_HIP(hipStreamSynchronize(stream));
    SPH_HIP(hipMemcpy(x_.get(), hx.data(), n * sizeof(float4), hipMemcpyHostToDevice));
    SPH_HIP(hipMemcpy(v_.get(), hv.data(), n * sizeof(float4), hipMemcpyHostToDevice));
    for (DBuf<float4> *b : {&a_, &ap_})
        SPH_HIP(hipMemcpy(b->get(), zero.data(), n * sizeof(float4), hipMemcpyHostToDevice));
    SPH_HIP(hipMemcpy(vdiff_.get(), vdiff ? vdiff : zero.data(), n * sizeof(float4), hipMemcpyHostToDevice));
    SPH_HIP(hipMemcpy(xc_.get(), xc ? xc : zero.data(), n * sizeof(float4), hipMemcpyHostToDevice));
    for (size_t o = 0; o < std::max<size_t>(nobj, 1); o++) {
        SPH_HIP(hipMemcpy(vmb_.get() + o * S, zero.data(), n * sizeof(float4), hipMemcpyHostToDevice));
        if (dmg_.get()) SPH_HIP(hipMemcpy(dmg_.get() + o * S, zero.data(), n * sizeof(float4), hipMemcpyHostToDevice));
    }
    for (DBuf<float> *b : {&rho_, &alpha_, &radv_})
        SPH_HIP(hipMemcpy(b->get(), zf.data(), n * sizeof(float), hipMemcpyHostToDevice));
    SPH_HIP(hipMemcpy(p_.get(), p ? p : zf.data(), n * sizeof(float), hipMemcpyHostToDevice));
    SPH_HIP(hipMemcpy(pv_.get(), pv ? pv : zf.data(), n * sizeof(float), hipMemcpyHostToDevice));
    SPH_HIP(hipMemcpy(id_.get(), ids.data(), n * sizeof(unsigned), hipMemcpyHostToDevice));
    if (states_) {
        const std::vector<unsigned> active(n, 0u);
        SPH_HIP(hipMemcpy(pst_.get(), active.data(), n * sizeof(unsigned), hipMemcpyHostToDevice));
    }
    // PCISPH's predicted positions start at zero (SimulationDataPCISPH::init)
    if (method_ == SPH_METHOD_PCISPH)
        SPH_HIP(hipMemcpy(predx_.get(), zero.data(), n * sizeof(float4), hipMemcpyHostToDevice));
}

void DFSPH::init() {
    SPH_REQUIRE(n_ > 0, SPH_ERR_STATE, "set_fluid must be called first");
    const size_t n = n_;
    // room for the emitters' particles up front (the reference's capacity
    // numParticles = initial + maxEmitterParticles, FluidModel::initModel)
    cap_emit_ = n + max_emit_;
    stride_ = (unsigned)(((emitters_.empty() ? n : cap_emit_) + 255) / 256 * 256);
    const size_t S = stride_;
    const size_t nobj = maps() ? vm_shapes_.size() : 0;
    alloc_particles();
    upload_particles(n, hx_.data(), hv_.data(), nullptr, nullptr, nullptr, nullptr);
    // grid over fluid, boundary particles and the volume-map box
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    auto ext = [&](const std::vector<float> &a) {
        for (size_t i = 0; i + 2 < a.size(); i += 3)
            for (int c = 0; c < 3; c++) {
                lo[c] = std::min(lo[c], (double)a[i + c]);
                hi[c] = std::max(hi[c], (double)a[i + c]);
            }
    };
    ext(hx_);
    ext(hbx_);
    for (const Shape &sh : vm_shapes_)
        for (int c = 0; c < 3; c++) {
            const bool sp = sh.kind == SHAPE_SPHERE;
            lo[c] = std::min(lo[c], sp ? sh.centre[c] - sh.radius : sh.box_lo[c]);
            hi[c] = std::max(hi[c], sp ? sh.centre[c] + sh.radius : sh.box_hi[c]);
        }
    for (const EmitterDesc &e : emitters_) {
        double size[3];
        emitter_size(e, size);
        const double L = 0.5 * std::max(size[0], std::max(size[1], size[2])) + hs;
        for (int c = 0; c < 3; c++) {
            lo[c] = std::min(lo[c], e.x[c] - L);
            hi[c] = std::max(hi[c], e.x[c] + L);
        }
    }
    for (int c = 0; c < 3; c++) {
        lo[c] -= 2.0 * hs;
        hi[c] += 2.0 * hs;
    }
    // x sub-cells of a quarter edge: each query trims its rows to the reach
    // of its own position, about half the candidates of whole cells
    grid_ = make_grid(lo, hi, hs, (size_t)1 << 27, 4);
    // Akinci boundary: sort once, volumes from boundary-boundary neighbours
    if (nb_ > 0) {
        const size_t nbp = nb_;
        const unsigned bstride = (unsigned)((nbp + 255) / 256 * 256);
        DBuf<float4> tmp;
        tmp.reserve(nbp);
        std::vector<float4> hb(nbp);
        for (size_t i = 0; i < nbp; i++) hb[i] = make_float4(hbx_[3 * i], hbx_[3 * i + 1], hbx_[3 * i + 2], 0.f);
        SPH_HIP(hipMemcpy(tmp.get(), hb.data(), nbp * sizeof(float4), hipMemcpyHostToDevice));
        bsort_.sort(stream, tmp.get(), (unsigned)nbp, grid_, timer);
        bx_.reserve(nbp);
        permute_f4(stream, bsort_.perm.get(), (unsigned)nbp, tmp.get(), bx_.get());
        bperm_.reserve(nbp);
        SPH_HIP(hipMemcpyAsync(bperm_.get(), bsort_.perm.get(), nbp * sizeof(unsigned), hipMemcpyDeviceToDevice,
                               stream));
        bstart_.reserve((size_t)grid_.ncells + 1);
        SPH_HIP(hipMemcpyAsync(bstart_.get(), bsort_.start.get(), ((size_t)grid_.ncells + 1) * sizeof(unsigned),
                               hipMemcpyDeviceToDevice, stream));
        unsigned cap = 64;
        DBuf<unsigned> bl, bc;
        bc.reserve(bstride);
        for (;;) {
            bl.reserve((size_t)cap * bstride);
            k_reset<<<1, 1, 0, stream>>>(ctl_.get(), 2);
            build_lists_colmajor(stream, bx_.get(), (unsigned)nbp, bx_.get(), bstart_.get(), grid_, hs, true,
                                 bl.get(), bstride, cap, bc.get(), &ctl_.get()->maxcnt_f, timer, "boundary_lists");
            read_ctl();
            if (hctl_->maxcnt_f <= cap) break;
            cap = (hctl_->maxcnt_f + 15) / 16 * 16;
        }
        k_boundary_volume<<<nblocks(nbp), BLOCK, 0, stream>>>(bx_.get(), (unsigned)nbp, bl.get(), bc.get(), bstride,
                                                              K);
        SPH_HIP(hipGetLastError());
        SPH_HIP(hipStreamSynchronize(stream));
    }
    vmaps.clear();
    for (size_t o = 0; o < nobj; o++) {
        vmaps.emplace_back(new VolumeMap());
        vmaps.back()->build(stream, vm_shapes_[o], vm_res_[o].data(), hs,
                            P.boundary_handling_method == SPH_BOUNDARY_KOSCHIER2017);
        vmaps.back()->d.obj = (unsigned)o;
    }
    nvm_ = (unsigned)nobj;
    apply_motion();
    initialized_ = true;
    if (mode_[0] || mode_[1] || stride_s_[0] || stride_s_[1]) ensure_learn_buffers();
    have_lists_ = false;
    (void)S;
}

// TimeStepDFSPH::reset (TimeStepDFSPH.cpp:710-716) with
// SimulationDataDFSPH::reset (SimulationDataDFSPH.cpp:64-81): the solver's
// per-particle fields and iteration counters return to zero; positions,
// velocities and the viscosity warm start (Viscosity_Weiler2018::reset
// keeps vDiff) are unchanged.
void DFSPH::reset() {
    itLast_ = itVLast_ = cgLast_ = 0;
    lastIt_ = 2;
    lastItV_ = 1;
    lastCg_ = 4;
    totIt_ = totItV_ = totVisco_ = 0;
    steps_ = 0;
    capped_ = cappedV_ = 0;
    learnedSolves_ = learnedSolvesV_ = 0;
    engaged_[0] = engaged_[1] = false;
    // EmitterSystem::reset (EmitterSystem.cpp:82-91)
    emitted_ = reused_ = 0;
    for (EmitterDesc &e : emitters_) {
        e.next = e.start;
        e.counter = 0;
    }
    if (!initialized_) return;
    const size_t n = n_;
    for (DBuf<float> *b : {&alpha_, &radv_, &p_, &pv_})
        SPH_HIP(hipMemsetAsync(b->get(), 0, n * sizeof(float), stream));
    SPH_HIP(hipMemsetAsync(ap_.get(), 0, n * sizeof(float4), stream));
    for (int which : {0, 1, 3}) k_reset<<<1, 1, 0, stream>>>(ctl_.get(), which);
    SPH_HIP(hipGetLastError());
    SPH_HIP(hipStreamSynchronize(stream));
}

void DFSPH::build_lists() {
    const Dev D = dev();
    for (;;) {
        nf_.reserve((size_t)capF_ * stride_);
        nf16_.reserve((size_t)((capF_ + 1) / 2) * stride_);
        if (D.bmode == 1) nb_l_.reserve((size_t)capB_ * stride_);
        build_lists_colmajor(stream, x_.get(), (unsigned)n_, x_.get(), fsort_.start.get(), grid_, hs, true,
                             nf_.get(), stride_, capF_, cf_.get(), &ctl_.get()->maxcnt_f, timer, "fluid_lists",
                             nf16_.get(), &ctl_.get()->ovf16);
        if (P.boundary_handling_method == SPH_BOUNDARY_AKINCI2012 && nb_ > 0)
            build_lists_colmajor(stream, x_.get(), (unsigned)n_, bx_.get(), bstart_.get(), grid_, hs, false,
                                 nb_l_.get(), stride_, capB_, cb_.get(), &ctl_.get()->maxcnt_b, timer,
                                 "boundary_lists");
        read_ctl();
        bool again = false;
        if (hctl_->maxcnt_f > capF_) {
            capF_ = (hctl_->maxcnt_f + 16) / 16 * 16;
            again = true;
        }
        if (hctl_->maxcnt_b > capB_) {
            capB_ = (hctl_->maxcnt_b + 16) / 16 * 16;
            again = true;
        }
        if (!again) break;
        k_reset<<<1, 1, 0, stream>>>(ctl_.get(), 2);
    }
    use16_ = hctl_->ovf16 == 0u;
    lists_max_ = hctl_->maxcnt_f;
    tiled_ = tiles_known_ = false;
    list_its_ = 0;
    // how many tiles were overfull counts for the next 16 lists
    if (tiles_over_ && ++tiles_wait_ > 16) tiles_over_ = 0;
    lists_n_ = n_;
    have_lists_ = true;
}

// Whether tiles gain more in the iterations on these lists than they cost.
// At n particles the two tiled sweeps of an iteration save about 35 ps n -
// 2.5 us and the tiles take 27 us + 60 ps n (measured / formula, us, 1 or 2
// lanes: 111k saved 2.0-3.4 / 1.4, built 33 / 34; 176k 3.4-6.6 / 3.6, 35 /
// 38; 262k 6.0-8.7 / 6.7, 38 / 43; 593k 15-20 / 18, 59 / 63; 1M 31-34 / 33,
// 85 / 87; 2M 56-77 / 68, 158 / 147): they pay from 3 iterations on at 1M, 10
// at 176k, 25 at 111k. Expected are the iterations of the last solves, or half
// as many again as the lists have already seen (a solve that ends near the
// last one's count is not worth tiles at its end). An overfull tile is taken to
// lose what another saves: its blocks gather beside LDS that they do not use
// (62-64 % of the tiles overfull, us an iteration gathered / tiled: 133k 57 /
// 63, 293k 94 / 98, 547k 159 / 150). Four lanes read tiles no faster than
// memory (1M: 124 us an iteration, 126 gathered), and below SMALL_PARTICLES
// the 16 ordered lanes hide the latency that staging would add.
bool DFSPH::tiles_pay() const {
    const double n = (double)n_, its = std::max(lastIt_ + (P.enable_divergence_solver ? lastItV_ : 0), list_its_ / 2);
    const double fit = 1.0 - 2.0 * tiles_over_ * TILE / n;
    return its * fit * (0.035 * n - 2500.0) >= 27000.0 + 0.06 * n;  // ns
}

// The lists of the iterations' sweeps (single-model scenes whose lists are
// packed), built when an iteration asks for them and they pay: a search, a
// density or a batched solve has no use for them.
void DFSPH::build_tiles() {
    if (tiles_known_) return;
    const bool can = have_lists_ && lists_n_ == n_ && use16_ && !models_ && method_ == SPH_METHOD_DFSPH &&
                     n_ >= SMALL_PARTICLES && lpp_ <= 2 && lppA_ <= 2 && !no_tile_room_;
    if (can && !tiles_pay()) return;
    tiles_known_ = true;
    if (!can) return;
    const unsigned nt = ((unsigned)n_ + TILE - 1) / TILE;
    try {
        nt16_.reserve(4 * (size_t)((capF_ + 7) / 8) * stride_);
        tslot_.reserve((size_t)nt * (TILE_CAP / 2));
        tcount_.reserve(nt);
    } catch (const Error &e) {
        if (e.code != SPH_ERR_OOM) throw;
        // the sweeps gather, until the particles' buffers change size
        (void)hipGetLastError();
        nt16_.release();
        tslot_.release();
        tcount_.release();
        no_tile_room_ = true;
        return;
    }
    tiled_ = true;
    tiles_wait_ = 0;
    TimedScope ts(timer, stream, "tile_lists");
    k_tile_lists<<<nt, TILE, 0, stream>>>(dev(), reinterpret_cast<uint4 *>(nt16_.get()), tslot_.get(), tcount_.get());
    SPH_HIP(hipGetLastError());
}

// Lanes per particle of a small count. The two give the same sums
// bit for bit, so the rule only weighs time: shared pairs hide the memory
// latency of a nearly idle GPU and cost three times the instructions.
// Whole steps (us), one lane / shared, Akinci walls and plain start: 2,197
// particles 550 / 407, 12,167 particles 895 / 687, 32,768 particles 1307 /
// 1203, 50,653 particles 1335 / 1425. Eight scenes of 20k-80k particles
// stepped together (24.4 / 28.0 ms for six steps) fill the GPU with one lane
// each, so a scene counts with those it is stepped with.
constexpr size_t ORDERED_MAX = 40960;
static int small_lanes(size_t n) { return n <= ORDERED_MAX ? ORDERED_LANES : 1; }

void DFSPH::neighborhood_search() {
    if (!initialized_) init();
    if (!lpp_fixed_ && !picked_large_) lpp_ = lppA_ = small_lanes(std::max(n_, company_));
    const unsigned n = (unsigned)n_;
    fsort_.sort(stream, x_.get(), n, grid_, timer);
    {
        TimedScope ts(timer, stream, "permute");
        const unsigned *perm = fsort_.perm.get();
        const FluidArrays src{x_.get(), v_.get(), xc_.get(), vdiff_.get(), p_.get(), pv_.get(), id_.get()};
        const FluidArrays dst{x2_.get(), v2_.get(), xc2_.get(), vdiff2_.get(), p2_.get(), pv2_.get(), id2_.get()};
        k_permute_fluid<<<std::max(nblocks(n), 1u), BLOCK, 0, stream>>>(perm, n, src, dst, ctl_.get());
        SPH_HIP(hipGetLastError());
        x_.swap(x2_);
        v_.swap(v2_);
        xc_.swap(xc2_);
        vdiff_.swap(vdiff2_);
        p_.swap(p2_);
        pv_.swap(pv2_);
        id_.swap(id2_);
        if (states_) {
            permute_u1(stream, perm, n, pst_.get(), pst2_.get());
            pst_.swap(pst2_);
        }
        if (models_) {
            permute_u1(stream, perm, n, model_.get(), model2_.get());
            model_.swap(model2_);
            // The first Jacobi sweep of a model reads the other models'
            // accelerations as the last sweep left them (TimeStepDFSPH.cpp:
            // 324-341 with compute_aij_pj, :1370-1420), so they move with
            // their particles (v2_ holds the stale velocities here).
            permute_f4(stream, perm, n, ap_.get(), v2_.get());
            ap_.swap(v2_);
        }
        if (method_ == SPH_METHOD_PCISPH) {
            permute_f4(stream, perm, n, predx_.get(), predx2_.get());
            predx_.swap(predx2_);
        }
    }
    build_lists();
}

// Boundary records of every map object. With `xin` the particles are
// sampled at those positions (PCISPH's predicted positions), `skip` leaves
// particles with a non-zero entry alone and `stop` makes the launches no-ops
// once a solve has converged.
void DFSPH::volume_maps(const float4 *xin, const unsigned *skip, const int *stop) {
    if (!maps() || nvm_ == 0) return;
    const unsigned *st = (states_ && !skip) ? pst_.get() : nullptr;
    if (P.boundary_handling_method == SPH_BOUNDARY_KOSCHIER2017) {
        // TimeStep::computeDensityAndGradient (TimeStep.cpp:349-468), objects
        // in insertion order as for the volume maps
        const double *dt = &ctl_.get()->h;
        if (nvm_ == 1) {
            sample_density_map(stream, vmaps[0]->d, (unsigned)n_, x_.get(), v_.get(), xc_.get(), vmb_.get(),
                               dmg_.get(), dt, hs, r, timer, xin, skip, stop);
            return;
        }
        for (unsigned o = 0; o < nvm_; o++)
            sample_density_map(stream, vmaps[o]->d, (unsigned)n_, x_.get(), v_.get(), xc_.get(),
                               vmraw_.get() + (size_t)o * stride_, dmgraw_.get() + (size_t)o * stride_, dt, hs, r,
                               timer, xin, skip, stop);
        pack_volume_maps(stream, (unsigned)n_, stride_, nvm_, vmraw_.get(), vmb_.get(), timer, dmgraw_.get(),
                         dmg_.get(), stop);
        return;
    }
    // objects in insertion order: a particle projected out of one object is
    // sampled against the next at its new position (TimeStep.cpp:177-222)
    // with moving bodies every record gets the body's velocity at x_b beside it
    if (nvm_ == 1) {
        sample_volume_map(stream, vmaps[0]->d, (unsigned)n_, x_.get(), v_.get(), xc_.get(), vmb_.get(), st, hs, r,
                          timer, xin, skip, stop, moving_ ? vmv_.get() : nullptr);
        return;
    }
    for (unsigned o = 0; o < nvm_; o++)
        sample_volume_map(stream, vmaps[o]->d, (unsigned)n_, x_.get(), v_.get(), xc_.get(),
                          vmraw_.get() + (size_t)o * stride_, st, hs, r, timer, xin, skip, stop,
                          moving_ ? vmvraw_.get() + (size_t)o * stride_ : nullptr);
    pack_volume_maps(stream, (unsigned)n_, stride_, nvm_, vmraw_.get(), vmb_.get(), timer,
                     moving_ ? vmvraw_.get() : nullptr, moving_ ? vmv_.get() : nullptr, stop);
}

#define LAUNCH(name, kern, ...)                                   \
    do {                                                          \
        TimedScope ts_(timer, stream, name);                      \
        kern<<<nblocks(n_), BLOCK, 0, stream>>>(__VA_ARGS__);     \
        SPH_HIP(hipGetLastError());                               \
    } while (0)
// One-block kernels finishing a grid reduction.
#define REDUCE(name, kern, ...)                                   \
    do {                                                          \
        TimedScope ts_(timer, stream, name);                      \
        kern<<<1, RBLOCK, 0, stream>>>(__VA_ARGS__);              \
        SPH_HIP(hipGetLastError());                               \
    } while (0)

// Launch of kernel template K<..., LPP> with `lanes` lanes per particle.
#define LAUNCH_LPP_AS(name, lanes, K, ...)                                         \
    do {                                                                           \
        TimedScope ts_(timer, stream, name);                                       \
        const int l_ = (lanes);                                                    \
        const unsigned nb_ = nblocks((size_t)n_ * l_);                             \
        if (l_ == ORDERED_LANES)                                                   \
            K<__VA_ARGS__, ORDERED_LANES><<<nb_, BLOCK, 0, stream>>>(D);           \
        else if (l_ == 4)                                                          \
            K<__VA_ARGS__, 4><<<nb_, BLOCK, 0, stream>>>(D);                       \
        else if (l_ == 2)                                                          \
            K<__VA_ARGS__, 2><<<nb_, BLOCK, 0, stream>>>(D);                       \
        else                                                                       \
            K<__VA_ARGS__, 1><<<nb_, BLOCK, 0, stream>>>(D);                       \
        SPH_HIP(hipGetLastError());                                                \
    } while (0)
// The same for the sweeps that keep the plain sequential sum at every count.
#define LAUNCH_SEQ(name, K, ...)                                                   \
    do {                                                                           \
        TimedScope ts_(timer, stream, name);                                       \
        const unsigned nb_ = nblocks((size_t)n_ * seq_lanes());                    \
        if (seq_lanes() == ORDERED_LANES)                                          \
            K<__VA_ARGS__, ORDERED_LANES><<<nb_, BLOCK, 0, stream>>>(D);           \
        else                                                                       \
            K<__VA_ARGS__, 1><<<nb_, BLOCK, 0, stream>>>(D);                       \
        SPH_HIP(hipGetLastError());                                                \
    } while (0)
// ... with the handle's lanes per particle.
#define LAUNCH_LPP(name, K, ...) LAUNCH_LPP_AS(name, lpp_, K, __VA_ARGS__)

// Same for kernel templates whose only parameter is LPP.
#define LAUNCH_LPP1(name, K)                                                       \
    do {                                                                           \
        TimedScope ts_(timer, stream, name);                                       \
        const unsigned nb_ = nblocks((size_t)n_ * lpp_);                           \
        if (lpp_ == ORDERED_LANES)                                                 \
            K<ORDERED_LANES><<<nb_, BLOCK, 0, stream>>>(D);                        \
        else if (lpp_ == 4)                                                        \
            K<4><<<nb_, BLOCK, 0, stream>>>(D);                                    \
        else if (lpp_ == 2)                                                        \
            K<2><<<nb_, BLOCK, 0, stream>>>(D);                                    \
        else                                                                       \
            K<1><<<nb_, BLOCK, 0, stream>>>(D);                                    \
        SPH_HIP(hipGetLastError());                                                \
    } while (0)

template <int LPP>
void DFSPH::sweep_init_l(bool dens, bool fact, bool div) {
    Dev D = dev();
    if (div && learn_or_collect(1)) D.kprev = kprev_.get();
    const unsigned nb = nblocks((size_t)n_ * LPP);
    const char *name = (dens && fact && div) ? "density_factor_divsetup"
                       : (dens && fact)      ? "density_factor"
                       : dens                ? "density"
                       : fact                ? "factor"
                                             : "divergence_setup";
    TimedScope ts(timer, stream, name);
    if (dens && fact && div)
        k_sweep_init<true, true, true, LPP><<<nb, BLOCK, 0, stream>>>(D);
    else if (dens && fact)
        k_sweep_init<true, true, false, LPP><<<nb, BLOCK, 0, stream>>>(D);
    else if (dens)
        k_sweep_init<true, false, false, LPP><<<nb, BLOCK, 0, stream>>>(D);
    else if (fact)
        k_sweep_init<false, true, false, LPP><<<nb, BLOCK, 0, stream>>>(D);
    else if (div)
        k_sweep_init<false, false, true, LPP><<<nb, BLOCK, 0, stream>>>(D);
    SPH_HIP(hipGetLastError());
}

void DFSPH::sweep_init(bool dens, bool fact, bool div) {
    if (!picked_ && have_lists_) pick_lanes();
    if (lpp_ == ORDERED_LANES)
        sweep_init_l<ORDERED_LANES>(dens, fact, div);
    else if (lpp_ == 4)
        sweep_init_l<4>(dens, fact, div);
    else if (lpp_ == 2)
        sweep_init_l<2>(dens, fact, div);
    else
        sweep_init_l<1>(dens, fact, div);
}

// Launches the acceleration or Jacobi sweep with `lanes` lanes per particle.
template <bool PRESSURE, bool JACOBI>
static void launch_sweep(int lanes, unsigned n, hipStream_t s, const Dev &D, int check_done) {
    const unsigned nb = nblocks((size_t)n * lanes);
#define SWEEP(L)                                                        \
    if (lanes == L) {                                                   \
        if (JACOBI)                                                     \
            k_jacobi<PRESSURE, L><<<nb, BLOCK, 0, s>>>(D, check_done);  \
        else                                                            \
            k_accel<PRESSURE, L><<<nb, BLOCK, 0, s>>>(D, check_done);   \
    }
    SWEEP(1) SWEEP(2) SWEEP(4) SWEEP(ORDERED_LANES)
#undef SWEEP
    SPH_HIP(hipGetLastError());
}
// The same from tiles where the lists have them.
template <bool PRESSURE, bool JACOBI>
static void launch_iteration_sweep(int lanes, unsigned n, hipStream_t s, const Dev &D, int check_done) {
    const unsigned nb = (n + TILE - 1) / TILE;
#define SWEEP(L)                                                                  \
    if (lanes == L) {                                                             \
        if (JACOBI)                                                               \
            k_jacobi_tile<PRESSURE, L><<<nb, TILE * L, 0, s>>>(D, check_done);    \
        else                                                                      \
            k_accel_tile<PRESSURE, L><<<nb, TILE * L, 0, s>>>(D, check_done);     \
    }
    if (D.nt16 && lanes <= 2) {
        SWEEP(1) SWEEP(2)
        SPH_HIP(hipGetLastError());
    } else {
        launch_sweep<PRESSURE, JACOBI>(lanes, n, s, D, check_done);
    }
#undef SWEEP
}

// One Jacobi iteration: accelerations, then the update (each sweep with its
// own lanes per particle).
template <bool PRESSURE>
void DFSPH::iteration_any(bool force) {
    if (models_) {
        // the models one after the other, each seeing the stiffness the
        // models before it have just updated (TimeStepDFSPH.cpp:324-341)
        Dev D = dev();
        for (int m = 0; m < (int)materials_.size(); m++) {
            D.solveModel = m;
            {
                TimedScope ts(timer, stream, PRESSURE ? "pressure_accel" : "pressure_accel_v");
                launch_sweep<PRESSURE, false>(lppA_, (unsigned)n_, stream, D, force ? 0 : 1);
            }
            {
                TimedScope ts(timer, stream, PRESSURE ? "jacobi" : "jacobi_v");
                launch_sweep<PRESSURE, true>(lpp_, (unsigned)n_, stream, D, force ? 0 : 1);
            }
            REDUCE("jacobi_reduce", k_jacobi_reduce<PRESSURE>, D, nblocks((size_t)n_ * lpp_), force ? 0 : 1);
        }
        return;
    }
    build_tiles();
    list_its_++;
    const Dev D = dev();
    {
        TimedScope ts(timer, stream, PRESSURE ? "pressure_accel" : "pressure_accel_v");
        launch_iteration_sweep<PRESSURE, false>(lppA_, (unsigned)n_, stream, D, force ? 0 : 1);
    }
    {
        TimedScope ts(timer, stream, PRESSURE ? "jacobi" : "jacobi_v");
        launch_iteration_sweep<PRESSURE, true>(lpp_, (unsigned)n_, stream, D, force ? 0 : 1);
    }
    REDUCE("jacobi_reduce", k_jacobi_reduce<PRESSURE>, D, nblocks((size_t)n_ * lpp_), force ? 0 : 1);
}

// One Jacobi iteration of many scenes: three launches in all (see kb_accel).
void launch_batch_iteration(bool pressure, int lanesA, int lanesJ, const Dev *Ds, const uint4 *bmapA, unsigned nbA,
                            const uint4 *bmapJ, unsigned nbJ, unsigned nscenes, hipStream_t s) {
#define KB(K, LN, L, nb, map)                                      \
    if (LN == L) {                                                 \
        if (pressure)                                              \
            K<true, L><<<nb, BLOCK, 0, s>>>(Ds, map, 1);           \
        else                                                       \
            K<false, L><<<nb, BLOCK, 0, s>>>(Ds, map, 1);          \
    }
#define KBL(K, LN, nb, map) \
    KB(K, LN, 1, nb, map) KB(K, LN, 2, nb, map) KB(K, LN, 4, nb, map) KB(K, LN, ORDERED_LANES, nb, map)
    KBL(kb_accel, lanesA, nbA, bmapA)
    KBL(kb_jacobi, lanesJ, nbJ, bmapJ)
    if (pressure)
        kb_jacobi_reduce<true><<<nscenes, RBLOCK, 0, s>>>(Ds, lanesJ, 1);
    else
        kb_jacobi_reduce<false><<<nscenes, RBLOCK, 0, s>>>(Ds, lanesJ, 1);
#undef KBL
#undef KB
    SPH_HIP(hipGetLastError());
}

void launch_batch_done(bool pressure, const Dev *Ds, unsigned nscenes, int *done, hipStream_t s) {
    if (pressure)
        kb_done<true><<<nblocks(nscenes), BLOCK, 0, s>>>(Ds, nscenes, done);
    else
        kb_done<false><<<nblocks(nscenes), BLOCK, 0, s>>>(Ds, nscenes, done);
    SPH_HIP(hipGetLastError());
}

// XSPH acts in some model (the parameters' coefficients, or a fluid
// model's own).
bool DFSPH::any_xsph() const {
    if (P.xsph != 0.0 || P.xsph_boundary != 0.0) return true;
    if (models_)
        for (const auto &m : materials_)
            if (m[3] != 0.0 || m[4] != 0.0) return true;
    return false;
}

bool DFSPH::batchable() const {
    return method_ == SPH_METHOD_DFSPH && mode_[0] == 0 && mode_[1] == 0 && stride_s_[0] == 0 && stride_s_[1] == 0 &&
           !models_;
}

void DFSPH::div_iteration(bool force) { iteration_any<false>(force); }

void DFSPH::pressure_iteration(bool force) { iteration_any<true>(force); }

// The lanes per particle of a large scene (from SMALL_PARTICLES on), by a rule
// on its count and lists at the first sweep, kept until the caller adds
// particles or sets lanes. The lanes fix the order of every FP32 neighbour
// sum, and velocities differ by about a per cent after some tens of steps in
// another order: a choice by timings made results depend on the noise of
// those timings (85k particles: four choices in twelve fresh handles).
// The lines are where the gathering sweeps cross (us at 1 / 2 / 4 lanes,
// collapsing dam in a box, k_accel with every pair active and k_jacobi):
//  - Jacobi and the other sweeps: 4 lanes below 84k particles, 2 above
//    (k_jacobi 69k 16.6 / 14.2 / 13.9, 85k 16.7 / 14.1 / 14.2, 111k 17.5 /
//    17.0 / 17.5, 1M 78.6 / 66.1 / 83.0);
//  - accelerations: 4 below 112k (111k 11.9 / 10.7 / 10.4), 2 below 236k
//    (176k 14.6 / 14.4 / 14.3), above it 1, the fastest with every pair
//    active (in a flow, where many pairs carry no pressure, 2 lanes gain up
//    to 10 %: 1M 42.0 / 37.8 / 43.4), but 2 from 32-bit lists (4M 274 / 241 /
//    270);
//  - long lists (88 or more: dense clouds; fluid at rest has 53 at most) take
//    4 for both (70k points, K = 100: k_jacobi 46.8 / 29.8 / 25.0, 500k 160 /
//    131 / 119).
// The tiled sweeps of the iterations differ less between 1 and 2 lanes (1M:
// k_accel_tile 27.3 / 25.4, k_jacobi_tile 54.4 / 49.7) and keep this order.
void DFSPH::pick_lanes() {
    picked_ = true;
    if (n_ < SMALL_PARTICLES || lpp_fixed_) return;
    picked_large_ = true;
    const bool longl = lists_max_ >= 88u;
    lpp_ = longl || n_ < 84000 ? 4 : 2;
    lppA_ = longl || n_ < 112000 ? 4 : (n_ < 236000 || !use16_ ? 2 : 1);
}

void DFSPH::set_lanes_per_particle(int lpp) {
    SPH_REQUIRE(lpp == 0 || lpp == 1 || lpp == 2 || lpp == 4, SPH_ERR_INVALID, "lanes per particle must be 0, 1, 2 or 4");
    lpp_fixed_ = lpp != 0;
    lpp_ = lpp ? lpp : 1;
    lppA_ = lpp_;
    picked_ = lpp_fixed_;
    picked_large_ = false;
}

void DFSPH::div_finish(bool scale_pv) {
    const Dev D = dev();
    LAUNCH_LPP_AS("divergence_finish", lppA_, k_finish, false);
    if (dynamic_) body_forces_pressure(false);
    if (scale_pv) LAUNCH("scale", k_scale, D, pv_.get(), 1);
}

// ------------------------------------------------------------ moving bodies
void DFSPH::set_body_motion(unsigned o, const double pos[3], const double R[9], const double vel[3],
                            const double omega[3], int kind) {
    SPH_REQUIRE(P.boundary_handling_method == SPH_BOUNDARY_BENDER2019, SPH_ERR_STATE,
                "moving bodies need Bender2019 volume maps");
    SPH_REQUIRE(o < vm_shapes_.size(), SPH_ERR_INVALID, "boundary object out of range");
    SPH_REQUIRE(kind >= 0 && kind <= 2, SPH_ERR_INVALID, "body kind must be 0 (at rest), 1 (animated) or 2 (dynamic)");
    SPH_REQUIRE(method_ == SPH_METHOD_DFSPH, SPH_ERR_STATE, "moving bodies are supported by the DFSPH step only");
    SPH_REQUIRE(!(P.viscosity_method == SPH_VISCOSITY_WEILER2018 && P.viscosity_boundary != 0.0), SPH_ERR_STATE,
                "moving bodies with Weiler2018 boundary viscosity are not supported");
    for (int c = 0; c < 12; c++) SPH_REQUIRE(std::isfinite(c < 3 ? pos[c] : c < 6 ? vel[c - 3] : c < 9 ? omega[c - 6] : 0.0),
                                             SPH_ERR_INVALID, "body motion: non-finite value");
    for (int c = 0; c < 9; c++) SPH_REQUIRE(std::isfinite(R[c]), SPH_ERR_INVALID, "body motion: non-finite rotation");
    motion_.resize(vm_shapes_.size());
    BodyMotion &m = motion_[o];
    m.kind = kind;
    for (int c = 0; c < 3; c++) {
        m.pos[c] = pos[c];
        m.vel[c] = vel[c];
        m.omega[c] = omega[c];
    }
    for (int c = 0; c < 9; c++) m.R[c] = R[c];
    if (initialized_) apply_motion();
}

void DFSPH::apply_motion() {
    const size_t nobj = vmaps.size();
    motion_.resize(vm_shapes_.size());
    bool mov = false, dyn = false;
    double mv = 0.0;
    std::vector<float4> tab(2 * std::max<size_t>(nobj, 1), make_float4(0.f, 0.f, 0.f, 0.f));
    for (size_t o = 0; o < nobj; o++) {
        VMapDesc &d = vmaps[o]->d;
        const BodyMotion &m = motion_[o];
        if (m.kind >= 0) {
            d.moved = 1;
            d.moving = m.kind != 0;
            for (int c = 0; c < 3; c++) {
                d.pos[c] = m.pos[c];
                d.vel[c] = m.vel[c];
                d.omega[c] = m.omega[c];
            }
            for (int c = 0; c < 9; c++) d.R[c] = m.R[c];
        }
        if (d.moving) {
            mov = true;
            // SimulatorBase::updateVMVelocity (SimulatorBase.cpp:1670-1687)
            const double md = vmaps[o]->max_dist;
            const double w[3] = {d.vel[0], d.vel[1] + d.omega[2] * md, d.vel[2] - d.omega[1] * md};
            mv = std::max(mv, std::sqrt((w[0] * w[0] + w[1] * w[1]) + w[2] * w[2]));
        }
        if (m.kind == 2) dyn = true;
        tab[o] = make_float4((float)d.omega[0], (float)d.omega[1], (float)d.omega[2], m.kind == 2 ? 1.f : 0.f);
        tab[nobj + o] = make_float4((float)d.pos[0], (float)d.pos[1], (float)d.pos[2], 0.f);
    }
    body_max_vel_ = mv;
    if (mov && !moving_) {
        moving_ = true;
        if (stride_) {
            vmv_.reserve(std::max<size_t>(nobj, 1) * stride_);
            if (nobj > 1) vmvraw_.reserve(nobj * stride_);
        }
    }
    dynamic_ = dyn;
    if (nobj) {
        body_.reserve(2 * nobj);
        SPH_HIP(hipMemcpyAsync(body_.get(), tab.data(), 2 * nobj * sizeof(float4), hipMemcpyHostToDevice, stream));
        if (!bforce_.get()) {
            bforce_.reserve(6 * nobj);
            fill_u32(stream, reinterpret_cast<unsigned *>(bforce_.get()), 12 * nobj, 0u);
        }
        SPH_HIP(hipStreamSynchronize(stream));
    }
}

void DFSPH::body_forces_pressure(bool pressure) {
    const Dev D = dev();
    if (!D.nbody) return;
    const unsigned nb = nblocks(n_);
    bpart_.reserve((size_t)nb * D.nbody * 6);
    const Dev E = dev();
    {
        TimedScope ts(timer, stream, "body_forces");
        if (pressure)
            k_body_force_p<true><<<nb, BLOCK, 0, stream>>>(E);
        else
            k_body_force_p<false><<<nb, BLOCK, 0, stream>>>(E);
        k_body_reduce<<<1, RBLOCK, 0, stream>>>(E, nb);
        SPH_HIP(hipGetLastError());
    }
}

void DFSPH::body_forces_nonpressure(const Dev &D0) {
    if (!D0.nbody || (D0.xsphB == 0.f && D0.sviscB == 0.f)) return;
    const unsigned nb = nblocks(n_);
    bpart_.reserve((size_t)nb * D0.nbody * 6);
    Dev E = D0;
    E.bpart = bpart_.get();
    TimedScope ts(timer, stream, "body_forces");
    k_body_force_np<<<nb, BLOCK, 0, stream>>>(E);
    k_body_reduce<<<1, RBLOCK, 0, stream>>>(E, nb);
    SPH_HIP(hipGetLastError());
}

void DFSPH::body_force(unsigned o, double force[3], double torque[3], bool clear) {
    SPH_REQUIRE(o < vm_shapes_.size(), SPH_ERR_INVALID, "boundary object out of range");
    for (int c = 0; c < 3; c++) force[c] = torque[c] = 0.0;
    if (!bforce_.get() || o >= vmaps.size()) return;
    double f[6];
    SPH_HIP(hipMemcpyAsync(f, bforce_.get() + 6 * o, sizeof(f), hipMemcpyDeviceToHost, stream));
    SPH_HIP(hipStreamSynchronize(stream));
    for (int c = 0; c < 3; c++) {
        force[c] = f[c];
        torque[c] = f[3 + c];
    }
    if (clear) {
        fill_u32(stream, reinterpret_cast<unsigned *>(bforce_.get() + 6 * o), 12, 0u);
        SPH_HIP(hipStreamSynchronize(stream));
    }
}

void DFSPH::body_reference(unsigned o, double pos0[3], double *max_dist) {
    SPH_REQUIRE(o < vm_shapes_.size(), SPH_ERR_INVALID, "boundary object out of range");
    shape_reference_point(vm_shapes_[o], pos0, max_dist);
}

// ------------------------------------------------------- several fluid models
void DFSPH::set_fluid_models(const unsigned *model, size_t n, const double *mat, unsigned nm) {
    if (!initialized_) init();
    SPH_REQUIRE(n == n_, SPH_ERR_INVALID, "fluid models: one model index per particle");
    SPH_REQUIRE(nm >= 1 && nm <= 8, SPH_ERR_INVALID, "fluid models: 1 to 8 models");
    SPH_REQUIRE(method_ == SPH_METHOD_DFSPH, SPH_ERR_STATE, "several fluid models need the DFSPH step");
    SPH_REQUIRE(P.viscosity_method != SPH_VISCOSITY_WEILER2018, SPH_ERR_STATE,
                "several fluid models with Weiler2018 viscosity are not supported");
    SPH_REQUIRE(emitters_.empty(), SPH_ERR_STATE, "several fluid models with emitters are not supported");
    SPH_REQUIRE(mode_[0] == 0 && mode_[1] == 0 && stride_s_[0] == 0 && stride_s_[1] == 0, SPH_ERR_STATE,
                "several fluid models need the reference's warm start");
    std::vector<unsigned> cnt(nm, 0);
    for (size_t i = 0; i < n; i++) {
        SPH_REQUIRE(model[i] < nm, SPH_ERR_INVALID, "fluid models: model index out of range");
        cnt[model[i]]++;
    }
    for (unsigned m = 0; m < nm; m++)
        SPH_REQUIRE(mat[5 * m] > 0.0 && std::isfinite(mat[5 * m]), SPH_ERR_INVALID, "fluid models: density0 must be > 0");
    materials_.clear();
    for (unsigned m = 0; m < nm; m++)
        materials_.push_back({mat[5 * m], mat[5 * m + 1], mat[5 * m + 2], mat[5 * m + 3], mat[5 * m + 4]});
    model_count_ = cnt;
    model_.reserve(stride_);
    model2_.reserve(stride_);
    const std::vector<unsigned> id = ids_host();
    std::vector<unsigned> t(n);
    for (size_t sl = 0; sl < n; sl++) t[sl] = model[id[sl]];
    SPH_HIP(hipStreamSynchronize(stream));
    SPH_HIP(hipMemcpy(model_.get(), t.data(), n * sizeof(unsigned), hipMemcpyHostToDevice));
    models_ = true;
    mrho_w_ = false;
}

void DFSPH::pressure_setup() {
    Dev D = dev();
    if (learn_or_collect(0)) D.kprev = kprev_.get();
    LAUNCH_LPP1("pressure_setup", k_psetup);
}

// Scale, features and (with a model) the network's start plus the first
// iteration from the per-particle better start. Returns iterations done.
bool DFSPH::learned_start(bool pressure) {
    const int solver = pressure ? 0 : 1;
    const bool was = engaged_[solver];
    engaged_[solver] = false;
    if (!learn_or_collect(solver)) return false;
    // A better start pays only when the reference's start is far from the
    // solution. After a solve from the reference's start, engage it if that
    // solve took at least engage_min_ iterations; after a solve from the
    // better start, keep it unless that solve ended at the minimum count
    // (then the next step tries the reference's start again).
    const int mode = mode_[solver];
    const int prev = pressure ? itLast_ : itVLast_;
    const int floor = pressure ? std::max(P.min_iterations, 1) : 1;
    const bool use = mode != 0 && (engage_min_[solver] == 0 || (was ? prev > floor : prev >= engage_min_[solver]));
    const bool collecting = stride_s_[solver] > 0;
    if (!use && !collecting) return false;
    Dev D = dev();
    D.kprev = kprev_.get();
    if (collecting || mode == 2) {
        LAUNCH("learn_scale", k_max_partial, D, kprev_.get());
        if (pressure)
            REDUCE("learn_scale", k_kref_reduce<true>, D, nblocks(n_));
        else
            REDUCE("learn_scale", k_kref_reduce<false>, D, nblocks(n_));
        if (pressure)
            LAUNCH_SEQ("learn_features", k_features, true);
        else
            LAUNCH_SEQ("learn_features", k_features, false);
    }
    if (!use) return false;
    engaged_[solver] = true;
    (pressure ? learnedSolves_ : learnedSolvesV_)++;
    D.strictP = engaged_[0];
    D.strictV = engaged_[1];
    if (mode == 2) {
        TimedScope ts(timer, stream, "learn_mlp");
        mlp_forward(stream, theta_[solver].get(), feats_[solver].get(), (unsigned)n_, pred_.get());
    }
    if (pressure) {
        if (mode == 2)
            LAUNCH("learn_start", (k_pred_start<true, true>), D);
        else
            LAUNCH("learn_start", (k_pred_start<true, false>), D);
        LAUNCH_SEQ("learn_accel2", k_accel2, true);
        LAUNCH_SEQ("learn_jacobi2", k_jacobi2, true);
        REDUCE("jacobi_reduce", (k_jacobi_reduce<true, true>), D, nblocks((size_t)n_ * seq_lanes()), 0);
    } else {
        if (mode == 2)
            LAUNCH("learn_start", (k_pred_start<false, true>), D);
        else
            LAUNCH("learn_start", (k_pred_start<false, false>), D);
        LAUNCH_SEQ("learn_accel2", k_accel2, false);
        LAUNCH_SEQ("learn_jacobi2", k_jacobi2, false);
        REDUCE("jacobi_reduce", (k_jacobi_reduce<false, true>), D, nblocks((size_t)n_ * seq_lanes()), 0);
    }
    return true;
}

void DFSPH::collect(bool pressure) {
    const int solver = pressure ? 0 : 1;
    if (stride_s_[solver] == 0) return;
    const Dev D = dev();
    if (pressure)
        LAUNCH("learn_collect", k_collect<true>, D);
    else
        LAUNCH("learn_collect", k_collect<false>, D);
}

void DFSPH::set_warm_start_model(int solver, const float *theta) {
    SPH_REQUIRE(solver == 0 || solver == 1, SPH_ERR_INVALID, "solver must be 0 (pressure) or 1 (divergence)");
    if (!theta) {
        learned_[solver] = false;
        mode_[solver] = 0;
        return;
    }
    theta_[solver].reserve(MLP_NPARAM);
    SPH_HIP(hipMemcpy(theta_[solver].get(), theta, MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice));
    learned_[solver] = true;
    mode_[solver] = 2;
    ensure_learn_buffers();
}

void DFSPH::set_warm_start_mode(int solver, int mode) {
    SPH_REQUIRE(solver == 0 || solver == 1, SPH_ERR_INVALID, "solver must be 0 (pressure) or 1 (divergence)");
    SPH_REQUIRE(mode >= 0 && mode <= 2, SPH_ERR_INVALID, "warm-start mode must be 0, 1 or 2");
    SPH_REQUIRE(mode != 2 || learned_[solver], SPH_ERR_STATE, "mode 2 needs a network (set_warm_start_model)");
    SPH_REQUIRE(mode == 0 || !models_, SPH_ERR_STATE, "several fluid models need the reference's warm start");
    mode_[solver] = mode;
    if (mode) ensure_learn_buffers();
}

void DFSPH::set_warm_start_policy(int solver, int min_prev_iterations) {
    SPH_REQUIRE(solver == 0 || solver == 1, SPH_ERR_INVALID, "solver must be 0 (pressure) or 1 (divergence)");
    SPH_REQUIRE(min_prev_iterations >= 0, SPH_ERR_INVALID, "min_prev_iterations must be >= 0");
    engage_min_[solver] = min_prev_iterations;
}

void DFSPH::collect_training(int solver, unsigned stride, size_t capacity) {
    SPH_REQUIRE(solver == 0 || solver == 1, SPH_ERR_INVALID, "solver must be 0 (pressure) or 1 (divergence)");
    SPH_REQUIRE(capacity < (size_t)0xffffffffu, SPH_ERR_INVALID, "capacity too large");
    SPH_REQUIRE(stride == 0 || !models_, SPH_ERR_STATE, "training samples need a single fluid model");
    stride_s_[solver] = stride;
    cap_s_[solver] = stride ? capacity : 0;
    if (stride) {
        sx_[solver].reserve(std::max<size_t>(capacity, 1) * 8);
        st_[solver].reserve(std::max<size_t>(capacity, 1));
        ensure_learn_buffers();
    }
    const unsigned zero = 0;
    upload_ctl_field(solver == 0 ? offsetof(Ctl, nsamp) : offsetof(Ctl, nsamp_v), &zero, sizeof(unsigned));
}

void DFSPH::get_training(int solver, float *x, float *t, size_t capacity, size_t *n) {
    SPH_REQUIRE(solver == 0 || solver == 1, SPH_ERR_INVALID, "solver must be 0 (pressure) or 1 (divergence)");
    read_ctl();
    const size_t have = std::min<size_t>(solver == 0 ? hctl_->nsamp : hctl_->nsamp_v, cap_s_[solver]);
    const size_t k = std::min(have, capacity);
    if (k && x) SPH_HIP(hipMemcpy(x, sx_[solver].get(), k * 8 * sizeof(float), hipMemcpyDeviceToHost));
    if (k && t) SPH_HIP(hipMemcpy(t, st_[solver].get(), k * sizeof(float), hipMemcpyDeviceToHost));
    if (n) *n = k;
    const unsigned zero = 0;
    upload_ctl_field(solver == 0 ? offsetof(Ctl, nsamp) : offsetof(Ctl, nsamp_v), &zero, sizeof(unsigned));
}

void DFSPH::ensure_learn_buffers() {
    if (!initialized_) return;  // init() allocates them
    const size_t S = stride_;
    feats_[0].reserve(8 * S);
    feats_[1].reserve(8 * S);
    pred_.reserve(S);
    kprev_.reserve(S);
    ap2_.reserve(S);
}

void DFSPH::pressure_finish(bool finalize_too) {
    const Dev D = dev();
    LAUNCH_LPP_AS("pressure_finish", lppA_, k_finish, true);
    if (dynamic_) body_forces_pressure(true);
    if (finalize_too) finalize(true, true);
}

void DFSPH::finalize(bool scale_p, bool update_x) {
    const Dev D = dev();
    if (scale_p && update_x)
        LAUNCH("finalize", (k_final<true, true>), D);
    else if (scale_p)
        LAUNCH("finalize", (k_final<true, false>), D);
    else if (update_x)
        LAUNCH("finalize", (k_final<false, true>), D);
}

void DFSPH::post_forces(bool clear, bool apply, int expl, bool cfl, bool vupd, bool scale_pv) {
    Dev D = dev();
    if (!(expl & 1)) {
        D.xsph = D.xsphB = 0.f;
        for (int m = 0; m < 8; m++) D.xsm[m] = D.xsbm[m] = 0.f;
    }
    if (!(expl & 2)) {
        D.svisc = D.sviscB = 0.f;
        for (int m = 0; m < 8; m++) D.svm[m] = D.svbm[m] = 0.f;
    }
    const bool xsph = D.xsph != 0.f || D.xsphB != 0.f || D.svisc != 0.f;
    if ((D.xsph != 0.f || D.svisc != 0.f) && !mrho_w_) LAUNCH("mass_density_copy", k_mrho_to_w, D);
    if (dynamic_ && xsph) {
        Dev E = D;
        if (E.svisc == 0.f) E.sviscB = 0.f;  // boundary viscosity belongs to the standard viscosity
        body_forces_nonpressure(E);
    }
    // the step uses the full fusion; single stages use the one-flag forms
    if (clear && !apply && !xsph && !cfl && !vupd && !scale_pv)
        LAUNCH_LPP("clear_accel", k_post, true, false, false, false, false, false);
    else if (!clear && apply && !xsph && !cfl && !vupd)
        LAUNCH_LPP("viscosity_apply", k_post, false, true, false, false, false, false);
    else if (!clear && !apply && xsph && !cfl && !vupd)
        LAUNCH_LPP("xsph", k_post, false, false, true, false, false, false);
    else if (!clear && !apply && !xsph && cfl && !vupd)
        LAUNCH_LPP("cfl", k_post, false, false, false, true, false, false);
    else if (!clear && !apply && !xsph && !cfl && vupd)
        LAUNCH_LPP("update_velocity", k_post, false, false, false, false, true, false);
    else {
        // step: clear, [apply], [xsph], [cfl], v update, [pv scale]
#define POSTV(A, X, C, S) LAUNCH_LPP("post_forces", k_post, true, A, X, C, true, S)
        const int key = (apply ? 8 : 0) | (xsph ? 4 : 0) | (cfl ? 2 : 0) | (scale_pv ? 1 : 0);
        switch (key) {
            case 0: POSTV(false, false, false, false); break;
            case 1: POSTV(false, false, false, true); break;
            case 2: POSTV(false, false, true, false); break;
            case 3: POSTV(false, false, true, true); break;
            case 4: POSTV(false, true, false, false); break;
            case 5: POSTV(false, true, false, true); break;
            case 6: POSTV(false, true, true, false); break;
            case 7: POSTV(false, true, true, true); break;
            case 8: POSTV(true, false, false, false); break;
            case 9: POSTV(true, false, false, true); break;
            case 10: POSTV(true, false, true, false); break;
            case 11: POSTV(true, false, true, true); break;
            case 12: POSTV(true, true, false, false); break;
            case 13: POSTV(true, true, false, true); break;
            case 14: POSTV(true, true, true, false); break;
            default: POSTV(true, true, true, true); break;
        }
#undef POSTV
    }
    if (cfl) REDUCE("cfl_reduce", k_cfl_reduce, D, nblocks((size_t)n_ * lpp_));
    if (vupd) v_.swap(v2_);
}

void DFSPH::stiff_to_w(bool pressure) {
    const Dev D = dev();
    if (pressure)
        LAUNCH("stiffness_copy", k_stiff_to_w<true>, D);
    else
        LAUNCH("stiffness_copy", k_stiff_to_w<false>, D);
}

int DFSPH::run_solver(bool pressure, int already, bool copy_w) {
    if (!picked_) pick_lanes();
    if (copy_w) stiff_to_w(pressure);
    const int maxIt = pressure ? P.max_iterations : P.max_iterations_v;
    int launched = already;
    int chunk = std::max(1, pressure ? std::max(lastIt_, P.min_iterations) : lastItV_);
    for (;;) {
        for (int c = 0; c < chunk && launched < maxIt; c++, launched++) {
            if (pressure)
                pressure_iteration(false);
            else
                div_iteration(false);
        }
        read_ctl();
        if (tiled_) tiles_over_ = hctl_->tiles_over;
        const int done = pressure ? hctl_->done : hctl_->done_v;
        if (done || launched >= maxIt) break;
        // past the predicted count: two iterations per round trip (an
        // iteration of a converged solve costs a few microseconds of early
        // exits, a host round trip tens)
        chunk = 2;
    }
    return solve_result(pressure, false);
}

int DFSPH::first_chunk(bool pressure) const {
    return std::max(1, pressure ? std::max(lastIt_, P.min_iterations) : lastItV_);
}

// Iterations of the solve that just ended (its counters read back), with
// the solves stopped by the cap counted.
int DFSPH::solve_result(bool pressure, bool read) {
    if (read) read_ctl();
    const int maxIt = pressure ? P.max_iterations : P.max_iterations_v;
    const int it = pressure ? hctl_->it : hctl_->it_v;
    if (it >= maxIt) {
        // stopped by the cap: count it unless the tolerance was met anyway
        const double eta = pressure ? P.max_error * 0.01 * P.density0
                                    : (1.0 / hctl_->h) * P.max_error_v * 0.01 * P.density0;
        const bool strict = engaged_[pressure ? 0 : 1];
        const double err = pressure ? hctl_->avg_err : hctl_->avg_err_v;
        const double over = pressure ? hctl_->avg_over : hctl_->avg_over_v;
        if (!(err <= eta) || (strict && !(over <= eta))) (pressure ? capped_ : cappedV_)++;
    }
    return it;
}

int DFSPH::run_cg() {
    const Dev D = dev();
    if (!mrho_w_) LAUNCH("mass_density_copy", k_mrho_to_w, D);
    k_reset<<<1, 1, 0, stream>>>(ctl_.get(), 3);
    LAUNCH("cg_x0", k_weiler_x0, D);
    LAUNCH_LPP1("cg_init", k_weiler_r0);
    REDUCE("cg_reduce", k_cg_init_reduce, D, nblocks((size_t)n_ * lpp_));
    LAUNCH_LPP1("cg_precond", k_weiler_precond);
    REDUCE("cg_reduce", k_cg_rz_reduce, D, nblocks((size_t)n_ * lpp_));
    int launched = 0, chunk = std::max(1, lastCg_ + 1);
    for (;;) {
        for (int c = 0; c < chunk && launched < P.visco_max_iter; c++, launched++) {
            LAUNCH_LPP1("cg_matvec", k_cg_matvec);
            REDUCE("cg_reduce", k_cg_alpha, D, nblocks((size_t)n_ * lpp_));
            LAUNCH("cg_update", k_cg_update, D);
            REDUCE("cg_reduce", k_cg_update_reduce, D, nblocks(n_));
            LAUNCH("cg_pupdate", k_cg_pupdate, D);
        }
        read_ctl();
        if (hctl_->cg_done || launched >= P.visco_max_iter) break;
        chunk = 2;
    }
    return hctl_->cg_it;
}

// computeViscosity. Weiler2018: the implicit solve (its result is applied
// with the other forces of the step, or here for a stand-alone stage);
// the explicit standard viscosity is part of the step's force sweep and
// runs here only as a stand-alone stage.
void DFSPH::viscosity(bool apply_separately) {
    if (n_ == 0) return;
    if (P.viscosity_method == SPH_VISCOSITY_STANDARD) {
        if (apply_separately) post_forces(false, false, 2, false, false, false);
        return;
    }
    if (P.viscosity_method != SPH_VISCOSITY_WEILER2018) return;
    cgLast_ = run_cg();
    lastCg_ = cgLast_;
    totVisco_ += cgLast_;
    if (apply_separately) post_forces(false, true, 0, false, false, false);
}

// m / rho into the w of the fluid positions for the non-pressure forces.
void DFSPH::mrho_copy() {
    const Dev D = dev();
    LAUNCH("mass_density_copy", k_mrho_to_w, D);
    mrho_w_ = true;
}

void DFSPH::step() {
    if (!initialized_) init();
    if (method_ == SPH_METHOD_PCISPH) {
        step_pcisph();
        return;
    }
    if (method_ == SPH_METHOD_IISPH) {
        step_iisph();
        return;
    }
    if (method_ == SPH_METHOD_WCSPH) {
        step_wcsph();
        return;
    }
    const bool div = step_begin();
    if (div) {
        const bool lv = learned_start(false);
        step_after_divergence(run_solver(false, lv ? 1 : 0, false));  // the set-up wrote the copy
    }
    step_middle(div);
    const bool lp = learned_start(true);
    step_after_pressure(run_solver(true, lp ? 1 : 0, false));
}

// The step around its two solves (TimeStepDFSPH::step, TimeStepDFSPH.cpp:117-249):
// neighbours, boundary records, densities, factor and the divergence set-up.
bool DFSPH::step_begin() {
    if (!initialized_) init();
    neighborhood_search();
    volume_maps();
    const bool div = P.enable_divergence_solver != 0;
    if (div) k_reset<<<1, 1, 0, stream>>>(ctl_.get(), 1);
    sweep_init(true, true, div);
    return div;
}

void DFSPH::step_after_divergence(int it) {
    itVLast_ = it;
    lastItV_ = std::max(1, itVLast_);
    totItV_ += itVLast_;
    div_finish(false);
}

// Non-pressure forces, CFL, velocity update and the pressure set-up.
void DFSPH::step_middle(bool div) {
    if (!div) itVLast_ = 0;
    const bool weiler = P.viscosity_method == SPH_VISCOSITY_WEILER2018;
    const bool stdv = P.viscosity_method == SPH_VISCOSITY_STANDARD;
    if ((weiler || stdv || any_xsph()) && n_) mrho_copy();
    if (weiler) viscosity(false);
    const int expl = (any_xsph() ? 1 : 0) | (stdv ? 2 : 0);
    post_forces(true, weiler, expl, P.cfl_method == 1 || P.cfl_method == 2, true, div);
    mrho_w_ = false;
    if (div) collect(false);
    k_reset<<<1, 1, 0, stream>>>(ctl_.get(), 0);
    pressure_setup();
}

void DFSPH::step_after_pressure(int it) {
    itLast_ = it;
    lastIt_ = std::max(P.min_iterations, itLast_);
    totIt_ += itLast_;
    pressure_finish(true);
    collect(true);
    emitter_system_step();
    soff_++;
    steps_++;
}

void DFSPH::stage(int s) {
    if (!initialized_) init();
    if (s != SPH_STAGE_NEIGHBORHOOD_SEARCH) SPH_REQUIRE(have_lists_, SPH_ERR_STATE, "run the neighbourhood search first");
    switch (s) {
        case SPH_STAGE_NEIGHBORHOOD_SEARCH: neighborhood_search(); break;
        case SPH_STAGE_VOLUME_MAPS: volume_maps(); break;
        case SPH_STAGE_DENSITIES: sweep_init(true, false, false); break;
        case SPH_STAGE_DFSPH_FACTOR: sweep_init(false, true, false); break;
        case SPH_STAGE_DIVERGENCE_SETUP:
            k_reset<<<1, 1, 0, stream>>>(ctl_.get(), 1);
            sweep_init(false, false, true);
            break;
        case SPH_STAGE_DIVERGENCE_ITER:
            stiff_to_w(false);
            div_iteration(true);
            break;
        case SPH_STAGE_DIVERGENCE_FINISH:
            stiff_to_w(false);
            div_finish(true);
            break;
        case SPH_STAGE_DIVERGENCE_SOLVE:
            k_reset<<<1, 1, 0, stream>>>(ctl_.get(), 1);
            sweep_init(false, false, true);
            itVLast_ = run_solver(false, learned_start(false) ? 1 : 0);
            totItV_ += itVLast_;
            div_finish(true);
            break;
        case SPH_STAGE_CLEAR_ACCEL: post_forces(true, false, 0, false, false, false); break;
        case SPH_STAGE_VISCOSITY: viscosity(true); break;
        case SPH_STAGE_XSPH:
            if (any_xsph()) post_forces(false, false, 1, false, false, false);
            break;
        case SPH_STAGE_CFL:
            if (P.cfl_method == 1 || P.cfl_method == 2) post_forces(false, false, 0, true, false, false);
            break;
        case SPH_STAGE_UPDATE_VELOCITY: post_forces(false, false, 0, false, true, false); break;
        case SPH_STAGE_PRESSURE_SETUP:
            k_reset<<<1, 1, 0, stream>>>(ctl_.get(), 0);
            pressure_setup();
            break;
        case SPH_STAGE_PRESSURE_ITER:
            stiff_to_w(true);
            pressure_iteration(true);
            break;
        case SPH_STAGE_PRESSURE_FINISH:
            stiff_to_w(true);
            pressure_finish(false);
            finalize(true, false);
            break;
        case SPH_STAGE_PRESSURE_SOLVE:
            k_reset<<<1, 1, 0, stream>>>(ctl_.get(), 0);
            pressure_setup();
            itLast_ = run_solver(true, learned_start(true) ? 1 : 0);
            totIt_ += itLast_;
            pressure_finish(false);
            finalize(true, false);
            break;
        case SPH_STAGE_UPDATE_POSITION:
            finalize(false, true);
            emitter_system_step();
            break;
        default: throw Error(SPH_ERR_INVALID, "unknown stage");
    }
    SPH_HIP(hipStreamSynchronize(stream));
}

// --------------------------------------------------------------- fields
std::vector<unsigned> DFSPH::ids_host() {
    std::vector<unsigned> id(n_);
    SPH_HIP(hipStreamSynchronize(stream));
    if (n_) SPH_HIP(hipMemcpy(id.data(), id_.get(), n_ * sizeof(unsigned), hipMemcpyDeviceToHost));
    return id;
}

namespace {
struct FieldInfo {
    int comps;      // 1 or 3
    int kind;       // 0 float4 array, 1 float array, 2 unsigned array, 3 vmb.w, 4 vmb.xyz
    const char *name;
};
}  // namespace

void DFSPH::get_field(const std::string &name, void *host, size_t bytes) {
    SPH_REQUIRE(initialized_, SPH_ERR_STATE, "not initialised");
    const size_t n = n_;
    if (name == "boundary particle volume") {
        SPH_REQUIRE(bytes == nb_ * sizeof(float), SPH_ERR_INVALID, "size mismatch");
        if (!nb_) return;
        std::vector<float4> b(nb_);
        std::vector<unsigned> perm(nb_);
        SPH_HIP(hipStreamSynchronize(stream));
        SPH_HIP(hipMemcpy(b.data(), bx_.get(), nb_ * sizeof(float4), hipMemcpyDeviceToHost));
        SPH_HIP(hipMemcpy(perm.data(), bperm_.get(), nb_ * sizeof(unsigned), hipMemcpyDeviceToHost));
        float *out = static_cast<float *>(host);
        for (size_t s = 0; s < nb_; s++) out[perm[s]] = b[s].w;
        return;
    }
    const float4 *f4 = nullptr;
    const float *f1 = nullptr;
    const unsigned *u1 = nullptr;
    int comps = 1, vmpart = 0;
    if (name == "position") f4 = x_.get(), comps = 3;
    else if (name == "velocity") f4 = v_.get(), comps = 3;
    else if (name == "acceleration") f4 = a_.get(), comps = 3;
    else if (name == "pressure acceleration") f4 = ap_.get(), comps = 3;
    else if (name == "velocity difference") f4 = vdiff_.get(), comps = 3;
    else if (name == "predicted position") {
        SPH_REQUIRE(method_ == SPH_METHOD_PCISPH, SPH_ERR_NOTFOUND, "predicted positions exist with PCISPH only");
        f4 = predx_.get(), comps = 3;
    }
    else if (name.rfind("boundary x", 0) == 0 || name.rfind("boundary volume", 0) == 0 ||
             name.rfind("boundary density", 0) == 0) {
        // "boundary x" / "boundary volume" of map object 0, or "... <o>";
        // with Koschier2017 the volume is the boundary density and
        // "boundary density gradient" is its gradient
        const bool isg = name.rfind("boundary density gradient", 0) == 0;
        SPH_REQUIRE(!isg || P.boundary_handling_method == SPH_BOUNDARY_KOSCHIER2017, SPH_ERR_NOTFOUND,
                    "boundary density gradients exist with Koschier2017 only");
        const bool isx = isg || name.rfind("boundary x", 0) == 0;
        const size_t plen = isg ? 25 : (name.rfind("boundary x", 0) == 0 ? 10 : (name.rfind("boundary volume", 0) == 0 ? 15 : 16));
        const std::string rest = name.substr(plen);
        unsigned o = 0;
        if (!rest.empty()) {
            SPH_REQUIRE(rest[0] == ' ' && rest.size() > 1 && rest.find_first_not_of("0123456789", 1) == std::string::npos,
                        SPH_ERR_NOTFOUND, "unknown field '" + name + "'");
            o = (unsigned)std::stoul(rest.substr(1));
        }
        SPH_REQUIRE(o < std::max(nvm_, 1u), SPH_ERR_NOTFOUND, "no volume map " + std::to_string(o));
        f4 = (isg ? (nvm_ > 1 ? dmgraw_.get() : dmg_.get()) : (nvm_ > 1 ? vmraw_.get() : vmb_.get())) +
             (size_t)o * stride_;
        comps = isx ? 3 : 1;
        vmpart = isx ? 1 : 2;
    }
    else if (name == "density") f1 = rho_.get();
    else if (name == "factor") f1 = alpha_.get();
    else if (name == "advected density") f1 = radv_.get();
    else if (name == "p / rho^2" || name == "pressure") f1 = p_.get();  // "pressure": WCSPH, PCISPH, IISPH
    else if (name == "p_v / rho^2") f1 = pv_.get();
    else if (name == "id") u1 = id_.get();
    else if (name == "state") u1 = pst_.get();
    else if (name == "fluid model") {
        if (!models_) {  // one model: every particle is in model 0
            SPH_REQUIRE(bytes == n * 4, SPH_ERR_INVALID, "size mismatch for field 'fluid model'");
            std::memset(host, 0, bytes);
            return;
        }
        u1 = model_.get();
    }
    else if (name == "fluid neighbor count") u1 = cf_.get();
    else if (name == "boundary neighbor count") u1 = cb_.get();
    else throw Error(SPH_ERR_NOTFOUND, "unknown field '" + name + "'");
    SPH_REQUIRE(bytes == n * comps * 4, SPH_ERR_INVALID, "size mismatch for field '" + name + "'");
    if (n == 0) return;
    if ((name == "boundary neighbor count" && !(P.boundary_handling_method == SPH_BOUNDARY_AKINCI2012 && nb_ > 0)) ||
        (name == "state" && !states_)) {
        std::memset(host, 0, bytes);
        return;
    }
    io_.reserve(3 * (size_t)stride_);
    const unsigned nn = (unsigned)n;
    if (f4 && vmpart != 2)
        k_field_out4<3><<<nblocks(n), BLOCK, 0, stream>>>(f4, id_.get(), nn, io_.get());
    else if (f4)
        k_field_out4<1><<<nblocks(n), BLOCK, 0, stream>>>(f4, id_.get(), nn, io_.get());
    else
        k_field_out1<<<nblocks(n), BLOCK, 0, stream>>>(f1 ? reinterpret_cast<const unsigned *>(f1) : u1, id_.get(), nn,
                                                       reinterpret_cast<unsigned *>(io_.get()));
    SPH_HIP(hipGetLastError());
    SPH_HIP(hipMemcpyAsync(host, io_.get(), bytes, hipMemcpyDeviceToHost, stream));
    SPH_HIP(hipStreamSynchronize(stream));
}

void DFSPH::set_field(const std::string &name, const void *host, size_t bytes) {
    SPH_REQUIRE(initialized_, SPH_ERR_STATE, "not initialised");
    const size_t n = n_;
    float4 *f4 = nullptr;
    float *f1 = nullptr;
    int comps = 1;
    if (name == "position") f4 = x_.get(), comps = 3;
    else if (name == "velocity") f4 = v_.get(), comps = 3;
    else if (name == "acceleration") f4 = a_.get(), comps = 3;
    else if (name == "pressure acceleration") f4 = ap_.get(), comps = 3;
    else if (name == "velocity difference") f4 = vdiff_.get(), comps = 3;
    else if (name == "predicted position" && method_ == SPH_METHOD_PCISPH) f4 = predx_.get(), comps = 3;
    else if (name == "density") f1 = rho_.get();
    else if (name == "factor") f1 = alpha_.get();
    else if (name == "advected density") f1 = radv_.get();
    else if (name == "p / rho^2" || name == "pressure") f1 = p_.get();  // "pressure": WCSPH, PCISPH, IISPH
    else if (name == "p_v / rho^2") f1 = pv_.get();
    else if (name != "state") throw Error(SPH_ERR_NOTFOUND, "unknown or read-only field '" + name + "'");
    SPH_REQUIRE(bytes == n * comps * 4, SPH_ERR_INVALID, "size mismatch for field '" + name + "'");
    if (name == "state") {
        // ParticleState: 0 active, 1 animated by an emitter, 2 fixed
        const unsigned *in = static_cast<const unsigned *>(host);
        for (size_t k = 0; k < n; k++) SPH_REQUIRE(in[k] <= 2u, SPH_ERR_INVALID, "particle state must be 0, 1 or 2");
        enable_states();
    }
    if (n == 0) return;
    io_.reserve(3 * (size_t)stride_);
    const unsigned nn = (unsigned)n;
    SPH_HIP(hipMemcpyAsync(io_.get(), host, bytes, hipMemcpyHostToDevice, stream));
    if (f4)
        k_field_in4<<<nblocks(n), BLOCK, 0, stream>>>(io_.get(), id_.get(), nn, f4,
                                                      name == "position" ? xc_.get() : nullptr);
    else
        k_field_in1<<<nblocks(n), BLOCK, 0, stream>>>(reinterpret_cast<const unsigned *>(io_.get()), id_.get(), nn,
                                                      f1 ? reinterpret_cast<unsigned *>(f1) : pst_.get());
    SPH_HIP(hipGetLastError());
    SPH_HIP(hipStreamSynchronize(stream));
}

void DFSPH::get_neighbors(int boundary, unsigned *offsets, unsigned *indices, size_t capacity, size_t *nnz) {
    SPH_REQUIRE(have_lists_, SPH_ERR_STATE, "no neighbour lists yet");
    const size_t n = n_;
    const bool bset = boundary != 0;
    const bool akinci = P.boundary_handling_method == SPH_BOUNDARY_AKINCI2012 && nb_ > 0;
    const unsigned cap = bset ? capB_ : capF_;
    std::vector<unsigned> cnt(n, 0u), lists, id = ids_host(), bperm;
    if (!bset || akinci) {
        SPH_HIP(hipMemcpy(cnt.data(), bset ? cb_.get() : cf_.get(), n * sizeof(unsigned), hipMemcpyDeviceToHost));
        lists.resize((size_t)cap * stride_);
        SPH_HIP(hipMemcpy(lists.data(), bset ? nb_l_.get() : nf_.get(), lists.size() * sizeof(unsigned),
                          hipMemcpyDeviceToHost));
    }
    if (bset && akinci) {
        bperm.resize(nb_);
        SPH_HIP(hipMemcpy(bperm.data(), bperm_.get(), nb_ * sizeof(unsigned), hipMemcpyDeviceToHost));
    }
    std::vector<unsigned> rowcnt(n);
    for (size_t s = 0; s < n; s++) rowcnt[id[s]] = cnt[s];
    std::vector<size_t> off(n + 1, 0);
    for (size_t i = 0; i < n; i++) off[i + 1] = off[i] + rowcnt[i];
    if (nnz) *nnz = off[n];
    if (offsets)
        for (size_t i = 0; i <= n; i++) offsets[i] = (unsigned)off[i];
    if (!indices) return;
    SPH_REQUIRE(capacity >= off[n], SPH_ERR_INVALID, "neighbour capacity too small");
    for (size_t s = 0; s < n; s++) {
        const size_t row = id[s];
        unsigned *o = indices + off[row];
        for (unsigned k = 0; k < cnt[s]; k++) {
            const unsigned j = lists[(size_t)k * stride_ + s];
            o[k] = bset ? bperm[j] : id[j];
        }
        std::sort(o, o + cnt[s]);
    }
}

void DFSPH::counters(sph_dfsph_counters_t *c) {
    read_ctl();
    std::memset(c, 0, sizeof(*c));
    c->time = hctl_->time;
    c->time_step_size = hctl_->h;
    c->avg_density_err = hctl_->avg_err;
    c->avg_divergence_err = hctl_->avg_err_v;
    c->iterations = hctl_->it;
    c->iterations_v = P.enable_divergence_solver ? hctl_->it_v : 0;
    c->visco_iterations = hctl_->cg_it;
    c->steps = steps_;
    c->total_iterations = totIt_;
    c->total_iterations_v = totItV_;
    c->total_visco_iterations = totVisco_;
    c->max_fluid_neighbors = (int)hctl_->maxcnt_f;
    c->max_boundary_neighbors = (int)hctl_->maxcnt_b;
    c->flags = hctl_->flags;
    c->learned_particles = engaged_[0] ? (int)hctl_->nlearn : 0;
    c->learned_particles_v = engaged_[1] ? (int)hctl_->nlearn_v : 0;
    c->learned_solves = learnedSolves_;
    c->lanes_per_particle = lpp_;
    c->lanes_per_particle_accel = lppA_;
    c->packed_lists = use16_ ? 1 : 0;
    c->host_syncs = syncs_;
    c->learned_solves_v = learnedSolvesV_;
    c->capped_solves = capped_;
    c->capped_solves_v = cappedV_;
    c->avg_overpressure_err = hctl_->avg_over;
    c->avg_overpressure_err_v = hctl_->avg_over_v;
}

void DFSPH::set_time(double t, double h) {
    SPH_REQUIRE(h > 0, SPH_ERR_INVALID, "time step size must be > 0");
    // h_step is taken from h by the next neighbourhood search
    k_set_time<<<1, 1, 0, stream>>>(ctl_.get(), t, h);
    SPH_HIP(hipGetLastError());
}

void DFSPH::sync() { SPH_HIP(hipStreamSynchronize(stream)); }

}  // namespace sph
