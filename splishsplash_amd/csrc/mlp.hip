// mlp.hip -- BF16 MFMA inference and training kernels of the warm-start
// network (see mlp.hpp).
//
// One wave computes a tile of 32 rows with v_mfma_f32_32x32x8bf16_1k
// (32x8 A, 8x32 B, 32x32 FP32 accumulator). Operand layouts of that
// instruction, lane l = 32 g + r:
//   A[m][k]: lane holds m = r, k = 4g .. 4g+3
//   B[k][n]: lane holds n = r, k = 4g .. 4g+3
//   C[m][n]: lane holds n = r, element e at m = 8 (e / 4) + 4 g + e % 4
// Between layers the activations go through LDS ([32][SP] BF16 per wave) to
// turn the C layout into the next A layout.
#include <algorithm>
#include <cmath>
#include <numeric>
#include <random>
#include <vector>

#include "grid.hpp"
#include "mlp.hpp"

namespace sph {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int SP = 68;        // LDS row pitch (BF16 elements)
constexpr int MWAVES = 4;     // waves per block

__device__ __forceinline__ short f2bf(float f) {
    unsigned u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
    return (short)(u >> 16);
}
// SiLU z * sigmoid(z) with the hardware reciprocal (1 ulp): the activations
// are rounded to BF16 (8 bits) right after, so a correctly rounded division
// would buy nothing.
__device__ __forceinline__ float sigm(float z) { return __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }
__device__ __forceinline__ float silu(float z) { return z * sigm(z); }
__device__ __forceinline__ f32x16 mfma(bf16x4 a, bf16x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ int crow(int e, int g) { return 8 * (e >> 2) + 4 * g + (e & 3); }
__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int e = 0; e < 16; e++) z[e] = 0.0f;
    return z;
}

// The staging buffers of a tile belong to one wave, and a wave's LDS
// accesses execute in program order, so passing activations between its
// lanes needs no block barrier: only the compiler must keep the order.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct Wregs {
    float w1[2][MLP_NIN];  // layer 1 (FP32): W1[k][32 h + r] of this lane's two columns
    bf16x4 B2[8][2];  // layer 2: 8 K-chunks, two halves
    bf16x4 B3[8];     // layer 3: only column 0 non-zero
    float b1[2], b2[2], w3[2], b3;
};

__device__ __forceinline__ void load_w(const float *__restrict__ th, Wregs &R, int r, int g) {
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int k = 0; k < MLP_NIN; k++) R.w1[h][k] = th[MLP_OFF_W1 + k * 64 + 32 * h + r];
#pragma unroll
    for (int kc = 0; kc < 8; kc++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int k = 8 * kc + 4 * g + j;
            R.B2[kc][0][j] = f2bf(th[MLP_OFF_W2 + k * 64 + r]);
            R.B2[kc][1][j] = f2bf(th[MLP_OFF_W2 + k * 64 + 32 + r]);
            R.B3[kc][j] = (r == 0) ? f2bf(th[MLP_OFF_W3 + k]) : (short)0;
        }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        R.b1[h] = th[MLP_OFF_B1 + 32 * h + r];
        R.b2[h] = th[MLP_OFF_B2 + 32 * h + r];
        R.w3[h] = th[MLP_OFF_W3 + 32 * h + r];
    }
    R.b3 = th[MLP_OFF_B3];
}

// Forward pass of one 32-row tile. Returns the pre-activations z1, z2 (with
// bias) in C layout and the output (valid in lanes r == 0). Leaves SiLU(z2)
// in S. Layer 1 (K = 6) runs in FP32 on the vector units from the inputs
// staged in XF, so the features keep their full precision (a normalisation
// folded into W1 and b1 costs nothing); layers 2 and 3 run on MFMA.
__device__ __forceinline__ void fwd_tile(const Wregs &R, const float *__restrict__ X, unsigned n, unsigned row0,
                                         short *S, float *XF, int r, int g, f32x16 &z1a, f32x16 &z1b, f32x16 &z2a,
                                         f32x16 &z2b, f32x16 &yv) {
    const unsigned row = row0 + (unsigned)r;
    float4 xv = make_float4(0.f, 0.f, 0.f, 0.f);
    if (row < n) xv = *reinterpret_cast<const float4 *>(X + (size_t)row * MLP_XSTRIDE + 4 * g);
    *reinterpret_cast<float4 *>(XF + r * MLP_XSTRIDE + 4 * g) = xv;
    wave_sync();
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const float *xr = XF + crow(e, g) * MLP_XSTRIDE;
        float a = 0.f, b = 0.f;
#pragma unroll
        for (int k = 0; k < MLP_NIN; k++) {
            a += xr[k] * R.w1[0][k];
            b += xr[k] * R.w1[1][k];
        }
        z1a[e] = a;
        z1b[e] = b;
    }
#pragma unroll
    for (int e = 0; e < 16; e++) {
        z1a[e] += R.b1[0];
        z1b[e] += R.b1[1];
        S[crow(e, g) * SP + r] = f2bf(silu(z1a[e]));
        S[crow(e, g) * SP + 32 + r] = f2bf(silu(z1b[e]));
    }
    wave_sync();
    z2a = zero16();
    z2b = zero16();
#pragma unroll
    for (int kc = 0; kc < 8; kc++) {
        const bf16x4 ak = *reinterpret_cast<const bf16x4 *>(S + r * SP + 8 * kc + 4 * g);
        z2a = mfma(ak, R.B2[kc][0], z2a);
        z2b = mfma(ak, R.B2[kc][1], z2b);
    }
    wave_sync();
#pragma unroll
    for (int e = 0; e < 16; e++) {
        z2a[e] += R.b2[0];
        z2b[e] += R.b2[1];
        S[crow(e, g) * SP + r] = f2bf(silu(z2a[e]));
        S[crow(e, g) * SP + 32 + r] = f2bf(silu(z2b[e]));
    }
    wave_sync();
    yv = zero16();
#pragma unroll
    for (int kc = 0; kc < 8; kc++) {
        const bf16x4 ak = *reinterpret_cast<const bf16x4 *>(S + r * SP + 8 * kc + 4 * g);
        yv = mfma(ak, R.B3[kc], yv);
    }
#pragma unroll
    for (int e = 0; e < 16; e++) yv[e] += R.b3;
    wave_sync();
}

__global__ __launch_bounds__(64 * MWAVES) void k_mlp_fwd(const float *__restrict__ th, const float *__restrict__ X,
                                                        unsigned n, float *__restrict__ y) {
    __shared__ short sm[MWAVES][32 * SP];
    __shared__ float xf[MWAVES][32 * MLP_XSTRIDE];
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 31, g = lane >> 5;
    Wregs R;
    load_w(th, R, r, g);
    const unsigned ntiles = (n + 31u) / 32u;
    for (unsigned t0 = blockIdx.x * MWAVES; t0 < ntiles; t0 += gridDim.x * MWAVES) {
        const unsigned row0 = (t0 + wid) * 32u;
        f32x16 z1a, z1b, z2a, z2b, yv;
        fwd_tile(R, X, n, row0, sm[wid], xf[wid], r, g, z1a, z1b, z2a, z2b, yv);
        if (r == 0)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const unsigned row = row0 + crow(e, g);
                if (row < n) y[row] = yv[e];
            }
    }
}

// BF16 weights of layers 2 and 3 in the order the matrix instructions take
// them: group c of lane l (16 bytes, eight values) at (c * 64 + l), so a wave
// loads a group of all lanes in one coalesced instruction. Groups 0-7: B2 of
// K-chunk c (half h, element j at 4 h + j), 8-15: W2^T the same way, 16-19:
// B3 of two K-chunks each (zero except in the lanes r == 0). A block that
// gathers and rounds the 140 values per lane from the FP32 parameters itself
// spends more time on that than on a tile.
constexpr int PACK_GROUPS = 20;
constexpr int PACK_WORDS = PACK_GROUPS * 64 * 8;  // shorts

// Parameter k rounded into every place of the packed weights that holds it.
__device__ __forceinline__ void pack_param(int k, float v, short *__restrict__ pk) {
    const short b = f2bf(v);
    if (k >= MLP_OFF_W2 && k < MLP_OFF_W2 + 64 * 64) {
        const int m = (k - MLP_OFF_W2) / 64, n = (k - MLP_OFF_W2) % 64;
        pk[((m / 8) * 64 + ((m % 8) / 4) * 32 + n % 32) * 8 + (n / 32) * 4 + m % 4] = b;
        pk[((8 + n / 8) * 64 + ((n % 8) / 4) * 32 + m % 32) * 8 + (m / 32) * 4 + n % 4] = b;
    } else if (k >= MLP_OFF_W3 && k < MLP_OFF_W3 + 64) {
        const int m = k - MLP_OFF_W3;
        pk[((16 + m / 16) * 64 + ((m % 8) / 4) * 32) * 8 + ((m / 8) % 2) * 4 + m % 4] = b;
    }
}
__global__ void k_mlp_pack(const float *__restrict__ th, short *__restrict__ pk) {
    const int k = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    // the lanes r != 0 of B3
    if (k < 4 * 64 * 8 && (k / 8) % 32 != 0) pk[16 * 64 * 8 + k] = 0;
    if (k < MLP_NPARAM) pack_param(k, th[k], pk);
}

// A wave's partial sums: the parameters' gradients, then the loss, in rows of
// whole 128-byte lines.
constexpr int PART_STRIDE = (MLP_NPARAM + 1 + 31) / 32 * 32;

// Gradients of sum_i (y_i - t_i)^2 / n, one partial row per wave. Each tile
// keeps the activations' derivatives (and h1 in LDS, h2 in registers) from
// the forward pass. 16,384 rows: 34.6 us before, 19 us now.
__global__ __launch_bounds__(64 * MWAVES) void k_mlp_grad(const float *__restrict__ th, const short *__restrict__ pk,
                                                         const float *__restrict__ X, const float *__restrict__ T,
                                                         unsigned n, float *__restrict__ partial) {
    __shared__ short sm[MWAVES][32 * SP];  // h1
    __shared__ short sd[MWAVES][32 * SP];  // h2, then dz2, then dz1
    __shared__ float xf[MWAVES][32 * MLP_XSTRIDE];
    __shared__ float sy[MWAVES][32];
    __shared__ uint4 W[PACK_GROUPS * 64];
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 31, g = lane >> 5;
    for (int k = threadIdx.x; k < PACK_GROUPS * 64; k += 64 * MWAVES) W[k] = reinterpret_cast<const uint4 *>(pk)[k];
    // group c of the packed weights, read where a tile needs it: the
    // registers are full of sums
    union Group {
        uint4 u;
        bf16x4 b[2];
    };
    auto group = [&](int c) {
        Group a;
        a.u = W[c * 64 + lane];
        return a;
    };
    float w1[2][MLP_NIN], b1[2], b2[2], w3[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int k = 0; k < MLP_NIN; k++) w1[h][k] = th[MLP_OFF_W1 + k * 64 + 32 * h + r];
        b1[h] = th[MLP_OFF_B1 + 32 * h + r];
        b2[h] = th[MLP_OFF_B2 + 32 * h + r];
        w3[h] = th[MLP_OFF_W3 + 32 * h + r];
    }
    const float b3 = th[MLP_OFF_B3];
    f32x16 gW2[2][2], gW1[2];
    gW2[0][0] = gW2[0][1] = gW2[1][0] = gW2[1][1] = gW1[0] = gW1[1] = zero16();
    float gW3[2] = {0.f, 0.f}, gb1[2] = {0.f, 0.f}, gb2[2] = {0.f, 0.f}, gb3 = 0.f, L = 0.f;
    const float invn = 1.0f / (float)n;
    short *S = sm[wid], *D = sd[wid];
    float *XF = xf[wid], *SY = sy[wid];
    __syncthreads();
    const unsigned ntiles = (n + 31u) / 32u;
    for (unsigned tile = blockIdx.x * MWAVES + wid; tile < ntiles; tile += gridDim.x * MWAVES) {
        const unsigned row0 = tile * 32u;
        {
            const unsigned row = row0 + (unsigned)r;
            float4 xv = make_float4(0.f, 0.f, 0.f, 0.f);
            if (row < n) xv = *reinterpret_cast<const float4 *>(X + (size_t)row * MLP_XSTRIDE + 4 * g);
            *reinterpret_cast<float4 *>(XF + r * MLP_XSTRIDE + 4 * g) = xv;
        }
        wave_sync();
        // layer 1 (FP32): h1 to S, the activation's derivative kept
        f32x16 d1a, d1b, d2a, d2b, h2a, h2b;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const float *xr = XF + crow(e, g) * MLP_XSTRIDE;
            float a = 0.f, b = 0.f;
#pragma unroll
            for (int k = 0; k < MLP_NIN; k++) {
                a += xr[k] * w1[0][k];
                b += xr[k] * w1[1][k];
            }
            a += b1[0];
            b += b1[1];
            const float sa = sigm(a), sb = sigm(b);
            S[crow(e, g) * SP + r] = f2bf(a * sa);
            S[crow(e, g) * SP + 32 + r] = f2bf(b * sb);
            d1a[e] = sa * (1.0f + a * (1.0f - sa));
            d1b[e] = sb * (1.0f + b * (1.0f - sb));
        }
        wave_sync();
        h2a = zero16();
        h2b = zero16();
#pragma unroll
        for (int kc = 0; kc < 8; kc++) {
            const bf16x4 ak = *reinterpret_cast<const bf16x4 *>(S + r * SP + 8 * kc + 4 * g);
            const Group B2 = group(kc);
            h2a = mfma(ak, B2.b[0], h2a);
            h2b = mfma(ak, B2.b[1], h2b);
        }
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const float a = h2a[e] + b2[0], b = h2b[e] + b2[1];
            const float sa = sigm(a), sb = sigm(b);
            h2a[e] = a * sa;
            h2b[e] = b * sb;
            D[crow(e, g) * SP + r] = f2bf(h2a[e]);
            D[crow(e, g) * SP + 32 + r] = f2bf(h2b[e]);
            d2a[e] = sa * (1.0f + a * (1.0f - sa));
            d2b[e] = sb * (1.0f + b * (1.0f - sb));
        }
        wave_sync();
        f32x16 yv = zero16();
#pragma unroll
        for (int kc = 0; kc < 8; kc++) {
            const bf16x4 ak = *reinterpret_cast<const bf16x4 *>(D + r * SP + 8 * kc + 4 * g);
            yv = mfma(ak, group(16 + kc / 2).b[kc % 2], yv);
        }
        if (r == 0)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const unsigned row = row0 + crow(e, g);
                float d = 0.f;
                if (row < n) {
                    const float diff = (yv[e] + b3) - T[row];
                    L += diff * diff;
                    d = 2.0f * diff * invn;
                }
                SY[crow(e, g)] = d;
                gb3 += d;
            }
        wave_sync();
        // dW3, db2 and dz2 (into D)
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const float d = SY[crow(e, g)];
            const float dza = d * w3[0] * d2a[e];
            const float dzb = d * w3[1] * d2b[e];
            gW3[0] += h2a[e] * d;
            gW3[1] += h2b[e] * d;
            gb2[0] += dza;
            gb2[1] += dzb;
            D[crow(e, g) * SP + r] = f2bf(dza);
            D[crow(e, g) * SP + 32 + r] = f2bf(dzb);
        }
        wave_sync();
        // dW2 += h1^T dz2 (M = 64 inputs, N = 64 outputs, K = 32 rows)
#pragma unroll
        for (int kc = 0; kc < 4; kc++) {
            bf16x4 A0, A1, Bn0, Bn1;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int row = 8 * kc + 4 * g + j;
                A0[j] = S[row * SP + r];
                A1[j] = S[row * SP + 32 + r];
                Bn0[j] = D[row * SP + r];
                Bn1[j] = D[row * SP + 32 + r];
            }
            gW2[0][0] = mfma(A0, Bn0, gW2[0][0]);
            gW2[0][1] = mfma(A0, Bn1, gW2[0][1]);
            gW2[1][0] = mfma(A1, Bn0, gW2[1][0]);
            gW2[1][1] = mfma(A1, Bn1, gW2[1][1]);
        }
        // dh1 = dz2 W2^T (M = 32 rows, N = 64, K = 64)
        f32x16 dh0 = zero16(), dh1 = zero16();
#pragma unroll
        for (int kc = 0; kc < 8; kc++) {
            const bf16x4 ak = *reinterpret_cast<const bf16x4 *>(D + r * SP + 8 * kc + 4 * g);
            const Group B2T = group(8 + kc);
            dh0 = mfma(ak, B2T.b[0], dh0);
            dh1 = mfma(ak, B2T.b[1], dh1);
        }
        wave_sync();
        // dz1 (into D), db1
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const float da = dh0[e] * d1a[e];
            const float db = dh1[e] * d1b[e];
            gb1[0] += da;
            gb1[1] += db;
            D[crow(e, g) * SP + r] = f2bf(da);
            D[crow(e, g) * SP + 32 + r] = f2bf(db);
        }
        wave_sync();
        // dW1 += x^T dz1 (M = features, padded to 32; N = 64; K = 32 rows)
#pragma unroll
        for (int kc = 0; kc < 4; kc++) {
            bf16x4 A, Bn0, Bn1;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int row = 8 * kc + 4 * g + j;
                A[j] = (r < MLP_NIN) ? f2bf(XF[row * MLP_XSTRIDE + r]) : (short)0;
                Bn0[j] = D[row * SP + r];
                Bn1[j] = D[row * SP + 32 + r];
            }
            gW1[0] = mfma(A, Bn0, gW1[0]);
            gW1[1] = mfma(A, Bn1, gW1[1]);
        }
        wave_sync();
    }
    float *const P = partial + (size_t)(blockIdx.x * MWAVES + wid) * PART_STRIDE;
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int m = crow(e, g);
            if (m < MLP_NIN) P[MLP_OFF_W1 + m * 64 + 32 * h + r] = gW1[h][e];
        }
#pragma unroll
    for (int mh = 0; mh < 2; mh++)
#pragma unroll
        for (int nh = 0; nh < 2; nh++)
#pragma unroll
            for (int e = 0; e < 16; e++) P[MLP_OFF_W2 + (32 * mh + crow(e, g)) * 64 + 32 * nh + r] = gW2[mh][nh][e];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const float v3 = gW3[h] + __shfl_xor(gW3[h], 32, 64);
        const float v1 = gb1[h] + __shfl_xor(gb1[h], 32, 64);
        const float v2 = gb2[h] + __shfl_xor(gb2[h], 32, 64);
        if (g == 0) {
            P[MLP_OFF_W3 + 32 * h + r] = v3;
            P[MLP_OFF_B1 + 32 * h + r] = v1;
            P[MLP_OFF_B2 + 32 * h + r] = v2;
        }
    }
    const float v3 = gb3 + __shfl_xor(gb3, 32, 64);
    const float l2 = L + __shfl_xor(L, 32, 64);
    if (lane == 0) {
        P[MLP_OFF_B3] = v3;
        P[MLP_NPARAM] = l2;
    }
}

// grad[k] = sum over waves of partial[w][k], one wave's after the other;
// loss = the same of the last column / n; with ADAM also the parameter update
// and its packed copy. A lane that loads what it adds takes 136 us for 512
// rows: here a block stages REDUCE_ROWS rows of 32 columns in LDS, 16 loads
// of every thread in flight, and 32 lanes add them from there, which is bound
// by the chain of dependent adds. 7.2 us for 512 rows, the update (5 us as
// a kernel of its own) included. Sums by block or by slices would be shorter
// (4.6 us) but add in another order.
constexpr int REDUCE_COLS = 32, REDUCE_ROWS = 512, REDUCE_THREADS = 1024;
struct AdamArgs {
    float *th, *m, *v;
    short *pk;
    float b1t, b2t, lr;
};
template <bool ADAM>
__global__ __launch_bounds__(REDUCE_THREADS) void k_mlp_grad_reduce(const float *__restrict__ partial, unsigned nparts,
                                                                   unsigned n, float *__restrict__ grad,
                                                                   float *__restrict__ loss, AdamArgs A) {
    constexpr unsigned STEP = REDUCE_THREADS / REDUCE_COLS, PER = REDUCE_ROWS / STEP;
    __shared__ float T[REDUCE_ROWS][REDUCE_COLS];
    const unsigned c = threadIdx.x % REDUCE_COLS, r0 = threadIdx.x / REDUCE_COLS;
    const unsigned k = blockIdx.x * REDUCE_COLS + c;
    float v[PER], s = 0.f;
    auto load = [&](unsigned w0) {
#pragma unroll
        for (unsigned q = 0; q < PER; q++) {
            const unsigned w = w0 + q * STEP + r0;
            v[q] = partial[(size_t)(w < nparts ? w : nparts - 1u) * PART_STRIDE + k];
        }
    };
    load(0);
    for (unsigned w0 = 0; w0 < nparts; w0 += REDUCE_ROWS) {
        if (w0) __syncthreads();
#pragma unroll
        for (unsigned q = 0; q < PER; q++) T[q * STEP + r0][c] = v[q];
        __syncthreads();
        if (w0 + REDUCE_ROWS < nparts) load(w0 + REDUCE_ROWS);
        if (r0 == 0) {
            const unsigned m = nparts - w0 < (unsigned)REDUCE_ROWS ? nparts - w0 : REDUCE_ROWS;
#pragma unroll 16
            for (unsigned w = 0; w < m; w++) s += T[w][c];
        }
    }
    if (r0 != 0 || k > (unsigned)MLP_NPARAM) return;
    if (k == (unsigned)MLP_NPARAM) {
        *loss = s / (float)n;
        return;
    }
    grad[k] = s;
    if (ADAM) {
        const float mk = 0.9f * A.m[k] + 0.1f * s;
        const float vk = 0.999f * A.v[k] + 0.001f * s * s;
        A.m[k] = mk;
        A.v[k] = vk;
        const float t = A.th[k] - A.lr * (mk / (1.0f - A.b1t)) / (sqrtf(vk / (1.0f - A.b2t)) + 1e-8f);
        A.th[k] = t;
        pack_param((int)k, t, A.pk);
    }
}

// dst row i = src row order[i] (rows of MLP_XSTRIDE floats and a target).
__global__ void k_gather_rows(const unsigned *__restrict__ order, size_t n, const float *__restrict__ x,
                              const float *__restrict__ t, float *__restrict__ xs, float *__restrict__ ts) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * n) return;
    const size_t row = i >> 1, src = order[row];
    reinterpret_cast<float4 *>(xs)[i] = reinterpret_cast<const float4 *>(x)[2 * src + (i & 1)];
    if ((i & 1) == 0) ts[row] = t[src];
}

static unsigned mlp_blocks(unsigned n) {
    const unsigned tiles = (n + 31u) / 32u;
    return std::max(1u, std::min(1024u, (tiles + MWAVES - 1) / MWAVES));
}

static unsigned grad_blocks(unsigned n) { return std::min(256u, mlp_blocks(n)); }

void mlp_forward(hipStream_t s, const float *theta, const float *x, unsigned n, float *y) {
    if (!n) return;
    k_mlp_fwd<<<mlp_blocks(n), 64 * MWAVES, 0, s>>>(theta, x, n, y);
    SPH_HIP(hipGetLastError());
}

void MLPTrainer::pack(hipStream_t s, const float *theta) {
    packed.reserve(PACK_WORDS);
    k_mlp_pack<<<(MLP_NPARAM + 255) / 256, 256, 0, s>>>(theta, packed.get());
    SPH_HIP(hipGetLastError());
}

void MLPTrainer::sums(hipStream_t s, const float *theta, const float *x, const float *t, unsigned n) {
    SPH_REQUIRE(n > 0, SPH_ERR_INVALID, "empty training batch");
    const unsigned blocks = grad_blocks(n);
    parts = blocks * MWAVES;
    partial.reserve((size_t)parts * PART_STRIDE);
    grad.reserve(MLP_NPARAM);
    loss.reserve(1);
    k_mlp_grad<<<blocks, 64 * MWAVES, 0, s>>>(theta, packed.get(), x, t, n, partial.get());
    SPH_HIP(hipGetLastError());
}

void MLPTrainer::loss_grad(hipStream_t s, const float *theta, const float *x, const float *t, unsigned n) {
    pack(s, theta);
    sums(s, theta, x, t, n);
    k_mlp_grad_reduce<false><<<PART_STRIDE / REDUCE_COLS, REDUCE_THREADS, 0, s>>>(partial.get(), parts, n, grad.get(),
                                                                                  loss.get(), AdamArgs{});
    SPH_HIP(hipGetLastError());
}

void MLPTrainer::start(hipStream_t s, const float *theta, unsigned n) {
    pack(s, theta);
    partial.reserve((size_t)grad_blocks(n) * MWAVES * PART_STRIDE);
    adam_m.reserve(MLP_NPARAM);
    adam_v.reserve(MLP_NPARAM);
    fill_u32(s, reinterpret_cast<unsigned *>(adam_m.get()), MLP_NPARAM, 0u);
    fill_u32(s, reinterpret_cast<unsigned *>(adam_v.get()), MLP_NPARAM, 0u);
}

void MLPTrainer::step(hipStream_t s, float *theta, const float *x, const float *t, unsigned n, int step, float lr) {
    sums(s, theta, x, t, n);
    const AdamArgs a{theta, adam_m.get(), adam_v.get(), packed.get(), (float)std::pow(0.9, step),
                     (float)std::pow(0.999, step), lr};
    k_mlp_grad_reduce<true><<<PART_STRIDE / REDUCE_COLS, REDUCE_THREADS, 0, s>>>(partial.get(), parts, n, grad.get(),
                                                                                 loss.get(), a);
    SPH_HIP(hipGetLastError());
}

}  // namespace sph

using namespace sph;

extern "C" {

int sph_mlp_num_params(void) { return MLP_NPARAM; }

int sph_mlp_forward(const float *theta, const float *x, size_t n, float *y) {
    return guarded([&] {
        SPH_REQUIRE(theta && x && y, SPH_ERR_INVALID, "null argument");
        require_device();
        if (!n) return;
        DBuf<float> dt, dx, dy;
        dt.reserve(MLP_NPARAM);
        dx.reserve(n * MLP_XSTRIDE);
        dy.reserve(n);
        SPH_HIP(hipMemcpy(dt.get(), theta, MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice));
        SPH_HIP(hipMemcpy(dx.get(), x, n * MLP_XSTRIDE * sizeof(float), hipMemcpyHostToDevice));
        mlp_forward(nullptr, dt.get(), dx.get(), (unsigned)n, dy.get());
        SPH_HIP(hipMemcpy(y, dy.get(), n * sizeof(float), hipMemcpyDeviceToHost));
    });
}

int sph_mlp_loss_grad(const float *theta, const float *x, const float *t, size_t n, float *grad, float *loss) {
    return guarded([&] {
        SPH_REQUIRE(theta && x && t && grad && loss && n > 0, SPH_ERR_INVALID, "bad arguments");
        require_device();
        DBuf<float> dt, dx, dtt;
        dt.reserve(MLP_NPARAM);
        dx.reserve(n * MLP_XSTRIDE);
        dtt.reserve(n);
        SPH_HIP(hipMemcpy(dt.get(), theta, MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice));
        SPH_HIP(hipMemcpy(dx.get(), x, n * MLP_XSTRIDE * sizeof(float), hipMemcpyHostToDevice));
        SPH_HIP(hipMemcpy(dtt.get(), t, n * sizeof(float), hipMemcpyHostToDevice));
        MLPTrainer tr;
        tr.loss_grad(nullptr, dt.get(), dx.get(), dtt.get(), (unsigned)n);
        SPH_HIP(hipMemcpy(grad, tr.grad.get(), MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost));
        SPH_HIP(hipMemcpy(loss, tr.loss.get(), sizeof(float), hipMemcpyDeviceToHost));
    });
}

int sph_mlp_train(float *theta, const float *x, const float *t, size_t n, int steps, int batch, double lr,
                  unsigned seed, float *loss_out) {
    return guarded([&] {
        SPH_REQUIRE(theta && x && t && n > 0 && steps >= 0 && batch > 0, SPH_ERR_INVALID, "bad arguments");
        require_device();
        // shuffled copy of the samples, gathered on the device; minibatches
        // are consecutive windows
        std::vector<unsigned> order(n);
        std::iota(order.begin(), order.end(), 0u);
        std::mt19937 rng(seed);
        std::shuffle(order.begin(), order.end(), rng);
        DBuf<float> dt, dx, dtt, ux, ut;
        DBuf<unsigned> dorder;
        dt.reserve(MLP_NPARAM);
        dx.reserve(n * MLP_XSTRIDE);
        dtt.reserve(n);
        ux.reserve(n * MLP_XSTRIDE);
        ut.reserve(n);
        dorder.reserve(n);
        SPH_HIP(hipMemcpy(dt.get(), theta, MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice));
        SPH_HIP(hipMemcpy(ux.get(), x, n * MLP_XSTRIDE * sizeof(float), hipMemcpyHostToDevice));
        SPH_HIP(hipMemcpy(ut.get(), t, n * sizeof(float), hipMemcpyHostToDevice));
        SPH_HIP(hipMemcpy(dorder.get(), order.data(), n * sizeof(unsigned), hipMemcpyHostToDevice));
        k_gather_rows<<<nblocks(2 * n), BLOCK>>>(dorder.get(), n, ux.get(), ut.get(), dx.get(), dtt.get());
        SPH_HIP(hipGetLastError());
        MLPTrainer tr;
        tr.start(nullptr, dt.get(), (unsigned)n);
        const size_t b = std::min<size_t>((size_t)batch, n);
        const size_t nbatches = std::max<size_t>(1, n / b);
        for (int it = 0; it < steps; it++) {
            const size_t o = (size_t)(it % nbatches) * b;
            tr.step(nullptr, dt.get(), dx.get() + o * MLP_XSTRIDE, dtt.get() + o, (unsigned)b, it + 1, (float)lr);
        }
        tr.loss_grad(nullptr, dt.get(), dx.get(), dtt.get(), (unsigned)n);
        SPH_HIP(hipMemcpy(theta, dt.get(), MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost));
        if (loss_out) SPH_HIP(hipMemcpy(loss_out, tr.loss.get(), sizeof(float), hipMemcpyDeviceToHost));
    });
}

}  // extern "C"
