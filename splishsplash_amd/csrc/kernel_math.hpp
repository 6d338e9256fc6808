// kernel_math.hpp -- device evaluation of the cubic-spline SPH kernel with
// the semantics of PrecomputedKernel<CubicKernel, 10000>
// (SPlisHSPlasH/SPHKernels.h:614-691):
//
//   W(r)     = 0.5 (T[p] + T[p+1]),            T[i] = W_cubic(i s)
//   gradW(r) = 0.5 (G[p] + G[p+1]) r,          G[i] = dW_cubic/dx(i s) / (i s)
//   p        = min(floor(|r| / s), 9998),      s = h / 9999
//
// The table entries are evaluated in closed form from q = i / 9999 instead of
// being read from memory, so the sweeps spend no bandwidth on the table. The
// index p is taken from an FP32 distance; when |r|/s lies close enough to an
// integer that the FP32 value could round to the other side of the step, p
// is recomputed from the FP64 distance of the original FP32 coordinates --
// the value an FP64 build computes from the same positions.
#pragma once
#include <hip/hip_runtime.h>

namespace sph {

struct KernelConst {
    float h, h2;        // support radius, h*h (float)
    float invStep_f;    // 9999 / h
    float k, l;         // 8/(pi h^3), 48/(pi h^3)
    float W0;           // W(0) = k
    float invH2;        // 1 / h^2
    float lh2;          // l / h^2
    float stepq;        // 1 / 9999
    double invStep_d;   // 1 / (h / 9999) in double, as the reference computes it
    double invStep2_d;  // invStep_d^2
    double h_d;
    float band;         // half-width of the FP64 band of table_step, per step
    float G0;           // the gradient entry of step 0: 0.5 (G[0] + G[1]) with G[0] = 0
};

KernelConst make_kernel_const(double h);

constexpr unsigned KRES = 10000u;

// The table average 0.5 (T[p] + T[p+1]) is evaluated as the smooth kernel
// at the step midpoint q = (p + 1/2) s / h: both W and G = W'(r)/r are C1
// across q = 1/2 and smooth on each side, so the two differ by
// f'' s^2 / 8, about 1e-8 of the value for s = h / 9999. G[0] = 0 (the
// reference's special case at r = 0) is kept exactly.
//
// Steps are floats (exact integers). A step past the table (9999 and up)
// stands for a pair outside the support: 1 - q is clamped to zero, which the
// subtraction does by itself, and both outer pieces vanish.
__device__ __forceinline__ float table_f(float q) { return __builtin_amdgcn_fmed3f(1.0f - q, 0.0f, 1.0f); }
__device__ __forceinline__ float table_W_avg(float p, const KernelConst &K) {
    const float q = fmaf(p, K.stepq, 0.5f * K.stepq);
    const float q2 = q * q, f = table_f(q);
    const float inner = K.k * fmaf(6.0f * q2, q - 1.0f, 1.0f);  // 6 q^3 - 6 q^2 + 1
    const float outer = K.k * (2.0f * f * f * f);
    return (q <= 0.5f) ? inner : outer;
}
// Both pieces are evaluated and one is selected: the lanes of a wave take
// both sides of q = 1/2, so a branch would run both anyway.
__device__ __forceinline__ float table_G_past0(float p, const KernelConst &K) {
    const float q = fmaf(p, K.stepq, 0.5f * K.stepq);
    const float f = table_f(q);
    const float inner = K.lh2 * fmaf(3.0f, q, -2.0f);
    const float outer = -K.lh2 * f * f * __builtin_amdgcn_rcpf(q);
    return (q <= 0.5f) ? inner : outer;
}
__device__ __forceinline__ float table_G_avg(float p, const KernelConst &K) {
    return p == 0.0f ? K.G0 : table_G_past0(p, K);
}

__device__ __forceinline__ float sqn(float x, float y, float z) { return (x * x + y * y) + z * z; }
// |r|^2 for the kernel evaluations, with fused multiply-adds (fewer
// roundings than sqn; the neighbour lists decide membership with sqn, the
// FP32 expression of the reference's float build).
__device__ __forceinline__ float sqn_fma(float x, float y, float z) { return fmaf(z, z, fmaf(y, y, x * x)); }

// Table step of the pair (xi, xj) with FP32 squared distance d2. With
// u = 2^-24 the FP32 value t = |r| / s is within 5.5 u t plus the rounding of
// the factor 1 / s of the FP64 one: coordinate differences, squares and sums
// are at most 5 u on d2, with or without fused multiply-adds, halved by the
// square root; the root itself is good to one ulp (2 u), the product to u.
// Inside a band K.band t of that width (3.3e-7 to 3.9e-7) around an integer
// m the step is decided in FP64 from the original FP32
// coordinates: floor(|r| / s) >= m  <=>  |r|^2 / s^2 >= m^2, which is what an
// FP64 build computes from the same positions up to its last-bit rounding.
// A wave takes that path for about every third pair (a lane in 150), 12 % of
// k_jacobi's time.
// The band around the last entry also decides the support: d2 <= h^2 differs
// from t <= 9999 by less than the band, so only there the two are compared
// (inside: at most step 9998; outside: 9999), and everywhere else floor(t)
// says it. Against a test and a select per pair on top of an integer step
// with its clamp and conversions: 12 % fewer vector instructions in k_accel
// (1.71e7 for 1.94e7 a launch at 1M particles), which the gathering sweeps
// hardly notice (1-2 %) and the tiled ones, bound by them, do.
__device__ __forceinline__ float table_step(const float4 &xi, const float4 &xj, float d2, const KernelConst &K) {
    const float t = __builtin_amdgcn_sqrtf(d2) * K.invStep_f;
    float p = floorf(t);
    const float m = rintf(t);
    if (fabsf(t - m) < fmaf(K.band, t, 2.0e-6f)) {
        const double dx = (double)xi.x - (double)xj.x;
        const double dy = (double)xi.y - (double)xj.y;
        const double dz = (double)xi.z - (double)xj.z;
        const double d2d = __dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz));
        const double md = (double)m;
        p = (__dmul_rn(d2d, K.invStep2_d) >= md * md) ? m : m - 1.0f;
        p = (d2 <= K.h2) ? fminf(p, (float)(KRES - 2u)) : (float)(KRES - 1u);
    }
    return p;
}

// W(xi - xj); zero outside the support.
__device__ __forceinline__ float kernel_W(const float4 &xi, const float4 &xj, const KernelConst &K) {
    const float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
    return table_W_avg(table_step(xi, xj, sqn_fma(dx, dy, dz), K), K);
}

// Scalar g with gradW(xi - xj) = g (xi - xj); zero outside the support.
// Also returns r = xi - xj.
__device__ __forceinline__ float kernel_G(const float4 &xi, const float4 &xj, const KernelConst &K, float3 &r) {
    r = make_float3(xi.x - xj.x, xi.y - xj.y, xi.z - xj.z);
    return table_G_avg(table_step(xi, xj, sqn_fma(r.x, r.y, r.z), K), K);
}

// kernel_G of N neighbours; whether any pair is within the first step is
// asked once for all.
template <unsigned N>
__device__ __forceinline__ void kernel_Gs(const float4 &xi, const float4 *xj, const KernelConst &K, float3 *r, float *g) {
    float p[N], p0 = (float)KRES;
#pragma unroll
    for (unsigned q = 0; q < N; q++) {
        r[q] = make_float3(xi.x - xj[q].x, xi.y - xj[q].y, xi.z - xj[q].z);
        p[q] = table_step(xi, xj[q], sqn_fma(r[q].x, r[q].y, r[q].z), K);
        g[q] = table_G_past0(p[q], K);
        p0 = fminf(p0, p[q]);
    }
    if (__builtin_expect(p0 == 0.0f, 0)) {
#pragma unroll
        for (unsigned q = 0; q < N; q++)
            if (p[q] == 0.0f) g[q] = K.G0;
    }
}

// Both W and the gradient scalar for one pair.
__device__ __forceinline__ void kernel_WG(const float4 &xi, const float4 &xj, const KernelConst &K, float3 &r, float &w,
                                          float &g) {
    r = make_float3(xi.x - xj.x, xi.y - xj.y, xi.z - xj.z);
    const float p = table_step(xi, xj, sqn_fma(r.x, r.y, r.z), K);
    w = table_W_avg(p, K);
    g = table_G_avg(p, K);
}

__device__ __forceinline__ float dot3(const float3 &a, const float3 &b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }

// Cubic spline W(r) for a scalar distance, double (SPHKernels.h:36-54).
__device__ __forceinline__ double cubic_W_d(double r, double h, double k) {
    const double q = r / h;
    if (q <= 1.0) {
        if (q <= 0.5) {
            const double q2 = q * q;
            return k * (6.0 * (q2 * q) - 6.0 * q2 + 1.0);
        }
        const double f = 1.0 - q;
        return k * (2.0 * (f * f * f));
    }
    return 0.0;
}

}  // namespace sph
