// Shared device / host helpers of the gfx950 hot path.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstring>

#include "../../include/sponge_amd.h"

namespace sa {

constexpr int kWave = 64;  // CDNA wavefront

// LTMatrix3 {a11, a21, a22, a31, a32, a33} (SPONGE/utils/vector.hpp:245-252)
struct LT6 {
    float a11, a21, a22, a31, a32, a33;
};

inline LT6 lt_from(const float* p) { return {p[0], p[1], p[2], p[3], p[4], p[5]}; }

inline bool lt_is_orthorhombic(const LT6& c) {
    return c.a21 == 0.0f && c.a31 == 0.0f && c.a32 == 0.0f;
}

#define SA_CHECK(expr)                                          \
    do {                                                        \
        hipError_t sa_err_ = (expr);                            \
        if (sa_err_ != hipSuccess) return (int)sa_err_;         \
    } while (0)

#define SA_LAUNCH_CHECK() SA_CHECK(hipGetLastError())

template <typename T>
inline int dmalloc(T** p, size_t n) {
    *p = nullptr;
    if (n == 0) n = 1;
    hipError_t e = hipMalloc((void**)p, n * sizeof(T));
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
        return SPONGE_AMD_ERROR_MALLOC_FAILED;
    }
    return 0;
}

template <typename T>
inline void dfree(T*& p) {
    if (p) (void)hipFree((void*)p);
    p = nullptr;
}

inline int grid_for(long long n, int block) { return (int)((n + block - 1) / block); }

// Minimum-image displacement a - b in the exact operation order of the
// reference's Get_Displacement<Periodic> (SPONGE/utils/boundary.h:22-31):
// dr - floorf(dr * rcell + 0.5f) * cell, with VECTOR * LTMatrix3 =
// {x a11 + y a21 + z a31, y a22 + z a32, z a33}.  FMA contraction is off so
// the neighbor-list criterion is reproduced bit for bit.
template <bool ORTHO>
__device__ __forceinline__ float3 disp_pbc(float3 a, float3 b, const LT6& c, const LT6& r) {
#pragma clang fp contract(off)
    float dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
    float3 o;
    if (ORTHO) {
        // the zero off-diagonal products of the general form add exact zeros
        float sx = floorf(dx * r.a11 + 0.5f);
        float sy = floorf(dy * r.a22 + 0.5f);
        float sz = floorf(dz * r.a33 + 0.5f);
        o.x = dx - sx * c.a11;
        o.y = dy - sy * c.a22;
        o.z = dz - sz * c.a33;
    } else {
        float sx = floorf(dx * r.a11 + dy * r.a21 + dz * r.a31 + 0.5f);
        float sy = floorf(dy * r.a22 + dz * r.a32 + 0.5f);
        float sz = floorf(dz * r.a33 + 0.5f);
        o.x = dx - (sx * c.a11 + sy * c.a21 + sz * c.a31);
        o.y = dy - (sy * c.a22 + sz * c.a32);
        o.z = dz - sz * c.a33;
    }
    return o;
}

// The periodic image of x nearest the point C (orthorhombic box).
__device__ __forceinline__ float3 near_image(float3 x, float3 C, const LT6& c, const LT6& r) {
    return make_float3(x.x - c.a11 * rintf((x.x - C.x) * r.a11),
                       x.y - c.a22 * rintf((x.y - C.y) * r.a22),
                       x.z - c.a33 * rintf((x.z - C.z) * r.a33));
}

// A cell's centre C on one axis of the box, moved by at most 1/32 to L - k / 16
// so that C and C - L are both exact, and the image of x nearest to it,
// relative to it: (x - n L) - C for n >= 0, (x - (n + 1) L) - (C - L) below, one
// rounding near zero for an x inside the box, where x + L would round to the
// box's precision (in a 35 A box that made the direct Coulomb forces an eighth
// less exact than the minimum image's).
__device__ __forceinline__ float image_centre(float mid, float L) {
    return L - rintf(16.f * (L - mid)) * 0.0625f;
}
__device__ __forceinline__ float image_offset(float x, float C, float L, float rL) {
    const float n = rintf((x - C) * rL);
    const float m = __builtin_amdgcn_fmed3f(n, -1.f, 0.f);  // the box taken off C
    return fmaf(m - n, L, x) - fmaf(m, L, C);
}
// the distance C may be moved by, with room for rounding
constexpr float kCentreMargin = 0.05f;
__device__ __forceinline__ float3 image_centre(float3 mid, const LT6& c) {
    return make_float3(image_centre(mid.x, c.a11), image_centre(mid.y, c.a22), image_centre(mid.z, c.a33));
}
__device__ __forceinline__ float3 image_offset(float3 x, float3 C, const LT6& c, const LT6& r) {
    return make_float3(image_offset(x.x, C.x, c.a11, r.a11), image_offset(x.y, C.y, c.a22, r.a22),
                       image_offset(x.z, C.z, c.a33, r.a33));
}

// r^2 as the reference's VECTOR dot product ((x*x + y*y) + z*z), no FMA.
__device__ __forceinline__ float norm2_exact(float3 d) {
#pragma clang fp contract(off)
    return d.x * d.x + d.y * d.y + d.z * d.z;
}

__device__ __forceinline__ int lane_id() { return __lane_id(); }

// LDS written by one lane of the wavefront is read by another: its LDS
// operations complete in order, so this only stops the compiler from moving
// them past each other.
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// number of set bits of mask in lanes below this one
__device__ __forceinline__ int lanes_below(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, kWave));
    return v;
}

// Scaled complementary error function erfcx(x) = exp(x^2) erfc(x) on
// 0 <= x <= kErfcxMax, as t P(t) with t = 1 / (1 + 0.4 x) and P of degree 7,
// coefficients fitted by iteratively reweighted least squares to minimise the
// largest relative error (2.9e-8 for the fit in FP64, under 4e-7 evaluated in
// FP32; generator and pins: tests/golden/make_erfcx_fit.py,
// tests/test_erfcx_fit.py).  The Ewald direct term then needs one
// exponential, exp(-x^2), for both erfc(x) and its derivative.  The rcp is the
// hardware reciprocal (1 ulp).
constexpr float kErfcxMax = 4.5f;
constexpr float kErfcxT = 0.4f;  // t = 1 / (1 + kErfcxT x)
// erfcx from t itself (callers that form t = 1 / (1 + kErfcxT x) their own way)
__device__ __forceinline__ float erfcx_poly_t(float t) {
    float p = 7.614902268e-02f;
    p = fmaf(p, t, -4.040216792e-01f);
    p = fmaf(p, t, 7.048484256e-01f);
    p = fmaf(p, t, -3.981623732e-01f);
    p = fmaf(p, t, 4.256499008e-01f);
    p = fmaf(p, t, 1.327632050e-01f);
    p = fmaf(p, t, 2.379624228e-01f);
    p = fmaf(p, t, 2.248110469e-01f);
    return p * t;
}
__device__ __forceinline__ float erfcx_poly(float x) {
    return erfcx_poly_t(__builtin_amdgcn_rcpf(1.0f + kErfcxT * x));
}

// Ewald direct force bracket B(x) = erfc(x) + 2 x / sqrt(pi) exp(-x^2), x = beta
// r: the force factor of a pair is qq B / r^3.  B = p(s)^2 with a polynomial p of
// degree 14 in s = 2 x / kBracketXMax - 1 on 0 <= x <= kBracketXMax, highest
// power first: neither an exponential nor a reciprocal beside 1/r, and no
// difference of nearly equal numbers where B falls to 8e-4.  (1/r^3 minus a
// polynomial in r^2 was 1.2e-4 of a pair's force off near the cutoff, against
// 3.4e-6, in the same time; direct Coulomb forces of 4,143 atoms at 8 A are 4.4e-7 from
// 64 bits, 5.9e-7 so, 4.3e-7 with the erfcx form, which takes a step of 95,000
// atoms 2 % longer.)  Generator and pins: tests/golden/make_ewald_bracket_fit.py,
// tests/test_ewald_bracket_fit.py.
constexpr float kBracketXMax = 2.91547595f;
constexpr int kBracketDegree = 14;
constexpr float kBracket[kBracketDegree + 1] = {
    7.479681517e-04f, 2.240266185e-04f, -3.764042864e-03f, -1.395790488e-03f, 9.287165478e-03f,
    1.515761670e-02f, -5.182155594e-02f, -2.190603316e-02f, 2.106313556e-01f, -1.537583619e-01f,
    -3.431663215e-01f, 5.348452926e-01f, 2.058848590e-01f, -8.598744273e-01f, 4.854928851e-01f};

// B(beta r) of r.  scale = 0: beta * cutoff lies beyond the fit (an Ewald
// tolerance below about 4e-6 at 10 A) and the callers take the erfcx form.
struct EwaldBracket {
    float scale;
    __device__ __forceinline__ float operator()(float r) const {
        const float s = fmaf(r, scale, -1.0f);
        float p = kBracket[0];
#pragma unroll
        for (int k = 1; k <= kBracketDegree; ++k) p = fmaf(p, s, kBracket[k]);
        return p * p;
    }
};

inline EwaldBracket ewald_bracket(float beta, float cutoff) {
    const double x = (double)beta * cutoff;
    return {x <= (double)kBracketXMax ? (float)(2.0 * beta / (double)kBracketXMax) : 0.f};
}

// Reciprocal part of an Ewald pair's force factor, qq beta^3 H(beta^2 r^2) with
// H(z) = (erf x - 2/sqrt(pi) x e^{-x^2}) / x^3, z = x^2 (the learned form's pair
// field), without an exponential and with nothing to cancel at small r.
// Polynomial of degree 12 in s = 2 z / kEwaldZMax - 1 on 0 <= z <= kEwaldZMax,
// highest power first.  Its error in FP64 is below 9e-9 beyond z = 2 and below
// 7e-9 of 3 / x^3 nearer (relative to H, at the splitting of a 10 A cutoff: 6e-7
// at 1 A, 1e-6 at 0.5 A; generator and pins: tests/golden/make_ewald_force_fit.py,
// tests/test_ewald_force_fit.py).
constexpr float kEwaldZMax = 8.5f;
constexpr int kEwaldDegree = 12;
constexpr float kEwaldForce[kEwaldDegree + 1] = {
    1.267232437e-04f, -4.884292139e-04f, 1.131965197e-03f, -2.847726457e-03f, 7.243126165e-03f,
    -1.631908305e-02f, 3.275954351e-02f, -5.882190540e-02f, 9.326564521e-02f, -1.286694109e-01f,
    1.518190950e-01f, -1.488173455e-01f, 1.099418998e-01f};

// beta^3 H(beta^2 r^2) as a polynomial of r^2: beta^3 folded into the
// coefficients, s = r^2 scale - 1.  scale = 0: beta * cutoff lies beyond the
// fit and the caller takes erff and exp.
struct EwaldPoly {
    float c[kEwaldDegree + 1];
    float scale;
    __device__ __forceinline__ float operator()(float r2) const {
        const float s = fmaf(r2, scale, -1.0f);
        float p = c[0];
#pragma unroll
        for (int k = 1; k <= kEwaldDegree; ++k) p = fmaf(p, s, c[k]);
        return p;
    }
};

inline EwaldPoly ewald_poly(float beta, float cutoff) {
    EwaldPoly e{};
    const double x = (double)beta * cutoff, b3 = (double)beta * beta * beta;
    for (int k = 0; k <= kEwaldDegree; ++k) e.c[k] = (float)(b3 * (double)kEwaldForce[k]);
    if (x * x <= (double)kEwaldZMax) e.scale = (float)(2.0 * beta * beta / (double)kEwaldZMax);
    return e;
}

// Lower-triangle packed pair index (Get_LJ_Type, Lennard_Jones_force.h:17-28):
// max(a,b) * (max(a,b)+1) / 2 + min(a,b).
__host__ __device__ __forceinline__ int lj_pair_index(int a, int b) {
    int hi = a > b ? a : b, lo = a > b ? b : a;
    return (hi * (hi + 1) >> 1) + lo;
}

// Fill kernel used instead of hipMemsetAsync so every step can be captured
// in a HIP graph.
template <typename T>
__global__ void k_fill(T* p, T v, long long n) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

template <typename T>
inline int fill_async(T* p, T v, long long n, hipStream_t s) {
    if (n <= 0) return 0;
    int blocks = grid_for(n, 256);
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_fill<T>, dim3(blocks), dim3(256), 0, s, p, v, n);
    SA_LAUNCH_CHECK();
    return 0;
}

// Smallest float t with sqrtf(t) >= rc: for r2 >= 0, (sqrtf(r2) < rc) <=>
// (r2 < t).  sqrtf is correctly rounded and monotone, so this reproduces the
// reference's strict "dr_abs < cutoff" test on r2 without a square root.
inline float sqrt_threshold(float rc) {
    float t = rc * rc;
    // walk to the boundary; a few ulps at most
    for (int it = 0; it < 64 && std::sqrt(t) >= rc; ++it) t = std::nextafter(t, 0.0f);
    for (int it = 0; it < 64 && std::sqrt(t) < rc; ++it) t = std::nextafter(t, 1e30f);
    return t;
}

}  // namespace sa
