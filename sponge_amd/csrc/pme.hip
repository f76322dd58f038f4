// PME reciprocal part and excluded-pair correction for gfx950.
//
// Reference: SPONGE/PM_force/PM_force.cpp.
//   Initial          :295-654   beta, grid, B-spline moduli, BC / virial_BC
//   PME_Atom_Near    :699-762   fractional coordinates, base point u, f
//   PME_Q_Spread     :765-814   order-4 cardinal B-spline charge spreading
//   R2C, PME_Sum_Virial, PME_BCFQ, C2R   :1102-1125
//   PME_Final        :829-893   force gather, device_add_force :1014-1022
//   energies         :1142-1166
//   MPI_PME_Excluded_Force_With_Atom_Energy_Correction :1745-1817
//
// The 3D FFT is our own: five passes over lines.  A line length with two
// factors up to 16 (every length up to 120, and most beyond) is transformed in
// registers with one exchange through LDS (fft_small.h); other lengths take an
// LDS-staged mixed-radix (4,2,3,5,7) Stockham transform.  The complex half
// spectrum is kept as [kz][x][y] so every pass reads and writes whole 128-byte
// segments:
//   z-R2C (two real lines per complex transform) -> y-FFT ->
//   x-FFT + BC multiply + energy / virial sums + inverse x-FFT ->
//   inverse y-FFT -> z-C2R (two real lines per complex transform).
// The stencil indices of PME_Atom_Near are recomputed on the fly in spread
// and gather (they are a pure function of the coordinates), so no 64-int
// per-atom table is stored.
#include <algorithm>
#include <cmath>
#include <vector>

#include "internal.h"
#include "fft_small.h"
#include "batch_launch.h"
#include "timing.h"

using namespace sa;

namespace {

constexpr float kPI = 3.1415926f;                      // PM_force.cpp:17
constexpr float kTwoOverSqrtPi = 1.1283791670218446f;  // PM_force.cpp:19

__constant__ float cMa[4] = {(float)(1.0 / 6.0), -0.5f, 0.5f, (float)(-1.0 / 6.0)};
__constant__ float cMb[4] = {0.f, 0.5f, -1.f, 0.5f};
__constant__ float cMc[4] = {0.f, 0.5f, 0.f, -0.5f};
__constant__ float cMd[4] = {0.f, (float)(1.0 / 6.0), (float)(4.0 / 6.0), (float)(1.0 / 6.0)};

// ---------------------------------------------------------------------------
// Stockham transforms of line lengths without two factors up to 16

// One radix-R Stockham stage over nl lines of length n (line stride ld) held
// in LDS: out[(j/Ns)*Ns*R + j%Ns + r*Ns] = DFT_R(in[j + r*n/R] * w^(r*(j%Ns))).
template <int R, int SIGN>
__device__ __forceinline__ void stockham_stage(const float2* a, float2* b, int nl, int n, int ld,
                                               int Ns, const float2* __restrict__ tw) {
    const int nb = n / R;
    const int total = nl * nb;
    const int step = n / (Ns * R);
    for (int t = threadIdx.x; t < total; t += blockDim.x) {
        const int line = t / nb, j = t - line * nb;
        const float2* in = a + line * ld;
        float2* out = b + line * ld;
        float2 v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = in[j + r * nb];
        const int k = j % Ns;
#pragma unroll
        for (int r = 1; r < R; ++r) {
            float2 w = tw[r * k * step];
            if (SIGN > 0) w.y = -w.y;
            v[r] = cmul(v[r], w);
        }
        Dft<R, SIGN>::run(v);
        const int idx = (j / Ns) * Ns * R + k;
#pragma unroll
        for (int r = 0; r < R; ++r) out[idx + r * Ns] = v[r];
    }
}

// Transform nl lines in place (result returned; ping-pong between a and b).
// tw: the line length's twiddles, staged in LDS by the caller.
template <int SIGN>
__device__ __forceinline__ float2* fft_lines(float2* a, float2* b, int nl, int n, int ld, const sa_radix_plan& pl,
                             const float2* __restrict__ tw) {
    int Ns = 1;
    for (int s = 0; s < pl.nst; ++s) {
        const int R = pl.r[s];
        switch (R) {
            case 4: stockham_stage<4, SIGN>(a, b, nl, n, ld, Ns, tw); break;
            case 2: stockham_stage<2, SIGN>(a, b, nl, n, ld, Ns, tw); break;
            case 3: stockham_stage<3, SIGN>(a, b, nl, n, ld, Ns, tw); break;
            case 5: stockham_stage<5, SIGN>(a, b, nl, n, ld, Ns, tw); break;
            default: stockham_stage<7, SIGN>(a, b, nl, n, ld, Ns, tw); break;
        }
        __syncthreads();
        float2* t = a;
        a = b;
        b = t;
        Ns *= R;
    }
    return a;
}

constexpr int kMaxFftLen = 512;  // largest grid dimension (checked at init)

// brick of grid coordinate x on one axis (the last brick takes the remainder)
__device__ __forceinline__ int brick_of(int x, int B, int nbk) {
    const int h = x / B;
    return h < nbk ? h : nbk - 1;
}

// Tile geometry (host and device).  A tile is sized for the largest brick,
// m = B or the remainder brick: (mx + 3) x (my + 3) x (mz + 3) points, dense
// in global memory.  In LDS the z stride is 1, the y stride mz + 3 rounded up
// to 4 and the x stride is rounded up to 16 mod 32 floats, which puts the 64
// stencil offsets kx*sx + ky*sy + kz of one atom into distinct banks per half
// wavefront for mz = 8.
struct TileGeom {
    int tx, ty, tz;  // tile extent (points)
    int sy, sx;      // LDS strides (floats)
    __host__ __device__ int lds_floats() const { return tx * sx; }
    __host__ __device__ int points() const { return tx * ty * tz; }
};

// z pass, real -> half spectrum: block = (y block, x).  (Summing the spread's
// tiles here as the lines are read, without the reduce pass and the grid in
// memory, took 32 us at 96^3 against 5.4 for the reduce and 6 for this pass:
// its loads are guarded and scattered.)
__device__ __forceinline__ void fft_z_r2c_body(int sa_block, const float* __restrict__ Q,
                                                   float2* __restrict__ FQ, int fx, int fy, int fz,
                                                   int fzc, int TL, const sa_radix_plan& pl,
                                                   const float2* __restrict__ tw) {
    extern __shared__ float2 sm[];
    const int gy = (fy + TL - 1) / TL;  // y blocks per x line (1D grid: x-major)
    const int x = sa_block / gy, y0 = (sa_block - x * gy) * TL;
    const int nl = min(TL, fy - y0), npair = (nl + 1) >> 1;
    const float* src = Q + ((size_t)x * fy + y0) * fz;
    const float2* res;
    int ldz;
    if (pl.r1) {
        const int R1 = pl.r1, R2 = pl.r2, ld = R1 * (R2 + 1);
        float2* z = sm + ((TL + 1) >> 1) * ld;
        ldz = fz + 1;
        const float inv2 = __builtin_amdgcn_rcpf((float)R2), inv1 = __builtin_amdgcn_rcpf((float)R1);
        with_radix(R1, [&](auto radix) {
            constexpr int R = decltype(radix)::value;
            for (int t = threadIdx.x; t < npair * R2; t += blockDim.x) {
                const int m = div_small(t, inv2), n2 = t - m * R2;
                // an absent second line reads the first and counts as zero
                const bool has = 2 * m + 1 < nl;
                const float* q0 = src + (size_t)(2 * m) * fz + n2;
                const float* q1 = q0 + (has ? fz : 0);
                float2 v[R], w[R];
#pragma unroll
                for (int r = 0; r < R; ++r) v[r] = make_float2(q0[R2 * r], q1[R2 * r]);
#pragma unroll
                for (int k1 = 1; k1 < R; ++k1) w[k1] = tw[n2 * k1];
                if (!has)
#pragma unroll
                    for (int r = 0; r < R; ++r) v[r].y = 0.f;
                Dft<R, -1>::run(v);
                sm[m * ld + n2] = v[0];
#pragma unroll
                for (int k1 = 1; k1 < R; ++k1) sm[m * ld + k1 * (R2 + 1) + n2] = cmul(v[k1], w[k1]);
            }
        });
        __syncthreads();
        with_radix(R2, [&](auto radix) {
            constexpr int R = decltype(radix)::value;
            for (int t = threadIdx.x; t < npair * R1; t += blockDim.x) {
                const int m = div_small(t, inv1), k1 = t - m * R1;
                float2 v[R];
#pragma unroll
                for (int n2 = 0; n2 < R; ++n2) v[n2] = sm[m * ld + k1 * (R2 + 1) + n2];
                Dft<R, -1>::run(v);
#pragma unroll
                for (int k2 = 0; k2 < R; ++k2) z[m * ldz + k1 + R1 * k2] = v[k2];
            }
        });
        __syncthreads();
        res = z;
    } else {
        float2* a = sm;
        float2* b = sm + npair * fz;
        float2* stw = sm + 2 * ((TL + 1) >> 1) * fz;
        ldz = fz;
        for (int k = threadIdx.x; k < fz; k += blockDim.x) stw[k] = tw[k];
        for (int e = threadIdx.x; e < npair * fz; e += blockDim.x) {
            const int m = e / fz, zz = e - m * fz;
            const float v0 = src[(size_t)(2 * m) * fz + zz];
            const float v1 = (2 * m + 1 < nl) ? src[(size_t)(2 * m + 1) * fz + zz] : 0.f;
            a[e] = make_float2(v0, v1);
        }
        __syncthreads();
        res = fft_lines<-1>(a, b, npair, fz, fz, pl, stw);
    }
    for (int e = threadIdx.x; e < fzc * nl; e += blockDim.x) {
        const int kz = e / nl, l = e - kz * nl;
        const int m = l >> 1;
        const float2 Z = res[m * ldz + kz];
        const float2 Zm = res[m * ldz + (kz == 0 ? 0 : fz - kz)];
        float2 v;
        if ((l & 1) == 0) v = make_float2(0.5f * (Z.x + Zm.x), 0.5f * (Z.y - Zm.y));
        else v = make_float2(0.5f * (Z.y + Zm.y), -0.5f * (Z.x - Zm.x));
        FQ[((size_t)kz * fx + x) * fy + y0 + l] = v;
    }
}

__global__ void __launch_bounds__(128) k_fft_z_r2c(const float* __restrict__ Q,
                                                   float2* __restrict__ FQ, int fx, int fy, int fz,
                                                   int fzc, int TL, sa_radix_plan pl,
                                                   const float2* __restrict__ tw) {
    fft_z_r2c_body(blockIdx.x, Q, FQ, fx, fy, fz, fzc, TL, pl, tw);
}

// y pass over contiguous lines [kz][x][0..fy)
template <int SIGN>
__device__ __forceinline__ void fft_y_body(int sa_block, float2* __restrict__ FQ, int nlines, int fy, int TL,
                                               const sa_radix_plan& pl, const float2* __restrict__ tw) {
    extern __shared__ float2 sm[];
    const int l0 = sa_block * TL;
    const int nl = min(TL, nlines - l0);
    float2* base = FQ + (size_t)l0 * fy;
    if (pl.r1) {
        const int R1 = pl.r1, R2 = pl.r2, ld = R1 * (R2 + 1);
        const float inv2 = __builtin_amdgcn_rcpf((float)R2), inv1 = __builtin_amdgcn_rcpf((float)R1);
        with_radix(R1, [&](auto radix) {
            constexpr int R = decltype(radix)::value;
            for (int t = threadIdx.x; t < nl * R2; t += blockDim.x) {
                const int l = div_small(t, inv2), n2 = t - l * R2;
                float2 v[R], w[R];
#pragma unroll
                for (int r = 0; r < R; ++r) v[r] = base[l * fy + n2 + R2 * r];
#pragma unroll
                for (int k1 = 1; k1 < R; ++k1) w[k1] = tw[n2 * k1];
                Dft<R, SIGN>::run(v);
                sm[l * ld + n2] = v[0];
#pragma unroll
                for (int k1 = 1; k1 < R; ++k1)
                    sm[l * ld + k1 * (R2 + 1) + n2] =
                        cmul(v[k1], make_float2(w[k1].x, SIGN > 0 ? -w[k1].y : w[k1].y));
            }
        });
        __syncthreads();
        with_radix(R2, [&](auto radix) {
            constexpr int R = decltype(radix)::value;
            for (int t = threadIdx.x; t < nl * R1; t += blockDim.x) {
                const int l = div_small(t, inv1), k1 = t - l * R1;
                float2 v[R];
#pragma unroll
                for (int n2 = 0; n2 < R; ++n2) v[n2] = sm[l * ld + k1 * (R2 + 1) + n2];
                Dft<R, SIGN>::run(v);
#pragma unroll
                for (int k2 = 0; k2 < R; ++k2) base[l * fy + k1 + R1 * k2] = v[k2];
            }
        });
        return;
    }
    float2* a = sm;
    float2* b = sm + TL * fy;
    float2* stw = sm + 2 * TL * fy;
    for (int k = threadIdx.x; k < fy; k += blockDim.x) stw[k] = tw[k];
    for (int e = threadIdx.x; e < nl * fy; e += blockDim.x) a[e] = base[e];
    __syncthreads();
    const float2* res = fft_lines<SIGN>(a, b, nl, fy, fy, pl, stw);
    for (int e = threadIdx.x; e < nl * fy; e += blockDim.x) base[e] = res[e];
}

template <int SIGN>
__global__ void __launch_bounds__(256) k_fft_y(float2* __restrict__ FQ, int nlines, int fy, int TL,
                                               sa_radix_plan pl, const float2* __restrict__ tw) {
    fft_y_body<SIGN>(blockIdx.x, FQ, nlines, fy, TL, pl, tw);
}

// x pass with the reciprocal-space convolution: block = (y block, kz).
// acc[0] += sum w(kz) BC |F|^2 (w = 1 on kz = 0 and kz = fz/2 for even fz,
// 2 otherwise: the full-spectrum sum of the reference's real-space
// 0.5 * sum Q * FBCFQ, PM_force.cpp:896-919); acc[1..6] -= factor |F|^2
// virial_BC with factor 0.5 on kz = 0 and kz = fzc-1 (PME_Sum_Virial,
// :1024-1068, including its odd-fz weighting), virial_BC = BC / 2 (delta -
// 2 / m^2 (1 + pi^2 m^2 / beta^2) m m) evaluated from m (:589-604; six stored
// planes of it were 24 of the 32 bytes per point that an energy and virial
// evaluation read here).
// ACC: accumulate the energy (and, with need_virial, the virial) sums; off on
// force-only evaluations.  BCt is laid out [kz][kx][ky] (the spectrum's order
// at this pass).
struct ReciprocalGeom {
    LT6 rc;
    float pre;  // pi^2 / beta^2
};

// frequency index of a grid of n points (PM_force.cpp:553-565)
__device__ __forceinline__ float frequency(int k, int n) { return (float)(k > n / 2 ? k - n : k); }

// energy and virial terms of one point of the half spectrum
struct SpectrumSums {
    double e = 0.0;
    double v[6] = {0, 0, 0, 0, 0, 0};
    __device__ __forceinline__ void add(float2 F, float bc, int kx, int ky, int kz, int fx, int fy,
                                        double wE, float vfac, int need_virial,
                                        const ReciprocalGeom& rg) {
        const float mag = F.x * F.x + F.y * F.y;
        e += wE * (double)bc * (double)mag;
        if (!need_virial || bc == 0.f) return;
        // in double: 1 - t m m cancels, and the terms of a pass are few (1 us at
        // 84 x 90 x 38 points)
        const double x = frequency(kx, fx), y = frequency(ky, fy), z = kz;
        const double mx = x * rg.rc.a11;
        const double my = x * rg.rc.a21 + y * rg.rc.a22;
        const double mz = x * rg.rc.a31 + y * rg.rc.a32 + z * rg.rc.a33;
        const double msq = mx * mx + my * my + mz * mz;
        const double t = 2 / msq * (1 + rg.pre * msq);
        const double s = 0.5 * vfac * (double)bc * (double)mag;
        v[0] -= s * (1 - t * mx * mx);
        v[1] += s * (t * my * mx);
        v[2] -= s * (1 - t * my * my);
        v[3] += s * (t * mz * mx);
        v[4] += s * (t * mz * my);
        v[5] -= s * (1 - t * mz * mz);
    }
};

// A workgroup's sums to part[c][block] of n workgroups, added up by the gather
// (228 workgroups at 96 x 96 x 96 adding seven FP64 sums each to the same
// addresses took 17 of a 27 us pass).
__device__ __forceinline__ void store_sums(SpectrumSums& sums, int need_virial, double* __restrict__ part,
                                           int n, int block) {
    __shared__ double red[7][16];
    const double e = wave_sum(sums.e);
    if (need_virial)
        for (int c = 0; c < 6; ++c) sums.v[c] = wave_sum(sums.v[c]);
    const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    if (lane == 0) {
        red[0][w] = e;
        for (int c = 0; c < 6; ++c) red[1 + c][w] = sums.v[c];
    }
    __syncthreads();
    if (threadIdx.x < 7) {
        const int nw = blockDim.x / kWave;
        double t = 0;
        for (int k = 0; k < nw; ++k) t += red[threadIdx.x][k];
        part[(size_t)threadIdx.x * n + block] = t;
    }
}

template <bool ACC>
__device__ __forceinline__ void fft_x_conv_body(int sa_block, 
    float2* __restrict__ FQ, const float* __restrict__ BCt, const ReciprocalGeom& rg,
    int fx, int fy, int fz, int fzc, int TL, const sa_radix_plan& pl,
    const float2* __restrict__ tw, int need_virial, double* __restrict__ part) {
    extern __shared__ float2 sm[];
    const int gy = (fy + TL - 1) / TL;  // y blocks per kz plane (1D grid: kz-major)
    const int kz = sa_block / gy, y0 = (sa_block - kz * gy) * TL;
    const int nl = min(TL, fy - y0);
    const double wE = (kz == 0 || 2 * kz == fz) ? 1.0 : 2.0;
    const float vfac = (kz == 0 || kz == fzc - 1) ? 0.5f : 1.0f;
    SpectrumSums sums;
    float2* plane = FQ + (size_t)kz * fx * fy + y0;
    const float* bcp = BCt + (size_t)kz * fx * fy + y0;
    if (pl.r1) {
        // l runs fastest over the threads: loads and stores of TL adjacent
        // columns; the inverse transform is the mirrored decomposition, which
        // starts from the points a thread holds and ends on the ones it loaded
        const int R1 = pl.r1, R2 = pl.r2, ld = nl + 1;
        const float invl = __builtin_amdgcn_rcpf((float)nl);
        with_radix(R1, [&](auto radix) {
            constexpr int R = decltype(radix)::value;
            for (int t = threadIdx.x; t < nl * R2; t += blockDim.x) {
                const int n2 = div_small(t, invl), l = t - n2 * nl;
                float2 v[R], w[R];
#pragma unroll
                for (int r = 0; r < R; ++r) v[r] = plane[(size_t)(n2 + R2 * r) * fy + l];
#pragma unroll
                for (int k1 = 1; k1 < R; ++k1) w[k1] = tw[n2 * k1];
                Dft<R, -1>::run(v);
                sm[n2 * ld + l] = v[0];
#pragma unroll
                for (int k1 = 1; k1 < R; ++k1) sm[(k1 * R2 + n2) * ld + l] = cmul(v[k1], w[k1]);
            }
        });
        __syncthreads();
        with_radix(R2, [&](auto radix) {
            constexpr int R = decltype(radix)::value;
            for (int t = threadIdx.x; t < nl * R1; t += blockDim.x) {
                const int k1 = div_small(t, invl), l = t - k1 * nl;
                float bc[R];
#pragma unroll
                for (int k2 = 0; k2 < R; ++k2) bc[k2] = bcp[(size_t)(k1 + R1 * k2) * fy + l];
                float2 v[R], w[R];
#pragma unroll
                for (int n2 = 0; n2 < R; ++n2) v[n2] = sm[(k1 * R2 + n2) * ld + l];
#pragma unroll
                for (int n2 = 1; n2 < R; ++n2) w[n2] = tw[n2 * k1];
                Dft<R, -1>::run(v);
#pragma unroll
                for (int k2 = 0; k2 < R; ++k2) {
                    if (ACC)
                        sums.add(v[k2], bc[k2], k1 + R1 * k2, y0 + l, kz, fx, fy, wE, vfac,
                                 need_virial, rg);
                    v[k2] = make_float2(v[k2].x * bc[k2], v[k2].y * bc[k2]);
                }
                Dft<R, +1>::run(v);
                sm[(k1 * R2) * ld + l] = v[0];
#pragma unroll
                for (int n2 = 1; n2 < R; ++n2)
                    sm[(k1 * R2 + n2) * ld + l] = cmul(v[n2], make_float2(w[n2].x, -w[n2].y));
            }
        });
        __syncthreads();
        with_radix(R1, [&](auto radix) {
            constexpr int R = decltype(radix)::value;
            for (int t = threadIdx.x; t < nl * R2; t += blockDim.x) {
                const int n2 = div_small(t, invl), l = t - n2 * nl;
                float2 v[R];
#pragma unroll
                for (int k1 = 0; k1 < R; ++k1) v[k1] = sm[(k1 * R2 + n2) * ld + l];
                Dft<R, +1>::run(v);
#pragma unroll
                for (int n1 = 0; n1 < R; ++n1) plane[(size_t)(n2 + R2 * n1) * fy + l] = v[n1];
            }
        });
    } else {
        float2* a = sm;
        float2* b = sm + TL * fx;
        float2* stw = sm + 2 * TL * fx;
        for (int k = threadIdx.x; k < fx; k += blockDim.x) stw[k] = tw[k];
        for (int e = threadIdx.x; e < fx * nl; e += blockDim.x) {
            const int xi = e / nl, l = e - xi * nl;
            a[l * fx + xi] = plane[(size_t)xi * fy + l];
        }
        __syncthreads();
        float2* res = fft_lines<-1>(a, b, nl, fx, fx, pl, stw);
        float2* other = (res == a) ? b : a;
        for (int e = threadIdx.x; e < nl * fx; e += blockDim.x) {
            const int kx = e / nl, l = e - kx * nl;
            const float2 F = res[l * fx + kx];
            const float bc = bcp[(size_t)kx * fy + l];
            if (ACC) sums.add(F, bc, kx, y0 + l, kz, fx, fy, wE, vfac, need_virial, rg);
            res[l * fx + kx] = make_float2(F.x * bc, F.y * bc);
        }
        __syncthreads();
        const float2* out = fft_lines<+1>(res, other, nl, fx, fx, pl, stw);
        for (int e = threadIdx.x; e < fx * nl; e += blockDim.x) {
            const int xi = e / nl, l = e - xi * nl;
            plane[(size_t)xi * fy + l] = out[l * fx + xi];
        }
    }
    if (ACC) store_sums(sums, need_virial, part, gy * fzc, sa_block);
}

template <bool ACC>
__global__ void __launch_bounds__(256) k_fft_x_conv(
    float2* __restrict__ FQ, const float* __restrict__ BCt, ReciprocalGeom rg,
    int fx, int fy, int fz, int fzc, int TL, sa_radix_plan pl,
    const float2* __restrict__ tw, int need_virial, double* __restrict__ part) {
    fft_x_conv_body<ACC>(blockIdx.x, FQ, BCt, rg, fx, fy, fz, fzc, TL, pl, tw, need_virial, part);
}

// y pass, x pass with the convolution, and back, in one kernel: block = one kz
// plane, held in LDS.  The two factors of a line are transformed in place, so
// a line's frequencies stand at k1 R2 + k2 in place of k1 + R1 k2; the inverse
// runs the mirrored decomposition from there.  Global loads and stores are
// those of the first and the last transform, and the twiddles wait in LDS.  It
// takes the place of three launches whose time is the latency of their loads,
// stores and barriers: about 28 x 28 x 28, 3 x 3.6 -> 6.5 us (a step of 2,000
// atoms 64 -> 59 us), 54 x 54 x 54, 13.3 -> 8.8 us.  A plane is one
// workgroup's, and there are only fz / 2 + 1 of them: at 96 x 96 x 96 it takes
// 15 us against 14.4, so planes beyond kPlaneLds (64 x 64) keep the three
// passes, as do lengths without two factors.
template <bool ACC>
__device__ __forceinline__ void fft_plane_body(int sa_block, float2* __restrict__ FQ,
                                               const float* __restrict__ BCt, const ReciprocalGeom& rg,
                                               int fx, int fy, int fz, int fzc, const sa_radix_plan& px,
                                               const sa_radix_plan& py, const float2* __restrict__ twx,
                                               const float2* __restrict__ twy, int need_virial,
                                               double* __restrict__ part) {
    extern __shared__ float2 sm[];
    const int kz = sa_block;
    const double wE = (kz == 0 || 2 * kz == fz) ? 1.0 : 2.0;
    const float vfac = (kz == 0 || kz == fzc - 1) ? 0.5f : 1.0f;
    SpectrumSums sums;
    float2* plane = FQ + (size_t)kz * fx * fy;
    const float* bcp = BCt + (size_t)kz * fx * fy;
    const int X1 = px.r1, X2 = px.r2, Y1 = py.r1, Y2 = py.r2;
    const int ld = fy | 1;  // odd: lanes over x hit distinct banks
    const float inv_y2 = __builtin_amdgcn_rcpf((float)Y2), inv_fx = __builtin_amdgcn_rcpf((float)fx);
    const float inv_fy = __builtin_amdgcn_rcpf((float)fy);
    // the twiddles beside the plane: a later pass waits for LDS only
    float2* tx = sm + fx * ld;
    float2* ty = tx + fx;
    for (int k = threadIdx.x; k < fx + fy; k += blockDim.x) tx[k] = k < fx ? twx[k] : twy[k - fx];
    with_radix(Y1, [&](auto radix) {
        constexpr int R = decltype(radix)::value;
        for (int t = threadIdx.x; t < fx * Y2; t += blockDim.x) {
            const int x = div_small(t, inv_y2), n2 = t - x * Y2;
            float2 v[R], w[R];
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = plane[x * fy + n2 + Y2 * r];
#pragma unroll
            for (int k1 = 1; k1 < R; ++k1) w[k1] = twy[n2 * k1];
            Dft<R, -1>::run(v);
            sm[x * ld + n2] = v[0];
#pragma unroll
            for (int k1 = 1; k1 < R; ++k1) sm[x * ld + k1 * Y2 + n2] = cmul(v[k1], w[k1]);
        }
    });
    __syncthreads();
    with_radix(Y2, [&](auto radix) {
        constexpr int R = decltype(radix)::value;
        for (int t = threadIdx.x; t < fx * Y1; t += blockDim.x) {
            const int k1 = div_small(t, inv_fx), x = t - k1 * fx;
            float2* a = sm + x * ld + k1 * Y2;
            float2 v[R];
#pragma unroll
            for (int n2 = 0; n2 < R; ++n2) v[n2] = a[n2];
            Dft<R, -1>::run(v);
#pragma unroll
            for (int k2 = 0; k2 < R; ++k2) a[k2] = v[k2];
        }
    });
    __syncthreads();
    with_radix(X1, [&](auto radix) {
        constexpr int R = decltype(radix)::value;
        for (int t = threadIdx.x; t < fy * X2; t += blockDim.x) {
            const int n2 = div_small(t, inv_fy), q = t - n2 * fy;
            float2 v[R], w[R];
#pragma unroll
            for (int k1 = 1; k1 < R; ++k1) w[k1] = tx[n2 * k1];
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = sm[(n2 + X2 * r) * ld + q];
            Dft<R, -1>::run(v);
            sm[n2 * ld + q] = v[0];
#pragma unroll
            for (int k1 = 1; k1 < R; ++k1) sm[(k1 * X2 + n2) * ld + q] = cmul(v[k1], w[k1]);
        }
    });
    __syncthreads();
    with_radix(X2, [&](auto radix) {
        constexpr int R = decltype(radix)::value;
        for (int t = threadIdx.x; t < fy * X1; t += blockDim.x) {
            const int k1 = div_small(t, inv_fy), q = t - k1 * fy;
            const int qy = div_small(q, inv_y2), ky = qy + Y1 * (q - qy * Y2);
            float bc[R];
#pragma unroll
            for (int k2 = 0; k2 < R; ++k2) bc[k2] = bcp[(k1 + X1 * k2) * fy + ky];
            float2 v[R], w[R];
#pragma unroll
            for (int n2 = 1; n2 < R; ++n2) w[n2] = tx[n2 * k1];
#pragma unroll
            for (int n2 = 0; n2 < R; ++n2) v[n2] = sm[(k1 * X2 + n2) * ld + q];
            Dft<R, -1>::run(v);
#pragma unroll
            for (int k2 = 0; k2 < R; ++k2) {
                if (ACC)
                    sums.add(v[k2], bc[k2], k1 + X1 * k2, ky, kz, fx, fy, wE, vfac, need_virial, rg);
                v[k2] = make_float2(v[k2].x * bc[k2], v[k2].y * bc[k2]);
            }
            Dft<R, +1>::run(v);
            sm[(k1 * X2) * ld + q] = v[0];
#pragma unroll
            for (int n2 = 1; n2 < R; ++n2)
                sm[(k1 * X2 + n2) * ld + q] = cmul(v[n2], make_float2(w[n2].x, -w[n2].y));
        }
    });
    __syncthreads();
    with_radix(X1, [&](auto radix) {
        constexpr int R = decltype(radix)::value;
        for (int t = threadIdx.x; t < fy * X2; t += blockDim.x) {
            const int n2 = div_small(t, inv_fy), q = t - n2 * fy;
            float2 v[R];
#pragma unroll
            for (int k1 = 0; k1 < R; ++k1) v[k1] = sm[(k1 * X2 + n2) * ld + q];
            Dft<R, +1>::run(v);
#pragma unroll
            for (int n1 = 0; n1 < R; ++n1) sm[(n2 + X2 * n1) * ld + q] = v[n1];
        }
    });
    __syncthreads();
    with_radix(Y2, [&](auto radix) {
        constexpr int R = decltype(radix)::value;
        for (int t = threadIdx.x; t < fx * Y1; t += blockDim.x) {
            const int k1 = div_small(t, inv_fx), x = t - k1 * fx;
            float2* a = sm + x * ld + k1 * Y2;
            float2 v[R], w[R];
#pragma unroll
            for (int n2 = 1; n2 < R; ++n2) w[n2] = ty[n2 * k1];
#pragma unroll
            for (int k2 = 0; k2 < R; ++k2) v[k2] = a[k2];
            Dft<R, +1>::run(v);
            a[0] = v[0];
#pragma unroll
            for (int n2 = 1; n2 < R; ++n2) a[n2] = cmul(v[n2], make_float2(w[n2].x, -w[n2].y));
        }
    });
    __syncthreads();
    with_radix(Y1, [&](auto radix) {
        constexpr int R = decltype(radix)::value;
        for (int t = threadIdx.x; t < fx * Y2; t += blockDim.x) {
            const int x = div_small(t, inv_y2), n2 = t - x * Y2;
            float2 v[R];
#pragma unroll
            for (int k1 = 0; k1 < R; ++k1) v[k1] = sm[x * ld + k1 * Y2 + n2];
            Dft<R, +1>::run(v);
#pragma unroll
            for (int n1 = 0; n1 < R; ++n1) plane[x * fy + n2 + Y2 * n1] = v[n1];
        }
    });
    if (ACC) store_sums(sums, need_virial, part, fzc, sa_block);
}

constexpr int kPlaneThreads = 512;
constexpr size_t kPlaneLds = 40 * 1024;
template <bool ACC>
__global__ void __launch_bounds__(kPlaneThreads) k_fft_plane(
    float2* __restrict__ FQ, const float* __restrict__ BCt, ReciprocalGeom rg, int fx, int fy, int fz,
    int fzc, sa_radix_plan px, sa_radix_plan py, const float2* __restrict__ twx,
    const float2* __restrict__ twy, int need_virial, double* __restrict__ part) {
    fft_plane_body<ACC>(blockIdx.x, FQ, BCt, rg, fx, fy, fz, fzc, px, py, twx, twy, need_virial, part);
}

// z pass, half spectrum -> real (unnormalised C2R): block = (y block, x)
__device__ __forceinline__ void fft_z_c2r_body(int sa_block, const float2* __restrict__ FQ,
                                                   float* __restrict__ out, int fx, int fy, int fz,
                                                   int fzc, int TL, const sa_radix_plan& pl,
                                                   const float2* __restrict__ tw) {
    extern __shared__ float2 sm[];
    const int gy = (fy + TL - 1) / TL;  // y blocks per x line (1D grid: x-major)
    const int x = sa_block / gy, y0 = (sa_block - x * gy) * TL;
    const int nl = min(TL, fy - y0), npair = (nl + 1) >> 1;
    // half spectra of the lines, [kz][l] with an odd row length
    const int ldh = TL | 1;
    float2* h = sm;
    for (int e = threadIdx.x; e < fzc * nl; e += blockDim.x) {
        const int kz = e / nl, l = e - kz * nl;
        float2 v = FQ[((size_t)kz * fx + x) * fy + y0 + l];
        // the imaginary parts of the DC and Nyquist terms do not enter a
        // real-to-complex inverse
        if (kz == 0 || 2 * kz == fz) v.y = 0.f;
        h[kz * ldh + l] = v;
    }
    float2* a = sm + fzc * ldh;
    float* dst = out + ((size_t)x * fy + y0) * fz;
    // spectrum of line 2m + i line 2m+1 at k
    auto paired = [&](int m, int k) -> float2 {
        const bool up = k >= fzc;
        const int kk = up ? fz - k : k;
        float2 A = h[kk * ldh + 2 * m];
        float2 B = 2 * m + 1 < nl ? h[kk * ldh + 2 * m + 1] : make_float2(0.f, 0.f);
        if (up) {
            A.y = -A.y;
            B.y = -B.y;
        }
        return make_float2(A.x - B.y, A.y + B.x);
    };
    if (pl.r1) {
        const int R1 = pl.r1, R2 = pl.r2, ld = R1 * (R2 + 1);
        const float inv2 = __builtin_amdgcn_rcpf((float)R2), inv1 = __builtin_amdgcn_rcpf((float)R1);
        __syncthreads();
        with_radix(R1, [&](auto radix) {
            constexpr int R = decltype(radix)::value;
            for (int t = threadIdx.x; t < npair * R2; t += blockDim.x) {
                const int m = div_small(t, inv2), n2 = t - m * R2;
                float2 v[R], w[R];
#pragma unroll
                for (int k1 = 1; k1 < R; ++k1) w[k1] = tw[n2 * k1];
#pragma unroll
                for (int r = 0; r < R; ++r) v[r] = paired(m, n2 + R2 * r);
                Dft<R, +1>::run(v);
                a[m * ld + n2] = v[0];
#pragma unroll
                for (int k1 = 1; k1 < R; ++k1)
                    a[m * ld + k1 * (R2 + 1) + n2] = cmul(v[k1], make_float2(w[k1].x, -w[k1].y));
            }
        });
        __syncthreads();
        with_radix(R2, [&](auto radix) {
            constexpr int R = decltype(radix)::value;
            for (int t = threadIdx.x; t < npair * R1; t += blockDim.x) {
                const int m = div_small(t, inv1), k1 = t - m * R1;
                float2 v[R];
#pragma unroll
                for (int n2 = 0; n2 < R; ++n2) v[n2] = a[m * ld + k1 * (R2 + 1) + n2];
                Dft<R, +1>::run(v);
                float* d0 = dst + (size_t)(2 * m) * fz + k1;
#pragma unroll
                for (int k2 = 0; k2 < R; ++k2) d0[R1 * k2] = v[k2].x;
                if (2 * m + 1 < nl)
#pragma unroll
                    for (int k2 = 0; k2 < R; ++k2) d0[fz + R1 * k2] = v[k2].y;
            }
        });
        return;
    }
    float2* b = a + ((TL + 1) >> 1) * fz;
    float2* stw = b + ((TL + 1) >> 1) * fz;
    for (int k = threadIdx.x; k < fz; k += blockDim.x) stw[k] = tw[k];
    __syncthreads();
    for (int e = threadIdx.x; e < npair * fz; e += blockDim.x) {
        const int m = e / fz, k = e - m * fz;
        a[e] = paired(m, k);
    }
    __syncthreads();
    const float2* res = fft_lines<+1>(a, b, npair, fz, fz, pl, stw);
    for (int e = threadIdx.x; e < nl * fz; e += blockDim.x) {
        const int l = e / fz, z = e - l * fz;
        const float2 v = res[(l >> 1) * fz + z];
        dst[e] = (l & 1) ? v.y : v.x;
    }
}

__global__ void __launch_bounds__(128) k_fft_z_c2r(const float2* __restrict__ FQ,
                                                   float* __restrict__ out, int fx, int fy, int fz,
                                                   int fzc, int TL, sa_radix_plan pl,
                                                   const float2* __restrict__ tw) {
    fft_z_c2r_body(blockIdx.x, FQ, out, fx, fy, fz, fzc, TL, pl, tw);
}

// ---------------------------------------------------------------------------
// PME_Atom_Near (PM_force.cpp:706-733): base point u and fraction f
struct Near {
    int ux, uy, uz;
    float fx, fy, fz;
};

// FMA contraction stays off here: fused, frac * n - t would subtract the
// truncated base from the unrounded product, and an atom on a grid plane
// (frac * n rounding up to an integer) would get f = 1 - eps on the base
// below instead of f = 0 on its own plane: a charge one grid step away.
__device__ __forceinline__ void near_axis(float frac, int n, int& u, float& f) {
#pragma clang fp contract(off)
    frac *= n;
    int t = (int)frac;
    t = t < 0 ? 0 : (t < n ? t : n - 1);
    u = t;
    f = frac - t;
    f = f - floorf(f);
}

__device__ __forceinline__ Near atom_near(const float* __restrict__ crd, int i, const LT6& rc,
                                          int fx, int fy, int fz) {
#pragma clang fp contract(off)
    const float x = crd[3 * i], y = crd[3 * i + 1], z = crd[3 * i + 2];
    // VECTOR * LTMatrix3 then frac - floorf(frac)
    float sx = x * rc.a11 + y * rc.a21 + z * rc.a31;
    float sy = y * rc.a22 + z * rc.a32;
    float sz = z * rc.a33;
    if (!isfinite(sx) || !isfinite(sy) || !isfinite(sz)) sx = sy = sz = 0.f;
    // x - floorf(x), below 1: for -3e-8 < x < 0 the subtraction rounds to 1,
    // whose base point was then clamped to the last plane with fraction 0, a
    // charge one grid step away (one atom in 100 steps of 95,000, where a
    // molecule drifts through a box face)
    sx = __builtin_amdgcn_fractf(sx);
    sy = __builtin_amdgcn_fractf(sy);
    sz = __builtin_amdgcn_fractf(sz);
    Near o;
    near_axis(sx, fx, o.ux, o.fx);
    near_axis(sy, fy, o.uy, o.fy);
    near_axis(sz, fz, o.uz, o.fz);
    return o;
}

// The weight polynomials of one stencil index k, held in registers by a
// lane for its whole kernel (the lane's k never changes), so the hot loops
// do not reload the coefficient tables.
struct BspCoef {
    float a, b, c, d;     // M: ((a f + b) f + c) f + d
    __device__ __forceinline__ explicit BspCoef(int k) : a(cMa[k]), b(cMb[k]), c(cMc[k]), d(cMd[k]) {}
    __device__ __forceinline__ float w(float f) const { return fmaf(fmaf(fmaf(a, f, b), f, c), f, d); }
};


// Tile spread.  The charge grid is cut into bricks of Bx x By x Bz points (the
// last brick of an axis takes the remainder, Bx..2Bx-1 points).  An atom
// spreads onto the points u - k (k = 0..3 per axis) below its base point u;
// so every atom whose base point lies in a brick spreads inside that brick's
// halo tile, the brick extended by 3 points downwards on each axis.  One
// workgroup per brick spreads the atoms binned in it into the tile in LDS and
// stores the tile; a second pass sums, for every grid point, the entries of
// the (at most 8) tiles covering it in a fixed order.  Neither pass uses an
// atomic or needs the grid cleared, and the grid is the same on every run
// for the same binning.  Same weights and order as PME_Q_Spread
// (PM_force.cpp:787-812): q Mx(kx) My(ky) Mz(kz).

// Bin the atoms by the brick of their base point; with qpart, also the
// workgroup's sums of q^2 and q (q^2 first, [2][workgroups]).  Slots: an LDS histogram of the
// block's atoms per brick, then one global atomic per distinct brick of the
// block, all issued at once (one round trip instead of a chain); for grids
// with more bricks than the LDS table holds, one atomic per distinct brick of
// each wavefront.
constexpr int kBinLds = 4096;  // bricks tracked in LDS by the bin kernel

__device__ __forceinline__ void pme_bin_body(int sa_block, int N, const float* __restrict__ crd,
                                                 const float* __restrict__ charge, LT6 rc, int fx,
                                                 int fy, int fz, int bx, int by, int bz, int nbx,
                                                 int nby, int nbz, int nb, int bcap,
                                                 int* __restrict__ bcount, float4* __restrict__ bw,
                                                 int* __restrict__ bu, int* __restrict__ bi,
                                                 float4* __restrict__ ow, int* __restrict__ ou,
                                                 int* __restrict__ oi, double* __restrict__ qpart) {
    __shared__ int lcount[kBinLds];
    __shared__ int lbase[kBinLds];
    const int i = sa_block * blockDim.x + threadIdx.x;
    const bool live = i < N;
    int h = -1, u = 0;
    float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
    if (live) {
        const Near nr = atom_near(crd, i, rc, fx, fy, fz);
        h = (brick_of(nr.ux, bx, nbx) * nby + brick_of(nr.uy, by, nby)) * nbz +
            brick_of(nr.uz, bz, nbz);
        w = make_float4(nr.fx, nr.fy, nr.fz, charge[i]);
        u = nr.ux | (nr.uy << 10) | (nr.uz << 20);
    }
    if (qpart) {
        __shared__ double qs[2][4];
        const double s2 = wave_sum((double)(w.w * w.w)), s1 = wave_sum((double)w.w);
        const int wv = threadIdx.x / kWave;
        if ((threadIdx.x & (kWave - 1)) == 0) {
            qs[0][wv] = s2;
            qs[1][wv] = s1;
        }
        __syncthreads();
        if (threadIdx.x < 2)
            qpart[(size_t)threadIdx.x * ((N + 255) / 256) + sa_block] =
                qs[threadIdx.x][0] + qs[threadIdx.x][1] + qs[threadIdx.x][2] + qs[threadIdx.x][3];
    }
    int slot = 0;
    if (nb <= kBinLds) {
        if (live) lcount[h] = 0;
        __syncthreads();
        int local = 0;
        if (live) local = atomicAdd(&lcount[h], 1);
        __syncthreads();
        if (live && local == 0) lbase[h] = atomicAdd(&bcount[h], lcount[h]);
        __syncthreads();
        if (live) slot = lbase[h] + local;
    } else {
        unsigned long long todo = __ballot(live);
        while (todo) {
            const int leader = __builtin_ctzll(todo);
            const int hb = __builtin_amdgcn_readlane(h, leader);
            const unsigned long long peers = __ballot(h == hb);
            int base = 0;
            if (__lane_id() == leader) base = atomicAdd(&bcount[hb], __popcll(peers));
            base = __builtin_amdgcn_readlane(base, leader);
            if (h == hb) slot = base + lanes_below(peers);
            todo &= ~peers;
        }
    }
    if (!live) return;
    if (slot < bcap) {
        bw[(size_t)h * bcap + slot] = w;
        bu[(size_t)h * bcap + slot] = u;
        bi[(size_t)h * bcap + slot] = i;
    } else {
        const int o = atomicAdd(&bcount[nb], 1);
        ow[o] = w;
        ou[o] = u;
        oi[o] = i;
    }
}

__global__ void __launch_bounds__(256) k_pme_bin(int N, const float* __restrict__ crd,
                                                 const float* __restrict__ charge, LT6 rc, int fx,
                                                 int fy, int fz, int bx, int by, int bz, int nbx,
                                                 int nby, int nbz, int nb, int bcap,
                                                 int* __restrict__ bcount, float4* __restrict__ bw,
                                                 int* __restrict__ bu, int* __restrict__ bi,
                                                 float4* __restrict__ ow, int* __restrict__ ou,
                                                 int* __restrict__ oi, double* __restrict__ qpart) {
    pme_bin_body(blockIdx.x, N, crd, charge, rc, fx, fy, fz, bx, by, bz, nbx, nby, nbz, nb, bcap, bcount, bw, bu, bi, ow, ou, oi, qpart);
}

// Brick of a workgroup of the spread, tile-reduce and gather launches (one
// workgroup per brick).  Workgroups go to the 8 XCDs in turn, so workgroup i
// takes brick (i % 8) * (nb / 8) + i / 8: each XCD gets a contiguous range of
// bricks (x-major order), whose neighbours' tiles mostly sit in the same L2.
constexpr int kXcds = 8;
__device__ __forceinline__ int brick_for_block(int i, int nb) {
    if (nb % kXcds) return i;
    return (i % kXcds) * (nb / kXcds) + i / kXcds;
}

__device__ __forceinline__ float lane_f(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

inline TileGeom tile_geom(int mx, int my, int mz) {
    TileGeom g;
    g.tx = mx + 3;
    g.ty = my + 3;
    g.tz = mz + 3;
    g.sy = (g.tz + 3) / 4 * 4;
    const int p = g.ty * g.sy;
    g.sx = p + ((16 - p % 32) + 32) % 32;
    return g;
}

// One workgroup per brick.  Each lane of a wavefront owns one stencil offset
// (kx, ky, kz); the brick's atoms are taken one at a time with their base
// point in scalar registers, so an atom costs the three weight polynomials and
// one LDS read-add-write per lane, every lane in range.  Every wavefront
// accumulates into its own copy of the tile: the LDS operations of one
// wavefront complete in order, so the plain read-add-write needs no atomic (an
// LDS float atomic costs about three cycles per lane on CDNA4); the copies are
// summed when the tile is stored.
__device__ __forceinline__ void pme_spread_tiles_body(int sa_block, 
    int bx, int by, int bz, int nbx, int nby, int nbz, int nb, int bcap, TileGeom tg,
    const int* __restrict__ bcount, const float4* __restrict__ bw, const int* __restrict__ bu,
    const float4* __restrict__ ow, const int* __restrict__ ou, float* __restrict__ tiles) {
    extern __shared__ float acc[];
    const int b = brick_for_block(sa_block, nb);
    const int cz = b % nbz, cy = (b / nbz) % nby, cx = b / (nbz * nby);
    const int X0 = cx * bx, Y0 = cy * by, Z0 = cz * bz;
    const int nwave = blockDim.x / kWave;
    const int tsize = tg.lds_floats();
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    // the first chunk of the brick's slots is loaded alongside its count
    // (slots below bcap always exist; those past the count are ignored)
    const int g0 = lane * nwave + wave;
    float4 w0 = make_float4(0.f, 0.f, 0.f, 0.f);
    int u0 = 0;
    if (g0 < bcap) {
        w0 = bw[(size_t)b * bcap + g0];
        u0 = bu[(size_t)b * bcap + g0];
    }
    const int n_own = min(bcount[b], bcap);
    const int n_over = bcount[nb];
    for (int k = threadIdx.x; k < nwave * tsize; k += blockDim.x) acc[k] = 0.f;
    __syncthreads();
    float* __restrict__ mine = acc + wave * tsize;
    const int kx = lane >> 4, ky = (lane >> 2) & 3, kz = lane & 3;
    int loff = kx * tg.sx + ky * tg.sy + kz;
    // keep the tile-relative base point scalar: without this the compiler
    // folds the lane offset back into per-lane multiplies
    asm volatile("" : "+v"(loff));
    const BspCoef Cx(kx), Cy(ky), Cz(kz);
    // tile corner: (X0 - 3, Y0 - 3, Z0 - 3)
    const int sbase = (3 - X0) * tg.sx + (3 - Y0) * tg.sy + (3 - Z0);
    const int total = n_own + n_over;
    // atoms dealt to the wavefronts in turn (a brick holds about one
    // wavefront's worth)
    for (int base = 0; base < total; base += nwave * kWave) {
        const int g = base + lane * nwave + wave;
        float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
        int u = 0;
        bool hit = false;
        if (g < n_own) {
            if (base == 0) {
                w = w0;
                u = u0;
            } else {
                w = bw[(size_t)b * bcap + g];
                u = bu[(size_t)b * bcap + g];
            }
            hit = w.w != 0.f;  // an uncharged atom adds nothing
        } else if (g < total) {
            w = ow[g - n_own];
            u = ou[g - n_own];
            hit = w.w != 0.f && brick_of(u & 1023, bx, nbx) == cx &&
                  brick_of((u >> 10) & 1023, by, nby) == cy && brick_of(u >> 20, bz, nbz) == cz;
        }
        unsigned long long m = __ballot(hit);
        while (m) {
            const int src = __builtin_ctzll(m);
            m &= m - 1;
            const int us = __builtin_amdgcn_readlane(u, src);
            const int a0 = sbase + (us & 1023) * tg.sx + ((us >> 10) & 1023) * tg.sy + (us >> 20);
            const float wfx = lane_f(w.x, src);
            const float wfy = lane_f(w.y, src);
            const float wfz = lane_f(w.z, src);
            const float q = lane_f(w.w, src);
            float tq = q * Cx.w(wfx);
            tq = tq * Cy.w(wfy);
            tq = tq * Cz.w(wfz);
            mine[a0 - loff] += tq;
        }
    }
    __syncthreads();
    float* __restrict__ out = tiles + (size_t)b * tg.points();
    const int npts = tg.points();
    const float inv_tz = __builtin_amdgcn_rcpf((float)tg.tz);
    const float inv_ty = __builtin_amdgcn_rcpf((float)tg.ty);
    for (int k = threadIdx.x; k < npts; k += blockDim.x) {
        const int r = div_small(k, inv_tz), z = k - r * tg.tz;
        const int x = div_small(r, inv_ty), y = r - x * tg.ty;
        const int a = x * tg.sx + y * tg.sy + z;
        float v = acc[a];
        for (int w = 1; w < nwave; ++w) v += acc[w * tsize + a];
        out[k] = v;
    }
}

__global__ void __launch_bounds__(256) k_pme_spread_tiles(
    int bx, int by, int bz, int nbx, int nby, int nbz, int nb, int bcap, TileGeom tg,
    const int* __restrict__ bcount, const float4* __restrict__ bw, const int* __restrict__ bu,
    const float4* __restrict__ ow, const int* __restrict__ ou, float* __restrict__ tiles) {
    pme_spread_tiles_body(blockIdx.x, bx, by, bz, nbx, nby, nbz, nb, bcap, tg, bcount, bw, bu, ow, ou, tiles);
}

// Grid point (x, y, z) of brick c at local (lx, ly, lz) sums, per axis, its
// own tile at l + 3 and, for the top 3 points of the brick, the tile of the
// brick above at l - extent + 3 (the same tile when the axis has one brick).
// It also hands the bin counts to the gather (gcount) and clears them for the
// next evaluation's binning (the spread, their other reader, has finished).
__device__ __forceinline__ void pme_tiles_reduce_body(int sa_block, int fx, int fy, int fz, int bx, int by,
                                                          int bz, int nbx, int nby, int nbz,
                                                          int nb, TileGeom tg,
                                                          const float* __restrict__ tiles,
                                                          float* __restrict__ Q,
                                                          int* __restrict__ bcount,
                                                          int* __restrict__ gcount) {
    const int b = brick_for_block(sa_block, nb);
    if (threadIdx.x == 0) {
        gcount[b] = bcount[b];
        bcount[b] = 0;
        if (b == 0) {
            gcount[nb] = bcount[nb];
            bcount[nb] = 0;
        }
    }
    const int cz = b % nbz, cy = (b / nbz) % nby, cx = b / (nbz * nby);
    const int X0 = cx * bx, Y0 = cy * by, Z0 = cz * bz;
    const int ex = cx == nbx - 1 ? fx - X0 : bx;
    const int ey = cy == nby - 1 ? fy - Y0 : by;
    const int ez = cz == nbz - 1 ? fz - Z0 : bz;
    const int ax = cx + 1 == nbx ? 0 : cx + 1;
    const int ay = cy + 1 == nby ? 0 : cy + 1;
    const int az = cz + 1 == nbz ? 0 : cz + 1;
    const size_t tn = (size_t)tg.points();
    const int npts = ex * ey * ez;
    const float inv_ez = __builtin_amdgcn_rcpf((float)ez);
    const float inv_ey = __builtin_amdgcn_rcpf((float)ey);
#pragma unroll 2
    for (int k = threadIdx.x; k < npts; k += blockDim.x) {
        const int r = div_small(k, inv_ez), lz = k - r * ez;
        const int lx = div_small(r, inv_ey), ly = r - lx * ey;
        // the up to 8 covering tiles, loaded independently, summed in a fixed order
        const bool hx = lx >= ex - 3, hy = ly >= ey - 3, hz = lz >= ez - 3;
        // (an absent tile reads the own tile's entry and adds zero, so the
        // loads stay unconditional and all in flight together)
        float t[8];
        size_t at[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int dx = c >> 2, dy = (c >> 1) & 1, dz = c & 1;
            const int bxi = dx ? ax : cx, tx = dx ? lx - ex + 3 : lx + 3;
            const int byi = dy ? ay : cy, ty = dy ? ly - ey + 3 : ly + 3;
            const int bzi = dz ? az : cz, tz = dz ? lz - ez + 3 : lz + 3;
            at[c] = (size_t)((bxi * nby + byi) * nbz + bzi) * tn + (tx * tg.ty + ty) * tg.tz + tz;
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int dx = c >> 2, dy = (c >> 1) & 1, dz = c & 1;
            const bool ok = (!dx || hx) && (!dy || hy) && (!dz || hz);
            const float v = tiles[ok ? at[c] : at[0]];
            t[c] = ok ? v : 0.f;
        }
        const float v = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
        Q[((size_t)(X0 + lx) * fy + (Y0 + ly)) * fz + (Z0 + lz)] = v;
    }
}

__global__ void __launch_bounds__(256) k_pme_tiles_reduce(int fx, int fy, int fz, int bx, int by,
                                                          int bz, int nbx, int nby, int nbz,
                                                          int nb, TileGeom tg,
                                                          const float* __restrict__ tiles,
                                                          float* __restrict__ Q,
                                                          int* __restrict__ bcount,
                                                          int* __restrict__ gcount) {
    pme_tiles_reduce_body(blockIdx.x, fx, fy, fz, bx, by, bz, nbx, nby, nbz, nb, tg, tiles, Q, bcount, gcount);
}

// B-spline weight polynomials M_k and their derivatives dM_k as compile-time
// constants (M_k the same as cMa..cMd) for the thread-per-atom gather
struct BspK {
    static constexpr float a[4] = {(float)(1.0 / 6.0), -0.5f, 0.5f, (float)(-1.0 / 6.0)};
    static constexpr float b[4] = {0.f, 0.5f, -1.f, 0.5f};
    static constexpr float c[4] = {0.f, 0.5f, 0.f, -0.5f};
    static constexpr float d[4] = {0.f, (float)(1.0 / 6.0), (float)(4.0 / 6.0), (float)(1.0 / 6.0)};
    static constexpr float da[4] = {0.5f, -1.5f, 1.5f, -0.5f};
    static constexpr float db[4] = {0.f, 1.f, -2.f, 1.f};
    static constexpr float dc[4] = {0.f, 0.5f, 0.f, -0.5f};
    __device__ static __forceinline__ float w(int k, float f) {
        return fmaf(fmaf(fmaf(a[k], f, b[k]), f, c[k]), f, d[k]);
    }
    __device__ static __forceinline__ float dw(int k, float f) {
        return fmaf(fmaf(da[k], f, db[k]), f, dc[k]);
    }
};

// g(x) = 2/sqrt(pi) x e^{-x^2} - erf(x)
//      = 2/sqrt(pi) sum_{n>=1} (-1)^n 2n / ((2n+1) n!) x^{2n+1},
// series below x = 0.75 (truncation < 1e-9 relative), direct form above.
__device__ __forceinline__ float excl_bracket(float x) {
    if (x < 0.75f) {
        const float x2 = x * x;
        float s = 2.62450659e-7f;         // n = 10
        s = s * x2 - 2.61069340e-6f;      // n = 9
        s = s * x2 + 2.33426704e-5f;      // n = 8
        s = s * x2 - 1.85185185e-4f;      // n = 7
        s = s * x2 + 1.28205128e-3f;      // n = 6
        s = s * x2 - 7.57575758e-3f;      // n = 5
        s = s * x2 + 3.70370370e-2f;      // n = 4
        s = s * x2 - 1.42857143e-1f;      // n = 3
        s = s * x2 + 4.00000000e-1f;      // n = 2
        s = s * x2 - 6.66666667e-1f;      // n = 1
        return kTwoOverSqrtPi * s * x2 * x;
    }
    return x * kTwoOverSqrtPi * expf(-x * x) - erff(x);
}

// Force factor of the excluded-pair correction (PM_force.cpp:1774-1790):
// (2/sqrt(pi) x e^{-x^2} + erfc(x) - 1) / r^3 times -q_i q_j; the bracket
// cancels to a few percent of its terms for bonded distances, so it is summed
// as its odd Taylor series there.
__device__ __forceinline__ float excl_factor(float dr2, float qq, float beta) {
    const float dr = sqrtf(dr2);
    return -qq * (excl_bracket(beta * dr) / dr2 / dr);
}

// Self, neutralizing and reciprocal energies added to the potential
// (PM_force.cpp:1142-1166).
__device__ __forceinline__ void energy_final(const double* acc, float* ene, float* potential,
                                             float self_factor, float neutralizing_factor) {
    const float rec = (float)acc[0] * 0.5f;
    float self = (float)acc[7];
    self = self * self_factor;
    const float sumq = (float)acc[8];
    self += neutralizing_factor * sumq * sumq;
    ene[0] = rec;
    ene[1] = self;
    if (potential) potential[0] += self + rec;
}

// Totals of an evaluation with energy or virial, by one workgroup: the partial
// sums of the convolution ([7][nx]) and of the bin pass ([2][nq], with an
// energy) into acc, and from there the energies and the virial.
struct SpectrumTotals {
    const double* part = nullptr;
    const double* qpart = nullptr;
    int nx = 0, nq = 0;
    double* acc = nullptr;
    float* ene = nullptr;
    float* potential = nullptr;
    float* virial = nullptr;
    float self_factor = 0.f, neutralizing_factor = 0.f;
};

__device__ __forceinline__ void spectrum_totals(const SpectrumTotals& t, double* red) {
    const int lane = threadIdx.x & (kWave - 1), nw = blockDim.x / kWave;
    const int terms = t.qpart ? 9 : 7;
    // term by term over the wavefronts
    for (int c = threadIdx.x / kWave; c < terms; c += nw) {
        const double* p = c < 7 ? t.part + (size_t)c * t.nx : t.qpart + (size_t)(c - 7) * t.nq;
        const int n = c < 7 ? t.nx : t.nq;
        double v = 0.0;
#pragma unroll 4
        for (int i = lane; i < n; i += kWave) v += p[i];
        v = wave_sum(v);
        if (lane == 0) red[c] = v;
    }
    __syncthreads();
    if ((int)threadIdx.x < terms) t.acc[threadIdx.x] = red[threadIdx.x];
    if (t.virial && threadIdx.x < 6) t.virial[threadIdx.x] += (float)red[1 + threadIdx.x];
    if (t.qpart && threadIdx.x == 0)
        energy_final(red, t.ene, t.potential, t.self_factor, t.neutralizing_factor);
}

// PME_Final + device_add_force: frc += update_interval * F (PM_force.cpp:
// 852-892, 1014-1022).  One workgroup per brick: the brick's halo tile of the
// convolved grid (the points the stencils of its atoms reach) is read into
// LDS with coalesced loads, then each thread takes one of the brick's atoms, as
// binned by the spread: its 4 x 4 x 4 stencil is read from the tile as 16 rows
// of 4 points and contracted with the weights in registers (per row the z sums
// with M_z and dM_z, then the x / y factors).  On the step driver's force-only
// steps it is the pass that writes the force array (gb: see GatherBase): the
// pair forces and the excluded-pair correction of its atoms cost it 2 us at
// 95,000 atoms, against passes of their own of 4 (finalize) and 11 us
// (excluded pairs by atomics, and 5 to clear their array).  The partners'
// coordinates are loaded before the stencil is contracted.
// One workgroup more than bricks (sums.part set): that one adds up the partial
// sums of the convolution and the bin pass and finishes the energies and the
// virial, which cost four launches (13 us) of their own.
constexpr int kGatherThreads = 256;
constexpr int kGatherLoads = 8;

__device__ __forceinline__ void pme_gather_tiles_body(int sa_block, 
    int fx, int fy, int fz, int bx, int by, int bz, int nbx, int nby, int nbz, int nb, int bcap,
    TileGeom tg, const int* __restrict__ gcount, const float4* __restrict__ bw,
    const int* __restrict__ bu, const int* __restrict__ bi, const float4* __restrict__ ow,
    const int* __restrict__ ou, const int* __restrict__ oi, const float* __restrict__ phi, LT6 rc,
    float update_interval, float* __restrict__ frc, const GatherBase& gb, LT6 cell, float beta,
    const SpectrumTotals& sums) {
    extern __shared__ __align__(16) float tile[];
    if (sa_block == nb) {
        spectrum_totals(sums, reinterpret_cast<double*>(tile));
        return;
    }
    if (gb.reset && sa_block == 0 && threadIdx.x == 0) *gb.reset = 0;
    const int b = brick_for_block(sa_block, nb);
    const int cz = b % nbz, cy = (b / nbz) % nby, cx = b / (nbz * nby);
    const int X0 = cx * bx, Y0 = cy * by, Z0 = cz * bz;
    const int TX = (cx == nbx - 1 ? fx - X0 : bx) + 3;
    const int TY = (cy == nby - 1 ? fy - Y0 : by) + 3;
    const int TZ = (cz == nbz - 1 ? fz - Z0 : bz) + 3;
    const int npts = TX * TY * TZ;
    const float inv_tz = __builtin_amdgcn_rcpf((float)TZ);
    const float inv_ty = __builtin_amdgcn_rcpf((float)TY);
    // batches of kGatherLoads loads per thread in flight before their LDS writes
    for (int k0 = threadIdx.x; k0 < npts; k0 += blockDim.x * kGatherLoads) {
        float v[kGatherLoads];
        int at[kGatherLoads];
#pragma unroll
        for (int j = 0; j < kGatherLoads; ++j) {
            // points past the tile repeat its last one (loaded, not stored),
            // so the loads stay unconditional and all in flight together
            const int kk = k0 + j * (int)blockDim.x;
            const int k = kk < npts ? kk : npts - 1;
            const int r = div_small(k, inv_tz), tz = k - r * TZ;
            const int tx = div_small(r, inv_ty), ty = r - tx * TY;
            int gx = X0 - 3 + tx, gy = Y0 - 3 + ty, gz = Z0 - 3 + tz;
            gx += gx < 0 ? fx : 0;
            gy += gy < 0 ? fy : 0;
            gz += gz < 0 ? fz : 0;
            v[j] = phi[((size_t)gx * fy + gy) * fz + gz];
            at[j] = kk < npts ? tx * tg.sx + ty * tg.sy + tz : -1;
        }
#pragma unroll
        for (int j = 0; j < kGatherLoads; ++j)
            if (at[j] >= 0) tile[at[j]] = v[j];
    }
    __syncthreads();
    const int n_own = min(gcount[b], bcap);
    const int total = n_own + gcount[nb];
    for (int g = threadIdx.x; g < total; g += blockDim.x) {
        float4 w;
        int u, i;
        if (g < n_own) {
            w = bw[(size_t)b * bcap + g];
            u = bu[(size_t)b * bcap + g];
            i = bi[(size_t)b * bcap + g];
        } else {
            w = ow[g - n_own];
            u = ou[g - n_own];
            i = oi[g - n_own];
            if (brick_of(u & 1023, bx, nbx) != cx || brick_of((u >> 10) & 1023, by, nby) != cy ||
                brick_of(u >> 20, bz, nbz) != cz)
                continue;
        }
        // the pair force and up to two excluded partners (a water's), loaded
        // ahead of the contraction
        const bool ex = gb.ex_start != nullptr;
        float f0x, f0y, f0z;
        if (gb.base) {
            const float4 f0 = gb.base[gb.rank[i]];
            f0x = f0.x;
            f0y = f0.y;
            f0z = f0.z;
        } else {
            f0x = frc[3 * i];
            f0y = frc[3 * i + 1];
            f0z = frc[3 * i + 2];
        }
        int e0 = 0, ne = 0, ea = 0, eb = 0;
        float3 xi = make_float3(0.f, 0.f, 0.f), xa = xi, xb = xi;
        float qa = 0.f, qb = 0.f;
        if (ex) {
            e0 = gb.ex_start[i];
            ne = gb.ex_start[i + 1] - e0;
            ea = ne > 0 ? gb.ex_list[e0] : i;
            eb = ne > 1 ? gb.ex_list[e0 + 1] : i;
            const int ja = ea < 0 ? ~ea : ea, jb = eb < 0 ? ~eb : eb;
            xi = make_float3(gb.crd[3 * i], gb.crd[3 * i + 1], gb.crd[3 * i + 2]);
            xa = make_float3(gb.crd[3 * ja], gb.crd[3 * ja + 1], gb.crd[3 * ja + 2]);
            xb = make_float3(gb.crd[3 * jb], gb.crd[3 * jb + 1], gb.crd[3 * jb + 2]);
            qa = gb.charge[ja];
            qb = gb.charge[jb];
        }
        // base point in the tile: stencil point k lies at t - k
        const int rx = (u & 1023) - X0 + 3, ry = ((u >> 10) & 1023) - Y0 + 3, rz = (u >> 20) - Z0 + 3;
        float wx[4], wy[4], wz[4], dx[4], dy[4], dz[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            wx[k] = BspK::w(k, w.x);
            wy[k] = BspK::w(k, w.y);
            wz[k] = BspK::w(k, w.z);
            dx[k] = BspK::dw(k, w.x);
            dy[k] = BspK::dw(k, w.y);
            dz[k] = BspK::dw(k, w.z);
        }
        float gx = 0.f, gy = 0.f, gz = 0.f;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float* row = tile + (rx - a) * tg.sx + (ry - c) * tg.sy + rz;
                float sw = 0.f, sd = 0.f;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float v = row[-k];
                    sw = fmaf(v, wz[k], sw);
                    sd = fmaf(v, dz[k], sd);
                }
                gx = fmaf(dx[a] * wy[c], sw, gx);
                gy = fmaf(wx[a] * dy[c], sw, gy);
                gz = fmaf(wx[a] * wy[c], sd, gz);
            }
        }
        gx *= (float)fx;
        gy *= (float)fy;
        gz *= (float)fz;
        const float dq = -w.w;
        // MultiplyTranspose(g, rcell) = {gx a11, gx a21 + gy a22, gx a31 + gy a32 + gz a33}
        const float ox = dq * (gx * rc.a11);
        const float oy = dq * (gx * rc.a21 + gy * rc.a22);
        const float oz = dq * (gx * rc.a31 + gy * rc.a32 + gz * rc.a33);
        float ex_x = 0.f, ex_y = 0.f, ex_z = 0.f;
        // the displacement is taken from the atom whose list holds the pair (at
        // half a box length the reference's minimum image is not antisymmetric)
        auto excluded = [&](float3 xj, float qj, bool reverse) {
            float3 d = reverse ? disp_pbc<true>(xi, xj, cell, rc) : disp_pbc<true>(xj, xi, cell, rc);
            if (reverse) d = make_float3(-d.x, -d.y, -d.z);
            const float fa = excl_factor(norm2_exact(d), w.w * qj, beta);
            ex_x = fmaf(fa, d.x, ex_x);
            ex_y = fmaf(fa, d.y, ex_y);
            ex_z = fmaf(fa, d.z, ex_z);
        };
        if (ne > 0) excluded(xa, qa, ea < 0);
        if (ne > 1) excluded(xb, qb, eb < 0);
        for (int e = 2; e < ne; ++e) {
            const int en = gb.ex_list[e0 + e], j = en < 0 ? ~en : en;
            excluded(make_float3(gb.crd[3 * j], gb.crd[3 * j + 1], gb.crd[3 * j + 2]), gb.charge[j],
                     en < 0);
        }
        // every atom is in exactly one brick's list (own slots or overflow)
        frc[3 * i] = f0x + update_interval * ox + ex_x;
        frc[3 * i + 1] = f0y + update_interval * oy + ex_y;
        frc[3 * i + 2] = f0z + update_interval * oz + ex_z;
    }
}

__global__ void __launch_bounds__(kGatherThreads) k_pme_gather_tiles(
    int fx, int fy, int fz, int bx, int by, int bz, int nbx, int nby, int nbz, int nb, int bcap,
    TileGeom tg, const int* __restrict__ gcount, const float4* __restrict__ bw,
    const int* __restrict__ bu, const int* __restrict__ bi, const float4* __restrict__ ow,
    const int* __restrict__ ou, const int* __restrict__ oi, const float* __restrict__ phi, LT6 rc,
    float update_interval, float* __restrict__ frc, GatherBase gb, LT6 cell, float beta,
    SpectrumTotals sums) {
    pme_gather_tiles_body(blockIdx.x, fx, fy, fz, bx, by, bz, nbx, nby, nbz, nb, bcap, tg, gcount, bw, bu, bi, ow, ou, oi, phi, rc, update_interval, frc, gb, cell, beta, sums);
}

__global__ void k_pme_charge_sums(int N, const float* __restrict__ q, double* __restrict__ acc) {
    double s2 = 0, s1 = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        const float v = q[i];
        s2 += (double)(v * v);
        s1 += (double)v;
    }
    s2 = wave_sum(s2);
    s1 = wave_sum(s1);
    if ((threadIdx.x & (kWave - 1)) == 0) {
        unsafeAtomicAdd(&acc[7], s2);
        unsafeAtomicAdd(&acc[8], s1);
    }
}

__global__ void k_pme_energy_final(const double* __restrict__ acc, float* __restrict__ ene,
                                   float* __restrict__ potential, float self_factor,
                                   float neutralizing_factor) {
    energy_final(acc, ene, potential, self_factor, neutralizing_factor);
}

// MPI_PME_Excluded_Force_With_Atom_Energy_Correction with factor 1
// (PM_force.cpp:1744-1817), one thread per local atom.
template <bool ORTHO>
__device__ __forceinline__ void pme_excluded_body(int sa_block, int N, const float* __restrict__ crd,
                               const float* __restrict__ charge, LT6 c, LT6 r, float beta,
                               const int* __restrict__ ex_start, const int* __restrict__ ex_list,
                               const int* __restrict__ ex_num, float* __restrict__ frc,
                               int need_e, float* __restrict__ atom_ene,
                               float* __restrict__ corr_ene, int need_v,
                               float* __restrict__ atom_virial) {
    const int i = sa_block * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int n = ex_num[i];
    if (n <= 0) return;
    const int s = ex_start[i];
    const float qi = charge[i];
    const float3 r1 = make_float3(crd[3 * i], crd[3 * i + 1], crd[3 * i + 2]);
    float fx = 0, fy = 0, fz = 0, e = 0;
    float v0 = 0, v1 = 0, v2 = 0, v3 = 0, v4 = 0, v5 = 0;
    for (int k = s; k < s + n; ++k) {
        const int j = ex_list[k];
        const float3 r2 = make_float3(crd[3 * j], crd[3 * j + 1], crd[3 * j + 2]);
        const float qj = charge[j];
        const float3 d = disp_pbc<ORTHO>(r2, r1, c, r);
        const float dr2 = norm2_exact(d);
        const float dr_abs = sqrtf(dr2);
        const float br = beta * dr_abs;
        const float fa = excl_factor(dr2, qi * qj, beta);
        const float lx = fa * d.x, ly = fa * d.y, lz = fa * d.z;
        unsafeAtomicAdd(&frc[3 * j], -lx);
        unsafeAtomicAdd(&frc[3 * j + 1], -ly);
        unsafeAtomicAdd(&frc[3 * j + 2], -lz);
        fx += lx;
        fy += ly;
        fz += lz;
        if (need_e) e -= qi * qj * erff(br) / dr_abs;
        if (need_v) {
            v0 -= lx * d.x;
            v1 -= lx * d.y + ly * d.x;
            v2 -= ly * d.y;
            v3 -= lx * d.z + lz * d.x;
            v4 -= ly * d.z + lz * d.y;
            v5 -= lz * d.z;
        }
    }
    unsafeAtomicAdd(&frc[3 * i], fx);
    unsafeAtomicAdd(&frc[3 * i + 1], fy);
    unsafeAtomicAdd(&frc[3 * i + 2], fz);
    if (need_e) {
        unsafeAtomicAdd(&atom_ene[i], e);
        corr_ene[i] = e;
    }
    if (need_v) {
        float* o = atom_virial + (size_t)6 * i;
        unsafeAtomicAdd(&o[0], v0);
        unsafeAtomicAdd(&o[1], v1);
        unsafeAtomicAdd(&o[2], v2);
        unsafeAtomicAdd(&o[3], v3);
        unsafeAtomicAdd(&o[4], v4);
        unsafeAtomicAdd(&o[5], v5);
    }
}

template <bool ORTHO>
__global__ void k_pme_excluded(int N, const float* __restrict__ crd,
                               const float* __restrict__ charge, LT6 c, LT6 r, float beta,
                               const int* __restrict__ ex_start, const int* __restrict__ ex_list,
                               const int* __restrict__ ex_num, float* __restrict__ frc,
                               int need_e, float* __restrict__ atom_ene,
                               float* __restrict__ corr_ene, int need_v,
                               float* __restrict__ atom_virial) {
    pme_excluded_body<ORTHO>(blockIdx.x, N, crd, charge, c, r, beta, ex_start, ex_list, ex_num, frc, need_e, atom_ene, corr_ene, need_v, atom_virial);
}

__global__ void k_sum2_f32(int n, const float* __restrict__ a, const float* __restrict__ b,
                           double* out) {
    double sa_ = 0, sb = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        sa_ += a[i];
        sb += b[i];
    }
    sa_ = wave_sum(sa_);
    sb = wave_sum(sb);
    if ((threadIdx.x & (kWave - 1)) == 0) {
        unsafeAtomicAdd(&out[0], sa_);
        unsafeAtomicAdd(&out[1], sb);
    }
}

// ---------------------------------------------------------------------------
// host set-up

// getb (PM_force.cpp:42-64): |B(k)|^2 = 1 / |sum_kk M4(kk+1) e^{2 pi i k kk/N}|^2
// evaluated in float with the reference's expc / divc (SPONGE/utils/fft.hpp:26-51).
float bspline_M(float u, int n) {
    if (n == 2) {
        if (u > 2 || u < 0) return 0;
        return 1 - fabsf(u - 1);
    }
    return u / (n - 1) * bspline_M(u, n - 1) + (n - u) / (n - 1) * bspline_M(u - 1, n - 1);
}

float getb(int k, int NFFT, int order) {
    float t2r = 0, t2i = 0;
    const float ang0 = 2 * (order - 1) * kPI * k / NFFT;
    const float rr = cosf(ang0), ri = sinf(ang0);
    for (int kk = 0; kk < order - 1; ++kk) {
        const float ang = 2.0f * kPI * k / NFFT * kk;
        const float tf = bspline_M((float)(kk + 1), order);
        t2r += tf * cosf(ang);
        t2i += tf * sinf(ang);
    }
    const float den = t2r * t2r + t2i * t2i;
    const float re = (rr * t2r + ri * t2i) / den, im = (ri * t2r - rr * t2i) / den;
    return re * re + im * im;
}

bool make_plan(int n, sa_radix_plan* p) {
    p->n = n;
    two_factors(n, p->r1, p->r2);
    p->nst = 0;
    int m = n;
    for (int f : {4, 2, 3, 5, 7})
        while (m % f == 0) {
            if (p->nst >= 16) return false;
            p->r[p->nst++] = f;
            m /= f;
        }
    return m == 1;
}

// LDS of a plane transform: the plane (odd row length) and both twiddle tables
size_t plane_lds(int fx, int fy) { return sizeof(float2) * ((size_t)fx * (fy | 1) + fx + fy); }

int lines_per_block(int n) {
    int t = 2048 / n;
    if (t > 16) t = 16;
    if (t < 2) t = 2;
    return t & ~1;
}

// BC (PM_force.cpp:545-611; recomputed for a new box as up_box_bc does,
// :1171-1238) in the [kz][kx][ky] order of the convolution pass, from the
// module's cell, rcell, volume and beta.
void bc_table(const sponge_pme* p, std::vector<float>& bct) {
    const int fx = p->fx, fy = p->fy, fz = p->fz;
    std::vector<float> B1(fx), B2(fy), B3(fz);
    for (int k = 0; k < fx; ++k) B1[k] = getb(k, fx, 4);
    for (int k = 0; k < fy; ++k) B2[k] = getb(k, fy, 4);
    for (int k = 0; k < fz; ++k) B3[k] = getb(k, fz, 4);
    bct.assign(p->nfft, 0.f);
    const float mprefactor = kPI * kPI / p->beta / p->beta;
    const LT6& rc = p->rcell;
    for (int kx = 0; kx < fx; ++kx) {
        const float kxrp = kx > fx / 2 ? kx - fx : kx;
        for (int ky = 0; ky < fy; ++ky) {
            const float kyrp = ky > fy / 2 ? ky - fy : ky;
            for (int kz = 0; kz <= fz / 2; ++kz) {
                const float kzrp = kz;
                // m = MultiplyTranspose({kx, ky, kz}, rcell)
                const float mx = kxrp * rc.a11;
                const float my = kxrp * rc.a21 + kyrp * rc.a22;
                const float mz = kxrp * rc.a31 + kyrp * rc.a32 + kzrp * rc.a33;
                const float msq = mx * mx + my * my + mz * mz;
                float bc;
                if (kx + ky + kz == 0) {
                    bc = 0;
                } else {
                    bc = (float)1.0 / kPI / msq * expf(-mprefactor * msq) / p->volume;
                }
                bc *= B1[kx] * B2[ky] * B3[kz];
                bct[((size_t)kz * fx + kx) * fy + ky] = bc;
            }
        }
    }
}

void pme_free(sponge_pme* p) {
    for (auto& t : p->d_tw) dfree(t);
    dfree(p->d_Q);
    dfree(p->d_FQ);
    dfree(p->d_FBCFQ);
    dfree(p->d_BCt);
    dfree(p->d_acc);
    dfree(p->d_part);
    dfree(p->d_qpart);
    dfree(p->d_ene);
    dfree(p->d_direct_atom_energy);
    dfree(p->d_correction_atom_energy);
    dfree(p->d_sum);
    dfree(p->d_bcount);
    dfree(p->d_bw);
    dfree(p->d_bu);
    dfree(p->d_ow);
    dfree(p->d_ou);
    dfree(p->d_tiles);
    dfree(p->d_bi);
    dfree(p->d_oi);
    dfree(p->d_gcount);
}

// Brick edge on one axis: the divisor of the grid size closest to 8 among
// 3..16; for a larger size without one, 8 (the last brick then takes the
// remainder, 9..15 points).
int brick_edge(int f) {
    int best = f > 16 ? 8 : f, score = 1 << 30;
    for (int d = 3; d <= 16 && d <= f; ++d) {
        if (f % d) continue;
        const int sc = d > 8 ? d - 8 : 8 - d;
        if (sc < score) {
            score = sc;
            best = d;
        }
    }
    return best;
}

// tile geometry of the spread: sized for the largest brick of each axis
TileGeom pme_tile_geom(const sponge_pme* p) {
    return tile_geom(std::max(p->bx, p->fx - (p->nbx - 1) * p->bx),
                     std::max(p->by, p->fy - (p->nby - 1) * p->by),
                     std::max(p->bz, p->fz - (p->nbz - 1) * p->bz));
}

}  // namespace

// Register budgets of the batched FFT passes: at 6 wavefronts per SIMD they
// fit the standalone kernels' ~77 VGPRs (left free, the batched kernels took
// 100-118 and ran at 4 wavefronts).  The energy / virial convolution keeps
// the compiler's budget (it would spill).
template <>
struct sa::BodyWaves<&fft_z_r2c_body> {
    static constexpr int value = 6;
};
template <>
struct sa::BodyWaves<&fft_y_body<-1>> {
    static constexpr int value = 6;
};
template <>
struct sa::BodyWaves<&fft_y_body<1>> {
    static constexpr int value = 6;
};
template <>
struct sa::BodyWaves<&fft_x_conv_body<false>> {
    static constexpr int value = 6;
};
template <>
struct sa::BodyWaves<&fft_z_c2r_body> {
    static constexpr int value = 6;
};

extern "C" void sponge_pme_default_options(sponge_pme_options* o) {
    o->fftx = o->ffty = o->fftz = -1;
    o->grid_spacing = 1.0f;
    o->direct_tolerance = 0.00001f;
    o->update_interval = 1;
    o->calculate_reciprocal_part = 1;
    o->calculate_excluded_part = 1;
}

extern "C" float sponge_amd_get_beta(float cutoff, float tolerance) {
    // Get_Beta (PM_force.cpp:246-274).  The direct-space tail erfc(b rc) / rc
    // falls as b grows: an upper end is found by doubling from b = 1, then the
    // bracket [0, upper] is halved 50 times more than the doublings needed,
    // and the last midpoint tried is beta.  The tail is evaluated with the
    // library erfc and kept in float, as are b and the bracket, so that beta
    // comes out bit-identical to the reference's.
    auto tail = [cutoff](float b) -> float { return erfc(b * cutoff) / cutoff; };
    float upper = 1.0f;
    int doublings = 0;
    while (!(tail(upper) <= tolerance)) {
        upper *= 2.0f;
        ++doublings;
    }
    float lower = 0.0f, mid = 0.0f;
    for (int halving = 0; halving < doublings + 50; ++halving) {
        mid = (lower + upper) / 2;
        if (tail(mid) >= tolerance) lower = mid;
        else upper = mid;
    }
    return mid;
}

static int check_2357(int n) {
    if (n <= 0) return 0;
    for (int f : {2, 3, 5, 7})
        while (n % f == 0) n /= f;
    return n == 1;
}

extern "C" int sponge_amd_get_fft_parameter(float length) {
    // Get_Fft_Patameter (SPONGE/common.cpp:639-659)
    int t = (int)ceil(length + 3) >> 2 << 2;
    if (t >= 60 && t <= 68) t = 64;
    else if (t >= 120 && t <= 136) t = 128;
    else if (t >= 240 && t <= 272) t = 256;
    else if (t >= 480 && t <= 544) t = 512;
    else if (t >= 960 && t <= 1088) t = 1024;
    while (!check_2357(t)) t += 4;
    return t;
}

extern "C" int sponge_pme_initial(sponge_pme** out, int atom_numbers, const float* cell,
                                  const float* rcell, float cutoff, const sponge_pme_options* opt,
                                  void* stream) {
    if (!out || !cell || !rcell || atom_numbers <= 0 || !(cutoff > 0))
        return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    *out = nullptr;
    sponge_pme* p = new sponge_pme();
    if (opt) p->opt = *opt;
    else sponge_pme_default_options(&p->opt);
    p->N = atom_numbers;
    p->cutoff = cutoff;
    p->cell = lt_from(cell);
    p->rcell = lt_from(rcell);
    p->stream = (hipStream_t)stream;
    if (p->opt.update_interval <= 0 || !(p->opt.grid_spacing > 0)) {
        delete p;
        return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    }
    // grid (PM_force.cpp:383-394): box_length / grid_spacing when not given,
    // box_length being the lengths of the cell vectors (MD_core.cpp:257-262);
    // any lower-triangular cell: fractional coordinates, the BC tables and
    // the gathered forces go through the full rcell
    const LT6& cl = p->cell;
    const bool ortho = lt_is_orthorhombic(cl);
    const float lx = cl.a11;
    const float ly = ortho ? cl.a22 : sqrtf(cl.a21 * cl.a21 + cl.a22 * cl.a22);
    const float lz = ortho ? cl.a33 : sqrtf(cl.a31 * cl.a31 + cl.a32 * cl.a32 + cl.a33 * cl.a33);
    p->fx = p->opt.fftx > 0 ? p->opt.fftx : sponge_amd_get_fft_parameter(lx / p->opt.grid_spacing);
    p->fy = p->opt.ffty > 0 ? p->opt.ffty : sponge_amd_get_fft_parameter(ly / p->opt.grid_spacing);
    p->fz = p->opt.fftz > 0 ? p->opt.fftz : sponge_amd_get_fft_parameter(lz / p->opt.grid_spacing);
    const int dims[3] = {p->fx, p->fy, p->fz};
    for (int d = 0; d < 3; ++d) {
        if (dims[d] < 4 || dims[d] > kMaxFftLen || !make_plan(dims[d], &p->plan[d])) {
            delete p;
            return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
        }
    }
    const int fx = p->fx, fy = p->fy, fz = p->fz;
    p->fzc = fz / 2 + 1;
    p->nall = (long long)fx * fy * fz;
    p->nfft = (long long)fx * fy * p->fzc;
    p->volume = p->cell.a11 * p->cell.a22 * p->cell.a33;
    p->beta = sponge_amd_get_beta(cutoff, p->opt.direct_tolerance);
    p->neutralizing_factor = -0.5 * 3.1415926535897932f / (p->beta * p->beta * p->volume);
    p->tl_z = lines_per_block(fz);
    p->tl_y = lines_per_block(fy);
    p->tl_x = lines_per_block(fx);

    std::vector<float> bct;
    bc_table(p, bct);
    int e = 0;
    for (int d = 0; d < 3; ++d) e |= dmalloc(&p->d_tw[d], dims[d]);
    e |= dmalloc(&p->d_Q, p->nall);
    e |= dmalloc(&p->d_FQ, p->nfft);
    e |= dmalloc(&p->d_FBCFQ, p->nall);
    e |= dmalloc(&p->d_BCt, p->nfft);
    p->plane = p->plan[0].r1 && p->plan[1].r1 && plane_lds(p->fx, p->fy) <= kPlaneLds;
    e |= dmalloc(&p->d_acc, 9);
    e |= dmalloc(&p->d_part, (size_t)7 * p->fy * p->fzc);  // tilings down to one line
    e |= dmalloc(&p->d_qpart, (size_t)2 * grid_for(p->N, 256));
    e |= dmalloc(&p->d_ene, 2);
    e |= dmalloc(&p->d_direct_atom_energy, p->N);
    e |= dmalloc(&p->d_correction_atom_energy, p->N);
    e |= dmalloc(&p->d_sum, 2);
    p->bx = brick_edge(p->fx);
    p->by = brick_edge(p->fy);
    p->bz = brick_edge(p->fz);
    p->nbx = p->fx / p->bx;
    p->nby = p->fy / p->by;
    p->nbz = p->fz / p->bz;
    p->nb = p->nbx * p->nby * p->nbz;
    {
        // four times the mean occupancy plus a margin; denser bins go to the
        // overflow list
        const long long mean = ((long long)p->N + p->nb - 1) / p->nb;
        p->bcap = (int)(((4 * mean + 64) + 63) / 64 * 64);
    }
    e |= dmalloc(&p->d_bcount, (size_t)p->nb + 1);
    e |= dmalloc(&p->d_bw, (size_t)p->nb * p->bcap);
    e |= dmalloc(&p->d_bu, (size_t)p->nb * p->bcap);
    e |= dmalloc(&p->d_ow, (size_t)p->N);
    e |= dmalloc(&p->d_ou, (size_t)p->N);
    e |= dmalloc(&p->d_bi, (size_t)p->nb * p->bcap);
    e |= dmalloc(&p->d_oi, (size_t)p->N);
    e |= dmalloc(&p->d_gcount, (size_t)p->nb + 1);
    {
        // tile copies per spread workgroup: as many as let every brick's
        // workgroup be resident at once (160 KB of LDS per CU, 256 CUs), 1..4
        const TileGeom tg = pme_tile_geom(p);
        const long long per_cu = (p->nb + 255) / 256;
        const long long bytes = (long long)tg.lds_floats() * (long long)sizeof(float);
        const long long fit = (160LL * 1024) / (per_cu * bytes);
        p->spread_waves = (int)std::max(1LL, std::min(4LL, fit));
        e |= dmalloc(&p->d_tiles, (size_t)p->nb * tg.points());
    }
    if (e) {
        pme_free(p);
        delete p;
        return SPONGE_AMD_ERROR_MALLOC_FAILED;
    }
    hipStream_t s = p->stream;
    hipError_t he = hipSuccess;
    for (int d = 0; d < 3 && he == hipSuccess; ++d) {
        std::vector<float2> tw(dims[d]);
        for (int t = 0; t < dims[d]; ++t) {
            const double a = -2.0 * M_PI * (double)t / dims[d];
            tw[t] = make_float2((float)cos(a), (float)sin(a));
        }
        he = hipMemcpyAsync(p->d_tw[d], tw.data(), tw.size() * sizeof(float2), hipMemcpyHostToDevice, s);
        if (he == hipSuccess) he = hipStreamSynchronize(s);
    }
    if (he == hipSuccess)
        he = hipMemcpyAsync(p->d_BCt, bct.data(), bct.size() * sizeof(float), hipMemcpyHostToDevice, s);
    int fe = 0;
    if (he == hipSuccess) {
        fe |= fill_async(p->d_acc, 0.0, 9, s);
        fe |= fill_async(p->d_bcount, 0, p->nb + 1, s);
        fe |= fill_async(p->d_ene, 0.f, 2, s);
        fe |= fill_async(p->d_Q, 0.f, p->nall, s);
        fe |= fill_async(p->d_FBCFQ, 0.f, p->nall, s);
        fe |= fill_async(p->d_direct_atom_energy, 0.f, p->N, s);
        fe |= fill_async(p->d_correction_atom_energy, 0.f, p->N, s);
        he = hipStreamSynchronize(s);
    }
    if (he != hipSuccess || fe) {
        pme_free(p);
        delete p;
        return he != hipSuccess ? (int)he : fe;
    }
    *out = p;
    return 0;
}

extern "C" int sponge_pme_info(sponge_pme* p, float* beta, int* fft) {
    if (!p) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    if (beta) *beta = p->beta;
    if (fft) {
        fft[0] = p->fx;
        fft[1] = p->fy;
        fft[2] = p->fz;
    }
    return 0;
}

extern "C" float* sponge_pme_direct_atom_energy(sponge_pme* p) {
    return p ? p->d_direct_atom_energy : nullptr;
}

// (energy and virial leave as partial sums per workgroup, which the gather adds up)
static int pme_fft_convolve(sponge_pme* p, int need_virial, int need_energy) {
    hipStream_t s = p->stream;
    const int fx = p->fx, fy = p->fy, fz = p->fz, fzc = p->fzc;
    // LDS of a line transform: the exchange array of two factors, or two
    // ping-pong buffers and the twiddles
    auto exchange = [](const sa_radix_plan& pl) { return pl.r1 * (pl.r2 + 1); };
    {
        const int TL = p->tl_z, np = (TL + 1) / 2;
        const sa_radix_plan& pl = p->plan[2];
        const size_t sh = (pl.r1 ? (size_t)np * (exchange(pl) + fz + 1) : (size_t)(2 * np + 1) * fz) * sizeof(float2);
        ScopedTimer timer("pme_fft_z_r2c", s);
        SA_LAUNCH(128, (&fft_z_r2c_body), (k_fft_z_r2c), dim3(grid_for(fy, TL) * fx), dim3(128),
                  sh, s, p->d_Q, p->d_FQ, fx, fy, fz, fzc, TL, pl, p->d_tw[2]);
        SA_LAUNCH_CHECK();
    }
    const ReciprocalGeom rg{p->rcell, kPI * kPI / p->beta / p->beta};
    if (pme_plane(p)) {
        const size_t sh = plane_lds(fx, fy);
        ScopedTimer timer("pme_fft_plane", s);
        if (need_energy || need_virial)
            SA_LAUNCH(kPlaneThreads, (&fft_plane_body<true>), (k_fft_plane<true>), dim3(fzc),
                      dim3(kPlaneThreads), sh, s, p->d_FQ, p->d_BCt, rg, fx, fy, fz, fzc, p->plan[0],
                      p->plan[1], p->d_tw[0], p->d_tw[1], need_virial, p->d_part);
        else
            SA_LAUNCH(kPlaneThreads, (&fft_plane_body<false>), (k_fft_plane<false>), dim3(fzc),
                      dim3(kPlaneThreads), sh, s, p->d_FQ, p->d_BCt, rg, fx, fy, fz, fzc, p->plan[0],
                      p->plan[1], p->d_tw[0], p->d_tw[1], need_virial, p->d_part);
        SA_LAUNCH_CHECK();
    } else {
        auto y_lds = [&](int TL) {
            const sa_radix_plan& pl = p->plan[1];
            return (size_t)(pl.r1 ? TL * exchange(pl) : (2 * TL + 1) * fy) * sizeof(float2);
        };
        {
            const int TL = p->tl_y, nlines = fzc * fx;
            ScopedTimer timer("pme_fft_y", s);
            SA_LAUNCH(256, (&fft_y_body<-1>), (k_fft_y<-1>), dim3(grid_for(nlines, TL)), dim3(256), y_lds(TL),
                      s, p->d_FQ, nlines, fy, TL, p->plan[1], p->d_tw[1]);
            SA_LAUNCH_CHECK();
        }
        {
            const int TL = p->tl_x;
            const sa_radix_plan& pl = p->plan[0];
            const size_t sh = (pl.r1 ? (size_t)fx * (TL + 1) : (size_t)(2 * TL + 1) * fx) * sizeof(float2);
            ScopedTimer timer("pme_fft_x_conv", s);
            const dim3 grid(grid_for(fy, TL) * fzc);
            if (need_energy || need_virial)
                SA_LAUNCH(256, (&fft_x_conv_body<true>), (k_fft_x_conv<true>), grid, dim3(256), sh, s,
                          p->d_FQ, p->d_BCt, rg, fx, fy, fz, fzc, TL, pl, p->d_tw[0], need_virial, p->d_part);
            else
                SA_LAUNCH(256, (&fft_x_conv_body<false>), (k_fft_x_conv<false>), grid, dim3(256), sh, s,
                          p->d_FQ, p->d_BCt, rg, fx, fy, fz, fzc, TL, pl, p->d_tw[0], need_virial, p->d_part);
            SA_LAUNCH_CHECK();
        }
        {
            const int TL = p->tl_y, nlines = fzc * fx;
            ScopedTimer timer("pme_ifft_y", s);
            SA_LAUNCH(256, (&fft_y_body<+1>), (k_fft_y<+1>), dim3(grid_for(nlines, TL)), dim3(256), y_lds(TL),
                      s, p->d_FQ, nlines, fy, TL, p->plan[1], p->d_tw[1]);
            SA_LAUNCH_CHECK();
        }
    }
    {
        const int TL = p->tl_z, np = (TL + 1) / 2;
        const sa_radix_plan& pl = p->plan[2];
        const size_t sh = ((size_t)fzc * (TL | 1) + (size_t)(pl.r1 ? np * exchange(pl) : (2 * np + 1) * fz)) * sizeof(float2);
        ScopedTimer timer("pme_fft_z_c2r", s);
        SA_LAUNCH(128, (&fft_z_c2r_body), (k_fft_z_c2r), dim3(grid_for(fy, TL) * fx), dim3(128),
                  sh, s, p->d_FQ, p->d_FBCFQ, fx, fy, fz, fzc, TL, pl, p->d_tw[2]);
        SA_LAUNCH_CHECK();
    }
    return 0;
}

// The reciprocal force in two halves, so that a caller can run the first (bin,
// spread, FFT convolution: it reads only the coordinates and charges) on a
// stream of its own beside other work and join before the second (gather,
// energy), which adds to the force array.  Both use the module's stream.
bool sa::pme_plane(const sponge_pme* p) { return p->plane && (!g_recorder || g_recorder->plane); }

int sa::pme_spread_waves(const sponge_pme* p) { return p->spread_waves; }

void sa::pme_set_spread_waves(sponge_pme* p, int waves) {
    if (waves >= 1 && waves <= p->spread_waves) p->spread_waves = waves;
}

int sa::pme_recip_begin(sponge_pme* p, const float* crd, const float* cell, const float* rcell,
                        const float* charge, int need_virial, int need_energy, int step) {
    const LT6 c = lt_from(cell), r = lt_from(rcell);
    if (memcmp(&c, &p->cell, sizeof(LT6)) != 0) return SPONGE_AMD_ERROR_CONFLICTING_COMMAND;
    if (step % p->opt.update_interval != 0) return 0;
    hipStream_t s = p->stream;
    const int N = p->N;
    {
        ScopedTimer timer("pme_spread", s);
        SA_LAUNCH(256, (&pme_bin_body), (k_pme_bin), dim3(grid_for(N, 256)), dim3(256), 0, s, N, crd, charge, r, p->fx, p->fy, p->fz, p->bx, p->by, p->bz, p->nbx, p->nby, p->nbz, p->nb,
                           p->bcap, p->d_bcount, p->d_bw, p->d_bu, p->d_bi, p->d_ow, p->d_ou,
                           p->d_oi, need_energy ? p->d_qpart : nullptr);
        SA_LAUNCH_CHECK();
        const TileGeom tg = pme_tile_geom(p);
        const size_t sh = sizeof(float) * (size_t)p->spread_waves * tg.lds_floats();
        SA_LAUNCH(256, (&pme_spread_tiles_body), (k_pme_spread_tiles), dim3(p->nb), dim3(kWave * p->spread_waves), sh, s,
                           p->bx, p->by, p->bz, p->nbx, p->nby, p->nbz, p->nb, p->bcap, tg,
                           p->d_bcount, p->d_bw, p->d_bu, p->d_ow, p->d_ou, p->d_tiles);
        SA_LAUNCH_CHECK();
        SA_LAUNCH(256, (&pme_tiles_reduce_body), (k_pme_tiles_reduce), dim3(p->nb), dim3(256), 0, s, p->fx, p->fy, p->fz,
                           p->bx, p->by, p->bz, p->nbx, p->nby, p->nbz, p->nb, tg, p->d_tiles,
                           p->d_Q, p->d_bcount, p->d_gcount);
        SA_LAUNCH_CHECK();
    }
    // the energy sum is kept for the energy of later steps between
    // reciprocal updates, so it is accumulated on every update then
    return pme_fft_convolve(p, need_virial, need_energy || p->opt.update_interval > 1);
}

int sa::pme_recip_end(sponge_pme* p, const float* rcell, const float* charge, float* frc,
                      int need_virial, int need_energy, float* d_virial, float* d_potential,
                      int step, GatherBase gb) {
    const LT6 r = lt_from(rcell);
    hipStream_t s = p->stream;
    const int N = p->N;
    if (step % p->opt.update_interval == 0) {
        SpectrumTotals sums;
        if (need_virial || need_energy || p->opt.update_interval > 1) {
            sums.part = p->d_part;
            sums.nx = pme_plane(p) ? p->fzc : grid_for(p->fy, p->tl_x) * p->fzc;
            sums.acc = p->d_acc;
            sums.virial = need_virial ? d_virial : nullptr;
            if (need_energy) {
                sums.qpart = p->d_qpart;
                sums.nq = grid_for(N, 256);
                sums.ene = p->d_ene;
                sums.potential = d_potential;
                sums.self_factor = -p->beta / sqrtf(kPI);
                sums.neutralizing_factor = p->neutralizing_factor;
            }
        }
        ScopedTimer timer("pme_gather", s);
        const TileGeom tg = pme_tile_geom(p);
        SA_LAUNCH(256, (&pme_gather_tiles_body), (k_pme_gather_tiles), dim3(p->nb + (sums.part ? 1 : 0)), dim3(kGatherThreads),
                           sizeof(float) * tg.lds_floats(), s, p->fx, p->fy, p->fz, p->bx, p->by,
                           p->bz, p->nbx, p->nby, p->nbz, p->nb, p->bcap, tg, p->d_gcount, p->d_bw,
                           p->d_bu, p->d_bi, p->d_ow, p->d_ou, p->d_oi, p->d_FBCFQ, r,
                           (float)p->opt.update_interval, frc, gb, p->cell, p->beta, sums);
        SA_LAUNCH_CHECK();
    } else if (need_energy) {
        // between updates: the energy sum of the last one, this call's charges
        int rc = fill_async(p->d_acc + 7, 0.0, 2, s);
        if (rc) return rc;
        hipLaunchKernelGGL(k_pme_charge_sums, dim3(64), dim3(256), 0, s, N, charge, p->d_acc);
        SA_LAUNCH_CHECK();
        const float self_factor = -p->beta / sqrtf(kPI);
        hipLaunchKernelGGL(k_pme_energy_final, dim3(1), dim3(1), 0, s, p->d_acc, p->d_ene,
                           d_potential, self_factor, p->neutralizing_factor);
        SA_LAUNCH_CHECK();
    }
    return 0;
}

hipStream_t sa::pme_stream(const sponge_pme* p) { return p->stream; }
bool sa::pme_calculates_reciprocal(const sponge_pme* p) { return p->opt.calculate_reciprocal_part != 0; }
bool sa::pme_updates_on(const sponge_pme* p, int step) { return step % p->opt.update_interval == 0; }
void sa::pme_set_stream(sponge_pme* p, hipStream_t s) { p->stream = s; }

extern "C" int sponge_pme_reciprocal_force(sponge_pme* p, const float* crd, const float* cell,
                                           const float* rcell, const float* charge, float* frc,
                                           int need_virial, int need_energy, float* d_virial,
                                           float* d_potential, int step) {
    if (!p || !crd || !cell || !rcell || !charge || !frc) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    if (!p->opt.calculate_reciprocal_part) return 0;
    if ((need_virial && !d_virial) || (need_energy && !d_potential))
        return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    int rc = sa::pme_recip_begin(p, crd, cell, rcell, charge, need_virial, need_energy, step);
    if (rc) return rc;
    return sa::pme_recip_end(p, rcell, charge, frc, need_virial, need_energy, d_virial,
                             d_potential, step);
}

extern "C" int sponge_pme_excluded_force(sponge_pme* p, int local_atom_numbers,
                                         const int* atom_local, const int* atom_local_id,
                                         const float* crd, const float* cell, const float* rcell,
                                         const float* charge, const int* excluded_list_start,
                                         const int* excluded_list, const int* excluded_numbers,
                                         float* frc, int need_energy, float* atom_energy,
                                         int need_virial, float* atom_virial) {
    (void)atom_local;
    (void)atom_local_id;
    if (!p || !crd || !cell || !rcell || !charge || !frc) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    if (!p->opt.calculate_excluded_part) return 0;
    if (!excluded_list_start || !excluded_list || !excluded_numbers)
        return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    if ((need_energy && !atom_energy) || (need_virial && !atom_virial))
        return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    if (local_atom_numbers <= 0) return 0;
    if (local_atom_numbers > p->N) return SPONGE_AMD_ERROR_CONFLICTING_COMMAND;
    hipStream_t s = p->stream;
    if (need_energy) {
        int rc = fill_async(p->d_correction_atom_energy, 0.f, local_atom_numbers, s);
        if (rc) return rc;
    }
    const LT6 c = lt_from(cell), r = lt_from(rcell);
    dim3 grid(grid_for(local_atom_numbers, 256)), block(256);
    if (lt_is_orthorhombic(c))
        SA_LAUNCH(256, (&pme_excluded_body<true>), (k_pme_excluded<true>), grid, block, 0, s, local_atom_numbers, crd, charge, c, r, p->beta, excluded_list_start, excluded_list, excluded_numbers, frc,
                           need_energy, atom_energy, p->d_correction_atom_energy, need_virial,
                           atom_virial);
    else
        SA_LAUNCH(256, (&pme_excluded_body<false>), (k_pme_excluded<false>), grid, block, 0, s, local_atom_numbers, crd, charge, c, r, p->beta, excluded_list_start, excluded_list,
                           excluded_numbers, frc, need_energy, atom_energy,
                           p->d_correction_atom_energy, need_virial, atom_virial);
    SA_LAUNCH_CHECK();
    return 0;
}

extern "C" int sponge_pme_step_print(sponge_pme* p, float* PM, float* direct, float* reciprocal,
                                     float* self_energy, float* correction) {
    if (!p) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    hipStream_t s = p->stream;
    int rc = fill_async(p->d_sum, 0.0, 2, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_sum2_f32, dim3(64), dim3(256), 0, s, p->N, p->d_direct_atom_energy,
                       p->d_correction_atom_energy, p->d_sum);
    SA_LAUNCH_CHECK();
    double hs[2];
    float he[2];
    SA_CHECK(hipMemcpyAsync(hs, p->d_sum, sizeof(hs), hipMemcpyDeviceToHost, s));
    SA_CHECK(hipMemcpyAsync(he, p->d_ene, sizeof(he), hipMemcpyDeviceToHost, s));
    SA_CHECK(hipStreamSynchronize(s));
    const float dir = (float)hs[0], corr = (float)hs[1];
    if (direct) *direct = dir;
    if (correction) *correction = corr;
    if (reciprocal) *reciprocal = he[0];
    if (self_energy) *self_energy = he[1];
    if (PM) *PM = dir + he[0] + he[1] + corr;
    return 0;
}

extern "C" int sponge_pme_grids(sponge_pme* p, float* Q, float* FBCFQ) {
    if (!p) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    if (Q) SA_CHECK(hipMemcpyAsync(Q, p->d_Q, p->nall * sizeof(float), hipMemcpyDeviceToDevice, p->stream));
    if (FBCFQ)
        SA_CHECK(hipMemcpyAsync(FBCFQ, p->d_FBCFQ, p->nall * sizeof(float), hipMemcpyDeviceToDevice,
                                p->stream));
    return 0;
}

// Particle_Mesh::Update_Box (PM_force.cpp:1240-1256): the BC table and the
// neutralizing factor of a new box (same grid); synchronises.
extern "C" int sponge_pme_update_box(sponge_pme* p, const float* cell, const float* rcell) {
    if (!p || !cell || !rcell) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    const LT6 c = lt_from(cell);
    p->cell = c;
    p->rcell = lt_from(rcell);
    p->volume = p->cell.a11 * p->cell.a22 * p->cell.a33;
    p->neutralizing_factor = -0.5 * 3.1415926535897932f / (p->beta * p->beta * p->volume);
    std::vector<float> bct;
    bc_table(p, bct);
    SA_CHECK(hipMemcpyAsync(p->d_BCt, bct.data(), bct.size() * sizeof(float), hipMemcpyHostToDevice,
                            p->stream));
    SA_CHECK(hipStreamSynchronize(p->stream));
    return 0;
}

// Autotuner of the FFT passes' tiling: lines per workgroup of the z, y and
// x passes, each chosen in turn (the others held) as the fastest of a few
// candidates by HIP-event timing of whole reciprocal-force calls on the
// module's stream.  Every tiling computes the same per-line transforms, so
// forces do not depend on the choice.  On a grid whose planes are transformed in
// LDS only the z tiling reaches a kernel: the other two keep their values.
extern "C" int sponge_pme_autotune(sponge_pme* p, const float* crd, const float* charge, int reps,
                                   int* chosen) {
    if (!p || !crd || !charge || reps < 1) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    hipStream_t s = p->stream;
    float* frc = nullptr;
    int rc = dmalloc(&frc, (size_t)3 * p->N);
    if (rc) return rc;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        if (e0) (void)hipEventDestroy(e0);
        dfree(frc);
        return SPONGE_AMD_ERROR_MALLOC_FAILED;
    }
    const float* cell = &p->cell.a11;
    const float* rcell = &p->rcell.a11;
    float best_ms = 0.f;
    auto measure = [&](float* ms) -> int {
        int r = sponge_pme_reciprocal_force(p, crd, cell, rcell, charge, frc, 0, 0, nullptr, nullptr, 0);
        if (r) return r;
        SA_CHECK(hipEventRecord(e0, s));
        for (int k = 0; k < reps && !r; ++k)
            r = sponge_pme_reciprocal_force(p, crd, cell, rcell, charge, frc, 0, 0, nullptr, nullptr, 0);
        if (r) return r;
        SA_CHECK(hipEventRecord(e1, s));
        SA_CHECK(hipEventSynchronize(e1));
        SA_CHECK(hipEventElapsedTime(ms, e0, e1));
        return 0;
    };
    int* axes[3] = {&p->tl_z, &p->tl_y, &p->tl_x};
    const int cand[4] = {2, 4, 8, 16};
    rc = measure(&best_ms);
    const int tuned = pme_plane(p) ? 1 : 3;
    for (int a = 0; a < tuned && !rc; ++a) {
        const int keep = *axes[a];
        int best = keep;
        for (int c : cand) {
            if (c == keep) continue;
            *axes[a] = c;
            float ms = 0.f;
            rc = measure(&ms);
            if (rc) break;
            if (ms < best_ms) {
                best_ms = ms;
                best = c;
            }
        }
        *axes[a] = best;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipStreamSynchronize(s);
    dfree(frc);
    if (!rc && chosen) {
        chosen[0] = p->tl_z;
        chosen[1] = p->tl_y;
        chosen[2] = p->tl_x;
    }
    return rc;
}

extern "C" int sponge_pme_set_fft_tiling(sponge_pme* p, const int* tiles) {
    if (!p || !tiles) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    // even line counts up to 16 (the candidates of the autotuner)
    for (int a = 0; a < 3; ++a)
        if (tiles[a] < 2 || tiles[a] > 16 || (tiles[a] & 1)) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    p->tl_z = tiles[0];
    p->tl_y = tiles[1];
    p->tl_x = tiles[2];
    return 0;
}

extern "C" int sponge_pme_clear(sponge_pme* p) {
    if (!p) return 0;
    (void)hipStreamSynchronize(p->stream);
    pme_free(p);
    delete p;
    return 0;
}

extern "C" const char* sponge_amd_version(void) { return "sponge_amd 0.1.0 (gfx950)"; }
