// Learned reciprocal-force surrogate: a per-atom MLP over local charge-
// environment features that stands in for the PME reciprocal force on the
// steps between full PME evaluations.  It has no counterpart in the
// reference; it sits beside PM_force (SPONGE/PM_force/PM_force.cpp), whose
// PME_Reciprocal_Force_With_Energy_And_Virial (:1070-1169) stays the
// fallback and the reference force every sampled step is checked against.
//
// Features of atom i (partners j on the neighbor list with r < Rf; d = r_j -
// r_i, u = r / Rf, fc = (1 - u^2)^2, w_j = q_j fc, x = 2u - 1, T_k Chebyshev):
//   R_k = sum w_j T_k(x), k < 32;  P_a = sum w_j T_a(x) d / r, a < 5;
//   S = sum w_j d d^T / r^2, Q = S - R_0 / 3 I;
//   angular = [P_a . P_b, a <= b] (15) + |Q|_F^2 (1).
// Basis vectors: U_0 = sum q_j fc phi'(r) d / r over the list partners,
// U_1 = sum q_j phi'(r) d / r over the excluded partners, U_2 = P_0, with
// phi(r) = erf(beta r) / r.  Predicted reciprocal force of atom i:
//   F_i = q_i (c_0 U_0 + c_1 U_1 + c_2 U_2),  c = MLP(normalised features),
// MLP 48 -> 64 -> 64 -> 3 with SiLU.  The coefficients (1, 1, 0) are the
// near-field reciprocal force itself (the physics baseline the network
// starts from and is compared with).
//
// Layout in HBM: features [N][48] FP32 and basis [N][3] float4 in the neighbor
// list's sorted order; model parameters FP32 (master) with BF16 copies in the
// MFMA operand order; training frames (features, basis, target force + charge)
// kept resident, [F][N] each.  The MLP runs on v_mfma_f32_16x16x16_bf16: a
// wave owns 16 atoms and computes every layer transposed (outputs x atoms),
// so that one layer's accumulator fragment is the next layer's B operand
// without a shuffle.
#include <algorithm>
#include <cmath>
#include <random>
#include <vector>

#include "internal.h"
#include "timing.h"

using namespace sa;

namespace {

constexpr int kRadial = 32, kVec = 5, kAngular = 16, kFeat = kRadial + kAngular;
constexpr int kHidden = 64, kOut = 3;
constexpr int oW1 = 0, oB1 = oW1 + kHidden * kFeat, oW2 = oB1 + kHidden;
constexpr int oB2 = oW2 + kHidden * kHidden, oW3 = oB2 + kHidden, oB3 = oW3 + kOut * kHidden;
constexpr int kParams = oB3 + kOut;
constexpr int kModel = kParams + 2 * kFeat;  // + feature mean and inverse std
constexpr int kFeatStage = 3584;
constexpr float kTwoOverSqrtPiF = 1.1283791670955126f;

}  // namespace

struct sponge_rsur {
    int N = 0;
    float rf = 0, beta = 0;
    sponge_rsur_options opt{};
    hipStream_t stream = nullptr;
    StreamOwner owner;             // of the stream, when it is a step driver's
    int stage = 0;
    const int* sidx = nullptr;     // sorted -> local order of the last feature call's list
    const float4* pos_last = nullptr;  // sorted positions + charges the last features used
    float4* d_pos = nullptr;       // [N] sorted x, y, z, charge
    float* d_feat = nullptr;       // [N][48] sorted order
    float4* d_basis = nullptr;     // [N][3] sorted order
    float4* d_uex = nullptr;       // [N] exclusion field, local order
    int* d_moved = nullptr;        // epoch of the last call with an atom beyond the list's skin bound
    int epoch = 0;                 // feature calls on the module's own pack
    float* d_params = nullptr;     // [kParams] FP32 master copy
    float* d_norm = nullptr;       // [96] feature mean, inverse std
    unsigned short* d_w1 = nullptr;   // [64][48] bf16
    unsigned short* d_w2 = nullptr;   // [64][64]
    unsigned short* d_w2t = nullptr;  // [64][64] transposed
    unsigned short* d_w3 = nullptr;   // [16][64], rows >= 3 zero
    unsigned short* d_w3t = nullptr;  // [64][16], columns >= 3 zero
    float* d_part = nullptr;       // partial gradients of a training pass
    double* d_lpart = nullptr;     // its partial losses
    float* h_grad = nullptr;       // pinned: gradient and loss of a gradient call
    float* d_m = nullptr;          // Adam moments
    float* d_v = nullptr;
    double* d_acc = nullptr;       // [0] loss, [1..3] sums, [8..104) feature stats, [104..110) evaluation
    long long adam_t = 0;
    int n_frames = 0;
    float* d_ffeat = nullptr;      // [F][N][48]
    float4* d_fbasis = nullptr;    // [F][N][3]
    float4* d_ftarget = nullptr;   // [F][N] target force, w = charge
};

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned short f2bf(float f) {
    // round to nearest even (finite inputs)
    unsigned u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x4 pack4(float a, float b, float c, float d) {
    bf16x4 v;
    v[0] = (short)f2bf(a);
    v[1] = (short)f2bf(b);
    v[2] = (short)f2bf(c);
    v[3] = (short)f2bf(d);
    return v;
}

__device__ __forceinline__ bf16x4 load4(const unsigned short* p) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    bf16x4 v;
    v[0] = (short)(u.x & 0xffffu);
    v[1] = (short)(u.x >> 16);
    v[2] = (short)(u.y & 0xffffu);
    v[3] = (short)(u.y >> 16);
    return v;
}

__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }

// DPP read of another lane of the row (VALU only, no LDS traffic)
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_read(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xf, true));
}

// d/dr [erf(beta r) / r] / r, times the caller's weights
__device__ __forceinline__ float dphi_over_r(float r, float rinv, float beta) {
    const float x = beta * r;
    return (kTwoOverSqrtPiF * x * __expf(-x * x) - erff(x)) * rinv * rinv * rinv;
}

// Sorted positions and charges of the call; clears the excluded partners'
// field, and marks the call (moved = epoch) when an atom is further from its
// build position than the list's skin permits.
__global__ void k_rs_pack(int N, const int* __restrict__ sidx, const float4* __restrict__ spos,
                          const float* __restrict__ crd, const float* __restrict__ charge, LT6 c,
                          LT6 r, float permit2, int epoch, float4* __restrict__ pos,
                          float4* __restrict__ uex, int* __restrict__ moved) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const int i = sidx[p];
    const float4 b = spos[p];
    const float3 x = make_float3(crd[3 * i], crd[3 * i + 1], crd[3 * i + 2]);
    pos[p] = make_float4(x.x, x.y, x.z, charge[i]);
    uex[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!(norm2_exact(disp_pbc<false>(x, make_float3(b.x, b.y, b.z), c, r)) <= permit2)) *moved = epoch;
}

// U_1: the reciprocal pair field of the excluded partners (both directions
// of the reference's half exclusion list)
template <bool ORTHO>
__global__ void k_rs_exfield(int N, const float* __restrict__ crd, const float* __restrict__ charge,
                             const int* __restrict__ ex_start, const int* __restrict__ ex_num,
                             const int* __restrict__ ex_list, LT6 c, LT6 r, float beta,
                             float4* __restrict__ uex) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int n = ex_num[i];
    if (n <= 0) return;
    const float3 pi = make_float3(crd[3 * i], crd[3 * i + 1], crd[3 * i + 2]);
    const float qi = charge[i];
    const int* lst = ex_list + ex_start[i];
    float fx = 0.f, fy = 0.f, fz = 0.f;
    for (int e = 0; e < n; ++e) {
        const int j = lst[e];
        const float3 pj = make_float3(crd[3 * j], crd[3 * j + 1], crd[3 * j + 2]);
        const float3 d = disp_pbc<ORTHO>(pj, pi, c, r);
        const float r2 = d.x * d.x + d.y * d.y + d.z * d.z;
        const float rinv = 1.0f / sqrtf(r2);
        const float g = dphi_over_r(r2 * rinv, rinv, beta);
        const float qj = charge[j];
        fx += qj * g * d.x;
        fy += qj * g * d.y;
        fz += qj * g * d.z;
        unsafeAtomicAdd(&uex[j].x, -qi * g * d.x);
        unsafeAtomicAdd(&uex[j].y, -qi * g * d.y);
        unsafeAtomicAdd(&uex[j].z, -qi * g * d.z);
    }
    unsafeAtomicAdd(&uex[i].x, fx);
    unsafeAtomicAdd(&uex[i].y, fy);
    unsafeAtomicAdd(&uex[i].z, fz);
}

// Features and basis vectors, one workgroup of 8 wavefronts per neighbor-list
// cell (or `split` of them): the cell's candidate stream (positions and
// charges) is staged in LDS once; one wavefront per row.
//
// The kernel is bound by VALU issue: about 110 instructions per pair within the
// feature radius, and two fifths of a row's list lie beyond it (radius 10,
// list 12 A).  So a row's entries are first tested (displacement and r^2 only)
// and those in range appended, 16 bytes each, to the wavefront's ring in LDS;
// the sums run on full batches of 64 of them.  The 32 radial sums are kept as
// products
//   M_pq = sum w T_8p T_q,  p < 4, q < 8,
// which cost 46 instructions against 62 for the recurrence up to T_31, and give
// R_8p+q = 2 M_pq - R_8p-q at the end.  The pair field takes the Ewald force
// polynomial where it holds (EwaldPoly), against erff and exp.  The row's 56
// lane sums are reduced by halving exchanges between lanes (lane 32 and 16
// swaps: two instructions per pair of sums) instead of six steps each, and the
// 48 features leave in one store.
// 24,000 atoms: 178 -> 70 us.  RMS error of the features against 64 bits there
// 1.4e-6 -> 1.0e-6 of a column's RMS (U_0 1.25e-6 -> 0.80e-6).
constexpr int kRsWaves = 8;    // wavefronts per workgroup
constexpr int kRsRing = 128;   // ring entries of a wavefront
constexpr int kRsSums = 56;    // 32 M, 15 P, 6 S, 3 U

// sum over the 16 lanes of a row, in every lane of it
__device__ __forceinline__ float row_total(float v) {
    v += dpp_read<0xb1, 0xf>(v);   // quad_perm [1, 0, 3, 2]
    v += dpp_read<0x4e, 0xf>(v);   // quad_perm [2, 3, 0, 1]
    v += dpp_read<0x141, 0xf>(v);  // row_half_mirror
    v += dpp_read<0x140, 0xf>(v);  // row_mirror
    return v;
}

// a and b over all 64 lanes -> lanes 0..31 hold a's sums of lane l and l + 32,
// lanes 32..63 b's
__device__ __forceinline__ float halve32(float a, float b) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// the same between the odd and even rows of 16 lanes: rows 0, 2 keep a, rows
// 1, 3 keep b
__device__ __forceinline__ float halve16(float a, float b) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// One batch of up to 64 in-range pairs added to the sums (d: displacement, q:
// the partner's charge, 0 in lanes without a pair).
template <bool POLY>
__device__ __forceinline__ void rs_batch(float4 dq, float inv_rf, float beta, const EwaldPoly& ew,
                                         float* __restrict__ acc) {
    const float r2 = fmaf(dq.z, dq.z, fmaf(dq.y, dq.y, dq.x * dq.x));
    const float rinv = __builtin_amdgcn_rsqf(r2);
    const float rr = r2 * rinv;
    const float u = rr * inv_rf;
    const float fb = fmaf(-u, u, 1.0f);
    const float w = dq.w * (fb * fb);
    const float x = 2.0f * u - 1.0f, x2 = 2.0f * x;
    float T[9];
    T[0] = 1.0f;
    T[1] = x;
#pragma unroll
    for (int k = 2; k <= 8; ++k) T[k] = fmaf(x2, T[k - 1], -T[k - 2]);
    const float t16 = fmaf(2.0f * T[8], T[8], -1.0f);
    const float t24 = fmaf(2.0f * T[8], t16, -T[8]);
    const float wp[4] = {w, w * T[8], w * t16, w * t24};
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        acc[8 * p] += wp[p];
#pragma unroll
        for (int q = 1; q < 8; ++q) acc[8 * p + q] = fmaf(wp[p], T[q], acc[8 * p + q]);
    }
    const float ex = dq.x * rinv, ey = dq.y * rinv, ez = dq.z * rinv;
#pragma unroll
    for (int a = 0; a < kVec; ++a) {
        const float b = a ? w * T[a] : w;
        acc[32 + 3 * a] = fmaf(b, ex, acc[32 + 3 * a]);
        acc[33 + 3 * a] = fmaf(b, ey, acc[33 + 3 * a]);
        acc[34 + 3 * a] = fmaf(b, ez, acc[34 + 3 * a]);
    }
    const float sx = w * ex, sy = w * ey, sz = w * ez;
    acc[47] = fmaf(sx, ex, acc[47]);
    acc[48] = fmaf(sx, ey, acc[48]);
    acc[49] = fmaf(sy, ey, acc[49]);
    acc[50] = fmaf(sx, ez, acc[50]);
    acc[51] = fmaf(sy, ez, acc[51]);
    acc[52] = fmaf(sz, ez, acc[52]);
    const float g = w * (POLY ? -ew(r2) : dphi_over_r(rr, rinv, beta));
    acc[53] = fmaf(g, dq.x, acc[53]);
    acc[54] = fmaf(g, dq.y, acc[54]);
    acc[55] = fmaf(g, dq.z, acc[55]);
}

// One row.  SHIFT: the staged positions and pi are offsets from the cell's
// centre at the images nearest to it.
template <bool ORTHO, bool STAGED, bool SHIFT, bool POLY>
__device__ __forceinline__ void rs_row(int p, int lane, int n, const unsigned short* __restrict__ row,
                                       const float4* src, const int* __restrict__ strm, float3 pi,
                                       const LT6& c, const LT6& r, float rf2, float inv_rf,
                                       float beta, const EwaldPoly& ew, float4* ring, float* sums,
                                       float* __restrict__ feat, float4* __restrict__ basis,
                                       const float4* __restrict__ uex_i) {
    float acc[kRsSums];
#pragma unroll
    for (int k = 0; k < kRsSums; ++k) acc[k] = 0.f;
    int head = 0, have = 0;
    // the next pass's entry is loaded before the current one is used, so
    // that the list's memory latency overlaps the arithmetic
    int cur = n > 0 ? (int)row[lane < n ? lane : n - 1] : 0;
    for (int e = lane; e - lane < n; e += kWave) {
        const bool has = e < n;
        const int en = e + kWave;
        int nxt = (int)row[en < n ? en : n - 1];
        const float4 pj = src[STAGED ? cur : strm[cur]];
        float3 d;
        float r2;
        if (SHIFT) {
            d = make_float3(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z);
            r2 = fmaf(d.z, d.z, fmaf(d.y, d.y, d.x * d.x));
        } else {
            d = disp_pbc<ORTHO>(make_float3(pj.x, pj.y, pj.z), pi, c, r);
            r2 = norm2_exact(d);
        }
        const bool in = has && r2 < rf2;
        const unsigned long long m = __ballot(in);
        if (in) ring[(head + have + lanes_below(m)) & (kRsRing - 1)] = make_float4(d.x, d.y, d.z, pj.w);
        have += (int)__popcll(m);
        if (have >= kWave) {
            wave_fence();
            rs_batch<POLY>(ring[(head + lane) & (kRsRing - 1)], inv_rf, beta, ew, acc);
            wave_fence();
            head = (head + kWave) & (kRsRing - 1);
            have -= kWave;
        }
        asm volatile("" : "+v"(nxt));
        cur = nxt;
    }
    if (have > 0) {
        wave_fence();
        float4 v = ring[(head + lane) & (kRsRing - 1)];
        // lanes without a pair: no charge, at a distance of the radius's order
        if (lane >= have) v = make_float4(1.f, 0.f, 0.f, 0.f);
        rs_batch<POLY>(v, inv_rf, beta, ew, acc);
        wave_fence();
    }
    // 56 sums over 64 lanes: after the two halvings register k (of 14) holds,
    // in row j of 16 lanes, sum 4 k + (0, 2, 1, 3)[j]
#pragma unroll
    for (int k = 0; k < 14; ++k) {
        const float lo = halve32(acc[4 * k], acc[4 * k + 1]), hi = halve32(acc[4 * k + 2], acc[4 * k + 3]);
        const float t = row_total(halve16(lo, hi));
        // row 0: a of lo, row 1: a of hi, row 2: b of lo, row 3: b of hi
        const int j = lane >> 4;
        if ((lane & 15) == 0) sums[4 * k + ((j & 1) << 1 | j >> 1)] = t;
    }
    wave_fence();
    // lane k: feature k
    float f = 0.f;
    if (lane < kRadial) {
        const int pp = lane >> 3, q = lane & 7;
        if (q == 0) {
            f = sums[8 * pp];
        } else {
            // R_8p+q = 2 M_p,q - 2 M_p-1,8-q + 2 M_p-2,q - ... with the last
            // term (M_0) single
            float sign = 1.f;
            for (int k = pp; k >= 0; --k) {
                const int qq = ((pp - k) & 1) ? 8 - q : q;
                f = fmaf(k ? 2.f * sign : sign, sums[8 * k + qq], f);
                sign = -sign;
            }
        }
    } else if (lane < kFeat - 1) {
        int a = 0, o = lane - kRadial;  // pair (a, b >= a) number o
        while (o >= kVec - a) {
            o -= kVec - a;
            ++a;
        }
        const float* A = sums + 32 + 3 * a;
        const float* B = sums + 32 + 3 * (a + o);
        f = A[0] * B[0] + A[1] * B[1] + A[2] * B[2];
    } else if (lane == kFeat - 1) {
        const float tr = sums[0] * (1.0f / 3.0f);
        const float q0 = sums[47] - tr, q2 = sums[49] - tr, q5 = sums[52] - tr;
        f = q0 * q0 + q2 * q2 + q5 * q5 +
            2.0f * (sums[48] * sums[48] + sums[50] * sums[50] + sums[51] * sums[51]);
    }
    if (lane < kFeat) feat[(size_t)kFeat * p + lane] = f;
    if (lane >= kFeat && lane < kFeat + 3) {
        const int m = lane - kFeat;
        const float4 ue = *uex_i;
        const float* u = m == 0 ? sums + 53 : sums + 32;
        basis[(size_t)3 * p + m] = m == 1 ? make_float4(ue.x, ue.y, ue.z, 0.f)
                                          : make_float4(u[0], u[1], u[2], 0.f);
    }
    wave_fence();  // sums is written again by the next row
}

// reach >= 0: every row atom lies within the pair kernel's bound of its build
// cell (and, with moved given, *moved != epoch: the pack of these coordinates
// found no atom beyond it), so partners are staged as offsets from the cell's
// centre, at their images nearest to it, in a box wide enough (see
// lj_cells_body).
template <bool ORTHO>
__global__ void __launch_bounds__(64 * kRsWaves) k_rs_features(
    const int* __restrict__ start, const int* __restrict__ g_stream,
    const long long* __restrict__ g_soff, const int* __restrict__ g_slen,
    const int* __restrict__ list_count, const unsigned short* __restrict__ list, int cap,
    const float4* __restrict__ pos, const int* __restrict__ sidx, LT6 c, LT6 r, float rf2,
    float inv_rf, float beta, EwaldPoly ew, int stage, int split, float3 width, int Nx, int Ny,
    int Nz, float reach, const int* __restrict__ moved, int epoch, const float4* __restrict__ uex,
    float* __restrict__ feat, float4* __restrict__ basis) {
    extern __shared__ float4 cpos[];
    const int cell = blockIdx.x / split, part = blockIdx.x - cell * split;
    const int a0 = start[cell], a1 = start[cell + 1];
    if (a0 + part * kRsWaves >= a1) return;
    float3 C = make_float3(0.f, 0.f, 0.f);
    bool shift = false;
    const int total = g_slen[cell];
    const bool staged = total <= stage;
    if (ORTHO && staged && reach >= 0.f && (!moved || *moved != epoch)) {
        const int ix = cell / (Ny * Nz), iy = (cell / Nz) % Ny, iz = cell % Nz;
        float lx, hx, ly, hy, lz, hz;
        cell_faces(ix, Nx, width.x, c.a11, lx, hx);
        cell_faces(iy, Ny, width.y, c.a22, ly, hy);
        cell_faces(iz, Nz, width.z, c.a33, lz, hz);
        C = image_centre(make_float3(0.5f * (lx + hx), 0.5f * (ly + hy), 0.5f * (lz + hz)), c);
        shift = 0.5f * c.a11 > reach + 0.5f * (hx - lx) + kCentreMargin &&
                0.5f * c.a22 > reach + 0.5f * (hy - ly) + kCentreMargin &&
                0.5f * c.a33 > reach + 0.5f * (hz - lz) + kCentreMargin;
    }
    const int* __restrict__ strm = g_stream + g_soff[cell];
    if (staged)
        stage_stream(
            strm, total, [&](int q) { return pos[q]; },
            [&](int t, const float4& v) {
                float4 x = v;
                if (shift) {
                    const float3 o = image_offset(make_float3(v.x, v.y, v.z), C, c, r);
                    x = make_float4(o.x, o.y, o.z, v.w);
                }
                cpos[t] = x;
            });
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    float4* ring = cpos + stage + kRsRing * wave;
    float* sums = reinterpret_cast<float*>(cpos + stage + kRsRing * kRsWaves) + kWave * wave;
    const bool poly = ew.scale > 0.f;
    for (int p = a0 + part * kRsWaves + wave; p < a1; p += split * kRsWaves) {
        const int n = list_count[p];
        const unsigned short* row = list + (size_t)p * cap;
        const float4* ue = uex + sidx[p];
        const float4 x = pos[p];
        float3 pi = make_float3(x.x, x.y, x.z);
        if (shift) pi = image_offset(pi, C, c, r);
#define SA_RS_ROW(S, SH, P, SRC)                                                                  \
    rs_row<ORTHO, S, SH, P>(p, lane, n, row, SRC, strm, pi, c, r, rf2, inv_rf, beta, ew, ring, sums, \
                            feat, basis, ue)
        if (shift && poly) SA_RS_ROW(true, true, true, cpos);
        else if (staged && poly) SA_RS_ROW(true, false, true, cpos);
        else if (staged)  // (offsets: disp_pbc holds for them as well)
            SA_RS_ROW(true, false, false, cpos);
        else SA_RS_ROW(false, false, false, pos);
#undef SA_RS_ROW
    }
}

// ----------------------------------------------------------------------------
// MLP on MFMA.  Lane l of a wave: atom column l & 15 of the wave's 16-atom
// tile, k-group kq = l >> 4.  Operand fragments of v_mfma_f32_16x16x16_bf16:
// A (M x K): row l & 15, k = 4 kq + j;  B (K x N): column l & 15, k = 4 kq + j;
// C (M x N): column l & 15, row 4 kq + j  (j = 0..3, the vector element).
// ----------------------------------------------------------------------------

struct Fwd {
    f32x4 d1[4], d2[4], c;  // d: SiLU's derivative (training only)
    bf16x4 x[3], h1[4], h2[4];
};

// SiLU of a tile as a bf16 fragment; training takes the derivative from the
// same sigmoid.
template <bool TRAIN>
__device__ __forceinline__ bf16x4 activate(const f32x4& z, f32x4& d) {
    float h[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (TRAIN) {
            const float s = 1.0f / (1.0f + __expf(-z[j]));
            d[j] = s * (1.0f + z[j] * (1.0f - s));
            h[j] = z[j] * s;
        } else {
            h[j] = silu(z[j]);
        }
    }
    return pack4(h[0], h[1], h[2], h[3]);
}

// Forward pass of one tile (rows p0 .. p0+15 of feat; rows >= N read as zero).
// TRAIN: with the derivatives, and one layer's weights in flight at a time (64
// registers fewer).
template <bool TRAIN = false>
__device__ __forceinline__ void mlp_forward(int p0, int N, int lane, const float* __restrict__ feat,
                                            const float* __restrict__ norm,
                                            const unsigned short* __restrict__ w1,
                                            const unsigned short* __restrict__ w2,
                                            const unsigned short* __restrict__ w3,
                                            const float* __restrict__ params, Fwd& f) {
    const int col = lane & 15, kq = lane >> 4;
    const int a = p0 + col;
    const bool ok = a < N;
#pragma unroll
    for (int kc = 0; kc < 3; ++kc) {
        const int k = kc * 16 + kq * 4;
        float4 v = ok ? *reinterpret_cast<const float4*>(feat + (size_t)kFeat * a + k)
                      : make_float4(0.f, 0.f, 0.f, 0.f);
        if (!ok) {
            // padding rows: normalised zeros
            v = make_float4(norm[k], norm[k + 1], norm[k + 2], norm[k + 3]);
        }
        f.x[kc] = pack4((v.x - norm[k]) * norm[kFeat + k], (v.y - norm[k + 1]) * norm[kFeat + k + 1],
                        (v.z - norm[k + 2]) * norm[kFeat + k + 2],
                        (v.w - norm[k + 3]) * norm[kFeat + k + 3]);
    }
    if (TRAIN) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int o = t * 16 + kq * 4;
        f32x4 acc = {params[oB1 + o], params[oB1 + o + 1], params[oB1 + o + 2], params[oB1 + o + 3]};
#pragma unroll
        for (int kc = 0; kc < 3; ++kc)
            acc = mfma16(load4(w1 + (size_t)(t * 16 + col) * kFeat + kc * 16 + kq * 4), f.x[kc], acc);
        f.h1[t] = activate<TRAIN>(acc, f.d1[t]);
    }
    if (TRAIN) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int o = t * 16 + kq * 4;
        f32x4 acc = {params[oB2 + o], params[oB2 + o + 1], params[oB2 + o + 2], params[oB2 + o + 3]};
#pragma unroll
        for (int kc = 0; kc < 4; ++kc)
            acc = mfma16(load4(w2 + (size_t)(t * 16 + col) * kHidden + kc * 16 + kq * 4), f.h1[kc], acc);
        f.h2[t] = activate<TRAIN>(acc, f.d2[t]);
    }
    if (TRAIN) __builtin_amdgcn_sched_barrier(0);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (kq == 0) {
        acc[0] = params[oB3];
        acc[1] = params[oB3 + 1];
        acc[2] = params[oB3 + 2];
    }
#pragma unroll
    for (int kc = 0; kc < 4; ++kc)
        acc = mfma16(load4(w3 + (size_t)col * kHidden + kc * 16 + kq * 4), f.h2[kc], acc);
    f.c = acc;  // lanes kq == 0: c_0, c_1, c_2 of atom p0 + col
}

// Inference: frc[local] += q (c . U), over tiles of 16 sorted atoms.
__global__ void __launch_bounds__(256) k_rs_predict(
    int N, int ntiles, const float* __restrict__ feat, const float4* __restrict__ basis,
    const float4* __restrict__ pos, const int* __restrict__ sidx, const float* __restrict__ norm,
    const unsigned short* __restrict__ w1, const unsigned short* __restrict__ w2,
    const unsigned short* __restrict__ w3, const float* __restrict__ params, float* __restrict__ frc,
    int assign, const float* __restrict__ anchor) {
    const int lane = threadIdx.x & 63;
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int nw = (gridDim.x * blockDim.x) >> 6;
    for (int tile = wave; tile < ntiles; tile += nw) {
        Fwd f;
        mlp_forward(tile * 16, N, lane, feat, norm, w1, w2, w3, params, f);
        const int a = tile * 16 + (lane & 15);
        if ((lane >> 4) == 0 && a < N) {
            const float q = pos[a].w;
            const float4 u0 = basis[3 * (size_t)a], u1 = basis[3 * (size_t)a + 1],
                         u2 = basis[3 * (size_t)a + 2];
            float fx = q * (f.c[0] * u0.x + f.c[1] * u1.x + f.c[2] * u2.x);
            float fy = q * (f.c[0] * u0.y + f.c[1] * u1.y + f.c[2] * u2.y);
            float fz = q * (f.c[0] * u0.z + f.c[1] * u1.z + f.c[2] * u2.z);
            const size_t i = (size_t)sidx[a];
            if (anchor) {
                fx += anchor[3 * i];
                fy += anchor[3 * i + 1];
                fz += anchor[3 * i + 2];
            }
            float* o = frc + 3 * i;
            if (assign) {
                o[0] = fx;
                o[1] = fy;
                o[2] = fz;
            } else {
                o[0] += fx;
                o[1] += fy;
                o[2] += fz;
            }
        }
    }
}

// Training pass over one frame: forward, loss, backward, and the gradients of
// one workgroup's atoms, written as one partial per workgroup (k_rs_reduce
// sums them; every workgroup adding its 7,491 sums to the same addresses took
// most of the kernel's time).
//
// A workgroup of 8 wavefronts takes 128 atoms at a time.  Each wavefront runs
// 16 of them forward and back in registers, as in inference, and leaves its
// operands of the weight gradients in LDS as bf16 [row][atom] (x, h1, h2, dZ1,
// dZ2, dc).  The gradients are then 32 tiles of 16 x 16 contracted over the 128
// atoms, four tiles to a wavefront: 16 accumulator registers each against 128
// when every wavefront kept all of them, and two barriers per 128 atoms against
// about 50 per 16.  Rows are 132 entries (264 bytes) long: 8-byte fragment
// reads stay aligned and conflict at most in pairs, and two workgroups fit on
// a CU.
// 24,000 atoms (188 workgroups, one pass each): 124 -> 22 us, now the latency of
// one pass through 3,000 instructions; the sums take 4 us (k_rs_reduce).
constexpr int kTrWaves = 8, kTrAtoms = 16 * kTrWaves, kTrRow = kTrAtoms + 4;
constexpr int kTrX = 0, kTrH1 = kTrX + kFeat, kTrH2 = kTrH1 + kHidden, kTrZ1 = kTrH2 + kHidden;
constexpr int kTrZ2 = kTrZ1 + kHidden, kTrC = kTrZ2 + kHidden, kTrRows = kTrC + kOut;
constexpr int kTrGroups = 512;                       // workgroups (partials) at most
constexpr int kTrPart = (kParams + 63) / 64 * 64;    // floats of a partial

// Tile in C layout (rows 4 kq + 0..3 of it from `row`, column = atom) to LDS:
// two lanes exchange halves, so that each stores pairs of atoms.
template <int ROWS>
__device__ __forceinline__ void tr_store(unsigned short* T, int row, int wave, int lane, bf16x4 v) {
    const int col = lane & 15, kq = lane >> 4, odd = lane & 1;
    const unsigned a = (unsigned)(unsigned short)v[0] | (unsigned)(unsigned short)v[1] << 16;
    const unsigned b = (unsigned)(unsigned short)v[2] | (unsigned)(unsigned short)v[3] << 16;
    const unsigned oa = (unsigned)__builtin_amdgcn_update_dpp(0, (int)a, 0xb1, 0xf, 0xf, true);
    const unsigned ob = (unsigned)__builtin_amdgcn_update_dpp(0, (int)b, 0xb1, 0xf, 0xf, true);
    const unsigned sel = odd ? 0x03020706u : 0x05040100u;
    unsigned short* o = T + (row + 4 * kq + odd) * kTrRow + 16 * wave + (col & ~1);
    if (ROWS == 16 || kq == 0) {
        *reinterpret_cast<unsigned*>(o) = __builtin_amdgcn_perm(oa, a, sel);
        if (ROWS == 16 || !odd)
            *reinterpret_cast<unsigned*>(o + 2 * kTrRow) = __builtin_amdgcn_perm(ob, b, sel);
    }
}

__global__ void __launch_bounds__(64 * kTrWaves) __attribute__((amdgpu_waves_per_eu(4))) k_rs_train(
    int N, int chunks, const float* __restrict__ feat, const float4* __restrict__ basis,
    const float4* __restrict__ target, const float* __restrict__ norm,
    const unsigned short* __restrict__ w1, const unsigned short* __restrict__ w2,
    const unsigned short* __restrict__ w2t, const unsigned short* __restrict__ w3,
    const unsigned short* __restrict__ w3t, const float* __restrict__ params,
    float* __restrict__ part, double* __restrict__ lpart) {
    __shared__ __align__(16) unsigned short T[kTrRows * kTrRow];
    const int wave = threadIdx.x >> 6;
    const float scale = 2.0f / (3.0f * (float)N);
    // tiles of this wavefront: row block `wave` of dW2, or row block wave - 4
    // of dW1 and column block wave - 4 of dW3
    f32x4 g[4];
    // bias sums over the 16 atoms of a row of lanes: lane col holds hidden unit
    // 16 (col / 4) + 4 kq + col % 4
    float gb1 = 0.f, gb2 = 0.f, gb3[kOut];
#pragma unroll
    for (int t = 0; t < 4; ++t) g[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < kOut; ++m) gb3[m] = 0.f;
    float lsum = 0.f;
    for (int chunk = blockIdx.x; chunk < chunks; chunk += gridDim.x) {
        // (opaque: the weights and their addresses, 120 registers if kept over
        // the loop, are formed where they are used)
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        const int col = lane & 15, kq = lane >> 4;
        const int p0 = chunk * kTrAtoms + 16 * wave;
        const int a = p0 + col;
        const bool own = kq == 0 && a < N;  // lanes kq == 0 own the atom's c
        float4 u0 = make_float4(0.f, 0.f, 0.f, 0.f), u1 = u0, u2 = u0, tg = u0;
        if (own) {
            u0 = basis[3 * (size_t)a];
            u1 = basis[3 * (size_t)a + 1];
            u2 = basis[3 * (size_t)a + 2];
            tg = target[a];
        }
        Fwd f;
        mlp_forward<true>(p0, N, lane, feat, norm, w1, w2, w3, params, f);
#pragma unroll
        for (int kc = 0; kc < 3; ++kc) tr_store<16>(T, kTrX + 16 * kc, wave, lane, f.x[kc]);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            tr_store<16>(T, kTrH1 + 16 * t, wave, lane, f.h1[t]);
            tr_store<16>(T, kTrH2 + 16 * t, wave, lane, f.h2[t]);
        }
        __builtin_amdgcn_sched_barrier(0);
        // loss and dL/dc
        float dc0 = 0.f, dc1 = 0.f, dc2 = 0.f;
        if (own) {
            const float q = tg.w;
            const float rx = q * (f.c[0] * u0.x + f.c[1] * u1.x + f.c[2] * u2.x) - tg.x;
            const float ry = q * (f.c[0] * u0.y + f.c[1] * u1.y + f.c[2] * u2.y) - tg.y;
            const float rz = q * (f.c[0] * u0.z + f.c[1] * u1.z + f.c[2] * u2.z) - tg.z;
            lsum += rx * rx + ry * ry + rz * rz;
            dc0 = scale * q * (rx * u0.x + ry * u0.y + rz * u0.z);
            dc1 = scale * q * (rx * u1.x + ry * u1.y + rz * u1.z);
            dc2 = scale * q * (rx * u2.x + ry * u2.y + rz * u2.z);
        }
        gb3[0] += dc0;
        gb3[1] += dc1;
        gb3[2] += dc2;
        // dC as a B operand (k = output 4 kq + j, column = atom): lanes kq == 0
        const bf16x4 dcb = pack4(dc0, dc1, dc2, 0.f);
        tr_store<kOut>(T, kTrC, wave, lane, dcb);
        __builtin_amdgcn_sched_barrier(0);
        // dH2 = W3^T dC, dZ2 = dH2 * silu'(Z2)
        bf16x4 dz2b[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            acc = mfma16(load4(w3t + (size_t)(t * 16 + col) * 16 + kq * 4), dcb, acc);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[j] *= f.d2[t][j];
                const float s = row_total(acc[j]);
                gb2 += col == 4 * t + j ? s : 0.f;
            }
            dz2b[t] = pack4(acc[0], acc[1], acc[2], acc[3]);
            tr_store<16>(T, kTrZ2 + 16 * t, wave, lane, dz2b[t]);
        }
        __builtin_amdgcn_sched_barrier(0);
        // dH1 = W2^T dZ2, dZ1 = dH1 * silu'(Z1)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kc = 0; kc < 4; ++kc)
                acc = mfma16(load4(w2t + (size_t)(t * 16 + col) * kHidden + kc * 16 + kq * 4), dz2b[kc], acc);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[j] *= f.d1[t][j];
                const float s = row_total(acc[j]);
                gb1 += col == 4 * t + j ? s : 0.f;
            }
            tr_store<16>(T, kTrZ1 + 16 * t, wave, lane, pack4(acc[0], acc[1], acc[2], acc[3]));
        }
        __syncthreads();
        // weight gradients over the chunk's atoms (k = atom): A = dZ, B = h or x
        const unsigned short* at = T + col * kTrRow + 4 * kq;
#pragma unroll 2
        for (int ks = 0; ks < kTrWaves; ++ks) {
            if (wave < 4) {
                const bf16x4 A = load4(at + (kTrZ2 + 16 * wave) * kTrRow + 16 * ks);
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    g[t] = mfma16(A, load4(at + (kTrH1 + 16 * t) * kTrRow + 16 * ks), g[t]);
            } else {
                const bf16x4 A = load4(at + (kTrZ1 + 16 * (wave - 4)) * kTrRow + 16 * ks);
#pragma unroll
                for (int t = 0; t < 3; ++t)
                    g[t] = mfma16(A, load4(at + (kTrX + 16 * t) * kTrRow + 16 * ks), g[t]);
                bf16x4 C = {0, 0, 0, 0};  // output rows beyond kOut are zero
                if (col < kOut) C = load4(at + kTrC * kTrRow + 16 * ks);
                g[3] = mfma16(C, load4(at + (kTrH2 + 16 * (wave - 4)) * kTrRow + 16 * ks), g[3]);
            }
        }
        __syncthreads();
    }
    const int lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4;
    // C-layout element j of lane l is (row 4 kq + j, column col) of its tile
    float* o = part + (size_t)blockIdx.x * kTrPart;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = 16 * (wave & 3) + kq * 4 + j;
        if (wave < 4) {
#pragma unroll
            for (int t = 0; t < 4; ++t) o[oW2 + r * kHidden + t * 16 + col] = g[t][j];
        } else {
#pragma unroll
            for (int t = 0; t < 3; ++t) o[oW1 + r * kFeat + t * 16 + col] = g[t][j];
            if (kq * 4 + j < kOut) o[oW3 + (kq * 4 + j) * kHidden + (wave - 4) * 16 + col] = g[3][j];
        }
    }
    // biases and loss over the wavefronts (the loop ended with a barrier: T is
    // free)
    constexpr int kBias = 2 * kHidden + kOut + 1;
    float* red = reinterpret_cast<float*>(T);
    float* rw = red + kBias * wave;
    const int unit = 16 * (col >> 2) + 4 * kq + (col & 3);
    rw[unit] = gb1;
    rw[kHidden + unit] = gb2;
#pragma unroll
    for (int m = 0; m < kOut; ++m) {
        const float s3 = row_total(gb3[m]);
        if (lane == 0) rw[2 * kHidden + m] = s3;
    }
    lsum = row_total(lsum);
    if (lane == 0) rw[2 * kHidden + kOut] = lsum;
    __syncthreads();
    for (int k = threadIdx.x; k < kBias; k += blockDim.x) {
        if (k < kBias - 1) {
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < kTrWaves; ++w) s += red[kBias * w + k];
            o[k < kHidden ? oB1 + k : k < 2 * kHidden ? oB2 + k - kHidden : oB3 + k - 2 * kHidden] = s;
        } else {
            double s = 0.0;
            for (int w = 0; w < kTrWaves; ++w) s += (double)red[kBias * w + k];
            lpart[blockIdx.x] = s;
        }
    }
}

// BF16 copies of the weights in the kernels' operand order
__device__ __forceinline__ void cast_param(int i, float w, unsigned short* w1, unsigned short* w2,
                                           unsigned short* w2t, unsigned short* w3,
                                           unsigned short* w3t) {
    const unsigned short b = f2bf(w);
    if (i < oB1) {
        w1[i] = b;
    } else if (i >= oW2 && i < oB2) {
        const int k = i - oW2, o = k / kHidden, in = k % kHidden;
        w2[k] = b;
        w2t[in * kHidden + o] = b;
    } else if (i >= oW3 && i < oB3) {
        const int k = i - oW3, o = k / kHidden, in = k % kHidden;
        w3[o * kHidden + in] = b;
        w3t[in * 16 + o] = b;
    }
}

__global__ void k_rs_cast(const float* __restrict__ params, unsigned short* w1, unsigned short* w2,
                          unsigned short* w2t, unsigned short* w3, unsigned short* w3t) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kParams) cast_param(i, params[i], w1, w2, w2t, w3, w3t);
}

// Gradient = sum of the n partials, 64 parameters to a workgroup of 16
// wavefronts with every 16th partial each, and the loss (workgroup 0); then the
// Adam step, or the sums to out (which may be host memory) with the loss after.
template <bool ADAM>
__global__ void __launch_bounds__(1024) k_rs_reduce(
    int N, int n, const float* __restrict__ part, const double* __restrict__ lpart,
    float* __restrict__ out, double* __restrict__ loss, float* __restrict__ params,
    float* __restrict__ m, float* __restrict__ v, float lr, float c1, float c2, unsigned short* w1,
    unsigned short* w2, unsigned short* w2t, unsigned short* w3, unsigned short* w3t) {
    __shared__ float red[16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;  // < kTrPart
    float s = 0.f;
    if (i < kParams) {
#pragma unroll 8
        for (int w = wave; w < n; w += 16) s += part[(size_t)w * kTrPart + i];
    }
    red[wave][lane] = s;
    __syncthreads();
    if (wave == 1 && blockIdx.x == 0) {
        double l = 0.0;
        for (int w = lane; w < n; w += 64) l += lpart[w];
        l = wave_sum(l) / (3.0 * (double)N);
        if (lane == 0) *loss = ADAM ? *loss + l : l;
    }
    if (wave || i >= kParams) return;
    float g = 0.f;
#pragma unroll
    for (int w = 0; w < 16; ++w) g += red[w][lane];
    if (!ADAM) {
        out[i] = g;
        return;
    }
    const float mi = 0.9f * m[i] + 0.1f * g;
    const float vi = 0.999f * v[i] + 0.001f * g * g;
    m[i] = mi;
    v[i] = vi;
    const float w = params[i] - lr * (mi * c1) / (sqrtf(vi * c2) + 1e-8f);
    params[i] = w;
    cast_param(i, w, w1, w2, w2t, w3, w3t);
}

// feature sums over stored frames (FP64): acc[0..47] sum, acc[48..95] sum of squares
__global__ void __launch_bounds__(256) k_rs_stats(long long rows, const float* __restrict__ feat,
                                                  double* __restrict__ acc) {
    __shared__ double s1[256], s2[256];
    const int k = threadIdx.x % kFeat;
    const int lanes = (256 / kFeat) * kFeat;  // 240 threads, 5 rows per pass
    double a = 0, b = 0;
    if (threadIdx.x < lanes) {
        for (long long rr = (long long)blockIdx.x * 5 + threadIdx.x / kFeat; rr < rows;
             rr += (long long)gridDim.x * 5) {
            const double x = feat[rr * kFeat + k];
            a += x;
            b += x * x;
        }
    }
    s1[threadIdx.x] = a;
    s2[threadIdx.x] = b;
    __syncthreads();
    if (threadIdx.x < kFeat) {
        for (int t = threadIdx.x + kFeat; t < lanes; t += kFeat) {
            a += s1[t];
            b += s2[t];
        }
        atomicAdd(&acc[threadIdx.x], a);
        atomicAdd(&acc[kFeat + threadIdx.x], b);
    }
}

__global__ void k_rs_norm(long long rows, const double* __restrict__ acc, float* __restrict__ norm) {
    const int k = threadIdx.x;
    if (k >= kFeat) return;
    const double mu = acc[k] / (double)rows;
    const double var = std::max(acc[kFeat + k] / (double)rows - mu * mu, 0.0);
    const double sd = std::sqrt(var);
    norm[k] = (float)mu;
    norm[kFeat + k] = sd > 1e-12 * (1.0 + std::fabs(mu)) ? (float)(1.0 / sd) : 1.0f;
}

// FP64 sums of a force array: [0..2] components (for the mean)
__global__ void __launch_bounds__(256) k_rs_sum3(int N, const float* __restrict__ f,
                                                 double* __restrict__ out) {
    __shared__ double s[3][256];
    double a = 0, b = 0, c = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        a += f[3 * i];
        b += f[3 * i + 1];
        c += f[3 * i + 2];
    }
    s[0][threadIdx.x] = a;
    s[1][threadIdx.x] = b;
    s[2][threadIdx.x] = c;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w)
            for (int m = 0; m < 3; ++m) s[m][threadIdx.x] += s[m][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int m = 0; m < 3; ++m) atomicAdd(&out[m], s[m][0]);
}

// store the current features / basis and the target (rec - mean) with the
// charge, in atom order (frames of different list builds line up)
__global__ void k_rs_store(int N, const int* __restrict__ sidx, const float* __restrict__ feat,
                           const float4* __restrict__ basis, const float4* __restrict__ pos,
                           const float* __restrict__ rec, const double* __restrict__ sums,
                           float* __restrict__ ffeat, float4* __restrict__ fbasis,
                           float4* __restrict__ ftarget) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const int i = sidx[p];
    for (int k = 0; k < kFeat; ++k) ffeat[(size_t)kFeat * i + k] = feat[(size_t)kFeat * p + k];
    for (int m = 0; m < 3; ++m) fbasis[3 * (size_t)i + m] = basis[3 * (size_t)p + m];
    const float mx = (float)(sums[0] / N), my = (float)(sums[1] / N), mz = (float)(sums[2] / N);
    ftarget[i] = make_float4(rec[3 * i] - mx, rec[3 * i + 1] - my, rec[3 * i + 2] - mz, pos[p].w);
}

// model prediction q (c . U) of one atom of a stored frame (lanes kq == 0)
__device__ __forceinline__ float3 frame_pred(const Fwd& f, const float4* basis, const float4* target,
                                             int a) {
    const float4 u0 = basis[3 * (size_t)a], u1 = basis[3 * (size_t)a + 1], u2 = basis[3 * (size_t)a + 2];
    const float q = target[a].w;
    return make_float3(q * (f.c[0] * u0.x + f.c[1] * u1.x + f.c[2] * u2.x),
                       q * (f.c[0] * u0.y + f.c[1] * u1.y + f.c[2] * u2.y),
                       q * (f.c[0] * u0.z + f.c[1] * u1.z + f.c[2] * u2.z));
}

__device__ __forceinline__ float3 frame_base(const float4* basis, const float4* target, int a) {
    const float4 u0 = basis[3 * (size_t)a], u1 = basis[3 * (size_t)a + 1];
    const float q = target[a].w;
    return make_float3(q * (u0.x + u1.x), q * (u0.y + u1.y), q * (u0.z + u1.z));
}

__device__ __forceinline__ float sq3(float3 a, float4 t) {
    const float x = a.x - t.x, y = a.y - t.y, z = a.z - t.z;
    return x * x + y * y + z * z;
}

// evaluation sums over a stored frame f (and, with lag > 0, the frame
// f - lag it is anchored on): [0] |model - T|^2, [1] |T|^2, [2] |baseline -
// T|^2 (c = 1, 1, 0); anchored on the earlier frame's exact target:
// [3] |model + (T' - model') - T|^2, [4] the same for the baseline,
// [5] |T' - T|^2 (the stale force)
__global__ void __launch_bounds__(256) k_rs_eval(
    int N, int ntiles, const float* __restrict__ feat, const float4* __restrict__ basis,
    const float4* __restrict__ target, const float* __restrict__ feat0,
    const float4* __restrict__ basis0, const float4* __restrict__ target0,
    const float* __restrict__ norm, const unsigned short* __restrict__ w1,
    const unsigned short* __restrict__ w2, const unsigned short* __restrict__ w3,
    const float* __restrict__ params, double* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int nw = (gridDim.x * blockDim.x) >> 6;
    float e[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int tile = wave; tile < ntiles; tile += nw) {
        Fwd f;
        mlp_forward(tile * 16, N, lane, feat, norm, w1, w2, w3, params, f);
        Fwd f0;
        if (feat0) mlp_forward(tile * 16, N, lane, feat0, norm, w1, w2, w3, params, f0);
        const int a = tile * 16 + (lane & 15);
        if ((lane >> 4) == 0 && a < N) {
            const float4 tg = target[a];
            const float3 pm = frame_pred(f, basis, target, a), pb = frame_base(basis, target, a);
            e[0] += sq3(pm, tg);
            e[1] += tg.x * tg.x + tg.y * tg.y + tg.z * tg.z;
            e[2] += sq3(pb, tg);
            if (feat0) {
                const float4 t0 = target0[a];
                const float3 pm0 = frame_pred(f0, basis0, target0, a);
                const float3 pb0 = frame_base(basis0, target0, a);
                e[3] += sq3(make_float3(pm.x + t0.x - pm0.x, pm.y + t0.y - pm0.y, pm.z + t0.z - pm0.z), tg);
                e[4] += sq3(make_float3(pb.x + t0.x - pb0.x, pb.y + t0.y - pb0.y, pb.z + t0.z - pb0.z), tg);
                e[5] += sq3(make_float3(t0.x, t0.y, t0.z), tg);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const float v = wave_sum(e[k]);
        if (lane == 0) atomicAdd(&out[k], (double)v);
    }
}

__global__ void k_rs_permute_out(int N, const int* __restrict__ sidx, const float* __restrict__ feat,
                                 const float4* __restrict__ basis, float* __restrict__ feat_out,
                                 float* __restrict__ basis_out) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const int i = sidx[p];
    if (feat_out)
        for (int k = 0; k < kFeat; ++k) feat_out[(size_t)kFeat * i + k] = feat[(size_t)kFeat * p + k];
    if (basis_out)
        for (int m = 0; m < 3; ++m) {
            const float4 b = basis[3 * (size_t)p + m];
            basis_out[9 * (size_t)i + 3 * m] = b.x;
            basis_out[9 * (size_t)i + 3 * m + 1] = b.y;
            basis_out[9 * (size_t)i + 3 * m + 2] = b.z;
        }
}

int tiles_of(int N) { return (N + 15) / 16; }

// workgroups of a training pass: two fit on a CU
int train_groups(int N) { return std::min((N + kTrAtoms - 1) / kTrAtoms, kTrGroups); }

// forward, loss and backward over one stored frame: partial gradients
int train_pass(sponge_rsur* h, int frame) {
    const size_t f = (size_t)frame, N = (size_t)h->N;
    hipLaunchKernelGGL(k_rs_train, dim3(train_groups(h->N)), dim3(64 * kTrWaves), 0, h->stream, h->N,
                       (h->N + kTrAtoms - 1) / kTrAtoms, h->d_ffeat + f * N * kFeat,
                       h->d_fbasis + f * N * 3, h->d_ftarget + f * N, h->d_norm, h->d_w1, h->d_w2,
                       h->d_w2t, h->d_w3, h->d_w3t, h->d_params, h->d_part, h->d_lpart);
    SA_LAUNCH_CHECK();
    return 0;
}

int cast_weights(sponge_rsur* h) {
    hipLaunchKernelGGL(k_rs_cast, dim3(grid_for(kParams, 256)), dim3(256), 0, h->stream, h->d_params,
                       h->d_w1, h->d_w2, h->d_w2t, h->d_w3, h->d_w3t);
    SA_LAUNCH_CHECK();
    return 0;
}

void rsur_free(sponge_rsur* h) {
    dfree(h->d_pos);
    dfree(h->d_feat);
    dfree(h->d_basis);
    dfree(h->d_uex);
    dfree(h->d_moved);
    dfree(h->d_params);
    dfree(h->d_norm);
    dfree(h->d_w1);
    dfree(h->d_w2);
    dfree(h->d_w2t);
    dfree(h->d_w3);
    dfree(h->d_w3t);
    dfree(h->d_part);
    dfree(h->d_lpart);
    if (h->h_grad) (void)hipHostFree(h->h_grad);
    h->h_grad = nullptr;
    dfree(h->d_m);
    dfree(h->d_v);
    dfree(h->d_acc);
    dfree(h->d_ffeat);
    dfree(h->d_fbasis);
    dfree(h->d_ftarget);
}

// initial parameters: normal weights scaled by 1/sqrt(fan-in), zero biases,
// output layer zero with biases (1, 1, 0): the physics baseline
std::vector<float> initial_params(unsigned seed) {
    std::vector<float> p(kParams, 0.f);
    std::mt19937 gen(seed);
    std::normal_distribution<float> nd(0.f, 1.f);
    for (int i = 0; i < kHidden * kFeat; ++i) p[oW1 + i] = nd(gen) / std::sqrt((float)kFeat);
    for (int i = 0; i < kHidden * kHidden; ++i) p[oW2 + i] = nd(gen) / std::sqrt((float)kHidden);
    p[oB3] = 1.f;
    p[oB3 + 1] = 1.f;
    return p;
}

}  // namespace

namespace sa {

// Features of the current coordinates over the list (sorted positions given).
// own_pack: the module's own pack wrote them (and cleared the excluded
// partners' field); otherwise the step driver's list update did, whose
// automatic refresh bounds how far an atom is from its build position.
static int features(sponge_rsur* h, sponge_nl* nl, const float4* pos, const float* crd,
                    const float* charge, const float* cell, const float* rcell, const int* ex_start,
                    const int* ex_list, const int* ex_num, bool own_pack) {
    hipStream_t s = h->stream;
    const LT6 c = lt_from(cell), r = lt_from(rcell);
    const bool ortho = lt_is_orthorhombic(c);
    if (!own_pack) {
        const int rc = fill_async(reinterpret_cast<float*>(h->d_uex), 0.f, 4LL * h->N, s);
        if (rc) return rc;
    }
    if (ex_start && ex_num && ex_list) {
        if (ortho)
            hipLaunchKernelGGL(k_rs_exfield<true>, dim3(grid_for(h->N, 256)), dim3(256), 0, s, h->N,
                               crd, charge, ex_start, ex_num, ex_list, c, r, h->beta, h->d_uex);
        else
            hipLaunchKernelGGL(k_rs_exfield<false>, dim3(grid_for(h->N, 256)), dim3(256), 0, s, h->N,
                               crd, charge, ex_start, ex_num, ex_list, c, r, h->beta, h->d_uex);
        SA_LAUNCH_CHECK();
    }
    // two workgroups per CU fit by registers and LDS; two or three per cell
    // where that fills the last round of the chip better (a row costs about
    // three times its share of the staging)
    const int stage = h->stage;
    const size_t sh = sizeof(float4) * stage + kRsWaves * (kRsRing * sizeof(float4) + kWave * sizeof(float));
    int split = 1;
    double best = 0.0;
    for (int k = 1; k <= 3; ++k) {
        const double rounds = std::ceil((double)nl->G * k / (2 * 256));
        const double cost = rounds * (1.0 + 3.0 * std::ceil((double)nl->N / nl->G / (kRsWaves * k)));
        if (k == 1 || cost < 0.95 * best) {
            best = cost;
            split = k;
        }
    }
    const bool same_cell = memcmp(&c, &nl->cell0, sizeof(LT6)) == 0;
    const bool bounded = own_pack ? same_cell : nl->opt.refresh_interval <= 0;
    const float reach = bounded ? h->rf + nl->skin * nl->opt.skin_permit : -1.f;
    const float rf2 = h->rf * h->rf;
    const EwaldPoly ew = ewald_poly(h->beta, h->rf);
    timer_begin("rsur_features", s);
#define SA_RS_FEAT(O)                                                                               \
    hipLaunchKernelGGL(k_rs_features<O>, dim3(nl->G * split), dim3(64 * kRsWaves), sh, s,             \
                       nl->d_cell_start, nl->d_stream, nl->d_soff, nl->d_slen, nl->d_list_count,      \
                       nl->d_list, nl->cap, pos, nl->d_sidx, c, r, rf2, 1.0f / h->rf, h->beta, ew,    \
                       stage, split, nl->width, nl->Nx, nl->Ny, nl->Nz, reach,                        \
                       own_pack ? h->d_moved : nullptr, h->epoch, h->d_uex, h->d_feat, h->d_basis)
    if (ortho) SA_RS_FEAT(true);
    else SA_RS_FEAT(false);
#undef SA_RS_FEAT
    SA_LAUNCH_CHECK();
    timer_end("rsur_features", s);
    h->sidx = nl->d_sidx;
    h->pos_last = pos;
    return 0;
}

int rsur_features_sorted(sponge_rsur* h, sponge_nl* nl, const float4* pos, const float* crd,
                         const float* charge, const float* cell, const float* rcell,
                         const int* ex_start, const int* ex_list, const int* ex_num) {
    return features(h, nl, pos, crd, charge, cell, rcell, ex_start, ex_list, ex_num, false);
}

int rsur_predict_sorted(sponge_rsur* h, float* frc, int assign, const float* anchor) {
    if (!h->sidx) return SPONGE_AMD_ERROR_MISSING_COMMAND;
    const float4* pos = h->pos_last;
    const int nt = tiles_of(h->N);
    const int blocks = std::min(grid_for(nt, 4), 2048);
    timer_begin("rsur_mlp", h->stream);
    hipLaunchKernelGGL(k_rs_predict, dim3(blocks), dim3(256), 0, h->stream, h->N, nt, h->d_feat,
                       h->d_basis, pos, h->sidx, h->d_norm, h->d_w1, h->d_w2, h->d_w3, h->d_params,
                       frc, assign, anchor);
    SA_LAUNCH_CHECK();
    timer_end("rsur_mlp", h->stream);
    return 0;
}

void rsur_set_stream(sponge_rsur* h, hipStream_t s, const StreamOwner& owner) {
    h->stream = s;
    h->owner = owner;
}
int rsur_atoms(const sponge_rsur* h) { return h->N; }
float rsur_cutoff(const sponge_rsur* h) { return h->rf; }

}  // namespace sa

extern "C" {

void sponge_rsur_default_options(sponge_rsur_options* opt) {
    if (!opt) return;
    opt->feature_cutoff = 10.0f;
    opt->max_frames = 0;
    opt->seed = 1;
}

int sponge_rsur_model_size(void) { return kModel; }

int sponge_rsur_initial(sponge_rsur** out, int atom_numbers, float beta,
                        const sponge_rsur_options* opt, void* stream) {
    if (!out || atom_numbers <= 0 || beta <= 0.f) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    *out = nullptr;
    sponge_rsur* h = new sponge_rsur();
    h->N = atom_numbers;
    h->beta = beta;
    if (opt) h->opt = *opt;
    else sponge_rsur_default_options(&h->opt);
    if (!(h->opt.feature_cutoff > 0.f) || h->opt.max_frames < 0) {
        delete h;
        return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    }
    h->rf = h->opt.feature_cutoff;
    h->stream = (hipStream_t)stream;
    h->stage = stage_entries(sizeof(float4), kFeatStage,
                             kRsWaves * (kRsRing * sizeof(float4) + kWave * sizeof(float)));
    const size_t N = (size_t)atom_numbers, F = (size_t)h->opt.max_frames;
    int e = 0;
    e |= dmalloc(&h->d_pos, N);
    e |= dmalloc(&h->d_feat, N * kFeat);
    e |= dmalloc(&h->d_basis, N * 3);
    e |= dmalloc(&h->d_uex, N);
    e |= dmalloc(&h->d_moved, 1);
    e |= dmalloc(&h->d_params, kParams);
    e |= dmalloc(&h->d_norm, 2 * kFeat);
    e |= dmalloc(&h->d_w1, kHidden * kFeat);
    e |= dmalloc(&h->d_w2, kHidden * kHidden);
    e |= dmalloc(&h->d_w2t, kHidden * kHidden);
    e |= dmalloc(&h->d_w3, 16 * kHidden);
    e |= dmalloc(&h->d_w3t, kHidden * 16);
    e |= dmalloc(&h->d_m, kParams);
    e |= dmalloc(&h->d_v, kParams);
    e |= dmalloc(&h->d_acc, 16 + 2 * kFeat);
    if (F) {
        e |= dmalloc(&h->d_ffeat, F * N * kFeat);
        e |= dmalloc(&h->d_fbasis, F * N * 3);
        e |= dmalloc(&h->d_ftarget, F * N);
        e |= dmalloc(&h->d_part, (size_t)train_groups(atom_numbers) * kTrPart);
        e |= dmalloc(&h->d_lpart, train_groups(atom_numbers));
        if (hipHostMalloc(reinterpret_cast<void**>(&h->h_grad), sizeof(float) * kTrPart + sizeof(double)) !=
            hipSuccess)
            e = 1;
    }
    if (e) {
        rsur_free(h);
        delete h;
        return SPONGE_AMD_ERROR_MALLOC_FAILED;
    }
    hipStream_t s = h->stream;
    std::vector<float> p = initial_params((unsigned)h->opt.seed);
    std::vector<float> norm(2 * kFeat, 0.f);
    for (int k = 0; k < kFeat; ++k) norm[kFeat + k] = 1.f;
    int rc = 0;
    if (hipMemcpyAsync(h->d_params, p.data(), sizeof(float) * kParams, hipMemcpyHostToDevice, s) !=
            hipSuccess ||
        hipMemcpyAsync(h->d_norm, norm.data(), sizeof(float) * 2 * kFeat, hipMemcpyHostToDevice, s) !=
            hipSuccess)
        rc = SPONGE_AMD_ERROR_MALLOC_FAILED;
    // the bf16 copies carry zeros where no parameter maps (padding rows)
    rc |= fill_async(h->d_w3, (unsigned short)0, 16 * kHidden, s);
    rc |= fill_async(h->d_w3t, (unsigned short)0, kHidden * 16, s);
    rc |= fill_async(h->d_m, 0.f, kParams, s);
    rc |= fill_async(h->d_v, 0.f, kParams, s);
    rc |= fill_async(h->d_moved, 0, 1, s);
    rc |= fill_async(h->d_uex, make_float4(0.f, 0.f, 0.f, 0.f), (long long)N, s);
    if (!rc) rc = cast_weights(h);
    if (!rc && hipStreamSynchronize(s) != hipSuccess) rc = SPONGE_AMD_ERROR_MALLOC_FAILED;
    if (rc) {
        rsur_free(h);
        delete h;
        return rc;
    }
    *out = h;
    return 0;
}

int sponge_rsur_features(sponge_rsur* h, sponge_nl* nl, const float* crd, const float* cell,
                         const float* rcell, const float* charge, const int* excluded_list_start,
                         const int* excluded_list, const int* excluded_numbers) {
    if (!h || !nl || !crd || !cell || !rcell || !charge) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    if (nl->N != h->N || !nl->built) return SPONGE_AMD_ERROR_MISSING_COMMAND;
    // every partner within the feature cutoff is on the list between rebuilds
    if (h->rf > nl->cutoff) return SPONGE_AMD_ERROR_CONFLICTING_COMMAND;
    const float permit = nl->skin * nl->opt.skin_permit;
    h->epoch = h->epoch == 0x7fffffff ? 1 : h->epoch + 1;
    hipLaunchKernelGGL(k_rs_pack, dim3(grid_for(h->N, 256)), dim3(256), 0, h->stream, h->N,
                       nl->d_sidx, nl->d_spos, crd, charge, nl->cell0, nl->rcell0, permit * permit,
                       h->epoch, h->d_pos, h->d_uex, h->d_moved);
    SA_LAUNCH_CHECK();
    return sa::features(h, nl, h->d_pos, crd, charge, cell, rcell, excluded_list_start,
                        excluded_list, excluded_numbers, true);
}

int sponge_rsur_export_features(sponge_rsur* h, float* feat, float* basis) {
    if (!h) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    if (!h->sidx) return SPONGE_AMD_ERROR_MISSING_COMMAND;
    hipLaunchKernelGGL(k_rs_permute_out, dim3(grid_for(h->N, 256)), dim3(256), 0, h->stream, h->N,
                       h->sidx, h->d_feat, h->d_basis, feat, basis);
    SA_LAUNCH_CHECK();
    return 0;
}

int sponge_rsur_predict(sponge_rsur* h, float* frc) {
    if (!h || !frc) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    return rsur_predict_sorted(h, frc, 0, nullptr);
}

int sponge_rsur_get_model(sponge_rsur* h, float* model) {
    if (!h || !model) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    SA_CHECK(hipMemcpyAsync(model, h->d_params, sizeof(float) * kParams, hipMemcpyDeviceToHost,
                            h->stream));
    SA_CHECK(hipMemcpyAsync(model + kParams, h->d_norm, sizeof(float) * 2 * kFeat,
                            hipMemcpyDeviceToHost, h->stream));
    SA_CHECK(hipStreamSynchronize(h->stream));
    return 0;
}

int sponge_rsur_set_model(sponge_rsur* h, const float* model) {
    if (!h || !model) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    SA_CHECK(hipMemcpyAsync(h->d_params, model, sizeof(float) * kParams, hipMemcpyHostToDevice,
                            h->stream));
    SA_CHECK(hipMemcpyAsync(h->d_norm, model + kParams, sizeof(float) * 2 * kFeat,
                            hipMemcpyHostToDevice, h->stream));
    int rc = cast_weights(h);
    if (rc) return rc;
    SA_CHECK(hipStreamSynchronize(h->stream));
    return 0;
}

int sponge_rsur_add_frame(sponge_rsur* h, const float* rec_frc) {
    if (!h || !rec_frc) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    if (!h->sidx) return SPONGE_AMD_ERROR_MISSING_COMMAND;
    if (h->n_frames >= h->opt.max_frames) return SPONGE_AMD_ERROR_OVERFLOW;
    hipStream_t s = h->stream;
    int rc = fill_async(h->d_acc + 1, 0.0, 3, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_rs_sum3, dim3(std::min(grid_for(h->N, 256), 256)), dim3(256), 0, s, h->N,
                       rec_frc, h->d_acc + 1);
    SA_LAUNCH_CHECK();
    const size_t f = (size_t)h->n_frames, N = (size_t)h->N;
    hipLaunchKernelGGL(k_rs_store, dim3(grid_for(h->N, 256)), dim3(256), 0, s, h->N, h->sidx,
                       h->d_feat, h->d_basis, h->pos_last, rec_frc, h->d_acc + 1,
                       h->d_ffeat + f * N * kFeat, h->d_fbasis + f * N * 3, h->d_ftarget + f * N);
    SA_LAUNCH_CHECK();
    h->n_frames++;
    return 0;
}

int sponge_rsur_frame_count(sponge_rsur* h, int* n) {
    if (!h || !n) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    *n = h->n_frames;
    return 0;
}

int sponge_rsur_fit_normalization(sponge_rsur* h, int n_frames) {
    if (!h || n_frames <= 0 || n_frames > h->n_frames) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    hipStream_t s = h->stream;
    double* acc = h->d_acc + 8;
    int rc = fill_async(acc, 0.0, 2 * kFeat, s);
    if (rc) return rc;
    const long long rows = (long long)n_frames * h->N;
    hipLaunchKernelGGL(k_rs_stats, dim3(1024), dim3(256), 0, s, rows, h->d_ffeat, acc);
    SA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_rs_norm, dim3(1), dim3(64), 0, s, rows, acc, h->d_norm);
    SA_LAUNCH_CHECK();
    return 0;
}

int sponge_rsur_gradient(sponge_rsur* h, int frame, float* grad, double* loss) {
    if (!h || frame < 0 || frame >= h->n_frames) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    const int rc = train_pass(h, frame);
    if (rc) return rc;
    // the sums go to pinned host memory: no copies to queue behind the kernel
    double* l = reinterpret_cast<double*>(h->h_grad + kTrPart);
    hipLaunchKernelGGL(k_rs_reduce<false>, dim3(kTrPart / 64), dim3(1024), 0, h->stream, h->N,
                       train_groups(h->N), h->d_part, h->d_lpart, h->h_grad, l, nullptr, nullptr,
                       nullptr, 0.f, 0.f, 0.f, nullptr, nullptr, nullptr, nullptr, nullptr);
    SA_LAUNCH_CHECK();
    SA_CHECK(hipStreamSynchronize(h->stream));
    if (grad) memcpy(grad, h->h_grad, sizeof(float) * kParams);
    if (loss) *loss = *l;
    return 0;
}

int sponge_rsur_train(sponge_rsur* h, int n_train_frames, int epochs, float lr, double* epoch_loss) {
    if (!h || n_train_frames <= 0 || n_train_frames > h->n_frames || epochs < 0 || !(lr > 0.f))
        return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    hipStream_t s = h->stream;
    std::mt19937 gen((unsigned)h->opt.seed + 17u);
    std::vector<int> order(n_train_frames);
    for (int i = 0; i < n_train_frames; ++i) order[i] = i;
    int rc = 0;
    for (int ep = 0; ep < epochs; ++ep) {
        std::shuffle(order.begin(), order.end(), gen);
        rc = fill_async(h->d_acc, 0.0, 1, s);
        if (rc) return rc;
        for (int k = 0; k < n_train_frames; ++k) {
            rc = train_pass(h, order[k]);
            if (rc) return rc;
            h->adam_t++;
            const float c1 = (float)(1.0 / (1.0 - std::pow(0.9, (double)h->adam_t)));
            const float c2 = (float)(1.0 / (1.0 - std::pow(0.999, (double)h->adam_t)));
            hipLaunchKernelGGL(k_rs_reduce<true>, dim3(kTrPart / 64), dim3(1024), 0, s, h->N,
                               train_groups(h->N), h->d_part, h->d_lpart, nullptr, h->d_acc,
                               h->d_params, h->d_m, h->d_v, lr, c1, c2, h->d_w1, h->d_w2, h->d_w2t,
                               h->d_w3, h->d_w3t);
            SA_LAUNCH_CHECK();
        }
        if (epoch_loss) {
            double l = 0;
            SA_CHECK(hipMemcpyAsync(&l, h->d_acc, sizeof(double), hipMemcpyDeviceToHost, s));
            SA_CHECK(hipStreamSynchronize(s));
            epoch_loss[ep] = l / n_train_frames;
        }
    }
    SA_CHECK(hipStreamSynchronize(s));
    return 0;
}

int sponge_rsur_evaluate(sponge_rsur* h, int frame_begin, int frame_end, int lag, double* out) {
    if (!h || !out || frame_begin < 0 || frame_end > h->n_frames || frame_begin >= frame_end ||
        lag < 0 || frame_begin - lag < 0)
        return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    hipStream_t s = h->stream;
    double* acc = h->d_acc + 8 + 2 * kFeat;
    int rc = fill_async(acc, 0.0, 6, s);
    if (rc) return rc;
    const size_t N = (size_t)h->N;
    const int nt = tiles_of(h->N);
    for (int f = frame_begin; f < frame_end; ++f) {
        const size_t f0 = (size_t)(f - lag);
        hipLaunchKernelGGL(k_rs_eval, dim3(std::min(grid_for(nt, 4), 2048)), dim3(256), 0, s, h->N, nt,
                           h->d_ffeat + f * N * kFeat, h->d_fbasis + f * N * 3, h->d_ftarget + f * N,
                           lag ? h->d_ffeat + f0 * N * kFeat : nullptr, h->d_fbasis + f0 * N * 3,
                           h->d_ftarget + f0 * N, h->d_norm, h->d_w1, h->d_w2, h->d_w3, h->d_params,
                           acc);
        SA_LAUNCH_CHECK();
    }
    double a[6];
    SA_CHECK(hipMemcpyAsync(a, acc, sizeof(a), hipMemcpyDeviceToHost, s));
    SA_CHECK(hipStreamSynchronize(s));
    const double ref = a[1] > 0 ? a[1] : 1.0;
    out[0] = std::sqrt(a[0] / ref);
    out[1] = std::sqrt(a[2] / ref);
    out[2] = lag ? std::sqrt(a[3] / ref) : 0.0;
    out[3] = lag ? std::sqrt(a[4] / ref) : 0.0;
    out[4] = lag ? std::sqrt(a[5] / ref) : 0.0;
    return 0;
}

int sponge_rsur_clear(sponge_rsur* h) {
    if (!h) return 0;
    (void)hipStreamSynchronize(h->stream);
    rsur_free(h);
    delete h;
    return 0;
}

}  // extern "C"
