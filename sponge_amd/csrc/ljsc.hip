// LJ soft core with PME direct Coulomb for alchemical lambda windows: the
// reference's LJ_SOFT_CORE module (SPONGE/Lennard_Jones_force/
// LJ_soft_core.{h:9-214, cpp:195-440, 463-700, 757-946}).  State A (types and
// tables AA / AB) is weighted 1 - lambda, state B (BA / BB) lambda; a pair
// whose repulsion vanishes in exactly one state uses the soft-core distances
// r_A = (r^6 + alpha lambda^p sigma_A)^(1/6), r_B = (r^6 + alpha (1 -
// lambda)^p sigma_B)^(1/6), sigma = A / (2B) (sigma^6 of the options when A
// or B is zero, at least sigma_min^6).
//
// Same structure as the plain pair kernel: workgroups of a
// neighbor-list cell stage the cell's candidate stream (positions and
// charges, A / B types, charge_BA, global ids) and both square coefficient
// tables in LDS; one wavefront per row over the full 16-bit list.  Forces
// need no atomics (rows hold both directions); energies, virial and
// dU/dlambda are counted in the row of the lower global id.  Force-only
// steps take a lighter form (positions and types staged, two partners per
// lane and pass, the plain kernel's arithmetic for the pairs that are not
// soft-core): 0.88 -> 0.57 ms per step of the 16-window batch.
#include <algorithm>
#include <vector>

#include "internal.h"
#include "batch_launch.h"
#include "pair_term.h"
#include "timing.h"

using namespace sa;

struct sponge_ljsc {
    int N = 0, TA = 0, TB = 0;
    float cutoff = 0, rc2_thr = 0;
    float lambda = 0, alpha = 0.5f, p = 1.0f, sigma6 = 729.0f, sigma6_min = 0.0f;
    float long_range_factor = 0, long_range_factor_TI = 0;
    hipStream_t stream = nullptr;
    StreamOwner owner;             // of the stream, when it is a step driver's
    int stage = 0;                 // most stream entries staged in LDS
    float2* d_ABa = nullptr;       // [TA][TA] (A, B) of state A
    float2* d_ABb = nullptr;       // [TB][TB] of state B
    int* d_typeA = nullptr;        // [N] local order
    int* d_typeB = nullptr;
    int* d_typeAB = nullptr;       // [N] local order, typeA | typeB << 16
    float4* d_pos = nullptr;       // [N] sorted x, y, z, charge
    int* d_tp = nullptr;           // [N] sorted typeA | typeB << 16
    float* d_qba = nullptr;        // [N] sorted charge_BA
    int* d_gid = nullptr;          // [N] sorted global id
    float4* d_facc = nullptr;      // [N] per row
    float2* d_eacc = nullptr;      // [N] (LJ, Coulomb) per row
    float* d_vacc = nullptr;       // [N][6]
    float* d_LJ_energy_atom = nullptr;  // [N] local order
    double* d_du = nullptr;        // [0] LJ, [1] direct
    double* d_sum = nullptr;
};

namespace {

constexpr int kScStage = 3584;
// Rings of stream positions, two per wavefront (plain and soft-core pairs; or
// one of twice the length, the force-only kernel's soft-core pairs): pairs in
// range are appended and evaluated 64 at a time, so that a wavefront runs the
// long pair functions with every lane in use.  One soft-core pair in a pass of
// 64 cost all of them the soft-core function (some 640 instructions, against 45
// of a plain pair), which rows near a solvated 24-atom solute met in most of
// their passes; and 45 % of a row's list lies beyond the cutoff.
// With the powers of lambda from the host (ScParams): force-only, 8 windows of
// 3,600 atoms, 72 -> 54 us (58 with displacements from the cell's centre and the
// squared polynomial); energies and virial at 6,000 atoms 44 -> 36, dU/dlambda
// 40 -> 36.  (The soft-core pairs queued for a whole workgroup, 12 KB of LDS
// more: 83.)  What is left is the solute's own cells: all pairs of a solute row
// are soft-core ones, five batches against one elsewhere.
constexpr int kScRing = 128;
constexpr size_t kScRings = 2 * kScRing * sizeof(unsigned short) * 16;  // of 16 wavefronts
constexpr float kTwoOverSqrtPiF = 1.1283791670955126f;

__device__ __forceinline__ void ljsc_pack_body(int sa_block, int N, const int* __restrict__ sidx,
                            const float4* __restrict__ spos,
                            const float* __restrict__ crd, const float* __restrict__ charge,
                            const float* __restrict__ qba, const int* __restrict__ tA,
                            const int* __restrict__ tB, float4* __restrict__ pos, int* __restrict__ tp,
                            float* __restrict__ pqba, int* __restrict__ gid) {
    const int p = sa_block * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const int i = sidx[p];
    pos[p] = make_float4(crd[3 * i], crd[3 * i + 1], crd[3 * i + 2], charge[i]);
    tp[p] = tA[i] | (tB[i] << 16);
    pqba[p] = qba ? qba[i] : 0.f;
    gid[p] = __float_as_int(spos[p].w);
}

__global__ void k_ljsc_pack(int N, const int* __restrict__ sidx, const float4* __restrict__ spos,
                            const float* __restrict__ crd, const float* __restrict__ charge,
                            const float* __restrict__ qba, const int* __restrict__ tA,
                            const int* __restrict__ tB, float4* __restrict__ pos, int* __restrict__ tp,
                            float* __restrict__ pqba, int* __restrict__ gid) {
    ljsc_pack_body(blockIdx.x, N, sidx, spos, crd, charge, qba, tA, tB, pos, tp, pqba, gid);
}

// The powers of lambda and 1 - lambda come from the host: hoisted out of the
// rows by the compiler, each was 210 instructions of every wavefront, which has
// two or three rows of about 600.
struct ScParams {
    float lambda, alpha, p, sigma6, sigma6_min, beta;
    float pow_l, pow_l_;    // lambda^p, (1 - lambda)^p
    float pow1_l, pow1_l_;  // (lambda + FLT_MIN)^(p - 1) and of 1 - lambda
};

// Pair functions of LJ_soft_core.h: forces are F / r (the vector force is
// F d), energies the pair energies.
__device__ __forceinline__ float lj_f(float r, float A, float B) {
    const float ri2 = 1.0f / (r * r), r6 = ri2 * ri2 * ri2;
    return (B - A * r6) * r6 * ri2;
}
__device__ __forceinline__ float lj_e(float r, float A, float B) {
    const float ri2 = 1.0f / (r * r), r6 = ri2 * ri2 * ri2;
    return (0.083333333f * A * r6 - 0.166666667f * B) * r6;
}
__device__ __forceinline__ float cf_f(float qq, float r, float beta) {
    const float br = beta * r;
    return qq / (r * r * r) * (br * kTwoOverSqrtPiF * expf(-br * br) + erfcf(br));
}
__device__ __forceinline__ float cf_e(float qq, float r, float beta) { return qq * erfcf(beta * r) / r; }
__device__ __forceinline__ float sc_sigma(float A, float B, const ScParams& s) {
    return (A == 0.f || B == 0.f) ? s.sigma6 : fmaxf(0.5f * A / B, s.sigma6_min);
}
__device__ __forceinline__ float sc_dist(float sigma, float r2, float pow_l, const ScParams& s) {
    return powf(r2 * r2 * r2 + s.alpha * pow_l * sigma, 0.16666667f);
}
__device__ __forceinline__ float sc_lj_f(float r2, float rs, float A, float B) {
    const float rsi6 = 1.0f / (rs * rs * rs * rs * rs * rs);
    return r2 * r2 * (B - A * rsi6) * rsi6 * rsi6;
}
__device__ __forceinline__ float sc_cf_f(float qq, float r2, float rs, float beta) {
    const float b = rs * beta;
    const float rsi6 = 1.0f / (rs * rs * rs * rs * rs * rs);
    return qq * r2 * r2 * (expf(-b * b) * kTwoOverSqrtPiF * beta + erfcf(b) / rs) * rsi6;
}
__device__ __forceinline__ float sc_du(float F, float sigma, float rs, float lam, float pow1_l,
                                       const ScParams& s) {
    return 0.16666667f * s.p * s.alpha * (1.0f - lam) * pow1_l * F *
           sigma / (rs * rs * rs * rs);
}

struct ScTerm {
    float f, elj, ecf, dlj, dcf;
};

// whether a pair's LJ is present in both states or in neither (plain mixture)
__device__ __forceinline__ bool sc_plain(float2 a, float2 b) {
    return a.x * b.x != 0.f || a.x + b.x == 0.f;
}

// SOFT: a pair that is not plain
template <bool E, bool DU, bool SOFT>
__device__ __forceinline__ ScTerm sc_pair(float r2, float qi, float qj, float qbai, float qbaj,
                                          float2 a, float2 b, const ScParams& s) {
    ScTerm t{0.f, 0.f, 0.f, 0.f, 0.f};
    const float r = sqrtf(r2);
    const float lam = s.lambda, lam_ = 1.0f - s.lambda;
    const float qq = qi * qj;
    const float Aa = a.x, Ab = a.y, Ba = b.x, Bb = b.y;
    if (!SOFT) {
        t.f = lam_ * lj_f(r, Aa, Ab) + lam * lj_f(r, Ba, Bb) - cf_f(qq, r, s.beta);
        if (E) {
            t.ecf = cf_e(qq, r, s.beta);
            t.elj = lam_ * lj_e(r, Aa, Ab) + lam * lj_e(r, Ba, Bb);
        }
        if (DU) {
            t.dlj = lj_e(r, Ba, Bb) - lj_e(r, Aa, Ab);
            t.dcf = erfcf(s.beta * r) * (qbaj * qi + qj * qbai) / r;
        }
    } else {
        const float sA = sc_sigma(Aa, Ab, s), sB = sc_sigma(Ba, Bb, s);
        const float rA = sc_dist(sA, r2, s.pow_l, s), rB = sc_dist(sB, r2, s.pow_l_, s);
        t.f = lam_ * sc_lj_f(r2, rA, Aa, Ab) + lam * sc_lj_f(r2, rB, Ba, Bb) -
              (lam_ * sc_cf_f(qq, r2, rA, s.beta) + lam * sc_cf_f(qq, r2, rB, s.beta));
        if (E) {
            t.ecf = lam_ * cf_e(qq, rA, s.beta) + lam * cf_e(qq, rB, s.beta);
            t.elj = lam_ * lj_e(rA, Aa, Ab) + lam * lj_e(rB, Ba, Bb);
        }
        if (DU) {
            t.dlj = lj_e(rB, Ba, Bb) - lj_e(rA, Aa, Ab) + sc_du(lj_f(rA, Aa, Ab), sA, rA, lam, s.pow1_l, s) -
                    sc_du(lj_f(rB, Ba, Bb), sB, rB, lam_, s.pow1_l_, s);
            const float qx = qbaj * qi + qj * qbai;
            t.dcf = cf_e(qq, rB, s.beta) - cf_e(qq, rA, s.beta) +
                    sc_du(cf_f(qq, rB, s.beta), sB, rB, lam_, s.pow1_l_, s) -
                    sc_du(cf_f(qq, rA, s.beta), sA, rA, lam, s.pow1_l, s) +
                    lam * erfcf(s.beta * rB) * qx / rB + lam_ * erfcf(s.beta * rA) * qx / rA;
        }
    }
    return t;
}

// Cell geometry for the force-only kernel's cell-centre images: reach =
// cutoff + the largest distance a row atom may have moved since the list was
// built (< 0: no bound known, periodic displacements kept).
struct ShiftGeom {
    float3 width;
    int Nx, Ny, Nz;
    float reach;
};

// LDS types of a partner: A-state type in the low byte, B-state type in the
// high one (at most 64 each).
__device__ __forceinline__ unsigned short pack_types(int tp) {
    return (unsigned short)((tp & 0xff) | ((tp >> 16) << 8));
}

// One pair of the force-only soft-core rows (displacement d): the plain
// kernel's FAST arithmetic with the state-weighted coefficients
// (1 - lambda) A_A + lambda A_B for pairs whose LJ is present in both states or
// in neither; true for the others in range, left to the soft-core pair
// function.  has = false: an absent entry of a partial pass (r^2 = the cutoff
// threshold, out of range).
template <bool POLY>
__device__ __forceinline__ bool sc_pair_fast(const float3& d, float r2, float qj, float2 a, float2 b,
                                             float qi, float lam, float lam_, float rc2_thr,
                                             const ScParams& sp, EwaldBracket ew, bool has,
                                             float& fx, float& fy, float& fz) {
    r2 = has ? r2 : rc2_thr;
    const bool in = r2 < rc2_thr;
    const bool plain = sc_plain(a, b);
    const float rinv = __builtin_amdgcn_rsqf(r2);
    const float r2inv = rinv * rinv;
    const float pw6 = r2inv * r2inv * r2inv;
    const float pw8 = pw6 * r2inv;
    const float cA = fmaf(lam, b.x, lam_ * a.x), cB = fmaf(lam, b.y, lam_ * a.y);
    float fc;
    if (POLY) {
        fc = r2inv * rinv * ew(r2 * rinv);
    } else {
        float erfc_br, bracket;
        coul_fast(r2, r2 * rinv, sp.beta, erfc_br, bracket);
        fc = rinv * r2inv * bracket;
    }
    float f = (cB - cA * pw6) * pw8 - qi * qj * fc;
    f = in && plain ? f : 0.f;
    fx = fmaf(f, d.x, fx);
    fy = fmaf(f, d.y, fy);
    fz = fmaf(f, d.z, fz);
    return in && !plain;
}

// Force-only row of a staged cell at cell-centre images: two entries per
// lane per pass from one 32-bit word (prefetched a pass ahead), the passes in
// which all 128 entries exist without presence tests, the partial last pass
// masked.
template <bool POLY>
__device__ __forceinline__ void sc_row_fast(int p, int lane, int n, const unsigned short* __restrict__ row,
                                            const float4* cpos, const unsigned short* ctp,
                                            const float4* __restrict__ pos, const float2* rowA,
                                            const float2* rowB, const LT6& c, const LT6& r,
                                            float rc2_thr, const ScParams& sp, EwaldBracket ew,
                                            float4* __restrict__ facc, float3 C,
                                            unsigned short* ring) {
    const float lam = sp.lambda, lam_ = 1.0f - sp.lambda;
    const float4 pi4 = pos[p];
    const float3 pi = image_offset(make_float3(pi4.x, pi4.y, pi4.z), C, c, r);
    float fx = 0.f, fy = 0.f, fz = 0.f;
    const int npairs = (n + 1) >> 1;
    const int full = n >> 7;
    const unsigned* row2 = reinterpret_cast<const unsigned*>(row);
    const unsigned last = npairs > 0 ? npairs - 1 : 0;
    unsigned cur = row2[(unsigned)lane < last ? (unsigned)lane : last];
    int w = lane;
    int head = 0, have = 0;  // soft-core pairs waiting in the ring
    auto batch = [&](int k) __attribute__((always_inline)) {
        wave_fence();
        if (lane < k) {
            const int t = ring[(head + lane) & (2 * kScRing - 1)];
            const float4 pj = cpos[t];
            const int tp = ctp[t];
            const float3 d = make_float3(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z);
            // (charge_BA enters only dU/dlambda)
            const float f = sc_pair<false, false, true>(fmaf(d.z, d.z, fmaf(d.y, d.y, d.x * d.x)), pi4.w,
                                                        pj.w, 0.f, 0.f, rowA[tp & 0xff], rowB[tp >> 8], sp).f;
            fx = fmaf(f, d.x, fx);
            fy = fmaf(f, d.y, fy);
            fz = fmaf(f, d.z, fz);
        }
        wave_fence();
    };
    auto pair = [&](int t, bool has) {
        const float4 pj = cpos[t];
        const int tp = ctp[t];
        const float3 d = make_float3(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z);
        const bool soft =
            sc_pair_fast<POLY>(d, fmaf(d.z, d.z, fmaf(d.y, d.y, d.x * d.x)), pj.w, rowA[tp & 0xff],
                               rowB[tp >> 8], pi4.w, lam, lam_, rc2_thr, sp, ew, has, fx, fy, fz);
        const unsigned long long m = __ballot(soft);
        if (m) {
            if (soft) ring[(head + have + lanes_below(m)) & (2 * kScRing - 1)] = (unsigned short)t;
            have += (int)__popcll(m);
        }
    };
    for (int k = 0; k < full; ++k, w += kWave) {
        const unsigned wn = (unsigned)(w + kWave);
        unsigned nxt = row2[wn < last ? wn : last];
        const int ta = (int)(cur & 0xffffu), tb = (int)(cur >> 16);
        pair(ta, true);
        pair(tb, true);
        // (at most 63 + 128 pairs wait here)
        while (have >= kWave) {
            batch(kWave);
            head = (head + kWave) & (2 * kScRing - 1);
            have -= kWave;
        }
        // the loaded word is opaque from here: the compiler cannot fold the
        // prefetch back into a load at the top of the next pass
        asm volatile("" : "+v"(nxt));
        cur = nxt;
    }
    if (full * 2 * kWave < n) {
        // cur is the row's word w, or its last word for lanes past the end
        const bool has_a = w < npairs;
        const bool has_b = 2 * w + 1 < n;
        const int ta = (int)(cur & 0xffffu);
        const int tb = has_b ? (int)(cur >> 16) : ta;
        pair(ta, has_a);
        pair(tb, has_b);
    }
    while (have > 0) {
        batch(have);
        head = (head + kWave) & (2 * kScRing - 1);
        have -= kWave;
    }
    fx = wave_sum(fx);
    fy = wave_sum(fy);
    fz = wave_sum(fz);
    if (lane == 0) facc[p] = make_float4(fx, fy, fz, 0.f);
}

struct ScStaged {
    float4 x;
    int tp;
    float qba;
    int gid;
};

template <bool ORTHO, bool F, bool E, bool V, bool DU, bool FAST = false>
__device__ __forceinline__ void ljsc_cells_body(int sa_block,
    const int* __restrict__ start, const int* __restrict__ g_stream,
    const long long* __restrict__ g_soff, const int* __restrict__ g_slen,
    const int* __restrict__ list_count, const unsigned short* __restrict__ list, int cap,
    const float4* __restrict__ pos, const int* __restrict__ ptp, const float* __restrict__ pqba,
    const int* __restrict__ pgid, const float2* __restrict__ ABa, int TA,
    const float2* __restrict__ ABb, int TB, LT6 c, LT6 r, float rc2_thr, ScParams sp,
    EwaldBracket ew, int stage, int split,
    float4* __restrict__ facc, float2* __restrict__ eacc, float* __restrict__ vacc,
    double* __restrict__ du, ShiftGeom sg, const StreamReport& report) {
    extern __shared__ float4 cpos[];
    // force-only steps stage positions and types only (18 B per entry)
    float* cqba = reinterpret_cast<float*>(cpos + stage);
    int* cgid = reinterpret_cast<int*>(cqba + stage);
    float2* ta = FAST ? reinterpret_cast<float2*>(cpos + stage) : reinterpret_cast<float2*>(cgid + stage);
    float2* tb = ta + TA * TA;
    unsigned short* ctp = reinterpret_cast<unsigned short*>(tb + TB * TB);
    unsigned short* ring = ctp + stage + 2 * kScRing * (threadIdx.x / kWave);
    report_streams(report, sa_block, stage);
    const int cell = sa_block / split, part = sa_block - cell * split;
    const int a0 = start[cell], a1 = start[cell + 1];
    if (a0 + part * (int)(blockDim.x / kWave) >= a1) return;
    const int total = g_slen[cell];
    const int* __restrict__ strm = g_stream + g_soff[cell];
    for (int k = threadIdx.x; k < TA * TA; k += blockDim.x) ta[k] = ABa[k];
    for (int k = threadIdx.x; k < TB * TB; k += blockDim.x) tb[k] = ABb[k];
    const bool staged = total <= stage;
    // force-only steps in an orthorhombic box wider than twice (half the cell
    // + reach) on every axis: partners staged at their images nearest the
    // cell's centre C (the plain pair kernel's construction)
    float3 C = make_float3(0.f, 0.f, 0.f);
    bool shift = false;
    if (FAST && ORTHO && sg.reach >= 0.f) {
        const int ix = cell / (sg.Ny * sg.Nz), iy = (cell / sg.Nz) % sg.Ny, iz = cell % sg.Nz;
        float lx, hx, ly, hy, lz, hz;
        cell_faces(ix, sg.Nx, sg.width.x, c.a11, lx, hx);
        cell_faces(iy, sg.Ny, sg.width.y, c.a22, ly, hy);
        cell_faces(iz, sg.Nz, sg.width.z, c.a33, lz, hz);
        C = image_centre(make_float3(0.5f * (lx + hx), 0.5f * (ly + hy), 0.5f * (lz + hz)), c);
        shift = staged && 0.5f * c.a11 > sg.reach + 0.5f * (hx - lx) + kCentreMargin &&
                0.5f * c.a22 > sg.reach + 0.5f * (hy - ly) + kCentreMargin &&
                0.5f * c.a33 > sg.reach + 0.5f * (hz - lz) + kCentreMargin;
    }
    if (staged)
        stage_stream(
            strm, total,
            [&](int q) {
                ScStaged e;
                e.x = pos[q];
                e.tp = ptp[q];
                if (!FAST) {
                    e.qba = pqba[q];
                    e.gid = pgid[q];
                }
                return e;
            },
            [&](int t, const ScStaged& e) {
                float4 v = e.x;
                if (shift) {
                    const float3 im = image_offset(make_float3(v.x, v.y, v.z), C, c, r);
                    v = make_float4(im.x, im.y, im.z, v.w);
                }
                cpos[t] = v;
                ctp[t] = pack_types(e.tp);
                if (!FAST) {
                    cqba[t] = e.qba;
                    cgid[t] = e.gid;
                }
            });
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave, nwave = blockDim.x / kWave;
    if (FAST) {
        // force-only steps: two entries per lane per pass, branch-free; the
        // pairs whose LJ is present in both states or in neither (all but
        // the perturbed atoms' pairs) take the plain kernel's arithmetic with
        // the state-weighted coefficients (1 - lambda) A_A + lambda A_B, the
        // soft-core pairs the reference's pair function, in batches
        const float lam = sp.lambda, lam_ = 1.0f - sp.lambda;
        if (shift) {
            for (int p = a0 + part * nwave + wave; p < a1; p += split * nwave) {
                const int tpi = ptp[p];
                const float2* rowA = ta + (tpi & 0xffff) * TA;
                const float2* rowB = tb + (tpi >> 16) * TB;
                const unsigned short* row = list + (size_t)p * cap;
                if (ew.scale > 0.f)
                    sc_row_fast<true>(p, lane, list_count[p], row, cpos, ctp, pos, rowA, rowB, c, r,
                                      rc2_thr, sp, ew, facc, C, ring);
                else
                    sc_row_fast<false>(p, lane, list_count[p], row, cpos, ctp, pos, rowA, rowB, c, r,
                                       rc2_thr, sp, ew, facc, C, ring);
            }
            return;
        }
        for (int p = a0 + part * nwave + wave; p < a1; p += split * nwave) {
            const float4 pi4 = pos[p];
            const float3 pi = make_float3(pi4.x, pi4.y, pi4.z);
            const int tpi = ptp[p];
            const float2* rowA = ta + (tpi & 0xffff) * TA;
            const float2* rowB = tb + (tpi >> 16) * TB;
            const int n = list_count[p];
            const unsigned short* row = list + (size_t)p * cap;
            float fx = 0.f, fy = 0.f, fz = 0.f;
            for (int base = 0; base < n; base += 2 * kWave) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int e = base + h * kWave + lane;
                    const bool has = e < n;
                    const int t = row[has ? e : 0];
                    const int q = staged ? t : strm[t];
                    const float4 pj = staged ? cpos[q] : pos[q];
                    const int tpj = staged ? ctp[q] : pack_types(ptp[q]);
                    const float3 d = disp_pbc<ORTHO>(make_float3(pj.x, pj.y, pj.z), pi, c, r);
                    const float r2 = norm2_exact(d);
                    const float2 a = rowA[tpj & 0xff], b = rowB[tpj >> 8];
                    const bool soft =
                        ew.scale > 0.f
                            ? sc_pair_fast<true>(d, r2, pj.w, a, b, pi4.w, lam, lam_, rc2_thr, sp, ew,
                                                 has, fx, fy, fz)
                            : sc_pair_fast<false>(d, r2, pj.w, a, b, pi4.w, lam, lam_, rc2_thr, sp, ew,
                                                  has, fx, fy, fz);
                    if (soft) {
                        const float f = sc_pair<false, false, true>(r2, pi4.w, pj.w, 0.f, 0.f, a, b, sp).f;
                        fx = fmaf(f, d.x, fx);
                        fy = fmaf(f, d.y, fy);
                        fz = fmaf(f, d.z, fz);
                    }
                }
            }
            fx = wave_sum(fx);
            fy = wave_sum(fy);
            fz = wave_sum(fz);
            if (lane == 0) facc[p] = make_float4(fx, fy, fz, 0.f);
        }
        return;
    }
    double wdl = 0, wdc = 0;  // dU/dlambda of this wavefront's rows
    for (int p = a0 + part * nwave + wave; p < a1; p += split * nwave) {
        const float4 pi4 = pos[p];
        const float3 pi = make_float3(pi4.x, pi4.y, pi4.z);
        const int tpi = ptp[p], gi = pgid[p];
        const float qbai = pqba[p];
        const float2* rowA = ta + (tpi & 0xffff) * TA;
        const float2* rowB = tb + (tpi >> 16) * TB;
        const int n = list_count[p];
        const unsigned short* row = list + (size_t)p * cap;
        float fx = 0.f, fy = 0.f, fz = 0.f, elj = 0.f, ecf = 0.f, dlj = 0.f, dcf = 0.f;
        float v0 = 0.f, v1 = 0.f, v2 = 0.f, v3 = 0.f, v4 = 0.f, v5 = 0.f;
        // pairs in range to the rings, evaluated in batches of 64; without
        // forces only the half-list's pairs count
        auto batch = [&](auto soft, const unsigned short* from, int k) __attribute__((always_inline)) {
            wave_fence();
            if (lane < k) {
                const int t = from[lane];
                const int q = staged ? t : strm[t];
                const float4 pj = staged ? cpos[q] : pos[q];
                const int tpj = staged ? ctp[q] : pack_types(ptp[q]);
                const float3 d = disp_pbc<ORTHO>(make_float3(pj.x, pj.y, pj.z), pi, c, r);
                const float qbaj = staged ? cqba[q] : pqba[q];
                const int gj = staged ? cgid[q] : pgid[q];
                const ScTerm tm = sc_pair<E, DU, decltype(soft)::value>(
                    norm2_exact(d), pi4.w, pj.w, qbai, qbaj, rowA[tpj & 0xff], rowB[tpj >> 8], sp);
                if (F) {
                    fx += tm.f * d.x;
                    fy += tm.f * d.y;
                    fz += tm.f * d.z;
                }
                if (gj > gi) {
                    // the reference's half-list row: energies, virial, dU/dlambda
                    elj += tm.elj;
                    ecf += tm.ecf;
                    dlj += tm.dlj;
                    dcf += tm.dcf;
                    if (V) {
                        const float lx = tm.f * d.x, ly = tm.f * d.y, lz = tm.f * d.z;
                        v0 -= lx * d.x;
                        v1 -= lx * d.y + ly * d.x;
                        v2 -= ly * d.y;
                        v3 -= lx * d.z + lz * d.x;
                        v4 -= ly * d.z + lz * d.y;
                        v5 -= lz * d.z;
                    }
                }
            }
            wave_fence();
        };
        int hp = 0, np = 0, hs = 0, ns = 0;  // plain and soft pairs waiting
        unsigned short* soft_ring = ring + kScRing;
        int cur = n > 0 ? (int)row[lane < n ? lane : n - 1] : 0;
        for (int e = lane; e - lane < n; e += kWave) {
            const bool has = e < n;
            const int en = e + kWave;
            int nxt = (int)row[en < n ? en : n - 1];
            const int q = staged ? cur : strm[cur];
            const float4 pj = staged ? cpos[q] : pos[q];
            const int tpj = staged ? ctp[q] : pack_types(ptp[q]);
            const float3 d = disp_pbc<ORTHO>(make_float3(pj.x, pj.y, pj.z), pi, c, r);
            bool in = has && norm2_exact(d) < rc2_thr;
            if (!F) in = in && (staged ? cgid[q] : pgid[q]) > gi;
            const bool plain = sc_plain(rowA[tpj & 0xff], rowB[tpj >> 8]);
            const unsigned long long mp = __ballot(in && plain), ms = __ballot(in && !plain);
            if (in && plain) ring[(hp + np + lanes_below(mp)) & (kScRing - 1)] = (unsigned short)cur;
            np += (int)__popcll(mp);
            if (np >= kWave) {
                batch(std::false_type{}, ring + hp, kWave);
                hp ^= kWave;
                np -= kWave;
            }
            if (ms) {
                if (in && !plain) soft_ring[(hs + ns + lanes_below(ms)) & (kScRing - 1)] = (unsigned short)cur;
                ns += (int)__popcll(ms);
                if (ns >= kWave) {
                    batch(std::true_type{}, soft_ring + hs, kWave);
                    hs ^= kWave;
                    ns -= kWave;
                }
            }
            asm volatile("" : "+v"(nxt));
            cur = nxt;
        }
        if (np) batch(std::false_type{}, ring + hp, np);
        if (ns) batch(std::true_type{}, soft_ring + hs, ns);
        if (F) {
            fx = wave_sum(fx);
            fy = wave_sum(fy);
            fz = wave_sum(fz);
        }
        double de = 0, dc = 0;
        if (E) {
            de = wave_sum((double)elj);
            dc = wave_sum((double)ecf);
        }
        if (DU) {
            wdl += wave_sum((double)dlj);
            wdc += wave_sum((double)dcf);
        }
        double w0 = 0, w1 = 0, w2 = 0, w3 = 0, w4 = 0, w5 = 0;
        if (V) {
            w0 = wave_sum((double)v0);
            w1 = wave_sum((double)v1);
            w2 = wave_sum((double)v2);
            w3 = wave_sum((double)v3);
            w4 = wave_sum((double)v4);
            w5 = wave_sum((double)v5);
        }
        if (lane == 0) {
            if (F) facc[p] = make_float4(fx, fy, fz, 0.f);
            if (E) eacc[p] = make_float2((float)de, (float)dc);
            if (V) {
                float* v = vacc + (size_t)6 * p;
                v[0] = (float)w0; v[1] = (float)w1; v[2] = (float)w2;
                v[3] = (float)w3; v[4] = (float)w4; v[5] = (float)w5;
            }
        }
    }
    // one hardware FP64 atomic per workgroup and sum: a pair of them per row
    // on the same two addresses took 120 of the kernel's 161 us at 6,000 atoms
    if (DU) {
        __shared__ double red[2][16];
        if (lane == 0) {
            red[0][wave] = wdl;
            red[1][wave] = wdc;
        }
        __syncthreads();
        if (threadIdx.x < 2) {
            double t = 0;
            for (int w = 0; w < nwave; ++w) t += red[threadIdx.x][w];
            unsafeAtomicAdd(&du[threadIdx.x], t);
        }
    }
}

}  // namespace

// The force-only kernels run at 8 wavefronts per SIMD (at most 64 VGPRs), as
// the plain pair kernel does.
template <>
struct sa::BodyWaves<&ljsc_cells_body<true, true, false, false, false, true>> {
    static constexpr int value = 8;
};
template <>
struct sa::BodyWaves<&ljsc_cells_body<false, true, false, false, false, true>> {
    static constexpr int value = 8;
};

namespace {

template <bool ORTHO, bool F, bool E, bool V, bool DU, bool FAST = false>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(FAST ? 8 : 1)))
k_ljsc_cells(
    const int* __restrict__ start, const int* __restrict__ g_stream,
    const long long* __restrict__ g_soff, const int* __restrict__ g_slen,
    const int* __restrict__ list_count, const unsigned short* __restrict__ list, int cap,
    const float4* __restrict__ pos, const int* __restrict__ ptp, const float* __restrict__ pqba,
    const int* __restrict__ pgid, const float2* __restrict__ ABa, int TA,
    const float2* __restrict__ ABb, int TB, LT6 c, LT6 r, float rc2_thr, ScParams sp, EwaldBracket ew,
    int stage, int split,
    float4* __restrict__ facc, float2* __restrict__ eacc, float* __restrict__ vacc,
    double* __restrict__ du, ShiftGeom sg, StreamReport report) {
    ljsc_cells_body<ORTHO, F, E, V, DU, FAST>(blockIdx.x, start, g_stream, g_soff, g_slen,
                                         list_count, list, cap, pos, ptp, pqba, pgid, ABa, TA, ABb,
                                         TB, c, r, rc2_thr, sp, ew, stage, split, facc, eacc, vacc, du, sg, report);
}

// Scatter of the rows: frc +=; atom_energy += LJ + Coulomb; the module's LJ
// energy and the direct-Coulomb energy overwritten (the reference clears
// them first, LJ_soft_core.cpp:776-785); atom_virial +=.
// assign: frc = instead of += (the step driver's first force term);
// reset_flag (nullable) is cleared by the first thread (the step driver's
// list-rebuild flag, once the rows of this step have been read).
template <bool E, bool V>
__device__ __forceinline__ void ljsc_finalize_body(int sa_block, int N, const int* __restrict__ sidx,
                                const float4* __restrict__ facc,
                                const float2* __restrict__ eacc, const float* __restrict__ vacc,
                                float* __restrict__ frc, float* __restrict__ atom_energy,
                                float* __restrict__ lj_energy, float* __restrict__ direct_energy,
                                float* __restrict__ atom_virial, int assign,
                                int* __restrict__ reset_flag) {
    const int p = sa_block * blockDim.x + threadIdx.x;
    if (p == 0 && reset_flag) *reset_flag = 0;
    if (p >= N) return;
    const int i = sidx[p];
    const float4 f = facc[p];
    if (assign) {
        frc[3 * i] = f.x;
        frc[3 * i + 1] = f.y;
        frc[3 * i + 2] = f.z;
    } else {
        frc[3 * i] += f.x;
        frc[3 * i + 1] += f.y;
        frc[3 * i + 2] += f.z;
    }
    if (E) {
        const float2 e = eacc[p];
        if (atom_energy) atom_energy[i] += e.x + e.y;
        lj_energy[i] = e.x;
        if (direct_energy) direct_energy[i] = e.y;
    }
    if (V && atom_virial)
        for (int k = 0; k < 6; ++k) atom_virial[6 * i + k] += vacc[6 * (size_t)p + k];
}

template <bool E, bool V>
__global__ void k_ljsc_finalize(int N, const int* __restrict__ sidx, const float4* __restrict__ facc,
                                const float2* __restrict__ eacc, const float* __restrict__ vacc,
                                float* __restrict__ frc, float* __restrict__ atom_energy,
                                float* __restrict__ lj_energy, float* __restrict__ direct_energy,
                                float* __restrict__ atom_virial, int assign,
                                int* __restrict__ reset_flag) {
    ljsc_finalize_body<E, V>(blockIdx.x, N, sidx, facc, eacc, vacc, frc, atom_energy, lj_energy,
                             direct_energy, atom_virial, assign, reset_flag);
}

__global__ void k_ljsc_add_scalar(float* p, float v) { p[0] += v; }

__global__ void k_ljsc_add_diag(float* p, float v) {
    p[0] += v;
    p[2] += v;
    p[5] += v;
}

__global__ void k_ljsc_sum(int N, const float* __restrict__ e, double* out) {
    double s = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) s += e[i];
    s = wave_sum(s);
    if ((threadIdx.x & (kWave - 1)) == 0) atomicAdd(out, s);
}

std::vector<float2> square_table(int T, const float* A, const float* B) {
    std::vector<float2> t((size_t)T * T);
    for (int a = 0; a < T; ++a)
        for (int b = 0; b < T; ++b) {
            const int k = lj_pair_index(a, b);
            t[(size_t)a * T + b] = make_float2(A[k], B[k]);
        }
    return t;
}

void ljsc_free(sponge_ljsc* h) {
    dfree(h->d_ABa);
    dfree(h->d_ABb);
    dfree(h->d_typeA);
    dfree(h->d_typeB);
    dfree(h->d_typeAB);
    dfree(h->d_pos);
    dfree(h->d_tp);
    dfree(h->d_qba);
    dfree(h->d_gid);
    dfree(h->d_facc);
    dfree(h->d_eacc);
    dfree(h->d_vacc);
    dfree(h->d_LJ_energy_atom);
    dfree(h->d_du);
    dfree(h->d_sum);
}

template <bool ORTHO>
int launch(sponge_ljsc* h, sponge_nl* nl, LT6 c, LT6 r, float beta, bool F, bool E, bool V,
           bool DU, float reach = -1.f) {
    const float lam = h->lambda, lam_ = 1.0f - lam;
    const ScParams sp{lam, h->alpha, h->p, h->sigma6, h->sigma6_min, beta, powf(lam, h->p),
                      powf(lam_, h->p), powf(lam + 1.17549435e-38f, h->p - 1.0f),
                      powf(lam_ + 1.17549435e-38f, h->p - 1.0f)};
    const ShiftGeom sg{nl->width, nl->Nx, nl->Ny, nl->Nz, reach};
    const bool fast = F && !E && !V && !DU && beta * h->cutoff <= kErfcxMax;
    const PairLaunch pl = pair_launch(
        nl, sizeof(float4) + (fast ? 0 : 2 * sizeof(int)) + sizeof(unsigned short),
        sizeof(float2) * ((size_t)h->TA * h->TA + (size_t)h->TB * h->TB) + kScRings, h->stage);
    const EwaldBracket ew = ewald_bracket(beta, h->cutoff);
    const int stage = pl.stage;
    const size_t sh = pl.lds;
#define SA_SC(f, e, v, d, fa)                                                                      \
    SA_LAUNCH(1024, (&ljsc_cells_body<ORTHO, f, e, v, d, fa>), (k_ljsc_cells<ORTHO, f, e, v, d, fa>),  \
              dim3(nl->G * pl.split), dim3(pl.threads), sh, h->stream,                                        \
                       nl->d_cell_start, nl->d_stream, nl->d_soff, nl->d_slen,                      \
                       nl->d_list_count, nl->d_list, nl->cap, h->d_pos, h->d_tp, h->d_qba,          \
                       h->d_gid, h->d_ABa, h->TA, h->d_ABb, h->TB, c, r, h->rc2_thr, sp, ew, stage, pl.split, \
                       h->d_facc, h->d_eacc, h->d_vacc, h->d_du, sg, pl.report)
    if (DU) SA_SC(false, false, false, true, false);
    else if (E && V) SA_SC(true, true, true, false, false);
    else if (E) SA_SC(true, true, false, false, false);
    else if (V) SA_SC(true, false, true, false, false);
    else if (fast) SA_SC(true, false, false, false, true);
    else SA_SC(true, false, false, false, false);
#undef SA_SC
    (void)F;
    SA_LAUNCH_CHECK();
    return 0;
}

int prepare(sponge_ljsc* h, sponge_nl* nl, const float* crd, const float* charge,
            const float* charge_BA) {
    if (!nl->built || nl->N != h->N) return SPONGE_AMD_ERROR_MISSING_COMMAND;
    SA_LAUNCH(256, (&ljsc_pack_body), (k_ljsc_pack), dim3(grid_for(h->N, 256)), dim3(256), 0,
              h->stream, h->N, nl->d_sidx, nl->d_spos, crd, charge, charge_BA, h->d_typeA, h->d_typeB,
                       h->d_pos, h->d_tp, h->d_qba, h->d_gid);
    SA_LAUNCH_CHECK();
    return 0;
}

}  // namespace

extern "C" {

void sponge_ljsc_default_options(sponge_ljsc_options* o) {
    if (!o) return;
    o->lambda = 0.0f;
    o->alpha = 0.5f;
    o->p = 1.0f;
    o->sigma = 3.0f;
    o->sigma_min = 0.0f;
}

int sponge_ljsc_initial(sponge_ljsc** out, int atom_numbers, int type_numbers_A,
                        int type_numbers_B, const float* LJ_AA, const float* LJ_AB,
                        const float* LJ_BA, const float* LJ_BB, const int* atom_type_A,
                        const int* atom_type_B, float cutoff, const sponge_ljsc_options* opt,
                        void* stream) {
    if (!out || atom_numbers <= 0 || type_numbers_A <= 0 || type_numbers_B <= 0 || !LJ_AA ||
        !LJ_AB || !LJ_BA || !LJ_BB || !atom_type_A || !atom_type_B || !(cutoff > 0.f))
        return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    *out = nullptr;
    if (type_numbers_A > 64 || type_numbers_B > 64) return SPONGE_AMD_ERROR_NOT_IMPLEMENTED;
    sponge_ljsc_options o;
    if (opt) o = *opt;
    else sponge_ljsc_default_options(&o);
    if (!(o.lambda >= 0.f && o.lambda <= 1.f) || !(o.p > 0.f)) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    const int N = atom_numbers, TA = type_numbers_A, TB = type_numbers_B;
    for (int i = 0; i < N; ++i)
        if (atom_type_A[i] < 0 || atom_type_A[i] >= TA || atom_type_B[i] < 0 || atom_type_B[i] >= TB)
            return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    sponge_ljsc* h = new sponge_ljsc();
    h->N = N;
    h->TA = TA;
    h->TB = TB;
    h->cutoff = cutoff;
    h->rc2_thr = sqrt_threshold(cutoff);
    h->lambda = o.lambda;
    h->alpha = o.alpha;
    h->p = o.p;
    h->sigma6 = powf(o.sigma, 6);
    h->sigma6_min = powf(o.sigma_min, 6);
    h->stream = (hipStream_t)stream;
    const size_t tables = sizeof(float2) * ((size_t)TA * TA + (size_t)TB * TB) + kScRings;
    h->stage = stage_entries(sizeof(float4) + 2 * sizeof(int) + sizeof(unsigned short), kScStage, tables);
    // long-range factors (LJ_soft_core.cpp:83-195, 640-668): sums of the
    // lambda-mixed and B - A C6 coefficients over all ordered pairs, by type
    // histograms, in double, scaled in float
    std::vector<long long> nA(TA, 0), nB(TB, 0);
    for (int i = 0; i < N; ++i) {
        nA[atom_type_A[i]]++;
        nB[atom_type_B[i]]++;
    }
    double sA = 0, sB = 0;
    for (int a = 0; a < TA; ++a)
        for (int b = 0; b < TA; ++b) sA += (double)nA[a] * nA[b] * LJ_AB[lj_pair_index(a, b)];
    for (int a = 0; a < TB; ++a)
        for (int b = 0; b < TB; ++b) sB += (double)nB[a] * nB[b] * LJ_BB[lj_pair_index(a, b)];
    const float lam_ = 1.0f - o.lambda;
    const float scale = -2.0f / 3.0f * 3.1415926535897932f / cutoff / cutoff / cutoff / 6.0f;
    h->long_range_factor = (float)((double)lam_ * sA + (double)o.lambda * sB) * scale;
    h->long_range_factor_TI = (float)(sB - sA) * scale;
    int e = 0;
    e |= dmalloc(&h->d_ABa, (size_t)TA * TA);
    e |= dmalloc(&h->d_ABb, (size_t)TB * TB);
    e |= dmalloc(&h->d_typeA, N);
    e |= dmalloc(&h->d_typeB, N);
    e |= dmalloc(&h->d_typeAB, N);
    e |= dmalloc(&h->d_pos, N);
    e |= dmalloc(&h->d_tp, N);
    e |= dmalloc(&h->d_qba, N);
    e |= dmalloc(&h->d_gid, N);
    e |= dmalloc(&h->d_facc, N);
    e |= dmalloc(&h->d_eacc, N);
    e |= dmalloc(&h->d_vacc, (size_t)6 * N);
    e |= dmalloc(&h->d_LJ_energy_atom, N);
    e |= dmalloc(&h->d_du, 2);
    e |= dmalloc(&h->d_sum, 1);
    if (e) {
        ljsc_free(h);
        delete h;
        return SPONGE_AMD_ERROR_MALLOC_FAILED;
    }
    const std::vector<float2> ta = square_table(TA, LJ_AA, LJ_AB), tb = square_table(TB, LJ_BA, LJ_BB);
    hipStream_t s = h->stream;
    hipError_t he = hipMemcpyAsync(h->d_ABa, ta.data(), sizeof(float2) * ta.size(), hipMemcpyHostToDevice, s);
    if (he == hipSuccess)
        he = hipMemcpyAsync(h->d_ABb, tb.data(), sizeof(float2) * tb.size(), hipMemcpyHostToDevice, s);
    if (he == hipSuccess)
        he = hipMemcpyAsync(h->d_typeA, atom_type_A, sizeof(int) * N, hipMemcpyHostToDevice, s);
    if (he == hipSuccess)
        he = hipMemcpyAsync(h->d_typeB, atom_type_B, sizeof(int) * N, hipMemcpyHostToDevice, s);
    std::vector<int> tab(N);
    for (int i = 0; i < N; ++i) tab[i] = atom_type_A[i] | (atom_type_B[i] << 16);
    if (he == hipSuccess)
        he = hipMemcpyAsync(h->d_typeAB, tab.data(), sizeof(int) * N, hipMemcpyHostToDevice, s);
    int rc = he == hipSuccess ? fill_async(h->d_LJ_energy_atom, 0.f, N, s) : (int)he;
    if (!rc) rc = fill_async(h->d_qba, 0.f, N, s);
    if (!rc && hipStreamSynchronize(s) != hipSuccess) rc = SPONGE_AMD_ERROR_MALLOC_FAILED;
    if (rc) {
        ljsc_free(h);
        delete h;
        return rc;
    }
    *out = h;
    return 0;
}

int sponge_ljsc_long_range_factors(sponge_ljsc* h, float* factor, float* factor_TI) {
    if (!h) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    if (factor) *factor = h->long_range_factor;
    if (factor_TI) *factor_TI = h->long_range_factor_TI;
    return 0;
}

int sponge_ljsc_direct_force(sponge_ljsc* h, sponge_nl* nl, const float* crd, const float* charge,
                             float* frc, const float* cell, const float* rcell, float pme_beta,
                             int need_atom_energy, float* atom_energy, int need_virial,
                             float* atom_virial, float* atom_direct_pme_energy) {
    if (!h || !nl || !crd || !charge || !frc || !cell || !rcell)
        return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    int rc = prepare(h, nl, crd, charge, nullptr);
    if (rc) return rc;
    const LT6 c = lt_from(cell), r = lt_from(rcell);
    const bool E = need_atom_energy != 0, V = need_virial != 0;
    timer_begin("ljsc_pairs", h->stream);
    rc = lt_is_orthorhombic(c) ? launch<true>(h, nl, c, r, pme_beta, true, E, V, false)
                               : launch<false>(h, nl, c, r, pme_beta, true, E, V, false);
    timer_end("ljsc_pairs", h->stream);
    if (rc) return rc;
    const dim3 g(grid_for(h->N, 256)), b(256);
#define SA_FIN(e, v)                                                                              \
    SA_LAUNCH(256, (&ljsc_finalize_body<e, v>), (k_ljsc_finalize<e, v>), g, b, 0, h->stream, h->N, \
              nl->d_sidx, h->d_facc, h->d_eacc, h->d_vacc, frc, atom_energy, h->d_LJ_energy_atom, \
              atom_direct_pme_energy, atom_virial, 0, (int*)nullptr)
    if (E && V) SA_FIN(true, true);
    else if (E) SA_FIN(true, false);
    else if (V) SA_FIN(false, true);
    else SA_FIN(false, false);
#undef SA_FIN
    SA_LAUNCH_CHECK();
    return 0;
}

int sponge_ljsc_du_dlambda(sponge_ljsc* h, sponge_nl* nl, const float* crd, const float* charge,
                           const float* charge_BA, const float* cell, const float* rcell,
                           float pme_beta, float* du_lj, float* du_direct) {
    if (!h || !nl || !crd || !charge || !cell || !rcell) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    int rc = prepare(h, nl, crd, charge, charge_BA);
    if (!rc) rc = fill_async(h->d_du, 0.0, 2, h->stream);
    if (rc) return rc;
    const LT6 c = lt_from(cell), r = lt_from(rcell);
    rc = lt_is_orthorhombic(c) ? launch<true>(h, nl, c, r, pme_beta, false, false, false, true)
                               : launch<false>(h, nl, c, r, pme_beta, false, false, false, true);
    if (rc) return rc;
    double d[2];
    SA_CHECK(hipMemcpyAsync(d, h->d_du, sizeof(d), hipMemcpyDeviceToHost, h->stream));
    SA_CHECK(hipStreamSynchronize(h->stream));
    // Get_Partial_H_Partial_Lambda_With_Columb_Direct (LJ_soft_core.cpp:828-880)
    // adds the long-range TI term to the LJ part
    const float volume = c.a11 * c.a22 * c.a33;
    if (du_lj) *du_lj = (float)d[0] + h->long_range_factor_TI / volume;
    if (du_direct) *du_direct = (float)d[1];
    return 0;
}

// LJ_SOFT_CORE::Long_Range_Correction (LJ_soft_core.cpp:928-946)
int sponge_ljsc_long_range_correction(sponge_ljsc* h, int need_pressure, float* d_virial,
                                      int need_potential, float* d_potential, float volume) {
    if (!h || !(volume > 0.f)) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    if (need_pressure) {
        if (!d_virial) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
        hipLaunchKernelGGL(k_ljsc_add_diag, dim3(1), dim3(1), 0, h->stream, d_virial,
                           2 * h->long_range_factor / volume);
        SA_LAUNCH_CHECK();
    }
    if (need_potential) {
        if (!d_potential) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
        hipLaunchKernelGGL(k_ljsc_add_scalar, dim3(1), dim3(1), 0, h->stream, d_potential,
                           h->long_range_factor / volume);
        SA_LAUNCH_CHECK();
    }
    return 0;
}

int sponge_ljsc_step_print(sponge_ljsc* h, float* LJ_soft_short) {
    if (!h) return SPONGE_AMD_ERROR_VALUE_ERROR_COMMAND;
    int rc = fill_async(h->d_sum, 0.0, 1, h->stream);
    if (rc) return rc;
    hipLaunchKernelGGL(k_ljsc_sum, dim3(64), dim3(256), 0, h->stream, h->N, h->d_LJ_energy_atom,
                       h->d_sum);
    SA_LAUNCH_CHECK();
    double sum = 0;
    SA_CHECK(hipMemcpyAsync(&sum, h->d_sum, sizeof(double), hipMemcpyDeviceToHost, h->stream));
    SA_CHECK(hipStreamSynchronize(h->stream));
    if (LJ_soft_short) *LJ_soft_short = (float)sum;
    return 0;
}

int sponge_ljsc_clear(sponge_ljsc* h) {
    if (!h) return 0;
    (void)hipStreamSynchronize(h->stream);
    ljsc_free(h);
    delete h;
    return 0;
}

}  // extern "C"

// The step driver's form of the direct-force call: frc assigned (the step's
// first force term), the list's rebuild flag cleared once the rows were read,
// per-atom energies only on energy steps.
int sa::ljsc_direct_force_md(sponge_ljsc* h, sponge_nl* nl, const float* crd, const float* charge,
                             float* frc, const float* cell, const float* rcell, float pme_beta,
                             int need_atom_energy, float* atom_energy,
                             float* atom_direct_pme_energy, int* reset_flag, bool* deferred,
                             bool packed) {
    int rc = packed ? 0 : prepare(h, nl, crd, charge, nullptr);
    if (rc) return rc;
    const LT6 c = lt_from(cell), r = lt_from(rcell);
    const bool E = need_atom_energy != 0;
    // the automatic refresh rebuilds once any atom moved more than
    // skin * skin_permit: the force-only kernel may use cell-centre images
    const float reach = nl->opt.refresh_interval <= 0 ? h->cutoff + nl->skin * nl->opt.skin_permit
                                                      : -1.f;
    {
        ScopedTimer timer("ljsc_pairs", h->stream);
        rc = lt_is_orthorhombic(c)
                 ? launch<true>(h, nl, c, r, pme_beta, true, E, false, false, reach)
                 : launch<false>(h, nl, c, r, pme_beta, true, E, false, false, reach);
    }
    if (rc) return rc;
    // a force-only step may leave the per-row forces to the PME gather
    if (deferred) {
        *deferred = !E;
        if (!E) return 0;
    }
    const dim3 g(grid_for(h->N, 256)), b(256);
    if (E)
        SA_LAUNCH(256, (&ljsc_finalize_body<true, false>), (k_ljsc_finalize<true, false>), g, b, 0,
                  h->stream, h->N, nl->d_sidx, h->d_facc, h->d_eacc, h->d_vacc, frc, atom_energy,
                  h->d_LJ_energy_atom, atom_direct_pme_energy, (float*)nullptr, 1, reset_flag);
    else
        SA_LAUNCH(256, (&ljsc_finalize_body<false, false>), (k_ljsc_finalize<false, false>), g, b,
                  0, h->stream, h->N, nl->d_sidx, h->d_facc, h->d_eacc, h->d_vacc, frc,
                  atom_energy, h->d_LJ_energy_atom, atom_direct_pme_energy, (float*)nullptr, 1,
                  reset_flag);
    SA_LAUNCH_CHECK();
    return 0;
}

const float4* sa::ljsc_row_forces(const sponge_ljsc* h) { return h->d_facc; }
// (charge_BA enters only dU/dlambda, whose call packs its own)
PackTarget sa::ljsc_pack_target(sponge_ljsc* h, const float* charge) {
    return {h->d_pos, h->d_tp, h->d_gid, charge, h->d_typeAB};
}
void sa::ljsc_set_stream(sponge_ljsc* h, hipStream_t s, const StreamOwner& owner) {
    h->stream = s;
    h->owner = owner;
}
int sa::ljsc_atoms(const sponge_ljsc* h) { return h->N; }
float sa::ljsc_long_range_factor(const sponge_ljsc* h) { return h->long_range_factor; }
