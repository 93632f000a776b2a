// Per-pair arithmetic and tile loads of the all-pairs kernels, shared by the
// wave-per-item kernels (pair_kernels.hip) and the block-per-item kernels for
// small work lists (pair_wide.hip).  Both forms evaluate a pair with the same
// products in the same order, so their results agree bit for bit.  Which
// product is fused into which sum is written out and contraction is off in the
// functions below that form pair terms: left to the compiler it depends on the
// loop they are inlined into.
//
//   descreening   energy/src/gb.rs:271-283 (pair), :347-369 (h)
//   LJ + Coulomb  energy/src/forces_nonbonded.rs:196-232
//   GB pair force energy/src/forces_gb.rs:72-112
#pragma once
#include "og_device.h"
#include "og_kernels.h"

namespace {

constexpr float kGbK = (float)(1.0 - 1.0 / OG_EPS_WATER);
constexpr float kHalfLn2 = 0.34657359027997264f;

struct LaneData {
    float x, y, z, q;
    float4 par;   // se, rm, se14, rm14
    float4 gb;    // rho~, S, R, invRq
};

__device__ __forceinline__ LaneData load_lane(const og_pair_args& a, int tile, int atom0, int cnt,
                                              int lane, double ox, double oy, double oz) {
    LaneData d;
    const int slot = tile * OG_TILE + lane;
    if (lane < cnt) {
        const double* p = a.pos + 3 * (size_t)(atom0 + lane);
        d.x = (float)(p[0] - ox);
        d.y = (float)(p[1] - oy);
        d.z = (float)(p[2] - oz);
    } else {
        // Padding slot: far away and (via zero parameters) inert.
        d.x = 1.0e6f + 97.0f * (float)lane;
        d.y = 1.0e6f;
        d.z = 1.0e6f;
    }
    d.q = a.qs[slot];
    d.par = a.par[slot];
    d.gb = a.gb[slot];
    return d;
}

__device__ __forceinline__ float rl(float v, int j) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}

// one-lane rotation of a value around the wave (DPP wave_rol:1)
// (mov_dpp: every lane is written, so no "old" value has to be materialised)
__device__ __forceinline__ float rot(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x134, 0xF, 0xF, false));
}
__device__ __forceinline__ int roti(int v) { return __builtin_amdgcn_mov_dpp(v, 0x134, 0xF, 0xF, false); }
// exchange with the lane 32 away (halves of the wave)
__device__ __forceinline__ float swap32(float v) { return __shfl_xor(v, 32, 64); }

// Descreening integral term h(r, rho~_i, S_j) of energy/src/gb.rs:347-369,
// written with one reciprocal and one log:  1/L - 1/U = (U-L)/(LU),
// 1/U^2 - 1/L^2 = -(1/L - 1/U)(U+L)/(LU),  ln(L/U) = ln(L^2/(LU)), with
// L = max(r - S, rho~) covering both the overlapping and the separate case.
__device__ __forceinline__ float descreen_h(float r2, float inv_r, float rt, float S, float S2) {
#pragma clang fp contract(off)
    // r = r2 * inv_r is not rounded on its own (left to the compiler, some
    // loops did and some did not)
    const float U = fmaf(r2, inv_r, S);
    const float L = fmaxf(fmaf(r2, inv_r, -S), rt);
    const float UmL = U - L;
    const float UpL = U + L;
    const float w = __builtin_amdgcn_rcpf(L * U);
    const float t = UmL * w;
    const float s2q = S2 * (0.25f * inv_r);
    const float lg = __builtin_amdgcn_logf(L * L * w);   // log2
    float h = fmaf(0.5f, t, -(t * UpL * w) * s2q);
    h = fmaf(lg, kHalfLn2 * inv_r, h);
    return (U <= rt) ? 0.0f : h;
}

// Orders a wave's own LDS accesses across lanes for the compiler; a wave's
// LDS operations are performed in program order, so no wait is needed.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Far-field form of descreen_tile_lds for tile pairs whose atoms are all at
// least og_pair_args::ds_far apart: there S / r <= 0.1 and L = r - S, and
// the HCT term (1/r)[x/(1-x^2) - x^3/(1-x^2)^2 - atanh x], x = S/r, is the
// series (1/r) sum_n c_n x^(2n+1), c_n = 1 - n - 1/(2n+1):
//   h = -(S^3 / (3 r^4)) (1 + 3.6 y + (45/7) y^2 + (28/3) y^3),  y = x^2,
// whose next term, (135/11) y^4 relative, is below 1.3e-7 at x = 0.1 (FP32
// rounding is 6e-8); the closed form evaluated in FP32 there loses about
// 6e-8 / x^2 to cancellation.  Every term is negative, as h is.  Q[e].z holds
// -S^3/3 of j atom e.
template <bool MODEA, int PART>
__device__ __forceinline__ void descreen_tile_far(const og_pair_args& a, const LaneData& di,
                                                  const float4* P, const float4* Q, int lane,
                                                  float& acc_i, float& acc_j) {
#pragma clang fp contract(off)
    float gj = 0.0f;
    const float Si2 = di.gb.y * di.gb.y;
    const float ci3 = (-1.0f / 3.0f) * Si2 * di.gb.y;
    auto series = [](float y) { return fmaf(y, fmaf(y, fmaf(y, 28.0f / 3.0f, 45.0f / 7.0f), 3.6f), 1.0f); };
    auto step = [&](float4 pj, float4 qj) {
        const float dx = pj.x - di.x, dy = pj.y - di.y, dz = pj.z - di.z;
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
        const float inv_r = __builtin_amdgcn_rsqf(r2);
        const float inv_r2 = inv_r * inv_r;
        const float inv_r4 = inv_r2 * inv_r2;
        const float ki = qj.z * inv_r4, si = series(qj.y * inv_r2);
        const float kj = ci3 * inv_r4, sj = series(Si2 * inv_r2);
        if (MODEA) {
            const bool ok = r2 <= a.rc2_ds;
            acc_i += ok ? ki * si : 0.0f;
            gj += ok ? kj * sj : 0.0f;
        } else {
            acc_i = fmaf(ki, si, acc_i);
            gj = fmaf(kj, sj, gj);
        }
        gj = rot(gj);                  // after step 63 this is the way home
    };
    constexpr int kb = PART == 1 ? 32 : 0, ke = PART == 0 ? 32 : 64;
    for (int k = kb; k < ke; k += 2) {
        const int idx = (lane + k) & 63;
        const float4 p0 = P[idx], p1 = P[idx + 1];
        const float4 q0 = Q[idx], q1 = Q[idx + 1];
        step(p0, q0);
        step(p1, q1);
    }
    if (PART == 0) gj = swap32(gj);
    acc_j += gj;
}

__device__ __forceinline__ float wave_max_f(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// Radius of a tile's atoms (lanes below cnt) about the point (x0, y0, z0).
__device__ __forceinline__ float tile_radius(const LaneData& d, int cnt, int lane, float x0, float y0, float z0) {
    const float ex = d.x - x0, ey = d.y - y0, ez = d.z - z0;
    return wave_max_f(lane < cnt ? sqrtf(fmaf(ex, ex, fmaf(ey, ey, ez * ez))) : 0.0f);
}

// Every pair of a tile pair lies beyond a cutoff (rc2 its square): the
// distance of the two first atoms (positions are relative to the i side's
// origin) less both tiles' radii about them bounds every pair's distance from
// below; the margin covers the FP32 rounding at any size.  Such a tile pair
// adds exact zeros under a cutoff and is left out.  A bound that is not finite
// leaves nothing out.
__device__ __forceinline__ bool tiles_beyond(float rad_i, const LaneData& dj, int cj, int lane, float rc2) {
    const float jx0 = rl(dj.x, 0), jy0 = rl(dj.y, 0), jz0 = rl(dj.z, 0);
    const float rad_j = tile_radius(dj, cj, lane, jx0, jy0, jz0);
    const float d0 = sqrtf(fmaf(jx0, jx0, fmaf(jy0, jy0, jz0 * jz0)));
    const float far = d0 - rad_i - rad_j - (1e-3f + 1e-6f * (d0 + rad_i + rad_j));
    return far > 0.0f && far < 1e15f && far * far > rc2;
}

__device__ __forceinline__ float force_cutoff2(const og_pair_args& a) { return fmaxf(a.rc2_nb, a.rc2_gb); }

// Far tile pair of the descreening pass: the distance of the two first atoms
// less the radii of both tiles about them (positions are relative to the i
// tile's first atom, so lane 0's i position is the origin) bounds every pair's
// distance from below; 1e-3 A covers the FP32 rounding.
__device__ __forceinline__ bool descreen_far(const og_pair_args& a, const LaneData& di, const LaneData& dj, int ci,
                                             int cj, int lane) {
    const float jx0 = rl(dj.x, 0), jy0 = rl(dj.y, 0), jz0 = rl(dj.z, 0);
    const float ri = lane < ci ? sqrtf(fmaf(di.x, di.x, fmaf(di.y, di.y, di.z * di.z))) : 0.0f;
    const float ex = dj.x - jx0, ey = dj.y - jy0, ez = dj.z - jz0;
    const float rj = lane < cj ? sqrtf(fmaf(ex, ex, fmaf(ey, ey, ez * ez))) : 0.0f;
    const float d0 = sqrtf(fmaf(jx0, jx0, fmaf(jy0, jy0, jz0 * jz0)));
    return a.ds_far > 0.0f && d0 - wave_max_f(ri) - wave_max_f(rj) - 1e-3f >= a.ds_far;
}

// Pair coefficient c (force on i = c * d, d = x_j - x_i) of a tile pair's
// fused LJ + Coulomb + GB-pair force.  MASKED: excl drops the LJ and Coulomb
// terms, one4 selects the 1-4 parameters.
template <bool MODEA, bool MASKED>
__device__ __forceinline__ float tile_coef(const og_pair_args& a, const LaneData& di, float qki, float qj, float sej,
                                           float rmj, float se14j, float rm14j, float Rj, float iRj, bool excl,
                                           bool one4, float dx, float dy, float dz) {
#pragma clang fp contract(off)
    const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
    const float inv_r = __builtin_amdgcn_rsqf(r2);
    const float inv_r2 = inv_r * inv_r;
    float rmin, eij;
    if (MASKED) {
        rmin = one4 ? di.par.w + rm14j : di.par.y + rmj;
        eij = one4 ? di.par.z * se14j : di.par.x * sej;
    } else {
        rmin = di.par.y + rmj;
        eij = di.par.x * sej;
    }
    const float t2 = rmin * rmin * inv_r2;
    const float t6 = t2 * t2 * t2;
    const float qq = di.q * qj;
    float coul;
    if (MODEA) coul = -qq * fmaf(inv_r2, inv_r, -a.inv_rc3);
    else coul = -qq * inv_r2 * inv_r;
    float cnb = fmaf(eij * inv_r2, fmaf(-t6, t6, t6), coul);
    if (MODEA) cnb = (r2 <= a.rc2_nb) ? cnb : 0.0f;
    if (MASKED) cnb = excl ? 0.0f : cnb;
    // GB pair (frozen radii): f^2 = r^2 + R_i R_j exp(-r^2 / (4 R_i R_j))
    const float Rp = di.gb.z * Rj;
    const float e = __builtin_amdgcn_exp2f(-r2 * (di.gb.w * iRj));
    const float f2 = fmaf(Rp, e, r2);
    const float inv_f = __builtin_amdgcn_rsqf(f2);
    const float qgb = qki * qj;
    const float k = qgb * fmaf(-0.25f, e, 1.0f), f3 = inv_f * inv_f * inv_f;
    const float c = MODEA ? cnb + (r2 <= a.rc2_gb ? k * f3 : 0.0f) : fmaf(k, f3, cnb);
    return r2 >= 1e-18f ? c : 0.0f;
}

// One i atom of a strip: position relative to the strip's origin, charge,
// LJ and GB parameters, and its force sum over the strip.
struct StripAtom {
    float x, y, z, q;
    float se, rm, R, gw;
    float fx, fy, fz;
};

__device__ __forceinline__ StripAtom strip_atom(const LaneData& d) {
    return {d.x, d.y, d.z, d.q, d.par.x, d.par.y, d.gb.z, d.gb.w, 0.0f, 0.0f, 0.0f};
}

// Pair coefficient c (force on i = c * d, d = x_j - x_i) of the fused
// LJ + Coulomb + GB-pair force for an unmasked pair; j data as in the LDS
// layout of force_tile_lds (P = x, y, z, q; Q = se, rm, R, 1/R scaled).
// Mode B groups the two charge terms: q_i q_j (k_GB (1 - e/4) / f^3 - 1/r^3).
// FAR: every pair of the j tile has r^2 gw_i gw_j >= 32 (gw = sqrt(log2 e / 4)
// / R), so e = exp2(-r^2 gw_i gw_j) <= 2^-32.  Then R_i R_j e is below 1e-11
// r^2 (r^2 = 4 R_i R_j x, x = r^2 gw_i gw_j / log2 e >= 22), far under half an
// FP32 ulp of r^2, so f^2 = fma(R_i R_j, e, r^2) rounds to r^2 and 1/f is the
// 1/r above; likewise k (1 - e/4) rounds to k.  The exponential and the
// second square root are left out, with the same products in the same order:
// the coefficient is bit-identical.
template <bool MODEA, bool FAR = false>
__device__ __forceinline__ float strip_coef(const og_pair_args& a, const StripAtom& I, float4 pj, float4 qj,
                                            float dx, float dy, float dz) {
#pragma clang fp contract(off)
    const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
    const float inv_r = __builtin_amdgcn_rsqf(r2);
    const float inv_r2 = inv_r * inv_r;
    const float rmin = I.rm + qj.y;
    const float t2 = rmin * rmin * inv_r2;
    const float t6 = t2 * t2 * t2;
    const float lj = (I.se * qj.x) * inv_r2 * fmaf(-t6, t6, t6);
    const float qq = I.q * pj.w;
    float k, f3;
    if (FAR) {
        k = kGbK;
        f3 = inv_r * inv_r * inv_r;
    } else {
        const float e = __builtin_amdgcn_exp2f(-r2 * (I.gw * qj.w));
        const float f2 = fmaf(I.R * qj.z, e, r2);
        const float inv_f = __builtin_amdgcn_rsqf(f2);
        k = fmaf(-0.25f * kGbK, e, kGbK);
        f3 = inv_f * inv_f * inv_f;
    }
    if (MODEA) {
        float cnb = fmaf(-qq, fmaf(inv_r2, inv_r, -a.inv_rc3), lj);
        cnb = (r2 <= a.rc2_nb) ? cnb : 0.0f;
        const float gbc = (r2 <= a.rc2_gb) ? qq * (k * f3) : 0.0f;
        return cnb + gbc;
    }
    return fmaf(qq, fmaf(k, f3, -(inv_r2 * inv_r)), lj);
}

// Bounds of a strip's two i tiles about the origin (the first one's first
// atom; both tiles are full) and their smallest gw, for the far test.
struct StripBound {
    float rad, gw;
};

__device__ __forceinline__ StripBound strip_bound(const StripAtom& A, const StripAtom& B) {
    return {wave_max_f(fmaxf(sqrtf(fmaf(A.x, A.x, fmaf(A.y, A.y, A.z * A.z))),
                             sqrtf(fmaf(B.x, B.x, fmaf(B.y, B.y, B.z * B.z))))),
            -wave_max_f(-fminf(A.gw, B.gw))};
}

// Far j tile: the smallest pair distance (distance of the first atoms less
// both tiles' radii, 1e-3 A for FP32 rounding) gives r^2 gw_i gw_j >= 33 for
// every pair (padding slots excluded).
__device__ __forceinline__ bool strip_far(const StripBound& b, const LaneData& dj, int cj, int lane) {
    const float jx0 = rl(dj.x, 0), jy0 = rl(dj.y, 0), jz0 = rl(dj.z, 0);
    const float ex = dj.x - jx0, ey = dj.y - jy0, ez = dj.z - jz0;
    const float rad_j = wave_max_f(lane < cj ? sqrtf(fmaf(ex, ex, fmaf(ey, ey, ez * ez))) : 0.0f);
    const float gw_j = -wave_max_f(lane < cj ? -dj.gb.w : -1.0e30f);
    const float rmn = sqrtf(fmaf(jx0, jx0, fmaf(jy0, jy0, jz0 * jz0))) - b.rad - rad_j - 1e-3f;
    return rmn > 0.0f && rmn * rmn * (b.gw * gw_j) >= 33.0f;
}

// ---------------------------------------------------------------------------
// FP64 pair energies (og_k_energy64, og_k_wide_energy)
// ---------------------------------------------------------------------------
// 1/sqrt(x) for x > 0 in FP64: the hardware estimate refined by two Newton
// steps (each doubles the number of correct bits), in place of a correctly
// rounded square root and division.
__device__ __forceinline__ double rsqrt64(double x) {
    double y = __builtin_amdgcn_rsq(x);
    double h = x * y;
    double e = fma(-h, y, 1.0);
    y = fma(0.5 * y, e, y);
    h = x * y;
    e = fma(-h, y, 1.0);
    return fma(0.5 * y, e, y);
}

// j atom data for the FP64 energy pass, one entry per j atom of the tile in
// the wave's LDS: every lane reads the same entry in a step (a broadcast).
struct EJ {
    double x, y, z, q;
    double rm, se, rm14, se14;     // Rmin/2, sqrt(eps), 1-4 variants
    double R, iR;                  // Born radius and its reciprocal
};


// The lane's i atom.
struct EI {
    double x, y, z, q, rm, se, rm14, se14, R, iR;
    bool valid;
};
struct ESum {
    double lj, c, g;
};

__device__ __forceinline__ EI energy_i(const og_pair_args& a, const og_energy64_args& e, int gi, bool valid, double R) {
    return {a.pos[3 * (size_t)gi], a.pos[3 * (size_t)gi + 1], a.pos[3 * (size_t)gi + 2], e.charge[gi], e.rmin[gi],
            sqrt(e.eps[gi]), e.rmin14[gi], sqrt(e.eps14[gi]), R, 1.0 / R, valid};
}

__device__ __forceinline__ EJ energy_j(const og_pair_args& a, const og_energy64_args& e, int gj, double R) {
    EJ m;
    m.x = a.pos[3 * (size_t)gj]; m.y = a.pos[3 * (size_t)gj + 1]; m.z = a.pos[3 * (size_t)gj + 2];
    m.q = e.charge[gj];
    m.rm = e.rmin[gj]; m.se = sqrt(e.eps[gj]);
    m.rm14 = e.rmin14[gj]; m.se14 = sqrt(e.eps14[gj]);
    m.R = R; m.iR = 1.0 / R;
    return m;
}

// j atoms [j0, j1) of an off-diagonal tile pair without excluded or 1-4
// pairs: the terms with the mask and 1-4 selects left out.
template <bool MODEA>
__device__ __forceinline__ void energy_plain(const og_energy64_args& e, const EI& I, const EJ* J, int j0, int j1,
                                             ESum& t) {
    const double xo = I.valid ? I.x : I.x + 1.0e6;       // padding lanes: far away, added as 0
    for (int jj = j0; jj < j1; ++jj) {
        const EJ d = J[jj];
        const double dx = xo - d.x, dy = I.y - d.y, dz = I.z - d.z;
        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
        const double qq = I.q * d.q;
        const double inv_r = rsqrt64(r2);
        const double s = (I.rm + d.rm) * inv_r;
        const double t2 = s * s;
        const double t6 = t2 * t2 * t2;
        const double lj = (I.se * d.se) * fma(t6, t6, -2.0 * t6);
        double c = qq * inv_r;
        bool nb = I.valid;
        if (MODEA) {
            c = qq * (inv_r + e.kappa * r2 - e.crf);
            nb = nb && (r2 <= e.rc2_nb);
        }
        t.lj += nb ? lj : 0.0;
        t.c += nb ? c : 0.0;
        // f_GB^2 = r^2 + R_i R_j exp(-x), x = r^2 / (4 R_i R_j).  From
        // x >= 60 on, R_i R_j exp(-x) < 1e-12 x 2^-52 r^2 (r^2 = 4 x R_i R_j),
        // far below half an ulp of r^2, so the fma rounds to r^2 exactly
        // and 1/f_GB is the 1/r above: the exponential and the second
        // square root are left out there, bit for bit.
        const double x = 0.25 * r2 * (I.iR * d.iR);
        double inv_f = inv_r;
        if (!(x >= 60.0)) inv_f = rsqrt64(fma(I.R * d.R, exp(-x), r2));
        t.g += I.valid ? qq * inv_f : 0.0;
    }
}

// The same where every pair is beyond the LJ and Coulomb cutoff and has
// x >= 60 (energy_tiles_far): only q_i q_j / r is left, the same bits.
__device__ __forceinline__ void energy_far(const EI& I, const EJ* J, int j0, int j1, ESum& t) {
    for (int jj = j0; jj < j1; ++jj) {
        const double dx = I.x - J[jj].x, dy = I.y - J[jj].y, dz = I.z - J[jj].z;
        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
        t.g += I.valid ? I.q * J[jj].q * rsqrt64(r2) : 0.0;
    }
}

// j atoms [j0, j1) of a diagonal or masked tile pair.
template <bool MODEA>
__device__ __forceinline__ void energy_masked(const og_energy64_args& e, const EI& I, const EJ* J, int j0, int j1,
                                              int lane, bool diag, unsigned long long xm, unsigned long long m14,
                                              ESum& t) {
    for (int jj = j0; jj < j1; ++jj) {
        const EJ d = J[jj];
        const double dx = I.x - d.x, dy = I.y - d.y, dz = I.z - d.z;
        const bool ok = I.valid && (!diag || jj > lane);
        const double r2 = ok ? fma(dx, dx, fma(dy, dy, dz * dz)) : 1.0;
        const double qq = I.q * d.q;
        const bool one4 = (m14 >> jj) & 1ull;
        bool nb = ok && !((xm >> jj) & 1ull);
        if (MODEA) nb = nb && (r2 <= e.rc2_nb);
        const double inv_r = rsqrt64(r2);
        const double rmij = one4 ? I.rm14 + d.rm14 : I.rm + d.rm;
        const double eij = one4 ? I.se14 * d.se14 : I.se * d.se;
        const double s = rmij * inv_r;
        const double t2 = s * s;
        const double t6 = t2 * t2 * t2;
        const double lj = eij * fma(t6, t6, -2.0 * t6);
        double c = qq * inv_r;
        if (MODEA) c = qq * (inv_r + e.kappa * r2 - e.crf);
        t.lj += nb ? lj : 0.0;
        t.c += nb ? c : 0.0;
        const double x = 0.25 * r2 * (I.iR * d.iR);      // as in energy_plain
        double inv_f = inv_r;
        if (!(x >= 60.0)) inv_f = rsqrt64(fma(I.R * d.R, exp(-x), r2));
        t.g += ok ? qq * inv_f : 0.0;
    }
}

// Every pair of the tile pair is beyond the LJ and Coulomb cutoff and has
// r^2 / (4 R_i R_j) >= 60 (tiles_beyond's bound against the larger distance;
// 1 % to spare on R).
__device__ __forceinline__ bool energy_tiles_far(const og_pair_args& a, int a0i, int ci, int a0j, int cj, int lane,
                                                 double iRi, double iRj) {
    const double* o = a.pos + 3 * (size_t)a0i;
    LaneData di, dj;
    const double* p = a.pos + 3 * (size_t)(a0i + (lane < ci ? lane : 0));
    di.x = (float)(p[0] - o[0]); di.y = (float)(p[1] - o[1]); di.z = (float)(p[2] - o[2]);
    p = a.pos + 3 * (size_t)(a0j + (lane < cj ? lane : 0));
    dj.x = (float)(p[0] - o[0]); dj.y = (float)(p[1] - o[1]); dj.z = (float)(p[2] - o[2]);
    const float g = -wave_max_f(-(float)iRi) * -wave_max_f(-(float)iRj);     // smallest 1 / (R_i R_j)
    const float rc2 = fmaxf(a.rc2_nb, 245.0f / g);
    return g > 0.0f && tiles_beyond(tile_radius(di, ci, lane, 0.0f, 0.0f, 0.0f), dj, cj, lane, rc2);
}

}  // namespace
