// All-pairs kernels for short work lists: a block of 8 waves per work item.
//
// With one wave per item (pair_kernels.hip) a force evaluation of one chain or
// a few is bound by that wave's chain of steps, not by the chip: a strip of
// four j tiles is 512 pair steps in a row, 35-55 us, while 4 to 400 waves run
// on 1 024 SIMDs.  Here the pair terms of an item, which do not depend on one
// another, are spread over the block's waves (8 of the 64 steps each) and left
// in LDS; then one wave per force component adds them up in the order in
// which the one-wave form does.  Pair terms and sums keep their products and
// their order, so both forms give the same bits.
//
// The Born radii are formed where the force pass loads its atoms, so that the
// force evaluation is two dependent launches instead of three:
//   og_k_wide_descreen  descreening items | bonded terms
//   og_k_wide_energy    energies only: tile pairs | radii, GB self | gather
//   og_k_wide_force     strips, force items | radii (stored for the readers
//                       after this pass) | bonded gather and next step's noise
#include "og_device.h"
#include "og_kernels.h"
#include "bonded_core.h"
#include "md_core.h"
#include "pair_core.h"

#define OG_WIDE_THREADS 512
#define OG_WIDE_WAVES (OG_WIDE_THREADS / 64)
#define OG_WIDE_GROUP 4                // j tiles of a strip held in LDS at a time

namespace {

// ---------------------------------------------------------------------------
// Descreening
// ---------------------------------------------------------------------------
// a tile pair's form: as it stands, the far-field one, beyond the cutoff
enum { WK_NEAR = 0, WK_FAR, WK_NONE };
struct WideDescreen {
    float4 pq[2 * (OG_TILE + 1)];      // j atoms as in descreen_tile_lds: P, then Q
    float h[2][OG_TILE][OG_TILE];      // [i side, j side][step][lane]
    int kind;                          // WK_*
};

// Steps [KB, KE) of the tile pair in the wave's lanes: step k pairs lane l with
// j atom (l + k) mod 64.  A diagonal tile runs steps 1..32, step 32 on lanes
// 0..31.
template <bool MODEA, bool DIAG, int KB, int KE>
__device__ __forceinline__ void wide_descreen_near(WideDescreen& L, const og_pair_args& a, const LaneData& di,
                                                   int lane, int wave, float& sum) {
    const float4* P = L.pq;
    const float4* Q = L.pq + (OG_TILE + 1);
    constexpr int N = (KE - KB) / OG_WIDE_WAVES;
    const float Si2 = di.gb.y * di.gb.y;
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const int k = KB + wave * N + u;
        const float4 pj = P[(lane + k) & 63], qj = Q[(lane + k) & 63];
        const float dx = pj.x - di.x, dy = pj.y - di.y, dz = pj.z - di.z;
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
        const float inv_r = __builtin_amdgcn_rsqf(r2);
        const float hij = descreen_h(r2, inv_r, di.gb.x, qj.x, qj.y);
        const float hji = descreen_h(r2, inv_r, pj.w, di.gb.y, Si2);
        bool ok = r2 >= 1e-18f;
        if (MODEA) ok = ok && (r2 <= a.rc2_ds);
        if (DIAG) ok = ok && (k < 32 || lane < 32);
        L.h[0][k - KB][lane] = ok ? hij : 0.0f;
        L.h[1][k - KB][lane] = ok ? hji : 0.0f;
    }
    __syncthreads();
    sum = 0.0f;
    if (wave == 0) {
#pragma unroll 16
        for (int k = KB; k < KE; ++k) sum += L.h[0][k - KB][lane];
    } else if (wave == 1) {            // lane = j atom: its partner at step k is lane - k
#pragma unroll 16
        for (int k = KB; k < KE; ++k) sum += L.h[1][k - KB][(lane - k) & 63];
    }
}

template <bool MODEA>
__device__ __forceinline__ void wide_descreen_item(WideDescreen& L, const og_pair_args& a, const og_work& it,
                                                   int lane, int wave) {
    const int a0i = a.tile_atom0[it.ti], ci = a.tile_cnt[it.ti];
    const int a0j = a.tile_atom0[it.tj], cj = a.tile_cnt[it.tj];
    const double ox = a.pos[3 * (size_t)a0i], oy = a.pos[3 * (size_t)a0i + 1], oz = a.pos[3 * (size_t)a0i + 2];
    const LaneData di = load_lane(a, it.ti, a0i, ci, lane, ox, oy, oz);
    float4* P = L.pq;
    float4* Q = L.pq + (OG_TILE + 1);
    if (wave == 0) {
        const LaneData dj = it.ti == it.tj ? di : load_lane(a, it.tj, a0j, cj, lane, ox, oy, oz);
        const float4 pj = make_float4(dj.x, dj.y, dj.z, dj.gb.x);
        const float4 qj = make_float4(dj.gb.y, dj.gb.y * dj.gb.y, (-1.0f / 3.0f) * (dj.gb.y * dj.gb.y) * dj.gb.y,
                                      0.0f);
        P[lane] = pj;
        Q[lane] = qj;
        if (lane == 0) { P[OG_TILE] = pj; Q[OG_TILE] = qj; }
        const bool far = it.ti != it.tj && descreen_far(a, di, dj, ci, cj, lane);
        const bool none = MODEA && it.ti != it.tj && it.part < 0 &&
                          tiles_beyond(tile_radius(di, ci, lane, 0.0f, 0.0f, 0.0f), dj, cj, lane, a.rc2_ds);
        if (lane == 0) L.kind = none ? WK_NONE : far ? WK_FAR : WK_NEAR;
    }
    __syncthreads();
    int* fl = a.sflag ? a.sflag + it.sys : nullptr;
    if (MODEA && L.kind == WK_NONE) return;
    if (L.kind == WK_FAR) {                  // the series is short: one wave runs it whole
        if (wave != 0) return;
        float acc_i = 0.0f, acc_j = 0.0f;
        if (it.part < 0) descreen_tile_far<MODEA, -1>(a, di, P, Q, lane, acc_i, acc_j);
        else if (it.part == 0) descreen_tile_far<MODEA, 0>(a, di, P, Q, lane, acc_i, acc_j);
        else descreen_tile_far<MODEA, 1>(a, di, P, Q, lane, acc_i, acc_j);
        if (lane < ci) og_atomic_add_fix(a.iacc + a0i + lane, og_to_fix_chk((double)acc_i, fl));
        if (lane < cj) og_atomic_add_fix(a.iacc + a0j + lane, og_to_fix_chk((double)acc_j, fl));
        return;
    }
    float sum;
    if (it.ti == it.tj) wide_descreen_near<MODEA, true, 1, 33>(L, a, di, lane, wave, sum);
    else if (it.part < 0) wide_descreen_near<MODEA, false, 0, 64>(L, a, di, lane, wave, sum);
    else if (it.part == 0) wide_descreen_near<MODEA, false, 0, 32>(L, a, di, lane, wave, sum);
    else wide_descreen_near<MODEA, false, 32, 64>(L, a, di, lane, wave, sum);
    if (wave == 0 && lane < ci) og_atomic_add_fix(a.iacc + a0i + lane, og_to_fix_chk((double)sum, fl));
    if (wave == 1 && lane < cj) og_atomic_add_fix(a.iacc + a0j + lane, og_to_fix_chk((double)sum, fl));
}

// ---------------------------------------------------------------------------
// Force
// ---------------------------------------------------------------------------
// x, y, z, q, sqrt(eps), Rmin/2, R, gw of the j atoms of a group of tiles
enum { WJ_X = 0, WJ_Y, WJ_Z, WJ_Q, WJ_SE, WJ_RM, WJ_R, WJ_GW, WJ_N };
struct WideForce {
    float j[OG_WIDE_GROUP][WJ_N][OG_TILE];
    float i[2][3][OG_TILE];            // positions of the (two) i tiles
    float j14[2][OG_TILE];             // 1-4 parameters (items)
    int kind[OG_STRIP_J];              // per j tile: WK_*
    float c[2][2][OG_TILE][OG_TILE];   // [buffer][i tile][step][lane] pair coefficients
};

// The position of a tile's atom relative to the origin (as load_lane).
__device__ __forceinline__ void wide_pos(LaneData& d, const og_pair_args& a, int atom0, int cnt, int lane, double ox,
                                         double oy, double oz) {
    if (lane < cnt) {
        const double* p = a.pos + 3 * (size_t)(atom0 + lane);
        d.x = (float)(p[0] - ox);
        d.y = (float)(p[1] - oy);
        d.z = (float)(p[2] - oz);
    } else {
        d.x = 1.0e6f + 97.0f * (float)lane;
        d.y = 1.0e6f;
        d.z = 1.0e6f;
    }
}

// The rest of load_lane, the Born radius formed from the descreening integral
// (padding slots keep R = gw = 1, as the engine lays them out).
__device__ __forceinline__ void wide_fill(LaneData& d, const og_pair_args& a, const double* rho, int tile, int atom0,
                                          int cnt, int lane) {
    const int slot = tile * OG_TILE + lane;
    float R = 1.0f, gw = 1.0f;
    if (lane < cnt) {
        bool clamped;
        const double Rd = born_radius((double)a.iacc[atom0 + lane] * OG_FIX_INV, rho[atom0 + lane], clamped);
        R = (float)Rd;
        gw = (float)(kGbWidth / Rd);
    }
    d.q = a.qs[slot];
    d.par = a.par[slot];
    d.gb = make_float4(0.0f, 0.0f, R, gw);
}

__device__ __forceinline__ LaneData wide_lane(const og_pair_args& a, const double* rho, int tile, int atom0, int cnt,
                                              int lane, double ox, double oy, double oz) {
    LaneData d;
    wide_pos(d, a, atom0, cnt, lane, ox, oy, oz);
    wide_fill(d, a, rho, tile, atom0, cnt, lane);
    return d;
}

__device__ __forceinline__ void wide_store_j(WideForce& L, int g, const LaneData& d, int lane) {
    float(*J)[OG_TILE] = L.j[g];
    J[WJ_X][lane] = d.x; J[WJ_Y][lane] = d.y; J[WJ_Z][lane] = d.z; J[WJ_Q][lane] = d.q;
    J[WJ_SE][lane] = d.par.x; J[WJ_RM][lane] = d.par.y; J[WJ_R][lane] = d.gb.z; J[WJ_GW][lane] = d.gb.w;
}

__device__ __forceinline__ void wide_store_i(WideForce& L, int h, const LaneData& d, int lane) {
    L.i[h][0][lane] = d.x; L.i[h][1][lane] = d.y; L.i[h][2][lane] = d.z;
}

// Coefficients of steps [KB, KE) of a tile pair, 1/8 of them per wave.
template <bool MODEA, bool MASKED, bool DIAG, int KB, int KE>
__device__ __forceinline__ void wide_item_coefs(WideForce& L, const og_pair_args& a, const LaneData& di, int lane,
                                                int wave, unsigned long long xm, unsigned long long m14) {
    constexpr int N = (KE - KB) / OG_WIDE_WAVES;
    const float(*J)[OG_TILE] = L.j[0];
    const float qki = kGbK * di.q;
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const int k = KB + wave * N + u, e = (lane + k) & 63;
        const float dx = J[WJ_X][e] - di.x, dy = J[WJ_Y][e] - di.y, dz = J[WJ_Z][e] - di.z;
        const bool excl = MASKED && ((xm >> e) & 1ull), one4 = MASKED && ((m14 >> e) & 1ull);
        float c = tile_coef<MODEA, MASKED>(a, di, qki, J[WJ_Q][e], J[WJ_SE][e], J[WJ_RM][e], MASKED ? L.j14[0][e] : 0.0f,
                                           MASKED ? L.j14[1][e] : 0.0f, J[WJ_R][e], J[WJ_GW][e], excl, one4, dx, dy, dz);
        if (DIAG) c = (k < 32 || lane < 32) ? c : 0.0f;
        L.c[0][0][k][lane] = c;
    }
}

// One component's sum over the steps: the i side (wave 0-2, lane = i atom) or
// the j side (wave 3-5, lane = j atom, whose partner at step k is lane - k).
template <int KB, int KE>
__device__ __forceinline__ float wide_item_sum(const WideForce& L, int lane, int wave) {
    float f = 0.0f;
    if (wave < 3) {
        const float* xj = L.j[0][wave];
        const float xi = L.i[0][wave][lane];
#pragma unroll 16
        for (int k = KB; k < KE; ++k) f = fmaf(L.c[0][0][k][lane], xj[(lane + k) & 63] - xi, f);
    } else {
        const float xj = L.j[0][wave - 3][lane];
        const float* xi = L.i[0][wave - 3];
#pragma unroll 16
        for (int k = KB; k < KE; ++k) {
            const int l = (lane - k) & 63;
            f = fmaf(-L.c[0][0][k][l], xj - xi[l], f);
        }
    }
    return f;
}

template <bool MODEA>
__device__ __forceinline__ void wide_force_item(WideForce& L, const og_pair_args& a, const double* rho,
                                                const og_work& it, int lane, int wave) {
    const int a0i = a.tile_atom0[it.ti], ci = a.tile_cnt[it.ti];
    const int a0j = a.tile_atom0[it.tj], cj = a.tile_cnt[it.tj];
    const double ox = a.pos[3 * (size_t)a0i], oy = a.pos[3 * (size_t)a0i + 1], oz = a.pos[3 * (size_t)a0i + 2];
    LaneData di, dj;
    wide_pos(di, a, a0i, ci, lane, ox, oy, oz);
    const bool diag = it.ti == it.tj;
    // half tile pairs (systems of up to four tiles) are short and mostly within
    // the cutoff: the test would cost them more than it saves
    if (MODEA && !diag && it.part < 0) {
        // every wave decides for itself, so that they agree without a barrier
        wide_pos(dj, a, a0j, cj, lane, ox, oy, oz);
        if (tiles_beyond(tile_radius(di, ci, lane, 0.0f, 0.0f, 0.0f), dj, cj, lane, force_cutoff2(a))) return;
    }
    wide_fill(di, a, rho, it.ti, a0i, ci, lane);
    unsigned long long xm = 0, m14 = 0;
    if (it.mask >= 0) {
        xm = a.masks[(size_t)it.mask * 128 + lane];
        m14 = a.masks[(size_t)it.mask * 128 + 64 + lane];
    }
    if (wave == 0) {
        dj = diag ? di : wide_lane(a, rho, it.tj, a0j, cj, lane, ox, oy, oz);
        wide_store_j(L, 0, dj, lane);
        L.j14[0][lane] = dj.par.z;
        L.j14[1][lane] = dj.par.w;
    } else if (wave == 1) {
        wide_store_i(L, 0, di, lane);
    }
    __syncthreads();
    float f = 0.0f;
    if (diag) {                        // its own tile holds excluded pairs or none: masks of zero select nothing
        wide_item_coefs<MODEA, true, true, 1, 33>(L, a, di, lane, wave, xm, m14);
        __syncthreads();
        if (wave < 6) f = wide_item_sum<1, 33>(L, lane, wave);
    } else if (it.part < 0) {
        if (it.mask >= 0) wide_item_coefs<MODEA, true, false, 0, 64>(L, a, di, lane, wave, xm, m14);
        else wide_item_coefs<MODEA, false, false, 0, 64>(L, a, di, lane, wave, xm, m14);
        __syncthreads();
        if (wave < 6) f = wide_item_sum<0, 64>(L, lane, wave);
    } else if (it.part == 0) {
        if (it.mask >= 0) wide_item_coefs<MODEA, true, false, 0, 32>(L, a, di, lane, wave, xm, m14);
        else wide_item_coefs<MODEA, false, false, 0, 32>(L, a, di, lane, wave, xm, m14);
        __syncthreads();
        if (wave < 6) f = wide_item_sum<0, 32>(L, lane, wave);
    } else {
        if (it.mask >= 0) wide_item_coefs<MODEA, true, false, 32, 64>(L, a, di, lane, wave, xm, m14);
        else wide_item_coefs<MODEA, false, false, 32, 64>(L, a, di, lane, wave, xm, m14);
        __syncthreads();
        if (wave < 6) f = wide_item_sum<32, 64>(L, lane, wave);
    }
    int* fl = a.sflag ? a.sflag + it.sys : nullptr;
    if (wave < 3) {
        if (lane < ci) og_atomic_add_fix(a.facc + 3 * (size_t)(a0i + lane) + wave, og_to_fix_chk((double)f, fl));
    } else if (wave < 6) {
        if (lane < cj) og_atomic_add_fix(a.facc + 3 * (size_t)(a0j + lane) + (wave - 3), og_to_fix_chk((double)f, fl));
    }
}

// What a block does with a strip (force_strip of pair_kernels.hip).
//   WS_BOTH   everything; two coefficient buffers, one barrier per j tile: the
//             waves that sum tile q's coefficients do so while the others form
//             tile q + 1's
//   WS_I + h  i tile h's sums only: its coefficients with every j tile of a
//             group, then 64 steps per j tile in a row on one wave a component
//   WS_J + q  j tile q's sums only
// The split forms evaluate each pair twice but take a strip over 2 + nj CUs.
enum { WS_BOTH = 0, WS_I = 1, WS_J = 3 };

// i-side sum of component `wave`, continued over 64 steps; the j position
// comes around the wave by rotation as in force_tile.
__device__ __forceinline__ void wide_sum_i(const float (*c)[OG_TILE], const float* xj, float xi, int lane, float& f) {
    float x = xj[lane];
#pragma unroll 16
    for (int k = 0; k < OG_TILE; ++k) {
        f = fmaf(c[k][lane], x - xi, f);
        x = rot(x);
    }
}

// j-side sum of one component: lane = j atom, whose partners at step k are
// lane - k of both i tiles, the first tile's added first.
__device__ __forceinline__ float wide_sum_j(const float (*ca)[OG_TILE], const float (*cb)[OG_TILE], float x,
                                            const float* xa, const float* xb, int lane) {
    float g = 0.0f;
#pragma unroll 16
    for (int k = 0; k < OG_TILE; ++k) {
        const int l = (lane - k) & 63;
        g = fmaf(-cb[k][l], x - xb[l], fmaf(-ca[k][l], x - xa[l], g));
    }
    return g;
}

template <bool MODEA>
__device__ __forceinline__ void wide_force_strip(WideForce& L, const og_pair_args& a, const double* rho,
                                                 const og_strip* sp, int role, int lane, int wave) {
    const int ta = __builtin_amdgcn_readfirstlane(sp->ti), tb = ta + 1;
    int nj = __builtin_amdgcn_readfirstlane(sp->nj), j0 = 0;
    if (role >= WS_J) {
        j0 = role - WS_J;
        if (j0 >= nj) return;
        nj = j0 + 1;
    }
    const int a0 = a.tile_atom0[ta], b0 = a.tile_atom0[tb];
    const int ca = a.tile_cnt[ta], cb = a.tile_cnt[tb];
    const double ox = a.pos[3 * (size_t)a0], oy = a.pos[3 * (size_t)a0 + 1], oz = a.pos[3 * (size_t)a0 + 2];
    LaneData da, db;
    wide_pos(da, a, a0, ca, lane, ox, oy, oz);
    wide_pos(db, a, b0, cb, lane, ox, oy, oz);
    if (MODEA) {
        // the j tiles beyond the cutoff, before anything else is formed
        const float rad = fmaxf(tile_radius(da, ca, lane, 0.0f, 0.0f, 0.0f), tile_radius(db, cb, lane, 0.0f, 0.0f, 0.0f));
        const int q = j0 + wave;
        if (q < nj) {
            const int tj = __builtin_amdgcn_readfirstlane(sp->tj[q]);
            const int cj = a.tile_cnt[tj];
            LaneData dj;
            wide_pos(dj, a, a.tile_atom0[tj], cj, lane, ox, oy, oz);
            const bool none = tiles_beyond(rad, dj, cj, lane, force_cutoff2(a));
            if (lane == 0) L.kind[q] = none ? WK_NONE : WK_NEAR;
        }
        __syncthreads();
        bool any = false;
        for (int k = j0; k < nj; ++k) any = any || L.kind[k] != WK_NONE;
        if (!any) return;
    }
    wide_fill(da, a, rho, ta, a0, ca, lane);
    wide_fill(db, a, rho, tb, b0, cb, lane);
    const StripAtom A = strip_atom(da), B = strip_atom(db);
    const StripBound bi = strip_bound(A, B);
    if (wave == 4) wide_store_i(L, 0, da, lane);
    if (wave == 5) wide_store_i(L, 1, db, lane);
    int* fl = a.sflag ? a.sflag + sp->sys : nullptr;
    float fa = 0.0f, fb = 0.0f;        // waves 0-2: this component's i-side sums
    // coefficients of i atom I and j tile q into c, 1/8 of the steps per wave
    auto coefs = [&](const StripAtom& I, int q, float (*c)[OG_TILE], auto far_tag) {
        constexpr bool F = decltype(far_tag)::value;
        constexpr int N = OG_TILE / OG_WIDE_WAVES;
        const float(*J)[OG_TILE] = L.j[q];
#pragma unroll 4
        for (int u = 0; u < N; ++u) {
            const int k = wave * N + u, e = (lane + k) & 63;
            const float4 pj = make_float4(J[WJ_X][e], J[WJ_Y][e], J[WJ_Z][e], J[WJ_Q][e]);
            const float4 qj = make_float4(J[WJ_SE][e], J[WJ_RM][e], J[WJ_R][e], J[WJ_GW][e]);
            c[k][lane] = strip_coef<MODEA, F>(a, I, pj, qj, pj.x - I.x, pj.y - I.y, pj.z - I.z);
        }
    };
    auto flush_j = [&](int tj, int d, float g) {
        if (lane < a.tile_cnt[tj])
            og_atomic_add_fix(a.facc + 3 * (size_t)(a.tile_atom0[tj] + lane) + d, og_to_fix_chk((double)g, fl));
    };
    int buf = 0;
    for (int g0 = j0; g0 < nj; g0 += OG_WIDE_GROUP) {
        if (wave < OG_WIDE_GROUP && g0 + wave < nj && !(MODEA && L.kind[g0 + wave] == WK_NONE)) {
            const int tj = __builtin_amdgcn_readfirstlane(sp->tj[g0 + wave]);
            const int cj = a.tile_cnt[tj];
            const LaneData dj = wide_lane(a, rho, tj, a.tile_atom0[tj], cj, lane, ox, oy, oz);
            wide_store_j(L, wave, dj, lane);
            const bool far = strip_far(bi, dj, cj, lane);
            if (lane == 0) L.kind[g0 + wave] = far ? WK_FAR : WK_NEAR;
        }
        __syncthreads();
        const int ng = nj - g0 < OG_WIDE_GROUP ? nj - g0 : OG_WIDE_GROUP;
        if (role == WS_I || role == WS_I + 1) {
            const StripAtom& I = role == WS_I ? A : B;
            float(*c)[OG_TILE] = &L.c[0][0][0];
            for (int q = 0; q < ng; ++q) {
                if (MODEA && L.kind[g0 + q] == WK_NONE) continue;
                if (L.kind[g0 + q] == WK_FAR) coefs(I, q, c + q * OG_TILE, std::true_type{});
                else coefs(I, q, c + q * OG_TILE, std::false_type{});
            }
            __syncthreads();
            if (wave < 3) {
                const float xi = L.i[role - WS_I][wave][lane];
                for (int q = 0; q < ng; ++q) {
                    if (MODEA && L.kind[g0 + q] == WK_NONE) continue;
                    wide_sum_i(c + q * OG_TILE, L.j[q][wave], xi, lane, fa);
                }
            }
        } else {
            for (int q = 0; q < ng; ++q) {
                if (MODEA && L.kind[g0 + q] == WK_NONE) continue;
                buf ^= 1;
                if (L.kind[g0 + q] == WK_FAR) {
                    coefs(A, q, L.c[buf][0], std::true_type{});
                    coefs(B, q, L.c[buf][1], std::true_type{});
                } else {
                    coefs(A, q, L.c[buf][0], std::false_type{});
                    coefs(B, q, L.c[buf][1], std::false_type{});
                }
                __syncthreads();
                if (wave < 3) {
                    if (role == WS_BOTH) {
                        wide_sum_i(L.c[buf][0], L.j[q][wave], L.i[0][wave][lane], lane, fa);
                        wide_sum_i(L.c[buf][1], L.j[q][wave], L.i[1][wave][lane], lane, fb);
                    }
                } else if (wave < 6) {
                    const int d = wave - 3;
                    const float g = wide_sum_j(L.c[buf][0], L.c[buf][1], L.j[q][d][lane], L.i[0][d], L.i[1][d], lane);
                    flush_j(__builtin_amdgcn_readfirstlane(sp->tj[g0 + q]), d, g);
                }
            }
        }
        if (g0 + OG_WIDE_GROUP < nj) __syncthreads();      // the group's sums are done with its j atoms
    }
    if (wave < 3 && role < WS_J) {
        if (role == WS_I + 1) {
            if (lane < cb) og_atomic_add_fix(a.facc + 3 * (size_t)(b0 + lane) + wave, og_to_fix_chk((double)fa, fl));
            return;
        }
        if (lane < ca) og_atomic_add_fix(a.facc + 3 * (size_t)(a0 + lane) + wave, og_to_fix_chk((double)fa, fl));
        if (role == WS_BOTH && lane < cb)
            og_atomic_add_fix(a.facc + 3 * (size_t)(b0 + lane) + wave, og_to_fix_chk((double)fb, fl));
    }
}

}  // namespace

// blocks [0, n_work): descreening items; the rest: bonded terms, whose
// registers (164, with energies 182) leave one block a CU
template <bool MODEA, bool ENERGY>
__global__ void __launch_bounds__(OG_WIDE_THREADS) og_k_wide_descreen(og_pair_args a, og_bonded_args b) {
    __shared__ WideDescreen L;
    if ((int)blockIdx.x < a.n_work) {
        const og_work it = a.work[blockIdx.x];
        if (ENERGY && a.skip_sys && a.skip_sys[it.sys]) return;
        wide_descreen_item<MODEA>(L, a, it, threadIdx.x & 63, threadIdx.x >> 6);
    } else {
        bonded_body<ENERGY>(b, blockIdx.x - a.n_work, gridDim.x - a.n_work);
    }
}

// blocks: strips (ns blocks each), force items, then nr blocks of radii, the
// rest the gather
// (four waves per SIMD, so that two blocks share a CU: left to itself the
// compiler spends up to 149 registers, with the noise code)
template <bool MODEA, bool NOISE>
__global__ void __launch_bounds__(OG_WIDE_THREADS) __attribute__((amdgpu_waves_per_eu(4)))
og_k_wide_force(og_pair_args a, og_radii_args r, og_bonded_args b, int ns, int nr) {
    __shared__ union {
        WideForce f;
        double t[3 * OG_GATHER_CHUNK];
    } L;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int k = blockIdx.x;
    if (k < a.n_strip * ns) {
        // the i-side blocks, the longer ones, come first
        const int sub = k / a.n_strip;
        wide_force_strip<MODEA>(L.f, a, r.rho, a.strips + (k - sub * a.n_strip), ns == 1 ? (int)WS_BOTH : WS_I + sub, lane,
                                wave);
        return;
    }
    k -= a.n_strip * ns;
    if (k < a.n_fwork) {
        const og_work it = a.fwork[k];
        wide_force_item<MODEA>(L.f, a, r.rho, it, lane, wave);
        return;
    }
    k -= a.n_fwork;
    if (k < nr) radii_body<false>(r, k * OG_WIDE_THREADS + threadIdx.x);
    else gather_lds_body<NOISE, OG_WIDE_THREADS>(b, k - nr, L.t);
}

// Energies only: blocks [0, n_work) tile pairs (a split pair whole, once), nr
// blocks of radii and GB self energies, the rest the gather (its sums are
// range-checked as in a force evaluation).  Each wave takes 8 of the 64 j
// atoms; one fixed-point value per tile pair and term, as in the one-wave form.
template <bool MODEA>
__global__ void __launch_bounds__(OG_WIDE_THREADS) og_k_wide_energy(og_pair_args a, og_energy64_args e, og_radii_args r,
                                                                    og_bonded_args b, int nr) {
    __shared__ union {
        struct {
            EJ j[OG_TILE];
            double part[OG_WIDE_WAVES][3];
            int far_pair;
        } e;
        double t[3 * OG_GATHER_CHUNK];
    } L;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int k = blockIdx.x;
    if (k >= a.n_work) {
        k -= a.n_work;
        if (k < nr) radii_body<true>(r, k * OG_WIDE_THREADS + threadIdx.x);
        else gather_lds_body<false, OG_WIDE_THREADS>(b, k - nr, L.t);
        return;
    }
    const og_work it = a.work[k];
    if (it.part == 1 || (a.skip_sys && a.skip_sys[it.sys])) return;
    const int a0i = a.tile_atom0[it.ti], ci = a.tile_cnt[it.ti];
    const int a0j = a.tile_atom0[it.tj], cj = a.tile_cnt[it.tj];
    const bool vi = lane < ci, diag = it.ti == it.tj, plain = !diag && it.mask < 0;
    const int gi = a0i + (vi ? lane : 0), gj = a0j + (lane < cj ? lane : 0);
    auto radius = [&](int g) {
        bool clamped;
        return born_radius((double)a.iacc[g] * OG_FIX_INV, r.rho[g], clamped);
    };
    const EI I = energy_i(a, e, gi, vi, radius(gi));
    unsigned long long xm = 0, m14 = 0;
    if (it.mask >= 0) {
        xm = a.masks[(size_t)it.mask * 128 + lane];
        m14 = a.masks[(size_t)it.mask * 128 + 64 + lane];
    }
    if (wave == 0) {
        const EJ mine = energy_j(a, e, gj, radius(gj));
        L.e.j[lane] = mine;
        const bool far = MODEA && plain && energy_tiles_far(a, a0i, ci, a0j, cj, lane, I.iR, mine.iR);
        if (lane == 0) L.e.far_pair = far;
    }
    __syncthreads();
    ESum t = {0.0, 0.0, 0.0};
    constexpr int N = OG_TILE / OG_WIDE_WAVES;
    const int j0 = wave * N, j1 = j0 + N < cj ? j0 + N : cj;
    if (MODEA && L.e.far_pair) energy_far(I, L.e.j, j0, j1, t);
    else if (plain) energy_plain<MODEA>(e, I, L.e.j, j0, j1, t);
    else energy_masked<MODEA>(e, I, L.e.j, j0, j1, lane, diag, xm, m14, t);
    t.lj = og_wave_sum_d(t.lj);
    t.c = og_wave_sum_d(t.c);
    t.g = og_wave_sum_d(t.g);
    if (lane == 0) {
        L.e.part[wave][0] = t.lj;
        L.e.part[wave][1] = t.c;
        L.e.part[wave][2] = t.g;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const double unit = threadIdx.x == 0   ? OG_KCAL_TO_KJ
                            : threadIdx.x == 1 ? OG_COULOMB_KCAL * OG_KCAL_TO_KJ
                                               : -(1.0 - 1.0 / OG_EPS_WATER) * OG_COULOMB_KCAL * OG_KCAL_TO_KJ;
        const int term = threadIdx.x == 0 ? OG_E_LJ : threadIdx.x == 1 ? OG_E_COUL : OG_E_GB_PAIR;
        double sum = 0.0;
        for (int w = 0; w < OG_WIDE_WAVES; ++w) sum += L.e.part[w][threadIdx.x];
        og_atomic_add_fix(a.eacc + (size_t)it.sys * OG_NE + term,
                          og_to_fix_chk(sum * unit, a.sflag ? a.sflag + it.sys : nullptr));
    }
}

void og_launch_wide_energy(const og_pair_args& a, const og_energy64_args& e, const og_radii_args& r,
                           const og_bonded_args& b, bool mode_a, hipStream_t s) {
    const int nr = (r.n_atoms + OG_WIDE_THREADS - 1) / OG_WIDE_THREADS;
    const int ng = (b.n_atoms + OG_GATHER_ATOMS - 1) / OG_GATHER_ATOMS;
    const dim3 g(a.n_work + nr + ng), t(OG_WIDE_THREADS);
    if (mode_a) hipLaunchKernelGGL(og_k_wide_energy<true>, g, t, 0, s, a, e, r, b, nr);
    else hipLaunchKernelGGL(og_k_wide_energy<false>, g, t, 0, s, a, e, r, b, nr);
}

void og_launch_wide_descreen(const og_pair_args& a, const og_bonded_args& b, bool mode_a, bool energy, hipStream_t s) {
    const int total = b.nb + b.na + b.nd + b.ni;
    const dim3 g(a.n_work + (total + OG_WIDE_THREADS - 1) / OG_WIDE_THREADS), t(OG_WIDE_THREADS);
    if (mode_a && energy) hipLaunchKernelGGL((og_k_wide_descreen<true, true>), g, t, 0, s, a, b);
    else if (mode_a) hipLaunchKernelGGL((og_k_wide_descreen<true, false>), g, t, 0, s, a, b);
    else if (energy) hipLaunchKernelGGL((og_k_wide_descreen<false, true>), g, t, 0, s, a, b);
    else hipLaunchKernelGGL((og_k_wide_descreen<false, false>), g, t, 0, s, a, b);
}

void og_launch_wide_force(const og_pair_args& a, const og_radii_args& r, const og_bonded_args& b, bool mode_a,
                          hipStream_t s) {
    const int nr = (r.n_atoms + OG_WIDE_THREADS - 1) / OG_WIDE_THREADS;
    const int ng = (b.n_atoms + OG_GATHER_ATOMS - 1) / OG_GATHER_ATOMS;
    const int ns = 2 * a.strip_j * a.n_strip <= OG_WIDE_SPLIT_MAX ? 2 + a.strip_j : 1;
    const dim3 g(a.n_strip * ns + a.n_fwork + nr + ng), t(OG_WIDE_THREADS);
    const bool noise = b.noise.noise != nullptr;
    if (mode_a && noise) hipLaunchKernelGGL((og_k_wide_force<true, true>), g, t, 0, s, a, r, b, ns, nr);
    else if (mode_a) hipLaunchKernelGGL((og_k_wide_force<true, false>), g, t, 0, s, a, r, b, ns, nr);
    else if (noise) hipLaunchKernelGGL((og_k_wide_force<false, true>), g, t, 0, s, a, r, b, ns, nr);
    else hipLaunchKernelGGL((og_k_wide_force<false, false>), g, t, 0, s, a, r, b, ns, nr);
}
