// All-pairs tile kernels: GB descreening integral and the fused
// LJ + Coulomb + GB-pair force (optionally with energies).
//
// Work decomposition: one wave64 per tile pair (I <= J) of one system,
// grid-stride over a flattened work list that covers every system of the
// batch.  Lane l owns i-atom I*64+l.  The j atoms travel around the wave:
// lane l starts with j-atom l and, after every pair step, each lane passes
// its j data and its running j-side reaction (Newton's third law) to the
// neighbouring lane with one DPP wave rotate (v_mov_dpp wave_rol:1), so in
// 64 steps every lane meets every j atom and the j-side sums arrive back
// home.  On off-diagonal tiles without exclusions (most of the work) the j
// data are read from the wave's LDS instead, entry (l + k) mod 64 at step k,
// which is exactly what the rotation would deliver, so only the three (one)
// j-side sums rotate.  A diagonal tile (I = J) runs steps 1..32 (step 32 on
// lanes 0..31) and swaps the halves of the wave at the end.  Per tile pair every lane
// flushes one FP32 partial per component into the int64 fixed-point
// accumulators.  The FP64 energy kernel reads its j atoms from LDS (every lane
// the same entry: a broadcast) and accumulates the pair energies per lane.
//
// Physics follows origami's SoA kernels:
//   descreening   energy/src/gb.rs:271-283 (pair), :347-369 (h)
//   LJ + Coulomb  energy/src/forces_nonbonded.rs:196-232
//   GB pair force energy/src/forces_gb.rs:72-112
//   energies      energy/src/nonbonded.rs:97-174, energy/src/gb.rs:146-182
// Mode B (all pairs) is the fast path; Mode A adds origami's integrator
// cutoffs (10 Å LJ + reaction-field Coulomb, 10 Å GB force, 20 Å descreen).
#include "og_device.h"
#include "og_kernels.h"
#include "bonded_core.h"
#include "md_core.h"
#include "pair_core.h"

namespace {

template <bool MODEA, bool DIAG>
__device__ __forceinline__ void descreen_tile(const og_pair_args& a, const LaneData& di,
                                              const LaneData& dj, int lane, float& acc_i, float& acc_j) {
    float xj = dj.x, yj = dj.y, zj = dj.z, rtj = dj.gb.x, Sj = dj.gb.y;
    float gj = 0.0f;
    const int k0 = DIAG ? 1 : 0, k1 = DIAG ? 32 : 63;
    if (DIAG) {
        xj = rot(xj); yj = rot(yj); zj = rot(zj); rtj = rot(rtj); Sj = rot(Sj);
    }
#pragma unroll 2
    for (int k = k0; k <= k1; ++k) {
        const float dx = xj - di.x, dy = yj - di.y, dz = zj - di.z;
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
        const float inv_r = __builtin_amdgcn_rsqf(r2);
        float hij = descreen_h(r2, inv_r, di.gb.x, Sj, Sj * Sj);
        float hji = descreen_h(r2, inv_r, rtj, di.gb.y, di.gb.y * di.gb.y);
        bool ok = r2 >= 1e-18f;
        if (MODEA) ok = ok && (r2 <= a.rc2_ds);
        if (DIAG) ok = ok && (k < 32 || lane < 32);
        acc_i += ok ? hij : 0.0f;
        gj += ok ? hji : 0.0f;
        if (k < k1) {
            xj = rot(xj); yj = rot(yj); zj = rot(zj); rtj = rot(rtj); Sj = rot(Sj);
            gj = rot(gj);
        }
    }
    // home: one more step around the wave (64 in all), or half a turn on a diagonal tile
    acc_j += DIAG ? swap32(gj) : rot(gj);
}

// Off-diagonal descreening tile with the j data in LDS: P[e] = (x, y, z, rho~)
// and Q[e] = (S, S^2, -, -) of j atom e, entries 0..63 plus entry 64 = entry
// 0, so that the pair of steps k, k + 1 reads entries idx and idx + 1 without
// a wrap (Q follows P in the same array: one address for all four reads).
// Same arithmetic, in the same order, as the rotating form.
// PART (og_work::part): -1 all 64 steps, 0 steps 0-31, 1 steps 32-63.  After
// steps 0-31 the j-side sums sit 32 lanes from home, hence the swap.
template <bool MODEA, int PART>
__device__ __forceinline__ void descreen_tile_lds(const og_pair_args& a, const LaneData& di,
                                                  const float4* P, const float4* Q, int lane,
                                                  float& acc_i, float& acc_j) {
    float gj = 0.0f;
    const float Si2 = di.gb.y * di.gb.y;
    auto step = [&](float4 pj, float4 qj) {
        const float dx = pj.x - di.x, dy = pj.y - di.y, dz = pj.z - di.z;
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
        const float inv_r = __builtin_amdgcn_rsqf(r2);
        const float hij = descreen_h(r2, inv_r, di.gb.x, qj.x, qj.y);
        const float hji = descreen_h(r2, inv_r, pj.w, di.gb.y, Si2);
        bool ok = r2 >= 1e-18f;
        if (MODEA) ok = ok && (r2 <= a.rc2_ds);
        acc_i += ok ? hij : 0.0f;
        gj += ok ? hji : 0.0f;
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

// One descreening work item (a tile pair, or half of one) of the wave; P, Q:
// the wave's LDS staging.
template <bool MODEA>
__device__ __forceinline__ void descreen_item(const og_pair_args& a, const og_work& it, int lane, float4* P,
                                              float4* Q) {
    {
        const int a0i = a.tile_atom0[it.ti], ci = a.tile_cnt[it.ti];
        const int a0j = a.tile_atom0[it.tj], cj = a.tile_cnt[it.tj];
        const double ox = a.pos[3 * (size_t)a0i], oy = a.pos[3 * (size_t)a0i + 1],
                     oz = a.pos[3 * (size_t)a0i + 2];
        const LaneData di = load_lane(a, it.ti, a0i, ci, lane, ox, oy, oz);
        float acc_i = 0.0f, acc_j = 0.0f;
        if (it.ti == it.tj) {
            descreen_tile<MODEA, true>(a, di, di, lane, acc_i, acc_j);
        } else {
            const LaneData dj = load_lane(a, it.tj, a0j, cj, lane, ox, oy, oz);
            if (MODEA && tiles_beyond(tile_radius(di, ci, lane, 0.0f, 0.0f, 0.0f), dj, cj, lane, a.rc2_ds)) return;
            const float4 pj = make_float4(dj.x, dj.y, dj.z, dj.gb.x);
            const float4 qj = make_float4(dj.gb.y, dj.gb.y * dj.gb.y, (-1.0f / 3.0f) * (dj.gb.y * dj.gb.y) * dj.gb.y,
                                          0.0f);
            wave_lds_order();                       // the previous tile's reads are done
            P[lane] = pj;
            Q[lane] = qj;
            if (lane == 0) { P[OG_TILE] = pj; Q[OG_TILE] = qj; }
            wave_lds_order();
            const bool far = descreen_far(a, di, dj, ci, cj, lane);
            if (far) {
                if (it.part < 0) descreen_tile_far<MODEA, -1>(a, di, P, Q, lane, acc_i, acc_j);
                else if (it.part == 0) descreen_tile_far<MODEA, 0>(a, di, P, Q, lane, acc_i, acc_j);
                else descreen_tile_far<MODEA, 1>(a, di, P, Q, lane, acc_i, acc_j);
            } else if (it.part < 0) descreen_tile_lds<MODEA, -1>(a, di, P, Q, lane, acc_i, acc_j);
            else if (it.part == 0) descreen_tile_lds<MODEA, 0>(a, di, P, Q, lane, acc_i, acc_j);
            else descreen_tile_lds<MODEA, 1>(a, di, P, Q, lane, acc_i, acc_j);
        }
        int* fl = a.sflag ? a.sflag + it.sys : nullptr;
        if (lane < ci) og_atomic_add_fix(a.iacc + a0i + lane, og_to_fix_chk((double)acc_i, fl));
        if (lane < cj) og_atomic_add_fix(a.iacc + a0j + lane, og_to_fix_chk((double)acc_j, fl));
    }
}

// blk / nblk: this block among the nblk blocks sharing the tile pairs.
template <bool MODEA>
__device__ __forceinline__ void descreen_body(const og_pair_args& a, int blk, int nblk) {
    __shared__ float4 s_pq[4][2 * (OG_TILE + 1)];       // per wave: P[65], then Q[65]
    float4* P = s_pq[threadIdx.x >> 6];
    float4* Q = P + (OG_TILE + 1);
    const int lane = threadIdx.x & 63;
    const int wave = (blk * blockDim.x + threadIdx.x) >> 6;
    const int n_waves = (nblk * blockDim.x) >> 6;
    for (int w = wave; w < a.n_work; w += n_waves) {
        const og_work it = a.work[w];
        if (a.skip_sys && a.skip_sys[it.sys]) continue;     // radii from the surrogate
        descreen_item<MODEA>(a, it, lane, P, Q);
    }
}

}  // namespace

__global__ void __launch_bounds__(256) og_k_descreen_b(og_pair_args a) {
    descreen_body<false>(a, blockIdx.x, gridDim.x);
}
__global__ void __launch_bounds__(256) og_k_descreen_a(og_pair_args a) {
    descreen_body<true>(a, blockIdx.x, gridDim.x);
}

// The descreening pass and the bonded terms (forces) in one launch, for small
// batches whose force evaluation is a chain of latency-bound launches: blocks
// [0, nd) take the tile pairs, the rest the bonded terms, side by side.
template <bool MODEA>
__global__ void __launch_bounds__(256) og_k_descreen_bonded(og_pair_args a, og_bonded_args b, int nd) {
    if ((int)blockIdx.x < nd) descreen_body<MODEA>(a, blockIdx.x, nd);
    else bonded_body<false>(b, blockIdx.x - nd, gridDim.x - nd);
}

namespace {

// ---------------------------------------------------------------------------
// Fused force tile.
// ---------------------------------------------------------------------------
struct ForceAcc {
    float fx, fy, fz;       // i-side
    float gx, gy, gz;       // j-side (lane j)
};

// PART (og_work::part, off-diagonal tiles): -1 all 64 steps, 0 steps 0-31,
// 1 steps 32-63 (the j data start half a turn round); after steps 0-31 the
// j-side sums sit 32 lanes from home, hence the swap.
template <bool MODEA, bool MASKED, bool DIAG, int PART>
__device__ __forceinline__ void force_tile(const og_pair_args& a, const LaneData& di,
                                           const LaneData& dj, int lane,
                                           unsigned long long xmask, unsigned long long m14,
                                           ForceAcc& acc) {
    float xj = dj.x, yj = dj.y, zj = dj.z, qj = dj.q;
    float sej = dj.par.x, rmj = dj.par.y, se14j = dj.par.z, rm14j = dj.par.w;
    float Rj = dj.gb.z, iRj = dj.gb.w;
    int jid = lane;                         // j index within tile J held by this lane
    float gx = 0.0f, gy = 0.0f, gz = 0.0f;
    const float qki = kGbK * di.q;
    constexpr int k0 = DIAG ? 1 : (PART == 1 ? 32 : 0), k1 = DIAG ? 32 : (PART == 0 ? 31 : 63);
    auto advance = [&]() {
        xj = rot(xj); yj = rot(yj); zj = rot(zj); qj = rot(qj);
        sej = rot(sej); rmj = rot(rmj); Rj = rot(Rj); iRj = rot(iRj);
        if (MASKED) { se14j = rot(se14j); rm14j = rot(rm14j); jid = roti(jid); }
    };
    if (DIAG) advance();
    if (!DIAG && PART == 1) {
        xj = swap32(xj); yj = swap32(yj); zj = swap32(zj); qj = swap32(qj);
        sej = swap32(sej); rmj = swap32(rmj); Rj = swap32(Rj); iRj = swap32(iRj);
        if (MASKED) { se14j = swap32(se14j); rm14j = swap32(rm14j); jid = lane ^ 32; }
    }
#pragma unroll 2
    for (int k = k0; k <= k1; ++k) {
        const float dx = xj - di.x, dy = yj - di.y, dz = zj - di.z;
        const bool excl = MASKED && ((xmask >> jid) & 1ull);
        const bool one4 = MASKED && ((m14 >> jid) & 1ull);
        float c = tile_coef<MODEA, MASKED>(a, di, qki, qj, sej, rmj, se14j, rm14j, Rj, iRj, excl, one4, dx, dy, dz);
        if (DIAG) c = (k < 32 || lane < 32) ? c : 0.0f;
        acc.fx = fmaf(c, dx, acc.fx);
        acc.fy = fmaf(c, dy, acc.fy);
        acc.fz = fmaf(c, dz, acc.fz);
        gx = fmaf(-c, dx, gx);
        gy = fmaf(-c, dy, gy);
        gz = fmaf(-c, dz, gz);
        if (k < k1) {
            advance();
            gx = rot(gx); gy = rot(gy); gz = rot(gz);
        }
    }
    // home: one more step around the wave (64 in all), or half a turn on a diagonal tile
    if (DIAG) {
        gx = swap32(gx); gy = swap32(gy); gz = swap32(gz);
    } else {
        gx = rot(gx); gy = rot(gy); gz = rot(gz);
        if (PART == 0) { gx = swap32(gx); gy = swap32(gy); gz = swap32(gz); }
    }
    acc.gx += gx;
    acc.gy += gy;
    acc.gz += gz;
}

// Off-diagonal force tile without exclusions, j data in LDS: P[e] = (x, y,
// z, q) and Q[e] = (se, rm, R, 1/R scaled) of j atom e, entries 0..63 plus
// entry 64 = entry 0 (steps k and k + 1 read entries idx and idx + 1; Q
// follows P in the same array).  The arithmetic is that of force_tile's
// unmasked path.
template <bool MODEA, int PART>
__device__ __forceinline__ void force_tile_lds(const og_pair_args& a, const LaneData& di,
                                               const float4* P, const float4* Q, int lane,
                                               ForceAcc& acc) {
    float gx = 0.0f, gy = 0.0f, gz = 0.0f;
    const float qki = kGbK * di.q;
    auto step = [&](float4 pj, float4 qj4) {
        const float dx = pj.x - di.x, dy = pj.y - di.y, dz = pj.z - di.z;
        const float c = tile_coef<MODEA, false>(a, di, qki, pj.w, qj4.x, qj4.y, 0.0f, 0.0f, qj4.z, qj4.w, false, false,
                                                dx, dy, dz);
        acc.fx = fmaf(c, dx, acc.fx);
        acc.fy = fmaf(c, dy, acc.fy);
        acc.fz = fmaf(c, dz, acc.fz);
        gx = rot(fmaf(-c, dx, gx));     // after step 63 this is the way home
        gy = rot(fmaf(-c, dy, gy));
        gz = rot(fmaf(-c, dz, gz));
    };
    constexpr int kb = PART == 1 ? 32 : 0, ke = PART == 0 ? 32 : 64;
    for (int k = kb; k < ke; k += 2) {
        const int idx = (lane + k) & 63;
        const float4 p0 = P[idx], p1 = P[idx + 1];
        const float4 q0 = Q[idx], q1 = Q[idx + 1];
        step(p0, q0);
        step(p1, q1);
    }
    if (PART == 0) { gx = swap32(gx); gy = swap32(gy); gz = swap32(gz); }
    acc.gx += gx;
    acc.gy += gy;
    acc.gz += gz;
}

// A strip: two i tiles (64 i atoms each, two per lane) against up to OG_STRIP_J j
// tiles of the same system, j data in the wave's LDS as in force_tile_lds.
// Each step evaluates the lane's two i atoms against one j atom, adds both
// reactions into the rotating j-side sums and rotates them once, so the
// rotation and the LDS read serve two pairs.  The i-side sums stay in
// registers over the whole strip and are flushed once.  No pair of a strip
// is excluded or 1-4, and no i atom is a padding slot (the i tiles precede a
// j tile of their system, so both are full); distinct atoms at one position
// give a non-finite coefficient, which the fixed-point conversion reports.
template <bool MODEA>
__device__ __forceinline__ void force_strip(const og_pair_args& a, const og_strip* sp, int lane,
                                            float4* P, float4* Q) {
    // fields read through the pointer (the j tile list is indexed at run
    // time, which a local copy would keep in scratch memory)
    const int ta = __builtin_amdgcn_readfirstlane(sp->ti), tb = ta + 1;
    const int nj = __builtin_amdgcn_readfirstlane(sp->nj);
    const int a0 = a.tile_atom0[ta], b0 = a.tile_atom0[tb];
    const int ca = a.tile_cnt[ta], cb = a.tile_cnt[tb];
    const double ox = a.pos[3 * (size_t)a0], oy = a.pos[3 * (size_t)a0 + 1], oz = a.pos[3 * (size_t)a0 + 2];
    StripAtom A = strip_atom(load_lane(a, ta, a0, ca, lane, ox, oy, oz));
    StripAtom B = strip_atom(load_lane(a, tb, b0, cb, lane, ox, oy, oz));
    int* fl = a.sflag ? a.sflag + sp->sys : nullptr;
    const StripBound bi = strip_bound(A, B);
    int tj = __builtin_amdgcn_readfirstlane(sp->tj[0]);
    LaneData dj = load_lane(a, tj, a.tile_atom0[tj], a.tile_cnt[tj], lane, ox, oy, oz);
    for (int q = 0; q < nj; ++q) {
        const int a0j = a.tile_atom0[tj], cj = a.tile_cnt[tj];
        const float4 pjl = make_float4(dj.x, dj.y, dj.z, dj.q);
        const float4 qjl = make_float4(dj.par.x, dj.par.y, dj.gb.z, dj.gb.w);
        wave_lds_order();                       // the previous j tile's reads are done
        P[lane] = pjl;
        Q[lane] = qjl;
        if (lane == 0) { P[OG_TILE] = pjl; Q[OG_TILE] = qjl; }
        wave_lds_order();
        const bool far = strip_far(bi, dj, cj, lane);
        const bool none = MODEA && tiles_beyond(bi.rad, dj, cj, lane, force_cutoff2(a));
        // the next j tile's data load while this one is evaluated
        const int tn = __builtin_amdgcn_readfirstlane(sp->tj[q + 1 < nj ? q + 1 : q]);
        dj = load_lane(a, tn, a.tile_atom0[tn], a.tile_cnt[tn], lane, ox, oy, oz);
        if (none) {
            tj = tn;
            continue;
        }
        float gx = 0.0f, gy = 0.0f, gz = 0.0f;
        auto step = [&](float4 pj, float4 qj, auto far_tag) {
            constexpr bool F = decltype(far_tag)::value;
            const float dxa = pj.x - A.x, dya = pj.y - A.y, dza = pj.z - A.z;
            const float dxb = pj.x - B.x, dyb = pj.y - B.y, dzb = pj.z - B.z;
            const float c_a = strip_coef<MODEA, F>(a, A, pj, qj, dxa, dya, dza);
            const float c_b = strip_coef<MODEA, F>(a, B, pj, qj, dxb, dyb, dzb);
            A.fx = fmaf(c_a, dxa, A.fx);
            A.fy = fmaf(c_a, dya, A.fy);
            A.fz = fmaf(c_a, dza, A.fz);
            B.fx = fmaf(c_b, dxb, B.fx);
            B.fy = fmaf(c_b, dyb, B.fy);
            B.fz = fmaf(c_b, dzb, B.fz);
            gx = rot(fmaf(-c_b, dxb, fmaf(-c_a, dxa, gx)));     // after step 63: home
            gy = rot(fmaf(-c_b, dyb, fmaf(-c_a, dya, gy)));
            gz = rot(fmaf(-c_b, dzb, fmaf(-c_a, dza, gz)));
        };
        if (far) {
            for (int k = 0; k < OG_TILE; k += 2) {
                const int idx = (lane + k) & 63;
                const float4 p0 = P[idx], q0 = Q[idx];
                const float4 p1 = P[idx + 1], q1 = Q[idx + 1];
                step(p0, q0, std::true_type{});
                step(p1, q1, std::true_type{});
            }
        } else {
            for (int k = 0; k < OG_TILE; k += 2) {
                const int idx = (lane + k) & 63;
                const float4 p0 = P[idx], q0 = Q[idx];
                const float4 p1 = P[idx + 1], q1 = Q[idx + 1];
                step(p0, q0, std::false_type{});
                step(p1, q1, std::false_type{});
            }
        }
        if (lane < cj) {
            long long* f = a.facc + 3 * (size_t)(a0j + lane);
            og_atomic_add_fix(f + 0, og_to_fix_chk((double)gx, fl));
            og_atomic_add_fix(f + 1, og_to_fix_chk((double)gy, fl));
            og_atomic_add_fix(f + 2, og_to_fix_chk((double)gz, fl));
        }
        tj = tn;
    }
    if (lane < ca) {
        long long* f = a.facc + 3 * (size_t)(a0 + lane);
        og_atomic_add_fix(f + 0, og_to_fix_chk((double)A.fx, fl));
        og_atomic_add_fix(f + 1, og_to_fix_chk((double)A.fy, fl));
        og_atomic_add_fix(f + 2, og_to_fix_chk((double)A.fz, fl));
    }
    if (lane < cb) {
        long long* f = a.facc + 3 * (size_t)(b0 + lane);
        og_atomic_add_fix(f + 0, og_to_fix_chk((double)B.fx, fl));
        og_atomic_add_fix(f + 1, og_to_fix_chk((double)B.fy, fl));
        og_atomic_add_fix(f + 2, og_to_fix_chk((double)B.fz, fl));
    }
}

// One force work item outside the strips (a diagonal, adjacent or masked
// tile pair, or a tile pair of a small system).
template <bool MODEA>
__device__ __forceinline__ void force_item(const og_pair_args& a, const og_work& it, int lane, float4* P,
                                           float4* Q) {
    {
        const int a0i = a.tile_atom0[it.ti], ci = a.tile_cnt[it.ti];
        const int a0j = a.tile_atom0[it.tj], cj = a.tile_cnt[it.tj];
        const double ox = a.pos[3 * (size_t)a0i], oy = a.pos[3 * (size_t)a0i + 1],
                     oz = a.pos[3 * (size_t)a0i + 2];
        const LaneData di = load_lane(a, it.ti, a0i, ci, lane, ox, oy, oz);
        ForceAcc acc = {0, 0, 0, 0, 0, 0};
        unsigned long long xm = 0, m14 = 0;
        if (it.mask >= 0) {
            xm = a.masks[(size_t)it.mask * 128 + lane];
            m14 = a.masks[(size_t)it.mask * 128 + 64 + lane];
        }
        if (it.ti == it.tj) {
            force_tile<MODEA, true, true, -1>(a, di, di, lane, xm, m14, acc);
        } else {
            const LaneData dj = load_lane(a, it.tj, a0j, cj, lane, ox, oy, oz);
            if (MODEA && tiles_beyond(tile_radius(di, ci, lane, 0.0f, 0.0f, 0.0f), dj, cj, lane, force_cutoff2(a)))
                return;
            if (it.mask >= 0) {
                if (it.part < 0) force_tile<MODEA, true, false, -1>(a, di, dj, lane, xm, m14, acc);
                else if (it.part == 0) force_tile<MODEA, true, false, 0>(a, di, dj, lane, xm, m14, acc);
                else force_tile<MODEA, true, false, 1>(a, di, dj, lane, xm, m14, acc);
            } else {
                const float4 pj = make_float4(dj.x, dj.y, dj.z, dj.q);
                const float4 qj = make_float4(dj.par.x, dj.par.y, dj.gb.z, dj.gb.w);
                wave_lds_order();                   // the previous tile's reads are done
                P[lane] = pj;
                Q[lane] = qj;
                if (lane == 0) { P[OG_TILE] = pj; Q[OG_TILE] = qj; }
                wave_lds_order();
                if (it.part < 0) force_tile_lds<MODEA, -1>(a, di, P, Q, lane, acc);
                else if (it.part == 0) force_tile_lds<MODEA, 0>(a, di, P, Q, lane, acc);
                else force_tile_lds<MODEA, 1>(a, di, P, Q, lane, acc);
            }
        }
        int* fl = a.sflag ? a.sflag + it.sys : nullptr;
        if (lane < ci) {
            long long* f = a.facc + 3 * (size_t)(a0i + lane);
            og_atomic_add_fix(f + 0, og_to_fix_chk((double)acc.fx, fl));
            og_atomic_add_fix(f + 1, og_to_fix_chk((double)acc.fy, fl));
            og_atomic_add_fix(f + 2, og_to_fix_chk((double)acc.fz, fl));
        }
        if (lane < cj) {
            long long* f = a.facc + 3 * (size_t)(a0j + lane);
            og_atomic_add_fix(f + 0, og_to_fix_chk((double)acc.gx, fl));
            og_atomic_add_fix(f + 1, og_to_fix_chk((double)acc.gy, fl));
            og_atomic_add_fix(f + 2, og_to_fix_chk((double)acc.gz, fl));
        }
    }
}

// The force pass: the strips first (the heavier items), then the remaining
// tile pairs (fwork), grid-stride over both.
template <bool MODEA>
__device__ __forceinline__ void force_body(const og_pair_args& a) {
    __shared__ float4 s_pq[4][2 * (OG_TILE + 1)];       // per wave: P[65], then Q[65]
    float4* P = s_pq[threadIdx.x >> 6];
    float4* Q = P + (OG_TILE + 1);
    const int lane = threadIdx.x & 63;
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int n_waves = (gridDim.x * blockDim.x) >> 6;
    const int total = a.n_strip + a.n_fwork;
    for (int w = wave; w < total; w += n_waves) {
        if (w < a.n_strip) {
            force_strip<MODEA>(a, a.strips + w, lane, P, Q);
            continue;
        }
        const og_work it = a.fwork[w - a.n_strip];
        force_item<MODEA>(a, it, lane, P, Q);
    }
}

}  // namespace

__global__ void __launch_bounds__(256) og_k_force_b(og_pair_args a) { force_body<false>(a); }
__global__ void __launch_bounds__(256) og_k_force_a(og_pair_args a) { force_body<true>(a); }

static int pair_grid(int n_work) {
    int blocks = (n_work + 3) / 4;
    const int cap = 256 * 16;
    if (blocks > cap) blocks = cap;
    return blocks < 1 ? 1 : blocks;
}

void og_launch_pair_descreen(const og_pair_args& a, bool mode_a, hipStream_t s) {
    if (a.n_work <= 0) return;
    const int g = a.grid > 0 ? a.grid : pair_grid(a.n_work);
    if (mode_a) hipLaunchKernelGGL(og_k_descreen_a, dim3(g), dim3(256), 0, s, a);
    else hipLaunchKernelGGL(og_k_descreen_b, dim3(g), dim3(256), 0, s, a);
}

void og_launch_descreen_bonded(const og_pair_args& a, const og_bonded_args& b, bool mode_a, hipStream_t s) {
    const int nd = a.n_work > 0 ? (a.grid > 0 ? a.grid : pair_grid(a.n_work)) : 0;
    const int total = b.nb + b.na + b.nd + b.ni;
    int nb = (total + 255) / 256;
    if (nb > 4096) nb = 4096;
    if (nd + nb <= 0) return;
    if (mode_a) hipLaunchKernelGGL(og_k_descreen_bonded<true>, dim3(nd + nb), dim3(256), 0, s, a, b, nd);
    else hipLaunchKernelGGL(og_k_descreen_bonded<false>, dim3(nd + nb), dim3(256), 0, s, a, b, nd);
}

void og_launch_pair_force(const og_pair_args& a, bool mode_a, hipStream_t s) {
    const int n = a.n_strip + a.n_fwork;
    if (n <= 0) return;
    // the force pass has fewer, larger work items than descreening (strips):
    // it runs one wave per item (measured fastest at every width tried:
    // 0.299 ms on the 157k-atom batch against 0.304-0.387 ms at 4096 to 512
    // blocks), whatever width the descreening pass takes
    const int g = (n + 3) / 4;
    if (mode_a) hipLaunchKernelGGL(og_k_force_a, dim3(g), dim3(256), 0, s, a);
    else hipLaunchKernelGGL(og_k_force_b, dim3(g), dim3(256), 0, s, a);
}

// ---------------------------------------------------------------------------
// FP64 pair energies (LJ, Coulomb, GB pair), used for energy totals, REMD
// exchange and the L-BFGS line search.  Same tile schedule; all arithmetic in
// double, evaluated as origami writes it:
//   LJ       eps_ij ((Rmin/r)^12 - 2 (Rmin/r)^6)         nonbonded.rs:410-415
//   Coulomb  k q_i q_j (1/r + kappa r^2 - c)  (Mode B: k q_i q_j / r)  nonbonded.rs:327-329
//   GB pair  2 (-1/2)(1 - 1/eps_w) k q_i q_j / f_GB, uncut  gb.rs:160-173
// ---------------------------------------------------------------------------
namespace {

template <bool MODEA>
__device__ void energy_body(const og_pair_args& a, const og_energy64_args& e) {
    __shared__ EJ s_j[4][OG_TILE];
    EJ* J = s_j[threadIdx.x >> 6];
    const int lane = threadIdx.x & 63;
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int n_waves = (gridDim.x * blockDim.x) >> 6;
    const double kc = OG_COULOMB_KCAL * OG_KCAL_TO_KJ;
    const double pref = -(1.0 - 1.0 / OG_EPS_WATER) * OG_COULOMB_KCAL * OG_KCAL_TO_KJ;
    for (int w = wave; w < a.n_work; w += n_waves) {
        const og_work it = a.work[w];
        if (it.part == 1) continue;                 // a split tile pair is evaluated whole once
        if (a.skip_sys && a.skip_sys[it.sys]) continue;
        const int a0i = a.tile_atom0[it.ti], ci = a.tile_cnt[it.ti];
        const int a0j = a.tile_atom0[it.tj], cj = a.tile_cnt[it.tj];
        const bool vi = lane < ci, vj = lane < cj;
        const int gi = a0i + (vi ? lane : 0), gj = a0j + (vj ? lane : 0);
        const EI I = energy_i(a, e, gi, vi, e.radii[gi]);
        unsigned long long xm = 0, m14 = 0;
        if (it.mask >= 0) {
            xm = a.masks[(size_t)it.mask * 128 + lane];
            m14 = a.masks[(size_t)it.mask * 128 + 64 + lane];
        }
        const EJ mine = energy_j(a, e, gj, e.radii[gj]);
        wave_lds_order();                           // the previous tile's reads are done
        J[lane] = mine;
        wave_lds_order();
        const bool diag = it.ti == it.tj;
        ESum t = {0.0, 0.0, 0.0};
        if (!diag && it.mask < 0) {
            if (MODEA && energy_tiles_far(a, a0i, ci, a0j, cj, lane, I.iR, mine.iR)) energy_far(I, J, 0, cj, t);
            else energy_plain<MODEA>(e, I, J, 0, cj, t);
        } else {
            energy_masked<MODEA>(e, I, J, 0, cj, lane, diag, xm, m14, t);
        }
        double elj = t.lj, ec = t.c, eg = t.g;
        elj = og_wave_sum_d(elj * OG_KCAL_TO_KJ);
        ec = og_wave_sum_d(ec * kc);
        eg = og_wave_sum_d(eg * pref);
        if (lane == 0) {
            long long* acc = a.eacc + (size_t)it.sys * OG_NE;
            int* fl = a.sflag ? a.sflag + it.sys : nullptr;
            og_atomic_add_fix(acc + OG_E_LJ, og_to_fix_chk(elj, fl));
            og_atomic_add_fix(acc + OG_E_COUL, og_to_fix_chk(ec, fl));
            og_atomic_add_fix(acc + OG_E_GB_PAIR, og_to_fix_chk(eg, fl));
        }
    }
}

}  // namespace

__global__ void __launch_bounds__(256) og_k_energy64_b(og_pair_args a, og_energy64_args e) { energy_body<false>(a, e); }
__global__ void __launch_bounds__(256) og_k_energy64_a(og_pair_args a, og_energy64_args e) { energy_body<true>(a, e); }

void og_launch_pair_energy64(const og_pair_args& a, const og_energy64_args& e, bool mode_a, hipStream_t s) {
    if (a.n_work <= 0) return;
    const int g = pair_grid(a.n_work);
    if (mode_a) hipLaunchKernelGGL(og_k_energy64_a, dim3(g), dim3(256), 0, s, a, e);
    else hipLaunchKernelGGL(og_k_energy64_b, dim3(g), dim3(256), 0, s, a, e);
}

// ---------------------------------------------------------------------------
// Persistent replica steps: block s owns system s for n_steps steps.  Each
// phase runs the same per-item code as the step's separate launches (the
// same FP32 partial sums per work item, the same FP64 per-atom and per-term
// arithmetic; integer sums do not depend on order), so the trajectory is the
// one the launches give, bit for bit.  A system that stops (non-finite
// velocities, a range flag) leaves the loop at that step.
// ---------------------------------------------------------------------------
// threads per block of the persistent replica-step kernel: 8 waves, which
// take the work items of each phase (tile pairs, strips) in turn
#define OG_PERSIST_THREADS 512
template <bool MODEA>
__global__ void __launch_bounds__(OG_PERSIST_THREADS) og_k_replica_steps(og_pair_args pa, og_bonded_args ba, og_radii_args ra,
                                                          og_cluster_args ca, og_back_args bk, og_noise_args nz,
                                                          og_persist_args pp) {
    constexpr int NT = OG_PERSIST_THREADS, NW = OG_PERSIST_THREADS / 64;
    __shared__ float4 s_pq[NW][2 * (OG_TILE + 1)];
    __shared__ int s_stop;
    const int s = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float4* P = s_pq[wave];
    float4* Q = P + (OG_TILE + 1);
    const int a0 = pp.atom_off[s], a1 = pp.atom_off[s + 1];
    for (int k = 0; k < pp.n_steps; ++k) {
        // one thread reads the stop flag and the block follows it, so every
        // thread leaves the loop at the same step
        if (tid == 0) s_stop = __hip_atomic_load(ca.diverged + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (s_stop) break;
        const uint32_t step = pp.step0 + (uint32_t)k;
        for (int i = a0 + tid; i < a1; i += NT) noise_atom_at(nz, i, step);
        __syncthreads();
        for (int q = pp.cl_small_off[s] + tid; q < pp.cl_small_off[s + 1]; q += NT)
            cluster_body<OG_SMALL_CL>(ca, pp.cl_small[q], step);
        __syncthreads();
#pragma unroll
        for (int kind = 0; kind < 4; ++kind) {
            // global term index of this kind's first term (bonds, angles, dihedrals, impropers)
            const int base = kind == 0 ? 0 : kind == 1 ? ba.nb : kind == 2 ? ba.nb + ba.na : ba.nb + ba.na + ba.nd;
            const int* off = pp.term_off + kind * (pp.n_sys + 1);
            for (int t = off[s] + tid; t < off[s + 1]; t += NT) {
                int e_slot = -1, e_sys = 0;
                long long e_fix = 0;
                bonded_term<false>(ba, base + t, e_slot, e_sys, e_fix);
            }
        }
        for (int w = pp.work_off[s] + wave; w < pp.work_off[s + 1]; w += NW) {
            const og_work it = pa.work[w];
            descreen_item<MODEA>(pa, it, lane, P, Q);
        }
        __syncthreads();
        for (int i = a0 + tid; i < a1; i += NT) {
            radii_body<false>(ra, i);
            gather_atom(ba, i);
        }
        __syncthreads();
        for (int w = pp.strip_off[s] + wave; w < pp.strip_off[s + 1]; w += NW) {
            force_strip<MODEA>(pa, pa.strips + w, lane, P, Q);
        }
        for (int w = pp.fwork_off[s] + wave; w < pp.fwork_off[s + 1]; w += NW) {
            const og_work it = pa.fwork[w];
            force_item<MODEA>(pa, it, lane, P, Q);
        }
        __syncthreads();
        og_back_args b = bk;
        b.ke_acc = pp.ke_acc ? pp.ke_acc + (size_t)k * pp.n_sys : nullptr;
        for (int i0 = a0; i0 < a1; i0 += NT) back_wave(b, i0 + tid, a1);
        __syncthreads();
    }
}

void og_launch_replica_steps(const og_pair_args& pa, const og_bonded_args& ba, const og_radii_args& ra,
                             const og_cluster_args& ca, const og_back_args& bk, const og_noise_args& nz,
                             const og_persist_args& pp, bool mode_a, hipStream_t s) {
    if (pp.n_sys <= 0 || pp.n_steps <= 0) return;
    const dim3 g(pp.n_sys), t(OG_PERSIST_THREADS);
    if (mode_a) hipLaunchKernelGGL(og_k_replica_steps<true>, g, t, 0, s, pa, ba, ra, ca, bk, nz, pp);
    else hipLaunchKernelGGL(og_k_replica_steps<false>, g, t, 0, s, pa, ba, ra, ca, bk, nz, pp);
}
