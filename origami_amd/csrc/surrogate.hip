// Learned Born-radius surrogate: descriptor, MLP forward, training (forward +
// backward + weight gradients + Adam), all hand-written for gfx950.
//
// There is no counterpart in origami: the surrogate stands in for the
// descreening pass of compute_born_radii_into_scratch (energy/src/gb.rs:203-342)
// and is trained on the radii that pass produces.  Plain GB stays the arbiter:
// systems whose surrogate radii drift more than a tolerance from the plain
// radii at a periodic check fall back to plain GB (engine.cpp).
//
// MFMA: v_mfma_f32_16x16x32_bf16.  A (16x32) lane l holds row l%16, k =
// 8*(l/16)..+7; B (32x16) lane l holds column l%16, the same k; D (16x16)
// lane l holds column l%16, rows 4*(l/16)..+3.
//
// Layouts (bf16 stored as raw 16-bit words):
//   X    [rows][192]  descriptors (row-major)       -> A operand, layer 1
//   W1t  layer-1 weights                             -> B operand, layer 1
//   W2t  layer-2 weights                             -> B operand, layer 2
//   W2i  layer-2 weights transposed                  -> B operand, dH1 = dZ2 W2^T
//        each by operands, [column / 16][k / 32][lane][8]: a wave's load of
//        one is 1 KB in a run (by rows it was 16 pieces of 64 bytes)
//   *T   [batch/16][feature][16] activations          -> operands of the
//        weight-gradient GEMMs, whose reduction runs over the batch.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "og_sur.h"

#pragma clang fp contract(off)

typedef __bf16 og_bf16x8 __attribute__((ext_vector_type(8)));
typedef float og_f32x4 __attribute__((ext_vector_type(4)));

static std::string g_sur_err;
const char* og_sur_error() { return g_sur_err.c_str(); }

// defined in sasa_kernel.hip
__global__ void og_k_tile_bounds(const double* pos, const int* tile_atom0, const int* tile_cnt,
                                 int n_tiles, double4* out, int* counters);

namespace {

__host__ __device__ inline unsigned short f2bf(float f) {
    unsigned u;
    memcpy(&u, &f, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);          // round to nearest even
    return (unsigned short)(u >> 16);
}

__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float((unsigned)h << 16); }

__device__ __forceinline__ og_bf16x8 ld8(const unsigned short* p) {
    const uint4 u = *reinterpret_cast<const uint4*>(p);
    return __builtin_bit_cast(og_bf16x8, u);
}

__device__ __forceinline__ og_f32x4 mfma(og_bf16x8 a, og_bf16x8 b, og_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float sigm(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float silu(float z) { return z * sigm(z); }
// silu'(z) from z and s = sigm(z)
__device__ __forceinline__ float dsilu(float z, float s) { return s * (1.0f + z * (1.0f - s)); }

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ double rld(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

struct DescArgs {
    const double* pos;
    const double* rho;
    const int* cls;
    const int* tile_atom0;
    const int* tile_cnt;
    const int* tile_sys;
    const int* sys_tile_b;
    const int* sys_tile_e;
    const double4* tile_bound;
    const int* mode;       // null: all systems
    unsigned short* X;
};

}  // namespace

// Descriptor: one block per 64-atom tile I.  The block lists the tiles J of
// the same system whose bounding spheres come within 12 Å of tile I, then its
// eight waves take halves of those tiles in turn: lane = atom i, the atoms j
// are broadcast one by one, and every j != i with r < 12 Å adds one count to
// i's histogram row in LDS (integer counts, so the result does not depend on
// the order).  Instruction issue bounds the kernel, so the bin floor(r / 0.375
// Å) is read off single-precision distances about tile I's centre; a lane
// whose r / 0.375 Å comes within SUR_EDGE of a whole number (each bin's edge,
// the range's end at 32 and a pair of coincident atoms are such) settles the
// bin on FP64 r^2 against the edges (0.375 k)^2 = 0.140625 k^2, which are
// exact.  With atoms i within SUR_NEAR_A of the centre a coordinate difference
// of a pair in range is off by at most 8.1e-6 Å, so r / 0.375 Å by 4.5e-5;
// a tile that reaches further settles every pair in FP64.  About one wave step
// in fifty has such a lane.  30 520 atoms of 16 chains: 67 us with FP64
// distances and four waves, 25 us this way.
// Counts are 16-bit, two bins to a word (25 KB of LDS per block, so that the
// kernel fits beside the SASA arrangement on a CU).
#define SUR_DESC_WAVES 8
#define SUR_HW ((OG_SUR_F + 1) / 2)                     // words per histogram row (81)
#define SUR_EDGE 1.0e-4f
#define SUR_NEAR_A 64.0

// bin of r^2, or 32 and more beyond the range
__device__ __forceinline__ int desc_bin(double dx, double dy, double dz) {
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (!(r2 < 144.0)) return 32;
    int k = (int)(sqrtf((float)r2) * (1.0f / 0.375f));
    k = k > 31 ? 31 : (k < 0 ? 0 : k);
    while (k < 31 && 0.140625 * (double)((k + 1) * (k + 1)) <= r2) ++k;
    while (k > 0 && 0.140625 * (double)(k * k) > r2) --k;
    return k;
}

__global__ void __launch_bounds__(64 * SUR_DESC_WAVES) og_k_sur_desc(DescArgs a) {
    __shared__ unsigned hist[64 * SUR_HW];            // odd stride: conflict-free rows
    __shared__ int near_list[1024];
    __shared__ int n_near;
    const int t = blockIdx.x;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sys = a.tile_sys[t];
    if (a.mode && !a.mode[sys]) return;
    for (int q = tid; q < 64 * SUR_HW; q += blockDim.x) hist[q] = 0u;
    if (tid == 0) n_near = 0;
    __syncthreads();
    const double4 bi = a.tile_bound[t];
    const int jb = a.sys_tile_b[sys], je = a.sys_tile_e[sys];
    for (int J = jb + tid; J < je; J += blockDim.x) {
        const double4 bj = a.tile_bound[J];
        const double cx = bj.x - bi.x, cy = bj.y - bi.y, cz = bj.z - bi.z;
        const double reach = bi.w + bj.w + 12.0;
        if (cx * cx + cy * cy + cz * cz <= reach * reach) {
            const int slot = atomicAdd(&n_near, 1);
            if (slot < 1024) near_list[slot] = J;
        }
    }
    __syncthreads();
    const int nn = n_near < 1024 ? n_near : 1024;
    const int a0 = a.tile_atom0[t], cnt = a.tile_cnt[t];
    const bool vi = lane < cnt;
    const int i = a0 + lane;
    const bool wide = !(bi.w <= SUR_NEAR_A);          // every pair in FP64
    double xi = 0.0, yi = 0.0, zi = 0.0;
    if (vi) { xi = a.pos[3 * (size_t)i]; yi = a.pos[3 * (size_t)i + 1]; zi = a.pos[3 * (size_t)i + 2]; }
    // lanes without an atom stay out of every range
    const float fx = vi ? (float)(xi - bi.x) : 1.0e9f, fy = (float)(yi - bi.y), fz = (float)(zi - bi.z);
    unsigned* row = hist + lane * SUR_HW;
    for (int q = wv; q < 2 * nn; q += SUR_DESC_WAVES) {
        const int J = near_list[q >> 1];
        const int b0 = a.tile_atom0[J] + (q & 1) * 32;
        const int cj = a.tile_cnt[J] - (q & 1) * 32 < 32 ? a.tile_cnt[J] - (q & 1) * 32 : 32;
        double xj = 0.0, yj = 0.0, zj = 0.0;
        int cl = 0;
        if (lane < cj) {
            const size_t j = 3 * (size_t)(b0 + lane);
            xj = a.pos[j]; yj = a.pos[j + 1]; zj = a.pos[j + 2];
            cl = a.cls[b0 + lane];
        }
        // slots past the tile's atoms stay out of every range
        const int gx = __float_as_int(lane < cj ? (float)(xj - bi.x) : 3.0e9f), gy = __float_as_int((float)(yj - bi.y)),
                  gz = __float_as_int((float)(zj - bi.z));
        for (int j0 = 0; j0 < cj; j0 += 4) {
            int k[4], c[4];
            bool in[4], near[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int jj = j0 + u;
                const float dx = __int_as_float(__builtin_amdgcn_readlane(gx, jj)) - fx,
                            dy = __int_as_float(__builtin_amdgcn_readlane(gy, jj)) - fy,
                            dz = __int_as_float(__builtin_amdgcn_readlane(gz, jj)) - fz;
                c[u] = __builtin_amdgcn_readlane(cl, jj);
                const float s = __builtin_amdgcn_sqrtf(fmaf(dx, dx, fmaf(dy, dy, dz * dz))) * (1.0f / 0.375f);
                k[u] = (int)s;
                in[u] = s < 32.0f;
                near[u] = vi && (wide || (!(s >= 32.0f + SUR_EDGE) && !(fabsf(s - rintf(s)) > SUR_EDGE)));
            }
            if (__any(near[0] | near[1] | near[2] | near[3])) {
#pragma unroll 1
                for (int u = 0; u < 4; ++u) {
                    const int jj = j0 + u;
                    const bool nu = u == 0 ? near[0] : u == 1 ? near[1] : u == 2 ? near[2] : near[3];
                    const int b = nu && jj < cj && b0 + jj != i
                                      ? desc_bin(rld(xj, jj) - xi, rld(yj, jj) - yi, rld(zj, jj) - zi) : 32;
#pragma unroll
                    for (int q4 = 0; q4 < 4; ++q4)
                        if (nu && q4 == u) {
                            k[q4] = b;
                            in[q4] = b < 32;
                        }
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (in[u]) {
                    const int b = c[u] * 32 + k[u];
                    atomicAdd(row + (b >> 1), 1u << ((b & 1) * 16));
                }
        }
    }
    __syncthreads();
    // write the rows, eight features at a time
    constexpr int V = OG_SUR_K1 / 8;
    for (int q = tid; q < cnt * V; q += blockDim.x) {
        const int rr = q / V, f = (q % V) * 8;
        unsigned v[4] = {0u, 0u, 0u, 0u};
        if (f < 160) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const unsigned h = hist[rr * SUR_HW + (f >> 1) + u];
                v[u] = f2bf((float)(h & 0xFFFFu) * 0.125f) | ((unsigned)f2bf((float)(h >> 16) * 0.125f) << 16);
            }
        } else if (f == 160) {
            v[0] = f2bf((float)((a.rho[a0 + rr] - 1.5) * 4.0));
        }
        *reinterpret_cast<uint4*>(a.X + (size_t)(a0 + rr) * OG_SUR_K1 + f) = make_uint4(v[0], v[1], v[2], v[3]);
    }
}

namespace {

struct MlpParams {
    const unsigned short* W1t;
    const unsigned short* W2t;
    const unsigned short* W2i;
    const float* p;            // FP32 master (b1, b2, w3, b3)
};

struct MlpOperands {
    unsigned short *W1t, *W2t, *W2i;
};

// place of column j, input k in a B operand with kk_n steps of 32 inputs, and
// a lane's eight inputs of step kk for the 16 columns nt
__device__ __forceinline__ int operand_at(int j, int k, int kk_n) {
    return (((j >> 4) * kk_n + (k >> 5)) * 64 + ((k >> 3) & 3) * 16 + (j & 15)) * 8 + (k & 7);
}
__device__ __forceinline__ og_bf16x8 operand(const unsigned short* w, int nt, int kk, int kk_n, int lane) {
    return ld8(w + ((nt * kk_n + kk) * 64 + lane) * 8);
}

// BF16 operand copy (copies, of W2) of parameter q
__device__ __forceinline__ void store_operand(const MlpOperands& o, int q, float w) {
    if (q < OG_SUR_OFF_B1) {
        const int k = q / OG_SUR_H, j = q % OG_SUR_H;
        o.W1t[operand_at(j, k, OG_SUR_K1 / 32)] = f2bf(w);
    } else if (q >= OG_SUR_OFF_W2 && q < OG_SUR_OFF_B2) {
        const int e = q - OG_SUR_OFF_W2;
        const int k = e / OG_SUR_H, j = e % OG_SUR_H;
        o.W2t[operand_at(j, k, OG_SUR_H / 32)] = f2bf(w);
        o.W2i[operand_at(k, j, OG_SUR_H / 32)] = f2bf(w);
    }
}

}  // namespace

// Inference, SUR_INFER_ROWS rows per block: each of the eight waves holds the
// weights of one 16-column group of both layers in registers and takes the
// 16-row groups in turn, with the activations exchanged over LDS (26 KB, so
// that the kernel fits beside the SASA arrangement on a CU).  Every element
// keeps its MFMA chain and the output sum its order over the column groups.
// 64 rows per wave, both layers unrolled over the column groups, took 26 us
// for 30 520 rows; columns over the waves with the rows and weights read in
// pieces of 64 bytes, eight waves the same rows, 24; rows through LDS and the
// weights in runs 12, of which about 10 are the exponentials and divisions.
#define SUR_INFER_ROWS 32
__global__ void __launch_bounds__(512) og_k_sur_infer(const unsigned short* X, int n_valid, int n_rows,
                                                      MlpParams P, double* r_out) {
    __shared__ __attribute__((aligned(16))) unsigned short h1s[SUR_INFER_ROWS][136];
    __shared__ __attribute__((aligned(16))) union {
        unsigned short x[SUR_INFER_ROWS][OG_SUR_K1 + 8];
        float h2[8][SUR_INFER_ROWS][17];
    } sh;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int j = w * 16 + r;
    const int row0 = blockIdx.x * SUR_INFER_ROWS;
    og_bf16x8 w1[6], w2[4];
#pragma unroll
    for (int kk = 0; kk < 6; ++kk) w1[kk] = operand(P.W1t, w, kk, OG_SUR_K1 / 32, lane);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) w2[kk] = operand(P.W2t, w, kk, OG_SUR_H / 32, lane);
    const float b1 = P.p[OG_SUR_OFF_B1 + j], b2 = P.p[OG_SUR_OFF_B2 + j];
    for (int q = threadIdx.x; q < SUR_INFER_ROWS * (OG_SUR_K1 / 8); q += 512) {
        const int rr = q / (OG_SUR_K1 / 8), c = q % (OG_SUR_K1 / 8) * 8;
        *reinterpret_cast<og_bf16x8*>(&sh.x[rr][c]) = ld8(X + (size_t)(row0 + rr < n_rows ? row0 + rr : 0) * OG_SUR_K1 + c);
    }
    __syncthreads();
#pragma unroll
    for (int rg = 0; rg < SUR_INFER_ROWS; rg += 16) {
        og_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 6; ++kk) acc = mfma(ld8(&sh.x[rg + r][kk * 32 + g * 8]), w1[kk], acc);
#pragma unroll
        for (int i = 0; i < 4; ++i) h1s[rg + g * 4 + i][j] = f2bf(silu(acc[i] + b1));
    }
    __syncthreads();
#pragma unroll
    for (int rg = 0; rg < SUR_INFER_ROWS; rg += 16) {
        og_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) acc = mfma(ld8(&h1s[rg + r][kk * 32 + g * 8]), w2[kk], acc);
#pragma unroll
        for (int i = 0; i < 4; ++i) sh.h2[w][rg + g * 4 + i][r] = silu(acc[i] + b2);
    }
    __syncthreads();
    // a wave sums four rows: over the column groups in order, then the columns
    const int row = w * 4 + g;
    float v = 0.0f;
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) v += sh.h2[nt][row][r] * P.p[OG_SUR_OFF_W3 + nt * 16 + r];
    v += __shfl_xor(v, 1, 64);
    v += __shfl_xor(v, 2, 64);
    v += __shfl_xor(v, 4, 64);
    v += __shfl_xor(v, 8, 64);
    const float y = v + P.p[OG_SUR_OFF_B3];
    if (r == 0 && row0 + row < n_valid) r_out[row0 + row] = OG_SUR_R0 + OG_SUR_RS * (double)y;
}

__device__ __forceinline__ unsigned long long sur_mix(unsigned long long x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

// h mod n with inv = (2^64 - 1) / n: the quotient guessed from inv is at most
// two too small
__device__ __forceinline__ unsigned long long sur_mod(unsigned long long h, unsigned long long n,
                                                      unsigned long long inv) {
    unsigned long long m = h - __umul64hi(h, inv) * n;
    if (m >= n) m -= n;
    if (m >= n) m -= n;
    return m;
}

// Training forward + backward, 16 batch rows per block: each of the eight
// waves takes one of the eight 16-column groups of every layer, with the
// activations exchanged over LDS.  What bounds the kernel at these sizes (a
// batch of 4 096 is 256 row groups) is one wave's chain of weight loads, MFMA
// and exponentials, so a group's chain is cut in eight.  Each element keeps its
// own MFMA chain and the output sum its order over the column groups, so the
// values are those of one wave per group.  The block also picks its rows out
// of the training set, row b being hash(seed, b) mod n_rows (n_rows 0: row b
// itself).  What the weight gradients read is left by groups of 16 rows,
// [B/16][columns][16]: a block writes whole lines, and a wave there reads the
// 32 rows of 16 columns as two runs of 512 bytes.  At 4 096 rows 50 us before
// (40 and a separate gather's 10), 14 now, of which 7 are the chain (2 blocks
// take as long) and the rest the 11 MB written.
__device__ __forceinline__ size_t sur_at(int col, int row, int cols) {
    return ((size_t)(row >> 4) * cols + col) * 16 + (row & 15);
}

struct TrainArgs {
    const unsigned short* X;    // [rows][K1]
    const float* t;             // [rows] normalised targets
    long long n_rows;
    unsigned long long inv;     // (2^64 - 1) / n_rows
    unsigned long long seed;
    int B;
    unsigned short* XbT;                 // [B/16][K1][16]
    unsigned short *H1T, *dZ1T, *dZ2T;   // [B/16][H][16] bf16
    float *dZ1Tf, *dZ2Tf, *H2Tf;         // [B/16][H][16] fp32
    float *dy, *lossr;                   // [B]
};

__device__ __forceinline__ void store4(unsigned short* p, const unsigned short (&v)[4]) {
    *reinterpret_cast<uint2*>(p) = make_uint2(v[0] | ((unsigned)v[1] << 16), v[2] | ((unsigned)v[3] << 16));
}
__device__ __forceinline__ void store4(float* p, const float (&v)[4]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}

__global__ void __launch_bounds__(512) og_k_sur_fwdbwd(TrainArgs a, MlpParams P) {
    __shared__ __attribute__((aligned(16))) unsigned short xs[16][OG_SUR_K1 + 8];
    __shared__ __attribute__((aligned(16))) unsigned short h1s[16][136], dz2s[16][136];
    __shared__ float h2s[8][16][17];                  // silu(z2) by column group, row, column
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int j = w * 16 + r;                          // this lane's column in every layer
    const int row0 = blockIdx.x * 16;
    const int rg = row0 + g * 4;                       // its four rows in the D layout
    // the weights load first, while the row's index is formed
    og_bf16x8 a1[6], w1[6], w2[4], w2i[4];
#pragma unroll
    for (int kk = 0; kk < 6; ++kk) w1[kk] = operand(P.W1t, w, kk, OG_SUR_K1 / 32, lane);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) w2[kk] = operand(P.W2t, w, kk, OG_SUR_H / 32, lane);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) w2i[kk] = operand(P.W2i, w, kk, OG_SUR_H / 32, lane);
    const float b1 = P.p[OG_SUR_OFF_B1 + j], b2 = P.p[OG_SUR_OFF_B2 + j], w3 = P.p[OG_SUR_OFF_W3 + j];
    const float b3 = P.p[OG_SUR_OFF_B3];
    float w3c[8];
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) w3c[nt] = P.p[OG_SUR_OFF_W3 + nt * 16 + r];
    long long src = row0 + r;
    if (a.n_rows > 0)
        src = (long long)sur_mod(sur_mix(a.seed ^ sur_mix((unsigned long long)src)), (unsigned long long)a.n_rows, a.inv);
#pragma unroll
    for (int kk = 0; kk < 6; ++kk) a1[kk] = ld8(a.X + src * OG_SUR_K1 + kk * 32 + g * 8);
    const float tr = a.t[src];

    og_f32x4 z1 = {0.f, 0.f, 0.f, 0.f}, s1;            // pre-activation and its sigmoid
#pragma unroll
    for (int kk = 0; kk < 6; ++kk) z1 = mfma(a1[kk], w1[kk], z1);
    unsigned short hb[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        z1[i] += b1;
        s1[i] = sigm(z1[i]);
        hb[i] = f2bf(z1[i] * s1[i]);
        h1s[g * 4 + i][j] = hb[i];
    }
#pragma unroll
    for (int kk = 0; kk < 6; ++kk)
        if (kk == w) *reinterpret_cast<og_bf16x8*>(&xs[r][kk * 32 + g * 8]) = a1[kk];
    __syncthreads();

    og_bf16x8 a2[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) a2[kk] = ld8(&h1s[r][kk * 32 + g * 8]);
    og_f32x4 z2 = {0.f, 0.f, 0.f, 0.f}, s2;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) z2 = mfma(a2[kk], w2[kk], z2);
    float h2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        z2[i] += b2;
        s2[i] = sigm(z2[i]);
        h2[i] = z2[i] * s2[i];
        h2s[w][g * 4 + i][r] = h2[i];
    }
    __syncthreads();

    // y of the lane's rows (every wave forms them), summed over the column
    // groups in order, then over the columns
    const float inv_b2 = 2.0f / (float)a.B;
    float dyv[4], dr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float v = 0.0f;
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) v += h2s[nt][g * 4 + i][r] * w3c[nt];
        v += __shfl_xor(v, 1, 64);
        v += __shfl_xor(v, 2, 64);
        v += __shfl_xor(v, 4, 64);
        v += __shfl_xor(v, 8, 64);
        dr[i] = (v + b3) - __shfl(tr, g * 4 + i, 64);
        dyv[i] = dr[i] * inv_b2;
    }
    // dZ2 = dy w3 * silu'(z2)
    float dz2[4], dz1[4];
    unsigned short db2[4], db1[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        dz2[i] = dyv[i] * w3 * dsilu(z2[i], s2[i]);
        db2[i] = f2bf(dz2[i]);
        dz2s[g * 4 + i][j] = db2[i];
    }
    __syncthreads();
    // dH1 = dZ2 W2^T, then dZ1 = dH1 * silu'(z1)
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) a2[kk] = ld8(&dz2s[r][kk * 32 + g * 8]);
    og_f32x4 dh = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) dh = mfma(a2[kk], w2i[kk], dh);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        dz1[i] = dh[i] * dsilu(z1[i], s1[i]);
        db1[i] = f2bf(dz1[i]);
    }

    // the weight gradients' operands
    const size_t o = sur_at(j, rg, OG_SUR_H);
    store4(a.H1T + o, hb);
    store4(a.H2Tf + o, h2);
    store4(a.dZ2Tf + o, dz2);
    store4(a.dZ2T + o, db2);
    store4(a.dZ1Tf + o, dz1);
    store4(a.dZ1T + o, db1);
    if (w == 0 && r == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a.dy[rg + i] = dyv[i];
            a.lossr[rg + i] = dr[i] * dr[i];
        }
    }
    if (threadIdx.x < OG_SUR_K1) {
        unsigned v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            v[u] = xs[2 * u][threadIdx.x] | ((unsigned)xs[2 * u + 1][threadIdx.x] << 16);
        uint4* q = reinterpret_cast<uint4*>(a.XbT + sur_at(threadIdx.x, row0, OG_SUR_K1));
        q[0] = make_uint4(v[0], v[1], v[2], v[3]);
        q[1] = make_uint4(v[4], v[5], v[6], v[7]);
    }
}

// Weight gradients and the Adam step, fixed reduction order (deterministic):
//   blocks [0, 96)     dW1 tiles: D[j][k] = sum_b dZ1T[j][b] XbT[k][b]
//   blocks [96, 160)   dW2 tiles: D[j][k] = sum_b dZ2T[j][b] H1T[k][b]
//   then a wave per sum: db1[j] = sum_b dZ1[b][j], db2[j] = sum_b dZ2[b][j],
//   dW3[j] = sum_b H2[b][j] dy[b], db3 = sum_b dy[b], loss = mean (y - t)^2
// A tile is one MFMA chain over the batch (its order is the result's), bound
// by the wait for its operands, not by the matrix cores: the block's eight
// waves each load SUR_WG_AHEAD steps at once and take the chain in turn,
// passing the accumulator on through LDS.  One wave per tile that waits for
// each step's loads took 34 us at 4 096 rows, one that loads 16 steps ahead
// 15.5, this 10.8, with the Adam update (6 us as a launch of its own) in it:
// an element's parameter and moments load before its gradient is formed.
struct GradArgs {
    const unsigned short *dZ1T, *XbT, *dZ2T, *H1T;
    const float *dZ1Tf, *dZ2Tf, *H2Tf, *dy, *lossr;
    int B;
    float* grad;               // gradient out, or (null) one Adam step on p, m, v
    float* loss;
    float *p, *m, *v;
    float lr, c1, c2;
    MlpOperands o;
};

// Where element q's gradient goes: out, or through Adam (w, m0, v0: the
// parameter and its moments) into the parameter and its BF16 copies.
__device__ __forceinline__ void apply_gradient(const GradArgs& a, int q, float gq, float w, float m0, float v0) {
    if (a.grad) {
        a.grad[q] = gq;
        return;
    }
    const float mq = 0.9f * m0 + 0.1f * gq;
    const float vq = 0.999f * v0 + 0.001f * gq * gq;
    a.m[q] = mq;
    a.v[q] = vq;
    w -= a.lr * (mq / a.c1) / (sqrtf(vq / a.c2) + 1e-8f);
    a.p[q] = w;
    store_operand(a.o, q, w);
}

#define SUR_WG_WAVES 8
#define SUR_WG_AHEAD 16
#define SUR_WG_TILES 160
#define SUR_WG_SUMS (3 * OG_SUR_H + 2)

// a lane's sum of x over rows lane, lane + 64, ... in order (stride: of x
// between those rows; DOT: of x y, y by row), the loads of 32 rows in flight
// together
template <bool DOT>
__device__ __forceinline__ float strided_sum(int B, int lane, const float* x, int stride, const float* y = nullptr) {
    const int n = (B - lane + 63) / 64;
    float s = 0.0f;
    for (int m0 = 0; m0 < n; m0 += 32) {
        float v[32], c[32];
#pragma unroll
        for (int u = 0; u < 32; ++u) {
            const int m = m0 + u < n ? m0 + u : m0;
            v[u] = x[(size_t)m * stride];
            if constexpr (DOT) c[u] = y[m * 64];
        }
#pragma unroll
        for (int u = 0; u < 32; ++u)
            if (m0 + u < n) {
                if constexpr (DOT) s += v[u] * c[u];
                else s += v[u];
            }
    }
    return s;
}

__global__ void __launch_bounds__(64 * SUR_WG_WAVES) og_k_sur_wgrad(GradArgs a) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (blockIdx.x < SUR_WG_TILES) {
        __shared__ og_f32x4 part[64];
        const int task = blockIdx.x;
        const int r = lane & 15, g = lane >> 4;
        const bool first = task < 96;
        const int jt = first ? task / 12 : (task - 96) / 8;
        const int kt = first ? task % 12 : (task - 96) % 8;
        const int bc = first ? OG_SUR_K1 : OG_SUR_H;
        const unsigned short* Ap = (first ? a.dZ1T : a.dZ2T) + sur_at(jt * 16 + r, g * 8, OG_SUR_H);
        const unsigned short* Bp = (first ? a.XbT : a.H1T) + sur_at(kt * 16 + r, g * 8, bc);
        const int n = a.B / 32;
        // thread t < 256 applies element (k, j) = (t / 16, t % 16) of the tile
        const int t = threadIdx.x;
        const int q = (first ? OG_SUR_OFF_W1 : OG_SUR_OFF_W2) + (kt * 16 + (t >> 4)) * OG_SUR_H + jt * 16 + (t & 15);
        float pq = 0.0f, mq = 0.0f, vq = 0.0f;
        if (t < 256 && !a.grad) {
            pq = a.p[q];
            mq = a.m[q];
            vq = a.v[q];
        }
        for (int k0 = 0; k0 < n; k0 += SUR_WG_WAVES * SUR_WG_AHEAD) {
            const int kw = k0 + w * SUR_WG_AHEAD;
            og_bf16x8 av[SUR_WG_AHEAD], bv[SUR_WG_AHEAD];
#pragma unroll
            for (int u = 0; u < SUR_WG_AHEAD; ++u)
                if (kw + u < n) {
                    av[u] = ld8(Ap + (size_t)(kw + u) * (32 * OG_SUR_H));
                    bv[u] = ld8(Bp + (size_t)(kw + u) * (32 * bc));
                }
            for (int turn = 0; turn < SUR_WG_WAVES && k0 + turn * SUR_WG_AHEAD < n; ++turn) {
                if (turn == w) {
                    og_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                    if (kw > 0) acc = part[lane];
#pragma unroll
                    for (int u = 0; u < SUR_WG_AHEAD; ++u)
                        if (kw + u < n) acc = mfma(av[u], bv[u], acc);
                    part[lane] = acc;
                }
                __syncthreads();
            }
        }
        if (t < 256) {
            // D layout: row j = 4 g + i, column k = r
            const int jl = t & 15, kl = t >> 4;
            apply_gradient(a, q, reinterpret_cast<const float*>(part)[((jl >> 2) * 16 + kl) * 4 + (jl & 3)], pq, mq, vq);
        }
        return;
    }
    const int task = (blockIdx.x - SUR_WG_TILES) * SUR_WG_WAVES + w;
    if (task >= SUR_WG_SUMS) return;
    float s = 0.0f;
    int out = -1;
    if (task < 3 * OG_SUR_H) {
        const size_t o = sur_at(task & (OG_SUR_H - 1), lane, OG_SUR_H);
        const int stride = 64 * OG_SUR_H;
        if (task < OG_SUR_H) {
            s = strided_sum<false>(a.B, lane, a.dZ1Tf + o, stride);
            out = OG_SUR_OFF_B1 + task;
        } else if (task < 2 * OG_SUR_H) {
            s = strided_sum<false>(a.B, lane, a.dZ2Tf + o, stride);
            out = OG_SUR_OFF_B2 + task - OG_SUR_H;
        } else {
            s = strided_sum<true>(a.B, lane, a.H2Tf + o, stride, a.dy + lane);
            out = OG_SUR_OFF_W3 + task - 2 * OG_SUR_H;
        }
    } else if (task == 3 * OG_SUR_H) {
        s = strided_sum<false>(a.B, lane, a.dy + lane, 64);
        out = OG_SUR_OFF_B3;
    } else {
        s = strided_sum<false>(a.B, lane, a.lossr + lane, 64);
    }
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) {
        if (out < 0) *a.loss = s / (float)a.B;
        else if (a.grad) a.grad[out] = s;
        else apply_gradient(a, out, s, a.p[out], a.m[out], a.v[out]);
    }
}

// BF16 operand copies of the FP32 master parameters.
__global__ void __launch_bounds__(256) og_k_sur_operands(const float* p, MlpOperands o) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < OG_SUR_P) store_operand(o, q, p[q]);
}

// Append descriptors and normalised plain radii of atoms [0, n) at row base.
__global__ void __launch_bounds__(256) og_k_sur_append(const unsigned short* X, const double* radii, int n,
                                                       unsigned short* Xtr, float* ttr, long long base) {
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long long)n * OG_SUR_K1) return;
    const int i = (int)(q / OG_SUR_K1), f = (int)(q % OG_SUR_K1);
    Xtr[(base + i) * OG_SUR_K1 + f] = X[(size_t)i * OG_SUR_K1 + f];
    if (f == 0) ttr[base + i] = (float)((radii[i] - OG_SUR_R0) / OG_SUR_RS);
}

// Fallback check: dev[s] = max over the system's atoms of |R_sur - R_plain| / R_plain
// (float bits; non-negative floats order like their bit patterns).
__global__ void og_k_sur_zero(unsigned* dev, int n) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) dev[q] = 0u;
}

__global__ void og_k_sur_fallback(int* mode, const unsigned* dev, int n, float tol) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n && mode[q] && !(__uint_as_float(dev[q]) <= tol)) mode[q] = 0;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
namespace {

template <class T>
bool dalloc(T** p, size_t n) {
    if (hipMalloc((void**)p, std::max<size_t>(n, 1) * sizeof(T)) != hipSuccess) return false;
    return hipMemset(*p, 0, std::max<size_t>(n, 1) * sizeof(T)) == hipSuccess;
}

template <class T>
bool upload(T** p, const std::vector<T>& v) {
    if (!dalloc(p, v.size())) return false;
    return v.empty() || hipMemcpy(*p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice) == hipSuccess;
}

int fail(const char* m) {
    g_sur_err = m;
    return -2;
}

MlpParams params_of(const og_sur* s) { return {s->W1t, s->W2t, s->W2i, s->p}; }
MlpOperands operands_of(const og_sur* s) { return {s->W1t, s->W2t, s->W2i}; }

int refresh_copies(og_sur* s) {
    hipLaunchKernelGGL(og_k_sur_operands, dim3((OG_SUR_P + 255) / 256), dim3(256), 0, s->stream, s->p, operands_of(s));
    return hipGetLastError() == hipSuccess ? 0 : fail("kernel launch failed");
}

// forward, backward and weight gradients of B rows of (X, t); the gradient
// goes to grad, or (null) one Adam step is taken
int batch_gradient(og_sur* s, const unsigned short* X, const float* t, long long n_rows, unsigned long long seed,
                   int B, float* grad, float lr, float c1, float c2, float* loss) {
    const unsigned long long inv = n_rows > 0 ? ~0ull / (unsigned long long)n_rows : 0;
    TrainArgs ta{X, t, n_rows, inv, seed, B, s->XbT, s->H1T, s->dZ1T, s->dZ2T, s->dZ1Tf, s->dZ2Tf, s->H2Tf, s->dy, s->lossr};
    hipLaunchKernelGGL(og_k_sur_fwdbwd, dim3(B / 16), dim3(512), 0, s->stream, ta, params_of(s));
    GradArgs ga{s->dZ1T, s->XbT, s->dZ2T, s->H1T, s->dZ1Tf, s->dZ2Tf, s->H2Tf, s->dy, s->lossr, B, grad, loss,
                s->p, s->m, s->v, lr, c1, c2, operands_of(s)};
    hipLaunchKernelGGL(og_k_sur_wgrad, dim3(SUR_WG_TILES + (SUR_WG_SUMS + SUR_WG_WAVES - 1) / SUR_WG_WAVES),
                       dim3(64 * SUR_WG_WAVES), 0, s->stream, ga);
    return hipGetLastError() == hipSuccess ? 0 : fail("kernel launch failed");
}

}  // namespace

int og_sur_create(og_sur* s, int n_atoms, int n_sys, const std::vector<double>& mass,
                  const std::vector<int>& sys_tile_off, const double* pos_dev, const double* rho_dev,
                  const int* tile_atom0_dev, const int* tile_cnt_dev, int n_tiles, long long capacity,
                  unsigned long long seed, hipStream_t stream) {
    s->n_atoms = n_atoms;
    s->n_pad = (n_atoms + 15) / 16 * 16;
    s->n_tiles = n_tiles;
    s->n_sys = n_sys;
    s->stream = stream;
    s->pos = pos_dev;
    s->rho = rho_dev;
    s->tile_atom0 = tile_atom0_dev;
    s->tile_cnt = tile_cnt_dev;
    std::vector<int> cls(n_atoms), tsys(n_tiles), tb(n_sys), te(n_sys);
    for (int i = 0; i < n_atoms; ++i) {
        const double mm = mass[i];
        cls[i] = mm < 2.0 ? 0 : mm < 13.0 ? 1 : mm < 15.0 ? 2 : mm < 17.0 ? 3 : 4;
    }
    for (int q = 0; q < n_sys; ++q) {
        tb[q] = sys_tile_off[q];
        te[q] = sys_tile_off[q + 1];
        if (te[q] - tb[q] > 1024) return fail("the descriptor kernel handles systems of up to 65536 atoms");
        for (int t = tb[q]; t < te[q]; ++t) tsys[t] = q;
    }
    if (!upload(&s->cls, cls) || !upload(&s->tile_sys, tsys) || !upload(&s->sys_tile_b, tb) ||
        !upload(&s->sys_tile_e, te) || !dalloc(&s->tile_bound, (size_t)n_tiles) ||
        !dalloc(&s->X, (size_t)s->n_pad * OG_SUR_K1) || !dalloc(&s->r_sur, (size_t)n_atoms) ||
        !dalloc(&s->mode, (size_t)n_sys) || !dalloc(&s->dev, (size_t)n_sys))
        return fail("device allocation failed");
    // parameters: W ~ N(0, 1/fan_in) from a seeded SplitMix64 + Box-Muller stream, biases 0
    std::vector<float> p(OG_SUR_P, 0.0f);
    unsigned long long st = seed;
    auto next = [&st]() {
        unsigned long long z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    };
    auto gauss = [&]() {
        const double u1 = ((next() >> 11) + 0.5) * 0x1.0p-53, u2 = ((next() >> 11) + 0.5) * 0x1.0p-53;
        return std::sqrt(-2.0 * std::log(u1)) * std::cos(2.0 * M_PI * u2);
    };
    for (int k = 0; k < OG_SUR_F; ++k)
        for (int j = 0; j < OG_SUR_H; ++j) p[OG_SUR_OFF_W1 + k * OG_SUR_H + j] = (float)(gauss() / std::sqrt((double)OG_SUR_F));
    for (int k = 0; k < OG_SUR_H; ++k)
        for (int j = 0; j < OG_SUR_H; ++j) p[OG_SUR_OFF_W2 + k * OG_SUR_H + j] = (float)(gauss() / std::sqrt((double)OG_SUR_H));
    for (int j = 0; j < OG_SUR_H; ++j) p[OG_SUR_OFF_W3 + j] = (float)(gauss() / std::sqrt((double)OG_SUR_H));
    if (!upload(&s->p, p) || !dalloc(&s->m, OG_SUR_P) || !dalloc(&s->v, OG_SUR_P) || !dalloc(&s->g, OG_SUR_P) ||
        !dalloc(&s->W1t, (size_t)OG_SUR_H * OG_SUR_K1) || !dalloc(&s->W2t, (size_t)OG_SUR_H * OG_SUR_H) ||
        !dalloc(&s->W2i, (size_t)OG_SUR_H * OG_SUR_H))
        return fail("device allocation failed");
    s->cap = capacity;
    s->n_train = 0;
    const size_t B = OG_SUR_BMAX;
    if (!dalloc(&s->Xtr, (size_t)std::max(capacity, 1ll) * OG_SUR_K1) || !dalloc(&s->ttr, (size_t)std::max(capacity, 1ll)) ||
        !dalloc(&s->Xb, B * OG_SUR_K1) || !dalloc(&s->XbT, B * OG_SUR_K1) || !dalloc(&s->H1T, B * OG_SUR_H) ||
        !dalloc(&s->dZ1T, B * OG_SUR_H) || !dalloc(&s->dZ2T, B * OG_SUR_H) || !dalloc(&s->dZ1Tf, B * OG_SUR_H) ||
        !dalloc(&s->dZ2Tf, B * OG_SUR_H) || !dalloc(&s->H2Tf, B * OG_SUR_H) || !dalloc(&s->tb, B) ||
        !dalloc(&s->dy, B) || !dalloc(&s->lossr, B) || !dalloc(&s->loss, OG_SUR_LOSSES))
        return fail("device allocation failed (training buffers)");
    s->adam_t = 0;
    if (refresh_copies(s)) return -2;
    return hipStreamSynchronize(stream) == hipSuccess ? 0 : fail("surrogate set-up failed");
}

void og_sur_free(og_sur* s) {
    void* ptrs[] = {s->cls, s->tile_sys, s->sys_tile_b, s->sys_tile_e, s->tile_bound, s->X, s->r_sur, s->mode,
                    s->dev, s->p, s->m, s->v, s->g, s->W1t, s->W2t, s->W2i, s->Xtr, s->ttr, s->Xb, s->XbT,
                    s->H1T, s->dZ1T, s->dZ2T, s->dZ1Tf, s->dZ2Tf, s->H2Tf, s->tb, s->dy, s->lossr, s->loss};
    for (void* q : ptrs)
        if (q) (void)hipFree(q);
    *s = og_sur{};
}

int og_sur_descriptors(og_sur* s, bool all) {
    if (s->n_tiles == 0) return 0;
    hipLaunchKernelGGL(og_k_tile_bounds, dim3(s->n_tiles), dim3(64), 0, s->stream, s->pos, s->tile_atom0,
                       s->tile_cnt, s->n_tiles, s->tile_bound, nullptr);
    DescArgs a{s->pos, s->rho, s->cls, s->tile_atom0, s->tile_cnt, s->tile_sys, s->sys_tile_b, s->sys_tile_e,
               s->tile_bound, all ? nullptr : s->mode, s->X};
    hipLaunchKernelGGL(og_k_sur_desc, dim3(s->n_tiles), dim3(64 * SUR_DESC_WAVES), 0, s->stream, a);
    return hipGetLastError() == hipSuccess ? 0 : fail("kernel launch failed");
}

int og_sur_infer(og_sur* s) {
    if (s->n_atoms == 0) return 0;
    hipLaunchKernelGGL(og_k_sur_infer, dim3((s->n_atoms + SUR_INFER_ROWS - 1) / SUR_INFER_ROWS), dim3(512), 0, s->stream, s->X, s->n_atoms,
                       s->n_pad, params_of(s), s->r_sur);
    return hipGetLastError() == hipSuccess ? 0 : fail("kernel launch failed");
}

int og_sur_collect(og_sur* s, const double* radii_dev) {
    const long long room = s->cap - s->n_train;
    const int n = (int)std::min<long long>(room, s->n_atoms);
    if (n <= 0) return 0;
    const long long tot = (long long)n * OG_SUR_K1;
    hipLaunchKernelGGL(og_k_sur_append, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s->stream, s->X,
                       radii_dev, n, s->Xtr, s->ttr, s->n_train);
    if (hipGetLastError() != hipSuccess) return fail("kernel launch failed");
    s->n_train += n;
    return 0;
}

int og_sur_train(og_sur* s, int n_steps, int batch, double lr, unsigned long long seed, float* loss_per_step) {
    if (n_steps > 0 && s->n_train <= 0) return fail("no training rows collected");
    if (n_steps > 0 && (batch < 32 || batch > OG_SUR_BMAX || batch % 32))
        return fail("batch must be a multiple of 32 in [32, 8192]");
    // the losses stay on the device and come back OG_SUR_LOSSES at a time: a
    // copy per step waited for every step
    for (int t = 0; t < n_steps; ++t) {
        const int slot = t % OG_SUR_LOSSES;
        s->adam_t += 1;
        const float c1 = (float)(1.0 - std::pow(0.9, s->adam_t)), c2 = (float)(1.0 - std::pow(0.999, s->adam_t));
        if (batch_gradient(s, s->Xtr, s->ttr, s->n_train, seed * 0x9E3779B97F4A7C15ull + (unsigned long long)t, batch,
                           nullptr, (float)lr, c1, c2, s->loss + slot))
            return -2;
        if (loss_per_step && (slot == OG_SUR_LOSSES - 1 || t == n_steps - 1) &&
            hipMemcpyAsync(loss_per_step + (t - slot), s->loss, (slot + 1) * sizeof(float), hipMemcpyDeviceToHost,
                           s->stream) != hipSuccess)
            return fail("copy failed");
    }
    return 0;
}

int og_sur_gradient(og_sur* s, const float* x, const float* r_target, int n, float* grad, double* loss) {
    if (n < 32 || n > OG_SUR_BMAX || n % 32) return fail("n must be a multiple of 32 in [32, 8192]");
    std::vector<unsigned short> xb((size_t)n * OG_SUR_K1, 0);
    std::vector<float> t(n);
    for (int b = 0; b < n; ++b) {
        for (int f = 0; f < OG_SUR_F; ++f) {
            xb[(size_t)b * OG_SUR_K1 + f] = f2bf(x[(size_t)b * OG_SUR_F + f]);
        }
        t[b] = (float)((r_target[b] - OG_SUR_R0) / OG_SUR_RS);
    }
    if (hipMemcpyAsync(s->Xb, xb.data(), xb.size() * 2, hipMemcpyHostToDevice, s->stream) != hipSuccess ||
        hipMemcpyAsync(s->tb, t.data(), t.size() * 4, hipMemcpyHostToDevice, s->stream) != hipSuccess)
        return fail("copy failed");
    if (batch_gradient(s, s->Xb, s->tb, 0, 0, n, s->g, 0.0f, 1.0f, 1.0f, s->loss)) return -2;
    float l = 0.0f;
    if (hipMemcpyAsync(grad, s->g, OG_SUR_P * sizeof(float), hipMemcpyDeviceToHost, s->stream) != hipSuccess ||
        hipMemcpyAsync(&l, s->loss, sizeof(float), hipMemcpyDeviceToHost, s->stream) != hipSuccess ||
        hipStreamSynchronize(s->stream) != hipSuccess)
        return fail("copy failed");
    if (loss) *loss = l;
    return 0;
}

int og_sur_set_params(og_sur* s, const float* p) {
    if (hipMemcpyAsync(s->p, p, OG_SUR_P * sizeof(float), hipMemcpyHostToDevice, s->stream) != hipSuccess)
        return fail("copy failed");
    if (refresh_copies(s)) return -2;
    return hipStreamSynchronize(s->stream) == hipSuccess ? 0 : fail("copy failed");
}

int og_sur_get_params(og_sur* s, float* p) {
    if (hipMemcpyAsync(p, s->p, OG_SUR_P * sizeof(float), hipMemcpyDeviceToHost, s->stream) != hipSuccess ||
        hipStreamSynchronize(s->stream) != hipSuccess)
        return fail("copy failed");
    return 0;
}

int og_sur_check_begin(og_sur* s) {
    hipLaunchKernelGGL(og_k_sur_zero, dim3((s->n_sys + 255) / 256), dim3(256), 0, s->stream, s->dev, s->n_sys);
    return hipGetLastError() == hipSuccess ? 0 : fail("kernel launch failed");
}

int og_sur_check_apply(og_sur* s) {
    hipLaunchKernelGGL(og_k_sur_fallback, dim3((s->n_sys + 255) / 256), dim3(256), 0, s->stream, s->mode, s->dev,
                       s->n_sys, (float)s->tol);
    return hipGetLastError() == hipSuccess ? 0 : fail("kernel launch failed");
}
