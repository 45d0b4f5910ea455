// replica_kernels.hpp -- thermal replicas of one cluster geometry.
//
// When every member of an ensemble is the same cluster (same positions,
// radii, anisotropy, axes, material and field) and only the Wiener stream
// (seed) and initial state differ, the dipolar field of all replicas at one
// Heun stage is one matrix product.  With the replica-major state
// Mt[r][3j+b] and the dipole tensor D[3i+a][3j+b] = w_j r_ij^-3 (3 u_a u_b -
// delta_ab) (lib/field.cpp:187-225; zero 3x3 blocks on the diagonal),
//   Ht[r][3i+a] = sum_k Mt[r][k] D[3i+a][k]
// i.e. Ht = Mt D^T.  Both MFMA operands are then "one row, consecutive k"
// reads of row-major matrices, and a wave's output lanes write consecutive
// columns of Ht.
//
// Columns are laid out component-blocked per 32 particles: particle i,
// component a sits in column 96 (i / 32) + 32 a + i % 32 (replica_col), with
// the particle count padded to a multiple of 64.  The same permutation is applied
// to both indices of D, so the product is unchanged; a 32-column MFMA tile then
// holds one component of 32 consecutive particles.
//
// State, field and increments are stored in tiles of 32 replicas x 32 columns, in
// the order in which a wave holds the tile as MFMA output with the tensor's rows as
// the first operand (replica_at): lane l holds replica l % 32 and, in its 16
// registers, particles 8 g + 4 (l / 32) + e.  The same 16 values in the same lane
// are a fragment of the second operand, for a sum over k in that order, which the
// tensor's fragments follow: what a lane computes is what it loads for the next
// product, every access is 16 bytes per lane and 1 KB per wave, and no operand goes
// through LDS.
//
// The product runs on MFMA in BF16 with the three-term split
// x = x_hi + x_lo (x_hi = bf16(x), x_lo = bf16(x - x_hi)):
//   Mt D^T ~ Mt_hi D_hi^T + Mt_hi D_lo^T + Mt_lo D_hi^T, FP32 accumulation,
// or in FP32 on MFMA, and the Heun stages run in its epilogue.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "sllg_kernels.hpp"

namespace mp {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kParticlePad = 64;   // particles per replica padded to a multiple of this
constexpr int kReplicaPad = 128;   // replicas padded to a multiple of this

__host__ __device__ inline int replica_col(int i, int a) { return 96 * (i >> 5) + 32 * a + (i & 31); }

// Place of (replica r, column c) in the state arrays: tiles of 1,024 values, rows
// of tiles along the columns.
__host__ __device__ inline size_t replica_at(int ld, int r, int c)
{
    const int p = c & 31, lane = (r & 31) + 32 * ((p >> 2) & 1);
    return (((size_t)(r >> 5) * (size_t)(ld >> 5) + (size_t)(c >> 5)) * 4 + (size_t)(p >> 3)) * 256 +
           (size_t)(4 * lane + (p & 3));
}

// Column of the tensor that lane l multiplies in slot j (0-7) of the product's step
// ks (16 columns): the state's particles in the order above.
__host__ __device__ inline int replica_k(int ks, int l, int j)
{
    return 32 * (ks >> 1) + 8 * (2 * (ks & 1) + (j >> 2)) + 4 * (l >> 5) + (j & 3);
}

// Place of part h (of two) of the tensor's fragments: particle block pb, step ks,
// component u; 64 lanes of 16 bytes from there.  BF16: part 0 is hi and part 1 lo of
// the eight slots of a lane; FP32: slots 0-3 and 4-7.
__host__ __device__ inline size_t replica_fragment(int ld, int pb, int ks, int u, int h)
{
    return ((((size_t)pb * (size_t)(ld >> 4) + (size_t)ks) * 3 + (size_t)u) * 2 + (size_t)h) * 64;
}

// ------------------------------------------------------------------ Heun stages
// Per-replica Heun stages around the product.  The applied field of the two stage
// times is uniform and passed in (h1, h2).
struct ReplicaArgs {
    int n;                  // particles per replica
    int reps;               // replicas
    int ld;                 // columns 3 Np (Np = n padded to a multiple of kParticlePad)
    int n_waves;            // waves in the grid (ensemble partial stride)
    const float *kex, *key, *kez, *edx, *edy, *edz;  // per particle: k e, e dt
    const float *sig;       // per particle: sr sqrt(dt)
    float dt, alpha;
    const uint32_t *key0, *key1;   // per replica Philox key (member seed)
    const double *msw;             // per replica Ms
    uint32_t tag;
    int renorm;
    float *m, *mt, *h;             // replica_at: state, predictor, field
    float *nz;                     // replica_at: the step's scaled Wiener increments (fused
                                   // product: stage 1 writes them, stage 2 reads them)
    uint32_t *status;              // [reps * n]
    // sampling
    const int64_t *sched;
    int64_t S;
    float *samples;                // [S][3][reps * n] or null
    double *ens_partial;           // [S][3][n_waves] or null
};

// Normals 3n, 3n+1, 3n+2 of particle p's stream under the Philox key
// (k0, k1) of its replica, scaled by sig: normal j is component j % 4 of
// Box-Muller over Philox call j / 4 (the stream of philox.h).  Only the
// Box-Muller pairs that hold the three are formed: the two of call 3n/4 when
// they start at component 0 or 1, else the second pair of that call and the
// first of the next.
__device__ inline void replica_normals(uint32_t k0, uint32_t k1, uint32_t tag, int p, int64_t n,
                                       float sig, float &sx, float &sy, float &sz)
{
    PhiloxKeys keys;
    keys.init(k0, k1);
    const uint64_t j0 = 3 * (uint64_t)n, c0 = j0 >> 2;
    const int o = (int)(j0 & 3);
    const u32x4 w = philox4x32_10(u32x4{(uint32_t)c0, (uint32_t)(c0 >> 32), (uint32_t)p, tag}, keys);
    float z0, z1, z2;
    if (o < 2) {
        float b0, b1, b2, b3;
        Num<float>::box_muller(w.x, w.y, b0, b1);
        Num<float>::box_muller(w.z, w.w, b2, b3);
        z0 = o == 0 ? b0 : b1;
        z1 = o == 0 ? b1 : b2;
        z2 = o == 0 ? b2 : b3;
    } else {
        const uint64_t c1 = c0 + 1;
        const u32x4 w1 =
            philox4x32_10(u32x4{(uint32_t)c1, (uint32_t)(c1 >> 32), (uint32_t)p, tag}, keys);
        float b2, b3, b4, b5;
        Num<float>::box_muller(w.z, w.w, b2, b3);
        Num<float>::box_muller(w1.x, w1.y, b4, b5);
        z0 = o == 2 ? b2 : b3;
        z1 = o == 2 ? b3 : b4;
        z2 = o == 2 ? b4 : b5;
    }
    sx = sig * z0;
    sy = sig * z1;
    sz = sig * z2;
}

// Per-particle constants of the stages: k e, e dt and sr sqrt(dt).
struct ReplicaParticle {
    float kex, key, kez, edx, edy, edz, sig;
};

__device__ inline ReplicaParticle replica_particle(const ReplicaArgs &a, int p)
{
    return ReplicaParticle{a.kex[p], a.key[p], a.kez[p], a.edx[p], a.edy[p], a.edz[p], a.sig[p]};
}

// The stage arithmetic of one (replica, particle) element from values
// already in registers: the field (hx, hy, hz) is the product's output,
// (sx, sy, sz) the step's scaled Wiener increments (replica_normals).  Both
// the fused epilogue and the elementwise kernels evaluate these same
// expressions.
// Stage 1: m~ = m + L(m, h dt + s).
__device__ inline void replica_stage1_math(const ReplicaArgs &a, const ReplicaParticle &c,
                                           float sx, float sy, float sz, float h1, float hx,
                                           float hy, float hz, float mx, float my, float mz,
                                           float &tx, float &ty, float &tz)
{
    const float dt = a.dt;
    const float d = mx * c.kex + my * c.key + mz * c.kez;
    const float vx = d * c.edx + (hx * dt + sx), vy = d * c.edy + (hy * dt + sy),
                vz = d * c.edz + ((hz + h1) * dt + sz);
    float ax, ay, az;
    llg_map(mx, my, mz, vx, vy, vz, a.alpha, ax, ay, az);
    tx = mx + ax;
    ty = my + ay;
    tz = mz + az;
}

// Stage 2: m' = m + (L(m, v1) + L(m~, v2)) / 2 with L(m, v1) = m~ - m,
// renormalised when asked.
__device__ inline void replica_stage2_math(const ReplicaArgs &a, const ReplicaParticle &c,
                                           float sx, float sy, float sz, float h2, float hx,
                                           float hy, float hz, float tx, float ty, float tz,
                                           float m0x, float m0y, float m0z, float &mx, float &my,
                                           float &mz)
{
    const float dt = a.dt;
    const float d = tx * c.kex + ty * c.key + tz * c.kez;
    const float vx = d * c.edx + (hx * dt + sx), vy = d * c.edy + (hy * dt + sy),
                vz = d * c.edz + ((hz + h2) * dt + sz);
    float bx, by, bz;
    llg_map(tx, ty, tz, vx, vy, vz, a.alpha, bx, by, bz);
    mx = m0x + 0.5f * ((tx - m0x) + bx);
    my = m0y + 0.5f * ((ty - m0y) + by);
    mz = m0z + 0.5f * ((tz - m0z) + bz);
    if (a.renorm) {
        const float nrm = sqrtf(mx * mx + my * my + mz * mz);
        mx = mx / nrm;
        my = my / nrm;
        mz = mz / nrm;
    }
}

// Flag a non-finite state.
__device__ inline void replica_check(const ReplicaArgs &a, int r, int p, float mx, float my,
                                     float mz)
{
    if (!(isfinite(mx) && isfinite(my) && isfinite(mz))) a.status[(size_t)r * a.n + p] |= 1u;
}

// Ht = Mt D^T, and in the epilogue kEpi the Heun stage 1 or 2 on the tile that the
// wave holds (kEpi 0: the field goes to a.h).  A pair of waves computes 32 particles
// (three tiles of D's rows, one per component) x 32 kT replicas; the two (kh) take
// alternate steps of 16 columns, so that 4,096 x 512 has two waves on each SIMD, and
// each finishes half of the tile from the sums of both (exchanged through LDS).  A
// block is kW x kW pairs, whose waves share operands in the CU's L1.  Operands go
// from memory to registers, a step of up to 10 KB per wave ahead, with no LDS and no
// barrier in the loop; the state is split to BF16 in registers.  Blocks are numbered
// so that the blocks one XCD runs (block ids b with equal b % 8) share panels: with
// row_panels, row panels of Mt (each XCD reads an eighth of Mt and all of D), else
// column panels of D.
//
// What bounds it (4,096 x 512, kW = kT = 2): 58 GFLOP of BF16 MFMA.  With operands
// of ordinary values the chip's power holds MFMA alone to 1,750-1,800 TFLOP/s (33 us;
// 24.5 on zeros) and a fed loop to about 1,130 (51 us), what a library product of
// 8,192^3 reaches.  The product with its field stored takes 55 us (44 on zeros);
// with both operands staged through LDS 61.4, the tensor alone 57.6, three steps
// ahead 56.9, one wave per SIMD with twice the tile 53.1 (but then nothing draws
// beside it, and the stages take longer alone).  With stage 1 61 us and with stage 2
// 66 in a trace; in a run 63.8 on average (70.7 with the operands through LDS and
// 4-byte accesses).
enum ReplicaMode { kReplicaBf16x3, kReplicaF32 };

template <int kMode, int kT>
struct ReplicaStep {
    f32x4 m[kT][2];    // state: replica tiles, groups 2 (ks % 2) and the next
    f32x4 d[3][2];     // tensor: component, part

    __device__ inline void load(const f32x4 *const state[kT], const f32x4 *tensor, int ks)
    {
#pragma unroll
        for (int t = 0; t < kT; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) m[t][h] = state[t][ks * 128 + h * 64];
#pragma unroll
        for (int u = 0; u < 3; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) d[u][h] = tensor[(ks * 6 + u * 2 + h) * 64];
    }

    __device__ inline void multiply(f32x16 acc[3][kT]) const
    {
        if constexpr (kMode == kReplicaBf16x3) {
            bf16x8 x[2][kT], y[3][2];
#pragma unroll
            for (int t = 0; t < kT; ++t)
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const float v = m[t][q >> 2][q & 3];
                    const __bf16 hi = (__bf16)v;
                    x[0][t][q] = hi;
                    x[1][t][q] = (__bf16)(v - (float)hi);
                }
#pragma unroll
            for (int u = 0; u < 3; ++u)
#pragma unroll
                for (int h = 0; h < 2; ++h) y[u][h] = __builtin_bit_cast(bf16x8, d[u][h]);
            // 3 kT independent accumulators between dependent instructions
#pragma unroll
            for (int term = 0; term < 3; ++term)
#pragma unroll
                for (int u = 0; u < 3; ++u)
#pragma unroll
                    for (int t = 0; t < kT; ++t)
                        acc[u][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            y[u][term == 1 ? 1 : 0], x[term == 2 ? 1 : 0][t], acc[u][t], 0, 0, 0);
        } else {
#pragma unroll
            for (int q = 0; q < 8; ++q)
#pragma unroll
                for (int u = 0; u < 3; ++u)
#pragma unroll
                    for (int t = 0; t < kT; ++t)
                        acc[u][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                            d[u][q >> 2][q & 3], m[t][q >> 2][q & 3], acc[u][t], 0, 0, 0);
        }
    }
};

template <int kMode, int kEpi, int kW, int kT>
static __global__ __launch_bounds__(128 * kW * kW, 2) void replica_product_kernel(
    const float *__restrict__ state, const f32x4 *__restrict__ tensor, ReplicaArgs a,
    int64_t n_step, float hstage, int64_t s_first, int n_rec, int n_row_blocks, int n_col_blocks,
    int row_panels)
{
    constexpr int kPairs = kW * kW;
    __shared__ f32x4 red[2 * kPairs][6 * kT * 64];
    __shared__ f32x4 constants[7][8 * kW];     // of the block's particles, four at a time
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), l = threadIdx.x & 63;
    const int kh = wave / kPairs, w = wave % kPairs, wr = w / kW, wc = w % kW;
    const int total = n_row_blocks * n_col_blocks;
    int logical = blockIdx.x;
    if (total % 8 == 0) logical = (blockIdx.x % 8) * (total / 8) + blockIdx.x / 8;
    const int cb = row_panels ? logical % n_col_blocks : logical / n_row_blocks;
    const int rb = row_panels ? logical / n_col_blocks : logical % n_row_blocks;
    const int rt0 = kT * (kW * rb + wr), pb = kW * cb + wc;   // first replica tile, particle block
    const int tiles = a.ld >> 5, steps = a.ld >> 4;
    if constexpr (kEpi != 0) {
        const float *src[7] = {a.kex, a.key, a.kez, a.edx, a.edy, a.edz, a.sig};
        if (wave == 0 && l < 32 * kW) {
            const int p = 32 * kW * cb + l;
#pragma unroll
            for (int c = 0; c < 7; ++c)
                reinterpret_cast<float *>(constants[c])[l] = src[c][p < a.n ? p : a.n - 1];
        }
    }
    // Each wave of the pair finishes half of the tile: of two replica tiles the one
    // kh, of one the groups 2 kh and 2 kh + 1 of four particles; the rest of its sums
    // goes to its partner.  i counts a wave's groups, 16 bytes a lane each.
    constexpr int kGroups = 2 * kT;
    const int rt = rt0 + (kT == 2 ? kh : 0), g0 = kT == 2 ? 0 : 2 * kh;
    const int r = 32 * rt + (l & 31);
    const size_t at0 = ((size_t)rt * tiles + 3 * (size_t)pb) * 256 + (size_t)(64 * g0 + l);
    auto place = [&](int u, int i) { return at0 + (size_t)(u * 256 + i * 64); };
    auto get = [&](const float *p, int u, int i) {
        return reinterpret_cast<const f32x4 *>(p)[place(u, i)];
    };
    auto put = [&](float *p, int u, int i, const f32x4 &v) {
        reinterpret_cast<f32x4 *>(p)[place(u, i)] = v;
    };
    // particles of group i, counted in groups of four from the block's first
    auto quad = [&](int i) { return 8 * wc + 2 * (g0 + i) + (l >> 5); };
    const int rk = r < a.reps ? r : 0;
    // Stage 1 draws the step's increments and stores them for both stages: one wave
    // of a tile before its sums and the other after them, so that on each SIMD one
    // draws (VALU) while the other multiplies: stage 1 of 4,096 x 512 70.7 -> 61.3 us.
    auto draw = [&]() {
        const uint32_t key0 = a.key0[rk], key1 = a.key1[rk];
#pragma unroll
        for (int i = 0; i < kGroups; ++i) {
            const f32x4 sig = constants[6][quad(i)];
            f32x4 inc[3];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float z[3];
                replica_normals(key0, key1, a.tag, 32 * kW * cb + 4 * quad(i) + e, n_step, sig[e],
                                z[0], z[1], z[2]);
#pragma unroll
                for (int u = 0; u < 3; ++u) inc[u][e] = z[u];
            }
#pragma unroll
            for (int u = 0; u < 3; ++u) put(a.nz, u, i, inc[u]);
        }
    };
    if constexpr (kEpi == 1) {
        __syncthreads();   // the particles' constants
        if (kh == 1) draw();
    }
    const f32x4 *st[kT];
#pragma unroll
    for (int t = 0; t < kT; ++t)
        st[t] = reinterpret_cast<const f32x4 *>(state) + (size_t)(rt0 + t) * tiles * 256 + l;
    const f32x4 *dt0 = tensor + replica_fragment(a.ld, pb, 0, 0, 0) + l;
    f32x16 acc[3][kT];
#pragma unroll
    for (int u = 0; u < 3; ++u)
#pragma unroll
        for (int t = 0; t < kT; ++t)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[u][t][q] = 0.f;
    // this wave's steps kh, kh + 2, ...: an even number (ld is a multiple of 192), each
    // loaded while the one before is multiplied (the scheduler would otherwise move
    // the loads down to their use); the load past the last is of the first step
    ReplicaStep<kMode, kT> f[2];
    const int mine = steps / 2;
    f[0].load(st, dt0, kh);
    for (int i = 0; i < mine; i += 2) {
        f[1].load(st, dt0, 2 * (i + 1) + kh);
        __builtin_amdgcn_sched_barrier(0);
        f[0].multiply(acc);
        f[0].load(st, dt0, 2 * (i + 2 < mine ? i + 2 : 0) + kh);
        __builtin_amdgcn_sched_barrier(0);
        f[1].multiply(acc);
    }
    f32x4 m[3][kGroups], mt[3][kGroups], nz[3][kGroups];
    auto load_half = [&](int half) {
#pragma unroll
        for (int j = 0; j < kT; ++j)
#pragma unroll
            for (int u = 0; u < 3; ++u) {
                const int i = half * kT + j;
                m[u][i] = get(a.m, u, i);
                nz[u][i] = get(a.nz, u, i);
                if constexpr (kEpi == 2) mt[u][i] = get(a.mt, u, i);
            }
    };
    if constexpr (kEpi == 1) {
        if (kh == 0) draw();
    }
    if constexpr (kEpi != 0) load_half(0);
    // the sum of group i, component u, of this wave (own) or its partner's groups
    auto sum = [&](bool own, int u, int i, int e) {
        const float first = acc[u][0][4 * i + e];
        const float second = kT == 2 ? acc[u][kT - 1][4 * i + e] : acc[u][0][8 + 4 * i + e];
        return (kh != 0) == own ? second : first;
    };
#pragma unroll
    for (int u = 0; u < 3; ++u)
#pragma unroll
        for (int i = 0; i < kGroups; ++i) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = sum(false, u, i, e);
            red[wave][(u * kGroups + i) * 64 + l] = v;
        }
    __syncthreads();
    const f32x4 *theirs = &red[kh ? wave - kPairs : wave + kPairs][l];
    double ex = 0.0, ey = 0.0, ez = 0.0;
    double msw = 0.0;
    if constexpr (kEpi == 2) msw = n_rec > 0 ? a.msw[rk] : 0.0;
#pragma unroll
    for (int i = 0; i < kGroups; ++i) {
        if constexpr (kEpi != 0)
            if (i == kT - 1) load_half(1);
        f32x4 h[3];
#pragma unroll
        for (int u = 0; u < 3; ++u) {
            h[u] = theirs[(u * kGroups + i) * 64];
#pragma unroll
            for (int e = 0; e < 4; ++e) h[u][e] += sum(true, u, i, e);
        }
        if constexpr (kEpi == 0) {
#pragma unroll
            for (int u = 0; u < 3; ++u) put(a.h, u, i, h[u]);
            continue;
        }
        f32x4 c[7], out[3];
#pragma unroll
        for (int k = 0; k < 7; ++k) c[k] = constants[k][quad(i)];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int p = 32 * kW * cb + 4 * quad(i) + e;
            const ReplicaParticle cp{c[0][e], c[1][e], c[2][e], c[3][e], c[4][e], c[5][e], c[6][e]};
            float x[3];
            if constexpr (kEpi == 1) {
                replica_stage1_math(a, cp, nz[0][i][e], nz[1][i][e], nz[2][i][e], hstage, h[0][e],
                                    h[1][e], h[2][e], m[0][i][e], m[1][i][e], m[2][i][e], x[0],
                                    x[1], x[2]);
            } else {
                replica_stage2_math(a, cp, nz[0][i][e], nz[1][i][e], nz[2][i][e], hstage, h[0][e],
                                    h[1][e], h[2][e], mt[0][i][e], mt[1][i][e], mt[2][i][e],
                                    m[0][i][e], m[1][i][e], m[2][i][e], x[0], x[1], x[2]);
            }
            const bool live = r < a.reps && p < a.n;
            if constexpr (kEpi == 2) {
                if (live) replica_check(a, r, p, x[0], x[1], x[2]);
                if (n_rec > 0 && live) {
                    ex += (double)x[0] * msw;
                    ey += (double)x[1] * msw;
                    ez += (double)x[2] * msw;
                    if (a.samples != nullptr) {
                        const size_t P = (size_t)a.n * a.reps, at = (size_t)r * a.n + p;
                        for (int k = 0; k < n_rec; ++k) {
                            float *base = a.samples + (size_t)(s_first + k) * 3 * P;
                            base[at] = x[0];
                            base[P + at] = x[1];
                            base[2 * P + at] = x[2];
                        }
                    }
                }
            }
            // the padding stays zero: it is an operand of the next product
#pragma unroll
            for (int u = 0; u < 3; ++u) out[u][e] = live ? x[u] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 3; ++u) put(kEpi == 1 ? a.mt : a.m, u, i, out[u]);
    }
    if constexpr (kEpi == 2) {
        if (n_rec > 0 && a.ens_partial != nullptr) {
            wave_sum3<float>(ex, ey, ez);
            if constexpr (kT == 1) {   // one partial per 32 replicas x 32 particles
                __shared__ double half[kPairs][3];
                if (kh == 1 && l == 0) {
                    half[w][0] = ex;
                    half[w][1] = ey;
                    half[w][2] = ez;
                }
                __syncthreads();
                ex += half[w][0];
                ey += half[w][1];
                ez += half[w][2];
            }
            if (l == 0 && (kT == 2 || kh == 0)) {
                const int wid = rt * (tiles / 3) + pb;
                for (int k = 0; k < n_rec; ++k) {
                    double *dst = a.ens_partial + (size_t)(s_first + k) * 3 * (size_t)a.n_waves;
                    dst[wid] = ex;
                    dst[(size_t)a.n_waves + wid] = ey;
                    dst[2 * (size_t)a.n_waves + wid] = ez;
                }
            }
        }
    }
}

// FP64 product on the VALU, one output per lane, of row-major matrices (reference
// for tests).
static __global__ void gemm_f64_kernel(const double *__restrict__ a, const double *__restrict__ b,
                                double *__restrict__ c, int rows, int cols, int K)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * cols) return;
    const int r = i / cols, col = i % cols;
    double s = 0.0;
    for (int k = 0; k < K; ++k) s += a[(size_t)r * K + k] * b[(size_t)col * K + k];
    c[(size_t)r * cols + col] = s;
}

// The stages as elementwise kernels around an unfused product: a thread per
// (replica, particle), in the order of replica_at.
struct ReplicaElement {
    int r, p;
    size_t at;     // of the x component; y and z are 1,024 and 2,048 further
    bool live;
    __device__ explicit ReplicaElement(const ReplicaArgs &a)
    {
        const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
        const int in = (int)(i & 1023), lane = (in >> 2) & 63, blocks = a.ld / 96;
        const int tile = (int)(i >> 10), pb = tile % blocks;
        r = 32 * (tile / blocks) + (lane & 31);
        p = 32 * pb + 8 * (in >> 8) + 4 * (lane >> 5) + (in & 3);
        at = ((size_t)(tile / blocks) * (size_t)(a.ld >> 5) + 3 * (size_t)pb) * 1024 + (size_t)in;
        live = r < a.reps && p < a.n;
    }
};

static __global__ __launch_bounds__(256) void replica_stage1_kernel(ReplicaArgs a, int64_t n_step, float h1)
{
    const ReplicaElement x(a);
    if (!x.live) return;
    const size_t y = x.at + 1024, z = x.at + 2048;
    const ReplicaParticle c = replica_particle(a, x.p);
    float sx, sy, sz, tx, ty, tz;
    replica_normals(a.key0[x.r], a.key1[x.r], a.tag, x.p, n_step, c.sig, sx, sy, sz);
    replica_stage1_math(a, c, sx, sy, sz, h1, a.h[x.at], a.h[y], a.h[z], a.m[x.at], a.m[y], a.m[z],
                        tx, ty, tz);
    a.mt[x.at] = tx;
    a.mt[y] = ty;
    a.mt[z] = tz;
}

// stage 2 and the samples s_first .. s_first + n_rec - 1 (all recorded after
// this step)
static __global__ __launch_bounds__(256) void replica_stage2_kernel(ReplicaArgs a, int64_t n_step, float h2,
                                                             int64_t s_first, int n_rec)
{
    const ReplicaElement x(a);
    const size_t yy = x.at + 1024, zz = x.at + 2048;
    const int p = x.live ? x.p : 0, r = x.live ? x.r : 0;
    const ReplicaParticle c = replica_particle(a, p);
    float sx, sy, sz, mx, my, mz;
    replica_normals(a.key0[r], a.key1[r], a.tag, p, n_step, c.sig, sx, sy, sz);
    replica_stage2_math(a, c, sx, sy, sz, h2, a.h[x.at], a.h[yy], a.h[zz], a.mt[x.at], a.mt[yy],
                        a.mt[zz], a.m[x.at], a.m[yy], a.m[zz], mx, my, mz);
    if (x.live) {
        a.m[x.at] = mx;
        a.m[yy] = my;
        a.m[zz] = mz;
        replica_check(a, r, p, mx, my, mz);
    }
    for (int k = 0; k < n_rec; ++k) {
        const int64_t s = s_first + k;
        if (a.samples != nullptr && x.live) {
            const size_t P = (size_t)a.n * a.reps, i = (size_t)r * a.n + p;
            float *base = a.samples + (size_t)s * 3 * P;
            base[i] = mx;
            base[P + i] = my;
            base[2 * P + i] = mz;
        }
        if (a.ens_partial != nullptr) {
            double ex = x.live ? (double)mx * a.msw[r] : 0.0;
            double ey = x.live ? (double)my * a.msw[r] : 0.0;
            double ez = x.live ? (double)mz * a.msw[r] : 0.0;
            wave_sum3<float>(ex, ey, ez);
            if ((threadIdx.x & (kWave - 1)) == 0) {
                const int wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
                double *dst = a.ens_partial + (size_t)s * 3 * (size_t)a.n_waves;
                dst[wave] = ex;
                dst[(size_t)a.n_waves + wave] = ey;
                dst[2 * (size_t)a.n_waves + wave] = ez;
            }
        }
    }
}

// The states of the live (replica, particle) elements as [reps n][3].
static __global__ __launch_bounds__(256) void replica_pack_kernel(ReplicaArgs a, float *out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n * a.reps) return;
    const size_t at = replica_at(a.ld, i / a.n, replica_col(i % a.n, 0));
#pragma unroll
    for (int d = 0; d < 3; ++d) out[3 * (size_t)i + d] = a.m[at + 1024 * (size_t)d];
}

}  // namespace mp
