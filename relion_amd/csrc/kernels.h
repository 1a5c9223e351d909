// Device kernels of the plain-FP32 E-step for CDNA4 (gfx950). Included by estep.hip only.
//
// Image geometry: an s x (s/2+1) half-complex image, pixel p = i*(s/2+1) + x, frequency
// (x, y) with y = i for i <= s/2 else i - s (FOR_ALL_ELEMENTS_IN_FFTW_TRANSFORM, src/fftw.h:99-102).
// Volume geometry: projector layout of src/projector.cpp:59-89, interleaved float2 [z][y][x].
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"

namespace rlnk {

// Whether any base voxel of brick br lies within squared distance reach2 of the origin.
__device__ __forceinline__ bool brick_in_reach(const VolGeom &g, int bx, int by, int bz, long long reach2) {
    constexpr int e = (1 << kBrickLog) - 1;
    const long long x = bx << kBrickLog;
    const int y0 = (by << kBrickLog) + g.starty, z0 = (bz << kBrickLog) + g.startz;
    const long long y = y0 > 0 ? y0 : y0 + e < 0 ? y0 + e : 0, z = z0 > 0 ? z0 : z0 + e < 0 ? z0 + e : 0;
    return x * x + y * y + z * z <= reach2;
}

// Builds the corner-packed volume from the plain [z][y][x] float2 volume: four lanes per base voxel, one 16-byte quarter
// (an x pair of corners) each, so that the stores of a wave are 1 KB of consecutive memory; kPackBricks bricks of 64
// base voxels per block, their loads in flight together. Bricks beyond squared radius reach2, where the plain volume
// is zero, are not read: they are cleared if clear_far, else they hold zeros already.
// Bound by the write of the packed volume: 2.3 GB of it in reach at box 256, 0.83 to 0.93 ms (a thread per base voxel, whose
// 64-byte stores lie 64 bytes apart, and every brick written: 1.85 ms).
constexpr int kPackBricks = 4;
__global__ void __launch_bounds__(kBlock) k_pack_volume(const float2 *__restrict__ plain, VolGeom g, long long reach2,
                                                        int clear_far, float4 *__restrict__ packed) {
    const int nx = brick_count(g.xdim), ny = brick_count(g.ydim), nz = brick_count(g.zdim);
    const int base = threadIdx.x >> 2, q = threadIdx.x & 3;
    const size_t row = (size_t)g.xdim, slab = row * (size_t)g.ydim;
    float2 lo[kPackBricks], hi[kPackBricks];
    bool on[kPackBricks];
#pragma unroll
    for (int u = 0; u < kPackBricks; ++u) {
        const int br = blockIdx.x * kPackBricks + u;
        const int bx = br % nx, by = (br / nx) % ny, bz = br / (nx * ny);
        const int x0 = 4 * bx + (base & 3), y0 = 4 * by + ((base >> 2) & 3), z0 = 4 * bz + (base >> 4);
        lo[u] = hi[u] = make_float2(0.f, 0.f);
        const bool far = !brick_in_reach(g, bx, by, bz, reach2);
        on[u] = bz < nz && x0 < g.xdim - 1 && y0 < g.ydim - 1 && z0 < g.zdim - 1 && (!far || clear_far);
        if (far || !on[u]) continue;
        const float2 *p = plain + (size_t)(z0 + (q >> 1)) * slab + (size_t)(y0 + (q & 1)) * row + x0;
        lo[u] = p[0];
        hi[u] = p[1];
    }
#pragma unroll
    for (int u = 0; u < kPackBricks; ++u)
        if (on[u])
            packed[((size_t)blockIdx.x * kPackBricks + u) * kBlock + threadIdx.x] =
                make_float4(lo[u].x, lo[u].y, hi[u].x, hi[u].y);
}
static_assert(kBrickLog == 2 && kBlock == 256, "k_pack_volume: 64 base voxels of 4 lanes per block");

// Backprojection accumulators in corner slots: per base voxel 32 floats = one 128-byte line,
// [re c0..c7 | im c0..c7 | weight c0..c7 | unused], corner c = 4*dz + 2*dy + dx. All 24 atomics of one
// trilinear scatter land in one line, so a wave's atomic instruction can be served line by line.
// k_fold_slots sums the slots into plain volumes.
constexpr int kSlot = 32;

// Base voxels that a backprojection can reach: samples lie within rr = xdim - 2 of the origin (the projector's
// dimensions are those of that radius), their base voxels within rr + sqrt(3). All other slots stay zero.
__host__ __device__ __forceinline__ long long slot_reach2(const VolGeom &g) {
    return (long long)g.xdim * g.xdim;  // (rr + 2)^2
}

// Zeroes the slots within reach (the others are zero from the allocation on). One brick of 64 base voxels (8 KB) per
// step of a block. Half of the box-256 slots (8.7 GB) lie in reach: 1.1 ms, all of them 2.0.
__global__ void __launch_bounds__(kBlock) k_zero_slots(float4 *__restrict__ slots, VolGeom g) {
    const int nx = brick_count(g.xdim), ny = brick_count(g.ydim), nz = brick_count(g.zdim);
    const int n = nx * ny * nz;
    const long long reach = slot_reach2(g);
    for (int br = blockIdx.x; br < n; br += gridDim.x) {
        const int bx = br % nx, by = (br / nx) % ny, bz = br / (nx * ny);
        if (!brick_in_reach(g, bx, by, bz, reach)) continue;
        float4 *p = slots + (size_t)br * (kSlot / 4 << 3 * kBrickLog);
        for (int i = threadIdx.x; i < kSlot / 4 << 3 * kBrickLog; i += kBlock) p[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
}

// Plain data/weight volumes from the slots: v(z,y,x) = sum over corners c (in order) of slot[base(z,y,x) - c][c], for
// planes [z0, z0 + nz); the outputs start at plane z0. A block marches along z over kFoldZ planes of a 16 x 16 tile: the
// slots of the 17 x 17 base voxels of a plane are staged in LDS (24 values each, the next plane's in registers
// meanwhile), each thread forms the lower (dz = 0) part of its voxel and carries the upper one (dz = 1) to the next
// plane. So every slot is read 1.16 times (tile and chunk edges), against 1.95 for a 4 x 4 x 4 brick per block, and
// those out of reach not at all. Bound by the read of the slots: 4.7 GB in 1.66 ms at box 256 (a brick per block: 8.7 GB,
// 5.2 ms).
constexpr int kFoldT = 16, kFoldZ = 32;
__global__ void __launch_bounds__(kBlock) k_fold_slots(const float4 *__restrict__ slots, VolGeom g, int z0, int nz,
                                                       float *__restrict__ re, float *__restrict__ im,
                                                       float *__restrict__ w) {
    constexpr int kB = kFoldT + 1, kN = kB * kB, kQ = (6 * kN + kBlock - 1) / kBlock;
    __shared__ float s[24][kN];  // [re c0..7 | im c0..7 | weight c0..7][base]; the row length 289 spreads the banks
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    const int bx = kFoldT * blockIdx.x, by = kFoldT * blockIdx.y;
    const int za = z0 + kFoldZ * (int)blockIdx.z, zb = min(za + kFoldZ, z0 + nz);
    const long long reach = slot_reach2(g);
    float4 q[kQ];
    auto load = [&](int z) {
#pragma unroll
        for (int i = 0; i < kQ; ++i) {
            const int u = tid + i * kBlock, base = u / 6;
            q[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            const int x0 = bx - 1 + base % kB, y0 = by - 1 + base / kB;
            if (u >= 6 * kN || x0 < 0 || y0 < 0 || z < 0 || x0 >= g.xdim - 1 || y0 >= g.ydim - 1 || z >= g.zdim - 1)
                continue;
            const long long ly = y0 + g.starty, lz = z + g.startz;
            if ((long long)x0 * x0 + ly * ly + lz * lz > reach) continue;
            q[i] = slots[(kSlot / 4) * packed_index(g, x0, y0, z) + u - 6 * base];
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int i = 0; i < kQ; ++i) {
            const int u = tid + i * kBlock, base = u / 6, f = 4 * (u - 6 * base);
            if (u >= 6 * kN) continue;
            s[f][base] = q[i].x;
            s[f + 1][base] = q[i].y;
            s[f + 2][base] = q[i].z;
            s[f + 3][base] = q[i].w;
        }
    };
    const int x = bx + tx, y = by + ty;
    const bool inside = x < g.xdim && y < g.ydim;
    float carry[3] = {0.f, 0.f, 0.f};
    load(za - 1);
    for (int z = za - 1; z < zb; ++z) {
        stage();
        __syncthreads();
        if (z + 1 < zb) load(z + 1);
        float lo[3], hi[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) lo[k] = hi[k] = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {  // base (x - dx, y - dy) is local (tx + 1 - dx, ty + 1 - dy)
            const int base = (tx + 1 - (c & 1)) + kB * (ty + 1 - (c >> 1));
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                lo[k] += s[8 * k + c][base];
                hi[k] += s[8 * k + 4 + c][base];
            }
        }
        if (z >= za && inside) {
            const size_t o = ((size_t)(z - z0) * g.ydim + y) * g.xdim + x;
            re[o] = lo[0] + carry[0];
            im[o] = lo[1] + carry[1];
            w[o] = lo[2] + carry[2];
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) carry[k] = hi[k];
        __syncthreads();
    }
}

// Grid of k_fold_slots for nz planes.
inline dim3 fold_grid(const VolGeom &g, int nz) {
    return dim3((g.xdim + kFoldT - 1) / kFoldT, (g.ydim + kFoldT - 1) / kFoldT, (nz + kFoldZ - 1) / kFoldZ);
}


// --------------------------------------------------------------------------------------------------
// Coarse pass
// --------------------------------------------------------------------------------------------------

// Orientations of one block of the coarse kernel (16 per wave).
constexpr int kCoTO = 64;

struct CoarseTile {
    int b;        // particle within the batch
    int o_begin;  // first orientation (within the particle's list)
};

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

// round-to-nearest-even FP32 -> BF16 bit pattern
__device__ __forceinline__ unsigned short f2bf(float x) {
    unsigned int u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}
__device__ __forceinline__ bf16x8_t load_bf16x8(const unsigned short *p) {
    return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4 *>(p));
}

// Lane layout of v_mfma_f32_16x16x32_bf16, which the pose proposal's kernels use: lane l supplies row l%16 of
// A and column l%16 of B, each with the 8 consecutive k = 8*(l/16) .. 8*(l/16)+7; it receives D rows
// 4*(l/16) .. 4*(l/16)+3 of column l%16.
__global__ void k_selftest_mfma(const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ D) {
    const int l = threadIdx.x;
    unsigned short a[8], b[8];
    for (int j = 0; j < 8; ++j) {
        a[j] = f2bf(A[(l % 16) * 32 + 8 * (l / 16) + j]);
        b[j] = f2bf(B[(8 * (l / 16) + j) * 16 + l % 16]);
    }
    floatx4_t acc = {0.f, 0.f, 0.f, 0.f};
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load_bf16x8(a), load_bf16x8(b), acc, 0, 0, 0);
    for (int j = 0; j < 4; ++j) D[(4 * (l / 16) + j) * 16 + l % 16] = acc[j];
}

// --------------------------------------------------------------------------------------------------
// Coarse squared differences (getAllSquaredDifferences, src/ml_optimiser.cpp:7430-7442):
//   diff2(o,t) = Xi2/2 + sum_p |c_p P_o(p) - y_t(p)|^2,  y_t(p) = q_p X(p) E_t(p),  c_p = q_p ctf_p s,
// with E_t(x, y) = exp(-2 pi i (x tx + y ty) / N) and |y_t| = |q X|, expanded to
//   Xi2/2 + sum |q X|^2 (FP64, per particle) + sum c^2 |P|^2 (per orientation) - 2 cross(o,t),
//   cross(o,t) = sum_p Re(conj(A_o(p)) E_t(p)),  A = P conj(w),  w = c q X.
// The translations lie on a lattice, so E factors into an x and a y phase and the cross term into two short
// contractions instead of one over all pixels for every translation: with A = a + i b, cx + i sx the x phase of tx and
// cy + i sy the y phase of ty,
//   U(y,tx) = sum_x a cx + b sx,  V(y,tx) = sum_x b cx - a sx,  cross = sum_y cy U + sy V.
// Opposite shifts share their sums (cos is even, sin odd): the x contraction is the real matrix product of the rows a
// and b with the columns cos(tx), sin(tx), tx > 0, on the matrix units; rows y and -y are added and subtracted
// before the y contraction, which runs in registers on each lane's tx.
//
// Pixel layout of that contraction: per row pair (y, -y), y = 0 .. s/2, steps of 16 complex slots: 8 consecutive x of
// row y, then the same 8 of row -y (zeros where there is no such row); a pair has steps up to its last pixel whose
// Minvsigma2 is non-zero, so rows and corners that carry no weight are not contracted. An empty step makes their number
// even. grp holds (row, x0) of every 8 slots (row -1: zeros). Kc = 16 * steps complex slots per projection.
// --------------------------------------------------------------------------------------------------

// Arithmetic of the contraction, by the precision setting.
//   double (RLN_PREC_PLAIN_FP32): the difference of the three sums loses what they have in common, so with FP32 sums the
//     error of diff2 follows the signal's power, where sums of squared FP32 differences follow diff2 itself. With FP64
//     operands, products and sums the expansion is exact to FP64, and the FP32 projections, images and stored diff2 are
//     what is left, as in the differences.
//   float (RLN_PREC_SPLIT_BF16): FP32 products and sums, the particle's power in FP64.
// The FP64 matrix product returns row g + 4 r in register r of lane group g, the FP32 one row 4 g + r (k_selftest_lattice).
typedef double doublex4_t __attribute__((ext_vector_type(4)));
// Tables read at wave-uniform addresses, in the constant address space: scalar loads, which do not queue behind the
// projection values in flight.
typedef const __attribute__((address_space(4))) float *UniformF;
typedef const __attribute__((address_space(4))) double *UniformD;
typedef const __attribute__((address_space(4))) int *UniformI;
template <typename T>
struct Lattice;
template <>
struct Lattice<float> {
    typedef float2 Pair;
    typedef floatx4_t Acc;
    typedef UniformF Uniform;
    static __device__ __forceinline__ Acc mfma(float a, float b, Acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int g, int r) { return 4 * g + r; }
    static __device__ __forceinline__ int reg(int row) { return row & 3; }
    static __device__ __forceinline__ int group(int row) { return row >> 2; }
};
template <>
struct Lattice<double> {
    typedef double2 Pair;
    typedef doublex4_t Acc;
    typedef UniformD Uniform;
    static __device__ __forceinline__ Acc mfma(double a, double b, Acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int g, int r) { return g + 4 * r; }
    static __device__ __forceinline__ int reg(int row) { return row >> 2; }
    static __device__ __forceinline__ int group(int row) { return row & 3; }
};

// D (16 x 16, row-major) = A (16 x 4) B (4 x 16) by one matrix instruction of the contraction: lane l supplies row or
// column l % 16 at k = l / 16 and receives its four rows of column l % 16.
template <typename T>
__global__ void k_selftest_lattice(const T *__restrict__ A, const T *__restrict__ B, T *__restrict__ D) {
    const int l = threadIdx.x, n = l & 15, g = l >> 4;
    typename Lattice<T>::Acc acc = {0, 0, 0, 0};
    acc = Lattice<T>::mfma(A[n * 4 + g], B[g * 16 + n], acc);
    for (int r = 0; r < 4; ++r) D[Lattice<T>::row(g, r) * 16 + n] = acc[r];
}

// Projections of every coarse orientation of every class in that layout: FP32 complex pf [K*n_or][Kc].
// grid (K*n_or, ceil(Kc/256)).
__global__ void __launch_bounds__(kBlock) k_project_grid(const float4 *const *__restrict__ vols, VolGeom vg,
                                                         const Frame *__restrict__ frames, int n_or, ImgGeom ig,
                                                         const int2 *__restrict__ grp, int Kc, float2 *__restrict__ pf) {
    const int idx = blockIdx.y * kBlock + threadIdx.x;  // complex slot 8g + j
    const int ko = blockIdx.x;
    if (idx >= Kc) return;
    const int2 gr = grp[idx >> 3];
    const int x = gr.y + (idx & 7), i = gr.x;
    const int y = (i < ig.xs) ? i : i - ig.s;
    float2 v = make_float2(0.f, 0.f);
    if (i >= 0 && x < ig.xs && x * x + y * y <= ig.proj_r2_max) {
        const int k = ko / n_or, o = ko - k * n_or;
        v = project_pixel(vols[k], vg, frames[o], x, y);
    }
    pf[(size_t)ko * Kc + idx] = v;
}

// Particle side in that layout: w[b][slot] = c_p q_p X(p), ctf2[b][slot] = c_p^2, and ynorm[b] = sum_p |q_p X(p)|^2
// over all pixels (summed in FP64). grid (ceil(max(Kc, P)/256), B).
template <typename T>
__global__ void __launch_bounds__(kBlock) k_prep_coarse(const float2 *__restrict__ fimg, const float *__restrict__ fctf,
                                                        const float *__restrict__ scale, int sf, int Pf, ImgGeom ig,
                                                        const float *__restrict__ q, const int2 *__restrict__ grp,
                                                        int Kc, int do_ctf, typename Lattice<T>::Pair *__restrict__ w,
                                                        T *__restrict__ ctf2, double *__restrict__ ynorm) {
    __shared__ double red[kBlock / 64];
    const int idx = blockIdx.x * kBlock + threadIdx.x;
    const int b = blockIdx.y;
    const T sc = scale[b];
    auto src_of = [&](int i, int x) {
        const int y = (i < ig.xs) ? i : i - ig.s;
        const int isrc = (y < 0) ? y + sf : y;
        return (size_t)b * Pf + (size_t)isrc * (sf / 2 + 1) + x;
    };
    if (idx < Kc) {
        const int2 gr = grp[idx >> 3];
        const int x = gr.y + (idx & 7), i = gr.x;
        typename Lattice<T>::Pair v;
        v.x = v.y = 0;
        T c2 = 0;
        if (i >= 0 && x < ig.xs) {
            const size_t src = src_of(i, x);
            const T qp = q[i * ig.xs + x];
            const T c = qp * (T)(do_ctf ? fctf[src] : 1.f) * sc;
            const float2 X = fimg[src];
            v.x = c * qp * (T)X.x;
            v.y = c * qp * (T)X.y;
            c2 = c * c;
        }
        w[(size_t)b * Kc + idx] = v;
        ctf2[(size_t)b * Kc + idx] = c2;
    }
    T yn = 0;
    if (idx < ig.P) {
        const int i = idx / ig.xs, x = idx - i * ig.xs;
        const T qp = q[idx];
        const float2 X = fimg[src_of(i, x)];
        yn = qp * qp * ((T)X.x * (T)X.x + (T)X.y * (T)X.y);
    }
    double s = yn;
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double t = red[0] + red[1] + red[2] + red[3];
        if (t != 0.) atomicAdd(&ynorm[b], t);
    }
}

// Per-particle state of the coarse weights and significance selection (k_wpart_init .. k_wsel_stats); the coarse
// kernel already folds its minimum diff2 into mn_bits.
struct WPart {
    unsigned int mn_bits;   // min diff2 (non-negative float bits)
    int status;
    double sum;             // sum of weights
    double target;          // adaptive_fraction * sum
    unsigned long long prefix, mask;  // radix selection state: the crossing bin's leading bits
    double above_sum;       // weights in bins above the crossing bin
    long long above_cnt;
    double dcut;            // entries with diff2 - min above it weigh less than every element of the crossing bin
    unsigned long long seen; // bits of the largest weight some finished segment has seen (a lower bound on the sum)
    int state;              // kSel*
    int ncand;
    double thr;             // significance threshold
    long long nr_sign;
    long long n_above;      // entries >= thr
};
// Selection state of a particle: crossing bin not fine enough yet; every entry from the crossing bin up fits the
// candidate list; only the crossing bin does; no weights (zero or NaN sum).
constexpr int kSelRefine = 0, kSelAll = 1, kSelBin = 2, kSelNone = 3;

// Columns of the x contraction: 16 lanes hold one signed x shift each, tx = +(n + 1) on lane n < 8 (matrix column
// cos) and -(n - 7) on lane n >= 8 (column sin), counted from kColShift * tile; where a tile
// has fewer than 8 positive shifts, lane 7 is tx = 0 (in the last tile) and lane 15 unused.
struct CoarseColumn {
    int t0;    // translation index of (tx, ty = 0)
    int half;  // ty = -half .. half exist, -1: no column
};
constexpr int kColShift = 8;
constexpr int kStepMinus = 1, kStepEnd = 2;  // the step has a row -y; it is the last of its row pair
constexpr int kStepChunk = 64;               // steps whose particle rows are staged in LDS at a time (even)

template <typename T>
struct CoarseArgs {
    typedef typename Lattice<T>::Pair Pair;
    const CoarseTile *tiles;
    const int *or_off, *or_cnt, *or_proj;
    const float2 *pf;         // projections [K*n_or][Kc]
    const float2 *zero_row;   // [Kc] zeros
    const Pair *w;            // [b][Kc]
    const T *ctf2;            // [b][Kc]
    const double *ynorm;
    const float *xi2half;
    const long long *d2_off;
    const int2 *steps;        // [n_steps] (offset of the step's x phases in xtab, flags: kStepMinus | kStepEnd)
    const T *ytab;            // per row pair: cos(2 pi y ty / N) for ty = 0 .. M, -sin for ty = 1 .. M
    const Pair *xtab;         // [column tile][step of a row][lane]: the two x phases of the lane's column
    const CoarseColumn *cols; // [column tile][16], then the tx = 0 column of M == 8
    const int *tile_of;       // column tile of each translation, null with one tile
    int n_steps, n_xsteps;    // n_steps even
    int NT, Kc;
    float *diff2;
    WPart *part;
};

// Value of the lane 8 further in its row of 16 lanes.
__device__ __forceinline__ float dpp_ror8(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, true));
}
__device__ __forceinline__ double dpp_ror8(double v) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x128, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x128, 0xf, 0xf, true));
}
__device__ __forceinline__ float fma_t(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return fma(a, b, c); }

// One block per tile of 64 orientations of one particle, 16 per wave, all translations of one column tile; M: number
// of positive shifts of the lattice; T: the arithmetic (Lattice). Each lane loads its row's projection values (lane l:
// orientation l % 16, x pairs 2 (l / 16) of every 8) and forms A in registers, so that the operands of the x contraction
// (16x16x4 products: lane l supplies row or column l % 16 at k = l / 16) go from memory to the matrix units through
// registers alone; the column operand is the same for every row, particle and orientation. The particle's rows, shared by
// the block, are staged in LDS: read from memory by every wave they took more of the vector memory path than the
// projections (busy 81% of the time). The steps alternate between two register sets, the next step's loads in flight. The
// results leave through LDS so that whole rows are stored. Bound by the matrix rate and the vector instructions that form
// A, about evenly.
// The lattice form needs 4 (2 M) + 4 (2 M + 1)^2 / s flops per pixel and orientation where the direct cross term needs
// 4 NT (113 translations, coarse size 54: 57 against 452), which is why FP32 matrix products here are faster than BF16
// hi+lo products of the direct form, and FP64 ones, at half the FP32 matrix rate and with twice the registers, much faster
// than direct FP32 squared differences on the vector units.
// Measured (box 128, coarse size 54, 36,864 orientations x 113 translations): 101 particles in FP64 9.3 to 10.3 ms (81 ms with
// direct FP32 squared differences; 5.5 ms with FP32 sums, whose error is 1e-7 of the signal's power), 151 particles and 4
// classes in FP32 30.6 to 31.5 ms (63.6 ms with BF16 hi+lo products of the direct cross term): 81 G poses/s. In FP32, reading all
// LDS operands of a step at once and running the missing row -y on zeros instead of a branch costs 16 registers, one wave
// per SIMD and 4 to 10% of the time.
// grid (tiles, column tiles), dynamic LDS: xtab of the column tile.
template <typename T, int M>
__global__ void __launch_bounds__(kBlock, 2) k_coarse_lattice(CoarseArgs<T> a) {
    typedef Lattice<T> L;
    typedef typename L::Pair Pair;
    constexpr bool kZero = M == kColShift;  // the tx = 0 column has no lane: summed beside the others
    constexpr int kY = 2 * M + 1;
    __shared__ union {
        struct {
            Pair w[16 * kStepChunk];
            Pair c[8 * kStepChunk];
        } in;
        float out[kBlock / 64][4][256];
    } lds;
    extern __shared__ __align__(16) unsigned char s_dyn[];
    Pair *s_x = reinterpret_cast<Pair *>(s_dyn);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform, and so is what follows from it
    const int n = lane & 15, g = lane >> 4;
    const CoarseTile tile = a.tiles[blockIdx.x];
    const int b = tile.b;
    const int n_o = a.or_cnt[b];
    const int o0 = tile.o_begin + 16 * wave;
    const int n_rows = max(0, min(16, n_o - o0));
    const int og = n < n_rows ? a.or_proj[a.or_off[b] + o0 + n] : -1;
    for (int i = tid; i < a.n_xsteps * 64; i += kBlock) s_x[i] = a.xtab[(size_t)blockIdx.y * a.n_xsteps * 64 + i];
    const float4 *pr = reinterpret_cast<const float4 *>(og >= 0 ? a.pf + (size_t)og * a.Kc : a.zero_row) + g;
    const Pair *wr = a.w + (size_t)b * a.Kc;
    const Pair *cr = reinterpret_cast<const Pair *>(a.ctf2 + (size_t)b * a.Kc);
    const T sgn = n < 8 ? 1 : -1;
    T cc[M + 1][4], cs[M + 1][4];  // cos and sin parts per |ty| of this lane's 4 rows (cs[0] unused)
    T zc[M + 1], zs[M + 1];        // the tx = 0 column, this lane's share of row n
#pragma unroll
    for (int k = 0; k <= M; ++k) {
#pragma unroll
        for (int r = 0; r < 4; ++r) cc[k][r] = cs[k][r] = 0;
        zc[k] = zs[k] = 0;
    }
    T an = 0;  // this lane's share of sum_p c_p^2 |P_o(p)|^2 of row n
    typename L::Acc da = {0, 0, 0, 0}, db = da, ea = da, eb = da;
    T zpa = 0, zpb = 0, zma = 0, zmb = 0;
    typename L::Uniform yt = (typename L::Uniform)a.ytab;
    UniformI steps = (UniformI)a.steps;
    // two complex slots of one row: A = P conj(w), its products with the lane's x phases, the row's norm
    auto half = [&](const float4 &p, int slot, const Pair &x, typename L::Acc &sa, typename L::Acc &sb, T &za, T &zb) {
        const Pair w0 = lds.in.w[2 * slot], w1 = lds.in.w[2 * slot + 1], c2 = lds.in.c[slot];
        const T p0 = p.x, p1 = p.y, p2 = p.z, p3 = p.w;
        const T a0 = p0 * w0.x + p1 * w0.y, b0 = p1 * w0.x - p0 * w0.y;
        const T a1 = p2 * w1.x + p3 * w1.y, b1 = p3 * w1.x - p2 * w1.y;
        sa = L::mfma(a0, x.x, sa);
        sb = L::mfma(b0, x.x, sb);
        sa = L::mfma(a1, x.y, sa);
        sb = L::mfma(b1, x.y, sb);
        an = fma_t(p0 * p0 + p1 * p1, c2.x, an);
        an = fma_t(p2 * p2 + p3 * p3, c2.y, an);
        if (kZero) {
            za += a0 + a1;
            zb += b0 + b1;
        }
    };
    // one step: a float4 (two complex slots) of row y (pp) and of row -y (pm) per lane; st within the staged chunk
    auto step = [&](const float4 &pp, const float4 &pm, int st, int xoff, int flags) {
        const Pair x = s_x[xoff + lane];
        half(pp, 8 * st + g, x, da, db, zpa, zpb);
        if (flags & kStepMinus) half(pm, 8 * st + 4 + g, x, ea, eb, zma, zmb);
        if (!(flags & kStepEnd)) return;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // cos lanes (+tx): U = Sa + Sb', V = Tb - Ta'; sin lanes (-tx): U = Sa' - Sb, V = Tb' + Ta, primes from
            // the partner lane, S and T the sum and difference of rows y and -y
            const T su = n < 8 ? da[r] + ea[r] : db[r] + eb[r];
            const T sv = n < 8 ? db[r] - eb[r] : da[r] - ea[r];
            const T U = fma_t(sgn, su, dpp_ror8(su)), V = fma_t(-sgn, dpp_ror8(sv), sv);
            cc[0][r] = fma_t(yt[0], U, cc[0][r]);
#pragma unroll
            for (int m = 1; m <= M; ++m) {
                cc[m][r] = fma_t(yt[m], U, cc[m][r]);
                cs[m][r] = fma_t(yt[M + m], V, cs[m][r]);
            }
        }
        if (kZero) {
            const T U = zpa + zma, V = zpb - zmb;
            zc[0] = fma_t(yt[0], U, zc[0]);
#pragma unroll
            for (int m = 1; m <= M; ++m) {
                zc[m] = fma_t(yt[m], U, zc[m]);
                zs[m] = fma_t(yt[M + m], V, zs[m]);
            }
            zpa = zpb = zma = zmb = 0;
        }
        da = db = ea = eb = typename L::Acc{0, 0, 0, 0};
        yt += kY;
    };
    for (int s0 = 0; s0 < a.n_steps; s0 += kStepChunk) {
        const int ns = min(kStepChunk, a.n_steps - s0);
        __syncthreads();  // the previous chunk's rows were read (and s_x is written, first time)
        for (int i = tid; i < 16 * ns; i += kBlock) lds.in.w[i] = wr[16 * s0 + i];
        for (int i = tid; i < 8 * ns; i += kBlock) lds.in.c[i] = cr[8 * s0 + i];
        __syncthreads();
        if (n_rows == 0) continue;  // uniform over the wave
        const float4 *p = pr + 8 * s0;
        float4 p0 = p[0], m0 = p[4], p1, m1;
        for (int st = 0; st < ns; st += 2) {
            p1 = p[8 * st + 8];
            m1 = p[8 * st + 12];
            step(p0, m0, st, steps[2 * (s0 + st)], steps[2 * (s0 + st) + 1]);
            const int nx = min(st + 2, ns - 1);  // the last load is repeated, not used
            p0 = p[8 * nx];
            m0 = p[8 * nx + 4];
            step(p1, m1, st + 1, steps[2 * (s0 + st) + 2], steps[2 * (s0 + st) + 3]);
        }
    }
    an += __shfl_xor(an, 16);  // the four lanes of row n
    an += __shfl_xor(an, 32);
    if (kZero) {
#pragma unroll
        for (int m = 0; m <= M; ++m) {
            zc[m] += __shfl_xor(zc[m], 16);
            zc[m] += __shfl_xor(zc[m], 32);
            zs[m] += __shfl_xor(zs[m], 16);
            zs[m] += __shfl_xor(zs[m], 32);
        }
    }
    const double base = (double)a.xi2half[b] + a.ynorm[b];
    const CoarseColumn col = a.cols[16 * blockIdx.y + n];
    CoarseColumn zcol{0, -1};
    if (kZero) zcol = a.cols[16 * gridDim.y];
    float *out = a.diff2 + a.d2_off[b];
    float mn = 3.0e38f;  // minimum of the non-negative values written, for the weights' exponent offset
    auto value = [&](T norm2, T cross) {
        const float v = (float)(base + (double)(norm2 - 2 * cross));
        return v < 0.f ? 0.f : v;  // rounding of a match without noise; NaN stays
    };
    float (*so)[256] = lds.out[wave];
    __syncthreads();  // the staged rows were read
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        // the rows of register r in the four lane groups; row n of the zero column's lanes may be one of them
        const T nr = __shfl(an, L::row(g, r));
        __syncthreads();
#pragma unroll
        for (int m = 0; m <= M; ++m) {
            if (m <= col.half) {
                so[g][col.t0 + m] = value(nr, cc[m][r] + cs[m][r]);
                if (m > 0) so[g][col.t0 - m] = value(nr, cc[m][r] - cs[m][r]);
            }
            if (kZero && g == 0 && L::reg(n) == r && m <= zcol.half) {
                so[L::group(n)][zcol.t0 + m] = value(an, zc[m] + zs[m]);
                if (m > 0) so[L::group(n)][zcol.t0 - m] = value(an, zc[m] - zs[m]);
            }
        }
        __syncthreads();
        for (int gg = 0; gg < 4; ++gg) {
            const int row = L::row(gg, r);
            if (row >= n_rows) break;
            const bool off = __shfl(og, row) < 0;  // orientation or class without prior: never evaluated
            for (int t = lane; t < a.NT; t += 64) {
                if (a.tile_of && a.tile_of[t] != (int)blockIdx.y) continue;
                const float v = off ? -999.f : so[gg][t];
                out[(size_t)(o0 + row) * a.NT + t] = v;
                if (v >= 0.f) mn = fminf(mn, v);
            }
        }
    }
    for (int o = 32; o > 0; o >>= 1) mn = fminf(mn, __shfl_xor(mn, o));
    // sign bit cleared: -0 orders as +0 among the unsigned bit patterns of non-negative floats
    if (lane == 0 && mn < 3.0e38f) atomicMin(&a.part[b].mn_bits, __float_as_uint(mn) & 0x7fffffffu);
}

// --------------------------------------------------------------------------------------------------
// Weights and significance (convertAllSquaredDifferencesToWeights, src/ml_optimiser.cpp:7704-8239)
// --------------------------------------------------------------------------------------------------

struct PassStats {
    double min_diff2;
    double sum_weight;
    double threshold;      // exp_significant_weight
    double max_weight;
    long long nr_sign;     // my_nr_significant_coarse_samples
    long long n_above;     // entries with weight >= threshold
    long long best_key;    // tie-break key of the max weight (wsum loop order)
    long long best_index;  // entry index of the max weight
    int status;            // 0 ok, RLN_ERR_* otherwise
    int pad_;
};

constexpr int kWBlock = 1024;
constexpr int kCand = 2048;  // threshold candidates sorted in LDS

__device__ __forceinline__ double block_sum_d(double v, double *red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[w] = v;
    __syncthreads();
    double t = 0.;
    if (threadIdx.x < 64) {
        t = (threadIdx.x < (blockDim.x >> 6)) ? red[threadIdx.x] : 0.;
        for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o);
        if (threadIdx.x == 0) red[0] = t;
    }
    __syncthreads();
    const double r = red[0];
    __syncthreads();
    return r;
}

__device__ __forceinline__ double block_min_d(double v, double *red) {
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o));
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[w] = v;
    __syncthreads();
    if (threadIdx.x < 64) {
        double t = (threadIdx.x < (blockDim.x >> 6)) ? red[threadIdx.x] : 1.0e300;
        for (int o = 32; o > 0; o >>= 1) t = fmin(t, __shfl_xor(t, o));
        if (threadIdx.x == 0) red[0] = t;
    }
    __syncthreads();
    const double r = red[0];
    __syncthreads();
    return r;
}

__device__ __forceinline__ int block_exclusive_scan_i(int v, int *tmp, int &total) {
    // wave-level inclusive scan
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    __syncthreads();
    if (lane == 63) tmp[w] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        int acc = 0;
        for (int i = 0; i < (int)(blockDim.x >> 6); ++i) {
            const int t = tmp[i];
            tmp[i] = acc;
            acc += t;
        }
        tmp[blockDim.x >> 6] = acc;
    }
    __syncthreads();
    const int r = x - v + tmp[w];
    total = tmp[blockDim.x >> 6];
    __syncthreads();
    return r;
}

__device__ __forceinline__ long long block_sum_ll(long long v, long long *red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[w] = v;
    __syncthreads();
    if (threadIdx.x < 64) {
        long long t = (threadIdx.x < (blockDim.x >> 6)) ? red[threadIdx.x] : 0;
        for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o);
        if (threadIdx.x == 0) red[0] = t;
    }
    __syncthreads();
    const long long r = red[0];
    __syncthreads();
    return r;
}

// Device-side header of a chunk's fine pass, written by k_fine_plan / k_fine_items and read by the persistent
// kernels, so that the fine pass needs no host round trip. When a count exceeds the capacity the host sized
// the buffers for, overflow is set, every later kernel of the pass returns at once, and the host grows the
// buffers and runs the pass again.
struct FinePlan {
    long long n_pairs;   // significant coarse poses of the chunk
    int n_jobs;          // (particle, orientation) jobs
    int n_small, n_wide; // work items of k_fine_diff2<2> and k_fine_diff2_wide
    int overflow;
    int B;               // particles in the chunk
    int next_fine;       // next work item of k_fine_diff2 (dynamic fetch; zeroed by k_fine_plan)
    int next_wsum;       // next work item of k_wsum_bp
    int next_fine_x[8];  // next work unit of each XCD's share (k_fine_diff2 with per-XCD queues)
    int next_wsum_x[8];  // the same for k_wsum_bp
    int fine_choice;     // log2 of the band count that fills the GPU with the chunk's items (k_fine_items)
    int wsum_choice;     // the same for the jobs of k_wsum_bp
    int pad_;
};

// log2 of the number of radial bands (1 .. 32) that cuts n items of n_pix pixels into at least 4 units per CU, as long
// as a band keeps kMinBandPix pixels (two of a block's four waves). For engines whose band count is not tuned or fixed:
// a few items on one band each leave most of the GPU idle. 11 items of 1,604 pixels: fine pass stage 165 us on 1 band, 54
// on 8; weighted sums 208 and 62 us; 108 items of 6,426 pixels: 650 and 190 us, 420 and 150 us.
constexpr int kMinBandPix = 128, kFillUnits = 1024;
__device__ __forceinline__ int fill_choice(int n, int n_pix) {
    int c = 0;
    while (c < 5 && ((long long)n << c) < kFillUnits && (n_pix >> (c + 1)) >= kMinBandPix) ++c;
    return c;
}

// Per-chunk input images (device pointers), read by the fine-pass kernels through one indirection so that a
// captured graph of the pass serves every chunk.
struct ChunkPtrs {
    const float2 *fimg;
    const float2 *fimg_nomask;
    const float *fctf;
    int B;  // particles in the chunk
    int pad_;
};

// Arguments of k_weights: entries of the fine pass are e = s*32 + r*4 + u where pair s holds the coarse index
// (o*NT + t) in pairs[].
struct WeightArgs {
    const double *diff2d;        // per particle at d2_off[b], every entry evaluated
    const long long *d2_off;
    const long long *n_entries;  // per particle
    const double *or_prior;      // normalised pdf_orientation per orientation entry (or_off based)
    const int *or_off;
    const double *tr_prior;      // normalised pdf_offset [b][NT]
    const int *pairs;            // coarse index per pair, at pair_off[b]
    const long long *pair_off;
    int NT;
    double adaptive_fraction;
    double *weight;              // out, same indexing as diff2d
    PassStats *stats;            // out [b]
    const FinePlan *plan;        // chunk header (overflow: skip; blocks >= plan->B: idle)
};

__device__ __forceinline__ double entry_prior(const WeightArgs &a, int b, long long e) {
    const int c = a.pairs[a.pair_off[b] + (e >> 5)];
    const int o = c / a.NT, t = c - o * a.NT;
    return a.or_prior[a.or_off[b] + o] * a.tr_prior[(size_t)b * a.NT + t];
}

// Key that orders entries like storeWeightedSums visits them (class, direction, psi, iover_rot, itrans,
// iover_trans; src/ml_optimiser.cpp:8329-8470), used to break ties of the max weight as the reference does.
__device__ __forceinline__ long long wsum_order_key(const WeightArgs &a, int b, long long e) {
    const long long s = e >> 5;
    const int r = (int)((e >> 2) & 7), u = (int)(e & 3);
    const long long c = a.pairs[a.pair_off[b] + s];
    const long long o = c / a.NT, t = c - o * a.NT;
    return ((o * 8 + r) * a.NT + t) * 4 + u;
}

// One 1024-thread block per particle: min diff2, weights in FP64, their sum, the significance threshold by
// radix selection over the weights' bit patterns (positive doubles order like their uint64 patterns) and the max
// weight. The threshold is the weight at which the descending
// cumulative sum first exceeds adaptive_fraction * sum (src/ml_optimiser.cpp:8145-8168).
__global__ void __launch_bounds__(kWBlock) k_weights(WeightArgs a) {
    __shared__ double red_d[16];
    __shared__ long long red_l[16];
    __shared__ unsigned int hcnt[256];
    __shared__ double hsum[256];
    __shared__ unsigned long long s_prefix, s_mask;
    __shared__ double s_cand[kCand];
    __shared__ int s_ncand, s_cand_ok;
    __shared__ double s_cand_thr;
    __shared__ long long s_cand_nsig;
    __shared__ double s_above_sum;
    __shared__ long long s_above_cnt;
    __shared__ int s_done;
    const int b = blockIdx.x;
    if (a.plan->overflow || b >= a.plan->B) return;
    const long long n = a.n_entries[b];
    double *w = a.weight + a.d2_off[b];
    const int tid = threadIdx.x;

    const double *d2d = a.diff2d + a.d2_off[b];
    double mind = 1.0e300;
    for (long long e = tid; e < n; e += kWBlock) mind = fmin(mind, d2d[e]);
    mind = block_min_d(mind, red_d);
    double sum = 0.;
    for (long long e = tid; e < n; e += kWBlock) {
        const double diff = d2d[e] - mind;
        const double wt = (diff > 700.) ? 0. : entry_prior(a, b, e) * exp(-diff);
        w[e] = wt;
        sum += wt;
    }
    sum = block_sum_d(sum, red_d);
    PassStats st;
    st.min_diff2 = mind;
    st.sum_weight = sum;
    st.threshold = 0.;
    st.max_weight = 0.;
    st.nr_sign = 0;
    st.n_above = 0;
    st.best_key = -1;
    st.best_index = -1;
    st.status = 0;
    st.pad_ = 0;
    if (!(sum > 0.)) {  // zero or NaN (src/ml_optimiser.cpp:8054-8104)
        if (tid == 0) {
            st.status = -6;
            a.stats[b] = st;
        }
        return;
    }

    const double target = a.adaptive_fraction * sum;
    double thr = 0.;
    long long nr_sign = 0;
    bool have_thr = false;
    // Candidates: only weights >= (1 - f) * sum / n can be the threshold, since all smaller weights together
    // hold less than the (1 - f) tail. When they are few, sort them in LDS and accumulate in descending order
    // exactly as the reference's loop does (src/ml_optimiser.cpp:8145-8168).
    {
        const double xmin = (1. - a.adaptive_fraction) * sum / (double)(n > 0 ? n : 1);
        if (tid == 0) s_ncand = 0;
        __syncthreads();
        for (long long e = tid; e < n; e += kWBlock) {
            const double v = w[e];
            if (v > 0. && v >= xmin) {
                const int slot = atomicAdd(&s_ncand, 1);
                if (slot < kCand) s_cand[slot] = v;
            }
        }
        __syncthreads();
        const int nc = s_ncand;
        if (nc <= kCand) {
            // sort size: the next power of two holding the candidates (uniform), padded with -1 below every weight
            int n2 = 2;
            while (n2 < nc) n2 <<= 1;
            for (int i = tid; i < n2; i += kWBlock)
                if (i >= nc) s_cand[i] = -1.;
            __syncthreads();
            // bitonic sort, ascending
            for (int ks = 2; ks <= n2; ks <<= 1)
                for (int j = ks >> 1; j > 0; j >>= 1) {
                    for (int i = tid; i < n2; i += kWBlock) {
                        const int l = i ^ j;
                        if (l > i) {
                            const double x = s_cand[i], y = s_cand[l];
                            if (((i & ks) == 0) ? (x > y) : (x < y)) {
                                s_cand[i] = y;
                                s_cand[l] = x;
                            }
                        }
                    }
                    __syncthreads();
                }
            // descending cumulative sum by wave 0, 64 candidates per step (inclusive lane scan)
            if (tid < 64) {
                double base = 0.;
                int crossed = 0;
                long long rank = -1;
                for (int r0 = 0; r0 < nc; r0 += 64) {
                    const int r = r0 + tid;
                    const double v = (r < nc) ? s_cand[n2 - 1 - r] : 0.;
                    double x = v;
                    for (int o = 1; o < 64; o <<= 1) {
                        const double y = __shfl_up(x, o);
                        if (tid >= o) x += y;
                    }
                    const double cum = base + x;
                    const unsigned long long hit = __ballot(r < nc && cum > target);
                    if (hit) {
                        crossed = 1;
                        rank = r0 + (__ffsll((long long)hit) - 1);
                        break;
                    }
                    base = __shfl(cum, 63);
                }
                if (tid == 0) {
                    long long nsig = rank + 1;
                    s_cand_ok = crossed;
                    s_cand_nsig = nsig;
                    s_cand_thr = crossed ? s_cand[n2 - nsig] : 0.;
                }
            }
            __syncthreads();
            if (s_cand_ok) {
                have_thr = true;
                thr = s_cand_thr;
                nr_sign = s_cand_nsig;
            }
        }
    }
    if (!have_thr) {
    // radix selection of the crossing element: 8 digits of 8 bits from the most significant
    if (tid == 0) {
        s_prefix = 0ULL;
        s_mask = 0ULL;
        s_above_sum = 0.;
        s_above_cnt = 0;
        s_done = 0;
    }
    __syncthreads();
    for (int shift = 56; shift >= 0; shift -= 8) {
        for (int i = tid; i < 256; i += kWBlock) {
            hcnt[i] = 0;
            hsum[i] = 0.;
        }
        __syncthreads();
        const unsigned long long pre = s_prefix, msk = s_mask;
        for (long long e = tid; e < n; e += kWBlock) {
            const double v = w[e];
            if (!(v > 0.)) continue;
            const unsigned long long key = (unsigned long long)__double_as_longlong(v);
            if ((key & msk) != pre) continue;
            const int bin = (int)((key >> shift) & 255ULL);
            atomicAdd(&hcnt[bin], 1u);
            atomicAdd(&hsum[bin], v);
        }
        __syncthreads();
        if (tid == 0) {
            double acc = s_above_sum;
            long long cnt = s_above_cnt;
            int bin = -1;
            for (int k = 255; k >= 0; --k) {
                if (hcnt[k] == 0) continue;
                if (acc + hsum[k] > target) {
                    bin = k;
                    break;
                }
                acc += hsum[k];
                cnt += hcnt[k];
            }
            if (bin < 0) {  // rounding: the total never exceeds the target; take the smallest present bin
                for (int k = 0; k < 256; ++k)
                    if (hcnt[k]) {
                        bin = k;
                        break;
                    }
                // undo its accumulation
                acc -= hsum[bin];
                cnt -= hcnt[bin];
            }
            s_above_sum = acc;
            s_above_cnt = cnt;
            s_prefix |= ((unsigned long long)bin << shift);
            s_mask |= (255ULL << shift);
        }
        __syncthreads();
    }
    thr = __longlong_as_double((long long)s_prefix);
    // elements equal to thr needed to cross the target
    {
        const double rem = target - s_above_sum;
        long long m = (long long)floor(rem / thr) + 1;
        if (m < 1) m = 1;
        nr_sign = s_above_cnt + m;
    }
    }  // radix selection
    // count above threshold, max weight with the reference's loop-order tie break
    long long above = 0;
    double bw = -1.;
    long long bkey = 0x7fffffffffffffffLL, bidx = -1;
    for (long long e = tid; e < n; e += kWBlock) {
        const double v = w[e];
        const bool sig = v >= thr && v > 0.;
        above += sig ? 1 : 0;
        if (v > 0.) {
            const long long key = wsum_order_key(a, b, e);
            if (v > bw || (v == bw && key < bkey)) {
                bw = v;
                bkey = key;
                bidx = e;
            }
        }
    }
    above = block_sum_ll(above, red_l);
    // arg-max across the block
    for (int o = 32; o > 0; o >>= 1) {
        const double ow = __shfl_xor(bw, o);
        const long long ok = __shfl_xor(bkey, o), oi = __shfl_xor(bidx, o);
        if (ow > bw || (ow == bw && ok < bkey)) {
            bw = ow;
            bkey = ok;
            bidx = oi;
        }
    }
    __shared__ double s_bw[16];
    __shared__ long long s_bk[16], s_bi[16];
    if ((tid & 63) == 0) {
        s_bw[tid >> 6] = bw;
        s_bk[tid >> 6] = bkey;
        s_bi[tid >> 6] = bidx;
    }
    __syncthreads();
    if (tid == 0) {
        for (int i = 1; i < (kWBlock >> 6); ++i)
            if (s_bw[i] > bw || (s_bw[i] == bw && s_bk[i] < bkey)) {
                bw = s_bw[i];
                bkey = s_bk[i];
                bidx = s_bi[i];
            }
        st.threshold = thr;
        st.nr_sign = nr_sign;
        st.n_above = above;
        st.max_weight = bw;
        st.best_key = bkey;
        st.best_index = bidx;
        a.stats[b] = st;
    }
}

// --------------------------------------------------------------------------------------------------
// Coarse weights over segments: min, FP64 weights, their sum, the significance threshold and the significant poses,
// with every pass over the entries split into blocks of a segment, so that a particle with millions of coarse poses
// (an exhaustive search) is spread over the whole GPU. The weights are not stored (unless they are asked for): every
// pass forms those it needs from the FP32 diff2, 4 bytes a pose, the same FP64 expression each time.
//   k_wseg_exp     weights' sum and a histogram of their binary exponents
//   k_wsel_pick    the crossing bin: where the descending cumulative sum exceeds the target or the count reaches the cap
//                  (maxsig), whichever comes first
//   k_wseg_refine  particles whose crossing bin holds more than the candidate list: a histogram of its entries' next 10
//                  mantissa bits, over the segments of a list that the pick made (nothing to do for sharp posteriors);
//                  then the pick again. Twice; entries alike to 20 bits are told apart by the last pick itself
//   k_wseg_gather  candidates: every entry from the crossing bin up when they fit the list (kSelAll), else the bin's
//                  (kSelBin)
//   k_wsel_final   exact threshold from the sorted candidates; for kSelAll also the significant poses in order, which
//                  are then all the fine pass needs
//   k_wseg_mask, k_wsel_stats  the mask, per-orientation counts and maximum over all entries of kSelBin particles
// Bound by the two reads of diff2 (4 bytes a pose each) and, where many poses are close, by the exponentials. Measured:
// 2.5e9 poses 20.0 -> 5.5 ms (20 GB: 3.7 TB/s), 4.2e8 poses 3.6 -> 1.1 ms, 2,048 particles of 35,000 poses 2.2 -> 0.66
// ms, against stored FP64 weights with 8-bit digits in a launch each. Several diff2 values a thread in flight: 1 8.8 ms,
// 4 5.5, 8 6.5. Finding the bin in the last block of a particle instead of a launch of its own needs device-wide fences,
// which made the first pass wait on the caches for 16 ms. Refining in the pick's block instead of over the segments, and
// the cap by a radix selection of its own in one block per particle, took 82 ms for 40 particles of 4.2e6 poses, broad
// posteriors and a cap of 500 (20.8 ms with stored weights and every digit over the segments): now 1.6 ms.
// --------------------------------------------------------------------------------------------------
constexpr double kWholeTail = 1. - 1e-9;  // fractions from which the weights below the threshold may hold nothing
constexpr int kExpBins = 1088;    // binary exponents of the weights (a weight is below 2^64: the prior's mean is 1)
constexpr int kGather = 4096;     // candidates sorted exactly
constexpr int kDigitBits = 10, kDigitBins = 1 << kDigitBits;  // mantissa bits per refinement (at most kExpBins bins)
constexpr int kRefines = 2;       // refinements over the segments
constexpr int kSegBatch = 4;      // diff2 values a thread has in flight
constexpr int kSegMin = 4096, kSegMax = 32768;  // entries per segment (choose_segment)

// Entries per segment of a chunk of `total` entries: long enough that a block's histogram (cleared and written once a
// segment) is a small part of its work, short enough that small chunks still fill the GPU.
inline long long choose_segment(long long total) {
    const long long want = total / 4096 / kBlock * kBlock;
    return want < kSegMin ? kSegMin : want > kSegMax ? kSegMax : want;
}

struct WSeg {
    int b;             // particle
    int pad_;
    long long begin;   // entry range [begin, end) within the particle
    long long end;
};

struct WSegBest {
    double w;
    long long key, idx;
};

struct CoarseWeightArgs {
    const WSeg *segs;
    const int *seg_first;        // [B + 1] first segment of each particle
    const float *diff2;          // per particle at d2_off[b]; entries < 0 were not evaluated
    const long long *d2_off;
    const long long *n_entries;  // per particle
    const double *or_prior;      // normalised pdf_orientation per orientation entry (or_off based)
    const int *or_off;
    const int *or_cnt;
    const int *oc_off;           // per-particle offsets of per-orientation state (ocnt)
    const double *tr_prior;      // normalised pdf_offset [b][NT]
    int NT;
    double prior_max;            // no entry's prior exceeds it
    double adaptive_fraction;
    long long maxsig;            // <= 0: none
    WPart *part;
    unsigned int *hcnt;          // [b][kExpBins] histogram: zero before k_wseg_exp, left zero for the next refinement
    double *hsum;
    int *refine;                 // particles and segments to refine: counts [kRefines][2], then per refinement particles
                                 // [B] and segments [n_seg]
    int n_seg;
    double *cand_w;              // [b][kGather] candidate weights
    int *cand_i;                 // [b][kGather] their entries; then the significant entries of kSelAll in order
    double *weight;              // out, same indexing as diff2, or null
    unsigned char *mask;         // out, weight >= threshold (kSelBin, or every particle with want_mask)
    int want_mask;
    WSegBest *best;              // per segment (kSelBin)
    int *ocnt;                   // significant translations per orientation entry (kSelBin)
    int *npairs, *njobs;         // out [b] significant poses, orientations with any
    PassStats *stats;            // out [b]
    int B;
};

// Entries of one segment as a block of S threads visits them: e, and its orientation and translation without a
// division per entry.
template <int S>
struct SegCursor {
    long long e;
    int o, t, step_o, step_t, NT;
    __device__ __forceinline__ SegCursor(long long begin, int nt) {
        NT = nt;
        step_o = S / nt;
        step_t = S % nt;
        e = begin + threadIdx.x;
        o = (int)((unsigned)e / (unsigned)nt);
        t = (int)e - o * nt;
    }
    __device__ __forceinline__ void next() {
        e += S;
        o += step_o;
        t += step_t;
        if (t >= NT) {
            t -= NT;
            ++o;
        }
    }
};

// Weight of a coarse pose: 0 where it was not evaluated or lies more than 700 above the minimum.
__device__ __forceinline__ double coarse_weight(float v, double mind, const double *orp, const double *trp, int o,
                                                int t) {
    if (!(v >= 0.f)) return 0.;
    const double diff = (double)v - mind;
    return (diff > 700.) ? 0. : orp[o] * trp[t] * exp(-diff);
}

// Lists of refinement r (0, 1) within CoarseWeightArgs::refine.
__host__ __device__ __forceinline__ long long refine_ints(long long B, long long n_seg) {
    return 2 * kRefines + kRefines * (B + n_seg);
}
__device__ __forceinline__ int *refine_count(const CoarseWeightArgs &a, int r) { return a.refine + 2 * r; }
__device__ __forceinline__ int *refine_parts(const CoarseWeightArgs &a, int r) {
    return a.refine + 2 * kRefines + (long long)r * (a.B + a.n_seg);
}
__device__ __forceinline__ int *refine_segs(const CoarseWeightArgs &a, int r) { return refine_parts(a, r) + a.B; }

// Particle states, histograms and refinement counts of a chunk.
__global__ void __launch_bounds__(kBlock) k_wpart_init(WPart *__restrict__ part, int B, unsigned int *__restrict__ hcnt,
                                                       double *__restrict__ hsum, int *__restrict__ refine) {
    const int b = blockIdx.x * kBlock + threadIdx.x;
    for (long long i = b; i < (long long)B * kExpBins; i += (long long)gridDim.x * kBlock) {
        hcnt[i] = 0;
        hsum[i] = 0.;
    }
    if (b < 2 * kRefines) refine[b] = 0;
    if (b >= B) return;
    WPart p{};
    p.mn_bits = 0x7f800000u;  // +inf
    part[b] = p;
}

// Weights of one segment, their sum, and the histogram of their exponents. Two bounds from the largest weight seen so
// far, s (at most the sum), spare most entries the LDS atomics and the exponential:
//   - the weights below x = (1 - f) sum / n together hold less than the (1 - f) tail, so the threshold is at least x and
//     its bin's lower edge at least x / 2: weights below (1 - f) s / (4 n) are left out of the histogram;
//   - weights below 2^-64 s / n, all together, do not change the FP64 sum: they are not formed.
// Neither holds where the tail is lost in the rounding of the sums (kWholeTail): every positive weight can then be the
// threshold, and all of them are formed and counted.
__global__ void __launch_bounds__(kBlock) k_wseg_exp(CoarseWeightArgs a) {
    __shared__ double red[kBlock / 64];
    __shared__ unsigned int c[kExpBins];
    __shared__ double sm[kExpBins];
    __shared__ unsigned long long s_seen;
    for (int k = threadIdx.x; k < kExpBins; k += kBlock) {
        c[k] = 0;
        sm[k] = 0.;
    }
    const WSeg sg = a.segs[blockIdx.x];
    const int b = sg.b;
    const float *d2 = a.diff2 + a.d2_off[b];
    const double *orp = a.or_prior + a.or_off[b], *trp = a.tr_prior + (size_t)b * a.NT;
    const double mind = (double)__uint_as_float(a.part[b].mn_bits);
    if (threadIdx.x == 0) s_seen = atomicAdd(&a.part[b].seen, 0ULL);
    __syncthreads();
    const bool bounded = a.adaptive_fraction < kWholeTail;
    const double n = (double)a.n_entries[b], tail = bounded ? (1. - a.adaptive_fraction) / (4. * n) : 0.;
    double sum = 0., seen = 0., hist_min = 0., cut = 1e300;
    for (SegCursor<kBlock> k(sg.begin, a.NT); k.e < sg.end;) {
        float v[kSegBatch];
#pragma unroll
        for (int u = 0; u < kSegBatch; ++u) v[u] = k.e + u * kBlock < sg.end ? d2[k.e + u * kBlock] : -1.f;
        const double s = __longlong_as_double(
            (long long)__hip_atomic_load(&s_seen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
        if (s > seen) {  // rare: the bounds follow the largest weight
            seen = s;
            hist_min = tail * s;
            if (bounded && !a.weight) cut = log(a.prior_max / s * n) + 44.4;  // 2^-64 = exp(-44.36)
        }
#pragma unroll
        for (int u = 0; u < kSegBatch; ++u, k.next()) {
            if (k.e >= sg.end || (double)v[u] - mind > cut) continue;
            const double wt = coarse_weight(v[u], mind, orp, trp, k.o, k.t);
            if (a.weight) a.weight[a.d2_off[b] + k.e] = wt;
            sum += wt;
            if (!(wt > 0.) || wt < hist_min) continue;
            const unsigned long long bits = (unsigned long long)__double_as_longlong(wt);
            const int bin = min((int)(bits >> 52), kExpBins - 1);
            atomicAdd(&c[bin], 1u);
            atomicAdd(&sm[bin], wt);
            if (wt > seen) atomicMax(&s_seen, bits);
        }
    }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < kBlock / 64; ++i) sum += red[i];
        atomicAdd(&a.part[b].sum, sum);
        if (s_seen) atomicMax(&a.part[b].seen, s_seen);
    }
    for (int k = threadIdx.x; k < kExpBins; k += kBlock)
        if (c[k]) {
            atomicAdd(&a.hcnt[(size_t)b * kExpBins + k], c[k]);
            atomicAdd(&a.hsum[(size_t)b * kExpBins + k], sm[k]);
        }
}

// The crossing bin of one particle among nb histogram bins (digit at `shift`) by wave 0: the bin where the descending
// cumulative sum from above_sum exceeds the target or the count from above_cnt reaches the cap, or (rounding: the total
// may not exceed the target) the smallest bin present.
__device__ __forceinline__ void pick_bin(const CoarseWeightArgs &a, WPart &p, const unsigned int *c, const double *sm,
                                         int nb, int shift, unsigned long long digit_mask) {
    const int lane = threadIdx.x;
    const long long cap = a.maxsig > 0 ? a.maxsig : 0x7fffffffffffffffLL;
    double acc = p.above_sum, low_sum = 0.;
    long long cnt = p.above_cnt, low_cnt = 0;
    int low = 0;
    unsigned int in_low = 0;
    for (int k0 = nb - 1; k0 >= 0; k0 -= 64) {
        const int k = k0 - lane;
        const unsigned int ck = k >= 0 ? c[k] : 0u;
        const unsigned long long present = __ballot(ck > 0);
        if (!present) continue;
        const double s = ck > 0 ? sm[k] : 0.;
        double xs = s;  // inclusive sums from the top
        long long xc = ck;
        for (int o = 1; o < 64; o <<= 1) {
            const double ys = __shfl_up(xs, o);
            const long long yc = __shfl_up(xc, o);
            if (lane >= o) {
                xs += ys;
                xc += yc;
            }
        }
        const unsigned long long hit = __ballot(ck > 0 && (acc + xs > p.target || cnt + xc >= cap));
        const int q = hit ? __ffsll((long long)hit) - 1 : 63 - __clzll((long long)present);
        low = k0 - q;
        low_sum = acc + __shfl(xs - s, q);
        low_cnt = cnt + __shfl(xc - (long long)ck, q);
        in_low = __shfl(ck, q);
        if (hit) break;
        acc += __shfl(xs, 63);
        cnt += __shfl(xc, 63);
    }
    p.above_sum = low_sum;
    p.above_cnt = low_cnt;
    p.prefix |= (unsigned long long)low << shift;
    p.mask |= digit_mask;
    // the smallest weight with this prefix; below it no entry is a candidate
    const double lo = __longlong_as_double((long long)p.prefix);
    p.dcut = lo > 0. ? log(a.prior_max / lo) + 1e-6 : 1e300;
    p.state = low_cnt + in_low <= kGather ? kSelAll : (in_low <= kGather || shift == 0) ? kSelBin : kSelRefine;
}

// Histogram of the next digit (nb bins at `shift`) of one particle's entries [begin, end) that match its prefix, by a
// block of S threads, into LDS; for kMinMax also the smallest and largest of their bit patterns.
template <int S, bool kMinMax>
__device__ __forceinline__ void digit_histogram(const CoarseWeightArgs &a, int b, const WPart &p, long long begin,
                                                long long end, int shift, int nb, unsigned int *c, double *sm,
                                                unsigned long long *mm) {
    const float *d2 = a.diff2 + a.d2_off[b];
    const double *orp = a.or_prior + a.or_off[b], *trp = a.tr_prior + (size_t)b * a.NT;
    const double mind = (double)__uint_as_float(p.mn_bits);
    unsigned long long lo = ~0ULL, hi = 0ULL;
    for (SegCursor<S> k(begin, a.NT); k.e < end;) {
        float v[kSegBatch];
#pragma unroll
        for (int u = 0; u < kSegBatch; ++u) v[u] = k.e + u * S < end ? d2[k.e + u * S] : -1.f;
#pragma unroll
        for (int u = 0; u < kSegBatch; ++u, k.next()) {
            if (!(v[u] >= 0.f) || !((double)v[u] - mind <= p.dcut)) continue;
            const double wt = coarse_weight(v[u], mind, orp, trp, k.o, k.t);
            const unsigned long long key = (unsigned long long)__double_as_longlong(wt);
            if (!(wt > 0.) || (key & p.mask) != p.prefix) continue;
            const int bin = (int)((key >> shift) & (unsigned long long)(nb - 1));
            atomicAdd(&c[bin], 1u);
            atomicAdd(&sm[bin], wt);
            if (kMinMax) {
                lo = key < lo ? key : lo;
                hi = key > hi ? key : hi;
            }
        }
    }
    if (kMinMax && hi) {
        atomicMin(&mm[0], lo);
        atomicMax(&mm[1], hi);
    }
}

// Refinement r: the histogram of the crossing bins' next kDigitBits mantissa bits, over the listed segments.
__global__ void __launch_bounds__(kBlock) k_wseg_refine(CoarseWeightArgs a, int r) {
    __shared__ unsigned int c[kDigitBins];
    __shared__ double sm[kDigitBins];
    const int n = refine_count(a, r)[1];
    const int *list = refine_segs(a, r);
    for (int q = blockIdx.x; q < n; q += gridDim.x) {
        const WSeg sg = a.segs[list[q]];
        const WPart p = a.part[sg.b];
        for (int k = threadIdx.x; k < kDigitBins; k += kBlock) {
            c[k] = 0;
            sm[k] = 0.;
        }
        __syncthreads();
        digit_histogram<kBlock, false>(a, sg.b, p, sg.begin, sg.end, 52 - kDigitBits * (r + 1), kDigitBins, c, sm, nullptr);
        __syncthreads();
        for (int k = threadIdx.x; k < kDigitBins; k += kBlock)
            if (c[k]) {
                atomicAdd(&a.hcnt[(size_t)sg.b * kExpBins + k], c[k]);
                atomicAdd(&a.hsum[(size_t)sg.b * kExpBins + k], sm[k]);
            }
        __syncthreads();  // the next segment clears the bins
    }
}

// The crossing bin of every particle (level 0: of the exponents, grid B) or of the particles that were refined (level
// 1, 2: of the refined digit, any grid). Particles whose bin still holds more than kGather entries are listed for the
// next refinement; the last level goes on by itself, one block per particle, through the remaining 32 bits, and stops
// after one pass where they are all alike.
template <bool kLast>
__global__ void __launch_bounds__(kLast ? kWBlock : kBlock) k_wsel_pick(CoarseWeightArgs a, int level) {
    constexpr int S = kLast ? kWBlock : kBlock;
    __shared__ unsigned int c[kExpBins];
    __shared__ double sm[kExpBins];
    __shared__ WPart s_p;
    __shared__ unsigned long long s_mm[2];
    __shared__ int s_slot;
    const int tid = threadIdx.x;
    const int n = level == 0 ? a.B : refine_count(a, level - 1)[0];
    const int nb0 = level == 0 ? kExpBins : kDigitBins;
    int shift = 52 - kDigitBits * level;
    for (int q = blockIdx.x; q < n; q += gridDim.x) {
        const int b = level == 0 ? q : refine_parts(a, level - 1)[q];
        unsigned int *hc = a.hcnt + (size_t)b * kExpBins;
        double *hs = a.hsum + (size_t)b * kExpBins;
        for (int k = tid; k < nb0; k += S) {
            c[k] = hc[k];
            sm[k] = hs[k];
        }
        if (tid == 0) {
            s_p = a.part[b];
            if (level == 0) {
                // the whole sum is never exceeded: every positive weight is significant, whatever the sums' rounding
                s_p.target = a.adaptive_fraction < 1. ? a.adaptive_fraction * s_p.sum : INFINITY;
                s_p.state = kSelRefine;
                if (!(s_p.sum > 0.)) {
                    s_p.status = -6;  // zero or NaN sum (src/ml_optimiser.cpp:8054-8104)
                    s_p.state = kSelNone;
                }
            }
        }
        __syncthreads();
        if (s_p.state == kSelRefine && tid < 64) {
            WPart p = s_p;
            const unsigned long long digit = level == 0 ? 0xfffULL << 52 : (unsigned long long)(kDigitBins - 1) << shift;
            pick_bin(a, p, c, sm, nb0, shift, digit);
            if (tid == 0) s_p = p;
        }
        __syncthreads();
        if (kLast) {
            for (int sh = shift - 8; sh >= 0; sh -= 8) {
                if (s_p.state != kSelRefine) break;
                const WPart p = s_p;
                for (int k = tid; k < 256; k += S) {
                    c[k] = 0;
                    sm[k] = 0.;
                }
                if (tid == 0) {
                    s_mm[0] = ~0ULL;
                    s_mm[1] = 0ULL;
                }
                __syncthreads();
                digit_histogram<S, true>(a, b, p, 0, a.n_entries[b], sh, 256, c, sm, s_mm);
                __syncthreads();
                if (tid < 64) {
                    WPart w = p;
                    pick_bin(a, w, c, sm, 256, sh, 255ULL << sh);
                    if (s_mm[0] == s_mm[1] && w.state == kSelRefine) {  // one value: all of its bits are known
                        w.prefix = s_mm[0];
                        w.mask = ~0ULL;
                        w.state = kSelBin;
                    }
                    if (tid == 0) s_p = w;
                }
                __syncthreads();
            }
        } else if (s_p.state == kSelRefine) {
            const int s0 = a.seg_first[b], ns = a.seg_first[b + 1] - s0;
            if (tid == 0) {
                refine_parts(a, level)[atomicAdd(refine_count(a, level), 1)] = b;
                s_slot = atomicAdd(refine_count(a, level) + 1, ns);
            }
            for (int k = tid; k < kDigitBins; k += S) {
                hc[k] = 0;
                hs[k] = 0.;
            }
            __syncthreads();
            for (int i = tid; i < ns; i += S) refine_segs(a, level)[s_slot + i] = s0 + i;
        }
        if (tid == 0) a.part[b] = s_p;
        __syncthreads();
    }
}

// Candidates into the particle's list: all entries from the crossing bin up, or the crossing bin's weights.
__global__ void __launch_bounds__(kBlock) k_wseg_gather(CoarseWeightArgs a) {
    const WSeg sg = a.segs[blockIdx.x];
    const int b = sg.b;
    const WPart p = a.part[b];
    if (p.state == kSelNone) return;
    const float *d2 = a.diff2 + a.d2_off[b];
    const double *orp = a.or_prior + a.or_off[b], *trp = a.tr_prior + (size_t)b * a.NT;
    const double mind = (double)__uint_as_float(p.mn_bits);
    for (SegCursor<kBlock> k(sg.begin, a.NT); k.e < sg.end;) {
        float v[kSegBatch];
#pragma unroll
        for (int u = 0; u < kSegBatch; ++u) v[u] = k.e + u * kBlock < sg.end ? d2[k.e + u * kBlock] : -1.f;
#pragma unroll
        for (int u = 0; u < kSegBatch; ++u, k.next()) {
            if (!(v[u] >= 0.f) || !((double)v[u] - mind <= p.dcut)) continue;
            const double wt = coarse_weight(v[u], mind, orp, trp, k.o, k.t);
            if (!(wt > 0.)) continue;
            const unsigned long long key = (unsigned long long)__double_as_longlong(wt);
            if (p.state == kSelAll ? key < p.prefix : (key & p.mask) != p.prefix) continue;
            const int slot = atomicAdd(&a.part[b].ncand, 1);
            if (slot < kGather) {
                a.cand_w[(size_t)b * kGather + slot] = wt;
                a.cand_i[(size_t)b * kGather + slot] = (int)k.e;
            }
        }
    }
}

// per particle (one block): exact threshold from the sorted candidates, maxsig cap by rank
// (src/ml_optimiser.cpp:8145-8168). kSelAll: also the significant entries in ascending order, their counts and the
// particle's statistics; kSelBin: its per-orientation counts cleared for k_wseg_mask.
__global__ void __launch_bounds__(kBlock) k_wsel_final(CoarseWeightArgs a) {
    __shared__ double s_w[kGather];
    __shared__ int s_i[kGather];
    __shared__ int s_rank, s_crossed, s_above;
    __shared__ int tmp[8];
    const int b = blockIdx.x, tid = threadIdx.x;
    WPart &p = a.part[b];
    PassStats st{};
    st.min_diff2 = (double)__uint_as_float(p.mn_bits);
    st.sum_weight = p.sum;
    st.best_key = st.best_index = -1;
    const int state = p.state;
    if (state == kSelNone) {
        if (tid == 0) {
            st.status = p.status;
            a.stats[b] = st;
            a.npairs[b] = a.njobs[b] = 0;
        }
        return;
    }
    // a list that does not hold every entry from the crossing bin up (the histogram counted fewer) selects nothing: the
    // particle goes by the mask, from the bin's lower edge up
    const int ncand = p.ncand, nc = min(ncand, kGather);
    const bool all = state == kSelAll && ncand <= kGather;
    const double above_sum = all ? 0. : p.above_sum;
    if (tid == 0) s_above = 0;
    // sort size: the next power of two holding the candidates (uniform over the block), padded with -1 below every
    // weight; descending weight, ascending entry among equal weights
    int n2 = 2;
    while (n2 < nc) n2 <<= 1;
    for (int i = tid; i < n2; i += kBlock) {
        s_w[i] = (i < nc) ? a.cand_w[(size_t)b * kGather + i] : -1.;
        s_i[i] = (i < nc) ? a.cand_i[(size_t)b * kGather + i] : 0x7fffffff;
    }
    __syncthreads();
    for (int ks = 2; ks <= n2; ks <<= 1)
        for (int j = ks >> 1; j > 0; j >>= 1) {
            for (int i = tid; i < n2; i += kBlock) {
                const int l = i ^ j;
                if (l > i) {
                    const double x = s_w[i], y = s_w[l];
                    const int xi = s_i[i], yi = s_i[l];
                    const bool after = x < y || (x == y && xi > yi);  // x belongs after y
                    if (((i & ks) == 0) == after) {
                        s_w[i] = y;
                        s_w[l] = x;
                        s_i[i] = yi;
                        s_i[l] = xi;
                    }
                }
            }
            __syncthreads();
        }
    // descending cumulative sum, 64 elements per step (wave 0)
    if (tid < 64) {
        double base = above_sum;
        int crossed = 0, rank = nc - 1;
        for (int r0 = 0; r0 < nc; r0 += 64) {
            const int r = r0 + tid;
            double x = (r < nc) ? s_w[r] : 0.;
            for (int o = 1; o < 64; o <<= 1) {
                const double y = __shfl_up(x, o);
                if (tid >= o) x += y;
            }
            const double cum = base + x;
            const unsigned long long hit = __ballot(r < nc && cum > p.target);
            if (hit) {
                crossed = 1;
                rank = r0 + (__ffsll((long long)hit) - 1);
                break;
            }
            base = __shfl(cum, 63);
        }
        if (tid == 0) {
            s_rank = rank;
            s_crossed = crossed;
        }
    }
    __syncthreads();
    double thr;
    long long nr_sign;
    if (ncand <= kGather && nc > 0) {
        // without a crossing (rounding) the smallest element, as the reference's loop ends
        const long long above = all ? 0 : p.above_cnt;
        const long long rank = a.maxsig > 0 ? min((long long)s_rank, a.maxsig - above - 1) : s_rank;
        thr = s_w[rank];
        nr_sign = above + rank + 1;
    } else {
        // all 64 bits fixed and more than kGather equal elements: the bin is one value
        thr = __longlong_as_double((long long)p.prefix);
        double room = ncand;
        if (a.maxsig > 0) room = fmin(room, (double)(a.maxsig - p.above_cnt));
        const long long m = (long long)fmax(1., fmin(floor((p.target - p.above_sum) / thr) + 1., room));
        nr_sign = p.above_cnt + m;
    }
    if (!all) {
        if (tid == 0) {
            p.state = kSelBin;
            p.thr = thr;
            p.nr_sign = nr_sign;
            a.njobs[b] = 0;
        }
        for (int o = tid; o < a.or_cnt[b]; o += kBlock) a.ocnt[a.oc_off[b] + o] = 0;
        return;
    }
    int mine = 0;
    for (int i = tid; i < nc; i += kBlock) mine += s_w[i] >= thr ? 1 : 0;
    if (mine) atomicAdd(&s_above, mine);
    const double best_w = s_w[0];
    const int best_i = s_i[0];
    __syncthreads();
    const int na = s_above;
    int m2 = 2;
    while (m2 < na) m2 <<= 1;
    for (int i = tid; i < m2; i += kBlock)
        if (i >= na) s_i[i] = 0x7fffffff;
    __syncthreads();
    for (int ks = 2; ks <= m2; ks <<= 1)  // ascending entries
        for (int j = ks >> 1; j > 0; j >>= 1) {
            for (int i = tid; i < m2; i += kBlock) {
                const int l = i ^ j;
                if (l > i) {
                    const int x = s_i[i], y = s_i[l];
                    if (((i & ks) == 0) ? (x > y) : (x < y)) {
                        s_i[i] = y;
                        s_i[l] = x;
                    }
                }
            }
            __syncthreads();
        }
    int jobs = 0;
    for (int i = tid; i < na; i += kBlock) {
        const int e = s_i[i];
        a.cand_i[(size_t)b * kGather + i] = e;
        jobs += (i == 0 || e / a.NT != s_i[i - 1] / a.NT) ? 1 : 0;
    }
    int n_jobs;
    block_exclusive_scan_i(jobs, tmp, n_jobs);
    if (tid == 0) {
        p.thr = thr;
        p.nr_sign = nr_sign;
        p.n_above = na;
        st.threshold = thr;
        st.nr_sign = nr_sign;
        st.n_above = na;
        st.max_weight = best_w;
        st.best_key = st.best_index = best_i;
        if (nr_sign == 0) st.status = -5;
        a.stats[b] = st;
        a.npairs[b] = na;
        a.njobs[b] = n_jobs;
    }
}

// Particles with more significant poses than the candidate list holds: mask, count above threshold, significant
// translations of every orientation entry (ocnt), orientations with at least one, and each segment's max weight, the
// first entry among equal ones. With want_mask the mask of every particle.
__global__ void __launch_bounds__(kBlock) k_wseg_mask(CoarseWeightArgs a) {
    __shared__ double s_bw[kBlock / 64];
    __shared__ long long s_bi[kBlock / 64], s_ab[kBlock / 64];
    const WSeg sg = a.segs[blockIdx.x];
    const int b = sg.b;
    const WPart p = a.part[b];
    const bool bin = p.state == kSelBin;
    if (!bin && !a.want_mask) return;
    const double thr = p.thr;
    const float *d2 = a.diff2 + a.d2_off[b];
    const double *orp = a.or_prior + a.or_off[b], *trp = a.tr_prior + (size_t)b * a.NT;
    const double mind = (double)__uint_as_float(p.mn_bits);
    long long above = 0;
    double bw = -1.;
    long long bidx = 0x7fffffffffffffffLL;
    for (SegCursor<kBlock> k(sg.begin, a.NT); k.e < sg.end; k.next()) {
        const double v = coarse_weight(d2[k.e], mind, orp, trp, k.o, k.t);
        const bool sig = p.state != kSelNone && v >= thr && v > 0.;
        a.mask[a.d2_off[b] + k.e] = sig ? 1 : 0;
        if (!bin) continue;
        above += sig ? 1 : 0;
        if (sig && atomicAdd(&a.ocnt[a.oc_off[b] + k.o], 1) == 0) atomicAdd(&a.njobs[b], 1);
        if (v > 0. && v > bw) {  // ascending entries: the first of equal weights stays
            bw = v;
            bidx = k.e;
        }
    }
    if (!bin) return;
    for (int o = 32; o > 0; o >>= 1) {
        above += __shfl_xor(above, o);
        const double ow = __shfl_xor(bw, o);
        const long long oi = __shfl_xor(bidx, o);
        if (ow > bw || (ow == bw && oi < bidx)) {
            bw = ow;
            bidx = oi;
        }
    }
    const int wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        s_bw[wv] = bw;
        s_bi[wv] = bidx;
        s_ab[wv] = above;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < kBlock / 64; ++i) {
            above += s_ab[i];
            if (s_bw[i] > bw || (s_bw[i] == bw && s_bi[i] < bidx)) {
                bw = s_bw[i];
                bidx = s_bi[i];
            }
        }
        if (above) atomicAdd((unsigned long long *)&a.part[b].n_above, (unsigned long long)above);
        a.best[blockIdx.x] = WSegBest{bw, bidx, bidx};
    }
}

// per particle of k_wseg_mask: PassStats from the particle state and its segments' maxima. One wave per particle.
__global__ void __launch_bounds__(kBlock) k_wsel_stats(CoarseWeightArgs a) {
    const int b = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (b >= a.B) return;
    const WPart p = a.part[b];
    if (p.state != kSelBin) return;
    double bw = -1.;
    long long bidx = 0x7fffffffffffffffLL;
    for (int s = a.seg_first[b] + lane; s < a.seg_first[b + 1]; s += 64) {
        const WSegBest q = a.best[s];
        if (q.w > bw || (q.w == bw && q.idx < bidx)) {
            bw = q.w;
            bidx = q.idx;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        const double ow = __shfl_xor(bw, o);
        const long long oi = __shfl_xor(bidx, o);
        if (ow > bw || (ow == bw && oi < bidx)) {
            bw = ow;
            bidx = oi;
        }
    }
    if (lane != 0) return;
    PassStats st{};
    st.min_diff2 = (double)__uint_as_float(p.mn_bits);
    st.sum_weight = p.sum;
    st.threshold = p.thr;
    st.nr_sign = p.nr_sign;
    st.n_above = p.n_above;
    st.max_weight = bw;
    st.best_key = st.best_index = bidx;
    if (p.nr_sign == 0) st.status = -5;
    a.npairs[b] = (int)p.n_above;
    a.stats[b] = st;
}

// --------------------------------------------------------------------------------------------------
// Fine-pass job lists from the coarse mask (the reference builds them on the host:
// makeJobsForDiff2Fine, src/acc/acc_helper_functions_impl.h:26-102).
// A job is one coarse orientation with >= 1 significant translation; its pairs are consecutive in
// ihidden order. pairs[] holds the particle-local coarse index o*NT + t of every significant pair.
// --------------------------------------------------------------------------------------------------

struct FineJob {
    int b;          // particle
    int o;          // orientation entry within the particle's list
    int s_begin;    // first pair (particle-local)
    int s_count;    // number of significant translations
};


// Offsets of the chunk's fine pass from the per-particle counts: exclusive scans over particles of pairs and
// jobs, fine-weight entry counts and offsets, totals and the capacity check. One block of 1024.
__global__ void __launch_bounds__(kWBlock) k_fine_plan(const int *__restrict__ n_pairs_b, const int *__restrict__ n_jobs_b,
                                                       const ChunkPtrs *__restrict__ cp, long long cap_pairs, int cap_jobs,
                                                       long long *__restrict__ pair_off, int *__restrict__ job_off,
                                                       long long *__restrict__ fine_n, long long *__restrict__ fine_off,
                                                       FinePlan *__restrict__ plan) {
    __shared__ int tmp[24];
    const int B = cp->B;
    long long pbase = 0;
    int jbase = 0;
    for (int b0 = 0; b0 < B; b0 += kWBlock) {
        const int b = b0 + threadIdx.x;
        const int np = b < B ? n_pairs_b[b] : 0, nj = b < B ? n_jobs_b[b] : 0;
        int tp, tj;
        const int ps = block_exclusive_scan_i(np, tmp, tp);
        const int js = block_exclusive_scan_i(nj, tmp, tj);
        if (b < B) {
            pair_off[b] = pbase + ps;
            job_off[b] = jbase + js;
            fine_n[b] = 32LL * np;
            fine_off[b] = 32LL * (pbase + ps);
        }
        pbase += tp;
        jbase += tj;
    }
    if (threadIdx.x == 0) {
        plan->n_pairs = pbase;
        plan->n_jobs = jbase;
        plan->n_small = plan->n_wide = 0;
        plan->next_fine = plan->next_wsum = 0;
        for (int x = 0; x < 8; ++x) plan->next_fine_x[x] = plan->next_wsum_x[x] = 0;
        plan->B = B;
        plan->overflow = (pbase > cap_pairs || jbase > cap_jobs) ? 1 : 0;
    }
}

// Writes pairs and jobs at the offsets computed by k_fine_plan: from the particle's ordered list of significant
// entries (kSelAll), or from the mask and the per-orientation significant counts (k_wseg_mask). grid (B), block 1024.
__global__ void __launch_bounds__(kWBlock) k_write_jobs(const WPart *__restrict__ part, const int *__restrict__ sig,
                                                        const unsigned char *__restrict__ mask,
                                                        const long long *__restrict__ d2_off,
                                                        const int *__restrict__ or_cnt, const int *__restrict__ oc_off,
                                                        const int *__restrict__ ocnt, int NT,
                                                        const long long *__restrict__ pair_off,
                                                        const int *__restrict__ job_off, int *__restrict__ pairs,
                                                        FineJob *__restrict__ jobs, const FinePlan *__restrict__ plan) {
    __shared__ int tmp[24];
    const int b = blockIdx.x;
    if (plan->overflow || b >= plan->B) return;
    const int state = part[b].state;
    if (state == kSelNone) return;
    int pair_base = 0, job_base = 0;
    if (state == kSelAll) {
        const int *e = sig + (size_t)b * kGather;
        const int na = (int)part[b].n_above;
        for (int i0 = 0; i0 < na; i0 += kWBlock) {
            const int i = i0 + threadIdx.x;
            int o = 0, first = 0;
            if (i < na) {
                o = e[i] / NT;
                first = (i == 0 || e[i - 1] / NT != o) ? 1 : 0;
                pairs[pair_off[b] + i] = e[i];
            }
            int tot_j;
            const int js = block_exclusive_scan_i(first, tmp, tot_j);
            if (first) {
                int c = 1;  // its entries follow
                while (i + c < na && e[i + c] / NT == o) ++c;
                jobs[job_off[b] + job_base + js] = FineJob{b, o, i, c};
            }
            job_base += tot_j;
        }
        return;
    }
    const unsigned char *m = mask + d2_off[b];
    const int n_o = or_cnt[b];
    for (int o0 = 0; o0 < n_o; o0 += kWBlock) {
        const int o = o0 + threadIdx.x;
        const int c = (o < n_o) ? ocnt[oc_off[b] + o] : 0;  // significant translations of orientation o
        int tot_p, tot_j;
        const int ps = block_exclusive_scan_i(c, tmp, tot_p);
        const int js = block_exclusive_scan_i(c > 0 ? 1 : 0, tmp, tot_j);
        if (o < n_o && c > 0) {
            int s = pair_base + ps;
            FineJob j;
            j.b = b;
            j.o = o;
            j.s_begin = s;
            j.s_count = c;
            jobs[job_off[b] + job_base + js] = j;
            for (int t = 0; t < NT; ++t)
                if (m[(size_t)o * NT + t]) pairs[pair_off[b] + (s++)] = o * NT + t;
        }
        pair_base += tot_p;
        job_base += tot_j;
    }
}

// --------------------------------------------------------------------------------------------------
// Fine pass: one block per (job, chunk of TC coarse translations); each thread owns pixels, projects the
// 8 oversampled orientations once per pixel and accumulates the 8 x 4*TC squared differences.
// --------------------------------------------------------------------------------------------------

// Jobs are keyed for the fine pass's order by class and coarse orientation (direction-major), key >> key_shift so that
// the keys fit the LDS histogram of k_fine_items.
constexpr int kJobKeys = 4096;

// Work items of the fine pass: jobs with at most small_max significant translations are one item of
// the small path of k_fine_diff2; the others one wide item per wide_tc translations. With `sorted`, the jobs are first
// put in the order of their class and coarse orientation (a counting sort over kJobKeys keys; the order within a key
// is arbitrary), so that consecutive items are jobs of nearby orientations, often of different particles: jobs of one
// coarse direction sample the same four fine-direction planes of the reference, and items processed together then
// share its corner blocks in the caches. job_order receives the order (the weighted sums follow it too); without
// `sorted` it is the identity (particle order). One block of 1024.
__global__ void __launch_bounds__(kWBlock) k_fine_items(const FineJob *__restrict__ jobs, const int *__restrict__ or_off,
                                                        const int *__restrict__ or_frame, const int *__restrict__ or_class,
                                                        int n_or_grid, int key_shift, int sorted, int small_max,
                                                        int wide_tc, int cap_small, int cap_wide, int n_pix, int n_wpix,
                                                        int *__restrict__ job_order, int2 *__restrict__ small_items,
                                                        int2 *__restrict__ wide_items, FinePlan *__restrict__ plan) {
    __shared__ int tmp[24];
    __shared__ int hist[kJobKeys];
    if (plan->overflow) return;
    const int n_jobs = plan->n_jobs;
    if (sorted) {
        for (int q = threadIdx.x; q < kJobKeys; q += kWBlock) hist[q] = 0;
        __syncthreads();
        auto key_of = [&](int j) {
            const FineJob jb = jobs[j];
            const int oe = or_off[jb.b] + jb.o;
            const long long g = (long long)or_class[oe] * n_or_grid + (or_frame[oe] >> 3);
            return (int)min((long long)(kJobKeys - 1), g >> key_shift);
        };
        for (int j = threadIdx.x; j < n_jobs; j += kWBlock) atomicAdd(&hist[key_of(j)], 1);
        __syncthreads();
        // exclusive scan of the histogram, kJobKeys / kWBlock consecutive keys per thread
        constexpr int kPer = kJobKeys / kWBlock;
        int loc[kPer], sum = 0;
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            loc[q] = hist[threadIdx.x * kPer + q];
            sum += loc[q];
        }
        int tot;
        int run = block_exclusive_scan_i(sum, tmp, tot);
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            hist[threadIdx.x * kPer + q] = run;
            run += loc[q];
        }
        __syncthreads();
        for (int j = threadIdx.x; j < n_jobs; j += kWBlock) job_order[atomicAdd(&hist[key_of(j)], 1)] = j;
    } else {
        for (int j = threadIdx.x; j < n_jobs; j += kWBlock) job_order[j] = j;
    }
    __syncthreads();
    int sbase = 0, wbase = 0;
    for (int j0 = 0; j0 < n_jobs; j0 += kWBlock) {
        const int jj = j0 + threadIdx.x;
        int ns = 0, nw = 0, sc = 0, j = 0;
        if (jj < n_jobs) {
            j = job_order[jj];
            sc = jobs[j].s_count;
            if (sc <= small_max) ns = 1;
            else nw = (sc + wide_tc - 1) / wide_tc;
        }
        int ts, tw;
        const int ss = block_exclusive_scan_i(ns, tmp, ts);
        const int ws = block_exclusive_scan_i(nw, tmp, tw);
        if (ns && sbase + ss < cap_small) small_items[sbase + ss] = make_int2(j, 0);
        for (int q = 0; q < nw; ++q)
            if (wbase + ws + q < cap_wide) wide_items[wbase + ws + q] = make_int2(j, q * wide_tc);
        sbase += ts;
        wbase += tw;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        plan->n_small = sbase;
        plan->n_wide = wbase;
        plan->fine_choice = fill_choice(sbase + wbase, n_pix);
        plan->wsum_choice = fill_choice(n_jobs, n_wpix);
        if (sbase > cap_small || wbase > cap_wide) plan->overflow = 1;
    }
}

struct FineArgs {
    const FineJob *jobs;
    const int2 *items_w;           // (job, first job-local pair) per wide work item (plan->n_wide)
    const int2 *items_s;           // per small work item (plan->n_small)
    FinePlan *plan;                // header; next_fine is the dynamic item counter
    const ChunkPtrs *cp;           // this chunk's images
    const int *pairs;
    const long long *pair_off;
    const int *or_off;
    const int *or_frame;           // fine frame base (coarse orientation * 8) per orientation entry
    const int *or_class;
    const float4 *const *vols;
    VolGeom vg;
    const Frame *fine_frames;      // [n_dir * n_psi * 8]
    ImgGeom ig;
    const float *scale;
    const float *q;                // sqrt(Minvsigma2/2) of the fine size
    const float2 *ex;              // [n_xs][xs] phase factors of the fine x shifts
    const float2 *ey;              // [n_ys][s]
    const int *tr_ix;              // [NT*4] x-shift index of fine translation t*4+u
    const int *tr_iy;
    const int2 *pix;               // sampled pixels (Minvsigma2 > 0, inside the projection radius) as (p, x | row
                                   // << 16), in n_bands bands of equal count by radius, pixel order within a band
    int n_pix;
    int n_bands;                   // band b: pix[b n_pix / n_bands .. (b + 1) n_pix / n_bands); 0: the plan's choice, pix
                                   // the lists of all choices one after the other
    int item_major;                // unit order: 0 band-major (all items of band 0, then band 1, ...), 1 item-major
    int xcd_queues;                // 1: each XCD takes its own eighth of the items (band-major), then helps the others
    int NT;
    int do_ctf;
    double *diff2;                 // [pair_off[b]*32 + s*32 + r*4 + u]: k_fine_init's base, plus each band's sum
};

// Pose-independent part of a particle's fine diff2, in FP64: highres_Xi2 / 2 + sum over the pixels with
// Minvsigma2 > 0 of |q X|^2 (q = sqrt(Minvsigma2 / 2)). The fine kernels accumulate only the pose-dependent
// remainder |A|^2 - 2 Re(A conj(Y)) of |A - Y|^2 (A the scaled projection, Y = q X shifted; |Y| = |q X|), whose
// magnitude is that of the signal, not of the noise power, so that FP32 partial sums keep the differences between
// poses that the weights exponentiate (the reference CPU path sums diff2 in double, src/ml_optimiser.cpp:7436-7442).
// grid (capacity of the chunk), block kBlock; blocks beyond the chunk's particle count return.
__global__ void __launch_bounds__(kBlock) k_fine_base(const ChunkPtrs *__restrict__ cp, const float *__restrict__ q,
                                                      int P, const double *__restrict__ xi2half,
                                                      double *__restrict__ fbase) {
    __shared__ double red[kBlock / 64];
    const int b = blockIdx.x;
    if (b >= cp->B) return;
    const float2 *X = cp->fimg + (size_t)b * P;
    double acc = 0.;
    for (int p = threadIdx.x; p < P; p += kBlock) {
        const float qp = q[p];
        if (qp == 0.f) continue;
        const float2 x = X[p];
        const double xr = (double)qp * x.x, xi = (double)qp * x.y;
        acc += xr * xr + xi * xi;
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = xi2half[b];
        for (int w = 0; w < kBlock / 64; ++w) t += red[w];
        fbase[b] = t;
    }
}

// Fine diff2 of the chunk's evaluated poses set to their particle's pose-independent part; the bands of the
// fine pass add their pose-dependent sums to it. grid (capacity of the chunk), block kBlock.
__global__ void __launch_bounds__(kBlock) k_fine_init(const int *__restrict__ n_pairs_b,
                                                      const long long *__restrict__ pair_off,
                                                      const double *__restrict__ fbase, const FinePlan *__restrict__ plan,
                                                      double *__restrict__ diff2) {
    const int b = blockIdx.x;
    if (plan->overflow || b >= plan->B) return;
    const long long n = 32LL * n_pairs_b[b];
    double *d = diff2 + 32LL * pair_off[b];
    const double v = fbase[b];
    for (long long e = threadIdx.x; e < n; e += kBlock) d[e] = v;
}

// Pixel range [i0, i1) of band `band` in FineArgs::pix.
__device__ __forceinline__ void band_range(const FineArgs &a, int band, int &i0, int &i1) {
    i0 = band * a.n_pix / a.n_bands;
    i1 = (band + 1) * a.n_pix / a.n_bands;
}

// Work-item shapes of the fine pass (chosen per engine by the tuner): a job with at most TC significant coarse
// translations is one small item; a larger job is split into wide items of 4 * CW coarse translations, CW per wave.
struct FineShape {
    int tc, cw;
};
constexpr FineShape kFineShapes[] = {{2, 2}, {1, 2}, {2, 1}, {1, 1}};
constexpr int kNumFineShapes = (int)(sizeof(kFineShapes) / sizeof(kFineShapes[0]));

// One work item on one band of pixels: a job with at most TC significant coarse translations. Each thread owns
// pixels, projects the 8 oversampled orientations once per pixel and accumulates the 8 x 4*TC squared differences.
template <int TC>
struct FineSmallLds {
    float red[kBlock / 64][8 * 4 * TC];
    int tix[4 * TC], tiy[4 * TC];
    int t[TC];
};

template <int TC>
__device__ __forceinline__ void fine_small_item(const FineArgs &a, int job_id, int first, int band,
                                                FineSmallLds<TC> &L) {
    constexpr int kFineSmallTC = TC;
    constexpr int kFineNF = 4 * kFineSmallTC;  // fine translations per block
    const FineJob job = a.jobs[job_id];
    const int b = job.b;
    const int nc = min(kFineSmallTC, job.s_count - first);
    const int tid = threadIdx.x;
    if (tid < kFineSmallTC) {
        const int s = job.s_begin + first + tid;
        L.t[tid] = (tid < nc) ? a.pairs[a.pair_off[b] + s] % a.NT : 0;
    }
    __syncthreads();
    if (tid < kFineNF) {
        const int c = tid >> 2, u = tid & 3;
        const int t = L.t[c];
        L.tix[tid] = a.tr_ix[t * 4 + u];
        L.tiy[tid] = a.tr_iy[t * 4 + u];
    }
    __syncthreads();
    const int oe = a.or_off[b] + job.o;
    const int k = a.or_class[oe];
    const Frame *fr = a.fine_frames + a.or_frame[oe];
    const float4 *vol = a.vols[k];
    const float2 *X = a.cp->fimg + (size_t)b * a.ig.P;
    const float *C = a.cp->fctf + (size_t)b * a.ig.P;
    const float sc = a.scale[b];
    float acc[8][kFineNF];
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
        for (int j = 0; j < kFineNF; ++j) acc[r][j] = 0.f;
    int i0, i1;
    band_range(a, band, i0, i1);
    // pixels with Minvsigma2 == 0 contribute nothing, those outside the projection radius only |Y|^2 (in fbase)
    for (int ip = i0 + tid; ip < i1; ip += kBlock) {
        const int2 pe = a.pix[ip];
        const int p = pe.x, x = pe.y & 0xffff, i = pe.y >> 16;
        const int y = (i < a.ig.xs) ? i : i - a.ig.s;
        const float qp = a.q[p];
        const float c = qp * (a.do_ctf ? C[p] : 1.f) * sc;
        float2 A[8];
        // every listed pixel is inside the projection radius; testing it anyway keeps the compiler from hoisting
        // all 32 corner-block loads of the 8 orientations at once (which spills registers at 3 waves per SIMD)
        const bool inside = x * x + y * y <= a.ig.proj_r2_max;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            float2 v = make_float2(0.f, 0.f);
            if (inside) v = project_pixel(vol, a.vg, fr[r], x, y);
            A[r] = make_float2(c * v.x, c * v.y);
        }
        const float2 Xp = X[p];
        const float2 Xq2 = make_float2(2.f * qp * Xp.x, 2.f * qp * Xp.y);
#pragma unroll
        for (int j = 0; j < kFineNF; ++j) {
            const float2 ph = cmul(a.ex[(size_t)L.tix[j] * a.ig.xs + x], a.ey[(size_t)L.tiy[j] * a.ig.s + i]);
            const float2 Y2 = cmul(Xq2, ph);  // 2 Y
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                // |A|^2 - 2 Re(A conj(Y)) = A.x (A.x - 2 Y.x) + A.y (A.y - 2 Y.y)
                acc[r][j] = fmaf(A[r].x, A[r].x - Y2.x, acc[r][j]);
                acc[r][j] = fmaf(A[r].y, A[r].y - Y2.y, acc[r][j]);
            }
        }
    }
    // block reduction: wave shuffles, then across the 4 waves
    const int lane = tid & 63, w = tid >> 6;
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
        for (int j = 0; j < kFineNF; ++j) {
            float v = acc[r][j];
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
            if (lane == 0) L.red[w][r * kFineNF + j] = v;
        }
    __syncthreads();
    if (tid < 8 * kFineNF) {
        const int r = tid / kFineNF, j = tid - r * kFineNF;
        const int c = j >> 2, u = j & 3;
        if (c < nc) {
            float v = 0.f;
            for (int ww = 0; ww < kBlock / 64; ++ww) v += L.red[ww][tid];
            const long long s = job.s_begin + first + c;
            atomicAdd(&a.diff2[(a.pair_off[b] + s) * 32 + r * 4 + u], (double)v);
        }
    }
}

// One work item of a job with more than TC significant translations: up to 4 * kWideCW coarse
// translations. Per tile of 64 pixels the four waves first project the 8 fine orientations together (two per
// thread) into LDS; then wave w accumulates the squared differences of its kWideCW coarse translations (4 * kWideCW
// fine translations) over the tile's pixels. A job with up to kWideTC significant translations reads each
// trilinear sample once.
template <int CW>
struct FineWideLds {
    float2 A[8][64];
    float2 X[64];
    int p[64];
    int tix[4][4 * CW], tiy[4][4 * CW];  // per wave
};

template <int CW>
__device__ __forceinline__ void fine_wide_item(const FineArgs &a, int job_id, int first, int band,
                                               FineWideLds<CW> &L) {
    constexpr int kWideCW = CW;            // coarse translations per wave
    constexpr int kWideTC = 4 * kWideCW;   // coarse translations per block
    constexpr int kNF = 4 * kWideCW;  // fine translations per wave
    const FineJob job = a.jobs[job_id];
    const int b = job.b;
    const int nc = min(kWideTC, job.s_count - first);  // coarse translations of this block
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid < 4 * kNF) {
        const int w = tid / kNF, j = tid % kNF;  // wave w, fine translation j = 4c + u
        const int c = kWideCW * w + (j >> 2), u = j & 3;
        int t = 0;
        if (c < nc) t = a.pairs[a.pair_off[b] + job.s_begin + first + c] % a.NT;
        L.tix[w][j] = a.tr_ix[t * 4 + u];
        L.tiy[w][j] = a.tr_iy[t * 4 + u];
    }
    const int oe = a.or_off[b] + job.o;
    const int k = a.or_class[oe];
    const Frame *fr = a.fine_frames + a.or_frame[oe];
    const float4 *vol = a.vols[k];
    const float2 *X = a.cp->fimg + (size_t)b * a.ig.P;
    const float *C = a.cp->fctf + (size_t)b * a.ig.P;
    const float sc = a.scale[b];
    const bool active = kWideCW * wave < nc;  // this wave has translations
    float acc[8][kNF];
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
        for (int j = 0; j < kNF; ++j) acc[r][j] = 0.f;
    int i0, i1;
    band_range(a, band, i0, i1);
    for (int t0 = i0; t0 < i1; t0 += 64) {
        __syncthreads();  // previous tile consumed (and the translation tables written, first time)
        // phase A: 8 projections of 64 sampled pixels, 2 per thread
        {
            const int ip = t0 + lane;
            float2 v0 = make_float2(0.f, 0.f), v1 = make_float2(0.f, 0.f);
            float c = 0.f;
            if (ip < i1) {
                const int2 pe = a.pix[ip];
                const int p = pe.x, x = pe.y & 0xffff, i = pe.y >> 16;
                const int y = (i < a.ig.xs) ? i : i - a.ig.s;
                const float qp = a.q[p];
                c = qp * (a.do_ctf ? C[p] : 1.f) * sc;
                v0 = project_pixel(vol, a.vg, fr[2 * wave], x, y);
                v1 = project_pixel(vol, a.vg, fr[2 * wave + 1], x, y);
                if (wave == 0) {
                    const float2 Xp = X[p];
                    L.X[lane] = make_float2(2.f * qp * Xp.x, 2.f * qp * Xp.y);  // 2 q X
                    L.p[lane] = p;
                }
            } else if (wave == 0) {
                L.p[lane] = -1;
            }
            L.A[2 * wave][lane] = make_float2(c * v0.x, c * v0.y);
            L.A[2 * wave + 1][lane] = make_float2(c * v1.x, c * v1.y);
        }
        __syncthreads();
        // phase B: this wave's fine translations over the tile
        if (active) {
            const int p = L.p[lane];
            if (p >= 0) {
                const int i = p / a.ig.xs, x = p - i * a.ig.xs;
                float2 A[8];
#pragma unroll
                for (int r = 0; r < 8; ++r) A[r] = L.A[r][lane];
                const float2 Xq2 = L.X[lane];
#pragma unroll
                for (int j = 0; j < kNF; ++j) {
                    const float2 ph = cmul(a.ex[(size_t)L.tix[wave][j] * a.ig.xs + x],
                                           a.ey[(size_t)L.tiy[wave][j] * a.ig.s + i]);
                    const float2 Y2 = cmul(Xq2, ph);  // 2 Y
#pragma unroll
                    for (int r = 0; r < 8; ++r) {
                        // pose-dependent part of |A - Y|^2 (|Y|^2 is in fbase)
                        acc[r][j] = fmaf(A[r].x, A[r].x - Y2.x, acc[r][j]);
                        acc[r][j] = fmaf(A[r].y, A[r].y - Y2.y, acc[r][j]);
                    }
                }
            }
        }
    }
    if (active) {
        // wave reduction; lanes 0 .. kWideCW-1 write the wave's translations
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int j = 0; j < kNF; ++j) {
                float v = acc[r][j];
                for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
                acc[r][j] = v;
            }
        if (lane < kWideCW) {
            const int c = kWideCW * wave + lane;  // one coarse translation per lane
            if (c < nc) {
                const long long s = job.s_begin + first + c;
                double *out = a.diff2 + (a.pair_off[b] + s) * 32;
#pragma unroll
                for (int r = 0; r < 8; ++r)
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        // acc index j = 4 * lane + u, selected without dynamic register indexing
                        float v = acc[r][u];
#pragma unroll
                        for (int q = 1; q < kWideCW; ++q)
                            if (lane == q) v = acc[r][4 * q + u];
                        atomicAdd(&out[r * 4 + u], (double)v);
                    }
            }
        }
    }
}

// Fine pass, persistent: blocks fetch work units from plan->next_fine until none is left, so uneven items spread
// over the GPU; every block exits once the counter passes the last unit. A unit is one work item on one band of
// pixels, either band-major (all items of band 0, then band 1, ...; within a band the wide items first, the heaviest,
// then the small ones), so that the units in flight sample one or two radial shells of the reference, or item-major
// (the bands of an item one after the other), so that with items in orientation order (k_fine_items) the units in
// flight sample the planes of few coarse directions. Each unit adds its partial
// sums to the FP64 diff2 (k_fine_init wrote the pose-independent part). Three waves per SIMD, as the two item
// paths have when compiled alone (at most 168 VGPRs). kTuning only separates the tuning launches from the production
// ones in kernel traces.
template <int kTuning, int TC, int CW>
__global__ void __launch_bounds__(kBlock, 3) k_fine_diff2(FineArgs a) {
    __shared__ union {
        FineSmallLds<TC> s;
        FineWideLds<CW> w;
    } lds;
    __shared__ int s_item;
    if (a.plan->overflow) return;
    if (a.n_bands == 0) {
        const int c = a.plan->fine_choice;
        a.n_bands = 1 << c;
        a.pix += (size_t)c * a.n_pix;
    }
    const int n_wide = a.plan->n_wide;
    const int n_items = n_wide + a.plan->n_small;
    const int n_units = n_items * a.n_bands;
    if (a.xcd_queues) {
        // Workgroups are dispatched to the 8 XCDs in turn, so block b runs on XCD b % 8. XCD x owns the x-th eighth of
        // the wide and of the small items (contiguous in orientation order: a subset of the directions for its L2)
        // and takes their units band-major; a block whose XCD's share is exhausted takes units of the next XCDs'
        // shares, so the pass ends when every share is. Each unit index comes from one atomic increment of its
        // share's counter, so every unit runs exactly once whichever XCD the blocks actually run on.
        __shared__ int s_queue;
        const int n_small = a.plan->n_small;
        const int home = blockIdx.x & 7;
        for (;;) {
            __syncthreads();
            if (threadIdx.x == 0) {
                int got = -1, q = 0;
                for (int k = 0; k < 8 && got < 0; ++k) {
                    const int x = (home + k) & 7;
                    const int nx = ((x + 1) * n_wide / 8 - x * n_wide / 8) + ((x + 1) * n_small / 8 - x * n_small / 8);
                    const int lim = nx * a.n_bands;
                    if (*(volatile int *)&a.plan->next_fine_x[x] >= lim) continue;  // exhausted (a stale read only
                                                                                    // costs the increment below)
                    const int u = atomicAdd(&a.plan->next_fine_x[x], 1);
                    if (u < lim) {
                        got = u;
                        q = x;
                    }
                }
                s_item = got;
                s_queue = q;
            }
            __syncthreads();
            const int unit = __builtin_amdgcn_readfirstlane(s_item);
            if (unit < 0) break;
            const int x = __builtin_amdgcn_readfirstlane(s_queue);
            const int wlo = x * n_wide / 8, nxw = (x + 1) * n_wide / 8 - wlo;
            const int slo = x * n_small / 8, nx = nxw + (x + 1) * n_small / 8 - slo;
            const int band = unit / nx, idx = unit - band * nx;
            if (idx < nxw) {
                const int2 it = a.items_w[wlo + idx];
                fine_wide_item<CW>(a, it.x, it.y, band, lds.w);
            } else {
                const int2 it = a.items_s[slo + idx - nxw];
                fine_small_item<TC>(a, it.x, it.y, band, lds.s);
            }
        }
        return;
    }
    for (;;) {
        __syncthreads();  // previous unit's LDS and s_item consumed
        if (threadIdx.x == 0) s_item = atomicAdd(&a.plan->next_fine, 1);
        __syncthreads();
        // one value per block: readfirstlane makes the branches below provably uniform, so the two item paths
        // are not linearised and do not hold their registers at the same time
        const int unit = __builtin_amdgcn_readfirstlane(s_item);
        if (unit >= n_units) break;
        int band, item;
        if (a.item_major) {
            item = unit / a.n_bands;
            band = unit - item * a.n_bands;
        } else {
            band = unit / n_items;
            item = unit - band * n_items;
        }
        if (item < n_wide) {
            const int2 it = a.items_w[item];
            fine_wide_item<CW>(a, it.x, it.y, band, lds.w);
        } else {
            const int2 it = a.items_s[item - n_wide];
            fine_small_item<TC>(a, it.x, it.y, band, lds.s);
        }
    }
}

// Resets the dynamic item counters (tuning launches of the fine pass reuse one plan).
__global__ void k_reset_items(FinePlan *plan) {
    if (threadIdx.x == 0) {
        plan->next_fine = 0;
        plan->next_wsum = 0;
        for (int x = 0; x < 8; ++x) plan->next_fine_x[x] = plan->next_wsum_x[x] = 0;
    }
}

// Sum over the B particles of each shell's weighted sigma2_noise contribution: block s sums column s of the
// [B][nshell] per-particle accumulators in a fixed order (strided partial sums, then a tree). grid (nshell).
__global__ void __launch_bounds__(kBlock) k_shell_total(const double *__restrict__ acc, int B, int nshell,
                                                        double *__restrict__ out) {
    __shared__ double red[kBlock];
    const int s = blockIdx.x, tid = threadIdx.x;
    double v = 0.;
    for (int b = tid; b < B; b += kBlock) v += acc[(size_t)b * nshell + s];
    red[tid] = v;
    __syncthreads();
    for (int o = kBlock / 2; o > 0; o >>= 1) {
        if (tid < o) red[tid] += red[tid + o];
        __syncthreads();
    }
    if (tid == 0) out[s] = red[0];
}

// What the host needs of a particle at the end of a chunk.
struct ChunkResult {
    PassStats c, f;    // coarse and fine pass
    double part[8];    // WsumArgs::part_acc
    int n_pairs;       // significant coarse poses
    int best_pair;     // coarse index of the pair that holds the best fine pose
};

// The chunk's results in one block of memory, so that they reach the host in one copy: [B] ChunkResult, then [B][K]
// pdf_class sums, the shell totals (k_shell_total) and the plan's header. (Ten separate copies of a chunk of 8 particles took 0.33 of 1.15 ms.)
__global__ void __launch_bounds__(kBlock) k_pack_results(const FinePlan *__restrict__ plan, int B, int K,
                                                         const PassStats *__restrict__ sc,
                                                         const PassStats *__restrict__ sf,
                                                         const double *__restrict__ part, const int *__restrict__ npairs,
                                                         const int *__restrict__ pairs,
                                                         const long long *__restrict__ pair_off,
                                                         const double *__restrict__ pdfc, ChunkResult *__restrict__ out,
                                                         double *__restrict__ out_pdfc, FinePlan *__restrict__ out_plan) {
    const int b = blockIdx.x * kBlock + threadIdx.x;
    if (b == 0) *out_plan = *plan;
    if (b >= B || plan->overflow) return;
    ChunkResult r;
    r.c = sc[b];
    r.f = sf[b];
    for (int i = 0; i < 8; ++i) r.part[i] = part[8 * (size_t)b + i];
    r.n_pairs = npairs[b];
    r.best_pair = r.f.best_index >= 0 ? pairs[pair_off[b] + (r.f.best_index >> 5)] : 0;
    out[b] = r;
    for (int k = 0; k < K; ++k) out_pdfc[(size_t)b * K + k] = pdfc[(size_t)b * K + k];
}

// Zero fill used inside captured graphs instead of memset nodes.
__global__ void __launch_bounds__(kBlock) k_zero_d(double *__restrict__ p, long long n) {
    for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) p[i] = 0.;
}

// --------------------------------------------------------------------------------------------------
// Weighted sums and backprojection (storeWeightedSums, src/ml_optimiser.cpp:8241-9156, with
// BackProjector::backproject2Dto3D, src/backprojector.cpp:55-357). Persistent blocks over (job, pixel band) units.
// --------------------------------------------------------------------------------------------------
constexpr int kMaxSigT = 1024;  // fine translations of one orientation (4 per coarse translation); host checks 4*NT

struct WsumArgs {
    const FineJob *jobs;
    const int *pairs;
    const long long *pair_off;
    const int *or_off;
    const int *or_frame;
    const int *or_class;
    const int *or_dir;              // global direction index per orientation entry
    const float4 *const *vols;
    VolGeom vg;
    const Frame *fine_frames;
    ImgGeom ig;
    const ChunkPtrs *cp;            // this chunk's images
    FinePlan *plan;                 // items: plan->n_jobs * 8, fetched through plan->next_wsum
    const int *job_order;           // jobs in the fine pass's order (k_fine_items)
    const float *scale_w;           // max(scale, 0.001) (src/ml_optimiser.cpp:8402-8416)
    const float *minv_w;            // Minvsigma2 with the origin restored
    const int *mresol;              // resolution shell per pixel, -1 excluded
    const int2 *wpix;               // the pixels that contribute (a shell >= 0 or backprojected) as (p, x | row << 16),
                                    // n_bands bands of equal count by radius, pixel order within a band
    int n_wpix;
    int n_bands;                    // 0: the plan's choice, wpix the lists of all choices one after the other
    int unit_order;                 // 0 band-major, 1 item-major (the bands of a job in a row), 2 band-major in per-XCD
                                    // queues
    const unsigned char *xa_shell;  // [K][nshell] data_vs_prior > 3 (scale correction) or null
    const float2 *ex;
    const float2 *ey;
    const int *tr_ix;
    const int *tr_iy;
    const double *over_x;           // [NT*4] fine shifts in pixels
    const double *over_y;
    const double *weight;           // fine weights [pair_off*32 + ...]
    const PassStats *stats;         // fine-pass stats per particle
    const double *old_off;          // [b][2]
    const double *prior_off;        // [b][2]
    double pixel_size;
    int NT;
    int nshell;
    int n_dir;
    int do_ctf;
    int do_scale;
    float *const *bp_slots;         // [K] corner-slot accumulators of the backprojectors
    double *shell_acc;              // [b][nshell] wsum sigma2_noise per particle
    double *part_acc;               // [b][8]: sumw, sigma2_offset, norm_corr, XA, AA, blocks, translations
    double *pdf_class;              // [b][K]
    double *pdf_direction;          // [K][n_dir] (all particles)
    int K;
};

__global__ void __launch_bounds__(kBlock, 5) k_wsum_bp(WsumArgs a) {
    __shared__ int s_ix[kMaxSigT], s_iy[kMaxSigT];
    __shared__ float s_w[kMaxSigT];
    __shared__ int s_tmp[24];
    __shared__ int s_cnt[8];
    __shared__ float shell[512];
    __shared__ double s_red[16];
    __shared__ long long sx_base[kBlock];
    __shared__ float sx_val[kBlock][3];
    __shared__ float sx_w[kBlock][8];
    __shared__ int s_item;
    if (a.plan->overflow) return;
    if (a.n_bands == 0) {
        const int c = a.plan->wsum_choice;
        a.n_bands = 1 << c;
        a.wpix += (size_t)c * a.n_wpix;
    }
    const int n_items = a.plan->n_jobs;
    const int n_units = n_items * a.n_bands;
    const int tid = threadIdx.x;
    // persistent: units fetched dynamically. A unit is one job (a coarse orientation of a particle with its
    // significant coarse translations) on one radial band of pixels; it visits the job's 8 oversampled orientations
    // and skips those without a significant fine pose (most of them). Band-major or item-major in one queue, or
    // band-major in per-XCD queues (XCD b % 8 first takes its eighth of the jobs, contiguous in the fine pass's
    // orientation order, then helps the others), in the fine pass's job order.
    __shared__ int s_queue;
    for (;;) {
    __syncthreads();  // previous unit's LDS and s_item consumed
    if (tid == 0) {
        if (a.unit_order == 2) {
            const int home = blockIdx.x & 7;
            int got = -1, q = 0;
            for (int k = 0; k < 8 && got < 0; ++k) {
                const int x = (home + k) & 7;
                const int lim = ((x + 1) * n_items / 8 - x * n_items / 8) * a.n_bands;
                if (*(volatile int *)&a.plan->next_wsum_x[x] >= lim) continue;
                const int u = atomicAdd(&a.plan->next_wsum_x[x], 1);
                if (u < lim) {
                    got = u;
                    q = x;
                }
            }
            s_item = got;
            s_queue = q;
        } else {
            s_item = atomicAdd(&a.plan->next_wsum, 1);
        }
    }
    __syncthreads();
    const int unit = s_item;
    if (unit >= n_units || unit < 0) break;
    int band, item;
    if (a.unit_order == 2) {
        const int x = s_queue;
        const int lo = x * n_items / 8, nx = (x + 1) * n_items / 8 - lo;
        band = unit / nx;
        item = lo + unit - band * nx;
    } else if (a.unit_order == 1) {
        item = unit / a.n_bands;
        band = unit - item * a.n_bands;
    } else {
        band = unit / n_items;
        item = unit - band * n_items;
    }
    const int job_id = a.job_order[item];
    const FineJob job = a.jobs[job_id];
    const int b = job.b;
    // a particle whose fine weights failed (zero or NaN sum) contributes nothing: its weights are not
    // normalisable and would turn the shared accumulators into NaN (the run returns the particle's status)
    if (a.stats[b].status != 0) continue;
    const double thr = a.stats[b].threshold;
    const double sumw = a.stats[b].sum_weight;
    for (int i = tid; i < a.nshell; i += kBlock) shell[i] = 0.f;
    const int oe = a.or_off[b] + job.o;
    const int k = a.or_class[oe];
    const float4 *vol = a.vols[k];
    const float2 *X = a.cp->fimg + (size_t)b * a.ig.P;
    const float2 *Xn = a.cp->fimg_nomask + (size_t)b * a.ig.P;
    const float *C = a.cp->fctf + (size_t)b * a.ig.P;
    const float scw = a.do_scale ? a.scale_w[b] : 1.f;
    float *slots = a.bp_slots[k];
    const unsigned char *xash = a.xa_shell ? a.xa_shell + (size_t)k * a.nshell : nullptr;
    double xa = 0., aa = 0., nc = 0.;
    const int sh = a.ig.xs;
    const long long base = (a.pair_off[b] + job.s_begin) * 32;
    const int n4 = 4 * job.s_count;  // fine translations of one oversampled orientation
    const int w0 = band * a.n_wpix / a.n_bands, w1 = (band + 1) * a.n_wpix / a.n_bands;
    const int n_chunks = (w1 - w0 + kBlock - 1) / kBlock;
    // significant fine poses per oversampled orientation, in one coalesced pass over the job's 32 weights per
    // significant coarse translation (entry sidx * 32 + r * 4 + u)
    if (tid < 8) s_cnt[tid] = 0;
    __syncthreads();
    for (int e = tid; e < 32 * job.s_count; e += kBlock)
        if (a.weight[base + e] >= thr) atomicAdd(&s_cnt[(e >> 2) & 7], 1);
    __syncthreads();
    for (int r = 0; r < 8; ++r) {
        if (s_cnt[r] == 0) continue;  // uniform
        // significant fine translations of orientation r, compacted in (coarse translation, sub-shift) order; their
        // normalised weights' sums (pdf_class, pdf_direction, sigma2_offset) once per job and orientation, with band 0
        int cnt = 0;
        double sw = 0., so = 0.;
        const double px2 = a.pixel_size * a.pixel_size;
        for (int e0 = 0; e0 < n4; e0 += kBlock) {
            const int e = e0 + tid;
            bool sig = false;
            double wn = 0.;
            int t = 0, u = 0;
            if (e < n4) {
                const int sidx = e >> 2;
                u = e & 3;
                const double wt = a.weight[base + (long long)sidx * 32 + r * 4 + u];
                sig = wt >= thr;
                if (sig) {
                    t = a.pairs[a.pair_off[b] + job.s_begin + sidx] % a.NT;
                    wn = wt / sumw;
                }
            }
            int tot;
            const int pos = cnt + block_exclusive_scan_i(sig ? 1 : 0, s_tmp, tot);
            if (sig) {
                if (pos < kMaxSigT) {
                    s_ix[pos] = a.tr_ix[t * 4 + u];
                    s_iy[pos] = a.tr_iy[t * 4 + u];
                    s_w[pos] = (float)wn;
                }
                if (band == 0) {
                    sw += wn;
                    const double dx = a.prior_off[2 * b] - a.old_off[2 * b] - a.over_x[t * 4 + u];
                    const double dy = a.prior_off[2 * b + 1] - a.old_off[2 * b + 1] - a.over_y[t * 4 + u];
                    so += wn * px2 * (dx * dx + dy * dy);
                }
            }
            cnt += tot;
        }
        if (cnt == 0) continue;  // uniform: cnt comes from the block scan
        if (band == 0) {
            sw = block_sum_d(sw, s_red);
            so = block_sum_d(so, s_red);
            if (tid == 0) {
                atomicAdd(&a.part_acc[8 * b + 0], sw);
                atomicAdd(&a.part_acc[8 * b + 1], so);
                atomicAdd(&a.part_acc[8 * b + 5], 1.0);
                atomicAdd(&a.part_acc[8 * b + 6], (double)cnt);
                atomicAdd(&a.pdf_class[(size_t)b * a.K + k], sw);
                atomicAdd(&a.pdf_direction[(size_t)k * a.n_dir + a.or_dir[oe]], sw);
            }
        }
        __syncthreads();  // compacted lists visible
        const int nsig = min(cnt, kMaxSigT);
        const Frame fr = a.fine_frames[a.or_frame[oe] + r];
        // the band's pixels in chunks of kBlock; each block starts at a different chunk so that concurrent blocks do
        // not all scatter into the same voxels at the same time
        const int c0 = n_chunks > 0 ? (int)(((unsigned)(8 * item + r) * 2654435761u) % (unsigned)n_chunks) : 0;
        for (int cc = 0; cc < n_chunks; ++cc) {
            int chunk = c0 + cc;
            if (chunk >= n_chunks) chunk -= n_chunks;
            const int ip = w0 + chunk * kBlock + tid;
            long long sc_base = -1;  // trilinear base voxel of this pixel's scatter (-1: none)
            float sc_val[3] = {0.f, 0.f, 0.f};
            float sc_w[8];
            if (ip < w1) {
                const int2 pe = a.wpix[ip];
                const int p = pe.x, x = pe.y & 0xffff, i = pe.y >> 16;
                const int y = (i < a.ig.xs) ? i : i - a.ig.s;
                const float ctf = (a.do_ctf ? C[p] : 1.f) * scw;
                float2 ref = make_float2(0.f, 0.f);
                if (x * x + y * y <= a.ig.proj_r2_max) {
                    const float2 v = project_pixel(vol, a.vg, fr, x, y);
                    ref = make_float2(ctf * v.x, ctf * v.y);
                }
                const int ires = a.mresol[p];
                const float minv = a.minv_w[p];
                const bool do_xa = a.do_scale && xash && ires > -1 && xash[ires];
                float wd2 = 0.f, fre = 0.f, fim = 0.f, fw = 0.f, pxa = 0.f, paa = 0.f;
                const float2 Xp = X[p], Xnp = Xn[p];
                for (int j = 0; j < nsig; ++j) {
                    const float wn = s_w[j];
                    const float2 ph = cmul(a.ex[(size_t)s_ix[j] * a.ig.xs + x], a.ey[(size_t)s_iy[j] * a.ig.s + i]);
                    if (ires > -1) {
                        const float2 Y = cmul(Xp, ph);
                        const float dr = ref.x - Y.x, di = ref.y - Y.y;
                        wd2 = fmaf(wn, dr * dr + di * di, wd2);
                        if (do_xa) {
                            pxa = fmaf(wn, ref.x * Y.x + ref.y * Y.y, pxa);
                            paa = fmaf(wn, ref.x * ref.x + ref.y * ref.y, paa);
                        }
                    }
                    const float2 Z = cmul(Xnp, ph);
                    const float wx = wn * ctf * minv;
                    fre = fmaf(Z.x, wx, fre);
                    fim = fmaf(Z.y, wx, fim);
                    fw = fmaf(wx, ctf, fw);
                }
                if (ires > -1) {
                    atomicAdd(&shell[ires], wd2);
                    nc += wd2;
                    xa += pxa;
                    aa += paa;
                }
                // backprojection of (fre, fim) with weight fw (backproject2Dto3D, src/backprojector.cpp:124-296)
                if (fw > 0.f && x * x + y * y <= a.ig.bp_r2_max && !(i >= sh && x == 0)) {
                    const float fxp = (float)x, fyp = (float)y;
                    float xp = fr.e0x * fxp + fr.e1x * fyp;
                    float yp = fr.e0y * fxp + fr.e1y * fyp;
                    float zp = fr.e0z * fxp + fr.e1z * fyp;
                    float vim = fim;
                    if (xp < 0.f) {
                        xp = -xp;
                        yp = -yp;
                        zp = -zp;
                        vim = -vim;
                    }
                    const float fx0 = floorf(xp), fy0 = floorf(yp), fz0 = floorf(zp);
                    const float fx = xp - fx0, fy = yp - fy0, fz = zp - fz0;
                    const int x0 = (int)fx0, y0 = (int)fy0 - a.vg.starty, z0 = (int)fz0 - a.vg.startz;
                    if (!(x0 < 0 || x0 + 1 >= a.vg.xdim || y0 < 0 || y0 + 1 >= a.vg.ydim || z0 < 0 ||
                          z0 + 1 >= a.vg.zdim)) {
                        const float mfx = 1.f - fx, mfy = 1.f - fy, mfz = 1.f - fz;
                        sc_base = (long long)packed_index(a.vg, x0, y0, z0);
                        sc_val[0] = fre;
                        sc_val[1] = vim;
                        sc_val[2] = fw;
                        sc_w[0] = mfz * mfy * mfx;
                        sc_w[1] = mfz * mfy * fx;
                        sc_w[2] = mfz * fy * mfx;
                        sc_w[3] = mfz * fy * fx;
                        sc_w[4] = fz * mfy * mfx;
                        sc_w[5] = fz * mfy * fx;
                        sc_w[6] = fz * fy * mfx;
                        sc_w[7] = fz * fy * fx;
                    }
                }
            }
            // Scatter of the block's pixels into the corner slots. The 24 values of one pixel share one 128-byte
            // slot line; lanes are regrouped through LDS so that each atomic instruction covers two pixels'
            // lines (32 lanes each) instead of 64 lines, which is what bounds atomic throughput.
            __syncthreads();
            sx_base[tid] = sc_base;
#pragma unroll
            for (int c = 0; c < 3; ++c) sx_val[tid][c] = sc_val[c];
#pragma unroll
            for (int c = 0; c < 8; ++c) sx_w[tid][c] = (sc_base >= 0) ? sc_w[c] : 0.f;
            __syncthreads();
            {
                const int lane = tid & 63, wave0 = tid & ~63;
                const int f = lane & 31;
                for (int k2 = 0; k2 < 32; ++k2) {
                    const int src = wave0 + 2 * k2 + (lane >> 5);
                    const long long sb = sx_base[src];
                    if (sb >= 0 && f < 24) atomicAdd(slots + kSlot * sb + f, sx_w[src][f & 7] * sx_val[src][f >> 3]);
                }
            }
        }
        __syncthreads();  // this orientation's lists consumed before the next one's are written
    }  // r
    nc = block_sum_d(nc, s_red);
    xa = block_sum_d(xa, s_red);
    aa = block_sum_d(aa, s_red);
    __syncthreads();
    double *sa = a.shell_acc + (size_t)b * a.nshell;
    for (int s2 = tid; s2 < a.nshell; s2 += kBlock)
        if (shell[s2] != 0.f) atomicAdd(&sa[s2], (double)shell[s2]);
    if (tid == 0 && (nc != 0. || xa != 0. || aa != 0.)) {
        atomicAdd(&a.part_acc[8 * b + 2], nc);
        atomicAdd(&a.part_acc[8 * b + 3], xa);
        atomicAdd(&a.part_acc[8 * b + 4], aa);
    }
    }  // units
}

}  // namespace rlnk
