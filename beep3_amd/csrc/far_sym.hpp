// Direct far field over symmetric tile pairs (the 1-point interaction of
// kernels_far.hip), for up to FAR_SYM_MAX patches.
//
// Targets in leaf order form super-tiles of 256.  A block takes one super-tile
// A (wave w, lane l: target 256 A + 64 w + l, in registers) and a run of
// 64-patch tiles J of the super-tiles A, A + 1, ..., A + nsup / 2 (cyclic), so
// every unordered pair of super-tiles meets once.  At step k lane l meets
// source (l + k) mod 64 of J (read from LDS, no two lanes the same) and the
// pair is evaluated once for both directions: distance, 1/r, e^-kr, the
// kernel derivatives and the three normal products are shared, 16 fused
// multiply-adds apply them.  The sums of the lane's own target stay in its
// registers; those of J's targets travel: a sum moves one lane down each step
// (DPP wave rotation), so it is always in the lane that meets its target and
// is back in lane j after 64 steps.  (LDS float atomics instead of the
// rotation took 90 us for one tile of 64 steps.)
//
// Bound by VALU issue: about 95 FP64 (57 FP32) instructions per unordered
// pair, where the one-directional kernel spends 153 issue slots per ordered
// pair (FP64).  Alone on an MI355X at 10,242 / 20,000 patches: 160 / 578 us
// FP64, 82 / 284 us FP32 (one-directional: 410 us FP64 at 10,242); occupancy
// 4 to 6 waves per SIMD makes no difference.
//
// Partial sums in far_part, in leaf order (no atomics in memory):
//   [segment][f, h][n]   of A's targets over the block's tiles
//   [distance][f, h][n]  of J's targets over A = J - distance (1 .. nsup / 2)
#pragma once

#include <hip/hip_runtime.h>

#include "device.hpp"

namespace beepdev {

constexpr int FAR_SUP = 256;

// nsup super-tiles; nseg segments of G tiles each per super-tile; npj
// partner distances
__host__ __device__ inline int far_sym_partners(int nsup, int a) {
    return nsup & 1 ? nsup / 2 : nsup / 2 - (a < nsup / 2 ? 0 : 1);
}
__host__ __device__ inline FarSymShape far_sym_shape(int n) {
    FarSymShape s;
    s.nsup = (n + FAR_SUP - 1) / FAR_SUP;
    s.npj = s.nsup / 2;
    // about 1,500 blocks (6 per CU) where there is that much work, at least
    // one tile per block
    const int tiles = 4 * (s.npj + 1);
    const long long total = (long long)s.nsup * tiles;
    s.G = int(total / 1536 < 1 ? 1 : total / 1536);
    s.nseg = (tiles + s.G - 1) / s.G;
    return s;
}

// e^-v for v >= 0 in FP64: v = n ln 2 - r with ln 2 split in two parts (Cody
// and Waite), |r| <= ln 2 / 2, e^r = 1 + r + r^2/2 + r^3 q(r) with q of degree 8
// by Remez's exchange (relative error of e^r below 2^-57.1 in exact arithmetic,
// with the coefficients rounded), scaled by 2^-n.  v is cut at 750 (e^-750 is
// zero), the only range check that arguments of one sign need.  Within
// 1.28 x 2^-53 of the exact value and 0.443 x 2^-53 in the mean square for v up
// to 700 (exp(-v): 1.25 and 0.443; 4 million values each).
__device__ __forceinline__ double exp_neg64(double v) {
    v = fmin(v, 750.0);
    const double n = rint(v * 1.4426950408889634);
    double r = fma(n, 0x1.62e42fee00000p-1, -v);
    r = fma(n, 0x1.a39ef35793c76p-33, r);
    double p = 0x1.ad9b514941fe2p-26;
    p = fma(p, r, 0x1.289c4059916afp-22);
    p = fma(p, r, 0x1.71def29152a3bp-19);
    p = fma(p, r, 0x1.a019aebd5ae4dp-16);
    p = fma(p, r, 0x1.a01a01551099fp-13);
    p = fma(p, r, 0x1.6c16c17b85d4bp-10);
    p = fma(p, r, 0x1.111111111a9f7p-7);
    p = fma(p, r, 0x1.555555555366ap-5);
    p = fma(p, r, 0x1.555555555554ep-3);
    p = fma(p, r, 0.5);
    p = fma(p, r, 1.0);
    p = fma(p, r, 1.0);
    return ldexp(p, -int(n));
}

template <typename T>
struct FarSymMath;
template <>
struct FarSymMath<float> {
    static __device__ __forceinline__ float rsqrt_(float v) { return __builtin_amdgcn_rsqf(v); }
    static __device__ __forceinline__ float exp_neg(float v) { return __expf(-v); }
};
template <>
struct FarSymMath<double> {
    static __device__ __forceinline__ double rsqrt_(double v) { return rsqrt_nr(v); }
    static __device__ __forceinline__ double exp_neg(double v) { return exp_neg64(v); }
};

// a patch as target and source: position relative to the block's origin,
// normal, a f (sf), a h (sh), 1/eps
template <typename T>
struct FarPatch {
    T x, y, z, nx, ny, nz, sf, sh, ie, isf;  // isf = sf / eps
};

template <typename T>
struct FarSymLds {
    static constexpr int NV = 16 / int(sizeof(T));           // values per 16-byte word
    static constexpr int NW = (10 + NV - 1) / NV;             // words per record
    typedef T word __attribute__((ext_vector_type(16 / sizeof(T))));
    word rec[NW][64];
    T acc[4][2][64];
};

// patch t of the leaf order (out of range: no source, far from everything)
template <typename T>
__device__ __forceinline__ FarPatch<T> far_sym_load(int t, int n, const int* __restrict__ order,
                                                    const Patch64* __restrict__ patches,
                                                    const double* __restrict__ x, double ox, double oy,
                                                    double oz) {
    if (t >= n) return FarPatch<T>{T(1e6), T(1e6), T(1e6 + 37.0 * (t - n)), T(0), T(0), T(0), T(0), T(0), T(0), T(0)};
    const int i = order[t];
    const Patch64 p = patches[i];
    const double sf = p.area * x[i];
    return FarPatch<T>{T(p.cx - ox), T(p.cy - oy), T(p.cz - oz), T(p.nx), T(p.ny), T(p.nz),
                       T(sf), T(p.area * x[n + i]), T(p.inv_eps), T(sf * p.inv_eps)};
}

// the value of lane l + 1 (of lane 0 in lane 63)
__device__ __forceinline__ float lane_above(float v) {
    constexpr int WAVE_ROL1 = 0x134;
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), WAVE_ROL1, 0xf, 0xf, false));
}
__device__ __forceinline__ double lane_above(double v) {
    constexpr int WAVE_ROL1 = 0x134;
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), WAVE_ROL1, 0xf, 0xf, false),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), WAVE_ROL1, 0xf, 0xf, false));
}

template <typename T>
struct FarPair {
    T A0, L1, E1, X, a, b;  // see far_sym_block
};
// what both directions of the pair (i, j) share, d = y_j - x_i:
// A0 = u - G, L1 = 1/r^3, E1 = g1, a = n_i.d, b = n_j.d,
// X = (gL1 - g1) n_i.n_j - a b (gL2 - g2)
template <typename T>
__device__ __forceinline__ FarPair<T> far_pair(const FarPatch<T>& i, const FarPatch<T>& j, T kappa) {
    const T dx = j.x - i.x, dy = j.y - i.y, dz = j.z - i.z;
    const T r2 = dx * dx + dy * dy + dz * dz;
    const T ir = FarSymMath<T>::rsqrt_(r2);
    const T kr = kappa * (r2 * ir);
    const T e = FarSymMath<T>::exp_neg(kr);
    const T ir2 = ir * ir;
    FarPair<T> p;
    p.A0 = e * ir - ir;
    p.L1 = ir2 * ir;
    p.E1 = (e * kr + e) * p.L1;
    p.a = i.nx * dx + i.ny * dy + i.nz * dz;
    p.b = j.nx * dx + j.ny * dy + j.nz * dz;
    const T nn = i.nx * j.nx + i.ny * j.ny + i.nz * j.nz;
    const T q = (kr * (kr + T(3)) + T(3)) * e;
    p.X = (p.L1 - p.E1) * nn - (T(3) - q) * (p.L1 * ir2) * (p.a * p.b);
    return p;
}

// block (super-tile, segment) number `task`
template <typename T>
__device__ __forceinline__ void far_sym_block(FarSymLds<T>& sm, int task, FarSymShape fs, int n,
                                              const int* __restrict__ order, const Patch64* __restrict__ patches,
                                              const double* __restrict__ x, T kappa, T* __restrict__ part) {
    using Lds = FarSymLds<T>;
    const int A = task / fs.nseg, seg = task - A * fs.nseg;
    const int tiles = 4 * (far_sym_partners(fs.nsup, A) + 1);
    const int q0 = seg * fs.G, q1 = min(q0 + fs.G, tiles);
    if (q0 >= q1) return;
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    const Patch64& org = patches[order[A * FAR_SUP]];
    const double ox = org.cx, oy = org.cy, oz = org.cz;
    const int ti = A * FAR_SUP + t;
    const FarPatch<T> me = far_sym_load<T>(ti, n, order, patches, x, ox, oy, oz);
    T fi = 0, hi = 0;
    for (int q = q0; q < q1; ++q) {
        const int dist = q >> 2;
        int B = A + dist;
        if (B >= fs.nsup) B -= fs.nsup;
        const int j0 = B * FAR_SUP + 64 * (q & 3);
        if (j0 >= n) continue;  // the last super-tile's missing tiles (uniform over the block)
        __syncthreads();        // the previous tile is consumed
        if (t < 64) {
            const FarPatch<T> p = far_sym_load<T>(j0 + t, n, order, patches, x, ox, oy, oz);
            T v[Lds::NW * Lds::NV] = {p.x, p.y, p.z, p.nx, p.ny, p.nz, p.sf, p.sh, p.ie, p.isf};
#pragma unroll
            for (int c = 0; c < Lds::NW; ++c) {
                typename Lds::word u;
#pragma unroll
                for (int e = 0; e < Lds::NV; ++e) u[e] = v[c * Lds::NV + e];
                sm.rec[c][t] = u;
            }
        }
        __syncthreads();
        auto record = [&](int jl) {
            T v[Lds::NW * Lds::NV];
#pragma unroll
            for (int c = 0; c < Lds::NW; ++c) {
                const typename Lds::word u = sm.rec[c][jl];
#pragma unroll
                for (int e = 0; e < Lds::NV; ++e) v[c * Lds::NV + e] = u[e];
            }
            return FarPatch<T>{v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9]};
        };
        if (dist == 0) {
            // within the super-tile: every wave meets all four tiles, its own
            // targets only; step 0 of its own tile is the patch itself
            for (int k = (q & 3) == w ? 1 : 0; k < 64; ++k) {
                const FarPatch<T> j = record((l + k) & 63);
                const FarPair<T> p = far_pair(me, j, kappa);
                fi = fma(j.sf * p.b, p.E1 - j.ie * p.L1, fma(j.sh, p.A0, fi));
                hi = fma(j.sh * p.a, j.ie * p.E1 - p.L1, fma(j.isf, p.X, hi));
            }
            continue;
        }
        T fj = 0, hj = 0;  // of target (l + k) mod 64 of J
#pragma unroll 2
        for (int k = 0; k < 64; ++k) {
            const FarPatch<T> j = record((l + k) & 63);
            const FarPair<T> p = far_pair(me, j, kappa);
            fi = fma(j.sf * p.b, p.E1 - j.ie * p.L1, fma(j.sh, p.A0, fi));
            hi = fma(j.sh * p.a, j.ie * p.E1 - p.L1, fma(j.isf, p.X, hi));
            // the other direction: d -> -d
            fj = fma(me.sf * p.a, me.ie * p.L1 - p.E1, fma(me.sh, p.A0, fj));
            hj = fma(me.sh * p.b, p.L1 - me.ie * p.E1, fma(me.isf, p.X, hj));
            fj = lane_above(fj);
            hj = lane_above(hj);
        }
        sm.acc[w][0][l] = fj;
        sm.acc[w][1][l] = hj;
        __syncthreads();
        if (t < 128 && j0 + l < n) {
            const T v = (sm.acc[0][w][l] + sm.acc[1][w][l]) + (sm.acc[2][w][l] + sm.acc[3][w][l]);
            part[(size_t(fs.nseg + dist - 1) * 2 + w) * n + j0 + l] = v;
        }
    }
    if (ti < n) {
        part[size_t(seg) * 2 * n + ti] = fi;
        part[(size_t(seg) * 2 + 1) * n + ti] = hi;
    }
}

// the far field of leaf-order target t: its partial sums in a fixed order
template <typename T>
__device__ __forceinline__ void far_sym_row(FarSymShape fs, int n, int t, const T* __restrict__ part, double& f,
                                            double& h) {
    const int A = t / FAR_SUP;
    const int nseg = (4 * (far_sym_partners(fs.nsup, A) + 1) + fs.G - 1) / fs.G;
    // distances at which A is met as a partner: every one below nsup / 2, and
    // that one too unless an even ring meets it from the other side
    const int npj = fs.nsup & 1 ? fs.npj : fs.npj - (A < fs.nsup / 2 ? 1 : 0);
    f = h = 0;
#pragma unroll 4
    for (int s = 0; s < nseg; ++s) {
        f += double(part[size_t(s) * 2 * n + t]);
        h += double(part[(size_t(s) * 2 + 1) * n + t]);
    }
#pragma unroll 4
    for (int s = fs.nseg; s < fs.nseg + npj; ++s) {
        f += double(part[size_t(s) * 2 * n + t]);
        h += double(part[(size_t(s) * 2 + 1) * n + t]);
    }
}

}  // namespace beepdev
