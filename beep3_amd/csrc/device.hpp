// Internal declarations shared by the HIP translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <string>
#include <unordered_map>

namespace beepdev {

constexpr double FOUR_PI_INV = 0.07957747154594767;  // 1 / (4 pi)

// One point of a node patch, stored relative to the centroid of the patch it
// belongs to (the "local frame": distances between nearby points are then
// formed from small numbers, which keeps FP32 differences accurate).
template <typename T>
struct alignas(16) Pt {
    T x, y, z, w;     // offset from own patch centroid, weight
    T nx, ny, nz, pad;
};
using Pt32 = Pt<float>;
using Pt64 = Pt<double>;

// Patch record: centroid and area, unit normal and 1/eps.
struct alignas(16) Patch64 {
    double cx, cy, cz, area;
    double nx, ny, nz, inv_eps;
};

// Far-field source record (FP64): position + 1/eps, dipole vector a f n and
// monopole a h.
struct alignas(16) Src64 {
    double x, y, z, inv_eps;
    double dx, dy, dz, sh;
};

// Workgroups are dispatched round-robin over the 8 XCDs of an MI355X, each
// with its own L2.  xcd_remap turns block b of n into a logical index such
// that consecutive logical indices run on the same XCD, so blocks that share
// data (same M2L offset, neighbouring leaves) share one L2.
__device__ __forceinline__ int xcd_remap(int b, int n) {
    constexpr int NX = 8;
    const int q = n / NX, r = n % NX;
    const int x = b % NX, k = b / NX;
    return x * q + min(x, r) + k;
}

// 1/sqrt(v) in FP64: the hardware estimate y (relative error below 2^-24)
// refined by the series of (1 - e)^(-1/2) to second order in e = 1 - v y^2,
// whose third-order remainder is below 2^-70.  Five operations, where two
// Newton steps take seven, and the same error: within 1.25 x 2^-53 of the exact
// value, 0.475 x 2^-53 in the mean square (4 million values each around 1, small,
// large and near either end of the range).
__device__ __forceinline__ double rsqrt_nr(double v) {
    const double y = __builtin_amdgcn_rsq(v);
    const double e = fma(-(v * y), y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// FMM leaf cell of a patch packed as x | y << 10 | z << 20 (leaf level
// <= 10): two patches meet in the FMM leaf pass iff every field differs by
// at most 1.
constexpr int FMM_CELL_BITS = 10;
__host__ __device__ inline bool fmm_cells_adjacent(unsigned a, unsigned b) {
    constexpr unsigned M = (1u << FMM_CELL_BITS) - 1;
    bool ok = true;
    for (int f = 0; f < 3; ++f) {
        const int u = int((a >> (FMM_CELL_BITS * f)) & M), v = int((b >> (FMM_CELL_BITS * f)) & M);
        ok = ok && u - v <= 1 && v - u <= 1;
    }
    return ok;
}

inline void hip_check(hipError_t e, const char* what) {
    if (e != hipSuccess)
        throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// Named grow-only device buffers.  A name keeps its allocation until a larger
// size is asked for, so a plan rebuilt for a new geometry of no larger size
// allocates and frees nothing (hipFree waits for the whole device, which
// would stall other contexts running on it).
struct DevArena {
    struct Slot {
        void* p = nullptr;
        size_t bytes = 0;
    };
    std::unordered_map<std::string, Slot> slots;
    size_t held = 0;
    DevArena() = default;
    DevArena(const DevArena&) = delete;
    DevArena& operator=(const DevArena&) = delete;
    ~DevArena() { release(); }
    // grow-only, a regrowth with 25 % headroom (plans of varying size reuse
    // their buffers; a free waits for the whole device)
    void* get(const std::string& name, size_t bytes) {
        Slot& sl = slots[name];
        if (sl.p && bytes <= sl.bytes) return sl.p;
        size_t b = bytes ? bytes : 16;
        if (sl.p) {
            b = std::max(b, sl.bytes + sl.bytes / 4);
            (void)hipFree(sl.p);
            held -= sl.bytes;
            sl = Slot{};
        }
        hip_check(hipMalloc(&sl.p, b), "hipMalloc");
        sl.bytes = b;
        held += b;
        return sl.p;
    }
    template <typename T>
    T* get(const std::string& name, size_t count) {
        return static_cast<T*>(get(name, count * sizeof(T)));
    }
    void release() {
        for (auto& kv : slots)
            if (kv.second.p) (void)hipFree(kv.second.p);
        slots.clear();
        held = 0;
    }
};

// A point set whose points come in runs of gs that lie in one plane and share
// its unit normal (a planar triangle's points): per run the normal n and n.p
// (local frame, FP64), and per patch an upper bound of |p|; for FP32 kernels the
// points again as position and weight alone.  Both point arrays have one unused
// entry behind the last (the kernels load one point ahead).  gs = 0: no such
// structure (curved triangles).  Run of a patch's first point k: k / gs.
struct PointPlanes {
    const double4* plane = nullptr;
    const float* radius = nullptr;
    const float4* xyzw = nullptr;
    int gs = 0;
};
// Shorter runs keep a normal per point: 10,242 patches with one point per
// sub-triangle (runs of 2), FP32, take 488 us so and 516 by runs, on the fly 784
// and 1,127 (FP64 697 and 680, 1,030 and 1,029).  8 is the next length a rule
// gives: FP32 998 us and 800 by runs, FP64 1,843 and 1,416.
constexpr int MIN_RUN = 4;

// ---- launchers (defined in the .hip files) ----
// singular self terms; a bad one (|v| > maxv or not finite) is zeroed and
// counted in *repaired; guard_only: check the stored terms and recompute only
// the bad ones
void launch_singular(hipStream_t s, int n, const Patch64* patches, const double* gc,
                     const int* gal_ptr, const Pt64* gal, double kappa, int guard_only,
                     double maxv, unsigned* repaired, double* diag4);

// Near-singular entries of an FP32 coefficient set, listed by the FP32
// coefficient kernel and computed in FP64 afterwards: global entry index,
// row patch, 2 * column patch + (1 if the entry stores full - 1 point).
struct NsRec {
    int64_t idx;
    int i, j2;
};
struct NsList {
    NsRec* rec = nullptr;      // null: no FP64 pass (every entry in FP32)
    unsigned* count = nullptr; // records listed (may exceed cap: the rest stay FP32)
    unsigned cap = 0;
};

// Entry idx of an FP64 coefficient set: (A, B) at coef64_at(idx), (C, D) 64
// places on (double2): runs of 64 entries hold their (A, B) and then their (C,
// D), so that a wave's load of consecutive entries reads one contiguous 1 KB
// (interleaved per entry, each of its two loads skips every other 16 bytes and
// a streaming load fetches every line twice).  With streaming loads the FP64
// SpMV at 163,842 patches takes 1,351 us (1,462 interleaved, ordinary loads).
__host__ __device__ inline int64_t coef64_at(int64_t idx) { return idx + (idx & ~int64_t(63)); }
constexpr int COEF64_CD = 64;
inline size_t coef64_size(long long entries) { return (size_t(entries) + 63) / 64 * 128; }
// near-field coefficients; coef points to float4 (FP32) or double2 (FP64)
void launch_near_coeffs_fp32(hipStream_t s, int n_blocks, int n_leaves, const int* blk_ptr,
                             const int* leaf_ptr, const int* leaf_idx, const int* nb_ptr,
                             const int* nb_idx, const int64_t* coef_off, const Patch64* patches,
                             const int* qual_ptr, const Pt32* qual, const int* quad_ptr,
                             const Pt32* quad, const PointPlanes& planes, float kappa, const unsigned* cellkey, const NsList& ns, const NsList& guard,
                             double maxv, float4* coef);
// the FP64 pass over the near-singular entries the FP32 kernel listed (a bad
// result is zeroed and counted in *repaired)
void launch_near_fix64(hipStream_t s, const NsList& ns, const Patch64* patches, const int* qual_ptr,
                       const Pt64* qual, const int* quad_ptr, const Pt64* quad, const PointPlanes& planes,
                       double kappa, double maxv, unsigned* repaired, float4* coef);
// coefficient guard: list the entries of a stored set with a value |v| >
// maxv or not finite (the coefficient kernels list theirs as they go), then
// recompute the listed ones in FP64 (zero if still bad, or a self pair).
// subtract_1pt: as the set was computed; 0, a set of full rules with no far
// field beside it, is judged by full - 1 point and falls back to the 1 point
void launch_coef_scan(hipStream_t s, int fp32, int n_blocks, int n_leaves, const int* blk_ptr,
                      const int* leaf_ptr, const int* leaf_idx, const int* nb_ptr, const int* nb_idx,
                      const int64_t* coef_off, const unsigned* cellkey, int subtract_1pt,
                      const Patch64* patches, double kappa, const void* coef, double maxv, const NsList& out);
void launch_coef_repair(hipStream_t s, int fp32, const NsList& list, const Patch64* patches,
                        const int* qual_ptr, const Pt64* qual, const int* quad_ptr, const Pt64* quad,
                        const PointPlanes& planes, double kappa, int subtract_1pt, double maxv,
                        unsigned* repaired, void* coef);
void launch_near_coeffs_fp64(hipStream_t s, int n_blocks, int n_leaves, const int* blk_ptr,
                             const int* leaf_ptr, const int* leaf_idx, const int* nb_ptr,
                             const int* nb_idx, const int64_t* coef_off, const Patch64* patches,
                             const int* qual_ptr, const Pt64* qual, const int* quad_ptr,
                             const Pt64* quad, const PointPlanes& planes, double kappa, int subtract_1pt,
                             const unsigned* cellkey, const NsList& guard, double maxv,
                             double2* coef);

// Work decomposition of the near-field SpMV (built on the host from the
// tree): work items (leaf, first row, first column, columns + rows << 16) of
// <= 256 rows x <= SPMV_CW columns, and row groups (leaf, first row, rows,
// first work item) with their work-item counts; the partials of consecutive
// items are pstride rows apart.
constexpr int SPMV_CW = 512;
// rows per work item of the on-the-fly near field (launch_near_fly)
constexpr int FLY_RB = 64;
struct SpmvPlan {
    const int4* work = nullptr;
    int n_work = 0;
    const int4* groups = nullptr;
    const int* group_nblk = nullptr;
    int n_groups = 0;
    int pstride = 256;
};
// y = near(x) + diag(x), overwriting y.  mode: 0 FP64 coef/FP64 sums,
// 1 FP32 coef/FP32 sums, 2 FP32 coef/FP64 sums.  part: scratch of
// n_work * pstride * 2 doubles.  max_blocks > 0 caps the grid (blocks then take
// the work items from the counter *next, zero before and after); depth (1, 2, 4) scales the coefficient
// loads each thread keeps in flight.
// ncopies (1 or 2) copies of the near field at patch offsets copy_offset
// (null: 0) share one pass over the coefficients; part then holds ncopies x
// n_work * pstride * 2 values.
void launch_near_spmv(hipStream_t s, int mode, int n, const SpmvPlan& p, const int* leaf_ptr,
                      const int* leaf_idx, const int* nb_ptr, const int* nb_idx,
                      const int64_t* coef_off, const float4* coef32, const double2* coef64,
                      const double* diag4, const double* x, void* part, double* y,
                      int max_blocks, int depth, unsigned* next, int ncopies = 1,
                      const int* copy_offset = nullptr);
// The same product with every explicit pair integrated on the fly (no
// coefficients stored), over a plan of row groups of <= FLY_RB rows; part
// holds 2 * FLY_RB values per work item.  subtract_1pt: pairs give full - 1
// point, except those of adjacent FMM leaf cells (cellkey; null with the
// direct far field); 0 (FP64 only): full rules, as a folded set's; ns64: FP32 near-singular pairs in FP64.
void launch_near_fly(hipStream_t s, int mode, int n, const SpmvPlan& p, const int* leaf_ptr,
                     const int* leaf_idx, const int* nb_ptr, const int* nb_idx, const Patch64* patches,
                     const int* qual_ptr, const Pt32* qual32, const Pt64* qual64, const int* quad_ptr,
                     const Pt32* quad32, const Pt64* quad64, const PointPlanes& planes, double kappa, int subtract_1pt,
                     const unsigned* cellkey,
                     int ns64, double maxv, const double* diag4, const double* x, void* part, double* y);

// explicit pairs listed one by one: coefficients (FP64, rounded to FP32 as
// well; bad values zeroed and counted), and y += their products over the
// rows that have pairs (CSR: rows, ptr, col; mode as launch_near_spmv)
void launch_pair_coeffs(hipStream_t s, long long n_pairs, const int* pi, const int* pj,
                        const Patch64* patches, const int* qual_ptr, const Pt64* qual, const int* quad_ptr,
                        const Pt64* quad, const PointPlanes& planes, double kappa, double maxv,
                        unsigned* repaired, float4* c32, double2* c64);
void launch_pair_spmv(hipStream_t s, int mode, int n, int n_rows, const int* rows, const int* ptr,
                      const int* col, const float4* c32, const double2* c64, const double* x, double* y);
// pairs between copies (contiguous ranges of ns patches at copy_off) closer
// than rc; sphere: per copy (centre xyz, radius); chunk_sph: per copy, the
// spheres of its chunks of 256 consecutive patches.  ptr null: count[i] =
// pairs of row i; else their columns at cols[ptr[i]..] (index order) and
// rows_of[] = i
void launch_cut_pairs(hipStream_t s, int N, int ncopies, int ns, const int* copy_off, const double4* sphere,
                      const double4* chunk_sph, const Patch64* patches, double rc, const int* ptr, int* count,
                      int* cols, int* rows_of);
void launch_iota(hipStream_t s, int n, int* out);
// exclusive prefix sum of n ints (temporary storage of the size the first
// function gives)
size_t exclusive_scan_temp_bytes(int n);
void launch_exclusive_scan(hipStream_t s, void* tmp, size_t tmp_bytes, const int* in, int* out, int n);

// far field: pack sources from x, then y += full 1-point sum over all pairs
void launch_far_pack(hipStream_t s, int n, const Patch64* patches, const int* order,
                     const double* x, Src64* src);
// source-run splits of the direct far field that fill the chip (n_cu CUs)
int far_direct_splits(int n, int n_cu);
// The direct far field over symmetric tile pairs (far_sym.hpp), up to
// FAR_SYM_MAX patches: its partial sums are (nseg + npj) * 2 n values of the
// far field's precision.
constexpr int FAR_SYM_MAX = 20480;
struct FarSymShape {
    int nsup = 0, G = 1, nseg = 0, npj = 0;
};
FarSymShape far_sym_plan(int n);
inline size_t far_sym_values(int n) {
    const FarSymShape s = far_sym_plan(n);
    return size_t(s.nseg + s.npj) * 2 * size_t(n);
}
// part = the far field's partial sums from x; then y += them
void launch_far_sym(hipStream_t s, int fp32, int n, const int* order, const Patch64* patches, const double* x,
                    double kappa, void* part);
void launch_far_sym_add(hipStream_t s, int fp32, int n, const int* order, const void* part, double* y);
// y = near(x) + diag(x) + direct far field(x) in two launches (modes as
// launch_near_spmv; part as there, far_part far_sym_values(n) doubles)
void launch_direct_matvec(hipStream_t s, int mode, int n, const SpmvPlan& p, const int* leaf_ptr,
                          const int* leaf_idx, const int* nb_ptr, const int* nb_idx, const int64_t* coef_off,
                          const float4* coef32, const double2* coef64, const double* diag4, const Patch64* patches,
                          double kappa, const double* x, int depth, void* part, void* far_part, double* y);
// y += direct far field; n_split > 1 needs part: 2 n n_split doubles
void launch_far_direct(hipStream_t s, int fp32, int n, int n_split, const int* order,
                       const Patch64* patches, const Src64* src, double kappa, double* y,
                       double* part);

// RHS and energy coefficients (FP64 direct sums)
void launch_rhs(hipStream_t s, int n, const int* qual_ptr, const Pt64* qual,
                const Patch64* patches, int n_charges, const double* xyzq, double scale,
                double* b);
void launch_energy_coeffs(hipStream_t s, int n, const int* gal_ptr, const Pt64* gal,
                          const Patch64* patches, const PointPlanes& planes, const int* patch_inst,
                          const int* inst_charge_ptr, const double* xyzq, double* ec_f,
                          double* ec_h);

// vector kernels for the GMRES driver
void launch_multi_dot(hipStream_t s, int n, const double* V, int ncols, const double* w,
                      double* partial, int n_part_blocks);
void launch_reduce_partials(hipStream_t s, int ncols, const double* partial, int n_part_blocks,
                            double* out);
void launch_gemv_sub(hipStream_t s, int n, const double* V, int ncols, const double* h,
                     double* w);
void launch_axpby(hipStream_t s, int n, double a, const double* x, double b, double* y);
void launch_fill(hipStream_t s, int n, double v, double* y);
// Arnoldi step (classical Gram-Schmidt against V[0..j], norm, V[j+1]) on
// the mat-vec output w, with j read from *jp; h receives the j + 2 values.
// h2 non-null: a second Gram-Schmidt pass (its coefficients in h2, added to h)
void launch_arnoldi_step(hipStream_t s, int n, int m, int nb, double* V, const int* jp,
                         double* partial, double* h, double* w, double* h2);
void launch_copy_col(hipStream_t s, int n, const double* V, const int* jp, double* out);
// dst row r = src row idx[r] over 64-byte rows (a scattered read of known size)
void launch_gather_rows64(hipStream_t s, const void* src, const int* idx, size_t rows, void* dst);

// octree build on the device (octree_dev.hip): descent keys of the patch
// centroids in the cube (centre, edge) when full is null, else the prefixes
// at `level` of the full keys; items[i] = i
void launch_tree_keys(hipStream_t s, int n, const Patch64* patches, const double* centre,
                      double edge, int level, const uint64_t* full, uint64_t* keys, int* items);
// stable radix sort of (key, item) pairs over key bits [0, end_bit)
size_t tree_sort_bytes(int n, int end_bit);
void tree_sort_pairs(hipStream_t s, void* tmp, size_t tmp_bytes, const uint64_t* kin,
                     uint64_t* kout, const int* vin, int* vout, int n, int end_bit);
// dst[seg.z + k] = src[seg.x + k] for k < seg.y, per segment
void launch_gather_segments(hipStream_t s, int nseg, const int4* seg, const int* src, int* dst);
void launch_set_int(hipStream_t s, int* p, int v);
void launch_inc_int(hipStream_t s, int* p);
// A triangle rule for point generation: k points per sub-triangle at
// barycentric (u, v) with weights w (k = 0: one centroid point per patch).
struct RuleDev {
    int k;
    double u[16], v[16], w[16];
};
// the point set of every patch from the surface, in the local frame
void launch_gen_points(hipStream_t s, int n, const double* verts, const int* tris,
                       const int* vt_ptr, const int* vt_tri, const int* vt_corner,
                       const int* ctl_idx, const double* ctl, const Patch64* patches,
                       const int* ptr, const RuleDev& rule, int per_area, Pt64* out64,
                       Pt32* out32);
// planes and radii of a point set in runs of gs; *bad counts the patches whose
// points are not (the outputs then hold nothing usable); xyzw may be null
void launch_point_planes(hipStream_t s, int n, const int* ptr, const Pt64* pts, int gs, double4* plane,
                         float* radius, float4* xyzw, int* bad);
// raw CSR points k0 .. k0+n-1 (7 doubles each) -> local-frame records
void launch_to_local(hipStream_t s, int n, int k0, const double* raw, const int* ptr, int N,
                     const Patch64* patches, Pt64* out64, Pt32* out32);
void launch_mfma_selftest(hipStream_t s, const double* a, const double* b, int fp32, double* out);
// y[k] = rsqrt_nr(x[k]) (which 0) or exp_neg64(x[k]) (1)
void launch_math_selftest(hipStream_t s, int which, int n, const double* x, double* y);
void launch_scale_copy(hipStream_t s, int n, const double* x, const double* scale_ptr,
                       double scale, double* y);

}  // namespace beepdev
