// Device task layouts and kernel launchers (implemented in kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace tns {

constexpr int DEV_MAXR = 8;

// One strided block copy: dst[i] = (neg ? -1 : 1) * src[i] over a rank-r box,
// i enumerated row-major over dims (destination order).  mul / sh: the
// round-up division magic of each dimension (perm_magic), so that the kernel
// decodes a flat index with multiply-shifts instead of integer divisions.
struct PermDev {
    const void* src;
    void* dst;
    int64_t n;
    int32_t rank, neg;
    int32_t dims[DEV_MAXR];
    int32_t ss[DEV_MAXR];
    int32_t ds[DEV_MAXR];
    uint32_t mul[DEV_MAXR];
    int32_t sh[DEV_MAXR];
};

// Granlund-Montgomery round-up magic for 31-bit dividends: with
// l = ceil(log2 d), mul = floor(2^(31+l) / d) + 1 (< 2^32 for every d >= 1)
// and sh = 31 + l, floor(x / d) = (x * mul) >> sh for all 0 <= x < 2^31.
inline void perm_magic(uint32_t d, uint32_t* mul, int32_t* sh) {
    const int l = d > 1 ? 32 - __builtin_clz(d - 1) : 0;
    *mul = uint32_t((uint64_t(1) << (31 + l)) / d + 1);
    *sh = 31 + l;
}

struct GemmDev {
    const void* a;
    const void* b;
    void* c;
    int32_t m, n, k, lda, ldb, ldc, ta, tb;
    double alpha;
    const int32_t* skip;  // non-null: nothing to do where *skip is set
};

struct TileDev {
    int32_t task, tm, tn, pad;
};

struct FillDev {
    void* p;
    int64_t n;
};

struct QrDev {
    const void* in;
    void* f1;
    void* f2;
    double* work;  // global scratch (mx*nx + k doubles) when not LDS-resident
    int32_t m, n, lq, pad;
};

struct SvdDev {
    const void* in;
    void* u;
    double* s;  // singular values are always stored in double
    void* v;
    double* work;  // global scratch (mx*kx + kx*kx + kx doubles) when not LDS-resident
    int32_t m, n;
    int32_t max_sweeps;  // Jacobi sweep limit; a sector not converged by then gets NaN singular values
    int32_t pad1;
    const int32_t* done;  // non-null: nothing to do where *done is set (the eigenvector path took the sector)
};
// default Jacobi sweep limit (the host can lower it to force the
// non-convergence path in tests)
constexpr int SVD_MAX_SWEEPS = 60;

// dtype: 0 = float64, 1 = float32
// A record of a permute or fill launch: `step` counts chunks of a task (one
// workgroup each, first in the list) or units of FLAT_UNIT elements (one wave).
// A task is cut into chunks; a rest of at most FLAT_UNIT elements is a unit, a
// longer one a shorter chunk.
struct FlatUnit {
    int32_t task;
    int32_t step;
};
constexpr int FLAT_LANE = 8;  // elements per lane
constexpr int FLAT_UNIT = 64 * FLAT_LANE, FLAT_CHUNK = 4 * FLAT_UNIT;
inline int64_t flat_chunks(int64_t n) { return (n + FLAT_CHUNK - FLAT_UNIT - 1) / FLAT_CHUNK; }
inline int64_t flat_units(int64_t n) { return n > flat_chunks(n) * FLAT_CHUNK; }
void launch_permute(const PermDev* tasks, const FlatUnit* units, int64_t num_chunks, int64_t num_units, int dtype,
                    hipStream_t stream);
// same copy with a float64 source (singular values into S)
void launch_permute_from_f64(const PermDev* tasks, const FlatUnit* units, int64_t num_chunks, int64_t num_units,
                             int dtype, hipStream_t stream);
void launch_fill(const FillDev* tasks, const FlatUnit* units, int64_t num_chunks, int64_t num_units, int dtype,
                 hipStream_t stream);
void launch_permute_to_f64(const PermDev* tasks, const FlatUnit* units, int64_t num_chunks, int64_t num_units,
                           hipStream_t stream);
// dtype: 0 float64, 1 float32, 2 float32 operands as split-bf16 x3 (hi*hi +
// hi*lo + lo*hi), 3 split-bf16 x6 (three-term split, all products of order
// <= 2); float32 accumulation for 1..3
// variant: tile 0 = 32x32, 1 = 64x64, 2 = 16x16 (split-bf16: 32x32 only)
void launch_gemm(const GemmDev* tasks, const TileDev* tiles, int64_t num_tiles, int dtype, int variant,
                 hipStream_t stream);
constexpr int GEMM_VARIANTS = 3;
constexpr int GEMM_TILE_OF[GEMM_VARIANTS] = {32, 64, 16};
// QR / SVD: one workgroup per block.  lds_bytes > 0 selects the LDS-resident
// kernel with that much dynamic LDS (every task of the launch must fit);
// 0 selects the kernel working in each task's global scratch.
constexpr int QR_WG = 512;
constexpr int SVD_WG = 256;
// largest LDS working set per workgroup (gfx950: 160 KiB per CU)
// LDS size classes: a launch reserves the largest working set among its
// tasks, so tasks are grouped by class (3, 2 or 1 workgroups per CU)
constexpr int64_t LDS_CLASS[3] = {48 * 1024, 76 * 1024, 152 * 1024};
constexpr int64_t QR_LDS_MAX = LDS_CLASS[2];
constexpr int64_t SVD_LDS_MAX = LDS_CLASS[2];
// scratch of a QR / LQ task beyond LDS: the block and its taus
inline int64_t qr_doubles(int64_t m, int64_t n) { return m * n + (m < n ? m : n); }
// Sectors that go through the eigenvectors of their Gram matrix first
// (svd_eig.hip).  Whole SVD passes with the Jacobi kernels alone and with this
// path: 64 tensors with sectors up to about 200 x 190 (some beyond the register
// kernel's 192 rows) 99.2 -> 4.4 ms; 4 tensors with sectors up to about
// 310 x 260 199 -> 5.2 ms; one stage of 128 8x8 D=8 configurations (register
// 24 / 16 and LDS kernels, one after the other) 11.1 -> 4.9 ms.  The lower line:
// tensors of one sector, whole passes with the LDS Jacobi kernel against this
// path, 1, 16 and 200 tensors a call: 31 x 30 599 / 1146 / 3118 against 415 /
// 1005 / 3152 us, 140 x 28 567 / 1140 / 3193 against 433 / 1045 / 3047, 24 x 24
// 483 / 1015 / 3029 against 360 / 996 / 3253, 30 x 20 433 / 909 / 2792 against 360 /
// 1002 / 3205, 200 x 16 390 / 889 / 2894 against 347 / 965 / 3149, 16 x 16 369 / 908 /
// 2864 against 369 / 939 / 3111 (host planning is most of a pass of many tensors,
// runs of one side differ by up to 20% there).  Where sectors of 16 to 31 columns
// are the largest of many tensors with smaller ones too, the LDS kernel runs
// anyway and the path adds 0.13 to 0.2 ms (21 tensors 1.52 -> 1.65 ms, 59 tensors
// 1.78 -> 1.97); beside larger sectors it adds next to nothing, and a launch of the
// LDS kernel for those of 16 to 23 columns would cost 10 to 20% of a pass of 1 to
// 2 ms.  The sector's size alone decides, so that its factors do not depend on
// what shares its launch.  A sector the path has to leave to the Jacobi kernels pays for
// both: 150 columns with singular values over 5 decades 7.8 -> 8.8 ms, over 12
// 12.5 -> 13.6, 32 columns 0.81 -> 1.03 and 0.95 -> 1.18, 210 columns 200 -> 206.
// Above 640 columns the eigenvector strips no longer fit the registers of one
// wave.
constexpr int SVD_EIG_MIN_COLS = 16, SVD_EIG_MAX_COLS = 640;
inline bool svd_eig_fits(int64_t m, int64_t n) {
    const int64_t mx = m > n ? m : n, kx = m < n ? m : n;
    return kx >= SVD_EIG_MIN_COLS && kx <= SVD_EIG_MAX_COLS && mx * kx <= (int64_t(1) << 28);
}
// blocks of 16 reflectors of that path
inline int64_t svd_eig_blocks(int64_t kx) { return (kx + 15) / 16; }
// scratch of an SVD task: the Jacobi kernels' columns, V and singular values;
// the eigenvector path's two column sets, four kx x kx matrices, the
// tridiagonal form, the block reflectors' factors, the order and the flags
inline int64_t svd_doubles(int64_t m, int64_t n) {
    const int64_t mx = m > n ? m : n, kx = m < n ? m : n;
    if (svd_eig_fits(m, n)) return 2 * mx * kx + 4 * kx * kx + 256 * svd_eig_blocks(kx) + 5 * kx + (kx + 1) / 2 + 2;
    return mx * kx + kx * kx + kx;
}
// the Jacobi kernels' LDS working set
inline int64_t svd_lds_doubles(int64_t m, int64_t n) {
    const int64_t mx = m > n ? m : n, kx = m < n ? m : n;
    return mx * kx + kx * kx + kx;
}
// variant 1: blocked Householder with the panel in LDS (global scratch
// blocks with at most QB_MAX_ROWS rows); otherwise LDS (lds_bytes > 0) or
// unblocked global scratch
void launch_qr(const QrDev* tasks, int64_t num, int64_t lds_bytes, int variant, int dtype, hipStream_t stream);
constexpr int64_t QB_LDS = 156 * 1024;
// rows for which the blocked kernel's panel keeps at least 4 columns
constexpr int64_t QB_MAX_ROWS = (QB_LDS - 8 * (16 * 16 * 2 + 16 * 128 + 16)) / (8 * 4);
// rpt > 0: register-resident kernel for blocks with at most 8 * rpt rows
// (rpt in {8, 16, 24}), V recovered from U; otherwise LDS (lds_bytes > 0)
// or global scratch.
void launch_svd(const SvdDev* tasks, int64_t num, int64_t lds_bytes, int rpt, int dtype, hipStream_t stream);

// A sector on the eigenvector path.  Rows are contiguous: row c of xt is
// column c of X.
struct SvdEigDev {
    SvdDev t;
    double *xt, *xt2;         // kx x mx
    double *b, *z, *s, *vt;   // kx x kx
    double *tb;               // 16 x 16 per block of reflectors
    double *de, *e, *tau;     // 2 kx (diagonal, squared off-diagonal), kx, kx
    double *sig;              // kx: reciprocal column norms in rank order
    int32_t *order, *flags;   // kx; done, not for this path, scale exponent, first form of the step
    int32_t mx, kx;
};
enum SvdEigStage {
    SVD_EIG_LOAD,     // per task
    SVD_EIG_TRIDIAG,  // per task; variant 0..4: at most 64 / 128 / 192 / 320 / 640 columns
    SVD_EIG_TFACTOR,  // per task and 16 columns (units)
    SVD_EIG_VECTORS,  // per task and 64 columns (units)
    SVD_EIG_BACK,     // per task and 64 columns (units); variant: 64 / 128 / 192 / 320 / 640 columns
    SVD_EIG_POLISH,   // per task
    SVD_EIG_REFINE,   // per task
    SVD_EIG_SECOND,   // per task
    SVD_EIG_VERIFY,   // per task
    SVD_EIG_ORDER,    // per task
    SVD_EIG_WRITE     // per task and 32 columns (units)
};
void launch_svd_eig(int stage, int variant, const SvdEigDev* tasks, const TileDev* units, int64_t num, int dtype,
                    hipStream_t stream);

// Copy n_i doubles from src_i to dst + off_i for every task, one workgroup
// per task: gathers the singular values of a batch of decompositions into
// one (host-mapped) buffer with a single launch.
struct GatherDev {
    const double* src;
    int64_t n;
    int64_t off;
};
void launch_gather_f64(const GatherDev* tasks, int64_t num, double* dst, hipStream_t stream);
constexpr int SVD_REG_MAX_ROWS = 192;

}  // namespace tns
