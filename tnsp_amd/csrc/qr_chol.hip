// QR (and LQ, through the transpose) of tall sector blocks by Cholesky
// factors, twice, with the signs of the Householder factorisation.
//
// X holds the nx = min(m, n) columns of the block (M or M^T) scaled by a power
// of two:
//   X^T X = R1^T R1,  Q1 = X R1^-1,  Q1^T Q1 = R2^T R2,  Q = Q1 R2^-1,
//   R = R2 R1.
// The second pass brings Q to orthogonality at rounding as long as the first
// left ||Q1^T Q1 - 1|| well below one, which is measured (QC_DEFECT); pivots
// that lose more than QC_PIVOT of their column (condition numbers beyond a few
// 10^5), entries that are not finite and columns that Householder would leave
// alone (zero below the diagonal: its sign rule differs there) leave the block
// to the Householder kernels, which run afterwards and skip what is done.
// Signs: the Householder R has the sign opposite to the pivot of each column;
// an elimination of the top block of Q without pivoting, with that sign taken
// from each pivot, meets the same numbers.
//
// Householder panels keep one workgroup per block busy with a serial chain of
// 2 nx columns; here the block's work is seven products spread over many
// workgroups and three nx-step eliminations in registers.
#include "device.hpp"
#include "kernels.hpp"

#include <stdexcept>
#include <string>

namespace tns {

namespace {

constexpr double QC_PIVOT = 1e-11, QC_DEFECT = 0.1;

inline void check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// The power of two that brings the block's largest entry into [1, 2), so that
// squares neither overflow nor vanish, and the flags
template<typename T>
__global__ __launch_bounds__(1024) void qc_range_kernel(const QrCholDev* __restrict__ tasks) {
    __shared__ double wmax[16];
    const QrCholDev& tk = tasks[blockIdx.x];
    const gptr<const T> in = to_global(static_cast<const T*>(tk.t.in));
    const int tid = threadIdx.x, total = tk.mx * tk.nx;
    double amax = 0.0;
    bool fine = true;
#pragma unroll 8
    for (int e = tid; e < total; e += 1024) {
        const double x = fabs(double(in[e]));
        fine = fine && x <= 1.79e308;
        amax = fmax(amax, x);
    }
    amax = wave_max(amax);
    if (tid % WAVE == 0) wmax[tid / WAVE] = amax;
    fine = __syncthreads_and(fine);
    if (tid != 0) return;
    for (int w = 0; w < 16; w++) amax = fmax(amax, wmax[w]);
    tk.flags[0] = 0;
    tk.flags[1] = (fine && amax > 0.0) ? 0 : 1;
    tk.flags[2] = jacobi_scale_exponent(amax);
}

// X (nx rows of mx, its columns one after the other) from the block, scaled, 32
// columns per workgroup, through LDS tiles where the block is stored the other
// way round
template<typename T>
__global__ __launch_bounds__(256) void qc_load_kernel(const QrCholDev* __restrict__ tasks,
                                                     const TileDev* __restrict__ units) {
    __shared__ double tile[32][33];
    const QrCholDev& tk = tasks[units[blockIdx.x].task];
    const int n = tk.nx, mx = tk.mx, c0 = 32 * units[blockIdx.x].tm, tx = threadIdx.x % 32, ty = threadIdx.x / 32;
    const gptr<const T> in = to_global(static_cast<const T*>(tk.t.in));
    const gptr<double> xt = to_global(tk.xt);
    const double scl = ldexp(1.0, -tk.flags[2]);
    if (tk.t.lq) {
        for (int q = ty; q < 32 && c0 + q < n; q += 8)
            for (int i = tx; i < mx; i += 32) xt[int64_t(c0 + q) * mx + i] = scl * double(in[int64_t(c0 + q) * mx + i]);
        return;
    }
    for (int i0 = 0; i0 < mx; i0 += 32) {
        for (int q = ty; q < 32; q += 8)
            if (i0 + q < mx && c0 + tx < n) tile[q][tx] = scl * double(in[int64_t(i0 + q) * n + c0 + tx]);
        __syncthreads();
        for (int q = ty; q < 32; q += 8)
            if (c0 + q < n && i0 + tx < mx) xt[int64_t(c0 + q) * mx + i0 + tx] = tile[tx][q];
        __syncthreads();
    }
}

// Cholesky factor R (upper, b = R^T R) and R^-T (lower) of a symmetric matrix
// in one elimination: thread (ti, tj) of TI x 16 holds rows ti + TI a and
// columns tj + 16 b.  Step j subtracts multiples of row j from the rows below,
// over all columns: right of j that is the Schur complement, left of j, where
// the eliminated columns have no further use, it builds the inverse of the
// unit lower factor in place.  The multipliers are row j itself (the complement
// is symmetric), so a step has one barrier; rows already done are skipped.
// Bound by the LDS reads of row j and the barrier per step; up to 224 columns
// 376 us, up to 192 267 us, up to 128 123 us.
template<int TI, int A, int BC>
__global__ __launch_bounds__(TI * 16) void qc_chol_kernel(const QrCholDev* __restrict__ tasks, int second) {
    constexpr int N = TI * A > 16 * BC ? TI * A : 16 * BC;
    __shared__ double xs[2][N], first[N], rs[N];
    const QrCholDev tk = tasks[blockIdx.x];
    const int n = tk.nx, tid = threadIdx.x, ti = tid / 16, tj = tid % 16;
    if (n > TI * A || n > 16 * BC || tk.flags[1]) return;
    const gptr<double> B = to_global(tk.b), G = to_global(tk.g), R = to_global(second ? tk.r2 : tk.r1);
    double w[A][BC];
    bool fine = true;
#pragma unroll
    for (int a = 0; a < A; a++) {
        const int r = ti + TI * a;
        double sum = 0.0;
#pragma unroll
        for (int b = 0; b < BC; b++) {
            const int c = tj + 16 * b;
            // the products below the diagonal are not formed
            w[a][b] = (r < n && c < n) ? (c >= r ? B[r * n + c] : B[c * n + r]) : 0.0;
            if (r < n && r == c) first[r] = w[a][b];
            sum += fabs(w[a][b] - (r < n && r == c ? 1.0 : 0.0));
        }
        if (second) fine = fine && row_sum16(sum) <= QC_DEFECT;
    }
    if (!__syncthreads_and(fine)) {
        if (tid == 0) tk.flags[1] = 1;
        return;
    }
    for (int j = 0; j < n; j++) {
        double* x = xs[j & 1];
#pragma unroll
        for (int a = 0; a < A; a++)
            if (j / TI == a && ti == j % TI) {
#pragma unroll
                for (int b = 0; b < BC; b++) x[tj + 16 * b] = w[a][b];
            }
        __syncthreads();
        const double d = x[j];
        if (!(d > QC_PIVOT * first[j])) {  // uniform: every thread reads the same pivot
            if (tid == 0) tk.flags[1] = 1;
            return;
        }
        const double rd = refined_rsqrt(d), inv = rd * rd;
        if (tid < n) R[j * n + tid] = tid < j ? 0.0 : x[tid] * rd;
        if (tid == 0) rs[j] = rd;
        double xv[BC];
#pragma unroll
        for (int b = 0; b < BC; b++) xv[b] = x[tj + 16 * b];
#pragma unroll
        for (int a = 0; a < A; a++) {
            if (TI * a + TI - 1 <= j) continue;
            const int r = ti + TI * a;
            const double f = r > j ? x[r] * inv : 0.0;
#pragma unroll
            for (int b = 0; b < BC; b++) w[a][b] -= f * xv[b];
            // column j starts the inverse
#pragma unroll
            for (int b = 0; b < BC; b++)
                if (j / 16 == b && tj == j % 16 && r > j) w[a][b] = -f;
        }
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < A; a++)
#pragma unroll
        for (int b = 0; b < BC; b++) {
            const int r = ti + TI * a, c = tj + 16 * b;
            if (r < n && c < n) G[r * n + c] = c > r ? 0.0 : rs[r] * (c == r ? 1.0 : w[a][b]);
        }
}

// The signs of the Householder R: elimination of the top nx x nx block of Q
// (xt: column c of Q is row c) without pivoting, each pivot moved away from
// zero by one.  A last column of a square block has nothing below its
// diagonal: Householder keeps its sign.
template<int TI, int A, int BC>
__global__ __launch_bounds__(TI * 16) void qc_sign_kernel(const QrCholDev* __restrict__ tasks) {
    constexpr int N = TI * A > 16 * BC ? TI * A : 16 * BC;
    __shared__ double row[2][N], col[2][N];
    const QrCholDev tk = tasks[blockIdx.x];
    const int n = tk.nx, mx = tk.mx, tid = threadIdx.x, ti = tid / 16, tj = tid % 16;
    if (n > TI * A || n > 16 * BC || tk.flags[1]) return;
    const gptr<const double> Q = to_global(tk.xt);
    double w[A][BC];
#pragma unroll
    for (int a = 0; a < A; a++)
#pragma unroll
        for (int b = 0; b < BC; b++) {
            const int r = ti + TI * a, c = tj + 16 * b;
            w[a][b] = (r < n && c < n) ? Q[int64_t(c) * mx + r] : 0.0;
        }
    for (int j = 0; j < n; j++) {
        double *x = row[j & 1], *y = col[j & 1];
#pragma unroll
        for (int a = 0; a < A; a++)
            if (j / TI == a && ti == j % TI) {
#pragma unroll
                for (int b = 0; b < BC; b++) x[tj + 16 * b] = w[a][b];
            }
#pragma unroll
        for (int b = 0; b < BC; b++)
            if (j / 16 == b && tj == j % 16) {
#pragma unroll
                for (int a = 0; a < A; a++) y[ti + TI * a] = w[a][b];
            }
        __syncthreads();
        const double t = x[j];
        const bool last = j + 1 == mx;
        if (!last && !(fabs(t) < 1.0 - 1e-12)) {  // nothing below the diagonal, or not finite
            if (tid == 0) tk.flags[1] = 1;
            return;
        }
        const double s = ((t >= 0.0) == last) ? 1.0 : -1.0;
        if (tid == 0) tk.sign[j] = s;
        if (last) break;
        const double inv = refined_rcp(t - s);
        double xv[BC];
#pragma unroll
        for (int b = 0; b < BC; b++) xv[b] = x[tj + 16 * b];
#pragma unroll
        for (int a = 0; a < A; a++) {
            if (TI * a + TI - 1 <= j) continue;
            const int r = ti + TI * a;
            const double f = r > j ? y[r] * inv : 0.0;
#pragma unroll
            for (int b = 0; b < BC; b++) w[a][b] -= f * xv[b];
        }
    }
}

// Q and R of the block with their signs, 32 columns of Q per workgroup; the
// first workgroup of a task marks it done.  The factor stored column by column
// goes through LDS tiles.
template<typename T>
__global__ __launch_bounds__(256) void qc_write_kernel(const QrCholDev* __restrict__ tasks,
                                                      const TileDev* __restrict__ units) {
    __shared__ double tile[32][33];
    const QrCholDev tk = tasks[units[blockIdx.x].task];
    if (tk.flags[1]) return;
    const int n = tk.nx, mx = tk.mx, c0 = 32 * units[blockIdx.x].tm, tx = threadIdx.x % 32, ty = threadIdx.x / 32;
    const bool lq = tk.t.lq != 0;
    const gptr<const double> Q = to_global(tk.xt), R = to_global(tk.b), sign = to_global(tk.sign);
    // lq: f1 = L (nx x nx), f2 = Q^T rows; otherwise f1 = Q, f2 = R
    const gptr<T> rout = to_global(static_cast<T*>(lq ? tk.t.f1 : tk.t.f2));
    const gptr<T> qout = to_global(static_cast<T*>(lq ? tk.t.f2 : tk.t.f1));
    const double scl = ldexp(1.0, tk.flags[2]);
    for (int q = ty; q < 32; q += 8) {
        const int j = c0 + q;
        if (j >= n) break;
        const double s = sign[j];
        for (int c = tx; c < n; c += 32) {
            const double v = c < j ? 0.0 : R[j * n + c] * (s * scl);
            rout[lq ? c * n + j : j * n + c] = T(v);
        }
        if (lq)
            for (int i = tx; i < mx; i += 32) qout[int64_t(j) * mx + i] = T(Q[int64_t(j) * mx + i] * s);
    }
    if (!lq)
        for (int i0 = 0; i0 < mx; i0 += 32) {
            for (int q = ty; q < 32; q += 8)
                if (c0 + q < n && i0 + tx < mx) tile[q][tx] = Q[int64_t(c0 + q) * mx + i0 + tx] * sign[c0 + q];
            __syncthreads();
            for (int q = ty; q < 32; q += 8)
                if (i0 + q < mx && c0 + tx < n) qout[int64_t(i0 + q) * n + c0 + tx] = T(tile[tx][q]);
            __syncthreads();
        }
    if (c0 == 0 && threadIdx.x == 0) tk.flags[0] = 1;
}

}  // namespace

void launch_qr_chol(int stage, int variant, const QrCholDev* tasks, const TileDev* units, int64_t num, int dtype,
                    hipStream_t st) {
    if (num <= 0) return;
    const dim3 grid(static_cast<unsigned>(num));
    auto chol = [&](int second) {
        if (variant == 0)
            hipLaunchKernelGGL((qc_chol_kernel<16, 4, 4>), grid, dim3(256), 0, st, tasks, second);
        else if (variant == 1)
            hipLaunchKernelGGL((qc_chol_kernel<32, 4, 8>), grid, dim3(512), 0, st, tasks, second);
        else if (variant == 2)
            hipLaunchKernelGGL((qc_chol_kernel<48, 4, 12>), grid, dim3(768), 0, st, tasks, second);
        else
            hipLaunchKernelGGL((qc_chol_kernel<32, 7, 14>), grid, dim3(512), 0, st, tasks, second);
    };
    switch (stage) {
        case QR_CHOL_RANGE:
            if (dtype == 0)
                hipLaunchKernelGGL(qc_range_kernel<double>, grid, dim3(1024), 0, st, tasks);
            else
                hipLaunchKernelGGL(qc_range_kernel<float>, grid, dim3(1024), 0, st, tasks);
            break;
        case QR_CHOL_LOAD:
            if (dtype == 0)
                hipLaunchKernelGGL(qc_load_kernel<double>, grid, dim3(256), 0, st, tasks, units);
            else
                hipLaunchKernelGGL(qc_load_kernel<float>, grid, dim3(256), 0, st, tasks, units);
            break;
        case QR_CHOL_FIRST:
            chol(0);
            break;
        case QR_CHOL_SECOND:
            chol(1);
            break;
        case QR_CHOL_SIGN:
            if (variant == 0)
                hipLaunchKernelGGL((qc_sign_kernel<16, 4, 4>), grid, dim3(256), 0, st, tasks);
            else if (variant == 1)
                hipLaunchKernelGGL((qc_sign_kernel<32, 4, 8>), grid, dim3(512), 0, st, tasks);
            else if (variant == 2)
                hipLaunchKernelGGL((qc_sign_kernel<48, 4, 12>), grid, dim3(768), 0, st, tasks);
            else
                hipLaunchKernelGGL((qc_sign_kernel<32, 7, 14>), grid, dim3(512), 0, st, tasks);
            break;
        case QR_CHOL_WRITE:
            if (dtype == 0)
                hipLaunchKernelGGL(qc_write_kernel<double>, grid, dim3(256), 0, st, tasks, units);
            else
                hipLaunchKernelGGL(qc_write_kernel<float>, grid, dim3(256), 0, st, tasks, units);
            break;
        default:
            throw std::runtime_error("qr: unknown stage");
    }
    check(hipGetLastError(), "qr cholesky stage launch");
}

}  // namespace tns
