// Singular value decomposition of sector blocks through the eigenvectors of
// their Gram matrix, with one exact refinement.
//
// X holds the kx = min(m, n) columns of the block (M or M^T) scaled by a power
// of two, as in the Jacobi kernels.  The path
//   B = X^T X                      (grouped GEMM)
//   B = Q T Q^T                    (Householder tridiagonalisation)
//   T Z = Z diag(lambda)           (bisection, twisted factorisations)
//   V = Q Z, V <- V (3 - V^T V)/2  (block reflectors, one Newton-Schulz step)
//   X' = X V, G = X'^T X'          (grouped GEMMs)
//   X'' = X' (I + E), V'' = V (I + E),  E_ij = G_ij / (G_jj - G_ii)
// leaves columns that are orthogonal to the tolerance of the Jacobi sweeps:
// squaring costs X' some of its orthogonality (cosines up to eps s1^2 /
// (si sj)), and I + E removes these cosines to first order, all pairs at once.
// For cosines up to c and row sums of |E| up to e, I + E is orthogonal up to
// e^2 and leaves cosines below kx c^2 + e c + e^2: with both at most EIG_SMALL
// these are rounding and less than half the sweeps' tolerance.  Above it the
// step is I + E + E^2 / 2 (orthogonal up to e^4 / 4, e at most EIG_TURN) and the
// cosines of X'' are measured.  Null columns (the Jacobi kernels' dead ones, up
// to EIG_DEAD of them) take part in none of this; their directions in U are
// completed to an orthonormal set at the end.  Any block that fails (close
// singular values, a larger null space, entries that are not finite) is left to
// the Jacobi kernels, which run after this path and skip the blocks marked
// done.  Of 1065 blocks of 32 to 190 columns of the 8x8 D=8 PEPS 0.4% and of 240
// of the 8x8 Z2 D=6 one 10% take the second form, and all pass; of 5972 blocks of
// 16 and more columns two have a null column.  The cosines before the step are
// 1.4e-13 in the median and 3.4e-6 at most.  One block left to the Jacobi kernels
// costs its launch the whole 5 ms of a block there.
//
// One-sided Jacobi does 10 to 14 sweeps of kx^2 / 2 rotations of length mx;
// this path does about 14 kx^3 multiply-adds, most of them on the matrix
// cores in launches that spread a block over many workgroups.  Times of both
// stand at the routing rule (svd_eig_fits).
#include "device.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <stdexcept>
#include <string>

namespace tns {

namespace {

// data written by an earlier kernel and read at uniform addresses: scalar loads
typedef const __attribute__((address_space(4))) double* cptr;

constexpr double EIG_SMALL = 1e-8, EIG_TURN = 1e-4;
constexpr int EIG_DEAD = 8;
// row sums of |V^T V - 1| above which one Newton-Schulz step (which squares
// the defect) does not reach rounding
constexpr double EIG_DEFECT = 1e-7;

inline void check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// ------------------------------------------------------------------- load
// X (kx rows of mx, the columns of X one after the other) from the block,
// scaled so that its largest entry lies in [1, 2).  32 x 32 tiles through LDS
// where the block is stored the other way round, so that both sides coalesce.
template<typename T>
__global__ __launch_bounds__(1024) void eig_load_kernel(const SvdEigDev* __restrict__ tasks) {
    const SvdEigDev tk = tasks[blockIdx.x];
    __shared__ double wmax[16];
    __shared__ double tile[32][33];
    const gptr<const T> in = to_global(static_cast<const T*>(tk.t.in));
    const gptr<double> xt = to_global(tk.xt);
    const int tid = threadIdx.x, mx = tk.mx, kx = tk.kx;
    double amax = 0.0;
    bool fine = true;
    for (int e = tid; e < mx * kx; e += 1024) {
        const double x = fabs(double(in[e]));
        fine = fine && x <= 1.79e308;
        amax = fmax(amax, x);
    }
    amax = wave_max(amax);
    if (tid % WAVE == 0) wmax[tid / WAVE] = amax;
    fine = __syncthreads_and(fine);
    for (int w = 0; w < 16; w++) amax = fmax(amax, wmax[w]);
    const int ex = jacobi_scale_exponent(amax);
    const double scl = ldexp(1.0, -ex);
    if (tid == 0) {
        tk.flags[0] = 0;                              // done
        tk.flags[1] = (fine && amax > 0.0) ? 0 : 1;  // not for this path
        tk.flags[2] = ex;
        tk.flags[3] = 1;  // the step's first form, no measurement
    }
    if (tk.t.m < tk.t.n) {
        // M^T: row c of the block is column c of X
        for (int e = tid; e < mx * kx; e += 1024) xt[e] = double(in[e]) * scl;
        return;
    }
    const int ti = tid / 32, tj = tid % 32;
    for (int r0 = 0; r0 < mx; r0 += 32) {
        for (int c0 = 0; c0 < kx; c0 += 32) {
            const int r = r0 + ti, c = c0 + tj;
            if (r < mx && c < kx) tile[ti][tj] = double(in[r * kx + c]) * scl;
            __syncthreads();
            if (c0 + ti < kx && r0 + tj < mx) xt[(c0 + ti) * mx + r0 + tj] = tile[tj][ti];
            __syncthreads();
        }
    }
}

// -------------------------------------------------------- tridiagonal form
// What both versions write per step j: the diagonal, the off-diagonal entry
// below it and its square (floored, so that the Sturm recurrence never meets
// a split matrix), and the reflector v (zero up to j, one at j + 1) as row j
// of `b`.
struct TriOut {
    gptr<double> de, e, tau;
    double floor2;
    __device__ void step(int j, int n, double d, double beta, double t) const {
        de[2 * j] = d;
        if (j == 0) de[1] = 0.0;
        tau[j] = t;
        if (j + 1 < n) {
            e[j] = beta;
            de[2 * j + 3] = fmax(beta * beta, floor2);
        }
    }
};

// Reflector scalars from one refined reciprocal square root and one refined
// reciprocal (every wave computes them: the division and square root
// sequences took a third of a step): beta, tau = 1 - alpha / beta and scale =
// 1 / (alpha - beta), each within a few ulp.
__device__ inline void tri_reflector(double alpha, double sigma, double& tau, double& beta, double& scale) {
    if (sigma == 0.0) {
        tau = scale = 0.0;
        beta = alpha;
        return;
    }
    const double s = fma(alpha, alpha, sigma), r = refined_rsqrt(s), root = s * r, a = fabs(alpha);
    beta = -copysign(root, alpha);
    tau = fma(a, r, 1.0);
    scale = copysign(refined_rcp(a + root), alpha);
}

// Matrix in registers: thread (ti, tj) of TI x 16 holds rows ti + TI a and
// columns tj + 16 b, a < A, b < BC.  Per column two barriers.  The 16 lanes
// that hold row j (column j by symmetry) put it into LDS with the square sum
// below the diagonal; every wave forms the reflector from them.  Then s = B v
// by partial rows and a sum over the 16 lanes of a row group, with v^T s summed
// per wave on the way, and the rank-two update.  Bound by the LDS reads of v
// and p (3 BC + 2 A values per thread and step) and by the chain of two
// barriers and one reciprocal square root per step; a block of rows or columns
// already reduced is skipped.  190 columns, one workgroup per CU: 640 us (770
// with v and w held in registers, 36 of them spilled).
template<int TI, int A, int BC>
__global__ __launch_bounds__(TI * 16) void eig_tridiag_kernel(const SvdEigDev* __restrict__ tasks) {
    constexpr int N = TI * A > 16 * BC ? TI * A : 16 * BC, NW = TI * 16 / WAVE;
    __shared__ double xs[2][N], ps[2][N], sg[2], dots[2][NW], wtr[NW];
    const SvdEigDev tk = tasks[blockIdx.x];
    const int n = tk.kx, tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE, ti = tid / 16, tj = tid % 16;
    if (n > TI * A || n > 16 * BC || tk.flags[1]) return;  // uniform over the workgroup
    const gptr<double> B = to_global(tk.b);
    double rb[A][BC];
    double trace = 0.0;
#pragma unroll
    for (int a = 0; a < A; a++)
#pragma unroll
        for (int b = 0; b < BC; b++) {
            const int r = ti + TI * a, c = tj + 16 * b;
            rb[a][b] = (r < n && c < n) ? B[r * n + c] : 0.0;
            if (r == c) {
                trace += rb[a][b];
                xs[0][r] = rb[a][b];
            }
        }
    for (int i = tid; i < 2 * N; i += TI * 16) (&ps[0][0])[i] = 0.0;
    trace = wave_sum(trace);
    if (lane == 0) wtr[wave] = trace;
    __syncthreads();
    trace = 0.0;
    for (int w = 0; w < NW; w++) trace += wtr[w];
    // Columns that are orthogonal already, to four times the sweeps' tolerance,
    // are left to the register and LDS Jacobi kernels, which only look them over
    // (an isometry of 150 columns: 1.67 ms through the whole path and the sweep,
    // 0.84 this way, 0.63 with the sweep alone).
    if (tk.mx <= SVD_REG_MAX_ROWS) {
        const double tol = 4.0 * 2.220446049250313e-16 * tk.mx;
        bool turn = false;
#pragma unroll
        for (int a = 0; a < A; a++)
#pragma unroll
            for (int b = 0; b < BC; b++) {
                const int r = ti + TI * a, c = tj + 16 * b;
                if (r < c && c < n) turn = turn || rb[a][b] * rb[a][b] > tol * xs[0][r] * (tol * xs[0][c]);
            }
        if (!__syncthreads_or(turn)) {
            if (tid == 0) tk.flags[1] = 1;
            return;
        }
    }
    const TriOut out{to_global(tk.de), to_global(tk.e), to_global(tk.tau), 1e-40 * trace * trace};
    for (int j = 0; j < n; j++) {
        double* x = xs[j & 1];
        double* p = ps[j & 1];
#pragma unroll
        for (int a = 0; a < A; a++)
            if (j / TI == a && ti == j % TI) {
                double s = 0.0;
#pragma unroll
                for (int b = 0; b < BC; b++) {
                    x[tj + 16 * b] = rb[a][b];
                    if (tj + 16 * b > j + 1) s += rb[a][b] * rb[a][b];
                }
                s = row_sum16(s);
                if (tj == 0) sg[j & 1] = s;
            }
        __syncthreads();
        double tau, beta, scale;
        tri_reflector(j + 1 < n ? x[j + 1] : 0.0, sg[j & 1], tau, beta, scale);
        if (tid == 0) out.step(j, n, x[j], beta, tau);
        if (tid < n) B[j * n + tid] = tid <= j ? 0.0 : (tid == j + 1 ? 1.0 : x[tid] * scale);
        // the next step writes the other buffers, and the one after it waits
        // for every wave to have left this step
        if (tau == 0.0) continue;
        // v is read again for the update: held, it would spill at A BC = 48
        double vr[A], sum[A], dot = 0.0;
#pragma unroll
        for (int a = 0; a < A; a++) {
            const int r = ti + TI * a;
            vr[a] = r <= j ? 0.0 : (r == j + 1 ? 1.0 : x[r] * scale);
            sum[a] = 0.0;
        }
#pragma unroll
        for (int b = 0; b < BC; b++) {
            if (16 * b + 15 <= j) continue;
            const int c = tj + 16 * b;
            const double v = c <= j ? 0.0 : (c == j + 1 ? 1.0 : x[c] * scale);
#pragma unroll
            for (int a = 0; a < A; a++) sum[a] += rb[a][b] * v;
        }
#pragma unroll
        for (int a = 0; a < A; a++) {
            if (TI * a + TI - 1 <= j) continue;
            const double s = row_sum16(sum[a]);
            dot += s * vr[a];
            if (tj == 0) p[ti + TI * a] = tau * s;
        }
        // the 16 lanes of a row group hold the same sums: four groups per wave
        dot = swap_sum<32>(swap_sum<16>(dot));
        if (lane == 0) dots[j & 1][wave] = dot;
        __syncthreads();
        double K = 0.0;
#pragma unroll
        for (int w = 0; w < NW; w++) K += dots[j & 1][w];
        K *= 0.5 * tau * tau;
        double wr[A];
#pragma unroll
        for (int a = 0; a < A; a++) wr[a] = ti + TI * a <= j ? 0.0 : p[ti + TI * a] - K * vr[a];
#pragma unroll
        for (int b = 0; b < BC; b++) {
            if (16 * b + 15 <= j) continue;
            const int c = tj + 16 * b;
            const double v = c <= j ? 0.0 : (c == j + 1 ? 1.0 : x[c] * scale);
            const double w = c <= j ? 0.0 : p[c] - K * v;
#pragma unroll
            for (int a = 0; a < A; a++) rb[a][b] -= vr[a] * w + wr[a] * v;
        }
    }
}

// Matrix in global memory (more columns than the registers hold): one pass
// over the trailing matrix per step, which applies the previous step's
// rank-two update, stores the result and multiplies it by the new reflector.
// One wave per TRI_GLB_R rows, lane l holds columns l + 64 t, t < TRI_GLB_T.
// Bound by those passes (kx^3 16 / 3 bytes through the XCD's L2 by one
// workgroup) and their latency.
template<int TRI_GLB_T, int TRI_GLB_R>
__global__ __launch_bounds__(1024) void eig_tridiag_glb_kernel(const SvdEigDev* __restrict__ tasks) {
    __shared__ double xs[SVD_EIG_MAX_COLS], vs[SVD_EIG_MAX_COLS], ws[SVD_EIG_MAX_COLS], ps[SVD_EIG_MAX_COLS], red[16];
    const SvdEigDev tk = tasks[blockIdx.x];
    const int n = tk.kx, tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    if (n > WAVE * TRI_GLB_T || tk.flags[1]) return;
    // the trailing matrix is updated in place in `s`, the reflectors go to `b`
    const gptr<double> B = to_global(tk.s), R = to_global(tk.b);
    double trace = 0.0;
    for (int r = wave; r < n; r += 16)
        for (int c = lane; c < n; c += WAVE) {
            const double v = R[r * n + c];
            B[r * n + c] = v;
            if (r == c) trace += v;
        }
    for (int i = tid; i < n; i += 1024) vs[i] = ws[i] = 0.0;
    trace = wave_sum(trace);
    if (lane == 0) red[wave] = trace;
    __syncthreads();
    trace = 0.0;
    for (int w = 0; w < 16; w++) trace += red[w];
    const TriOut out{to_global(tk.de), to_global(tk.e), to_global(tk.tau), 1e-40 * trace * trace};
    for (int j = 0; j < n; j++) {
        if (tid >= j && tid < n) xs[tid] = B[j * n + tid] - vs[j] * ws[tid] - ws[j] * vs[tid];
        __syncthreads();
        double alpha = 0.0, sigma = 0.0;
        if (j + 1 < n) {
            alpha = xs[j + 1];
            double s = 0.0;
            for (int i = j + 2 + lane; i < n; i += WAVE) s += xs[i] * xs[i];
            sigma = wave_sum(s);
        }
        double tau, beta, scale;
        tri_reflector(alpha, sigma, tau, beta, scale);
        if (tid == 0) out.step(j, n, xs[j], beta, tau);
        if (tid < n) R[j * n + tid] = tid <= j ? 0.0 : (tid == j + 1 ? 1.0 : xs[tid] * scale);
        // v, w of the previous step and the new v at this lane's columns
        double ov[TRI_GLB_T], ow[TRI_GLB_T], nv[TRI_GLB_T];
#pragma unroll
        for (int t = 0; t < TRI_GLB_T; t++) {
            const int c = lane + WAVE * t;
            const bool in = c < n && c > j;
            ov[t] = in ? vs[c] : 0.0;
            ow[t] = in ? ws[c] : 0.0;
            nv[t] = in ? (c == j + 1 ? 1.0 : xs[c] * scale) : 0.0;
        }
        // TRI_GLB_R rows at a time keep their loads in flight together
        for (int r0 = j + 1 + wave; r0 < n; r0 += 16 * TRI_GLB_R) {
            double vr[TRI_GLB_R], wr[TRI_GLB_R], s[TRI_GLB_R];
#pragma unroll
            for (int q = 0; q < TRI_GLB_R; q++) {
                const int r = min(r0 + 16 * q, n - 1);
                vr[q] = vs[r];
                wr[q] = ws[r];
                s[q] = 0.0;
            }
#pragma unroll
            for (int t = 0; t < TRI_GLB_T; t++) {
                if (WAVE * t >= n || WAVE * t + WAVE - 1 <= j) continue;
                const int c = lane + WAVE * t;
                if (c < n && c > j) {
                    double v[TRI_GLB_R];
#pragma unroll
                    for (int q = 0; q < TRI_GLB_R; q++) v[q] = B[min(r0 + 16 * q, n - 1) * n + c];
#pragma unroll
                    for (int q = 0; q < TRI_GLB_R; q++) {
                        v[q] -= vr[q] * ow[t] + wr[q] * ov[t];
                        if (r0 + 16 * q < n) B[(r0 + 16 * q) * n + c] = v[q];
                        s[q] += v[q] * nv[t];
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < TRI_GLB_R; q++) {
                const double sum = wave_sum(s[q]);
                if (lane == 0 && r0 + 16 * q < n) ps[r0 + 16 * q] = tau * sum;
            }
        }
        __syncthreads();
        double s = 0.0;
        for (int i = j + 1 + lane; i < n; i += WAVE) s += ps[i] * (i == j + 1 ? 1.0 : xs[i] * scale);
        const double K = 0.5 * tau * wave_sum(s);
        // every wave has read the old v, w (before the barrier above) and the
        // sums above read ps and xs only
        for (int i = tid; i < n; i += 1024) {
            const double v = i <= j ? 0.0 : (i == j + 1 ? 1.0 : xs[i] * scale);
            vs[i] = v;
            ws[i] = i <= j ? 0.0 : ps[i] - K * v;
        }
        __syncthreads();
    }
}

// T (16 x 16, upper) of the block reflectors of 16 consecutive columns,
// H = I - V T V^T (forward, columnwise): the Gram matrix of the reflectors on
// the fp64 MFMA, then the recurrence, one lane per row.  One wave per block.
__global__ __launch_bounds__(64) void eig_tfactor_kernel(const SvdEigDev* __restrict__ tasks,
                                                        const TileDev* __restrict__ units) {
    __shared__ double Gm[16][17], Tm[16][17];
    const SvdEigDev tk = tasks[units[blockIdx.x].task];
    const int blk = units[blockIdx.x].tm, n = tk.kx, lane = threadIdx.x, lm = lane % 16, lk = lane / 16;
    if (tk.flags[1]) return;
    const gptr<const double> R = to_global(tk.b);
    const int j = 16 * blk + lm;
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int r0 = 16 * blk; r0 < n; r0 += 4) {
        const int r = r0 + lk;
        const double v = (j < n && r < n) ? R[j * n + r] : 0.0;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v, v, acc, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) Gm[lk + 4 * i][lm] = acc[i];
    __syncthreads();
    if (lane < 16) {
        for (int i = 0; i < 16; i++) {
            const int col = 16 * blk + i;
            const double ti = col < n ? tk.tau[col] : 0.0;
            double v = 0.0;
            if (i == lane) {
                v = ti;
            } else if (i > lane) {
                double s = 0.0;
                for (int l = lane; l < i; l++) s += Tm[lane][l] * Gm[l][i];
                v = -ti * s;
            }
            Tm[lane][i] = v;
        }
    }
    __syncthreads();
    const gptr<double> out = to_global(tk.tb) + 256 * blk;
#pragma unroll
    for (int i = 0; i < 4; i++) out[(lk + 4 * i) * 16 + lm] = Tm[lk + 4 * i][lm];
}

// ------------------------------------------------ eigenvalues and -vectors
// Number of eigenvalues of T below x: sign changes of the leading minors,
// rescaled every four steps.
__device__ inline int sturm_count(cptr de, int n, double x) {
    double p0 = 1.0, p1 = de[0] - x;
    bool neg = p1 < 0.0;
    int c = neg;
    int i = 1;
    auto step = [&](int q) __attribute__((always_inline)) {
        const double p2 = (de[2 * q] - x) * p1 - de[2 * q + 1] * p0;
        const bool ng = p2 < 0.0;
        c += ng != neg;
        neg = ng;
        p0 = p1;
        p1 = p2;
    };
    for (; i + 4 <= n; i += 4) {
        step(i);
        step(i + 1);
        step(i + 2);
        step(i + 3);
        const int e = __builtin_amdgcn_frexp_exp(fmax(fabs(p0), fabs(p1)));
        p0 = __builtin_amdgcn_ldexp(p0, -e);
        p1 = __builtin_amdgcn_ldexp(p1, -e);
    }
    for (; i < n; i++) step(i);
    return c;
}

// 64 eigenvalues and eigenvectors of T per workgroup, one per lane.
// Eigenvalues: each step splits the intervals in five, one Sturm count per
// wave (24 steps, 5^24 > 2^55).  Vectors: the twisted factorisation of
// T - lambda (forward by wave 0, backward by wave 1 at the same time), the
// twist where its pivot is smallest, and the two back substitutions.  Every
// lane runs a serial chain of kx steps, so the time is their latency; the
// factors pass through global memory, lanes side by side.
// Eigenvectors of close eigenvalues come out less orthogonal; the caller
// measures and refines them.
__global__ __launch_bounds__(256) void eig_vectors_kernel(const SvdEigDev* __restrict__ tasks,
                                                         const TileDev* __restrict__ units) {
    __shared__ int cnt[4][64], gi[4][64];
    __shared__ double gm[4][64];
    const SvdEigDev tk = tasks[units[blockIdx.x].task];
    const int n = tk.kx, lane = threadIdx.x % WAVE, w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / WAVE);
    if (tk.flags[1]) return;
    const int k = 64 * units[blockIdx.x].tm + lane, kk = min(k, n - 1);
    const cptr de = (cptr)(tk.de), ee = (cptr)(tk.e);
    double lo = 0.0, hi = 0.0;
    {
        double a = -1e308, b = -1e308;
        for (int i = lane; i < n; i += WAVE) {
            const double r = (i > 0 ? fabs(tk.e[i - 1]) : 0.0) + (i + 1 < n ? fabs(tk.e[i]) : 0.0);
            a = fmax(a, tk.de[2 * i] + r);
            b = fmax(b, r - tk.de[2 * i]);
        }
        hi = wave_max(a);
        lo = -wave_max(b);
        const double pad = 1e-14 * fmax(fabs(lo), fabs(hi));
        hi += pad;
        lo -= pad;
    }
    const double pivmin = 1e-32 * (hi - lo);
    for (int it = 0; it < 24; it++) {
        const double h = (hi - lo) * 0.2;
        cnt[w][lane] = sturm_count(de, n, lo + h * (w + 1));
        __syncthreads();
        const double base = lo;
        double nlo = lo, nhi = hi;
#pragma unroll
        for (int s = 3; s >= 0; s--)
            if (cnt[s][lane] > kk) nhi = base + h * (s + 1);
#pragma unroll
        for (int s = 0; s < 4; s++)
            if (cnt[s][lane] <= kk) nlo = base + h * (s + 1);
        lo = nlo;
        hi = nhi;
        __syncthreads();
    }
    const double lam = 0.5 * (lo + hi);
    const gptr<double> Lp = to_global(tk.s), Lm = to_global(tk.vt), Z = to_global(tk.z);
    auto inv = [&](double q) __attribute__((always_inline)) {
        return refined_rcp(fabs(q) < pivmin ? copysign(pivmin, q) : q);
    };
    if (w == 0) {
        double q = de[0] - lam;
        for (int i = 0; i + 1 < n; i++) {
            const double l = ee[i] * inv(q);
            if (k < n) Lp[i * n + k] = l;
            q = de[2 * i + 2] - lam - ee[i] * l;
        }
    } else if (w == 1) {
        double q = de[2 * n - 2] - lam;
        for (int i = n - 2; i >= 0; i--) {
            const double l = ee[i] * inv(q);
            if (k < n) Lm[(i + 1) * n + k] = l;
            q = de[2 * i] - lam - ee[i] * l;
        }
    }
    __syncthreads();
    {
        double best = 1e308;
        int at = n * w / 4;
        for (int i = n * w / 4; i < n * (w + 1) / 4; i++) {
            double g = de[2 * i] - lam;
            if (k < n) {
                if (i > 0) g -= ee[i - 1] * Lp[(i - 1) * n + k];
                if (i + 1 < n) g -= ee[i] * Lm[(i + 1) * n + k];
            }
            if (fabs(g) < best) {
                best = fabs(g);
                at = i;
            }
        }
        gm[w][lane] = best;
        gi[w][lane] = at;
    }
    __syncthreads();
    int r = gi[0][lane];
    {
        double best = gm[0][lane];
#pragma unroll
        for (int v = 1; v < 4; v++)
            if (gm[v][lane] < best) {
                best = gm[v][lane];
                r = gi[v][lane];
            }
    }
    __syncthreads();
    double ss = 0.0;
    if (w == 0 && k < n) {
        double z = 1.0;
        Z[r * n + k] = 1.0;
#pragma unroll 4
        for (int i = n - 2; i >= 0; i--) {
            const double l = Lp[i * n + k];
            if (i < r) {
                z = -l * z;
                ss += z * z;
                Z[i * n + k] = z;
            }
        }
    } else if (w == 1 && k < n) {
        double z = 1.0;
#pragma unroll 4
        for (int i = 1; i < n; i++) {
            const double l = Lm[i * n + k];
            if (i > r) {
                z = -l * z;
                ss += z * z;
                Z[i * n + k] = z;
            }
        }
    }
    gm[w][lane] = ss;
    __syncthreads();
    const double f = refined_rsqrt(1.0 + gm[0][lane] + gm[1][lane]);
    if (k < n)
        for (int i = w; i < n; i += 4) Z[i * n + k] *= f;
}

// V = Q Z: the block reflectors, last first, applied to strips of 16 columns
// of Z, one strip per wave, in registers.  A strip's row tile t, register i,
// lane l holds row 16 t + 4 i + l / 16, column l % 16: the accumulator layout
// of the fp64 MFMA is also its B operand layout for the four rows of step i,
// so W = V^T Z and T W feed the next product without moving.  V's rows sit in
// LDS with a stride of 17, which both operand reads cross without conflicts.
template<int TILES>
__global__ __launch_bounds__(256) void eig_back_kernel(const SvdEigDev* __restrict__ tasks,
                                                      const TileDev* __restrict__ units) {
    extern __shared__ double lds[];
    const SvdEigDev tk = tasks[units[blockIdx.x].task];
    const int n = tk.kx, tid = threadIdx.x, lane = tid % WAVE, lm = lane % 16, lk = lane / 16;
    if (n > 16 * TILES || tk.flags[1]) return;
    double* Vs = lds;                      // 16 TILES rows of stride 17
    double* Ts = lds + 16 * TILES * 17;    // 16 x 17
    const int c = 64 * units[blockIdx.x].tm + 16 * (tid / WAVE) + lm;
    const gptr<double> Z = to_global(tk.z);
    const gptr<const double> R = to_global(tk.b), Tb = to_global(tk.tb);
    d4 z[TILES];
#pragma unroll
    for (int t = 0; t < TILES; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = 16 * t + 4 * i + lk;
            z[t][i] = (r < n && c < n) ? Z[r * n + c] : 0.0;
        }
    for (int blk = (n - 1) / 16; blk >= 0; blk--) {
        __syncthreads();
        for (int e = tid; e < 16 * 16 * TILES; e += 256) {
            const int jj = e / (16 * TILES), i = e % (16 * TILES), j = 16 * blk + jj;
            Vs[i * 17 + jj] = (j < n && i < n && i > j) ? R[j * n + i] : 0.0;
        }
        Ts[(tid / 16) * 17 + tid % 16] = Tb[256 * blk + tid];
        __syncthreads();
        d4 wv = {0.0, 0.0, 0.0, 0.0}, wv2 = wv;
#pragma unroll
        for (int t = 0; t < TILES; t++) {
            if (t < blk || 16 * t >= n) continue;
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                wv = __builtin_amdgcn_mfma_f64_16x16x4f64(Vs[(16 * t + 4 * i + lk) * 17 + lm], z[t][i], wv, 0, 0, 0);
                wv2 = __builtin_amdgcn_mfma_f64_16x16x4f64(Vs[(16 * t + 4 * i + 4 + lk) * 17 + lm], z[t][i + 1], wv2, 0,
                                                           0, 0);
            }
        }
        wv += wv2;
        d4 tw = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < 4; i++)
            tw = __builtin_amdgcn_mfma_f64_16x16x4f64(Ts[lm * 17 + 4 * i + lk], wv[i], tw, 0, 0, 0);
#pragma unroll
        for (int t = 0; t < TILES; t++) {
            if (t < blk || 16 * t >= n) continue;
#pragma unroll
            for (int i = 0; i < 4; i++)
                z[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-Vs[(16 * t + lm) * 17 + 4 * i + lk], tw[i], z[t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int t = 0; t < TILES; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = 16 * t + 4 * i + lk;
            if (r < n && c < n) Z[r * n + c] = z[t][i];
        }
}

// --------------------------------------------------- checks and corrections
// s <- (3 - s) / 2 for s = V^T V, after measuring its distance from one
__global__ __launch_bounds__(1024) void eig_polish_kernel(const SvdEigDev* __restrict__ tasks) {
    const SvdEigDev tk = tasks[blockIdx.x];
    const int n = tk.kx, lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    if (tk.flags[1]) return;
    const gptr<double> S = to_global(tk.s);
    bool fine = true;
    for (int r = wave; r < n; r += 16) {
        double sum = 0.0;
        for (int c = lane; c < n; c += WAVE) {
            const double v = S[r * n + c], one = r == c ? 1.0 : 0.0;
            sum += fabs(v - one);
            S[r * n + c] = 1.5 * one - 0.5 * v;
        }
        fine = fine && wave_sum(sum) <= EIG_DEFECT;  // false for NaN
    }
    if (!__syncthreads_and(fine) && threadIdx.x == 0) tk.flags[1] = 1;
}

// b <- I + E from b = G = X'^T X' and the checks that decide whether the block
// is this path's and which form of the step it takes
__global__ __launch_bounds__(1024) void eig_refine_kernel(const SvdEigDev* __restrict__ tasks) {
    __shared__ double d[SVD_EIG_MAX_COLS], root[SVD_EIG_MAX_COLS], red[16];
    const SvdEigDev tk = tasks[blockIdx.x];
    const int n = tk.kx, tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    if (n > SVD_EIG_MAX_COLS || tk.flags[1]) return;
    const gptr<double> G = to_global(tk.b);
    double fro = 0.0;
    for (int i = tid; i < n; i += 1024) {
        const double v = G[i * n + i];
        d[i] = v;
        root[i] = sqrt(v);
        fro += v;
    }
    fro = wave_sum(fro);
    if (lane == 0) red[wave] = fro;
    __syncthreads();
    fro = 0.0;
    for (int w = 0; w < 16; w++) fro += red[w];
    const double live = fmax(JACOBI_QUIET, JACOBI_DEAD2 * fro);
    const double tol = fmax(1e-15, 2.220446049250313e-16 * tk.mx);
    bool fine = true, small = true;
    int dead = 0;
    for (int r = wave; r < n; r += 16) {
        const double dr = d[r], rr = root[r];
        double sum = 0.0;
        for (int c = lane; c < n; c += WAVE) {
            const double g = G[r * n + c], scale = rr * root[c];
            double e = 1.0;
            if (c != r) {
                e = g / (d[c] - dr);
                // as orthogonal as the sweeps ask: turned only if the turn is
                // slight (close values would turn far for nothing)
                if (fabs(g) <= tol * scale && !(fabs(e) <= 1e-9)) e = 0.0;
                if (dr <= live || d[c] <= live) e = 0.0;
                small = small && (e == 0.0 || fabs(g) <= EIG_SMALL * scale);
                sum += fabs(e);
            }
            G[r * n + c] = e;
        }
        const double row = wave_sum(sum);
        small = small && row <= EIG_SMALL;
        fine = fine && row <= EIG_TURN && dr == dr;
        dead += dr <= live && lane == 0;
    }
    // a wave has at most kx / 16 rows: the count fits the vote's bits
    int total = 0;
    for (int q = 0; q < (SVD_EIG_MAX_COLS + 15) / 16; q++) total += __syncthreads_count(q < dead);
    fine = __syncthreads_and(fine && total <= EIG_DEAD);
    small = __syncthreads_and(small);
    if (tid == 0) {
        if (!fine) tk.flags[1] = 1;
        if (!small) tk.flags[3] = 0;
    }
}

// b <- I + E + E^2 / 2 = (1 + s) / 2 for s = (I + E)^2
__global__ __launch_bounds__(1024) void eig_second_kernel(const SvdEigDev* __restrict__ tasks) {
    const SvdEigDev tk = tasks[blockIdx.x];
    const int n = tk.kx;
    if (tk.flags[1] || tk.flags[3]) return;
    const gptr<const double> S = to_global(tk.s);
    const gptr<double> Q = to_global(tk.b);
    for (int e = threadIdx.x; e < n * n; e += 1024) Q[e] = 0.5 * S[e] + (e / n == e % n ? 0.5 : 0.0);
}

// Cosines of X'' after the second form (b = X''^T X'').  A pair left alone may
// measure a rounding above the tolerance now, hence the margin.
__global__ __launch_bounds__(1024) void eig_verify_kernel(const SvdEigDev* __restrict__ tasks) {
    __shared__ double root[SVD_EIG_MAX_COLS], red[16];
    const SvdEigDev tk = tasks[blockIdx.x];
    const int n = tk.kx, tid = threadIdx.x;
    if (n > SVD_EIG_MAX_COLS || tk.flags[1] || tk.flags[3]) return;
    const gptr<const double> G = to_global(tk.b);
    double fro = 0.0;
    for (int i = tid; i < n; i += 1024) {
        fro += G[i * n + i];
        root[i] = sqrt(G[i * n + i]);
    }
    fro = wave_sum(fro);
    if (tid % WAVE == 0) red[tid / WAVE] = fro;
    __syncthreads();
    fro = 0.0;
    for (int w = 0; w < 16; w++) fro += red[w];
    const double live = sqrt(fmax(JACOBI_QUIET, JACOBI_DEAD2 * fro));
    const double tol = fmax(1e-15, 2.220446049250313e-16 * tk.mx);
    bool fine = true;
    for (int r = tid / WAVE; r < n; r += 16)
        for (int c = tid % WAVE; c < n; c += WAVE)
            if (c != r && root[r] > live && root[c] > live)
                fine = fine && fabs(G[r * n + c]) <= 1.1 * tol * (root[r] * root[c]);
    if (!__syncthreads_and(fine) && tid == 0) tk.flags[1] = 1;
}

// Singular values (column norms), their descending order (ties by column),
// the directions of null columns and the mark that takes the block from the
// Jacobi kernels.  A null column keeps its tiny norm as its singular value.  Its
// direction starts from the first unit vector that keeps half its length
// outside the other columns' span, or from the one that keeps most (in a
// square block with one null column none may keep more than 1 / sqrt(mx)), and is
// what two passes of Gram-Schmidt against every other column leave of it.
__global__ __launch_bounds__(1024) void eig_order_kernel(const SvdEigDev* __restrict__ tasks) {
    __shared__ double sg[SVD_EIG_MAX_COLS], inv[SVD_EIG_MAX_COLS], coef[SVD_EIG_MAX_COLS], red[16];
    __shared__ int pos[16];
    const SvdEigDev tk = tasks[blockIdx.x];
    const int n = tk.kx, mx = tk.mx, tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    if (n > SVD_EIG_MAX_COLS || tk.flags[1]) return;
    const gptr<double> X = to_global(tk.xt);
    bool fine = true;
    double fro = 0.0;
    for (int c = wave; c < n; c += 16) {
        double s = 0.0;
        for (int r = lane; r < mx; r += WAVE) s += X[c * mx + r] * X[c * mx + r];
        s = wave_sum(s);
        fine = fine && s < 1e300;
        fro += s;
        if (lane == 0) sg[c] = s;
    }
    if (lane == 0) red[wave] = fro;
    if (!__syncthreads_and(fine)) return;
    fro = 0.0;
    for (int w = 0; w < 16; w++) fro += red[w];
    const double live = fmax(JACOBI_QUIET, JACOBI_DEAD2 * fro);
    bool null = false;
    for (int c = tid; c < n; c += 1024) {
        const double s = sg[c], root = sqrt(s);
        inv[c] = s > live ? 1.0 / root : 0.0;  // 0: no direction yet
        null = null || !(inv[c] > 0.0);
        sg[c] = root;
    }
    const int last = __syncthreads_or(null) ? n : 0;
    for (int c = 0; c < last; c++) {
        if (inv[c] > 0.0) continue;  // uniform over the workgroup
        // squared length of each unit vector outside the span, 1024 at a time
        double most = -1.0;
        int at = 0;
        for (int r0 = 0; r0 < mx && most <= 0.25; r0 += 1024) {
            const int r = r0 + tid;
            double left = -1.0;
            if (r < mx) {
                left = 1.0;
                for (int d = 0; d < n; d++) {
                    const double q = X[d * mx + r] * inv[d];
                    left -= q * q;
                }
            }
            // the first above a quarter, else the largest
            const double score = left > 0.25 ? 4.0 - 0x1p-10 * tid : left, top = wave_max(score);
            const int lane_at = __builtin_ctzll(__ballot(score == top));
            __syncthreads();
            if (lane == 0) {
                red[wave] = top;
                pos[wave] = r0 + WAVE * wave + lane_at;
            }
            __syncthreads();
            for (int w = 0; w < 16; w++)
                if (red[w] > most) {
                    most = red[w];
                    at = pos[w];
                }
        }
        for (int r = tid; r < mx; r += 1024) X[c * mx + r] = r == at ? 1.0 : 0.0;
        for (int pass = 0; pass < 2; pass++) {
            __syncthreads();
            for (int d = wave; d < n; d += 16) {
                double s = 0.0;
                if (inv[d] > 0.0)
                    for (int r = lane; r < mx; r += WAVE) s += X[c * mx + r] * X[d * mx + r];
                s = wave_sum(s);
                if (lane == 0) coef[d] = s * inv[d] * inv[d];
            }
            __syncthreads();
            for (int r = tid; r < mx; r += 1024) {
                double v = X[c * mx + r];
                for (int d = 0; d < n; d++)
                    if (inv[d] > 0.0) v -= coef[d] * X[d * mx + r];
                X[c * mx + r] = v;
            }
        }
        __syncthreads();
        double s = 0.0;
        for (int r = lane; r < mx; r += WAVE) s += X[c * mx + r] * X[c * mx + r];
        s = wave_sum(s);  // every wave: the same value
        // at least 1 / kx keeps some unit vector; what did not is not for here
        if (!(s > 1e-4)) {
            if (tid == 0) tk.flags[1] = 1;
            return;
        }
        if (tid == 0) inv[c] = 1.0 / sqrt(s);
        __syncthreads();
    }
    for (int c = tid; c < n; c += 1024) {
        const double sc = sg[c];
        int rank = 0;
        for (int q = 0; q < n; q++) rank += (sg[q] > sc) || (sg[q] == sc && q < c);
        tk.order[rank] = c;
        tk.sig[rank] = inv[c];
        tk.t.s[rank] = ldexp(sc, tk.flags[2]);
    }
    if (tid == 0) tk.flags[0] = 1;
}

// U and V^T of the block from the columns of X and V in rank order, 32 ranks
// per workgroup; the factor stored column by column goes through LDS tiles.
template<typename T>
__global__ __launch_bounds__(256) void eig_write_kernel(const SvdEigDev* __restrict__ tasks,
                                                       const TileDev* __restrict__ units) {
    __shared__ double tile[32][33];
    const SvdEigDev tk = tasks[units[blockIdx.x].task];
    if (!tk.flags[0]) return;
    const int n = tk.kx, r0 = 32 * units[blockIdx.x].tm, tx = threadIdx.x % 32, ty = threadIdx.x / 32;
    const bool trans = tk.t.m < tk.t.n;
    const gptr<const double> X = to_global(tk.xt), V = to_global(tk.z), inv = to_global(tk.sig);
    const gptr<const int32_t> order = to_global(tk.order);
    const gptr<T> U = to_global(static_cast<T*>(tk.t.u)), Vo = to_global(static_cast<T*>(tk.t.v));
    // rows: the columns of X (m < n) or V, as rows of V^T; cols: the others,
    // as columns of U
    const gptr<const double> rows = trans ? X : V, cols = trans ? V : X;
    const int rl = trans ? tk.mx : n, cl = trans ? n : tk.mx;
    for (int q = ty; q < 32; q += 8) {
        const int rank = r0 + q;
        if (rank >= n) break;
        const double f = trans ? inv[rank] : 1.0;
        const gptr<const double> p = rows + int64_t(order[rank]) * rl;
        for (int i = tx; i < rl; i += 32) Vo[int64_t(rank) * rl + i] = T(p[i] * f);
    }
    for (int i0 = 0; i0 < cl; i0 += 32) {
        for (int q = ty; q < 32; q += 8) {
            const int rank = r0 + q;
            if (rank < n && i0 + tx < cl)
                tile[q][tx] = cols[int64_t(order[rank]) * cl + i0 + tx] * (trans ? 1.0 : inv[rank]);
        }
        __syncthreads();
        for (int q = ty; q < 32; q += 8)
            if (i0 + q < cl && r0 + tx < n) U[int64_t(i0 + q) * n + r0 + tx] = T(tile[tx][q]);
        __syncthreads();
    }
}

}  // namespace

namespace {
template<int TILES>
void launch_back(const SvdEigDev* tasks, const TileDev* units, dim3 grid, hipStream_t st) {
    constexpr int lds = (16 * TILES * 17 + 16 * 17) * int(sizeof(double));
    // once per kernel and process: the static's initialisation is thread-safe
    static const bool allowed = [] {
        if (lds > 64 * 1024)
            check(hipFuncSetAttribute(reinterpret_cast<const void*>(eig_back_kernel<TILES>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, lds),
                  "dynamic LDS attribute");
        return true;
    }();
    (void)allowed;
    hipLaunchKernelGGL(eig_back_kernel<TILES>, grid, dim3(256), size_t(lds), st, tasks, units);
}
}  // namespace

void launch_svd_eig(int stage, int variant, const SvdEigDev* tasks, const TileDev* units, int64_t num, int dtype,
                    hipStream_t st) {
    if (num <= 0) return;
    const dim3 grid(static_cast<unsigned>(num));
    switch (stage) {
        case SVD_EIG_LOAD:
            if (dtype == 0)
                hipLaunchKernelGGL(eig_load_kernel<double>, grid, dim3(1024), 0, st, tasks);
            else
                hipLaunchKernelGGL(eig_load_kernel<float>, grid, dim3(1024), 0, st, tasks);
            break;
        case SVD_EIG_TRIDIAG:
            if (variant == 0)
                hipLaunchKernelGGL((eig_tridiag_kernel<16, 4, 4>), grid, dim3(256), 0, st, tasks);
            else if (variant == 1)
                hipLaunchKernelGGL((eig_tridiag_kernel<32, 4, 8>), grid, dim3(512), 0, st, tasks);
            else if (variant == 2)
                hipLaunchKernelGGL((eig_tridiag_kernel<48, 4, 12>), grid, dim3(768), 0, st, tasks);
            else if (variant == 3)
                hipLaunchKernelGGL((eig_tridiag_glb_kernel<5, 3>), grid, dim3(1024), 0, st, tasks);
            else
                hipLaunchKernelGGL((eig_tridiag_glb_kernel<SVD_EIG_MAX_COLS / WAVE, 1>), grid, dim3(1024), 0, st, tasks);
            break;
        case SVD_EIG_TFACTOR:
            hipLaunchKernelGGL(eig_tfactor_kernel, grid, dim3(64), 0, st, tasks, units);
            break;
        case SVD_EIG_VECTORS:
            hipLaunchKernelGGL(eig_vectors_kernel, grid, dim3(256), 0, st, tasks, units);
            break;
        case SVD_EIG_BACK:
            if (variant == 0)
                launch_back<4>(tasks, units, grid, st);
            else if (variant == 1)
                launch_back<8>(tasks, units, grid, st);
            else if (variant == 2)
                launch_back<12>(tasks, units, grid, st);
            else if (variant == 3)
                launch_back<20>(tasks, units, grid, st);
            else
                launch_back<SVD_EIG_MAX_COLS / 16>(tasks, units, grid, st);
            break;
        case SVD_EIG_POLISH:
            hipLaunchKernelGGL(eig_polish_kernel, grid, dim3(1024), 0, st, tasks);
            break;
        case SVD_EIG_REFINE:
            hipLaunchKernelGGL(eig_refine_kernel, grid, dim3(1024), 0, st, tasks);
            break;
        case SVD_EIG_SECOND:
            hipLaunchKernelGGL(eig_second_kernel, grid, dim3(1024), 0, st, tasks);
            break;
        case SVD_EIG_VERIFY:
            hipLaunchKernelGGL(eig_verify_kernel, grid, dim3(1024), 0, st, tasks);
            break;
        case SVD_EIG_ORDER:
            hipLaunchKernelGGL(eig_order_kernel, grid, dim3(1024), 0, st, tasks);
            break;
        case SVD_EIG_WRITE:
            if (dtype == 0)
                hipLaunchKernelGGL(eig_write_kernel<double>, grid, dim3(256), 0, st, tasks, units);
            else
                hipLaunchKernelGGL(eig_write_kernel<float>, grid, dim3(256), 0, st, tasks, units);
            break;
        default:
            throw std::runtime_error("svd: unknown stage");
    }
    check(hipGetLastError(), "svd eigenvector stage launch");
}

}  // namespace tns
