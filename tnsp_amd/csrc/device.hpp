// Device helpers shared by the kernel files: global-memory pointers, cross-lane
// sums on the VALU, Householder reflectors and the Jacobi block conventions.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace tns {

namespace {

constexpr int WG = 256;
constexpr int WAVE = 64;

// Device pointers read from task records are generic to the compiler, so
// accesses through them compile to flat instructions, and a flat load is
// counted by the LDS counter as well as the vector-memory one: a wait for an
// LDS read then also waits for every global load in flight (the prefetch of
// a pipelined loop included).  Every task buffer is global memory; accesses
// through these pointers compile to global_load / global_store.
template<typename T>
using gptr = __attribute__((address_space(1))) T*;
template<typename T>
__device__ inline gptr<T> to_global(T* p) {
    return (gptr<T>)(p);
}

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int DPP_ROW_ROR1 = 0x121, DPP_ROW_ROR2 = 0x122, DPP_ROW_ROR4 = 0x124, DPP_ROW_ROR8 = 0x128;

// a double moved across lanes by a DPP row shift (two 32-bit halves)
template<int CTRL>
__device__ inline double dpp_f64(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, int(unsigned(u)), CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, int(unsigned(u >> 32)), CTRL, 0xF, 0xF, true);
    return __builtin_bit_cast(double, (static_cast<unsigned long long>(unsigned(hi)) << 32) | unsigned(lo));
}

// v of lane l plus v of lane l ^ 16 (SWAP = 16) or l ^ 32 (SWAP = 32), by the
// gfx950 row / half swaps: permlane16_swap(x, x) leaves each lane one of
// {x_l, x_(l^16)} in each of its two results (even rows keep their own value
// in the first and receive the partner's in the second, odd rows the other
// way round), so the two results add up to the pair sum in every lane; the
// same holds for permlane32_swap with halves.  VALU only, no LDS.
template<int SWAP>
__device__ inline double swap_sum(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = unsigned(u), hi = unsigned(u >> 32);
    unsigned lo0, lo1, hi0, hi1;
    if constexpr (SWAP == 16) {
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        lo0 = l[0];
        lo1 = l[1];
        hi0 = h[0];
        hi1 = h[1];
    } else {
        const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        lo0 = l[0];
        lo1 = l[1];
        hi0 = h[0];
        hi1 = h[1];
    }
    const double a = __builtin_bit_cast(double, (static_cast<unsigned long long>(hi0) << 32) | lo0);
    const double b = __builtin_bit_cast(double, (static_cast<unsigned long long>(hi1) << 32) | lo1);
    return a + b;
}

// butterfly sum over the 8 lanes {l ^ 8k}: l ^ 8 by a DPP rotate by 8 within
// the 16-lane row, l ^ 16 and l ^ 32 by the row and half swaps; every lane
// ends with the same value (the additions commute)
__device__ inline double sum8(double v) {
    v += dpp_f64<DPP_ROW_ROR8>(v);
    v = swap_sum<16>(v);
    return swap_sum<32>(v);
}

// sum over the 16 lanes of a DPP row by rotations 8, 4, 2, 1: after the
// step with rotation r every lane holds the sum of its 16/r-lane orbit, and
// the two lanes of each addition hold the same two values, so every lane of
// the row ends with bitwise the same sum (IEEE addition commutes)
__device__ inline double row_sum16(double v) {
    v += dpp_f64<DPP_ROW_ROR8>(v);
    v += dpp_f64<DPP_ROW_ROR4>(v);
    v += dpp_f64<DPP_ROW_ROR2>(v);
    v += dpp_f64<DPP_ROW_ROR1>(v);
    return v;
}

// sum within aligned groups of G lanes (G = 16, 32 or 64), VALU only: every
// lane of the group ends with bitwise the same value
__device__ inline double group_sum(double v, int G) {
    v = row_sum16(v);
    if (G >= 32) v = swap_sum<16>(v);
    if (G >= 64) v = swap_sum<32>(v);
    return v;
}

__device__ inline double wave_sum(double v) { return group_sum(v, WAVE); }

// maximum over the wave (rotations within rows, then the row / half swaps)
__device__ inline double wave_max(double v) {
    v = fmax(v, dpp_f64<DPP_ROW_ROR8>(v));
    v = fmax(v, dpp_f64<DPP_ROW_ROR4>(v));
    v = fmax(v, dpp_f64<DPP_ROW_ROR2>(v));
    v = fmax(v, dpp_f64<DPP_ROW_ROR1>(v));
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = unsigned(u), hi = unsigned(u >> 32);
    {
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        const double a = __builtin_bit_cast(double, (static_cast<unsigned long long>(unsigned(h[0])) << 32) | unsigned(l[0]));
        const double b = __builtin_bit_cast(double, (static_cast<unsigned long long>(unsigned(h[1])) << 32) | unsigned(l[1]));
        v = fmax(a, b);
    }
    const unsigned long long u2 = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo2 = unsigned(u2), hi2 = unsigned(u2 >> 32);
    const auto l = __builtin_amdgcn_permlane32_swap(lo2, lo2, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(hi2, hi2, false, false);
    const double a = __builtin_bit_cast(double, (static_cast<unsigned long long>(unsigned(h[0])) << 32) | unsigned(l[0]));
    const double b = __builtin_bit_cast(double, (static_cast<unsigned long long>(unsigned(h[1])) << 32) | unsigned(l[1]));
    return fmax(a, b);
}

// Scale exponent of a block for the Jacobi SVDs: the block is multiplied by
// 2^-e (exact) so that its largest entry lies in [1, 2); squared column norms
// then neither overflow nor underflow for every column that matters.  0 for
// an all-zero or non-finite block.
__device__ inline int jacobi_scale_exponent(double amax) {
    return (amax > 0.0 && amax <= 1.79e308) ? ilogb(amax) : 0;
}

// Squared column norm (after the scaling) at or below which a column counts
// as zero: it takes part in no rotation and gets singular value 0.  Its true
// singular value is below 1e-100 of the largest entry.  A column of an
// exactly rank-deficient block shrinks by a rounding factor with every
// rotation against the columns spanning its space, and would otherwise keep
// rotating down into the underflow range, where its relative cosines stay
// of order one and the sweeps never end.
constexpr double JACOBI_QUIET = 1e-200;

// A column whose squared norm falls to JACOBI_DEAD2 times the block's squared
// Frobenius norm (1e-15 of the norm, about 4.5 ulp) is rounding noise: it
// takes part in no further rotation.  The columns of an exactly
// rank-deficient block that shrink into the null space are noise inside the
// span of the others, so their cosines with those stay of order one; they
// shrink only slowly as they mix among themselves, and would otherwise keep
// the sweeps going for dozens of sweeps or forever.  Their singular values
// come out at that noise level, as LAPACK's do.
constexpr double JACOBI_DEAD2 = 1e-30;

template<int NT>
__device__ inline double block_sum(double v, double* red) {
    v = wave_sum(v);
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    double t = 0;
    for (int w = 0; w < NT / WAVE; w++) t += red[w];
    return t;
}

// hardware reciprocal / reciprocal square root refined by two Newton steps:
// within a few ulp where argument and result are normal numbers (the Jacobi
// rotations' arguments lie in [1, inf); the tridiagonalisations' and twisted
// factorisations' come from blocks scaled to entries of order one, the pivots
// floored)
__device__ inline double refined_rcp(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
}

__device__ inline double refined_rsqrt(double y) {
    double r = __builtin_amdgcn_rsq(y);
    r = r * fma(-0.5 * y * r, r, 1.5);
    return r * fma(-0.5 * y * r, r, 1.5);
}

// Householder reflector of a column with diagonal entry alpha and squared
// norm sigma below it: H = I - tau v v^T, v = (1, x / (alpha - beta)),
// H (alpha, x) = (beta, 0).  Every thread computes the same values.
__device__ inline void householder(double alpha, double sigma, double& tau, double& beta) {
    if (sigma == 0.0) {
        tau = 0.0;
        beta = alpha;
    } else {
        beta = -copysign(sqrt(alpha * alpha + sigma), alpha);
        tau = (beta - alpha) / beta;
    }
}

}  // namespace

}  // namespace tns
