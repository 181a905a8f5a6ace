// Hop-proposal network for Metropolis sampling of fermion occupations on an
// H x W lattice: 3x3 convolutions (zero padding, NCHW, fp32 activations and
// accumulation, bf16 weights), ReLU, and the masked softmax over the 4 H W
// nearest-neighbour hops (direction d at site s: 0 up, 1 down, 2 left,
// 3 right; valid when s is filled and its neighbour exists and is empty).
// Forward, both backward passes, the loss gradient, Adam and the proposal
// sampling are written here; the caller owns every buffer.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <string>
#include <type_traits>

#include "proposal.hpp"

namespace tns {
namespace {

constexpr int NT = 256;
constexpr size_t CONV_LDS_MAX = 160 * 1024;

__device__ inline float bf16_to_f(uint16_t h) { return __uint_as_float(uint32_t(h) << 16); }

__device__ inline uint16_t f_to_bf16(float x) {
    uint32_t u = __float_as_uint(x);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return uint16_t(u >> 16);
}

typedef float f4 __attribute__((ext_vector_type(4)));

// LDS row of one padded channel plane of HP x WP values: with a stride of 4
// modulo 8 words the 16 channels x 4 positions (or 16 positions x 4 channels)
// of an MFMA operand read fall into different banks.  Without the padding
// where it would not fit.
inline int plane_stride(int HP, int WP) {
    int s = HP * WP;
    while (s % 8 != 4) s++;
    return s;
}

// One 3x3 convolution as a product on the fp32 MFMA (16x16x4), for the forward
// pass (out = y, in = x, channels m = co, k = ci) and for the data gradient
// (out = dx, in = dy masked by the ReLU of y, m = ci, k = co, flipped taps):
//   out[b, m, p] = bias[m] + sum_{tap, k} w[m, k, tap] in[b, k, p + tap]
// Rows of a tile are 16 output channels, columns 16 positions; the reduction
// runs tap by tap over groups of 4 input channels.  A workgroup keeps the
// weights (bf16) in LDS and walks samples; the padded input planes of the
// sample sit in LDS, so a tap is an offset.  Each wave takes every fourth
// column tile and all MT row tiles.
// Lane l holds w(m0 + l % 16, k0 + l / 16) and in(k0 + l / 16, p0 + l % 16);
// accumulator rows 4 (l / 16) + i.
// The VALU version read LDS twice per multiply-add: 66 (forward) and 84 us
// (data gradient) per launch on 1024 samples of 32 channels, 8 x 8; this
// kernel 25 us for either.  The floor is 8 us of fp32 arithmetic.
template<int MT>
__global__ __launch_bounds__(NT) void conv_mfma_kernel(const float* __restrict__ in, const float* __restrict__ relu_y,
                                                       const uint16_t* __restrict__ w, const float* __restrict__ bias,
                                                       float* __restrict__ out, int B, int M, int K, int H, int W,
                                                       int S, int flip, int relu) {
    extern __shared__ float sm[];
    const int HP = H + 2, WP = W + 2, HW = H * W;
    float* xs = sm;                                             // K planes of stride S
    uint16_t* ws = reinterpret_cast<uint16_t*>(sm + K * S);     // [tap][k][m]
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int lm = lane % 16, lk = lane / 16;
    for (int q = tid; q < M * K; q += NT) {
        const int m = flip ? q % M : q / K, k = flip ? q / M : q % K;
#pragma unroll
        for (int tap = 0; tap < 9; tap++) ws[((flip ? 8 - tap : tap) * K + k) * M + m] = w[q * 9 + tap];
    }
    // the border of every plane stays zero
    for (int e = tid; e < K * S; e += NT) xs[e] = 0.f;
    for (int b = blockIdx.x; b < B; b += gridDim.x) {
        __syncthreads();
        const float* ib = in + int64_t(b) * K * HW;
        const float* yb = relu_y ? relu_y + int64_t(b) * K * HW : nullptr;
        for (int e = tid; e < K * HW; e += NT) {
            const int k = e / HW, p = e - k * HW, i = p / W, j = p - i * W;
            float v = ib[e];
            if (yb && !(yb[e] > 0.f)) v = 0.f;
            xs[k * S + (i + 1) * WP + j + 1] = v;
        }
        __syncthreads();
        float* ob = out + int64_t(b) * M * HW;
        for (int p0 = 16 * wave; p0 < HW; p0 += 16 * (NT / 64)) {
            // columns beyond HW read position 0 and are not stored, rows
            // beyond M likewise read channel M - 1
            const int p = p0 + lm < HW ? p0 + lm : 0;
            const float* xp = xs + (p / W) * WP + p % W;
            f4 acc[MT];
            int mrow[MT];
#pragma unroll
            for (int t = 0; t < MT; t++) {
                mrow[t] = min(16 * t + lm, M - 1);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int m = 16 * t + 4 * lk + i;
                    acc[t][i] = bias && m < M ? bias[m] : 0.f;
                }
            }
            for (int tap = 0; tap < 9; tap++) {
                const float* xt = xp + (tap / 3) * WP + tap % 3;
                const uint16_t* wt = ws + tap * K * M;
#pragma unroll 2
                for (int k0 = 0; k0 < K; k0 += 4) {
                    // channels beyond K count nothing on either side
                    const int k = k0 + lk, kc = min(k, K - 1);
                    const bool ok = k < K;
                    const float x = ok ? xt[kc * S] : 0.f;
#pragma unroll
                    for (int t = 0; t < MT; t++) {
                        const float a = ok ? bf16_to_f(wt[kc * M + mrow[t]]) : 0.f;
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, x, acc[t], 0, 0, 0);
                    }
                }
            }
            if (p0 + lm < HW) {
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int m = 16 * t + 4 * lk + i;
                        if (m < M) ob[m * HW + p0 + lm] = relu ? fmaxf(acc[t][i], 0.f) : acc[t][i];
                    }
            }
        }
    }
}

// Partial weight / bias gradients over a chunk of samples per workgroup:
// part[chunk][co][ci][9] and partb[chunk][co], as a product on the fp32 MFMA
// with the positions as the reduction dimension:
//   part[co, n] = sum_{b, i, j} dy[b, co, i, j] x[b, ci, i + ky, j + kx],
//   n = (ci, ky, kx) flattened.
// A k step is 4 positions of one row; both operands are zero beyond the row.  Each wave takes every fourth tile of 16
// columns n and all MT row tiles of 16 channels co.
// Lane l holds dy(co0 + l % 16, p + l / 16) and x(p + l / 16, n0 + l % 16).
// The VALU version (one thread per weight, 64 samples per workgroup, 16
// workgroups for 1024 samples) took 3.8 ms per launch on 1024 samples of 32
// channels, 8 x 8; this kernel 31 us and its reduction 8.
template<int MT, int NPW>
__global__ __launch_bounds__(NT) void conv_bwd_weight_kernel(const float* __restrict__ dy,
                                                             const float* __restrict__ relu_y,
                                                             const float* __restrict__ x, float* __restrict__ part,
                                                             float* __restrict__ partb, int B, int per_chunk, int cin,
                                                             int cout, int H, int W, int S, int G) {
    extern __shared__ float sm[];
    const int WP = W + 2, HW = H * W;
    float* xs = sm;            // cin padded planes of stride S
    float* gs = sm + cin * S;  // cout planes H x W of stride G
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, chunk = blockIdx.x;
    const int lm = lane % 16, lk = lane / 16;
    const int nw = cout * cin * 9, N = cin * 9;
    f4 acc[MT][NPW];
    int xoff[NPW], goff[MT];
#pragma unroll
    for (int u = 0; u < NPW; u++) {
        // columns beyond N read column N - 1 and are not stored
        const int n = min(16 * (wave + 4 * u) + lm, N - 1);
        xoff[u] = (n / 9) * S + ((n % 9) / 3) * WP + n % 3;
#pragma unroll
        for (int t = 0; t < MT; t++) acc[t][u] = f4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int t = 0; t < MT; t++) goff[t] = min(16 * t + lm, cout - 1) * G;
    for (int e = tid; e < cin * S + cout * G; e += NT) sm[e] = 0.f;
    // bias: TB threads per channel, a power of two of neighbouring lanes
    int TB = 4;
    while (TB < 64 && 2 * TB * cout <= NT) TB *= 2;
    float accb = 0.f;
    const int b0 = chunk * per_chunk, b1 = min(B, b0 + per_chunk);
    for (int b = b0; b < b1; b++) {
        const float* xb = x + int64_t(b) * cin * HW;
        const float* gb = dy + int64_t(b) * cout * HW;
        const float* yb = relu_y ? relu_y + int64_t(b) * cout * HW : nullptr;
        __syncthreads();
        for (int e = tid; e < cin * HW; e += NT) {
            const int c = e / HW, p = e - c * HW, i = p / W, j = p - i * W;
            xs[c * S + (i + 1) * WP + j + 1] = xb[e];
        }
        for (int e = tid; e < cout * HW; e += NT) {
            const int c = e / HW, p = e - c * HW;
            float v = gb[e];
            if (yb && !(yb[e] > 0.f)) v = 0.f;
            gs[c * G + p] = v;
        }
        __syncthreads();
        for (int i = 0; i < H; i++) {
            for (int j = 0; j < W; j += 4) {
                // beyond the row both operands are zero
                const bool ok = j + lk < W;
                const int go = ok ? i * W + j + lk : 0, xo = ok ? i * WP + j + lk : 0;
                float a[MT];
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    const float v = gs[goff[t] + go];
                    a[t] = ok ? v : 0.f;
                }
#pragma unroll
                for (int u = 0; u < NPW; u++) {
                    const float r = xs[xoff[u] + xo];
                    const float v = ok ? r : 0.f;
#pragma unroll
                    for (int t = 0; t < MT; t++)
                        acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], v, acc[t][u], 0, 0, 0);
                }
            }
        }
        if (tid / TB < cout) {
            const float* gp = gs + (tid / TB) * G;
            for (int e = tid % TB; e < HW; e += TB) accb += gp[e];
        }
    }
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int u = 0; u < NPW; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int co = 16 * t + 4 * lk + i, n = 16 * (wave + 4 * u) + lm;
                if (co < cout && n < N) part[int64_t(chunk) * nw + co * N + n] = acc[t][u][i];
            }
    for (int o = 1; o < TB; o <<= 1) accb += __shfl_xor(accb, o, 64);
    if (tid / TB < cout && tid % TB == 0) partb[int64_t(chunk) * cout + tid / TB] = accb;
}

// out[k] = sum over the chunks of part[c][k], k < n, for the weights and the
// biases in one launch: 64 outputs per workgroup, its four waves take every
// fourth chunk and their sums meet in LDS (one thread per output left most of
// the chip idle behind a serial chain over the chunks).  A lane keeps eight
// sums: eight loads in flight, and chains of 16 additions over 512 chunks where
// one sum would make 128, whose rounding was most of the gradients' error.
__global__ __launch_bounds__(NT) void reduce_chunks_kernel(const float* __restrict__ part, const float* __restrict__ partb,
                                                           int chunks, int nw, int nb, float* __restrict__ dw,
                                                           float* __restrict__ db) {
    __shared__ float red[NT / 64][64];
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int wblocks = (nw + 63) / 64;
    const bool bias = int(blockIdx.x) >= wblocks;
    const int n = bias ? nb : nw;
    const float* src = bias ? partb : part;
    const int k = (int(blockIdx.x) - (bias ? wblocks : 0)) * 64 + lane;
    constexpr int R = 8;
    float s[R] = {};
    if (k < n) {
        for (int c = wave; c < chunks; c += R * (NT / 64)) {
            float v[R];
            // beyond the last chunk the last one is read and not added
#pragma unroll
            for (int u = 0; u < R; u++) v[u] = src[int64_t(min(c + u * (NT / 64), chunks - 1)) * n + k];
#pragma unroll
            for (int u = 0; u < R; u++) s[u] += c + u * (NT / 64) < chunks ? v[u] : 0.f;
        }
    }
    red[wave][lane] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    __syncthreads();
    if (wave == 0 && k < n) (bias ? db : dw)[k] = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
}

// hop h = d * H W + s: valid when site s is filled and its neighbour in
// direction d exists and is empty; returns the neighbour or -1
__device__ inline int hop_target(const int8_t* occ, int h, int H, int W) {
    const int HW = H * W, d = h / HW, s = h % HW, i = s / W, j = s % W;
    int ti = i, tj = j;
    if (d == 0) ti--;
    else if (d == 1) ti++;
    else if (d == 2) tj--;
    else tj++;
    if (ti < 0 || ti >= H || tj < 0 || tj >= W) return -1;
    const int t = ti * W + tj;
    return (occ[s] == 1 && occ[t] == 0) ? t : -1;
}

__device__ inline float wave_max(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ inline float wave_sumf(float v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// one wave per chain: masked log-softmax over the hops; with u != null draw
// a hop by inverse CDF (u in [0, 1)), else score the given hop.  logq gets
// log q(hop); hop gets -1 if no hop is valid.
__global__ __launch_bounds__(64) void hop_kernel(const float* __restrict__ logits, const int8_t* __restrict__ occ,
                                                 const float* __restrict__ u, int32_t* __restrict__ hop,
                                                 float* __restrict__ logq, int H, int W) {
    const int b = blockIdx.x, lane = threadIdx.x;
    const int n = 4 * H * W;
    const float* lg = logits + int64_t(b) * n;
    const int8_t* oc = occ + int64_t(b) * H * W;
    float mx = -INFINITY;
    for (int h = lane; h < n; h += 64)
        if (hop_target(oc, h, H, W) >= 0) mx = fmaxf(mx, lg[h]);
    mx = wave_max(mx);
    if (mx == -INFINITY) {
        if (lane == 0) {
            if (u) hop[b] = -1;
            logq[b] = 0.f;
        }
        return;
    }
    float z = 0.f;
    for (int h = lane; h < n; h += 64)
        if (hop_target(oc, h, H, W) >= 0) z += expf(lg[h] - mx);
    z = wave_sumf(z);
    if (!u) {
        if (lane == 0) {
            const int h = hop[b];
            logq[b] = (h >= 0 && h < n && hop_target(oc, h, H, W) >= 0) ? lg[h] - mx - logf(z) : -INFINITY;
        }
        return;
    }
    // inverse CDF in hop order, done by lane 0 over the (small) hop list
    if (lane == 0) {
        const float target = u[b] * z;
        float c = 0.f;
        int pick = -1, last = -1;
        for (int h = 0; h < n; h++) {
            if (hop_target(oc, h, H, W) < 0) continue;
            last = h;
            c += expf(lg[h] - mx);
            if (c > target) {
                pick = h;
                break;
            }
        }
        if (pick < 0) pick = last;
        hop[b] = pick;
        logq[b] = lg[pick] - mx - logf(z);
    }
}

// regression of the hop logit onto its target: loss_b = (l_h - t_b)^2,
// dlogits = 2 (l_h - t_b) / B at h, zero elsewhere
__global__ void hop_regression_kernel(const float* __restrict__ logits, const int32_t* __restrict__ hop,
                                      const float* __restrict__ target, float* __restrict__ dlogits,
                                      float* __restrict__ loss, int B, int n) {
    const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= int64_t(B) * n) return;
    const int b = int(e / n), h = int(e % n);
    float g = 0.f;
    if (h == hop[b]) {
        const float d = logits[e] - target[b];
        g = 2.f * d / float(B);
        loss[b] = d * d;
    }
    dlogits[e] = g;
}

__global__ void adam_kernel(float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
                            const float* __restrict__ g, uint16_t* __restrict__ wbf, int n, float lr, float b1,
                            float b2, float eps, float c1, float c2) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const float gk = g[k];
    const float mk = b1 * m[k] + (1.f - b1) * gk;
    const float vk = b2 * v[k] + (1.f - b2) * gk * gk;
    m[k] = mk;
    v[k] = vk;
    const float wk = w[k] - lr * (mk / c1) / (sqrtf(vk / c2) + eps);
    w[k] = wk;
    if (wbf) wbf[k] = f_to_bf16(wk);
}

__global__ void to_bf16_kernel(const float* __restrict__ w, uint16_t* __restrict__ wbf, int n) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) wbf[k] = f_to_bf16(w[k]);
}

__global__ void occ_to_input_kernel(const int8_t* __restrict__ occ, float* __restrict__ x, int64_t n) {
    const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < n) x[k] = float(occ[k]);
}

void check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

void allow(const void* k, size_t bytes) {
    if (bytes > 64 * 1024) (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes));
}

}  // namespace

void conv_check(int cin, int cout, int H, int W) {
    if (cin < 1 || cout < 1 || H < 1 || W < 1 || cin > 64 || cout > 64 || H > 32 || W > 32)
        throw std::runtime_error("conv3x3: channels must be in [1, 64] and the lattice at most 32 x 32");
    if (cout * cin * 9 > NT * 64) throw std::runtime_error("conv3x3: too many weights for the gradient kernel");
}

namespace {
void launch_conv_mfma(const float* in, const float* relu_y, const uint16_t* w, const float* bias, float* out, int B,
                      int M, int K, int H, int W, int flip, int relu, hipStream_t st) {
    const size_t wbytes = size_t(M) * K * 9 * sizeof(uint16_t);
    int S = plane_stride(H + 2, W + 2);
    if (size_t(K) * S * sizeof(float) + wbytes > CONV_LDS_MAX) S = (H + 2) * (W + 2);
    const size_t lds = size_t(K) * S * sizeof(float) + wbytes;
    // up to four workgroups per CU with the same number of samples each (one
    // more for some), the weights staged once per workgroup
    const int per = (B + 1023) / 1024;
    const dim3 grid(unsigned((B + per - 1) / per));
    auto go = [&](auto kernel) {
        allow(reinterpret_cast<const void*>(kernel), lds);
        hipLaunchKernelGGL(kernel, grid, dim3(NT), lds, st, in, relu_y, w, bias, out, B, M, K, H, W, S, flip, relu);
    };
    if (M <= 16)
        go(conv_mfma_kernel<1>);
    else if (M <= 32)
        go(conv_mfma_kernel<2>);
    else
        go(conv_mfma_kernel<4>);
}
}  // namespace

void launch_conv_fwd(const float* x, const uint16_t* w, const float* bias, float* y, int B, int cin, int cout, int H,
                     int W, int relu, hipStream_t st) {
    conv_check(cin, cout, H, W);
    if (B <= 0) return;
    if (size_t(cin * (H + 2) * (W + 2) + cout * cin * 9) * sizeof(float) > CONV_LDS_MAX)
        throw std::runtime_error("conv3x3: working set exceeds LDS");
    launch_conv_mfma(x, nullptr, w, bias, y, B, cout, cin, H, W, 0, relu, st);
    check(hipGetLastError(), "conv forward launch");
}

void launch_conv_bwd_data(const float* dy, const float* relu_y, const uint16_t* w, float* dx, int B, int cin, int cout,
                          int H, int W, hipStream_t st) {
    conv_check(cin, cout, H, W);
    if (B <= 0) return;
    if (size_t(cout * (H + 2) * (W + 2) + cout * cin * 9) * sizeof(float) > CONV_LDS_MAX)
        throw std::runtime_error("conv3x3: working set exceeds LDS");
    launch_conv_mfma(dy, relu_y, w, nullptr, dx, B, cin, cout, H, W, 1, 0, st);
    check(hipGetLastError(), "conv backward-data launch");
}

namespace {
// Samples per workgroup of the weight gradient: one while that gives at most
// 512 workgroups (each CU holds a few; a workgroup's samples are a serial
// chain), more beyond, so that the partial gradients (37 KB each at 32 channels)
// stay a small part of the traffic.  All layers with the reductions, 1 / 2 / 4 / 8
// samples per workgroup: 32 channels, 8 x 8, 64 samples 54 / 91 / 149 / 259 us,
// 512 samples 94 / 98 / 153 / 267, 1024 samples (2 at least) 128 / 156 / 269; 24
// channels, 10 x 10, 128 samples 51 / 84 / 145 / 259; 8 channels, 4 x 4, 512 samples
// 41 / 34 / 35 / 54.
constexpr int CONV_CHUNKS_MAX = 512;
int conv_chunk(int B) { return std::max(1, (B + CONV_CHUNKS_MAX - 1) / CONV_CHUNKS_MAX); }
}  // namespace

// Enough for every batch up to B, not only for B (513 samples make 257
// workgroups of two, 512 make 512 of one): a caller may keep the workspace of
// its largest batch.
int64_t conv_bwd_weight_workspace(int B, int cin, int cout) {
    const int chunks = std::max(0, std::min(B, CONV_CHUNKS_MAX));
    return int64_t(chunks) * (int64_t(cout) * cin * 9 + cout) * int64_t(sizeof(float));
}

void launch_conv_bwd_weight(const float* dy, const float* relu_y, const float* x, float* dw, float* db, int B, int cin,
                            int cout, int H, int W, float* workspace, hipStream_t st) {
    conv_check(cin, cout, H, W);
    if (B <= 0) return;
    if (size_t(cin * (H + 2) * (W + 2) + cout * H * W) * sizeof(float) > CONV_LDS_MAX)
        throw std::runtime_error("conv3x3: working set exceeds LDS");
    const int per = conv_chunk(B), chunks = (B + per - 1) / per;
    const int nw = cout * cin * 9;
    float* part = workspace;
    float* partb = workspace + int64_t(chunks) * nw;
    int S = plane_stride(H + 2, W + 2), G = plane_stride(H, W);
    auto bytes = [&] { return (size_t(cin) * S + size_t(cout) * G) * sizeof(float); };
    if (bytes() > CONV_LDS_MAX) {
        S = (H + 2) * (W + 2);
        G = H * W;
    }
    const size_t lds = bytes();
    const dim3 grid(static_cast<unsigned>(chunks));
    auto go = [&](auto kernel) {
        allow(reinterpret_cast<const void*>(kernel), lds);
        hipLaunchKernelGGL(kernel, grid, dim3(NT), lds, st, dy, relu_y, x, part, partb, B, per, cin, cout, H, W, S, G);
    };
    // column tiles per wave: ceil(ceil(9 cin / 16) / 4), 9 at 64 channels
    const int npw = ((cin * 9 + 15) / 16 + 3) / 4;
    auto pick = [&](auto mt) {
        constexpr int MT = decltype(mt)::value;
        if (npw <= 1)
            go(conv_bwd_weight_kernel<MT, 1>);
        else if (npw <= 3)
            go(conv_bwd_weight_kernel<MT, 3>);
        else if (npw <= 5)
            go(conv_bwd_weight_kernel<MT, 5>);
        else
            go(conv_bwd_weight_kernel<MT, 9>);
    };
    if (cout <= 16)
        pick(std::integral_constant<int, 1>());
    else if (cout <= 32)
        pick(std::integral_constant<int, 2>());
    else
        pick(std::integral_constant<int, 4>());
    check(hipGetLastError(), "conv backward-weight launch");
    hipLaunchKernelGGL(reduce_chunks_kernel, dim3(unsigned((nw + 63) / 64 + (cout + 63) / 64)), dim3(NT), 0, st, part,
                       partb, chunks, nw, cout, dw, db);
    check(hipGetLastError(), "conv gradient reduction launch");
}

void launch_hop(const float* logits, const int8_t* occ, const float* u, int32_t* hop, float* logq, int B, int H, int W,
                hipStream_t st) {
    if (B <= 0) return;
    if (H < 1 || W < 1 || H > 32 || W > 32) throw std::runtime_error("hop: lattice at most 32 x 32");
    hipLaunchKernelGGL(hop_kernel, dim3(unsigned(B)), dim3(64), 0, st, logits, occ, u, hop, logq, H, W);
    check(hipGetLastError(), "hop launch");
}

void launch_hop_regression(const float* logits, const int32_t* hop, const float* target, float* dlogits, float* loss,
                           int B, int n, hipStream_t st) {
    if (B <= 0) return;
    const int64_t total = int64_t(B) * n;
    hipLaunchKernelGGL(hop_regression_kernel, dim3(unsigned((total + 255) / 256)), dim3(256), 0, st, logits, hop, target,
                       dlogits, loss, B, n);
    check(hipGetLastError(), "hop regression launch");
}

void launch_adam(float* w, float* m, float* v, const float* g, uint16_t* wbf, int n, float lr, float b1, float b2,
                 float eps, int step, hipStream_t st) {
    if (n <= 0) return;
    const float c1 = 1.f - std::pow(b1, float(step)), c2 = 1.f - std::pow(b2, float(step));
    hipLaunchKernelGGL(adam_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, w, m, v, g, wbf, n, lr, b1, b2,
                       eps, c1, c2);
    check(hipGetLastError(), "adam launch");
}

void launch_to_bf16(const float* w, uint16_t* wbf, int n, hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(to_bf16_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, w, wbf, n);
    check(hipGetLastError(), "bf16 launch");
}

void launch_occ_to_input(const int8_t* occ, float* x, int64_t n, hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(occ_to_input_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, occ, x, n);
    check(hipGetLastError(), "input launch");
}

}  // namespace tns
