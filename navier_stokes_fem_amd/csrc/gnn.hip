// Learned warm start for the pressure CG: a 3-layer message-passing network
// over the pressure-matrix graph that maps the divergence right-hand side to
// an initial guess.  Forward and backward passes, the loss and an Adam step
// run here, on the GPU (the Adam step clips the gradient norm at 4 times its
// running average); CG still solves to the same tolerance afterwards, so
// a poor guess costs iterations, never accuracy.  (The reference has no
// learned component: the pressure solve is warm-started from the previous
// pressure, include/assembly.h:608-615.)
//
// Network (hidden width H = 32):
//   graph     w_ij = -A_ij / sqrt(A_ii A_jj), j != i (symmetric), a_i = node
//             area (lumped P1 mass), (X_i, Y_i) = coordinates scaled to the
//             unit box
//   input     d_i = b_i / a_i, s = sqrt(mean d^2), x0_i = [d_i/s, X_i, Y_i, 0]
//   layer l   m = W_hat h, z = [h | m] W_l + c_l, h' = relu(z)
//   readout   y_i = h3_i . w4 + c4, p_hat_i = s y_i
//   loss      sum (p_hat - p)^2 / sum p^2
// Storage: weights FP32 (master) with BF16 copies; [h | m] and dz in BF16 as
// MFMA operands; z, dX in FP32; v_mfma_f32_16x16x16_bf16 with FP32
// accumulation for every dense product (forward, dW = X^T dz, dX = dz W^T).
// Every reduction (sum of d^2, loss, dW, dc) uses per-block partials added
// in block order, so a given input gives bit-identical results run to run.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "nsfem_internal.hpp"

namespace nsfem {
namespace gnn {

constexpr int H = 32;
constexpr int K1 = 16;  // layer-1 operand width: x0 (4) | m0 (4) | zero padding
constexpr int K2 = 64;  // layers 2 and 3: h (32) | m (32)
constexpr int OFF_W1 = 0;                // [8][H]
constexpr int OFF_C1 = OFF_W1 + 8 * H;   // [H]
constexpr int OFF_W2 = OFF_C1 + H;       // [K2][H]
constexpr int OFF_C2 = OFF_W2 + K2 * H;
constexpr int OFF_W3 = OFF_C2 + H;       // [K2][H]
constexpr int OFF_C3 = OFF_W3 + K2 * H;
constexpr int OFF_W4 = OFF_C3 + H;       // [H]
constexpr int OFF_C4 = OFF_W4 + H;       // [1]
constexpr int NPARAM = OFF_C4 + 1;
constexpr int kRB = 256;  // threads per block of the elementwise kernels

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f) {  // round to nearest even
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint32_t b) { return __uint_as_float((b & 0xFFFFu) << 16); }

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// d = b / area
__global__ void k_ratio(int n, const double *__restrict__ b, const double *__restrict__ area,
                        double *__restrict__ d) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = b[i] / area[i];
}

// x0 = [d/s, X, Y, 0] into columns 0..3 of X1; columns 8..15 are padding
__global__ void k_input(int n, const double *__restrict__ d, const double *__restrict__ sumsq,
                        const float2 *__restrict__ xy, uint16_t *__restrict__ X1) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double s = sqrt(sumsq[0] / n) + 1e-30;
    const float2 c = xy[i];
    uint2 lo, hi;
    lo.x = (uint32_t)f2bf((float)(d[i] / s)) | ((uint32_t)f2bf(c.x) << 16);
    lo.y = (uint32_t)f2bf(c.y);
    hi.x = 0;
    hi.y = 0;
    uint2 *row = reinterpret_cast<uint2 *>(X1 + (size_t)i * K1);
    row[0] = lo;  // columns 0..3
    row[2] = hi;  // columns 8..11
    row[3] = hi;  // columns 12..15
}

// One layer: m_i = sum_j w_ij h_j (FP64 sums in CSR order, rounded to BF16),
// z = [h | m] W + c, h' = relu(z); a wave per 16 nodes, two 16x16 output
// tiles.  MFMA 16x16x16 operand layout: lane l holds A[l%16][4(l/16)+i],
// B[4(l/16)+i][l%16]; the result D[4(l/16)+j][l%16].  A lane so needs, of the
// aggregate, four columns (layer 1: the second lane group alone) or twice
// four of one node, and sums just those: the aggregate goes from registers
// into the product, and to memory (columns KS..2KS-1 of X, which nothing
// gathers) only for the backward pass, with z.  Bound by the gathers: the
// aggregation and the product apart were 9.3 and 10.9 us on the 65,656 nodes
// of the 512 x 128 channel and a launch gap (layer 1: 6.9 and 5.1), this is
// 19.3 (9.3).  Eight neighbours at a time take 21.6, as does a run of
// consecutive nodes per XCD.
template <int KP>
__global__ __launch_bounds__(kRB) void k_layer_fwd(int n, const int32_t *__restrict__ rs,
                                                   const int32_t *__restrict__ nbr,
                                                   const double *__restrict__ w, uint16_t *X,
                                                   const uint16_t *__restrict__ Wt,
                                                   const float *__restrict__ c,
                                                   float *__restrict__ z,
                                                   uint16_t *__restrict__ hout, int hstride) {
    constexpr int KS = KP == K1 ? 4 : KP / 2;  // columns of h
    constexpr int NG = KP == K1 ? 1 : 2;       // groups of four of them a lane sums
    constexpr int AHEAD = 4;                   // neighbours asked for at a time
    const int lane = threadIdx.x & 63;
    const int64_t r0 = ((blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6) * 16;
    if (r0 >= n) return;  // wave-uniform
    const int arow = (int)min((int64_t)n - 1, r0 + (lane & 15));
    const int kq = 4 * (lane >> 4);
    const int hq = KP == K1 ? 0 : kq;  // first column this lane sums
    const bool sums = KP != K1 || kq == KS;
    bf16x4 own[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g)
        own[g] = *reinterpret_cast<const bf16x4 *>(X + (size_t)arow * KP + 16 * g + kq);
    double a[NG][4];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int f = 0; f < 4; ++f) a[g][f] = 0.0;
    if (sums) {
        const int end = rs[arow + 1];
        for (int k = rs[arow]; k < end; k += AHEAD) {
            int jn[AHEAD];
            double wk[AHEAD];
            uint2 v[AHEAD][NG];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                const int ku = min(k + u, end - 1);
                jn[u] = nbr[ku];
                wk[u] = w[ku];
            }
#pragma unroll
            for (int u = 0; u < AHEAD; ++u)
#pragma unroll
                for (int g = 0; g < NG; ++g)
                    v[u][g] = *reinterpret_cast<const uint2 *>(X + (size_t)jn[u] * KP + 16 * g + hq);
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    if (k + u >= end) continue;
                    a[g][0] += wk[u] * (double)bf2f(v[u][g].x);
                    a[g][1] += wk[u] * (double)bf2f(v[u][g].x >> 16);
                    a[g][2] += wk[u] * (double)bf2f(v[u][g].y);
                    a[g][3] += wk[u] * (double)bf2f(v[u][g].y >> 16);
                }
            }
        }
    }
    bf16x4 m[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
#pragma unroll
        for (int f = 0; f < 4; ++f) m[g][f] = (short)f2bf((float)a[g][f]);
        if (z && sums && r0 + (lane & 15) < n)
            *reinterpret_cast<bf16x4 *>(X + (size_t)arow * KP + KS + 16 * g + hq) = m[g];
    }
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KP / 16; ++ks) {
        // layer 1 holds both halves in one operand
        const bf16x4 av = (KP == K1 ? kq == KS : ks >= NG) ? m[ks % NG] : own[ks % NG];
        const bf16x4 b0 =
            *reinterpret_cast<const bf16x4 *>(Wt + (size_t)(lane & 15) * KP + 16 * ks + kq);
        const bf16x4 b1 =
            *reinterpret_cast<const bf16x4 *>(Wt + (size_t)(16 + (lane & 15)) * KP + 16 * ks + kq);
        acc0 = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, b0, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, b1, acc1, 0, 0, 0);
    }
    const int col = lane & 15;
    const float c0 = c[col], c1 = c[col + 16];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t row = r0 + kq + j;
        if (row < n) {
            const float v0 = acc0[j] + c0, v1 = acc1[j] + c1;
            if (z) {
                z[row * H + col] = v0;
                z[row * H + col + 16] = v1;
            }
            hout[row * hstride + col] = f2bf(fmaxf(v0, 0.f));
            hout[row * hstride + col + 16] = f2bf(fmaxf(v1, 0.f));
        }
    }
}

// y = h3 . w4 + c4 (FP64 sum, rounded to FP32), p_hat = s y
__global__ void k_readout(int n, const uint16_t *__restrict__ h3, const float *__restrict__ prm,
                          const double *__restrict__ sumsq, double *__restrict__ p_hat) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double s = sqrt(sumsq[0] / n) + 1e-30;
    const uint4 *row = reinterpret_cast<const uint4 *>(h3 + (size_t)i * H);
    double acc = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint4 v = row[q];
        const uint32_t wv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc += (double)bf2f(wv[e]) * (double)prm[OFF_W4 + 8 * q + 2 * e];
            acc += (double)bf2f(wv[e] >> 16) * (double)prm[OFF_W4 + 8 * q + 2 * e + 1];
        }
    }
    const float y = (float)(acc + (double)prm[OFF_C4]);
    p_hat[i] = s * (double)y;
}

// block sum of K doubles into part[blockIdx.x * K + k]
template <int K>
__device__ void block_partial(double (&v)[K], double *part) {
    __shared__ double red[K][kRB / 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double s = wave_sum(v[k]);
        if (lane == 0) red[k][wv] = s;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < K; k += blockDim.x) {
        double s = 0.0;
        for (int w = 0; w < kRB / 64; ++w) s += red[k][w];
        part[(size_t)blockIdx.x * K + k] = s;
    }
}

// dy = 2 s (p_hat - p) / sum p^2 (FP32); partial sums of (p_hat - p)^2
__global__ __launch_bounds__(kRB) void k_loss(int n, const double *__restrict__ p_hat,
                                              const double *__restrict__ p,
                                              const double *__restrict__ scal,
                                              float *__restrict__ dy, double *__restrict__ part) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const double s = sqrt(scal[0] / n) + 1e-30;
    const double den = scal[1] + 1e-300;
    double v[1] = {0.0};
    if (i < n) {
        const double diff = p_hat[i] - p[i];
        v[0] = diff * diff;
        dy[i] = (float)(2.0 * s * diff / den);
    }
    block_partial<1>(v, part);
}

// dh3 = dy w4 (FP32), dz3 = bf16(dh3 [z3 > 0]); partials of h3 dy and dy.
// Bound by the loads of h3 and z3: 8 lanes a node, 4 features each (8-byte
// and 16-byte loads), a block striding over the nodes and summing its
// partials in registers, so that the lanes are added once a block.  One
// thread a node (2-byte loads and 33 sums over the wave per 64 nodes) took
// 34 us on the 65,656 nodes of the 512 x 128 channel; this takes 5.9.
__global__ __launch_bounds__(kRB) void k_readout_bwd(int n, const uint16_t *__restrict__ h3,
                                                     const float *__restrict__ dy,
                                                     const float *__restrict__ prm,
                                                     const float *__restrict__ z3,
                                                     uint16_t *__restrict__ dz3,
                                                     double *__restrict__ part) {
    constexpr int CH = H / 4, NW = kRB / 64;
    __shared__ double red[NW][H + 1];
    const int c = threadIdx.x % CH;
    double w4[4], v[4] = {0.0, 0.0, 0.0, 0.0}, vd = 0.0;
#pragma unroll
    for (int f = 0; f < 4; ++f) w4[f] = (double)prm[OFF_W4 + 4 * c + f];
    constexpr int NB = kRB / CH;  // nodes a block takes at a time
    for (int64_t i = blockIdx.x * (int64_t)NB + threadIdx.x / CH; i < n;
         i += (int64_t)gridDim.x * NB) {
        const float d = dy[i];
        const uint2 h = *reinterpret_cast<const uint2 *>(h3 + i * H + 4 * c);
        const float4 z = *reinterpret_cast<const float4 *>(z3 + i * H + 4 * c);
        const uint32_t hb[4] = {h.x, h.x >> 16, h.y, h.y >> 16};
        const float zz[4] = {z.x, z.y, z.z, z.w};
        uint16_t r[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            v[f] += (double)bf2f(hb[f]) * (double)d;
            const float dh = (float)((double)d * w4[f]);
            r[f] = zz[f] > 0.f ? f2bf(dh) : (uint16_t)0;
        }
        vd += (double)d;
        uint2 o;
        o.x = (uint32_t)r[0] | ((uint32_t)r[1] << 16);
        o.y = (uint32_t)r[2] | ((uint32_t)r[3] << 16);
        *reinterpret_cast<uint2 *>(dz3 + i * H + 4 * c) = o;
    }
    // lanes CH apart hold the same features
#pragma unroll
    for (int o = CH; o < 64; o *= 2) {
#pragma unroll
        for (int f = 0; f < 4; ++f) v[f] += __shfl_xor(v[f], o, 64);
        vd += __shfl_xor(vd, o, 64);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane < CH) {
#pragma unroll
        for (int f = 0; f < 4; ++f) red[wave][4 * c + f] = v[f];
        if (lane == 0) red[wave][H] = vd;
    }
    __syncthreads();
    if (threadIdx.x <= H) {
        double t = 0.0;
        for (int w = 0; w < NW; ++w) t += red[w][threadIdx.x];
        part[(size_t)blockIdx.x * (H + 1) + threadIdx.x] = t;
    }
}

// Partials of dW = X^T dz ([KP][H]) and dc = sum dz ([H]) per block of nbw:
// part[block][KP * H + H].  Waves stride over 16-node groups; rows past n
// contribute zeros.
template <int KP>
__device__ __forceinline__ void dense_bwd_w(int n, int block, int nbw,
                                            const uint16_t *__restrict__ X,
                                            const uint16_t *__restrict__ dz,
                                            double *__restrict__ part) {
    constexpr int MT = KP / 16;
    constexpr int NW = kRB / 64;
    __shared__ float lds[NW][KP * H];
    __shared__ float ldc[NW][H];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15;
    f32x4 acc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float dc0 = 0.f, dc1 = 0.f;
    const int64_t groups = ((int64_t)n + 15) / 16;
    for (int64_t g = (int64_t)block * NW + wave; g < groups; g += (int64_t)nbw * NW) {
        const int64_t base = g * 16 + 4 * (lane >> 4);
        bf16x4 b0, b1;
        int64_t nodec[4];
        bool ok[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            ok[i] = base + i < n;
            nodec[i] = ok[i] ? base + i : (int64_t)n - 1;
            const uint16_t v0 = dz[nodec[i] * H + col];
            const uint16_t v1 = dz[nodec[i] * H + 16 + col];
            b0[i] = ok[i] ? (short)v0 : (short)0;
            b1[i] = ok[i] ? (short)v1 : (short)0;
            dc0 += ok[i] ? bf2f(v0) : 0.f;
            dc1 += ok[i] ? bf2f(v1) : 0.f;
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            bf16x4 a;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint16_t xv = X[nodec[i] * KP + 16 * mt + col];
                a[i] = ok[i] ? (short)xv : (short)0;
            }
            acc[mt][0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b0, acc[mt][0], 0, 0, 0);
            acc[mt][1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b1, acc[mt][1], 0, 0, 0);
        }
    }
    // lanes l, l+16, l+32, l+48 hold the same columns
    dc0 += __shfl_xor(dc0, 16, 64);
    dc0 += __shfl_xor(dc0, 32, 64);
    dc1 += __shfl_xor(dc1, 16, 64);
    dc1 += __shfl_xor(dc1, 32, 64);
    const int kq = 4 * (lane >> 4);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int j = 0; j < 4; ++j) lds[wave][(16 * mt + kq + j) * H + 16 * nt + col] = acc[mt][nt][j];
    if (lane < 16) {
        ldc[wave][col] = dc0;
        ldc[wave][col + 16] = dc1;
    }
    __syncthreads();
    double *out = part + (size_t)block * (KP * H + H);
    for (int e = threadIdx.x; e < KP * H + H; e += blockDim.x) {
        double s = 0.0;
        for (int w = 0; w < NW; ++w) s += e < KP * H ? (double)lds[w][e] : (double)ldc[w][e - KP * H];
        out[e] = s;
    }
}

// dX = dz W^T: one wave per 16 rows, KP/16 output tiles, K = H
template <int KP>
__device__ __forceinline__ void dense_bwd_x(int n, int block, const uint16_t *__restrict__ dz,
                                            const uint16_t *__restrict__ Wr,
                                            float *__restrict__ dX) {
    constexpr int NT = KP / 16;
    const int lane = threadIdx.x & 63;
    const int64_t r0 = ((block * (int64_t)blockDim.x + threadIdx.x) >> 6) * 16;
    if (r0 >= n) return;
    const int arow = (int)min((int64_t)n - 1, r0 + (lane & 15));
    const int kq = 4 * (lane >> 4);
    const int col = lane & 15;
    f32x4 acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < H / 16; ++ks) {
        const bf16x4 a = *reinterpret_cast<const bf16x4 *>(dz + (size_t)arow * H + 16 * ks + kq);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const bf16x4 b =
                *reinterpret_cast<const bf16x4 *>(Wr + (size_t)(16 * nt + col) * H + 16 * ks + kq);
            acc[nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[nt], 0, 0, 0);
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t row = r0 + kq + j;
        if (row < n) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) dX[row * KP + 16 * nt + col] = acc[nt][j];
        }
    }
}

// Sums of per-block partials part[b][e], b < nb, e < count (FP64): a block
// takes kRedCols columns e, kRedSegs threads a column, each adding one
// contiguous run of b in order; the runs are then added in order, so the sum
// has one fixed order for a given nb.  The reads of a run are independent of
// each other and kRedCols consecutive doubles (a 128-byte line) wide; one
// thread a column, with its chain of nb dependent adds behind nb far-apart
// loads, took 60-65 us for the 256 x 2,080 partials of a layer and 39 us
// for 257 x 33, this 3.4 us each.
constexpr int kRedCols = 16;
constexpr int kRedSegs = kRB / kRedCols;

__device__ __forceinline__ double sum_partials(int nb, int count, int e,
                                               const double *__restrict__ part) {
    __shared__ double seg[kRedSegs][kRedCols];
    const int c = threadIdx.x % kRedCols, g = threadIdx.x / kRedCols;
    const int lo = (int)((int64_t)nb * g / kRedSegs), hi = (int)((int64_t)nb * (g + 1) / kRedSegs);
    double s = 0.0;
    if (e < count) {
#pragma unroll 8
        for (int b = lo; b < hi; ++b) s += part[(size_t)b * count + e];
    }
    seg[g][c] = s;
    __syncthreads();
    s = 0.0;
    if (g == 0) {
#pragma unroll
        for (int k = 0; k < kRedSegs; ++k) s += seg[k][c];
    }
    return s;  // whole in the threads with g == 0
}

// A sum of partials: out[e] = sum_b part[b][e] in FP32 and / or FP64 for
// e < keep, tail[e - split] for the columns from `split` on (a dense layer:
// the real rows of dW, then dc).
struct Reduction {
    int nb = 0, count = 0, keep = 0, split = 0;
    const double *part = nullptr;
    float *out = nullptr, *tail = nullptr;
    double *out64 = nullptr;
    int blocks() const { return (count + kRedCols - 1) / kRedCols; }
};

__device__ __forceinline__ void reduce_block(const Reduction &r, int block) {
    const int e = block * kRedCols + threadIdx.x % kRedCols;
    const double s = sum_partials(r.nb, r.count, e, r.part);
    if (threadIdx.x >= kRedCols || e >= r.count) return;
    if (e >= r.split) {
        r.tail[e - r.split] = (float)s;
    } else if (e < r.keep) {
        if (r.out) r.out[e] = (float)s;
        if (r.out64) r.out64[e] = s;
    }
}

// The sums that wait when a layer's dX is aggregated, in that launch's first
// blocks: they read what the launches before it wrote and nothing in it
// reads them.
constexpr int kReductions = 3;
struct Reductions {
    Reduction r[kReductions];
    int blocks = 0;
    void add(const Reduction &x) {
        for (Reduction &slot : r)
            if (slot.count == 0) {
                slot = x;
                blocks += x.blocks();
                return;
            }
    }
};

__device__ __forceinline__ void reduce_blocks(const Reductions &R, int block) {
#pragma unroll
    for (int k = 0; k < kReductions; ++k) {
        const int nb = (R.r[k].count + kRedCols - 1) / kRedCols;
        if (block < nb) {  // block-uniform
            reduce_block(R.r[k], block);
            return;
        }
        block -= nb;
    }
}

__global__ __launch_bounds__(kRB) void k_reduce(Reductions R) {
    reduce_blocks(R, blockIdx.x);
}

// dh = dX[:, :H] + W_hat dX[:, H:] (FP64 sums in CSR order, rounded to FP32),
// dz_prev = bf16(dh [z_prev > 0]); one thread per (node, 4 features)
__device__ __forceinline__ void agg_bwd(int n, int block, const int32_t *__restrict__ rs,
                                        const int32_t *__restrict__ col,
                                        const double *__restrict__ w,
                                        const float *__restrict__ dX,
                                        const float *__restrict__ zp,
                                        uint16_t *__restrict__ dzp) {
    constexpr int CH = H / 4;
    const int64_t t = block * (int64_t)blockDim.x + threadIdx.x;
    if (t >= (int64_t)n * CH) return;
    const int i = (int)(t / CH), c = (int)(t % CH);
    double a[4] = {0, 0, 0, 0};
    for (int k = rs[i]; k < rs[i + 1]; ++k) {
        const int j = col[k];
        const double wk = w[k];
        const float4 v = *reinterpret_cast<const float4 *>(dX + (size_t)j * K2 + H + 4 * c);
        a[0] += wk * (double)v.x;
        a[1] += wk * (double)v.y;
        a[2] += wk * (double)v.z;
        a[3] += wk * (double)v.w;
    }
    const float4 own = *reinterpret_cast<const float4 *>(dX + (size_t)i * K2 + 4 * c);
    const float4 z = *reinterpret_cast<const float4 *>(zp + (size_t)i * H + 4 * c);
    const float dh[4] = {(float)((double)own.x + a[0]), (float)((double)own.y + a[1]),
                         (float)((double)own.z + a[2]), (float)((double)own.w + a[3])};
    const float zz[4] = {z.x, z.y, z.z, z.w};
    uint2 o;
    uint16_t r[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) r[f] = zz[f] > 0.f ? f2bf(dh[f]) : (uint16_t)0;
    o.x = (uint32_t)r[0] | ((uint32_t)r[1] << 16);
    o.y = (uint32_t)r[2] | ((uint32_t)r[3] << 16);
    *reinterpret_cast<uint2 *>(dzp + (size_t)i * H + 4 * c) = o;
}

// A layer's weight gradient (first nbw blocks) and input gradient: two
// independent passes over dz, of 6.7 and 9.1 us each by itself on the 65,656
// nodes of the 512 x 128 channel, 9.6 us together.
template <int KP>
__global__ __launch_bounds__(kRB) void k_layer_bwd(int n, int nbw, const uint16_t *__restrict__ X,
                                                   const uint16_t *__restrict__ dz,
                                                   const uint16_t *__restrict__ Wr,
                                                   double *__restrict__ part,
                                                   float *__restrict__ dX) {
    if ((int)blockIdx.x < nbw) dense_bwd_w<KP>(n, blockIdx.x, nbw, X, dz, part);
    else dense_bwd_x<KP>(n, blockIdx.x - nbw, dz, Wr, dX);
}

// the first layer has no input gradient
template <int KP>
__global__ __launch_bounds__(kRB) void k_layer_bwd_w(int n, const uint16_t *__restrict__ X,
                                                     const uint16_t *__restrict__ dz,
                                                     double *__restrict__ part) {
    dense_bwd_w<KP>(n, blockIdx.x, gridDim.x, X, dz, part);
}

// The waiting sums and the gradient of the layer before
__global__ __launch_bounds__(kRB) void k_agg_bwd(Reductions R, int n,
                                                 const int32_t *__restrict__ rs,
                                                 const int32_t *__restrict__ col,
                                                 const double *__restrict__ w,
                                                 const float *__restrict__ dX,
                                                 const float *__restrict__ zp,
                                                 uint16_t *__restrict__ dzp) {
    if ((int)blockIdx.x < R.blocks) reduce_blocks(R, blockIdx.x);
    else agg_bwd(n, blockIdx.x - R.blocks, rs, col, w, dX, zp, dzp);
}

// Gradient-norm clipping, one block: |g| against a running average of the
// norms of earlier steps (clip[0]); the gradient is scaled by
// clip[1] = min(1, kClipRatio * average / |g|) before the Adam update, so a
// pair whose relative loss is far above the rest (a target that is nearly
// zero against its input scale) moves the weights no more than an ordinary
// pair.  The average starts at the first step's norm and follows the clipped
// norms with decay kClipDecay.
constexpr float kClipRatio = 4.f;
constexpr float kClipDecay = 0.95f;

__global__ __launch_bounds__(kRB) void k_clip(int count, const float *__restrict__ g,
                                              float *__restrict__ clip) {
    double v[1] = {0.0};
#pragma unroll 6
    for (int k = threadIdx.x; k < count; k += kRB) v[0] += (double)g[k] * (double)g[k];
    __shared__ double total;
    double *part = &total;
    block_partial<1>(v, part);
    __syncthreads();
    if (threadIdx.x != 0) return;
    const float norm = (float)sqrt(total);
    float avg = clip[0];
    if (!(avg > 0.f)) avg = norm;
    const float limit = kClipRatio * avg;
    const float f = norm > limit ? limit / norm : 1.f;
    clip[0] = kClipDecay * avg + (1.f - kClipDecay) * fminf(norm, limit);
    clip[1] = f;
}

// BF16 copies of the weights: Wt[o][k] (forward operand, k padded to the
// MFMA's 16 with zeros) and Wr[k][o] (dX operand)
struct Packed {
    uint16_t *wt1, *wt2, *wr2, *wt3, *wr3;
    __device__ __forceinline__ void put(int e, float w) const {  // parameter e
        const uint16_t b = f2bf(w);
        if (e < OFF_C1) {
            wt1[(e % H) * K1 + e / H] = b;
        } else if (e >= OFF_W2 && e < OFF_C2) {
            const int k = e - OFF_W2;
            wt2[(k % H) * K2 + k / H] = b;
            wr2[k] = b;
        } else if (e >= OFF_W3 && e < OFF_C3) {
            const int k = e - OFF_W3;
            wt3[(k % H) * K2 + k / H] = b;
            wr3[k] = b;
        }
    }
};

__global__ void k_adam(int count, float *__restrict__ w, const float *__restrict__ g,
                       const float *__restrict__ clip, float *__restrict__ m,
                       float *__restrict__ v, float lr, float b1, float b2, float eps, float bc1,
                       float bc2, Packed pk) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= count) return;
    const float gk = g[k] * clip[1];
    const float mk = b1 * m[k] + (1.f - b1) * gk;
    const float vk = b2 * v[k] + (1.f - b2) * gk * gk;
    m[k] = mk;
    v[k] = vk;
    const float wk = w[k] - lr * (mk / bc1) / (sqrtf(vk / bc2) + eps);
    w[k] = wk;
    pk.put(k, wk);
}

__global__ void k_pack(int count, const float *__restrict__ w, Packed pk) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < count) pk.put(k, w[k]);
}

// copy src into dst where ||b - A src|| < ||b - A dst||: scal[0] = the
// squared residual of dst, scal[1] that of src
__global__ void k_select(int n, const double *__restrict__ scal, const double *__restrict__ src,
                         double *__restrict__ dst) {
    if (!(scal[1] < scal[0])) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// x += c d with c = scal[0] / scal[1] = (d . r) / (d . A d), the step along
// d that minimises the A-norm error of x (r = b - A x); no step unless
// d . A d > 0 and c is finite
__global__ void k_line_step(int n, const double *__restrict__ scal, const double *__restrict__ dir,
                            double *__restrict__ x) {
    const double den = scal[1], c = scal[0] / den;
    if (!(den > 0.0) || !(c == c) || c - c != 0.0) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = __builtin_fma(c, dir[i], x[i]);
}

inline int blocks_for(int64_t work, int bs = kRB) { return (int)((work + bs - 1) / bs); }

}  // namespace gnn

// ------------------------------------------------------------------- host
namespace {

gnn::Packed packed(GnnNet &g) {
    return {g.wt1.ptr, g.wt2.ptr, g.wr2.ptr, g.wt3.ptr, g.wr3.ptr};
}

void gnn_pack(GnnNet &g) {
    Device &d = *g.dev;
    gnn::k_pack<<<gnn::blocks_for(gnn::NPARAM), gnn::kRB, 0, d.stream>>>(gnn::NPARAM, g.params.ptr,
                                                                        packed(g));
    NSFEM_HIP(hipGetLastError());
}

// Blocks of k_readout_bwd: 32 nodes each at a time, two blocks a CU at most.
int readout_blocks(int n) { return std::min(512, gnn::blocks_for(n, gnn::kRB * 4 / gnn::H)); }

void gnn_reserve(GnnNet &g, int n) {
    if (n <= g.cap) return;
    using namespace gnn;
    g.X1.resize((size_t)n * K1);
    g.X2.resize((size_t)n * K2);
    g.X3.resize((size_t)n * K2);
    g.h3.resize((size_t)n * H);
    g.dz.resize((size_t)n * H);
    g.z1.resize((size_t)n * H);
    g.z2.resize((size_t)n * H);
    g.z3.resize((size_t)n * H);
    g.dX.resize((size_t)n * K2);
    g.dy.resize(n);
    g.d.resize(n);
    g.phat.resize(n);
    const size_t nb = (size_t)blocks_for(n);
    const size_t groups = ((size_t)n + 15) / 16;
    const size_t nbw = std::max<size_t>(1, std::min<size_t>(256, (groups + 3) / 4));
    const size_t nbr = (size_t)readout_blocks(n);
    // a layer's, the loss's and the readout's, which are added together
    g.part.resize(nbw * (K2 * H + H) + nb + nbr * (H + 1));
    g.cap = n;
}

int bwd_w_blocks(int n) {
    const int64_t groups = ((int64_t)n + 15) / 16;
    return (int)std::max<int64_t>(1, std::min<int64_t>(256, (groups + 3) / 4));
}

// forward pass; stores z for the backward pass when `train`.  p_hat ==
// nullptr writes the prediction to the workspace (g.phat), resolved after
// the workspace has been sized: a pointer taken before gnn_reserve may be
// null or freed.
void gnn_forward(GnnNet &g, GnnGraph &gr, const double *b, double *p_hat, bool train) {
    using namespace gnn;
    Device &d = *g.dev;
    const int n = gr.n;
    gnn_reserve(g, n);
    if (!p_hat) p_hat = g.phat.ptr;
    const int nb = blocks_for(n);
    g.scal.ensure(4);
    launch_fill(d, 4, 0.0, g.scal.ptr);
    k_ratio<<<nb, kRB, 0, d.stream>>>(n, b, gr.area.ptr, g.d.ptr);
    launch_dot_accumulate(d, n, g.d.ptr, g.d.ptr, g.scal.ptr);
    k_input<<<nb, kRB, 0, d.stream>>>(n, g.d.ptr, g.scal.ptr, gr.xy.ptr, g.X1.ptr);
    const int nbt = blocks_for(((int64_t)n + 15) / 16 * 64);  // one wave per 16 rows
    k_layer_fwd<K1><<<nbt, kRB, 0, d.stream>>>(n, gr.rs.ptr, gr.col.ptr, gr.w.ptr, g.X1.ptr,
                                              g.wt1.ptr, g.params.ptr + OFF_C1,
                                              train ? g.z1.ptr : nullptr, g.X2.ptr, K2);
    k_layer_fwd<K2><<<nbt, kRB, 0, d.stream>>>(n, gr.rs.ptr, gr.col.ptr, gr.w.ptr, g.X2.ptr,
                                              g.wt2.ptr, g.params.ptr + OFF_C2,
                                              train ? g.z2.ptr : nullptr, g.X3.ptr, K2);
    k_layer_fwd<K2><<<nbt, kRB, 0, d.stream>>>(n, gr.rs.ptr, gr.col.ptr, gr.w.ptr, g.X3.ptr,
                                              g.wt3.ptr, g.params.ptr + OFF_C3,
                                              train ? g.z3.ptr : nullptr, g.h3.ptr, H);
    k_readout<<<nb, kRB, 0, d.stream>>>(n, g.h3.ptr, g.params.ptr, g.scal.ptr, p_hat);
    NSFEM_HIP(hipGetLastError());
}

// forward + loss + backward into g.grads; the loss lands in scal[2]
void gnn_backward(GnnNet &g, GnnGraph &gr, const double *b, const double *p) {
    using namespace gnn;
    Device &d = *g.dev;
    const int n = gr.n;
    gnn_forward(g, gr, b, nullptr, true);  // prediction into g.phat
    const int nb = blocks_for(n);
    launch_dot_accumulate(d, n, p, p, g.scal.ptr + 1);
    const int nbr = readout_blocks(n), nbw = bwd_w_blocks(n);
    const int nbt = blocks_for(((int64_t)n + 15) / 16 * 64);
    const int nba = blocks_for((int64_t)n * (H / 4));
    double *part = g.part.ptr, *part_loss = part + (size_t)nbw * (K2 * H + H),
           *part_readout = part_loss + nb;
    Reductions sums;
    k_loss<<<nb, kRB, 0, d.stream>>>(n, g.phat.ptr, p, g.scal.ptr, g.dy.ptr, part_loss);
    sums.add({nb, 1, 1, 1, part_loss, nullptr, nullptr, g.scal.ptr + 2});
    k_readout_bwd<<<nbr, kRB, 0, d.stream>>>(n, g.h3.ptr, g.dy.ptr, g.params.ptr, g.z3.ptr,
                                             g.dz.ptr, part_readout);
    sums.add({nbr, H + 1, H + 1, H + 1, part_readout, g.grads.ptr + OFF_W4, nullptr, nullptr});
    // layer 3
    k_layer_bwd<K2><<<nbw + nbt, kRB, 0, d.stream>>>(n, nbw, g.X3.ptr, g.dz.ptr, g.wr3.ptr, part,
                                                    g.dX.ptr);
    sums.add({nbw, K2 * H + H, K2 * H, K2 * H, part, g.grads.ptr + OFF_W3, g.grads.ptr + OFF_C3,
              nullptr});
    k_agg_bwd<<<sums.blocks + nba, kRB, 0, d.stream>>>(sums, n, gr.rs.ptr, gr.col.ptr, gr.w.ptr,
                                                       g.dX.ptr, g.z2.ptr, g.dz.ptr);
    // layer 2
    k_layer_bwd<K2><<<nbw + nbt, kRB, 0, d.stream>>>(n, nbw, g.X2.ptr, g.dz.ptr, g.wr2.ptr, part,
                                                    g.dX.ptr);
    sums = {};
    sums.add({nbw, K2 * H + H, K2 * H, K2 * H, part, g.grads.ptr + OFF_W2, g.grads.ptr + OFF_C2,
              nullptr});
    k_agg_bwd<<<sums.blocks + nba, kRB, 0, d.stream>>>(sums, n, gr.rs.ptr, gr.col.ptr, gr.w.ptr,
                                                       g.dX.ptr, g.z1.ptr, g.dz.ptr);
    // layer 1 (8 real input rows of the 16-row padded operand)
    k_layer_bwd_w<K1><<<nbw, kRB, 0, d.stream>>>(n, g.X1.ptr, g.dz.ptr, part);
    sums = {};
    sums.add({nbw, K1 * H + H, 8 * H, K1 * H, part, g.grads.ptr + OFF_W1, g.grads.ptr + OFF_C1,
              nullptr});
    k_reduce<<<sums.blocks, kRB, 0, d.stream>>>(sums);
    NSFEM_HIP(hipGetLastError());
}

}  // namespace

GnnNet *gnn_create(Device &d, uint64_t seed) {
    using namespace gnn;
    auto *g = new GnnNet();
    g->dev = &d;
    d.set_current();
    std::vector<float> h(NPARAM, 0.f);
    std::mt19937_64 rng(seed);
    std::normal_distribution<double> nd(0.0, 1.0);
    auto fill = [&](int off, int rows, int cols) {
        const double sc = std::sqrt(2.0 / rows);
        for (int e = 0; e < rows * cols; ++e) h[off + e] = (float)(nd(rng) * sc);
    };
    fill(OFF_W1, 8, H);
    fill(OFF_W2, K2, H);
    fill(OFF_W3, K2, H);
    // the readout starts at zero: an untrained network predicts 0 (loss 1),
    // and training only moves it from there
    for (int e = 0; e < H; ++e) h[OFF_W4 + e] = 0.f;
    g->params.resize(NPARAM);
    g->grads.resize(NPARAM);
    g->m.resize(NPARAM);
    g->v.resize(NPARAM);
    g->clip.resize(2);
    g->wt1.resize(H * K1);
    g->wt2.resize(H * K2);
    g->wr2.resize(H * K2);
    g->wt3.resize(H * K2);
    g->wr3.resize(H * K2);
    NSFEM_HIP(hipMemcpy(g->params.ptr, h.data(), NPARAM * sizeof(float), hipMemcpyHostToDevice));
    // (cleared on the stream that packs and trains: it does not wait for the
    // null stream, and a late clear of wt1 would wipe the packed weights)
    NSFEM_HIP(hipMemsetAsync(g->grads.ptr, 0, NPARAM * sizeof(float), d.stream));
    NSFEM_HIP(hipMemsetAsync(g->m.ptr, 0, NPARAM * sizeof(float), d.stream));
    NSFEM_HIP(hipMemsetAsync(g->v.ptr, 0, NPARAM * sizeof(float), d.stream));
    NSFEM_HIP(hipMemsetAsync(g->clip.ptr, 0, 2 * sizeof(float), d.stream));
    NSFEM_HIP(hipMemsetAsync(g->wt1.ptr, 0, H * K1 * sizeof(uint16_t), d.stream));  // the padding
    gnn_pack(*g);
    NSFEM_HIP(hipStreamSynchronize(d.stream));
    return g;
}

void gnn_set_params(GnnNet &g, const float *h) {
    using namespace gnn;
    Device &d = *g.dev;
    d.set_current();
    NSFEM_HIP(hipMemcpyAsync(g.params.ptr, h, NPARAM * sizeof(float), hipMemcpyHostToDevice,
                             d.stream));
    NSFEM_HIP(hipMemsetAsync(g.m.ptr, 0, NPARAM * sizeof(float), d.stream));
    NSFEM_HIP(hipMemsetAsync(g.v.ptr, 0, NPARAM * sizeof(float), d.stream));
    NSFEM_HIP(hipMemsetAsync(g.clip.ptr, 0, 2 * sizeof(float), d.stream));
    g.adam_t = 0;
    gnn_pack(g);
    NSFEM_HIP(hipStreamSynchronize(d.stream));
}

void gnn_get(GnnNet &g, const float *src, float *h) {
    Device &d = *g.dev;
    d.set_current();
    NSFEM_HIP(hipMemcpyAsync(h, src, gnn::NPARAM * sizeof(float), hipMemcpyDeviceToHost, d.stream));
    NSFEM_HIP(hipStreamSynchronize(d.stream));
}

// Graph of a pressure matrix: CSR without the diagonal, symmetric weights.
GnnGraph *gnn_graph_create(Device &d, int n, int64_t nnz, const int32_t *rs, const int32_t *col,
                           const double *val, const double *area, const float *xy) {
    NSFEM_REQUIRE(n > 0 && rs && col && val && area && xy, NSFEM_INVALID_ARGUMENT,
                  "gnn graph: empty or null input");
    NSFEM_REQUIRE(rs[0] == 0 && rs[n] == nnz, NSFEM_INVALID_ARGUMENT, "gnn graph: bad row_start");
    std::vector<double> diag(n, 0.0);
    for (int i = 0; i < n; ++i) {
        NSFEM_REQUIRE(rs[i + 1] >= rs[i], NSFEM_INVALID_ARGUMENT, "gnn graph: bad row_start");
        for (int k = rs[i]; k < rs[i + 1]; ++k) {
            NSFEM_REQUIRE(col[k] >= 0 && col[k] < n, NSFEM_INVALID_ARGUMENT,
                          "gnn graph: matrix must be square, column out of range");
            if (col[k] == i) diag[i] = val[k];
        }
        NSFEM_REQUIRE(diag[i] > 0 && area[i] > 0, NSFEM_INVALID_ARGUMENT,
                      "gnn graph: every row needs a positive diagonal and a positive area");
    }
    std::vector<int32_t> grs(n + 1, 0), gcol;
    std::vector<double> gw;
    gcol.reserve(nnz);
    gw.reserve(nnz);
    for (int i = 0; i < n; ++i) {
        for (int k = rs[i]; k < rs[i + 1]; ++k) {
            if (col[k] == i) continue;
            gcol.push_back(col[k]);
            gw.push_back(-val[k] / std::sqrt(diag[i] * diag[col[k]]));
        }
        grs[i + 1] = (int32_t)gcol.size();
    }
    double lo[2] = {1e300, 1e300}, hi[2] = {-1e300, -1e300};
    for (int i = 0; i < n; ++i)
        for (int a = 0; a < 2; ++a) {
            lo[a] = std::min(lo[a], (double)xy[2 * i + a]);
            hi[a] = std::max(hi[a], (double)xy[2 * i + a]);
        }
    const double ext = std::max(std::max(hi[0] - lo[0], hi[1] - lo[1]), 1e-30);
    std::vector<float2> nx(n);
    for (int i = 0; i < n; ++i)
        nx[i] = make_float2((float)(((double)xy[2 * i] - lo[0]) / ext),
                            (float)(((double)xy[2 * i + 1] - lo[1]) / ext));
    auto *g = new GnnGraph();
    g->dev = &d;
    g->n = n;
    g->ne = (int64_t)gcol.size();
    d.set_current();
    g->rs.resize(n + 1);
    g->col.resize(std::max<size_t>(1, gcol.size()));
    g->w.resize(std::max<size_t>(1, gw.size()));
    g->area.resize(n);
    g->xy.resize(n);
    NSFEM_HIP(hipMemcpy(g->rs.ptr, grs.data(), (n + 1) * sizeof(int32_t), hipMemcpyHostToDevice));
    if (!gcol.empty()) {
        NSFEM_HIP(hipMemcpy(g->col.ptr, gcol.data(), gcol.size() * sizeof(int32_t),
                            hipMemcpyHostToDevice));
        NSFEM_HIP(hipMemcpy(g->w.ptr, gw.data(), gw.size() * sizeof(double), hipMemcpyHostToDevice));
    }
    NSFEM_HIP(hipMemcpy(g->area.ptr, area, n * sizeof(double), hipMemcpyHostToDevice));
    NSFEM_HIP(hipMemcpy(g->xy.ptr, nx.data(), n * sizeof(float2), hipMemcpyHostToDevice));
    return g;
}

void gnn_predict(GnnNet &g, GnnGraph &gr, const double *b, double *p_hat) {
    g.dev->set_current();
    gnn_forward(g, gr, b, p_hat, false);
}

// gradients (device) and the loss; host copies when requested
void gnn_gradients(GnnNet &g, GnnGraph &gr, const double *b, const double *p, float *host_grads,
                   double *loss) {
    Device &d = *g.dev;
    d.set_current();
    gnn_backward(g, gr, b, p);
    if (host_grads)
        NSFEM_HIP(hipMemcpyAsync(host_grads, g.grads.ptr, gnn::NPARAM * sizeof(float),
                                 hipMemcpyDeviceToHost, d.stream));
    double h[3] = {0, 0, 0};
    if (loss)
        NSFEM_HIP(hipMemcpyAsync(h, g.scal.ptr, 3 * sizeof(double), hipMemcpyDeviceToHost, d.stream));
    NSFEM_HIP(hipStreamSynchronize(d.stream));
    if (loss) *loss = h[2] / (h[1] + 1e-300);
}

void gnn_train_step(GnnNet &g, GnnGraph &gr, const double *b, const double *p, float lr,
                    double *loss) {
    Device &d = *g.dev;
    d.set_current();
    gnn_backward(g, gr, b, p);
    ++g.adam_t;
    const float b1 = 0.9f, b2 = 0.999f;
    const float bc1 = 1.f - std::pow(b1, (float)g.adam_t), bc2 = 1.f - std::pow(b2, (float)g.adam_t);
    gnn::k_clip<<<1, gnn::kRB, 0, d.stream>>>(gnn::NPARAM, g.grads.ptr, g.clip.ptr);
    gnn::k_adam<<<gnn::blocks_for(gnn::NPARAM), gnn::kRB, 0, d.stream>>>(
        gnn::NPARAM, g.params.ptr, g.grads.ptr, g.clip.ptr, g.m.ptr, g.v.ptr, lr, b1, b2, 1e-8f,
        bc1, bc2, packed(g));
    NSFEM_HIP(hipGetLastError());
    if (loss) {
        double h[3];
        NSFEM_HIP(hipMemcpyAsync(h, g.scal.ptr, 3 * sizeof(double), hipMemcpyDeviceToHost, d.stream));
        NSFEM_HIP(hipStreamSynchronize(d.stream));
        *loss = h[2] / (h[1] + 1e-300);
    }
}

// dst = src where src has the smaller residual ||b - A x|| (device-side,
// no host synchronisation); tmp: n doubles of scratch
void select_better_guess(Device &d, Matrix &A, const double *b, const double *src, double *dst,
                         double *tmp, double *scal2) {
    const int n = A.rows;
    launch_fill(d, 2, 0.0, scal2);
    launch_spmv(d, A, dst, b, tmp, 1);
    launch_dot_accumulate(d, n, tmp, tmp, scal2);
    launch_spmv(d, A, src, b, tmp, 1);
    launch_dot_accumulate(d, n, tmp, tmp, scal2 + 1);
    gnn::k_select<<<gnn::blocks_for(n), gnn::kRB, 0, d.stream>>>(n, scal2, src, dst);
    NSFEM_HIP(hipGetLastError());
}

// x += c d, c the A-norm-optimal step along d from x (r = b - A x on entry;
// no host sync); w: n doubles of scratch (receives A d), scal2: 2 doubles
void line_search_step(Device &d, Matrix &A, const double *r, const double *dir, double *x,
                      double *w, double *scal2) {
    const int n = A.rows;
    launch_fill(d, 2, 0.0, scal2);
    launch_spmv(d, A, dir, nullptr, w, 0);
    launch_dot_accumulate(d, n, dir, r, scal2);
    launch_dot_accumulate(d, n, dir, w, scal2 + 1);
    gnn::k_line_step<<<gnn::blocks_for(n), gnn::kRB, 0, d.stream>>>(n, scal2, dir, x);
    NSFEM_HIP(hipGetLastError());
}

}  // namespace nsfem
