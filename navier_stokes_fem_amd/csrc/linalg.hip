// CSR products, BLAS-1 and the persistent conjugate-gradient kernel for
// gfx950.  Replaces gpu/matrix_math.cu of the reference (spRMult :19-51,
// spRMultSub :66-99, saxpy :106-122, saxpby :131-155, dotProduct :162-194,
// GridSync :209-249, conjugateGradientMegakernel :251-287) and the host
// orchestration of cpp/gpu_simulation_device.cpp:142-515.
//
// Layout in HBM: the reference CSR (int32 row_start[n+1], int32 col[nnz]
// ascending per row, values[nnz]) plus a tile table cutting the rows into
// runs of <= kTileRows rows and <= kTileNnz nonzeros.  A tile is staged
// through LDS: one coalesced pass over col/val computes every product
// val*x[col] into LDS, then one thread per row adds its products in row
// order.  That keeps the column and value streams fully coalesced for the
// 7 (P1) to 19 (P2) nonzeros per row of these matrices, and it adds the
// products of a row in the same order as the reference's row loop.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <type_traits>

#include "nsfem_internal.hpp"

namespace nsfem {

// ----------------------------------------------------------------- helpers
namespace {

constexpr int kWaves = kBlock / 64;
// The product loads a tile's columns and values in groups of 4 nonzeros
// starting at a multiple of 4 (16-byte column and 2 x 16-byte value loads
// per lane); tiles hold at most kTileNnz - 3 nonzeros so that the aligned
// span of any tile fits kTileNnz products, kGroups groups per thread.
constexpr int kSpmvTileNnz = kTileNnz - 3;
typedef short i16x4 __attribute__((ext_vector_type(4)));
constexpr int kGroups = kTileNnz / (4 * kBlock);
static_assert(kGroups * 4 * kBlock == kTileNnz, "tile must be whole groups per thread");
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Workgroups are dispatched round-robin over the 8 XCDs; this maps the
// hardware block id to a logical id so that each XCD (and its L2) works on
// one contiguous range of rows.
__device__ __forceinline__ int xcd_swizzle(int b, int nb) {
    constexpr int nx = 8;
    const int per = nb / nx, rem = nb % nx;
    const int xcd = b % nx, local = b / nx;
    return xcd < rem ? xcd * (per + 1) + local
                     : rem * (per + 1) + (xcd - rem) * per + local;
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Deterministic block sum of K doubles; every thread receives the totals.
template <int K, int BS>
__device__ __forceinline__ void block_sum(double (&v)[K], double *lds) {
    constexpr int NW = BS / 64;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = wave_sum(v[k]);
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) lds[k * NW + w] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < NW; ++i) s += lds[k * NW + i];
        v[k] = s;
    }
    __syncthreads();
}

// Matrix streams (column indices, values) are read once per product: load
// them non-temporally so they do not evict the vector entries the gathers
// reuse from L2.
#ifndef NSFEM_STREAM_LOADS
#define NSFEM_STREAM_LOADS 1
#endif
template <typename T>
__device__ __forceinline__ T ld_stream(const T *p) {
#if NSFEM_STREAM_LOADS
    return __builtin_nontemporal_load(p);
#else
    return *p;
#endif
}

// 16-bit column offsets unless NSFEM_CG_IDX16=0 (comparison runs)
bool want_idx16() {
    static const bool on = [] {
        const char *e = std::getenv("NSFEM_CG_IDX16");
        return !(e && std::atoi(e) == 0);
    }();
    return on;
}

template <typename T>
__device__ __forceinline__ T fma_t(T a, T b, T c);
template <>
__device__ __forceinline__ double fma_t<double>(double a, double b, double c) {
    return __builtin_fma(a, b, c);
}
template <>
__device__ __forceinline__ float fma_t<float>(float a, float b, float c) {
    return __builtin_fmaf(a, b, c);
}

}  // namespace

// ------------------------------------------------------------ tile tables
namespace {
// Greedy cut of the rows into runs of <= max_rows rows and <= max_nnz
// nonzeros; a single longer row forms a run of its own.
std::vector<int32_t> cut_rows(const std::vector<int32_t> &rs, int rows, int max_rows,
                              int max_nnz) {
    std::vector<int32_t> t;
    t.reserve((size_t)rows / std::max(1, max_rows / 2) + 2);
    int r = 0;
    t.push_back(0);
    while (r < rows) {
        int end = r;
        int64_t nz = 0;
        while (end < rows && end - r < max_rows) {
            const int64_t rn = rs[end + 1] - rs[end];
            if (end > r && nz + rn > max_nnz) break;
            nz += rn;
            ++end;
            if (nz > max_nnz) break;
        }
        t.push_back(end);
        r = end;
    }
    return t;
}
}  // namespace

namespace {
// dcol[k] = col[k] - first row of k's wave tile, one wave per tile; bad[0]
// is raised when an offset does not fit 16 bits.
__global__ void k_col_delta(int n_wtiles, const int4 *__restrict__ meta,
                            const int32_t *__restrict__ col, int16_t *__restrict__ dcol,
                            int *bad) {
    const int t = blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
    if (t >= n_wtiles) return;
    const int4 m = meta[t];
    int out = 0;
    for (int k = threadIdx.x & 63; k < m.w; k += 64) {
        const int dv = col[m.z + k] - m.x;
        out |= (dv < -32768 || dv > 32767) ? 1 : 0;
        dcol[m.z + k] = (int16_t)dv;
    }
    if (out) __hip_atomic_fetch_or(bad, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Kernels stream 16-bit column offsets instead of 32-bit columns when every
// offset from its tile's first row fits (banded numberings: the offsets span
// about twice the mesh width).  Returns whether they do; `out` is released
// if not.
bool col_delta(const Matrix &m, int n_tiles, const int4 *meta, DeviceArray<int16_t> &out) {
    out.release();
    if (m.nnz <= 0 || m.rows != m.cols || n_tiles <= 0) return false;
    out.resize((size_t)m.nnz + 8);  // 8 zero offsets of padding for group loads
    NSFEM_HIP(hipMemset(out.ptr + m.nnz, 0, 8 * sizeof(int16_t)));
    DeviceArray<int> bad;
    bad.resize(1);
    NSFEM_HIP(hipMemset(bad.ptr, 0, sizeof(int)));
    constexpr int kWavesPerBlock = 4;
    k_col_delta<<<(n_tiles + kWavesPerBlock - 1) / kWavesPerBlock, 64 * kWavesPerBlock>>>(
        n_tiles, meta, m.col.ptr, out.ptr, bad.ptr);
    NSFEM_HIP(hipGetLastError());
    int h = 1;
    NSFEM_HIP(hipMemcpy(&h, bad.ptr, sizeof(int), hipMemcpyDeviceToHost));
    if (h != 0) out.release();
    return h == 0;
}

// wave tiles: the persistent CG's offsets
void build_col_delta(Matrix &m) { m.dcol_ok = col_delta(m, m.n_wtiles, m.wmeta.ptr, m.dcol); }

// Group loads (8 nonzeros per lane from a multiple of 8) need the 16-bit
// offsets (padded by 8) and every multi-row tile within kStageNnz nonzeros.
void set_group_loads(Matrix &m) {
    m.groups_ok = m.dcol_ok && m.nnz > 0 && m.max_multirow_nz <= kStageNnz;
}

}  // namespace

namespace {
// out = {most nonzeros of a row, most columns below and above the diagonal}
// (columns ascend within a row)
__global__ void k_row_shape(int rows, const int32_t *__restrict__ rs,
                            const int32_t *__restrict__ col, int *__restrict__ out) {
    int nz = 0, lo = 0, hi = 0;
    for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < rows; r += gridDim.x * blockDim.x) {
        const int a = rs[r], b = rs[r + 1];
        if (a == b) continue;
        nz = max(nz, b - a);
        lo = max(lo, r - col[a]);
        hi = max(hi, col[b - 1] - r);
    }
    for (int o = 32; o >= 1; o >>= 1) {
        nz = max(nz, __shfl_xor(nz, o, 64));
        lo = max(lo, __shfl_xor(lo, o, 64));
        hi = max(hi, __shfl_xor(hi, o, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMax(out, nz);
        atomicMax(out + 1, lo);
        atomicMax(out + 2, hi);
    }
}

RowShape row_shape(const Matrix &m) {
    int h[3] = {0, 0, 0};
    if (m.rows == m.cols && m.nnz > 0) {
        DeviceArray<int> out;
        out.resize(3);
        NSFEM_HIP(hipMemset(out.ptr, 0, sizeof(h)));
        k_row_shape<<<std::max(1, std::min((m.rows + 255) / 256, 1024)), 256>>>(
            m.rows, m.row_start.ptr, m.col.ptr, out.ptr);
        NSFEM_HIP(hipGetLastError());
        NSFEM_HIP(hipMemcpy(h, out.ptr, sizeof(h), hipMemcpyDeviceToHost));
    }
    return {h[0], h[1], h[2]};
}
}  // namespace

void build_tiles(Matrix &m, const std::vector<int32_t> &rs, const RowShape *shape) {
    std::vector<int32_t> t = cut_rows(rs, m.rows, kTileRows, kSpmvTileNnz);
    m.n_tiles = (int)t.size() - 1;
    m.host_rs = rs;
    std::vector<int4> meta((size_t)std::max(m.n_tiles, 1));
    for (int i = 0; i < m.n_tiles; ++i)
        meta[i] = make_int4(t[i], t[i + 1], rs[t[i]], rs[t[i + 1]] - rs[t[i]]);
    m.tiles.resize(meta.size());
    NSFEM_HIP(hipMemcpy(m.tiles.ptr, meta.data(), meta.size() * sizeof(int4),
                        hipMemcpyHostToDevice));
    m.bcol_ok = col_delta(m, m.n_tiles, m.tiles.ptr, m.bcol);
    m.shape = shape ? *shape : row_shape(m);
    build_wave_tiles(m, kWaveRows, kStageNnz);
}

void build_wave_tiles(Matrix &m, int rows, int nnz) {
    NSFEM_REQUIRE(rows >= 1 && rows <= kWaveRows && nnz >= 64 && nnz <= kWaveNnz,
                  NSFEM_INVALID_ARGUMENT, "wave tile shape out of range");
    const std::vector<int32_t> &rs = m.host_rs;
    m.wave_rows = rows;
    m.wave_nnz = nnz;
    std::vector<int32_t> w = cut_rows(rs, m.rows, rows, nnz);
    m.n_wtiles = (int)w.size() - 1;
    m.host_wtiles = w;
    for (auto &plan : m.res_plan) plan = ResidentPlan{};
    for (auto &plan : m.batch_least) plan = ResidentPlan{};
    for (auto &plan : m.batch_plan) plan = ResidentPlan{};
    m.host_wtile_prefix.assign(w.size(), 0);
    for (int i = 0; i < m.n_wtiles; ++i)
        m.host_wtile_prefix[i + 1] =
            m.host_wtile_prefix[i] + (rs[w[i + 1]] - rs[w[i]]) + (w[i + 1] - w[i]);
    m.wtiles.resize(w.size());
    NSFEM_HIP(hipMemcpy(m.wtiles.ptr, w.data(), w.size() * sizeof(int32_t),
                        hipMemcpyHostToDevice));
    std::vector<int4> meta((size_t)std::max(m.n_wtiles, 1));
    m.max_multirow_nz = 0;
    for (int i = 0; i < m.n_wtiles; ++i) {
        meta[i] = make_int4(w[i], w[i + 1], rs[w[i]], rs[w[i + 1]] - rs[w[i]]);
        if (w[i + 1] - w[i] > 1) m.max_multirow_nz = std::max(m.max_multirow_nz, meta[i].w);
    }
    m.wmeta.resize(meta.size());
    NSFEM_HIP(hipMemcpy(m.wmeta.ptr, meta.data(), meta.size() * sizeof(int4),
                        hipMemcpyHostToDevice));
    m.block_tiles.resize(kMaxGridBlocks + 1);
    m.host_block_tiles.reserve(kMaxGridBlocks + 1);
    m.block_tiles_grid = 0;
    build_col_delta(m);
    set_group_loads(m);
}

namespace {
// Contiguous wave-tile ranges of `grid` blocks, balanced by (nnz + rows).
void split_tiles(const Matrix &m, int grid, std::vector<int32_t> &bt) {
    bt.resize((size_t)grid + 1);
    const int64_t total = m.host_wtile_prefix[m.n_wtiles];
    int t = 0;
    for (int b = 0; b <= grid; ++b) {
        const int64_t target = total * b / grid;
        while (t < m.n_wtiles && m.host_wtile_prefix[t] < target) ++t;
        bt[b] = t;
    }
    bt[0] = 0;
    bt[grid] = m.n_wtiles;
}
}  // namespace

// The persistent blocks' tiles.  The table lives in arrays sized for the
// largest grid at tiling time, so this only computes and copies.
void ensure_block_tiles(Device &d, Matrix &m, int grid) {
    NSFEM_REQUIRE(grid >= 1 && grid <= kMaxGridBlocks, NSFEM_ERROR, "grid size out of range");
    if (m.block_tiles_grid == grid) return;
    std::vector<int32_t> &bt = m.host_block_tiles;
    split_tiles(m, grid, bt);  // within the reserved capacity
    NSFEM_HIP(hipMemcpyAsync(m.block_tiles.ptr, bt.data(), bt.size() * sizeof(int32_t),
                             hipMemcpyHostToDevice, d.stream));
    NSFEM_HIP(hipStreamSynchronize(d.stream));
    m.block_tiles_grid = grid;
}

namespace {
__global__ void k_to_float(int64_t n, const double *__restrict__ a, float *__restrict__ b) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        b[i] = (float)a[i];
}
}  // namespace

// The FP32 copy of the values, with 8 zero entries of padding (the group-load
// product loads 8 values per lane from a multiple of 8).
void ensure_val32(Device &d, Matrix &m) {
    if (m.val32.ptr && m.val32.count == (size_t)m.nnz + 8) return;
    m.val32.resize((size_t)m.nnz + 8);
    NSFEM_HIP(hipMemsetAsync(m.val32.ptr + m.nnz, 0, 8 * sizeof(float), d.stream));
    if (m.nnz) {
        const int grid = (int)std::min<int64_t>((m.nnz + 255) / 256, 65536);
        k_to_float<<<grid, 256, 0, d.stream>>>(m.nnz, m.val.ptr, m.val32.ptr);
        NSFEM_HIP(hipGetLastError());
    }
}

// --------------------------------------------------------- Jacobi scaling
namespace {

// scale[r] = 1 / sqrt(a_rr) (the row's diagonal entries summed); a row
// without a positive diagonal sets *bad (and keeps scale 1)
__global__ void k_jacobi_scale(int n, const int32_t *__restrict__ rs,
                               const int32_t *__restrict__ col, const double *__restrict__ val,
                               double *__restrict__ scale, int32_t *__restrict__ bad) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    double d = 0.0;
    for (int32_t k = rs[r]; k < rs[r + 1]; ++k)
        if (col[k] == r) d += val[k];
    if (d > 0.0) {
        scale[r] = 1.0 / sqrt(d);
    } else {
        scale[r] = 1.0;
        *bad = 1;
    }
}

// out[k] = (float)(scale[row] * a_k * scale[col_k]): D^-1/2 A D^-1/2 in FP32
__global__ void k_jacobi_values(int n, const int32_t *__restrict__ rs,
                                const int32_t *__restrict__ col, const double *__restrict__ val,
                                const double *__restrict__ scale, float *__restrict__ out) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const double sr = scale[r];
    for (int32_t k = rs[r]; k < rs[r + 1]; ++k) out[k] = (float)(sr * val[k] * scale[col[k]]);
}
}  // namespace

// The Jacobi-scaled FP32 values and the row scales of a square matrix
// (built once; 8 zero entries of padding as val32).  False when a row has
// no positive diagonal entry: the solve then runs unscaled.
bool ensure_jacobi(Device &d, Matrix &m) {
    if (m.jacobi_built) return m.jacobi_ok;
    m.jacobi_built = true;
    m.jacobi_ok = false;
    if (m.rows != m.cols || m.rows == 0) return false;
    m.jscale.resize((size_t)m.rows);
    DeviceArray<int32_t> bad;
    bad.resize(1);
    NSFEM_HIP(hipMemsetAsync(bad.ptr, 0, sizeof(int32_t), d.stream));
    const int grid = (m.rows + 255) / 256;
    k_jacobi_scale<<<grid, 256, 0, d.stream>>>(m.rows, m.row_start.ptr, m.col.ptr, m.val.ptr,
                                               m.jscale.ptr, bad.ptr);
    NSFEM_HIP(hipGetLastError());
    int32_t h = 0;
    NSFEM_HIP(hipMemcpyAsync(&h, bad.ptr, sizeof(h), hipMemcpyDeviceToHost, d.stream));
    NSFEM_HIP(hipStreamSynchronize(d.stream));
    if (h) {
        m.jscale.release();
        return false;
    }
    m.jval32.resize((size_t)m.nnz + 8);
    NSFEM_HIP(hipMemsetAsync(m.jval32.ptr + m.nnz, 0, 8 * sizeof(float), d.stream));
    k_jacobi_values<<<grid, 256, 0, d.stream>>>(m.rows, m.row_start.ptr, m.col.ptr, m.val.ptr,
                                                m.jscale.ptr, m.jval32.ptr);
    NSFEM_HIP(hipGetLastError());
    m.jacobi_ok = true;
    return true;
}

// ------------------------------------------------------------- CSR product
namespace {

// MODE 0: y = A x.  MODE 1: y = lhs - A x (y may alias lhs).
// MODE 2: y = A x - lhs.  MODE 3: y = x + omega dinv (lhs - A x), a damped
// Jacobi sweep into another vector (y aliases neither x nor lhs; the same
// roundings as the residual product followed by a Jacobi update).
// MODE 4: y += A x (the roundings of the product followed by k_add).
// MODE 5: y = A x and y2 = omega dinv y, the Jacobi sweep from zero that
// follows a restriction (k_jacobi0's roundings).
// DOT: partial[tile] = the tile's rows' sum of y times x (MODE 0) or times
// rdot (MODE 3) in FP64, one wave after the other: a CG's (p, A p) and
// (r, z) without another pass over the vectors or another launch (a launch
// costs 3.3 us however little it does).
// IT = int16_t reads the columns as 16-bit offsets from the tile's first row
// (bcol, square matrices whose offsets fit): 2 bytes less per nonzero.
// T = double: the FP64 values; T = float: the FP32 copy (val32) with FP32
// x.  S: the type of the products, sums, lhs and y: T (FP32 throughout for
// the multigrid smoothing of mixed-precision solves), or double with FP32
// values and x (each FP32 x FP32 product exact in FP64, summed in FP64: the
// product of a CG's FP32 direction, free of the cancellation an FP32 sum
// suffers on smooth vectors).
template <typename S>
struct SpmvTail {
    const S *dinv = nullptr;
    S omega = S(0);
    S *y2 = nullptr;
    const double *rdot = nullptr;
    double *partial = nullptr;
};

template <int MODE, typename IT, typename T, typename S = T, bool DOT = false>
__global__ __launch_bounds__(kBlock) void k_spmv(int n_tiles, int n_rows, int64_t nnz,
                                                 const int4 *__restrict__ tiles,
                                                 const int32_t *__restrict__ rs,
                                                 const int32_t *__restrict__ col,
                                                 const int16_t *__restrict__ bcol,
                                                 const T *__restrict__ val,
                                                 const T *__restrict__ x,
                                                 const S *lhs, S *y, const SpmvTail<S> tail) {
    constexpr bool F64 = std::is_same<T, double>::value;
    constexpr bool S64 = std::is_same<S, double>::value;
    __shared__ __align__(16) S prod[kTileNnz];
    __shared__ S red[kWaves];
    __shared__ double dred[DOT ? kWaves : 1];
    double dsum[1] = {0.0};
    const int t = xcd_swizzle(blockIdx.x, gridDim.x);
    if (t >= n_tiles) return;
    const int tid = threadIdx.x;
    const int4 tile = tiles[t];
    const int r0 = tile.x, r1 = tile.y, k0 = tile.z, nz = tile.w;
    if (nz <= kSpmvTileNnz) {
        // groups of 4 nonzeros from ka = k0 rounded down to a multiple of 4;
        // entries of the neighbouring tiles in the first and last group are
        // multiplied too (their columns are valid) and never summed, entries
        // past the end of the matrix are column 0, value 0
        const int ka = k0 & ~3;
        const int ng = (k0 + nz - ka + 3) >> 2;
        i32x4 c[kGroups];
        T v[kGroups][4];
#pragma unroll
        for (int g = 0; g < kGroups; ++g) {
            const int grp = tid + g * kBlock;
            c[g] = i32x4{0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 4; ++e) v[g][e] = T(0);
            if (grp < ng) {
                const int64_t base = ka + 4 * (int64_t)grp;
                if (base + 4 <= nnz) {
                    if constexpr (std::is_same<IT, int16_t>::value) {
                        // entries of a neighbouring tile decode relative to
                        // the wrong row: clamped into the vector, never summed
                        const i16x4 d = ld_stream(reinterpret_cast<const i16x4 *>(bcol + base));
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            c[g][e] = min(max(r0 + (int)d[e], 0), n_rows - 1);
                    } else {
                        c[g] = ld_stream(reinterpret_cast<const i32x4 *>(col + base));
                    }
                    if constexpr (F64) {
                        const f64x2 a = ld_stream(reinterpret_cast<const f64x2 *>(val + base));
                        const f64x2 b = ld_stream(reinterpret_cast<const f64x2 *>(val + base + 2));
                        v[g][0] = a.x;
                        v[g][1] = a.y;
                        v[g][2] = b.x;
                        v[g][3] = b.y;
                    } else {
                        const f32x4_t a = ld_stream(reinterpret_cast<const f32x4_t *>(val + base));
                        v[g][0] = a.x;
                        v[g][1] = a.y;
                        v[g][2] = a.z;
                        v[g][3] = a.w;
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const bool in = base + e < nnz;
                        c[g][e] = in ? col[base + e] : 0;
                        v[g][e] = in ? val[base + e] : T(0);
                    }
                }
            }
        }
        // the row's own words, needed only after the barrier: asked for here,
        // behind the streams
        const int row = r0 + tid;
        int ra = ka, rb = ka;
        S lrow = S(0), drow = S(0), xrow = S(0);
        double dotrow = 0.0;
        if (row < r1) {
            ra = rs[row];
            rb = rs[row + 1];
            if (MODE >= 1 && MODE <= 3) lrow = lhs[row];
            if (MODE == 4) lrow = y[row];
            if (MODE == 3 || MODE == 5) drow = tail.dinv[row];
            if (MODE == 3 || (DOT && MODE == 0)) xrow = (S)x[row];
            if (DOT && MODE == 3) dotrow = tail.rdot[row];
        }
        // columns transposed through the wave's own slice of prod (256
        // products; the 256 columns take 1 KB of it), so that each gather
        // instruction covers 64 consecutive nonzeros
        const int lane = tid & 63;
#pragma unroll
        for (int g = 0; g < kGroups; ++g) {
            const int chunk = 4 * (g * kBlock + (tid & ~63));  // first element of the wave's slice
            int *cs = reinterpret_cast<int *>(prod + chunk);
            if (chunk < 4 * ng) {  // wave-uniform
                *reinterpret_cast<i32x4 *>(cs + 4 * lane) = c[g];
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
                int cc[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) cc[j] = cs[lane + 64 * j];
                T xv[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) xv[j] = x[cc[j]];
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int j = 0; j < 4; ++j) prod[chunk + lane + 64 * j] = (S)xv[j];
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if constexpr (S64) {
                    f64x2 p0 = *reinterpret_cast<const f64x2 *>(prod + chunk + 4 * lane);
                    f64x2 p1 = *reinterpret_cast<const f64x2 *>(prod + chunk + 4 * lane + 2);
                    p0.x = (double)v[g][0] * p0.x;
                    p0.y = (double)v[g][1] * p0.y;
                    p1.x = (double)v[g][2] * p1.x;
                    p1.y = (double)v[g][3] * p1.y;
                    *reinterpret_cast<f64x2 *>(prod + chunk + 4 * lane) = p0;
                    *reinterpret_cast<f64x2 *>(prod + chunk + 4 * lane + 2) = p1;
                } else {
                    f32x4_t p = *reinterpret_cast<const f32x4_t *>(prod + chunk + 4 * lane);
                    p.x = v[g][0] * p.x;
                    p.y = v[g][1] * p.y;
                    p.z = v[g][2] * p.z;
                    p.w = v[g][3] * p.w;
                    *reinterpret_cast<f32x4_t *>(prod + chunk + 4 * lane) = p;
                }
            }
        }
        __syncthreads();
        if (row < r1) {
            S s = S(0);
            for (int k = ra - ka; k < rb - ka; ++k) s += prod[k];
            if (MODE == 0) y[row] = s;
            if (MODE == 1) y[row] = lrow - s;
            if (MODE == 2) y[row] = s - lrow;
            if (MODE == 3) {
                const S r = lrow - s;
                s = __builtin_fma(tail.omega * drow, r, xrow);
                y[row] = s;
            }
            if (MODE == 4) y[row] = s + lrow;
            if (MODE == 5) {
                y[row] = s;
                tail.y2[row] = (tail.omega * drow) * s;
            }
            if (DOT) dsum[0] = (double)s * (MODE == 0 ? (double)xrow : dotrow);
        }
        if (DOT) {
            block_sum<1, kBlock>(dsum, dred);
            if (tid == 0) tail.partial[t] = dsum[0];
        }
    } else {  // one row longer than a tile
        S s = S(0);
        for (int k = tid; k < nz; k += kBlock) s += (S)val[k0 + k] * (S)x[col[k0 + k]];
        s = wave_sum(s);
        if ((tid & 63) == 0) red[tid >> 6] = s;
        __syncthreads();
        if (tid == 0) {
            S tot = S(0);
            for (int i = 0; i < kWaves; ++i) tot += red[i];
            if (MODE == 0) y[r0] = tot;
            if (MODE == 1) y[r0] = lhs[r0] - tot;
            if (MODE == 2) y[r0] = tot - lhs[r0];
            if (MODE == 3) {
                const S r = lhs[r0] - tot;
                tot = __builtin_fma(tail.omega * tail.dinv[r0], r, (S)x[r0]);
                y[r0] = tot;
            }
            if (MODE == 4) y[r0] = tot + y[r0];
            if (MODE == 5) {
                y[r0] = tot;
                tail.y2[r0] = (tail.omega * tail.dinv[r0]) * tot;
            }
            if (DOT) tail.partial[t] = (double)tot * (MODE == 0 ? (double)x[r0] : tail.rdot[r0]);
        }
    }
}

// y = A x with a dense row-major n x n matrix (a multigrid hierarchy's deepest
// inverse, some hundred to a thousand rows): a wave per row, its lanes
// striding over the row, kDenseAhead loads of the row and of x in flight
// each.  Bound by latency (4.7 MB at 1,089 rows, out of L2 or the Infinity
// Cache).  As a sparse product it gave each row a block and one thread the
// sum of the row's products: 28 / 33 / 45 / 61 us at 576 / 676 / 961 / 1,089
// rows in FP32 against 3.0 / 3.5 us at the first two here.
constexpr int kDenseAhead = 8;
template <typename T>
__global__ __launch_bounds__(kBlock) void k_dense(int n, const T *__restrict__ a,
                                                  const T *__restrict__ x, T *__restrict__ y) {
    const int row = blockIdx.x * kWaves + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= n) return;
    a += (size_t)row * n;
    T s = T(0);
    int k = lane;
    for (; k + 64 * (kDenseAhead - 1) < n; k += 64 * kDenseAhead) {
        T av[kDenseAhead], xv[kDenseAhead];
#pragma unroll
        for (int j = 0; j < kDenseAhead; ++j) {
            av[j] = a[k + 64 * j];
            xv[j] = x[k + 64 * j];
        }
#pragma unroll
        for (int j = 0; j < kDenseAhead; ++j) s = fma_t(av[j], xv[j], s);
    }
#pragma unroll 4
    for (; k < n; k += 64) s = fma_t(a[k], x[k], s);
    s = wave_sum(s);
    if (lane == 0) y[row] = s;
}

__global__ void k_axpy(int n, double a, const double *__restrict__ x, double *y) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        y[i] = __builtin_fma(a, x[i], y[i]);
}

// y = y0 + a_0 X_0 + ... + a_{l-1} X_{l-1} (y0 = 0, or y's own values when
// `accumulate`), X_k = X + k * stride, one fused multiply-add per term in k
// order: the bits of a fill (or nothing) followed by l k_axpy launches, in
// one pass over the vectors.  y2, when given, receives the same values.
constexpr int kCombineMax = 8;
struct CombineCoef {
    double a[kCombineMax];
};

__global__ void k_combine(int n, int l, CombineCoef c, const double *__restrict__ X,
                          size_t stride, int accumulate, double *__restrict__ y,
                          double *__restrict__ y2) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        double t = accumulate ? y[i] : 0.0;
        for (int k = 0; k < l; ++k) t = __builtin_fma(c.a[k], X[(size_t)k * stride + i], t);
        y[i] = t;
        if (y2) y2[i] = t;
    }
}

__global__ void k_axpby(int n, double a, double b, const double *x, const double *y,
                        double *out) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        out[i] = __builtin_fma(a, x[i], b * y[i]);
}

// Deterministic dot: block k sums the contiguous chunk k, a single block adds
// the chunk sums in order.  Chunks of 1,024 until there are kDotBlocks of
// them: with 4,096 a vector of some ten thousand entries had 16 dependent
// rounds on ten CUs (6.8 us on 40,401 entries, a launch's 3 us included).
__global__ __launch_bounds__(kBlock) void k_dot_partial(int n, int chunk,
                                                        const double *__restrict__ a,
                                                        const double *__restrict__ b,
                                                        double *__restrict__ partial) {
    __shared__ double lds[kWaves];
    const int lo = blockIdx.x * chunk;
    const int hi = min(n, lo + chunk);
    double s[1] = {0.0};
#pragma unroll 4
    for (int i = lo + threadIdx.x; i < hi; i += kBlock) s[0] = __builtin_fma(a[i], b[i], s[0]);
    block_sum<1, kBlock>(s, lds);
    if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

__global__ __launch_bounds__(kBlock) void k_dot_final(int nb, const double *__restrict__ partial,
                                                      double *result) {
    __shared__ double lds[kWaves];
    double s[1] = {0.0};
    for (int i = threadIdx.x; i < nb; i += kBlock) s[0] += partial[i];
    block_sum<1, kBlock>(s, lds);
    if (threadIdx.x == 0) result[0] += s[0];
}

// X_i . y for l <= kDotsMax vectors X_i = X + i * stride, each as
// k_dot_partial and k_dot_final add it (the same bits): y is read once and
// the l sums come in two launches.  The sums go to `out`, the host's page: the
// fill before and the copy after cost more than the sums of a vector of some
// ten thousand entries (2.4 and 4.1 us a launch, next to 3.4 for the dot):
// ten steps of the V-cycle chain on the 512 x 128 channel went from 44.3 to
// 38.6 ms, eight on the 200 x 200 cavity from 24.1 to 20.2.
constexpr int kDotsMax = 8;
__global__ __launch_bounds__(kBlock) void k_dots_partial(int n, int chunk, int l,
                                                         const double *__restrict__ X,
                                                         size_t stride,
                                                         const double *__restrict__ y,
                                                         double *__restrict__ partial) {
    __shared__ double lds[kDotsMax * kWaves];
    const int lo = blockIdx.x * chunk;
    const int hi = min(n, lo + chunk);
    double s[kDotsMax] = {};
#pragma unroll 2
    for (int i = lo + threadIdx.x; i < hi; i += kBlock) {
        const double yi = y[i];
#pragma unroll
        for (int k = 0; k < kDotsMax; ++k)
            if (k < l) s[k] = __builtin_fma(X[(size_t)k * stride + i], yi, s[k]);
    }
    block_sum<kDotsMax, kBlock>(s, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < kDotsMax; ++k)
            if (k < l) partial[(size_t)k * gridDim.x + blockIdx.x] = s[k];
    }
}

__global__ __launch_bounds__(kBlock) void k_dots_final(int nb, const double *__restrict__ partial,
                                                       double *out) {
    __shared__ double lds[kWaves];
    double s[1] = {0.0};
    for (int i = threadIdx.x; i < nb; i += kBlock) s[0] += partial[(size_t)blockIdx.x * nb + i];
    block_sum<1, kBlock>(s, lds);
    if (threadIdx.x == 0) out[blockIdx.x] = 0.0 + s[0];
}

// The sum of n partials, the same bits in every thread of every block.  One
// partial (folded before) is read as it is: with a block sum's two barriers
// in front of each block's work k_pcg_direction took 71 us on the 16.8 M
// velocity nodes of the 2048^2 cavity, without 51.
__device__ __forceinline__ double sum_partials(int n, const double *__restrict__ part,
                                               double *lds) {
    if (n == 1) return 0.0 + part[0];
    double s[1] = {0.0};
#pragma unroll 4
    for (int i = threadIdx.x; i < n; i += kBlock) s[0] += part[i];
    block_sum<1, kBlock>(s, lds);
    return s[0];
}

// out[block] = the sum of the block's contiguous share of part[0..n)
__global__ __launch_bounds__(kBlock) void k_fold(int n, const double *__restrict__ part,
                                                 double *__restrict__ out) {
    __shared__ double lds[kWaves];
    const int lo = (int)((int64_t)n * blockIdx.x / gridDim.x);
    const int hi = (int)((int64_t)n * (blockIdx.x + 1) / gridDim.x);
    const double s = sum_partials(hi - lo, part + lo, lds);
    if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// The update of a CG with FP32 directions p (q = A p in FP64) and an FP32
// preconditioner, step `k`: alpha = (r, z) / (p, q), (p, q) the sum of npq
// partials that every block adds for itself; x += alpha p and r -= alpha q
// in FP64, r32 = r rounded to FP32 (the preconditioner's input), x0 = omega
// dinv r32 (its first Jacobi sweep, from zero), and the partial sums of
// (r, r) per contiguous chunk.  A (p, q) or (r, z) that is not positive
// leaves x and r as they are, for the host to see.
__global__ __launch_bounds__(kBlock) void k_pcg_update(
    int n, int chunk, PcgScalars *sc, int k, int npq, const double *__restrict__ pq_part,
    const float *__restrict__ p, const double *__restrict__ q, double *__restrict__ x,
    double *__restrict__ r, float *__restrict__ r32, const float *__restrict__ dinv, float omega,
    float *__restrict__ x0, double *__restrict__ partial) {
    __shared__ double lds[kWaves];
    const double pq = sum_partials(npq, pq_part, lds);
    const double rz = sc->rz[k & 1];
    const double a = pq > 0.0 && rz > 0.0 ? rz / pq : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) sc->pq = pq;
    const int lo = blockIdx.x * chunk;
    const int hi = min(n, lo + chunk);
    double s[1] = {0.0};
    if (a > 0.0) {
#pragma unroll 2
        for (int i = lo + threadIdx.x; i < hi; i += kBlock) {
            x[i] = __builtin_fma(a, (double)p[i], x[i]);
            const double ri = __builtin_fma(-a, q[i], r[i]);
            const float rf = (float)ri;
            r[i] = ri;
            r32[i] = rf;
            x0[i] = (omega * dinv[i]) * rf;
            s[0] = __builtin_fma(ri, ri, s[0]);
        }
    }
    block_sum<1, kBlock>(s, lds);
    if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

// The step's scalars to the host's page: (r, r) from its partials, (p, q)
// and (r, z).  One block.
__global__ __launch_bounds__(kBlock) void k_pcg_report(int nrr, const double *__restrict__ rr_part,
                                                       const PcgScalars *__restrict__ sc, int k,
                                                       PcgReport *host) {
    __shared__ double lds[kWaves];
    const double rr = sum_partials(nrr, rr_part, lds);
    if (threadIdx.x == 0) {
        host->rr = rr;
        host->pq = sc->pq;
        host->rz = sc->rz[k & 1];
    }
}

// r32 = r rounded to FP32 and x0 = omega dinv r32 (see k_pcg_update)
__global__ void k_pcg_round(int n, const double *__restrict__ r, float *__restrict__ r32,
                            const float *__restrict__ dinv, float omega, float *__restrict__ x0) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const float rf = (float)r[i];
        r32[i] = rf;
        x0[i] = (omega * dinv[i]) * rf;
    }
}

// The direction of step k: p = z + beta p in FP32 storage, the sum in FP64,
// beta = (r, z) / the step before's (p = z at k = 0).  (r, z) is the sum of
// nrz partials, which every block adds for itself.
__global__ __launch_bounds__(kBlock) void k_pcg_direction(int n, int nrz,
                                                          const double *__restrict__ rz_part,
                                                          PcgScalars *sc, int k,
                                                          const float *__restrict__ z,
                                                          float *__restrict__ p) {
    __shared__ double lds[kWaves];
    const double rz = sum_partials(nrz, rz_part, lds);
    if (blockIdx.x == 0 && threadIdx.x == 0) sc->rz[k & 1] = rz;
    const double b = k > 0 ? rz / sc->rz[(k + 1) & 1] : 0.0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = k > 0 ? (float)__builtin_fma(b, (double)p[i], (double)z[i]) : z[i];
}

__global__ void k_scatter(int count, const int32_t *__restrict__ idx,
                          const double *__restrict__ val, double *__restrict__ dst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) dst[idx[i]] = val[i];
}

__global__ void k_gather(int count, const int32_t *__restrict__ idx,
                         const double *__restrict__ src, double *__restrict__ dst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) dst[i] = src[idx[i]];
}

template <typename T>
__global__ void k_scatter_value(int count, const int32_t *__restrict__ idx, T v,
                                T *__restrict__ dst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) dst[idx[i]] = v;
}

template <typename T>
__global__ void k_add(int n, const T *__restrict__ a, T *__restrict__ y) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        y[i] = a[i] + y[i];
}

// x = w * dinv .* b (the damped Jacobi sweep from x = 0)
template <typename T>
__global__ void k_jacobi0(int n, T w, const T *__restrict__ dinv, const T *__restrict__ b,
                          T *__restrict__ x) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        x[i] = (w * dinv[i]) * b[i];
}

// y = a rounded to (or widened from) y's type
template <typename A, typename Y>
__global__ void k_convert(int n, const A *__restrict__ a, Y *__restrict__ y) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        y[i] = (Y)a[i];
}

template <typename T>
__global__ void k_fill(int n, T v, T *__restrict__ y) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        y[i] = v;
}

__global__ void k_copy(int n, const double *__restrict__ a, double *__restrict__ y) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        y[i] = a[i];
}

constexpr int kDotBlocks = 1024;  // per-block partials of the dot product

// blocks and chunk of the deterministic dot over n entries
void dot_shape(int n, int &nb, int &chunk) {
    nb = (int)std::max<int64_t>(1, std::min<int64_t>(((int64_t)n + 1023) / 1024, kDotBlocks));
    chunk = (int)std::max<int64_t>(1, ((int64_t)n + nb - 1) / nb);
}

// One element per thread up to 2^28 elements: a full grid streams at
// 6.1 TB/s (copy) on MI355X where a grid-stride loop over 8192 blocks
// reaches 4.5.
inline int ew_grid(int n) { return std::max(1, std::min((n + kBlock - 1) / kBlock, 1 << 20)); }

}  // namespace

namespace {
template <typename T>
const T *values(Matrix &m);
template <>
const double *values<double>(Matrix &m) {
    return m.val.ptr;
}
template <>
const float *values<float>(Matrix &m) {
    return m.val32.ptr;
}

template <int MODE, typename T, typename S, bool DOT = false>
void spmv_launch(Device &d, Matrix &m, const T *x, const S *lhs, S *y,
                 const SpmvTail<S> &tail = SpmvTail<S>()) {
    if (m.bcol_ok && want_idx16())
        k_spmv<MODE, int16_t, T, S, DOT><<<m.n_tiles, kBlock, 0, d.stream>>>(
            m.n_tiles, m.rows, m.nnz, m.tiles.ptr, m.row_start.ptr, m.col.ptr, m.bcol.ptr,
            values<T>(m), x, lhs, y, tail);
    else
        k_spmv<MODE, int32_t, T, S, DOT><<<m.n_tiles, kBlock, 0, d.stream>>>(
            m.n_tiles, m.rows, m.nnz, m.tiles.ptr, m.row_start.ptr, m.col.ptr, m.bcol.ptr,
            values<T>(m), x, lhs, y, tail);
}

template <typename T>
void spmv_any(Device &d, Matrix &m, const T *x, const T *lhs, T *y, int mode) {
    if (m.rows == 0) return;
    if (mode == 0)
        spmv_launch<0>(d, m, x, lhs, y);
    else if (mode == 1)
        spmv_launch<1>(d, m, x, lhs, y);
    else
        spmv_launch<2>(d, m, x, lhs, y);
    NSFEM_HIP(hipGetLastError());
}
}  // namespace

void launch_spmv(Device &d, Matrix &m, const double *x, const double *lhs, double *y,
                 int mode) {
    spmv_any(d, m, x, lhs, y, mode);
}

// The FP32 product reads the FP32 copy of the values (val32, built by
// ensure_val32 before the first call).
void launch_spmv(Device &d, Matrix &m, const float *x, const float *lhs, float *y, int mode) {
    NSFEM_REQUIRE(m.rows == 0 || m.val32.ptr, NSFEM_NOT_READY,
                  "FP32 product without the FP32 copy of the values");
    spmv_any(d, m, x, lhs, y, mode);
}

namespace {
template <typename T>
void require_values(const Matrix &m) {
    NSFEM_REQUIRE((std::is_same<T, double>::value || m.val32.ptr), NSFEM_NOT_READY,
                  "FP32 product without the FP32 copy of the values");
}
}  // namespace

template <typename T>
void launch_sweep(Device &d, Matrix &m, double w, const T *dinv, const T *x, const T *b, T *y) {
    if (m.rows == 0) return;
    require_values<T>(m);
    SpmvTail<T> tail;
    tail.dinv = dinv;
    tail.omega = (T)w;
    spmv_launch<3>(d, m, x, b, y, tail);
    NSFEM_HIP(hipGetLastError());
}
template void launch_sweep(Device &, Matrix &, double, const double *, const double *,
                           const double *, double *);
template void launch_sweep(Device &, Matrix &, double, const float *, const float *, const float *,
                           float *);

template <typename T>
void launch_spmv_add(Device &d, Matrix &m, const T *x, T *y) {
    if (m.rows == 0) return;
    require_values<T>(m);
    spmv_launch<4>(d, m, x, (const T *)nullptr, y);
    NSFEM_HIP(hipGetLastError());
}
template void launch_spmv_add(Device &, Matrix &, const double *, double *);
template void launch_spmv_add(Device &, Matrix &, const float *, float *);

template <typename T>
void launch_restrict(Device &d, Matrix &m, const T *x, T *y, double w, const T *dinv, T *y2) {
    if (m.rows == 0) return;
    require_values<T>(m);
    SpmvTail<T> tail;
    tail.dinv = dinv;
    tail.omega = (T)w;
    tail.y2 = y2;
    spmv_launch<5>(d, m, x, (const T *)nullptr, y, tail);
    NSFEM_HIP(hipGetLastError());
}
template void launch_restrict(Device &, Matrix &, const double *, double *, double, const double *,
                              double *);
template void launch_restrict(Device &, Matrix &, const float *, float *, double, const float *,
                              float *);

// --------------------------------- CG with an FP32 preconditioner
namespace {
// Partials that a kernel's blocks add for themselves; more of them are folded
// to one first, which two launches over a thousand tiles hide.
constexpr int kPcgInline = 1024;
constexpr int kPcgFold = 256;

void fold_partials(Device &d, PcgDevice &w) {
    if (w.count <= kPcgInline) {
        w.sums = w.partial.ptr;
        return;
    }
    double *folded = w.partial.ptr + w.count, *one = folded + kPcgFold;
    k_fold<<<kPcgFold, kBlock, 0, d.stream>>>(w.count, w.partial.ptr, folded);
    k_fold<<<1, kBlock, 0, d.stream>>>(kPcgFold, folded, one);
    NSFEM_HIP(hipGetLastError());
    w.sums = one;
    w.count = 1;
}
}  // namespace

void pcg_reserve(Device &d, const Matrix &m, PcgDevice &w) {
    w.partial.ensure((size_t)m.n_tiles + kPcgFold + 1);
    w.scalars.ensure(1);
    w.report.ensure(1);
    d.dot_partial.ensure(kDotBlocks);
}

void launch_pcg_round(Device &d, int n, const double *r, float *r32, const float *dinv, double w,
                      float *x0) {
    if (n <= 0) return;
    k_pcg_round<<<ew_grid(n), kBlock, 0, d.stream>>>(n, r, r32, dinv, (float)w, x0);
    NSFEM_HIP(hipGetLastError());
}

void launch_pcg_product(Device &d, Matrix &m, const float *p, double *q, PcgDevice &w) {
    require_values<float>(m);
    SpmvTail<double> tail;
    tail.partial = w.partial.ptr;
    w.count = m.n_tiles;
    spmv_launch<0, float, double, true>(d, m, p, (const double *)nullptr, q, tail);
    NSFEM_HIP(hipGetLastError());
}

void launch_pcg_sweep(Device &d, Matrix &m, double omega, const float *dinv, const float *x,
                      const float *b, float *y, const double *r, PcgDevice &w) {
    require_values<float>(m);
    SpmvTail<float> tail;
    tail.dinv = dinv;
    tail.omega = (float)omega;
    tail.rdot = r;
    tail.partial = w.partial.ptr;
    w.count = m.n_tiles;
    spmv_launch<3, float, float, true>(d, m, x, b, y, tail);
    NSFEM_HIP(hipGetLastError());
}

void launch_pcg_direction(Device &d, int n, int k, const float *z, float *p, PcgDevice &w) {
    fold_partials(d, w);
    k_pcg_direction<<<ew_grid(n), kBlock, 0, d.stream>>>(n, w.count, w.sums, w.scalars.ptr, k, z,
                                                        p);
    NSFEM_HIP(hipGetLastError());
}

PcgReport pcg_update(Device &d, int n, int k, const float *p, const double *q, double *x,
                     double *r, float *r32, const float *dinv, double omega, float *x0,
                     PcgDevice &w) {
    fold_partials(d, w);
    int nb, chunk;
    dot_shape(n, nb, chunk);
    k_pcg_update<<<nb, kBlock, 0, d.stream>>>(n, chunk, w.scalars.ptr, k, w.count, w.sums, p, q, x,
                                              r, r32, dinv, (float)omega, x0, d.dot_partial.ptr);
    k_pcg_report<<<1, kBlock, 0, d.stream>>>(nb, d.dot_partial.ptr, w.scalars.ptr, k,
                                             w.report.device);
    NSFEM_HIP(hipGetLastError());
    NSFEM_HIP(hipStreamSynchronize(d.stream));
    return *w.report.host;
}

template <typename T>
void launch_dense(Device &d, int n, const T *a, const T *x, T *y) {
    if (n <= 0) return;
    k_dense<T><<<(n + kWaves - 1) / kWaves, kBlock, 0, d.stream>>>(n, a, x, y);
    NSFEM_HIP(hipGetLastError());
}
template void launch_dense<double>(Device &, int, const double *, const double *, double *);
template void launch_dense<float>(Device &, int, const float *, const float *, float *);

void launch_spmv_affine(Device &d, Matrix &m, const double *x, const double *c, double *y) {
    launch_spmv(d, m, x, c, y, 2);
}

void launch_axpy(Device &d, int n, double a, const double *x, double *y) {
    if (n <= 0) return;
    k_axpy<<<ew_grid(n), kBlock, 0, d.stream>>>(n, a, x, y);
    NSFEM_HIP(hipGetLastError());
}

void launch_combine(Device &d, int n, int l, const double *a, const double *X, size_t stride,
                    bool accumulate, double *y, double *y2) {
    if (n <= 0) return;
    if (l <= 0) {
        if (!accumulate) launch_fill(d, n, 0.0, y);
        if (y2) launch_copy(d, n, y, y2);
        return;
    }
    // terms beyond kCombineMax continue from the stored partial sum (an FP64
    // store and load: the same bits as one longer chain)
    for (int k0 = 0; k0 < l; k0 += kCombineMax) {
        const int m = std::min(kCombineMax, l - k0);
        CombineCoef c{};
        for (int k = 0; k < m; ++k) c.a[k] = a[k0 + k];
        const bool last = k0 + m == l;
        k_combine<<<ew_grid(n), kBlock, 0, d.stream>>>(n, m, c, X + (size_t)k0 * stride, stride,
                                                        (accumulate || k0 > 0) ? 1 : 0, y,
                                                        last ? y2 : nullptr);
        NSFEM_HIP(hipGetLastError());
    }
}

void launch_axpby(Device &d, int n, double a, double b, const double *x, const double *y,
                  double *out) {
    if (n <= 0) return;
    k_axpby<<<ew_grid(n), kBlock, 0, d.stream>>>(n, a, b, x, y, out);
    NSFEM_HIP(hipGetLastError());
}

namespace {

// partial: kDotBlocks doubles of scratch
void dot_accumulate(Device &d, int n, const double *a, const double *b, double *result,
                    double *partial) {
    int nb, chunk;
    dot_shape(n, nb, chunk);
    k_dot_partial<<<nb, kBlock, 0, d.stream>>>(n, chunk, a, b, partial);
    k_dot_final<<<1, kBlock, 0, d.stream>>>(nb, partial, result);
    NSFEM_HIP(hipGetLastError());
}
}  // namespace

void launch_dot_accumulate(Device &d, int n, const double *a, const double *b,
                           double *result) {
    d.dot_partial.ensure(kDotBlocks);
    dot_accumulate(d, n, a, b, result, d.dot_partial.ptr);
}

void launch_dots(Device &d, int n, int l, const double *X, size_t stride, const double *y,
                 int at) {
    NSFEM_REQUIRE(at >= 0 && l >= 0 && at + l <= kDotPage, NSFEM_INVALID_ARGUMENT,
                  "more dots than the page holds");
    d.dots.ensure(kDotPage);
    d.dot_partial.ensure((size_t)kDotsMax * kDotBlocks);
    int nb, chunk;
    dot_shape(n, nb, chunk);
    for (int k = 0; k < l; k += kDotsMax) {
        const int m = std::min(kDotsMax, l - k);
        const double *Xk = X + (size_t)k * stride;
        if (m == 1)
            k_dot_partial<<<nb, kBlock, 0, d.stream>>>(n, chunk, Xk, y, d.dot_partial.ptr);
        else
            k_dots_partial<<<nb, kBlock, 0, d.stream>>>(n, chunk, m, Xk, stride, y,
                                                        d.dot_partial.ptr);
        k_dots_final<<<m, kBlock, 0, d.stream>>>(nb, d.dot_partial.ptr, d.dots.device + at + k);
        NSFEM_HIP(hipGetLastError());
    }
}

const double *wait_dots(Device &d) {
    NSFEM_HIP(hipStreamSynchronize(d.stream));
    return d.dots.host;
}

void launch_scatter(Device &d, int count, const int32_t *idx, const double *val, double *dst) {
    if (count <= 0) return;
    k_scatter<<<(count + kBlock - 1) / kBlock, kBlock, 0, d.stream>>>(count, idx, val, dst);
    NSFEM_HIP(hipGetLastError());
}

void launch_gather(Device &d, int count, const int32_t *idx, const double *src, double *dst) {
    if (count <= 0) return;
    k_gather<<<(count + kBlock - 1) / kBlock, kBlock, 0, d.stream>>>(count, idx, src, dst);
    NSFEM_HIP(hipGetLastError());
}

void launch_scatter_value(Device &d, int count, const int32_t *idx, double v, double *dst) {
    if (count <= 0) return;
    k_scatter_value<<<(count + kBlock - 1) / kBlock, kBlock, 0, d.stream>>>(count, idx, v, dst);
    NSFEM_HIP(hipGetLastError());
}

void launch_scatter_value(Device &d, int count, const int32_t *idx, double v, float *dst) {
    if (count <= 0) return;
    k_scatter_value<<<(count + kBlock - 1) / kBlock, kBlock, 0, d.stream>>>(count, idx, (float)v,
                                                                            dst);
    NSFEM_HIP(hipGetLastError());
}

void launch_add(Device &d, int n, const double *a, double *y) {
    if (n <= 0) return;
    k_add<<<ew_grid(n), kBlock, 0, d.stream>>>(n, a, y);
    NSFEM_HIP(hipGetLastError());
}

void launch_jacobi0(Device &d, int n, double w, const double *dinv, const double *b, double *x) {
    if (n <= 0) return;
    k_jacobi0<<<ew_grid(n), kBlock, 0, d.stream>>>(n, w, dinv, b, x);
    NSFEM_HIP(hipGetLastError());
}

void launch_fill(Device &d, int n, double v, double *y) {
    if (n <= 0) return;
    k_fill<<<ew_grid(n), kBlock, 0, d.stream>>>(n, v, y);
    NSFEM_HIP(hipGetLastError());
}

void launch_fill(Device &d, int n, double v, float *y) {
    if (n <= 0) return;
    k_fill<<<ew_grid(n), kBlock, 0, d.stream>>>(n, (float)v, y);
    NSFEM_HIP(hipGetLastError());
}

void launch_convert(Device &d, int n, const double *a, float *y) {
    if (n <= 0) return;
    k_convert<<<ew_grid(n), kBlock, 0, d.stream>>>(n, a, y);
    NSFEM_HIP(hipGetLastError());
}

void launch_convert(Device &d, int n, const float *a, double *y) {
    if (n <= 0) return;
    k_convert<<<ew_grid(n), kBlock, 0, d.stream>>>(n, a, y);
    NSFEM_HIP(hipGetLastError());
}

void launch_copy(Device &d, int n, const double *a, double *y) {
    if (n <= 0) return;
    k_copy<<<ew_grid(n), kBlock, 0, d.stream>>>(n, a, y);
    NSFEM_HIP(hipGetLastError());
}

// =====================================================================
// Persistent conjugate gradient
// =====================================================================
//
// One cooperative launch runs a whole solve.  Each block owns a contiguous
// run of tiles (rows); per iteration there are two grid-wide reductions:
//
//   phase A  p_new = r + beta*p_old (owner rows, written),
//            q = A p_new, gathering r and p_old (p_new of a neighbour is
//            recomputed from them, bit-identically, so no extra barrier),
//            x += alpha_prev * p_old (the x update of the previous step,
//            deferred to here), delta += (p_new, q)        -> reduce delta
//   phase B  alpha = gamma/delta; r -= alpha q; gamma' += (r, r) -> reduce
//
// This is textbook CG (thesis Alg. CG; gpu/matrix_math.cu:256-286) with the
// reference's 4 grid barriers per iteration fused down to 2.
//
// Mixed precision (NSFEM_PRECISION_FP32_REFINED): the matrix values and the
// r, p, q vectors are FP32; products are accumulated in FP64 (an FP32 x FP32
// product is exact in FP64), every dot is accumulated in FP64, and the
// solution x is kept and updated in FP64.  The FP32 recursive residual is
// replaced by r = b - A x, computed in FP64 from the FP64 matrix and rounded
// to FP32, at "reliable updates" (Sleijpen & van der Vorst 1996): whenever
// ||r|| has fallen by reliable_delta since the last one (at least
// ru_min_gap iterations after it), after ru_gap
// iterations, or when the recurrence says the tolerance is met; the search
// direction is kept.  Convergence is decided only on that FP64 residual.
// Measured on the 2048^2 cavity pressure matrix: FP32 storage of x or FP32
// accumulation of the products each inflates the iteration count by 1.4-1.8x,
// and so do sparse reliable updates (reliable_delta 0.1: +33%); with x and
// the accumulations in FP64 and reliable_delta 0.5 the count equals FP64 CG's.
//
// Grid reduction of a solve over at most kFlatMax blocks: each block posts
// its partial sums and an epoch flag, then every block waits for all flags
// and adds all partials itself, in block order -- one write and one round of
// polling on the critical path, and every block holds the same bits.
// Larger grids use a tree: arrivals count on one counter per group of
// kGroup blocks, the last arrival of a group adds the group's partials in
// block order and arrives at the top counter, the last top arrival adds the
// group sums in group order and releases every group.  Either way the
// summation order is fixed, so results are deterministic.  Measured on the
// 512x128 channel's pressure matrix (65,656 rows), per reduction: flat
// 2.8-5.5 us against the tree's 5.1-10 us at 16-64 blocks, about even at
// 128, and the tree ahead at 256 (the flags of all blocks sit on a few
// cache lines that every block polls).

namespace {

constexpr int kGroup = 16;
constexpr int kMaxGroups = kMaxGridBlocks / kGroup;
constexpr int kFlatMax = 128;
constexpr int kResMaxBlocks = 256;  // blocks of a resident solve

struct alignas(256) SyncState {
    unsigned int arrive_top;
    unsigned int pad0[63];
    unsigned int abort;
    unsigned int pad1[63];
    unsigned int arrive_group[kMaxGroups][64];
    unsigned int release_group[kMaxGroups][64];
    double result[kMaxRed];
    double pad2[24];
    double gpartial[kMaxRed][kMaxGroups];
    double partial[kMaxRed][kMaxGridBlocks];
    // flat reduction: per block the last epoch whose partials are posted,
    // and the partials by epoch parity (a block overwrites a parity's slots
    // only after every block has posted the next epoch, i.e. has read them)
    unsigned int flag[kFlatMax];
    double fpart[2][kMaxRed][kFlatMax];
    // resident solves: per epoch parity, sum and block the two halves of the
    // block's partial sum, each tagged with the epoch
    unsigned long long tag[2][kMaxRed][kResMaxBlocks][2];
};

#ifdef NSFEM_CG_TRACE
// Phase timestamps of the first kTraceIters iterations (100 MHz wall clock):
// [0] block 0 iteration start, [1] latest phase A end over all blocks,
// [2] block 0 after the delta reduction, [3] latest phase B end,
// [4] block 0 after the gamma reduction.
constexpr int kTraceIters = 4096;
__device__ unsigned long long g_cg_trace[kTraceIters][5];
#define CG_TRACE_STAMP(it, slot)                                                    \
    do {                                                                            \
        if (threadIdx.x == 0 && (it) < kTraceIters && L == 0)                       \
            g_cg_trace[(it)][(slot)] = wall_clock64();                              \
    } while (0)
#define CG_TRACE_MAX(it, slot)                                                      \
    do {                                                                            \
        __syncthreads();                                                            \
        if (threadIdx.x == 0 && (it) < kTraceIters)                                 \
            atomicMax(&g_cg_trace[(it)][(slot)], (unsigned long long)wall_clock64()); \
    } while (0)
}  // namespace
// trace builds only: read / clear the phase timestamps
extern "C" int nsfem_trace_read(unsigned long long *out, int iters) {
    const int n = iters < kTraceIters ? iters : kTraceIters;
    if (hipMemcpyFromSymbol(out, HIP_SYMBOL(g_cg_trace), sizeof(unsigned long long) * 5 * n) !=
        hipSuccess)
        return -1;
    return n;
}
extern "C" int nsfem_trace_clear() {
    static unsigned long long zero[kTraceIters][5];
    return hipMemcpyToSymbol(HIP_SYMBOL(g_cg_trace), zero, sizeof(zero)) == hipSuccess ? 0 : -1;
}
namespace {
#else
#define CG_TRACE_STAMP(it, slot) \
    do {                         \
    } while (0)
#define CG_TRACE_MAX(it, slot) \
    do {                       \
    } while (0)
#endif

struct CgArgs {
    int n, nnz;
    const int4 *meta;  // wave tile descriptors
    const int32_t *tiles;
    const int32_t *block_tiles;
    const int32_t *rs;
    const int32_t *col;
    const int16_t *dcol;  // col - wave tile's first row (int16 kernels)
    const double *val64;
    const float *val32;
    const double *b;  // [NC][n]
    double *x;        // [NC][n]
    void *r, *p0, *p1, *q;  // interleaved [n][NC] (two-column solves)
    void *st[2];            // packed {r, p, q} rows of mixed solves
    int packed2;  // two-column mixed solves: 1 packed, 2 narrow-gather iteration (0 two-phase)
    double rtol, atol, rdelta;
    int max_iter, max_refine;
    int ru_gap;      // mixed: force a reliable update after this many iterations
    int ru_min_gap;  // mixed: no drop-triggered update sooner than this
    unsigned long long timeout_ticks;
    SyncState *sync;
    CgColumnResult *res;
    int nblocks;  // blocks of this solve (batched launches)
    int flat;     // flat grid reduction for solves of <= kFlatMax blocks
    // Jacobi scaling (mixed solves): 1/sqrt(diag A) per row, or null.  The
    // FP32 iteration runs on D^-1/2 A D^-1/2 (val32 holds it) with r, p, q
    // in that scaled space; x, b and the FP64 residual passes stay unscaled
    // (r_scaled = scale * (b - A x)), so convergence is decided on the
    // unscaled residual, as without scaling.
    const double *scale;
    // resident solves: the matrix's bandwidths below and above the diagonal,
    // and the most rows a block's window holds
    int band_lo, band_hi, win_cap;
};

// The FP64 step of x_row along the scaled search direction: x = D^-1/2 y.
__device__ __forceinline__ double x_step(const CgArgs &A, double pend, int row) {
    return A.scale ? pend * A.scale[row] : pend;
}

// Launched with at least kFlatMax threads; blocks > 0 clears that many blocks'
// tags too (a resident solve; a tag's epoch is never 0).
__global__ void k_sync_reset(SyncState *s, int ngroups, int blocks) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    for (int k = i; k < 4 * kMaxRed * blocks; k += gridDim.x * blockDim.x) {
        const int half = k & 1, b = (k >> 1) % blocks, j = (k >> 1) / blocks;
        s->tag[j / kMaxRed][j % kMaxRed][b][half] = 0ull;
    }
    if (i == 0) {
        s->arrive_top = 0;
        s->abort = 0;
    }
    if (i < kFlatMax) s->flag[i] = 0;
    if (i < ngroups) {
        s->arrive_group[i][0] = 0;
        s->release_group[i][0] = 0;
    }
}

__device__ __forceinline__ unsigned ld_acquire(const unsigned *p) {
    return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double ld_relaxed(const double *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Grid-wide sum of K values with barrier semantics.  Returns false if the
// barrier timed out or another block aborted (the caller must return).
// Memory ordering (gfx950: one L2 per XCD, not coherent across XCDs; an
// agent-scope release writes the L2 back, an agent-scope acquire invalidates
// it).  Every wave first waits for its own global stores to complete
// (s_waitcnt 0: the stores have reached its XCD's L2), the block
// synchronises, and then ONE thread per block performs the agent-scope
// release as part of its arrival (a single L2 write-back per block).  Waiting
// threads poll with relaxed agent-scope loads, which read the coherence
// point without touching the caches, and perform one acquire fence after the
// wait (a single invalidate per block), before the block reads data other
// blocks wrote.  The last arrival at a counter (the group's, then the top
// one) reads the counter's release sequence and performs an acquire fence
// before it adds the other blocks' partials.
//
// Flat form (nb <= kFlatMax): thread 0 posts the block's partials at the
// coherence point and then its flag with an agent-scope release (the
// block's stores, completed to L2 by every wave's s_waitcnt before the
// block barrier, are written back with it).  Wave 0 polls every block's
// flag with relaxed agent-scope loads, performs one acquire fence once all
// are posted, and adds the partials in block order (lane i takes blocks i,
// i + 64, ...; then a fixed butterfly), so every block computes the same
// sum.  A block posts epoch e + 1 only after its wave 0 has read epoch e's
// partials, which is what makes two parity slots enough.
template <int K, int BS>
__device__ bool grid_sum_flat(SyncState *S, double (&v)[K], const unsigned epoch,
                              unsigned long long timeout, const int b, const int nb) {
    static_assert(K <= kMaxRed, "reduction width");
    __shared__ double s_sum[K];
    __shared__ int s_ok;
    const int par = epoch & 1u;
    __builtin_amdgcn_s_waitcnt(0);  // this wave's stores are complete
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            __hip_atomic_store(&S->fpart[par][k][b], v[k], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&S->flag[b], epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        int ok = 1;
        const unsigned long long t0 = wall_clock64();
        for (;;) {
            bool mine = true;
            for (int i = lane; i < nb; i += 64)
                mine = mine && __hip_atomic_load(&S->flag[i], __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT) >= epoch;
            if (__all(mine)) break;
            if (__any(__hip_atomic_load(&S->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) !=
                      0u)) {
                ok = 0;
                break;
            }
            if (wall_clock64() - t0 > timeout) {
                if (lane == 0)
                    __hip_atomic_store(&S->abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                ok = 0;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#pragma unroll
        for (int k = 0; k < K; ++k) {
            double t = 0.0;
            for (int i = lane; i < nb; i += 64) t += ld_relaxed(&S->fpart[par][k][i]);
            t = wave_sum(t);
            if (lane == 0) s_sum[k] = t;
        }
        if (lane == 0) s_ok = ok;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = s_sum[k];
    return s_ok != 0;
}

template <int K, int BS>
__device__ bool grid_sum(SyncState *S, double (&v)[K], unsigned &epoch, double *lds,
                         unsigned long long timeout, const int b, const int nb, const bool flat) {
    // Each flag is written by thread 0 before a __syncthreads and read by
    // the block after it; none is rewritten until the next call, which
    // every thread reaches only after passing several more barriers.
    __shared__ int s_group_last, s_top_last, s_ok;
    block_sum<K, BS>(v, lds);
    if (flat && nb <= kFlatMax) return grid_sum_flat<K, BS>(S, v, ++epoch, timeout, b, nb);
    const int g = b / kGroup;
    const int ng = (nb + kGroup - 1) / kGroup;
    const int gsize = min(kGroup, nb - g * kGroup);
    ++epoch;
    __builtin_amdgcn_s_waitcnt(0);  // this wave's stores are complete
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) S->partial[k][b] = v[k];
        const unsigned prev = __hip_atomic_fetch_add(&S->arrive_group[g][0], 1u, __ATOMIC_RELEASE,
                                                     __HIP_MEMORY_SCOPE_AGENT);
        const bool last = prev == epoch * (unsigned)gsize - 1u;
        // the last arrival read the counter's release sequence (every
        // member's release RMW): an acquire fence after it synchronises with
        // all of them before the block reads their partials (the block
        // barrier below carries the order to the reading threads)
        if (last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        s_group_last = last ? 1 : 0;
    }
    __syncthreads();
    if (s_group_last) {
        // group sum, members in block order (lane i of wave 0 holds member i);
        // the partials are read at the coherence point
        double gs[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            double t = 0.0;
            if (threadIdx.x < gsize) t = ld_relaxed(&S->partial[k][g * kGroup + threadIdx.x]);
            gs[k] = threadIdx.x < 64 ? wave_sum(t) : 0.0;
        }
        if (threadIdx.x == 0) {
#pragma unroll
            for (int k = 0; k < K; ++k)
                __hip_atomic_store(&S->gpartial[k][g], gs[k], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            const unsigned prev = __hip_atomic_fetch_add(&S->arrive_top, 1u, __ATOMIC_RELEASE,
                                                         __HIP_MEMORY_SCOPE_AGENT);
            const bool last = prev == epoch * (unsigned)ng - 1u;
            if (last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // as above
            s_top_last = last ? 1 : 0;
        }
        __syncthreads();
        if (s_top_last) {
            double ts[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                double acc = 0.0;
                for (int i = threadIdx.x; i < ng; i += BS) acc += ld_relaxed(&S->gpartial[k][i]);
                ts[k] = acc;
            }
            block_sum<K, BS>(ts, lds);
            if (threadIdx.x == 0) {
#pragma unroll
                for (int k = 0; k < K; ++k)
                    __hip_atomic_store(&S->result[k], ts[k], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            }
            __syncthreads();
            for (int i = threadIdx.x; i < ng; i += BS)
                __hip_atomic_store(&S->release_group[i][0], epoch, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // wait for the release of this block's group (bounded)
    if (threadIdx.x == 0) {
        int ok = 1;
        const unsigned long long t0 = wall_clock64();
        while (__hip_atomic_load(&S->release_group[g][0], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT) < epoch) {
            if (__hip_atomic_load(&S->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                ok = 0;
                break;
            }
            if (wall_clock64() - t0 > timeout) {
                __hip_atomic_store(&S->abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                ok = 0;
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        s_ok = ok;
    }
    __syncthreads();
    const bool ok = s_ok != 0;
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = ld_relaxed(&S->result[k]);
    return ok;
}

template <int NC, typename T>
struct VecN {
    T v[NC];
};

template <int NC, typename T>
__device__ __forceinline__ VecN<NC, T> ldv(const T *p, int i) {
    VecN<NC, T> o;
    if constexpr (NC == 1) {
        o.v[0] = p[i];
    } else if constexpr (std::is_same<T, double>::value) {
        const double2 t = reinterpret_cast<const double2 *>(p)[i];
        o.v[0] = t.x;
        o.v[1] = t.y;
    } else {
        const float2 t = reinterpret_cast<const float2 *>(p)[i];
        o.v[0] = t.x;
        o.v[1] = t.y;
    }
    return o;
}

template <int NC, typename T>
__device__ __forceinline__ void stv(T *p, int i, const VecN<NC, T> &o) {
    if constexpr (NC == 1) {
        p[i] = o.v[0];
    } else if constexpr (std::is_same<T, double>::value) {
        reinterpret_cast<double2 *>(p)[i] = make_double2(o.v[0], o.v[1]);
    } else {
        reinterpret_cast<float2 *>(p)[i] = make_float2(o.v[0], o.v[1]);
    }
}

// ---------------------------------------------------------------------
// Wave tiles: the persistent CG partitions rows into tiles of at most 64
// rows and kWaveNnz nonzeros; each wavefront stages its own tile through
// its own LDS region (no block-wide synchronisation inside a phase), so the
// 16 waves of a block overlap their memory latencies independently.
constexpr int kWItems = kWaveNnz / 64;  // nonzeros per lane per tile

struct WTile {
    int r0, r1, k0, nz;
};

// Sum of a row's products p[ra..rb) in column order, four LDS reads in
// flight at a time (the adds stay sequential: bit-identical to one by one).
__device__ __forceinline__ double row_sum(const double *p, int ra, int rb) {
    double s = 0.0;
    int k = ra;
    for (; k + 4 <= rb; k += 4) {
        const double a0 = p[k], a1 = p[k + 1], a2 = p[k + 2], a3 = p[k + 3];
        s += a0;
        s += a1;
        s += a2;
        s += a3;
    }
    for (; k < rb; ++k) s += p[k];
    return s;
}

// The same for NC interleaved columns (products [k][NC]), added to s[c];
// two nonzeros' products in flight at a time, each column in column order.
template <int NC>
__device__ __forceinline__ void row_sums(const double *p, int ra, int rb, double (&s)[NC]) {
    if constexpr (NC == 1) {
        s[0] += row_sum(p, ra, rb);
    } else {
        int k = ra;
        for (; k + 2 <= rb; k += 2) {
            double a[2][NC];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int c = 0; c < NC; ++c) a[j][c] = p[(k + j) * NC + c];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int c = 0; c < NC; ++c) s[c] += a[j][c];
        }
        for (; k < rb; ++k)
#pragma unroll
            for (int c = 0; c < NC; ++c) s[c] += p[k * NC + c];
    }
}

// Tile metadata: read from global memory, or from the block's copy in LDS
// (MetaLds: indexed from the block's first tile), which keeps the per-tile
// descriptor read out of the vector-memory counter the gathers wait on.
// The LDS copy holds {first row, first nonzero} of the block's tiles and of
// one past its last (a tile ends where the next begins).
struct MetaLds {
    const int2 *m;
    int t0;
};
__device__ __forceinline__ WTile wave_tile(const int4 *meta, int t);
__device__ __forceinline__ WTile wave_tile(const MetaLds &meta, int t) {
    const int2 a = meta.m[t - meta.t0], b = meta.m[t - meta.t0 + 1];
    WTile w;
    w.r0 = __builtin_amdgcn_readfirstlane(a.x);
    w.r1 = __builtin_amdgcn_readfirstlane(b.x);
    w.k0 = __builtin_amdgcn_readfirstlane(a.y);
    w.nz = __builtin_amdgcn_readfirstlane(b.y) - w.k0;
    return w;
}

// Copy tiles T0 .. T1 - 1 of the block's descriptors (T1 > T0) into `lds`
// as MetaLds entries, T1 - T0 + 1 of them.
template <int BS>
__device__ __forceinline__ void load_meta_lds(const int4 *meta, int T0, int T1, int2 *lds) {
    for (int i = threadIdx.x; i <= T1 - T0; i += BS) {
        const int4 m = meta[i < T1 - T0 ? T0 + i : T1 - 1];
        lds[i] = i < T1 - T0 ? make_int2(m.x, m.z) : make_int2(m.y, m.z + m.w);
    }
    __syncthreads();
}

__device__ __forceinline__ WTile wave_tile(const int4 *meta, int t) {
    const int4 m = meta[t];
    WTile w;
    w.r0 = __builtin_amdgcn_readfirstlane(m.x);
    w.r1 = __builtin_amdgcn_readfirstlane(m.y);
    w.k0 = __builtin_amdgcn_readfirstlane(m.z);
    w.nz = __builtin_amdgcn_readfirstlane(m.w);
    return w;
}

// One-column mixed solves keep each row's FP32 CG state packed as {r, p, q}
// in 12 bytes, so that one dwordx3 gather brings everything a neighbour
// contributes.  A wave64 gather costs the same return-path time whatever its
// width per lane, so one wide gather replaces the two narrow ones (r, p) of
// the two-phase iteration.  (The solution stays FP64 and is updated every
// iteration: an FP32 accumulator between reliable updates, multiplied by an
// ill-conditioned A, pollutes the true residual at ~eps32 * cond(A) of its
// last level and cost the 2048^2 cavity's pressure solve 50% more
// iterations.)
struct alignas(4) RowState {
    float r, p, q;
};

__device__ __forceinline__ RowState ld_state(const void *st, int i) {
    return reinterpret_cast<const RowState *>(st)[i];
}
__device__ __forceinline__ void st_state(void *st, int i, const RowState &v) {
    reinterpret_cast<RowState *>(st)[i] = v;
}

// Two-column mixed solves keep both columns' FP32 {r, p} of a row in one
// 16-byte word {r0, r1, p0, p1} and their q in an 8-byte word {q0, q1}: a
// state copy holds the n words of the first kind, then the n of the second.
// A neighbour's contribution to both columns takes two gathers.
__device__ __forceinline__ float4 *st2_rp(void *st) { return reinterpret_cast<float4 *>(st); }
__device__ __forceinline__ const float4 *st2_rp(const void *st) {
    return reinterpret_cast<const float4 *>(st);
}
__device__ __forceinline__ float2 *st2_q(void *st, int n) {
    return reinterpret_cast<float2 *>(reinterpret_cast<float4 *>(st) + n);
}
__device__ __forceinline__ const float2 *st2_q(const void *st, int n) {
    return reinterpret_cast<const float2 *>(reinterpret_cast<const float4 *>(st) + n);
}

// Column word of nonzero k: the column (IT = int32_t) or its offset from the
// first row of the nonzero's wave tile (IT = int16_t).
template <typename IT>
__device__ __forceinline__ int col_word(const CgArgs &A, int k) {
    if constexpr (std::is_same<IT, int16_t>::value)
        return (int)ld_stream(A.dcol + k);
    else
        return ld_stream(A.col + k);
}
// Column from a column word of a wave tile whose first row is r0.
template <typename IT>
__device__ __forceinline__ int col_of(int word, int r0) {
    if constexpr (std::is_same<IT, int16_t>::value)
        return r0 + word;
    else
        return word;
}
template <typename IT>
__device__ __forceinline__ int col_at(const CgArgs &A, int r0, int k) {
    return col_of<IT>(col_word<IT>(A, k), r0);
}

// FP64 residual over the block's wave tiles: r = b - A x (x column-major).
// SETUP: also p_old = 0 and b.b.
// Accumulates per column: acc[c] = r.r (FP64), acc[NC+c] = b.b,
// acc[2NC+c] = (FP32 r).(FP32 r).
// PACKED (one-column mixed solves): r goes to the packed state `st`; SETUP
// also clears its p and q.
template <int NC, int BS, bool MIXED, bool SETUP, typename IT, bool PACKED = false,
          typename MP = const int4 *>
__device__ void residual_phase(const CgArgs &A, MP meta, int T0, int T1, double *lds_wave,
                               double (&acc)[3 * NC], void *st = nullptr) {
    static_assert(!PACKED || ((NC == 1 || NC == 2) && MIXED), "packed state: FP32 columns");
    using VT = typename std::conditional<MIXED, float, double>::type;
    constexpr int NW = BS / 64;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    VT *r = (VT *)A.r;
    VT *pold = (VT *)A.p0;
    for (int t = T0 + wave; t < T1; t += NW) {
        const WTile w = wave_tile(meta, t);
        const int row = w.r0 + lane;
        const bool has_row = row < w.r1;
        const int rowc = has_row ? row : w.r0;
        double s[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) s[c] = 0.0;
        double bb[NC];
        int ra = A.rs[rowc] - w.k0;
        int rb = A.rs[rowc + 1] - w.k0;
#pragma unroll
        for (int c = 0; c < NC; ++c) bb[c] = A.b[(size_t)c * A.n + rowc];
        if (!has_row) rb = ra;
        if (w.nz <= kWaveNnz) {
            // Branch-free staging: out-of-tile lanes read index 0 of the
            // column/value arrays (always allocated) and gather x[0] (the
            // matrix has >= 1 column); their products are zeroed and never
            // summed.  All loads of a batch issue back to back.
            constexpr int IB = (NC == 2 || MIXED) ? 4 : kWItems;  // register budget
#pragma unroll
            for (int i0 = 0; i0 < kWItems; i0 += IB) {
                int cj[IB];
                double vj[IB];
#pragma unroll
                for (int i = 0; i < IB; ++i) {
                    const int k = lane + 64 * (i0 + i);
                    const bool ok = k < w.nz;
                    const int idx = ok ? w.k0 + k : 0;
                    const int cc = col_at<IT>(A, w.r0, idx);
                    const double vv = A.val64[idx];
                    cj[i] = ok ? cc : 0;
                    vj[i] = ok ? vv : 0.0;
                }
#pragma unroll
                for (int i = 0; i < IB; ++i) {
                    const int k = lane + 64 * (i0 + i);
#pragma unroll
                    for (int c = 0; c < NC; ++c)
                        lds_wave[k * NC + c] = vj[i] * A.x[(size_t)c * A.n + cj[i]];
                }
            }
            __syncwarp();
            if (has_row) row_sums<NC>(lds_wave, ra, rb, s);
            __syncwarp();
        } else {  // a single row longer than a tile: wave-wide sum
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                double part = 0.0;
                for (int k = lane; k < w.nz; k += 64)
                    part += A.val64[w.k0 + k] *
                            A.x[(size_t)c * A.n + col_at<IT>(A, w.r0, w.k0 + k)];
                s[c] = wave_sum(part);
            }
        }
        if (has_row) {
            VecN<NC, VT> rv, zero;
            const double sc = A.scale ? A.scale[row] : 1.0;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const double rr = bb[c] - s[c];
                acc[c] += rr * rr;
                if (SETUP) acc[NC + c] += bb[c] * bb[c];
                rv.v[c] = (VT)(A.scale ? rr * sc : rr);
                if (MIXED) acc[2 * NC + c] += (double)rv.v[c] * (double)rv.v[c];
                zero.v[c] = (VT)0;
            }
            if constexpr (PACKED && NC == 1) {
                if constexpr (SETUP)
                    st_state(st, row, RowState{(float)rv.v[0], 0.f, 0.f});
                else
                    reinterpret_cast<RowState *>(st)[row].r = (float)rv.v[0];
            } else if constexpr (PACKED) {
                float4 *rp = st2_rp(st);
                if constexpr (SETUP) {
                    rp[row] = make_float4((float)rv.v[0], (float)rv.v[1], 0.f, 0.f);
                    st2_q(st, A.n)[row] = make_float2(0.f, 0.f);
                } else {
                    reinterpret_cast<float2 *>(rp + row)[0] =
                        make_float2((float)rv.v[0], (float)rv.v[1]);
                }
            } else {
                stv<NC, VT>(r, row, rv);
                if (SETUP) {
                    stv<NC, VT>(pold, row, zero);
                }
            }
        }
    }
}

// Phase A over the block's wave tiles:
//   p_new = r + beta p_old (owner rows), q = A p_new (gathering r, p_old),
//   deferred FP64 solution update x += pend * p_old, delta += (p_new, q).
// The products and row sums accumulate in FP64 in both precisions (the
// product of two FP32 numbers is exact in FP64); only q is stored as VT.
template <int NC, int BS, bool MIXED, typename IT, typename MP>
__device__ void phase_a(const CgArgs &A, MP meta, int T0, int T1, double *lds_wave,
                        const typename std::conditional<MIXED, float, double>::type *pold,
                        typename std::conditional<MIXED, float, double>::type *pnew,
                        const typename std::conditional<MIXED, float, double>::type (&beta)[NC],
                        const double (&pend)[NC], bool has_pend, double (&delta)[NC]) {
    using VT = typename std::conditional<MIXED, float, double>::type;
    using MT = VT;
    constexpr int NW = BS / 64;
    const MT *val = MIXED ? (const MT *)A.val32 : (const MT *)A.val64;
    const VT *r = (const VT *)A.r;
    VT *q = (VT *)A.q;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int t = T0 + wave;
    if (t >= T1) return;
    // Software pipeline: the column indices of the next tile load while the
    // current tile's values and gathers are in flight.  Lanes beyond a
    // tile's nonzeros read entry 0 of the column/value arrays (a valid
    // column: upload makes col[0] = 0 for an empty matrix); their products
    // land in LDS slots that no row sum reads, so no loaded value is masked
    // and no load has to be waited for before the products are staged.
    // The prefetched words stay raw until the tile is consumed (no ALU use
    // of a load in flight).  Lanes beyond the tile read its first nonzero
    // (a valid column of the tile); a tile without nonzeros gathers nothing.
    // Item slices wholly beyond a tile's nonzeros issue no loads (a 64-row
    // tile of a 7-point matrix fills 7 of its 8 slices): 5% faster here.
    WTile w = wave_tile(meta, t);
    int cn[kWItems];
    {
        const int kf = w.nz > 0 ? w.k0 : 0;
#pragma unroll
        for (int i = 0; i < kWItems; ++i) {
            const int k = lane + 64 * i;
            cn[i] = 64 * i < w.nz ? col_word<IT>(A, k < w.nz ? w.k0 + k : kf) : 0;
        }
    }
    for (; t < T1; t += NW) {
        const WTile cur = w;
        int cj[kWItems];
#pragma unroll
        for (int i = 0; i < kWItems; ++i) cj[i] = col_of<IT>(cn[i], cur.r0);
        // 1. next tile: descriptor and column words
        const int tn = t + NW;
        if (tn < T1) {
            w = wave_tile(meta, tn);
            const int kf = w.nz > 0 ? w.k0 : 0;
#pragma unroll
            for (int i = 0; i < kWItems; ++i) {
                const int k = lane + 64 * i;
                cn[i] = 64 * i < w.nz ? col_word<IT>(A, k < w.nz ? w.k0 + k : kf) : 0;
            }
        }
        // 2. owner rows (clamped so the loads stay unconditional)
        const int row = cur.r0 + lane;
        const bool has_row = row < cur.r1;
        const int rowc = has_row ? row : cur.r0;
        const int rsa = A.rs[rowc];
        const int rsb = A.rs[rowc + 1];
        const VecN<NC, VT> rv = ldv<NC, VT>(r, rowc);
        const VecN<NC, VT> pv = ldv<NC, VT>(pold, rowc);
        double xo[NC];
        if (has_pend) {
#pragma unroll
            for (int c = 0; c < NC; ++c) xo[c] = A.x[(size_t)c * A.n + rowc];
        }
        double s[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) s[c] = 0.0;
        if (cur.nz == 0) {
            // rows without nonzeros: q = 0
        } else if (cur.nz <= kWaveNnz) {
            // 3. values and gathers, then one wait for the whole tile
            constexpr int IB = (NC == 2) ? 4 : kWItems;  // register budget
#pragma unroll
            for (int i0 = 0; i0 < kWItems; i0 += IB) {
                if (64 * i0 >= cur.nz) break;
                MT vj[IB];
                VecN<NC, VT> rj[IB], pj[IB];
#pragma unroll
                for (int i = 0; i < IB; ++i) {
                    const int k = lane + 64 * (i0 + i);
                    if (64 * (i0 + i) < cur.nz) {
                        vj[i] = ld_stream(val + (k < cur.nz ? cur.k0 + k : 0));
                        rj[i] = ldv<NC, VT>(r, cj[i0 + i]);
                        pj[i] = ldv<NC, VT>(pold, cj[i0 + i]);
                    } else {
                        vj[i] = (MT)0;
#pragma unroll
                        for (int c = 0; c < NC; ++c) rj[i].v[c] = pj[i].v[c] = (VT)0;
                    }
                }
#pragma unroll
                for (int i = 0; i < IB; ++i) {
                    const int k = lane + 64 * (i0 + i);
                    if (64 * (i0 + i) < cur.nz) {
#pragma unroll
                        for (int c = 0; c < NC; ++c)
                            lds_wave[k * NC + c] =
                                (double)vj[i] * (double)fma_t<VT>(beta[c], pj[i].v[c], rj[i].v[c]);
                    }
                }
            }
            __syncwarp();
            const int ra = rsa - cur.k0;
            const int rb = has_row ? rsb - cur.k0 : ra;
            row_sums<NC>(lds_wave, ra, rb, s);
            __syncwarp();
        } else {
            // a single row longer than a tile: wave-wide sum
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                double part = 0.0;
                for (int k = lane; k < cur.nz; k += 64) {
                    const int j = col_at<IT>(A, cur.r0, cur.k0 + k);
                    const VecN<NC, VT> rjj = ldv<NC, VT>(r, j);
                    const VecN<NC, VT> pjj = ldv<NC, VT>(pold, j);
                    part += (double)val[cur.k0 + k] *
                            (double)fma_t<VT>(beta[c], pjj.v[c], rjj.v[c]);
                }
                s[c] = wave_sum(part);
            }
        }
        if (has_row) {
            VecN<NC, VT> pn, qq;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                pn.v[c] = fma_t<VT>(beta[c], pv.v[c], rv.v[c]);
                qq.v[c] = (VT)s[c];
                delta[c] += (double)pn.v[c] * s[c];
            }
            stv<NC, VT>(pnew, row, pn);
            stv<NC, VT>(q, row, qq);
            if (has_pend) {
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    A.x[(size_t)c * A.n + row] =
                        __builtin_fma(x_step(A, pend[c], row), (double)pv.v[c], xo[c]);
            }
        }
    }
}

// Phase B over the block's rows: r -= alpha q, g += (r, r); rows are
// processed 4 per thread with all loads issued first.
template <int NC, int BS, typename VT>
__device__ void phase_b(const CgArgs &A, int R0, int R1, const VT (&alpha)[NC], double (&g)[NC]) {
    VT *r = (VT *)A.r;
    const VT *q = (const VT *)A.q;
    constexpr int U = 4;
    for (int base = R0 + (int)threadIdx.x; base < R1; base += U * BS) {
        VecN<NC, VT> rv[U], qv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {  // clamped rows keep the loads unconditional
            const int row = min(base + u * BS, R1 - 1);
            rv[u] = ldv<NC, VT>(r, row);
            qv[u] = ldv<NC, VT>(q, row);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int row = base + u * BS;
            if (row < R1) {
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    rv[u].v[c] = fma_t<VT>(-alpha[c], qv[u].v[c], rv[u].v[c]);
                    g[c] += (double)rv[u].v[c] * (double)rv[u].v[c];
                }
                stv<NC, VT>(r, row, rv[u]);
            }
        }
    }
}

// x += pend p over the block's rows (FP64 solution, p in VT)
template <int NC, int BS, typename VT>
__device__ void flush_x(const CgArgs &A, int R0, int R1, const VT *p, const double (&pend)[NC]) {
    for (int row = R0 + (int)threadIdx.x; row < R1; row += BS) {
        const VecN<NC, VT> pv = ldv<NC, VT>(p, row);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            double *xp = A.x + (size_t)c * A.n + row;
            *xp = __builtin_fma(x_step(A, pend[c], row), (double)pv.v[c], *xp);
        }
    }
}

// The persistent CG run by one block of a solve that owns `nb` blocks: `bid`
// is the block's index among them (reduction slots), `L` its logical index
// (tile ownership).  prod_raw / lds are the block's LDS.
template <int NC, int BS, bool MIXED, typename IT, typename MP>
__device__ __forceinline__ void cg_body_m(const CgArgs &A, MP meta, const int bid, const int nb,
                                          const int L, double *prod_raw, double *lds) {
    using VT = typename std::conditional<MIXED, float, double>::type;
    const int T0 = A.block_tiles[L], T1 = A.block_tiles[L + 1];
    const int R0 = A.tiles[T0], R1 = A.tiles[T1];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double *lds64 = prod_raw + wave * kWaveNnz * NC;
    VT *pbuf[2] = {(VT *)A.p0, (VT *)A.p1};
    unsigned epoch = 0;
    const bool writer = (L == 0 && threadIdx.x == 0);

    // ------------------------------------------------------------ setup
    double acc[3 * NC];
#pragma unroll
    for (int k = 0; k < 3 * NC; ++k) acc[k] = 0.0;
    residual_phase<NC, BS, MIXED, true, IT, false, MP>(A, meta, T0, T1, lds64, acc);
    if (!grid_sum<3 * NC, BS>(A.sync, acc, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
    {
        double tol2[NC], gamma[NC], rmax2[NC], rho[NC];
        bool active[NC];
        int iters[NC], status[NC], refines = 0;
        VT beta[NC];
        double pend[NC];
        double last_rr[NC];
        bool any = false;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const double bn = sqrt(acc[NC + c]), r0n = sqrt(acc[c]);
            const double ref = bn > 0.0 ? bn : r0n;
            const double tol = fmax(A.rtol * ref, A.atol);
            tol2[c] = tol * tol;
            active[c] = acc[c] > tol2[c];
            any = any || active[c];
            gamma[c] = MIXED ? acc[2 * NC + c] : acc[c];
            // the drop triggers compare the recursion with the true residual
            // in the iteration's (scaled) space; rho converts a scaled norm
            // into the unscaled one the tolerance is on
            rmax2[c] = A.scale ? acc[2 * NC + c] : acc[c];
            rho[c] = A.scale && acc[2 * NC + c] > 0.0 ? acc[c] / acc[2 * NC + c] : 1.0;
            last_rr[c] = acc[c];
            iters[c] = 0;
            status[c] = NSFEM_OK;
            beta[c] = (VT)0;
            pend[c] = 0.0;
            if (writer) {
                A.res[c].rhs_norm = bn;
                A.res[c].initial_residual = r0n;
                A.res[c].tolerance = tol;
            }
        }
        int k = 0;
        int cur = 0;  // pbuf[cur] = p_old
        bool has_pend = false;
        int last_ru = 0;
        int stall[NC];
        double ru_rr[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            stall[c] = 0;
            ru_rr[c] = acc[c];
        }
        while (any) {
            VT *pold = pbuf[cur];
            VT *pnew = pbuf[cur ^ 1];
            double delta[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) delta[c] = 0.0;
            CG_TRACE_STAMP(k, 0);
            phase_a<NC, BS, MIXED, IT, MP>(A, meta, T0, T1, lds64, pold, pnew, beta, pend, has_pend, delta);
            CG_TRACE_MAX(k, 1);
            if (!grid_sum<NC, BS>(A.sync, delta, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
            CG_TRACE_STAMP(k, 2);
            double alpha[NC];
            VT alpha_v[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                alpha[c] = 0.0;
                if (active[c]) {
                    if (!(delta[c] > 0.0)) {
                        status[c] = NSFEM_BREAKDOWN;
                        active[c] = false;
                    } else {
                        alpha[c] = gamma[c] / delta[c];
                    }
                }
                alpha_v[c] = (VT)alpha[c];
            }
            double g[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) g[c] = 0.0;
            phase_b<NC, BS, VT>(A, R0, R1, alpha_v, g);
            CG_TRACE_MAX(k, 3);
            if (!grid_sum<NC, BS>(A.sync, g, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
            CG_TRACE_STAMP(k, 4);
            ++k;
            bool want_ru = false;
            bool dropped[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                dropped[c] = false;
                if (active[c]) {
                    iters[c] = k;
                    if (MIXED) {
                        // a drop by rdelta triggers the update once
                        // ru_min_gap iterations have passed, a drop by
                        // rdelta^2 at once (FP32 rounding must not pile up
                        // over a steep fall of the residual)
                        const double d2 = A.rdelta * A.rdelta;
                        dropped[c] = g[c] * rho[c] <= tol2[c] ||
                                     (g[c] < d2 * rmax2[c] &&
                                      (k - last_ru >= A.ru_min_gap || g[c] < d2 * d2 * rmax2[c]));
                        want_ru = want_ru || dropped[c];
                    } else if (g[c] <= tol2[c]) {
                        active[c] = false;  // its last update is still pending
                        last_rr[c] = g[c];
                    }
                }
                pend[c] = alpha[c];
            }
            has_pend = true;
            const bool out_of_iters = k >= A.max_iter;
            if (MIXED && k - last_ru >= A.ru_gap) want_ru = true;
            if (MIXED && (want_ru || out_of_iters)) {
                last_ru = k;
                // apply the pending x += alpha p_new (FP64), recompute r
                flush_x<NC, BS, VT>(A, R0, R1, pnew, pend);
                has_pend = false;
#pragma unroll
                for (int c = 0; c < NC; ++c) pend[c] = 0.0;
                double dummy[1] = {0.0};
                if (!grid_sum<1, BS>(A.sync, dummy, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
                double ra[3 * NC];
#pragma unroll
                for (int kk = 0; kk < 3 * NC; ++kk) ra[kk] = 0.0;
                residual_phase<NC, BS, MIXED, false, IT, false, MP>(A, meta, T0, T1, lds64, ra);
                if (!grid_sum<3 * NC, BS>(A.sync, ra, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
                ++refines;
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    last_rr[c] = ra[c];
                    if (active[c]) {
                        if (ra[c] <= tol2[c]) {
                            active[c] = false;
                        } else {
                            g[c] = ra[2 * NC + c];
                            rmax2[c] = A.scale ? ra[2 * NC + c] : ra[c];
                            rho[c] = A.scale && ra[2 * NC + c] > 0.0 ? ra[c] / ra[2 * NC + c]
                                                                     : 1.0;
                            // when the recursion reports a drop by rdelta,
                            // the FP64 residual must fall below
                            // (1 + rdelta)/2 of its best value so far; three
                            // misses in a row end the FP32 iteration for
                            // this column (an update forced by ru_gap alone
                            // is not judged)
                            if (dropped[c]) {
                                const double s = 0.5 * (1.0 + A.rdelta);
                                stall[c] = ra[c] > s * s * ru_rr[c] ? stall[c] + 1 : 0;
                            }
                            ru_rr[c] = fmin(ru_rr[c], ra[c]);
                            if (stall[c] >= 3) {
                                status[c] = NSFEM_STAGNATION;
                                active[c] = false;
                            }
                        }
                    }
                }
                if (refines >= A.max_refine) {
#pragma unroll
                    for (int c = 0; c < NC; ++c)
                        if (active[c]) {
                            status[c] = NSFEM_MAX_ITERATIONS_REACHED;
                            active[c] = false;
                        }
                }
            }
            any = false;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if (active[c] && out_of_iters) {
                    status[c] = NSFEM_MAX_ITERATIONS_REACHED;
                    active[c] = false;
                    last_rr[c] = g[c];
                }
                any = any || active[c];
                beta[c] = active[c] ? (VT)(g[c] / gamma[c]) : (VT)0;
                if (active[c]) gamma[c] = g[c];
            }
            if (!any) {
                // flush the pending x update of the last iteration
                if (has_pend) flush_x<NC, BS, VT>(A, R0, R1, pnew, pend);
                break;
            }
            cur ^= 1;
        }
        if (writer) {
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                A.res[c].iterations = iters[c];
                A.res[c].refinements = refines;
                A.res[c].status = status[c];
                A.res[c].last_residual = sqrt(last_rr[c]);
            }
        }
        return;
    }
timeout:
    if (writer) {
        for (int c = 0; c < NC; ++c) A.res[c].status = NSFEM_BARRIER_TIMEOUT;
    }
}

// Tile descriptors of a block: copied into LDS once per launch when they fit
// (one-column solves; the two-column solves' product slices fill the LDS).
// 4096 tiles cover the 2048^2 cavity's P2 matrices on 256 blocks (~2,500
// tiles each).
constexpr int kMetaLds = 4096;

template <int NC, int BS, bool MIXED, typename IT>
__device__ __forceinline__ void cg_body(const CgArgs &A, const int bid, const int nb, const int L,
                                        double *prod_raw, double *lds) {
    if constexpr (NC == 1) {
        __shared__ int2 tmeta[kMetaLds + 1];
        const int T0 = A.block_tiles[L], T1 = A.block_tiles[L + 1];
        if (T1 > T0 && T1 - T0 <= kMetaLds) {
            load_meta_lds<BS>(A.meta, T0, T1, tmeta);
            cg_body_m<NC, BS, MIXED, IT>(A, MetaLds{tmeta, T0}, bid, nb, L, prod_raw, lds);
            return;
        }
    }
    cg_body_m<NC, BS, MIXED, IT>(A, A.meta, bid, nb, L, prod_raw, lds);
}

// ---------------------------------------------------------------------
// One-column mixed solves: single-reduction iteration over the packed FP32
// row state.
//
// With r_{k-1}, p_{k-1}, q_{k-1} = A p_{k-1} of the last phase, one fused
// phase forms, over the block's wave tiles,
//   r_k = r_{k-1} - alpha q_{k-1},  p_k = r_k + beta p_{k-1}  (owner rows),
//   q_k = A p_k, each neighbour's p_k recomputed from its gathered state by
//   the same two roundings as its owner's (products summed in FP64),
//   the deferred FP64 solution update x += pend p_{k-1},
// and the FP64 sums (p_k, q_k), (r_k, r_k), (r_k, q_k), (q_k, q_k), all in one
// grid reduction: gamma_{k+1} = (r,r) - 2 alpha (r,q) + alpha^2 (q,q) gives
// beta_{k+1} without a second reduction (Meurant's single-synchronisation
// form of Hestenes-Stiefel CG, equal to it in exact arithmetic).  The state
// of step k goes to the other buffer, so no block overwrites rows that
// another still gathers.  (The streaming FP64 solve keeps the two-phase
// iteration: its packed state would need two gathers per nonzero, and
// measured slower.)
__device__ __forceinline__ float next_r(float alpha, float r, float q) {
    return __builtin_fmaf(-alpha, q, r);
}

// WI: nonzeros per lane per tile (the host's bound on every multi-row tile's
// nonzeros over 64); a single longer row is summed wave-wide.
template <int BS, typename IT, int WI, typename MP>
__device__ void phase_f1(const CgArgs &A, MP meta, int T0, int T1, double *lds_wave,
                         const void *st_old,
                         void *st_new, const float alpha, const float beta, const double pend,
                         const bool has_pend, double (&sums)[4]) {
    constexpr int NW = BS / 64;
    const float *val = A.val32;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int t = T0 + wave;
    if (t >= T1) return;
    // column words of the next tile stay raw until the tile is consumed;
    // lanes beyond a tile read its first nonzero (a valid column)
    WTile w = wave_tile(meta, t);
    int cn[WI];
    {
        const int kf = w.nz > 0 ? w.k0 : 0;
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            const int k = lane + 64 * i;
            cn[i] = col_word<IT>(A, k < w.nz ? w.k0 + k : kf);
        }
    }
    for (; t < T1; t += NW) {
        const WTile cur = w;
        int cj[WI];
#pragma unroll
        for (int i = 0; i < WI; ++i) cj[i] = col_of<IT>(cn[i], cur.r0);
        const int tn = t + NW;
        if (tn < T1) {
            w = wave_tile(meta, tn);
            const int kf = w.nz > 0 ? w.k0 : 0;
#pragma unroll
            for (int i = 0; i < WI; ++i) {
                const int k = lane + 64 * i;
                cn[i] = col_word<IT>(A, k < w.nz ? w.k0 + k : kf);
            }
        }
        const int row = cur.r0 + lane;
        const bool has_row = row < cur.r1;
        const int rowc = has_row ? row : cur.r0;
        const int rsa = A.rs[rowc];
        const int rsb = A.rs[rowc + 1];
        const RowState so = ld_state(st_old, rowc);
        double xo = 0.0;
        if (has_pend) xo = A.x[rowc];
        double s = 0.0;
        if (cur.nz == 0) {
            // rows without nonzeros: q = 0
        } else if (cur.nz <= 64 * WI) {
            constexpr int IB = 4;  // registers in flight
#pragma unroll
            // (loads stay unconditional: guarding the item slices beyond a
            // tile's nonzeros serialised this loop's gathers, 2x slower)
            for (int i0 = 0; i0 < WI; i0 += IB) {
                float vj[IB];
                RowState gj[IB];
#pragma unroll
                for (int i = 0; i < IB && i0 + i < WI; ++i) {
                    const int k = lane + 64 * (i0 + i);
                    vj[i] = ld_stream(val + (k < cur.nz ? cur.k0 + k : 0));
                    gj[i] = ld_state(st_old, cj[i0 + i]);
                }
#pragma unroll
                for (int i = 0; i < IB && i0 + i < WI; ++i) {
                    const int k = lane + 64 * (i0 + i);
                    lds_wave[k] = (double)vj[i] *
                                  (double)__builtin_fmaf(beta, gj[i].p, next_r(alpha, gj[i].r, gj[i].q));
                }
            }
            __syncwarp();
            const int ra = rsa - cur.k0;
            const int rb = has_row ? rsb - cur.k0 : ra;
            s = row_sum(lds_wave, ra, rb);
            __syncwarp();
        } else {
            // a single row longer than a tile: wave-wide sum
            double part = 0.0;
            for (int k = lane; k < cur.nz; k += 64) {
                const RowState g = ld_state(st_old, col_at<IT>(A, cur.r0, cur.k0 + k));
                part += (double)val[cur.k0 + k] *
                        (double)__builtin_fmaf(beta, g.p, next_r(alpha, g.r, g.q));
            }
            s = wave_sum(part);
        }
        if (has_row) {
            RowState sn;
            sn.r = next_r(alpha, so.r, so.q);
            sn.p = __builtin_fmaf(beta, so.p, sn.r);
            sn.q = (float)s;
            const double rd = (double)sn.r, qd = (double)sn.q;
            sums[0] += (double)sn.p * s;
            sums[1] += rd * rd;
            sums[2] += rd * qd;
            sums[3] += qd * qd;
            st_state(st_new, row, sn);
            if (has_pend) A.x[row] = __builtin_fma(x_step(A, pend, row), (double)so.p, xo);
        }
    }
}

// The same fused phase with group loads (one-column mixed solves on
// matrices with 16-bit offsets).  Each lane owns 8 consecutive nonzeros of a
// wave tile, counted from the tile's first nonzero rounded down to a
// multiple of 8, so a tile's values take two 16-byte loads per lane and its
// column words one, instead of one load per nonzero each.  Entries of the
// neighbouring tiles in the first and last group are computed too (their
// offsets, decoded against this tile's first row, are clamped into the
// matrix) into the slice's 8 entries of padding or its unused tail, and are
// never summed.  The next tile's column words and values load while the
// current tile's gathers are in flight.  Products and sums are those of
// phase_f1 (p_k with the owner's two roundings, FP64 products of FP32
// factors, row sums in column order), so the iterates are identical.
template <int BS, typename MP>
__device__ void phase_f1g(const CgArgs &A, MP meta, int T0, int T1, double *lds_wave,
                          const void *st_old, void *st_new, const float alpha, const float beta,
                          const double pend, const bool has_pend, double (&sums)[4]) {
    constexpr int NW = BS / 64;
    typedef short i16x8 __attribute__((ext_vector_type(8)));
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int t = T0 + wave;
    if (t >= T1) return;
    const int nmax = A.n - 1;
    struct Pre {  // a tile's group: column words and values
        i16x8 w;
        f32x4 v0, v1;
    };
    auto fetch = [&](const WTile &w, Pre &p) {
        const int kk = (w.k0 & ~7) + 8 * lane;
        const int kc = kk < w.k0 + w.nz ? kk : (w.k0 & ~7);  // idle lanes: the first group
        p.w = ld_stream(reinterpret_cast<const i16x8 *>(A.dcol + kc));
        p.v0 = ld_stream(reinterpret_cast<const f32x4 *>(A.val32 + kc));
        p.v1 = ld_stream(reinterpret_cast<const f32x4 *>(A.val32 + kc + 4));
    };
    WTile w = wave_tile(meta, t);
    Pre pn;
    if (w.nz > 0 && w.nz <= kStageNnz) fetch(w, pn);
    for (; t < T1; t += NW) {
        const WTile cur = w;
        const Pre pc = pn;
        const int tn = t + NW;
        if (tn < T1) {
            w = wave_tile(meta, tn);
            if (w.nz > 0 && w.nz <= kStageNnz) fetch(w, pn);
        }
        const int row = cur.r0 + lane;
        const bool has_row = row < cur.r1;
        const int rowc = has_row ? row : cur.r0;
        const int rsa = A.rs[rowc];
        const int rsb = A.rs[rowc + 1];
        const RowState so = ld_state(st_old, rowc);
        double xo = 0.0;
        if (has_pend) xo = A.x[rowc];
        double s = 0.0;
        if (cur.nz == 0) {
            // rows without nonzeros: q = 0
        } else if (cur.nz <= kStageNnz) {
            const int kk = (cur.k0 & ~7) + 8 * lane;
            RowState g[8];
#pragma unroll
            for (int e = 0; e < 8; ++e)
                g[e] = ld_state(st_old, min(max(cur.r0 + (int)pc.w[e], 0), nmax));
            if (kk < cur.k0 + cur.nz) {
                double *dst = lds_wave + (kk - cur.k0);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float v = e < 4 ? pc.v0[e] : pc.v1[e - 4];
                    dst[e] = (double)v *
                             (double)__builtin_fmaf(beta, g[e].p, next_r(alpha, g[e].r, g[e].q));
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const int ra = rsa - cur.k0;
            const int rb = has_row ? rsb - cur.k0 : ra;
            s = row_sum(lds_wave, ra, rb);
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
        } else {
            // a single row longer than a tile: wave-wide sum
            double part = 0.0;
            for (int k = lane; k < cur.nz; k += 64) {
                const RowState g = ld_state(st_old, col_at<int16_t>(A, cur.r0, cur.k0 + k));
                part += (double)A.val32[cur.k0 + k] *
                        (double)__builtin_fmaf(beta, g.p, next_r(alpha, g.r, g.q));
            }
            s = wave_sum(part);
        }
        if (has_row) {
            RowState sn;
            sn.r = next_r(alpha, so.r, so.q);
            sn.p = __builtin_fmaf(beta, so.p, sn.r);
            sn.q = (float)s;
            const double rd = (double)sn.r, qd = (double)sn.q;
            sums[0] += (double)sn.p * s;
            sums[1] += rd * rd;
            sums[2] += rd * qd;
            sums[3] += qd * qd;
            st_state(st_new, row, sn);
            if (has_pend) A.x[row] = __builtin_fma(x_step(A, pend, row), (double)so.p, xo);
        }
    }
}

// x += pend p over the block's rows (p from the packed state)
template <int BS>
__device__ void flush_x1(const CgArgs &A, int R0, int R1, const void *st, double pend) {
    for (int row = R0 + (int)threadIdx.x; row < R1; row += BS)
        A.x[row] = __builtin_fma(x_step(A, pend, row), (double)ld_state(st, row).p, A.x[row]);
}

// Control state of a single-reduction solve, in LDS: thread 0 updates it after
// every grid reduction and the block reads the step coefficients from it, so
// the bookkeeping holds no registers during the phases.  Two columns share
// one iteration count and reliable updates (a column that did not ask for one
// gets it too).
template <int NC>
struct CgCtl {
    double tol2[NC], gamma[NC], rmax2[NC], last_rr[NC], ru_rr[NC], rho[NC];
    double pend[NC], alpha[NC], beta[NC], g[NC];
    int iters[NC], status[NC], stall[NC], active[NC], dropped[NC];
    int k, last_ru, refines, ru, has_pend, out_of_iters, any;
};

// After the set-up residual: acc[c] = (r, r) in FP64, acc[NC + c] = (b, b),
// acc[2 NC + c] = (r, r) of the stored r.
template <int NC>
__device__ void ctl_start(CgCtl<NC> &C, const CgArgs &A, const double (&acc)[3 * NC], bool writer) {
    C.any = 0;
    for (int c = 0; c < NC; ++c) {
        const double bn = sqrt(acc[NC + c]), r0n = sqrt(acc[c]);
        const double ref = bn > 0.0 ? bn : r0n;
        const double tol = fmax(A.rtol * ref, A.atol);
        C.tol2[c] = tol * tol;
        C.active[c] = acc[c] > C.tol2[c];
        C.any = C.any || C.active[c];
        C.gamma[c] = acc[2 * NC + c];
        // the drop triggers compare the recursion with the true residual in
        // the iteration's (scaled) space; rho converts a scaled norm into
        // the unscaled one the tolerance is on
        C.rmax2[c] = A.scale ? acc[2 * NC + c] : acc[c];
        C.last_rr[c] = C.ru_rr[c] = acc[c];
        C.rho[c] = A.scale && acc[2 * NC + c] > 0.0 ? acc[c] / acc[2 * NC + c] : 1.0;
        C.g[c] = 0.0;
        C.iters[c] = 0;
        C.status[c] = NSFEM_OK;
        C.stall[c] = C.dropped[c] = 0;
        C.pend[c] = C.alpha[c] = C.beta[c] = 0.0;
        if (writer) {
            A.res[c].rhs_norm = bn;
            A.res[c].initial_residual = r0n;
            A.res[c].tolerance = tol;
        }
    }
    C.k = C.last_ru = C.refines = C.ru = C.has_pend = C.out_of_iters = 0;
}

// After the phase reduction: alpha_k, gamma_{k+1} and the reliable-update
// trigger.  A drop of the recursive residual by rdelta triggers the update
// once ru_min_gap iterations have passed, a drop by rdelta^2 at once (FP32
// rounding must not pile up over a steep fall); ru_gap iterations and the
// iteration limit force one.  sums[4 c ...] = (p, q), (r, r), (r, q), (q, q).
// MIXED = false (FP64): no updates; a column is done when its recursive
// residual meets the tolerance.
template <int NC, bool MIXED = true>
__device__ void ctl_after_phase(CgCtl<NC> &C, const CgArgs &A, const double (&sums)[4 * NC]) {
    const int k = ++C.k;
    const double d2 = A.rdelta * A.rdelta;
    bool want = false, any = false;
    for (int c = 0; c < NC; ++c) {
        double alpha = 0.0, g = 0.0;
        bool dropped = false;
        if (C.active[c]) {
            const double delta = sums[4 * c], gk = sums[4 * c + 1];
            if (!(delta > 0.0)) {
                C.status[c] = NSFEM_BREAKDOWN;
                C.active[c] = 0;
                C.last_rr[c] = gk;
            } else {
                alpha = gk / delta;
                // gk - 2 alpha (r, q) + alpha^2 (q, q), its roundings spelt out:
                // the same bits in every kernel this is inlined into
                g = fmax(__builtin_fma(alpha * alpha, sums[4 * c + 3],
                                       __builtin_fma(-2.0 * alpha, sums[4 * c + 2], gk)),
                         0.0);
                C.gamma[c] = gk;
                C.iters[c] = k;
                if (MIXED) {
                    dropped = g * C.rho[c] <= C.tol2[c] ||
                              (g < d2 * C.rmax2[c] &&
                               (k - C.last_ru >= A.ru_min_gap || g < d2 * d2 * C.rmax2[c]));
                } else if (g <= C.tol2[c]) {
                    C.active[c] = 0;  // its last step is still pending
                    C.last_rr[c] = g;
                }
            }
        }
        want = want || dropped;
        any = any || C.active[c];
        C.pend[c] = alpha;
        C.alpha[c] = alpha;
        C.g[c] = g;
        C.dropped[c] = dropped;
    }
    C.has_pend = 1;
    C.out_of_iters = k >= A.max_iter;
    C.ru = MIXED && any && (want || k - C.last_ru >= A.ru_gap || C.out_of_iters);
    if (C.ru) C.last_ru = k;
}

// After a reliable update (x flushed, r := b - A x in FP64; ra as ctl_start's
// acc): the FP64 residual decides convergence; after a drop reported by the
// recursion the FP64 residual must fall below (1 + rdelta)/2 of its best
// value so far, and three misses in a row end the FP32 iteration
// (stagnation; an update forced by ru_gap alone is not judged).
template <int NC>
__device__ void ctl_after_update(CgCtl<NC> &C, const CgArgs &A, const double (&ra)[3 * NC]) {
    C.has_pend = 0;
    ++C.refines;
    for (int c = 0; c < NC; ++c) {
        C.pend[c] = 0.0;
        C.alpha[c] = 0.0;
        C.last_rr[c] = ra[c];
        if (!C.active[c]) continue;
        if (ra[c] <= C.tol2[c]) {
            C.active[c] = 0;
            continue;
        }
        C.g[c] = ra[2 * NC + c];
        C.rmax2[c] = A.scale ? ra[2 * NC + c] : ra[c];
        C.rho[c] = A.scale && ra[2 * NC + c] > 0.0 ? ra[c] / ra[2 * NC + c] : 1.0;
        if (C.dropped[c]) {
            const double sr = 0.5 * (1.0 + A.rdelta);
            C.stall[c] = ra[c] > sr * sr * C.ru_rr[c] ? C.stall[c] + 1 : 0;
        }
        C.ru_rr[c] = fmin(C.ru_rr[c], ra[c]);
        if (C.stall[c] >= 3) {
            C.status[c] = NSFEM_STAGNATION;
            C.active[c] = 0;
        } else if (C.refines >= A.max_refine) {
            C.status[c] = NSFEM_MAX_ITERATIONS_REACHED;
            C.active[c] = 0;
        }
    }
}

// End of an iteration: iteration limit, beta_{k+1} = gamma_{k+1} / gamma_k.
template <int NC>
__device__ void ctl_end(CgCtl<NC> &C) {
    C.any = 0;
    for (int c = 0; c < NC; ++c) {
        if (C.active[c] && C.out_of_iters) {
            C.status[c] = NSFEM_MAX_ITERATIONS_REACHED;
            C.active[c] = 0;
            C.last_rr[c] = C.g[c];
        }
        C.beta[c] = C.active[c] ? C.g[c] / C.gamma[c] : 0.0;
        if (!C.active[c]) C.alpha[c] = 0.0;
        C.any = C.any || C.active[c];
    }
}

template <int NC>
__device__ void ctl_finish(const CgCtl<NC> &C, const CgArgs &A) {
    for (int c = 0; c < NC; ++c) {
        A.res[c].iterations = C.iters[c];
        A.res[c].refinements = C.refines;
        A.res[c].status = C.status[c];
        A.res[c].last_residual = sqrt(C.last_rr[c]);
    }
}

// The one-column mixed persistent CG run by one block (arguments as
// cg_body).  The recursive residual is replaced by the FP64 b - A x whenever
// it has fallen by rdelta (reliable updates).
template <int BS, typename IT, int WI, typename MP>
__device__ __forceinline__ void cg_body1_m(const CgArgs &A, MP meta, const int bid, const int nb,
                                           const int L, double *prod_raw, double *lds) {
    constexpr bool MIXED = true;  // residual_phase precision
    // WI 1: group loads (16-bit offsets only); else WI items per lane
    constexpr bool GROUPS = WI == 1;
    static_assert(!GROUPS || std::is_same<IT, int16_t>::value, "group loads read 16-bit words");
    __shared__ CgCtl<1> C;
    const int T0 = A.block_tiles[L], T1 = A.block_tiles[L + 1];
    const int R0 = A.tiles[T0], R1 = A.tiles[T1];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // the group-load product writes up to 7 entries before a tile's first
    // nonzero: each wave's slice starts 8 entries in
    double *lds64 = prod_raw + wave * (kWaveNnz + (GROUPS ? 8 : 0)) + (GROUPS ? 8 : 0);
    unsigned epoch = 0;
    const bool t0 = threadIdx.x == 0;
    const bool writer = (L == 0 && t0);
    int cur = 0;  // st[cur]: state of step k - 1

    {
        double acc[3] = {0.0, 0.0, 0.0};
        residual_phase<1, BS, MIXED, true, IT, true, MP>(A, meta, T0, T1, lds64, acc, A.st[0]);
        if (!grid_sum<3, BS>(A.sync, acc, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
        if (t0) ctl_start<1>(C, A, acc, writer);
        __syncthreads();
    }
    while (C.any) {
        const int nx = cur ^ 1;
        const float alpha = (float)C.alpha[0], beta = (float)C.beta[0];
        const double pend = C.pend[0];
        const bool has_pend = C.has_pend != 0;
        double sums[4] = {0.0, 0.0, 0.0, 0.0};
        CG_TRACE_STAMP(C.k, 0);
        if constexpr (GROUPS)
            phase_f1g<BS, MP>(A, meta, T0, T1, lds64, A.st[cur], A.st[nx], alpha, beta, pend,
                              has_pend, sums);
        else
            phase_f1<BS, IT, WI, MP>(A, meta, T0, T1, lds64, A.st[cur], A.st[nx], alpha, beta,
                                     pend, has_pend, sums);
        CG_TRACE_MAX(C.k, 1);
        if (!grid_sum<4, BS>(A.sync, sums, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
        CG_TRACE_STAMP(C.k, 2);
        if (t0) {
            ctl_after_phase<1>(C, A, sums);
            if (!C.ru) ctl_end<1>(C);
        }
        __syncthreads();
        if (C.ru) {
            // apply the pending x += alpha p_k (FP64), then replace the
            // recursive residual: r_k := b - A x, alpha := 0
            flush_x1<BS>(A, R0, R1, A.st[nx], C.pend[0]);
            double dummy[1] = {0.0};
            if (!grid_sum<1, BS>(A.sync, dummy, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
            double ra[3] = {0.0, 0.0, 0.0};
            residual_phase<1, BS, MIXED, false, IT, true, MP>(A, meta, T0, T1, lds64, ra, A.st[nx]);
            if (!grid_sum<3, BS>(A.sync, ra, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
            if (t0) {
                ctl_after_update<1>(C, A, ra);
                ctl_end<1>(C);
            }
            __syncthreads();
        }
        if (!C.any) {
            if (C.has_pend) flush_x1<BS>(A, R0, R1, A.st[nx], C.pend[0]);
            break;
        }
        cur = nx;
    }
    if (writer) ctl_finish<1>(C, A);
    return;
timeout:
    if (writer) A.res[0].status = NSFEM_BARRIER_TIMEOUT;
}

template <int BS, typename IT, int WI>
__device__ __forceinline__ void cg_body1(const CgArgs &A, const int bid, const int nb, const int L,
                                         double *prod_raw, double *lds) {
    __shared__ int2 tmeta[kMetaLds + 1];
    const int T0 = A.block_tiles[L], T1 = A.block_tiles[L + 1];
    if (T1 > T0 && T1 - T0 <= kMetaLds) {
        load_meta_lds<BS>(A.meta, T0, T1, tmeta);
        cg_body1_m<BS, IT, WI>(A, MetaLds{tmeta, T0}, bid, nb, L, prod_raw, lds);
    } else {
        cg_body1_m<BS, IT, WI>(A, A.meta, bid, nb, L, prod_raw, lds);
    }
}

// ---------------------------------------------------------------------
// Two-column mixed solves: the single-reduction iteration of the one-column
// solves (phase_f1) over both columns at once.  Each nonzero's column and
// value load once for both columns; a neighbour's {r0, r1, p0, p1} and
// {q0, q1} come in two gathers; each column's p_k is recomputed from its
// gathered state by the same two roundings as its owner's, and the FP64
// sums (p_k, q_k), (r_k, r_k), (r_k, q_k), (q_k, q_k) of both columns take
// one grid reduction of 8 values.  sums[4c + i] holds column c's i-th sum.
// IB: nonzeros per lane whose loads are in flight together (4 or 8).
template <int BS, typename IT, int IB, typename MP>
__device__ void phase_f2(const CgArgs &A, MP meta, int T0, int T1, double *lds_wave,
                         const void *st_old, void *st_new, const float (&alpha)[2],
                         const float (&beta)[2], const double (&pend)[2], const bool has_pend,
                         double (&sums)[8]) {
    constexpr int NW = BS / 64;
    constexpr int WI = kWItems;
    const int n = A.n;
    const float *val = A.val32;
    const float4 *rp_old = st2_rp(st_old);
    const float2 *q_old = st2_q(st_old, n);
    float4 *rp_new = st2_rp(st_new);
    float2 *q_new = st2_q(st_new, n);
    const bool pend0 = has_pend && pend[0] != 0.0, pend1 = has_pend && pend[1] != 0.0;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int t = T0 + wave;
    if (t >= T1) return;
    WTile w = wave_tile(meta, t);
    int cn[WI];
    {
        const int kf = w.nz > 0 ? w.k0 : 0;
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            const int k = lane + 64 * i;
            cn[i] = col_word<IT>(A, k < w.nz ? w.k0 + k : kf);
        }
    }
    for (; t < T1; t += NW) {
        const WTile cur = w;
        int cj[WI];
#pragma unroll
        for (int i = 0; i < WI; ++i) cj[i] = col_of<IT>(cn[i], cur.r0);
        const int tn = t + NW;
        if (tn < T1) {
            w = wave_tile(meta, tn);
            const int kf = w.nz > 0 ? w.k0 : 0;
#pragma unroll
            for (int i = 0; i < WI; ++i) {
                const int k = lane + 64 * i;
                cn[i] = col_word<IT>(A, k < w.nz ? w.k0 + k : kf);
            }
        }
        const int row = cur.r0 + lane;
        const bool has_row = row < cur.r1;
        const int rowc = has_row ? row : cur.r0;
        const int rsa = A.rs[rowc];
        const int rsb = A.rs[rowc + 1];
        const float4 so = rp_old[rowc];
        const float2 sq = q_old[rowc];
        // the row's solution entries and scale load with its state, ahead of
        // the gathers (a late load would wait behind the next tile's
        // prefetch)
        double xo0 = 0.0, xo1 = 0.0, scl = 1.0;
        if (pend0) xo0 = A.x[rowc];
        if (pend1) xo1 = A.x[(size_t)n + rowc];
        if (has_pend && A.scale) scl = A.scale[rowc];
        double s[2] = {0.0, 0.0};
        if (cur.nz == 0) {
            // rows without nonzeros: q = 0
        } else if (cur.nz <= 64 * WI) {
#pragma unroll
            for (int i0 = 0; i0 < WI; i0 += IB) {
                float vj[IB];
                float4 gj[IB];
                float2 gq[IB];
#pragma unroll
                for (int i = 0; i < IB; ++i) {
                    const int k = lane + 64 * (i0 + i);
                    vj[i] = ld_stream(val + (k < cur.nz ? cur.k0 + k : 0));
                    gj[i] = rp_old[cj[i0 + i]];
                    gq[i] = q_old[cj[i0 + i]];
                }
#pragma unroll
                for (int i = 0; i < IB; ++i) {
                    const int k = lane + 64 * (i0 + i);
                    const double v = (double)vj[i];
                    lds_wave[2 * k] =
                        v * (double)__builtin_fmaf(beta[0], gj[i].z, next_r(alpha[0], gj[i].x, gq[i].x));
                    lds_wave[2 * k + 1] =
                        v * (double)__builtin_fmaf(beta[1], gj[i].w, next_r(alpha[1], gj[i].y, gq[i].y));
                }
            }
            __syncwarp();
            const int ra = rsa - cur.k0;
            const int rb = has_row ? rsb - cur.k0 : ra;
            row_sums<2>(lds_wave, ra, rb, s);
            __syncwarp();
        } else {
            // a single row longer than a tile: wave-wide sums
            double part0 = 0.0, part1 = 0.0;
            for (int k = lane; k < cur.nz; k += 64) {
                const int j = col_at<IT>(A, cur.r0, cur.k0 + k);
                const float4 g = rp_old[j];
                const float2 q = q_old[j];
                const double v = (double)val[cur.k0 + k];
                part0 += v * (double)__builtin_fmaf(beta[0], g.z, next_r(alpha[0], g.x, q.x));
                part1 += v * (double)__builtin_fmaf(beta[1], g.w, next_r(alpha[1], g.y, q.y));
            }
            s[0] = wave_sum(part0);
            s[1] = wave_sum(part1);
        }
        if (has_row) {
            const float r0 = next_r(alpha[0], so.x, sq.x), r1 = next_r(alpha[1], so.y, sq.y);
            const float p0 = __builtin_fmaf(beta[0], so.z, r0);
            const float p1 = __builtin_fmaf(beta[1], so.w, r1);
            const float q0 = (float)s[0], q1 = (float)s[1];
            const double r0d = (double)r0, q0d = (double)q0, r1d = (double)r1, q1d = (double)q1;
            sums[0] += (double)p0 * s[0];
            sums[1] += r0d * r0d;
            sums[2] += r0d * q0d;
            sums[3] += q0d * q0d;
            sums[4] += (double)p1 * s[1];
            sums[5] += r1d * r1d;
            sums[6] += r1d * q1d;
            sums[7] += q1d * q1d;
            rp_new[row] = make_float4(r0, r1, p0, p1);
            q_new[row] = make_float2(q0, q1);
            // x_c += x_step(pend_c) p_c, x_step = pend_c * scale[row] (or pend_c)
            if (pend0) A.x[row] = __builtin_fma(pend[0] * scl, (double)so.z, xo0);
            if (pend1) A.x[(size_t)n + row] = __builtin_fma(pend[1] * scl, (double)so.w, xo1);
        }
    }
}

// x_c += pend_c p_c over the block's rows (p from the packed state)
template <int BS>
__device__ void flush_x2(const CgArgs &A, int R0, int R1, const void *st,
                         const double (&pend)[2]) {
    const float4 *rp = st2_rp(st);
    for (int row = R0 + (int)threadIdx.x; row < R1; row += BS) {
        const float4 v = rp[row];
        if (pend[0] != 0.0) A.x[row] = __builtin_fma(x_step(A, pend[0], row), (double)v.z, A.x[row]);
        if (pend[1] != 0.0) {
            double *x = A.x + (size_t)A.n + row;
            *x = __builtin_fma(x_step(A, pend[1], row), (double)v.w, *x);
        }
    }
}

// The two-column mixed persistent CG run by one block (arguments as
// cg_body), single-reduction iteration over the packed state.
template <int BS, typename IT, int IB, typename MP>
__device__ __forceinline__ void cg_body2_m(const CgArgs &A, MP meta, const int bid, const int nb,
                                           const int L, double *prod_raw, double *lds) {
    __shared__ CgCtl<2> C;
    const int T0 = A.block_tiles[L], T1 = A.block_tiles[L + 1];
    const int R0 = A.tiles[T0], R1 = A.tiles[T1];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double *lds64 = prod_raw + wave * kWaveNnz * 2;
    unsigned epoch = 0;
    const bool t0 = threadIdx.x == 0;
    const bool writer = (L == 0 && t0);
    int cur = 0;  // st[cur]: state of step k - 1

    {
        double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        residual_phase<2, BS, true, true, IT, true, MP>(A, meta, T0, T1, lds64, acc, A.st[0]);
        if (!grid_sum<6, BS>(A.sync, acc, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
        if (t0) ctl_start<2>(C, A, acc, writer);
        __syncthreads();
    }
    while (C.any) {
        const int nx = cur ^ 1;
        const float alpha[2] = {(float)C.alpha[0], (float)C.alpha[1]};
        const float beta[2] = {(float)C.beta[0], (float)C.beta[1]};
        const double pend[2] = {C.pend[0], C.pend[1]};
        const bool has_pend = C.has_pend != 0;
        double sums[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        CG_TRACE_STAMP(C.k, 0);
        phase_f2<BS, IT, IB, MP>(A, meta, T0, T1, lds64, A.st[cur], A.st[nx], alpha, beta, pend,
                             has_pend, sums);
        CG_TRACE_MAX(C.k, 1);
        if (!grid_sum<8, BS>(A.sync, sums, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
        CG_TRACE_STAMP(C.k, 2);
        if (t0) {
            ctl_after_phase<2>(C, A, sums);
            if (!C.ru) ctl_end<2>(C);
        }
        __syncthreads();
        if (C.ru) {
            // apply the pending x += alpha p_k (FP64), then replace both
            // recursive residuals: r_k := b - A x, alpha := 0
            const double pf[2] = {C.pend[0], C.pend[1]};
            flush_x2<BS>(A, R0, R1, A.st[nx], pf);
            double dummy[1] = {0.0};
            if (!grid_sum<1, BS>(A.sync, dummy, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
            double ra[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
            residual_phase<2, BS, true, false, IT, true, MP>(A, meta, T0, T1, lds64, ra, A.st[nx]);
            if (!grid_sum<6, BS>(A.sync, ra, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
            if (t0) {
                ctl_after_update<2>(C, A, ra);
                ctl_end<2>(C);
            }
            __syncthreads();
        }
        if (!C.any) {
            if (C.has_pend) {
                const double pf[2] = {C.pend[0], C.pend[1]};
                flush_x2<BS>(A, R0, R1, A.st[nx], pf);
            }
            break;
        }
        cur = nx;
    }
    if (writer) ctl_finish<2>(C, A);
    return;
timeout:
    if (writer) {
        for (int c = 0; c < 2; ++c) A.res[c].status = NSFEM_BARRIER_TIMEOUT;
    }
}

// ---------------------------------------------------------------------
// Two-column mixed solves, narrow-gather form: the packed iteration's
// arithmetic with p_k stored once instead of recomputed by every reader.
// After the reduction, a stream pass over the block's own rows forms
//   r_k = r_{k-1} - alpha q_{k-1},  p_k = r_k + beta p_{k-1},
//   x += pend p_{k-1} (FP64),
// a grid barrier follows, and the product q_k = A p_k gathers only the
// neighbours' {p0, p1} (8 bytes, one load per nonzero instead of two) with
// the sums (p_k, q_k), (r_k, r_k), (r_k, q_k), (q_k, q_k) of the packed
// form.  r, p and q are interleaved [n][2] FP32 arrays (one copy each: the
// stream pass touches only its own rows, the product writes only q).  The
// FP32 roundings, products and sums are those of the packed form, so the
// iterates are the same bits.
template <int BS>
__device__ void phase_u2(const CgArgs &A, int R0, int R1, float2 *r, float2 *p, const float2 *q,
                         const float (&alpha)[2], const float (&beta)[2], const double (&pend)[2],
                         const bool has_pend) {
    const bool pend0 = has_pend && pend[0] != 0.0, pend1 = has_pend && pend[1] != 0.0;
    const size_t n = (size_t)A.n;
    for (int row = R0 + (int)threadIdx.x; row < R1; row += BS) {
        const float2 ro = r[row], po = p[row], qo = q[row];
        double x0 = 0.0, x1 = 0.0, scl = 1.0;
        if (pend0) x0 = A.x[row];
        if (pend1) x1 = A.x[n + row];
        if (has_pend && A.scale) scl = A.scale[row];
        const float r0 = next_r(alpha[0], ro.x, qo.x), r1 = next_r(alpha[1], ro.y, qo.y);
        r[row] = make_float2(r0, r1);
        p[row] = make_float2(__builtin_fmaf(beta[0], po.x, r0), __builtin_fmaf(beta[1], po.y, r1));
        if (pend0) A.x[row] = __builtin_fma(pend[0] * scl, (double)po.x, x0);
        if (pend1) A.x[n + row] = __builtin_fma(pend[1] * scl, (double)po.y, x1);
    }
}

template <int BS, typename IT, int IB, typename MP>
__device__ void phase_q2(const CgArgs &A, MP meta, int T0, int T1, double *lds_wave,
                         const float2 *p, const float2 *r, float2 *q, double (&sums)[8]) {
    constexpr int NW = BS / 64;
    constexpr int WI = kWItems;
    const float *val = A.val32;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int t = T0 + wave;
    if (t >= T1) return;
    WTile w = wave_tile(meta, t);
    int cn[WI];
    {
        const int kf = w.nz > 0 ? w.k0 : 0;
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            const int k = lane + 64 * i;
            cn[i] = col_word<IT>(A, k < w.nz ? w.k0 + k : kf);
        }
    }
    for (; t < T1; t += NW) {
        const WTile cur = w;
        int cj[WI];
#pragma unroll
        for (int i = 0; i < WI; ++i) cj[i] = col_of<IT>(cn[i], cur.r0);
        const int tn = t + NW;
        if (tn < T1) {
            w = wave_tile(meta, tn);
            const int kf = w.nz > 0 ? w.k0 : 0;
#pragma unroll
            for (int i = 0; i < WI; ++i) {
                const int k = lane + 64 * i;
                cn[i] = col_word<IT>(A, k < w.nz ? w.k0 + k : kf);
            }
        }
        const int row = cur.r0 + lane;
        const bool has_row = row < cur.r1;
        const int rowc = has_row ? row : cur.r0;
        const int rsa = A.rs[rowc];
        const int rsb = A.rs[rowc + 1];
        const float2 po = p[rowc], ro = r[rowc];
        double s[2] = {0.0, 0.0};
        if (cur.nz == 0) {
            // rows without nonzeros: q = 0
        } else if (cur.nz <= 64 * WI) {
#pragma unroll
            for (int i0 = 0; i0 < WI; i0 += IB) {
                float vj[IB];
                float2 gj[IB];
#pragma unroll
                for (int i = 0; i < IB; ++i) {
                    const int k = lane + 64 * (i0 + i);
                    vj[i] = ld_stream(val + (k < cur.nz ? cur.k0 + k : 0));
                    gj[i] = p[cj[i0 + i]];
                }
#pragma unroll
                for (int i = 0; i < IB; ++i) {
                    const int k = lane + 64 * (i0 + i);
                    const double v = (double)vj[i];
                    lds_wave[2 * k] = v * (double)gj[i].x;
                    lds_wave[2 * k + 1] = v * (double)gj[i].y;
                }
            }
            __syncwarp();
            const int ra = rsa - cur.k0;
            const int rb = has_row ? rsb - cur.k0 : ra;
            row_sums<2>(lds_wave, ra, rb, s);
            __syncwarp();
        } else {
            // a single row longer than a tile: wave-wide sums
            double part0 = 0.0, part1 = 0.0;
            for (int k = lane; k < cur.nz; k += 64) {
                const float2 g = p[col_at<IT>(A, cur.r0, cur.k0 + k)];
                const double v = (double)val[cur.k0 + k];
                part0 += v * (double)g.x;
                part1 += v * (double)g.y;
            }
            s[0] = wave_sum(part0);
            s[1] = wave_sum(part1);
        }
        if (has_row) {
            const float q0 = (float)s[0], q1 = (float)s[1];
            const double r0d = (double)ro.x, q0d = (double)q0, r1d = (double)ro.y, q1d = (double)q1;
            sums[0] += (double)po.x * s[0];
            sums[1] += r0d * r0d;
            sums[2] += r0d * q0d;
            sums[3] += q0d * q0d;
            sums[4] += (double)po.y * s[1];
            sums[5] += r1d * r1d;
            sums[6] += r1d * q1d;
            sums[7] += q1d * q1d;
            q[row] = make_float2(q0, q1);
        }
    }
}

// The narrow-gather two-column mixed CG run by one block (control as
// cg_body2_m; one grid barrier and one reduction an iteration).
template <int BS, typename IT, int IB, typename MP>
__device__ __forceinline__ void cg_body2n_m(const CgArgs &A, MP meta, const int bid, const int nb,
                                            const int L, double *prod_raw, double *lds) {
    __shared__ CgCtl<2> C;
    const int T0 = A.block_tiles[L], T1 = A.block_tiles[L + 1];
    const int R0 = A.tiles[T0], R1 = A.tiles[T1];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double *lds64 = prod_raw + wave * kWaveNnz * 2;
    float2 *r = (float2 *)A.r, *p = (float2 *)A.p0, *q = (float2 *)A.q;
    unsigned epoch = 0;
    const bool t0 = threadIdx.x == 0;
    const bool writer = (L == 0 && t0);

    {
        // r = b - A x (FP64, stored FP32), p = 0, q = 0
        double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        residual_phase<2, BS, true, true, IT, false, MP>(A, meta, T0, T1, lds64, acc);
        for (int row = R0 + (int)threadIdx.x; row < R1; row += BS) q[row] = make_float2(0.f, 0.f);
        if (!grid_sum<6, BS>(A.sync, acc, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
        if (t0) ctl_start<2>(C, A, acc, writer);
        __syncthreads();
    }
    while (C.any) {
        {
            const float alpha[2] = {(float)C.alpha[0], (float)C.alpha[1]};
            const float beta[2] = {(float)C.beta[0], (float)C.beta[1]};
            const double pend[2] = {C.pend[0], C.pend[1]};
            phase_u2<BS>(A, R0, R1, r, p, q, alpha, beta, pend, C.has_pend != 0);
        }
        double dummy[1] = {0.0};
        if (!grid_sum<1, BS>(A.sync, dummy, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
        double sums[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        phase_q2<BS, IT, IB, MP>(A, meta, T0, T1, lds64, p, r, q, sums);
        if (!grid_sum<8, BS>(A.sync, sums, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
        if (t0) {
            ctl_after_phase<2>(C, A, sums);
            if (!C.ru) ctl_end<2>(C);
        }
        __syncthreads();
        if (C.ru) {
            // apply the pending x += alpha p_k (FP64), then replace both
            // recursive residuals: r_k := b - A x, alpha := 0
            const double pf[2] = {C.pend[0], C.pend[1]};
            flush_x<2, BS, float>(A, R0, R1, (const float *)p, pf);
            if (!grid_sum<1, BS>(A.sync, dummy, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
            double ra[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
            residual_phase<2, BS, true, false, IT, false, MP>(A, meta, T0, T1, lds64, ra);
            if (!grid_sum<6, BS>(A.sync, ra, epoch, lds, A.timeout_ticks, bid, nb, A.flat)) goto timeout;
            if (t0) {
                ctl_after_update<2>(C, A, ra);
                ctl_end<2>(C);
            }
            __syncthreads();
        }
        if (!C.any) {
            if (C.has_pend) {
                const double pf[2] = {C.pend[0], C.pend[1]};
                flush_x<2, BS, float>(A, R0, R1, (const float *)p, pf);
            }
            break;
        }
    }
    if (writer) ctl_finish<2>(C, A);
    return;
timeout:
    if (writer) {
        for (int c = 0; c < 2; ++c) A.res[c].status = NSFEM_BARRIER_TIMEOUT;
    }
}

// One block per CU: BS / 256 waves per SIMD (4 for 1024 threads, 128 VGPRs
// per wave; 2 for 512 threads, up to 256 VGPRs).
// WI (items per lane of a tile) < 8 is used by the one-column mixed solve only.
template <int NC, int BS, bool MIXED, typename IT, int WI>
__global__ __launch_bounds__(BS, BS / 256) void k_cg(const CgArgs A) {
    constexpr int NW = BS / 64;
    __shared__ double prod_raw[NW * (kWaveNnz * NC + (WI == 1 ? 8 : 0))];
    __shared__ double lds[kMaxRed * NW];
    const int L = xcd_swizzle(blockIdx.x, gridDim.x);
    if constexpr (NC == 1 && MIXED)
        cg_body1<BS, IT, WI>(A, blockIdx.x, gridDim.x, L, prod_raw, lds);
    else
        cg_body<NC, BS, MIXED, IT>(A, blockIdx.x, gridDim.x, L, prod_raw, lds);
}

// The two-column mixed solve's packed iteration: a kernel of its own, so
// that its registers are allocated for it alone.  (The tile descriptors
// stay in global memory: a copy in LDS beside the product slices measured
// no faster, 2,495 against 2,525 GB/s in the 2048^2 cavity's mass solve.)
template <int BS, typename IT, int IB>
__global__ __launch_bounds__(BS, BS / 256) void k_cg_p2(const CgArgs A) {
    constexpr int NW = BS / 64;
    __shared__ double prod_raw[NW * kWaveNnz * 2];
    __shared__ double lds[kMaxRed * NW];
    const int L = xcd_swizzle(blockIdx.x, gridDim.x);
    if (A.packed2 == 2)
        cg_body2n_m<BS, IT, IB>(A, A.meta, blockIdx.x, gridDim.x, L, prod_raw, lds);
    else
        cg_body2_m<BS, IT, IB>(A, A.meta, blockIdx.x, gridDim.x, L, prod_raw, lds);
}

// =====================================================================
// Resident CG: a solve whose matrix stays in the blocks' registers
// =====================================================================
//
// The persistent forms above stream the matrix from memory and gather the
// neighbours' vector entries every iteration, and publish what they wrote
// with an L2 write-back and invalidate at every grid reduction.  On a system
// of up to a few hundred thousand rows none of that is bandwidth: an
// iteration is a chain of load latencies and cache maintenance (12 us on the
// 512 x 128 channel's 65,656 pressure rows in FP32, 15-24 us in FP64).  Here,
// when the rows are short (at most W nonzeros) and banded:
//
// * a lane owns one row of up to R wave tiles and keeps the row's values, its
//   columns (16-bit positions in the block's window) and its r, q and x in
//   registers for the whole solve;
// * the block keeps p for its window -- its own rows and the rows its columns
//   reach, one contiguous run -- in LDS, and r for the window's rows that
//   other blocks own.  It updates both for itself from the neighbours' q, the
//   only vector that crosses blocks: r = r - alpha q and p = r + beta p round
//   the same in every block that computes them;
// * q and the sums cross through agent-scope relaxed stores and loads, which
//   meet at the coherence point and pass the caches by, so that nothing is
//   written back or invalidated: a wave waits for its stores of q, the block
//   meets, and the sums are posted with the epoch beside their bits, one read
//   giving arrival and value together.
//
// One exchange an iteration (the single-reduction iteration of the one-column
// mixed solves, in FP64 too).  In the one-column mixed form every product,
// sum and reduction has phase_f1g's order (wave tiles to waves, lanes to rows,
// the same grid; blocks as the flat reduction adds them), so up to kFlatMax
// blocks its iterates are that form's, bit for bit; past them the streaming
// form adds the blocks' sums as a tree.
//
// Measured per iteration, streaming -> resident, refined with the residual
// passes: 1,089 pressure rows in one block, FP64 11.5 -> 2.2 us, refined 10.9
// -> 3.2; 65,656 rows on 42 blocks 18.3 -> 4.6 and 12.5 -> 5.0; 261,247 rows
// on 170 blocks 26.9 -> 6.5 and 21.6 -> 6.7; P2 mass matrices in lattice
// order, 4,225 rows on 8 blocks, two columns, FP64 22.9 -> 10.4, refined (22
// passes in 27 iterations) 48.0 -> 19.8; 261,241 rows on 256 blocks, one
// column FP64 33.7 -> 15.6, two refined (23 passes in 47) 108 -> 42.8.
// Systems past the registers or the window (a million P2 rows, the
// vertices-first node order of larger meshes) keep the streaming forms.

constexpr int kResWaves = 12;  // 3 waves a SIMD: 168 VGPRs each
// Waves of a block of the refined one-column batch: those of the streaming
// batch's blocks, whose sums it repeats (4 waves a SIMD: 128 VGPRs each).
constexpr int kResWavesBatch = 16;

template <typename T>
__device__ __forceinline__ T ld_agent(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void st_agent(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// rows of NC interleaved columns
template <int NC, typename T>
__device__ __forceinline__ VecN<NC, T> ldv_agent(const T *p, int i) {
    VecN<NC, T> o;
    if constexpr (NC == 2 && sizeof(T) == 4) {
        const unsigned long long t =
            ld_agent(reinterpret_cast<const unsigned long long *>(p) + i);
        o.v[0] = __uint_as_float((unsigned)t);
        o.v[1] = __uint_as_float((unsigned)(t >> 32));
    } else {
#pragma unroll
        for (int c = 0; c < NC; ++c) o.v[c] = ld_agent(p + (size_t)i * NC + c);
    }
    return o;
}
template <int NC, typename T>
__device__ __forceinline__ void stv_agent(T *p, int i, const VecN<NC, T> &v) {
    if constexpr (NC == 2 && sizeof(T) == 4) {
        const unsigned long long t =
            (unsigned long long)__float_as_uint(v.v[0]) |
            ((unsigned long long)__float_as_uint(v.v[1]) << 32);
        st_agent(reinterpret_cast<unsigned long long *>(p) + i, t);
    } else {
#pragma unroll
        for (int c = 0; c < NC; ++c) st_agent(p + (size_t)i * NC + c, v.v[c]);
    }
}

// wave_sum's sum, in its order, without the LDS pipe: lanes 32 and 16 apart
// by row swaps, then rotations within rows of 16 (after each step the values
// repeat with that period, so a rotation pairs what an exclusive-or does).
template <int CTRL>
__device__ __forceinline__ double dpp_rotated(double v) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                            (unsigned long long)(unsigned)lo));
}
__device__ __forceinline__ double wave_sum_dpp(double v) {
    {
        const unsigned long long u = (unsigned long long)__double_as_longlong(v);
        const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)u, false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(u >> 32), (unsigned)(u >> 32),
                                                         false, false);
        v = __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
    }
    {
        const unsigned long long u = (unsigned long long)__double_as_longlong(v);
        const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)u, false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(u >> 32), (unsigned)(u >> 32),
                                                         false, false);
        v = __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
    }
    v += dpp_rotated<0x128>(v);  // row_ror:8
    v += dpp_rotated<0x124>(v);
    v += dpp_rotated<0x122>(v);
    v += dpp_rotated<0x121>(v);
    return v;
}

template <int NW>
struct ResShared {
    double part[2][kMaxRed][NW];  // by epoch parity
    double sum[kMaxRed];
    int fail;
    int range;  // FP64: a sum was past the recurrence's range
};

// Status of a resident FP64 solve that left the range of its recurrence (no
// public status is positive): x is as it was, and the streaming form, which
// sums (r, r) itself, runs the solve.
constexpr int kCgOutOfRange = 1;
// Least (r, r), (q, q) and alpha^2, 2^-963 or 1.3e-290 (high word), whose
// terms' underflow below 1e-307 is lost in rounding.
constexpr int kCgLeastSum = 60 << 20;

// Whether the next (r, r) of an FP64 column cannot be formed from an
// iteration's sums: (q, q) of a matrix near 1e-170 underflows and alpha^2
// overflows, (q, q) of one near 1e150 overflows, while (r, r) and (p, q) are in
// range.  The mark stays: whatever the recurrence does from there (converge
// on a clamped 0, break down on an infinity), x is written only at the end.
// A thread of its own tests while thread 0 steps the control state (on thread
// 0's chain the test took 0.7 to 1.6% of a solve).
template <int NC>
__device__ __forceinline__ bool past_range(const double *sums) {
    bool out = false;
    for (int c = 0; c < NC; ++c) {
        const double delta = sums[4 * c], gk = sums[4 * c + 1], qq = sums[4 * c + 3];
        if (!(delta > 0.0) || gk == 0.0) continue;  // a breakdown, or done
        const double alpha = gk / delta;
        const double g = __builtin_fma(alpha * alpha, qq,
                                       __builtin_fma(-2.0 * alpha, sums[4 * c + 2], gk));
        // (non-negative doubles compare as their high words)
        const int least = min(min(__double2hiint(gk), __double2hiint(qq)),
                              __double2hiint(alpha * alpha));
        out = out || least < kCgLeastSum ||
              (__double2hiint(g) & 0x7ff00000) == 0x7ff00000;  // infinite or NaN
    }
    return out;
}

// The grid's sums of K values a thread, into S.sum, and a barrier over the
// solve's blocks: every block's agent-scope stores before it are visible to
// agent-scope loads after it.  False when a block did not arrive in time.
//
// Wave k adds the block's partials of sum k in wave order, posts the two
// halves of the result, each in one 8-byte word with the epoch, and polls the
// other blocks' words; a word that carries the epoch is whole, so nothing
// orders the two halves.  The words alternate between two slots by epoch
// parity: a block posts epoch e + 2 only after every block has posted e + 1,
// which each does after it has read all of e.  Sums are added as in
// grid_sum_flat.  The waits on vmcnt before the first barrier are what makes
// the block's stores visible before its post.
template <int K, int NW>
__device__ __forceinline__ bool res_exchange(SyncState *G, ResShared<NW> &S, double (&v)[K],
                                             unsigned &epoch, const unsigned long long timeout,
                                             const int b, const int nb) {
    static_assert(K <= kMaxRed && K <= NW, "reduction width");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned e = ++epoch;
    const int par = e & 1u;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        v[k] = wave_sum_dpp(v[k]);
        if (lane == 0) S.part[par][k][wave] = v[k];
    }
    __builtin_amdgcn_s_waitcnt(0);  // this wave's stores are complete
    __syncthreads();
    if (wave < K) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < NW; ++i) s += S.part[par][wave][i];
        if (nb == 1) {
            if (lane == 0) S.sum[wave] = s;
        } else {
            unsigned long long(*words)[2] = G->tag[par][wave];
            const unsigned long long mark = (unsigned long long)e << 32;
            const unsigned long long bits = (unsigned long long)__double_as_longlong(s);
            if (lane < 2)
                st_agent(&words[b][lane], mark | (lane ? bits >> 32 : bits & 0xffffffffull));
            double t = 0.0;
            bool ok = true;
            const unsigned long long t0 = wall_clock64();
            for (int i = lane; i < nb; i += 64) {
                unsigned long long w0 = ld_agent(&words[i][0]), w1 = ld_agent(&words[i][1]);
                while (ok && ((w0 ^ mark) >> 32 != 0 || (w1 ^ mark) >> 32 != 0)) {
                    if (ld_agent(&G->abort) != 0u) {
                        ok = false;
                    } else if (wall_clock64() - t0 > timeout) {
                        st_agent(&G->abort, 1u);
                        ok = false;
                    }
                    w0 = ld_agent(&words[i][0]);
                    w1 = ld_agent(&words[i][1]);
                }
                t += __longlong_as_double((long long)((w1 << 32) | (w0 & 0xffffffffull)));
            }
            t = wave_sum_dpp(t);
            if (lane == 0) S.sum[wave] = t;
            if (!ok) S.fail = 1;
        }
    }
    __syncthreads();
    return S.fail == 0;
}

// The FP64 residual of the wave's rows: r = b - A x, scaled and rounded to VT,
// published in rbuf; the sums as residual_phase's, which it rounds as (the
// products before they are added, in column order).  SHARED: x as other
// blocks published it.  The loop over the wave's tiles stays rolled, so that
// its loads take no registers from the resident matrix more than once.
template <int NC, typename VT, bool SHARED, int NW>
__device__ __forceinline__ void res_residual(const CgArgs &A, const int T0, const int T1,
                                             const int wave, const int lane, VT *rbuf,
                                             double (&acc)[3 * NC]) {
#pragma unroll 1
    for (int t = T0 + wave; t < T1; t += NW) {
        const int4 m = A.meta[t];
        const int row = m.x + lane;
        if (row >= m.y) continue;
        double s[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) s[c] = 0.0;
        const int ka = A.rs[row], kb = A.rs[row + 1];
        // four nonzeros' loads in flight (past the row: its last, not added)
#pragma unroll 1
        for (int k0 = ka; k0 < kb; k0 += 4) {
            double pr[4][NC];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k = min(k0 + u, kb - 1);
                const double v = A.val64[k];
                const int j = A.col[k];
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const double *xp = A.x + (size_t)c * A.n + j;
                    pr[u][c] = v * (SHARED ? ld_agent(xp) : *xp);
                    asm("" : "+v"(pr[u][c]));  // no fused multiply-add
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    if (k0 + u < kb) s[c] += pr[u][c];
        }
        const double sc = A.scale ? A.scale[row] : 1.0;
        VecN<NC, VT> r;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const double bb = A.b[(size_t)c * A.n + row];
            const double rr = bb - s[c];
            acc[c] += rr * rr;
            if (!SHARED) acc[NC + c] += bb * bb;
            r.v[c] = (VT)(A.scale ? rr * sc : rr);
            acc[2 * NC + c] += (double)r.v[c] * (double)r.v[c];
        }
        stv_agent<NC, VT>(rbuf, row, r);
    }
}

// One block's part of a resident solve of `nb` blocks (`b`: its reduction
// slot, `L`: its index among the tiles' owners, as cg_body).  W: the most
// nonzeros of a row; R: the most wave tiles of a wave (the host checks both,
// and that the window fits win_cap); NW: the block's waves.  smem: win_cap + 1 rows of p, then r of
// the window's rows that other blocks own.
template <int NC, bool MIXED, int W, int R, int NW>
__device__ __forceinline__ void cg_resident(const CgArgs &A, const int b, const int nb,
                                            const int L, unsigned char *smem) {
    using VT = typename std::conditional<MIXED, float, double>::type;
    using Row = VecN<NC, VT>;
    __shared__ CgCtl<NC> C;
    __shared__ ResShared<NW> S;
    constexpr int BS = 64 * NW;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int T0 = A.block_tiles[L], T1 = A.block_tiles[L + 1];
    const int R0 = A.tiles[T0], R1 = A.tiles[T1];
    const int win0 = max(0, R0 - A.band_lo), win1 = min(A.n, R1 + A.band_hi);
    const int nl = R0 - win0, nh = nl + (win1 - R1), wn = win1 - win0;
    Row *pw = reinterpret_cast<Row *>(smem);
    Row *rh = pw + A.win_cap + 1;
    VT *rbuf = (VT *)A.r;
    VT *qbuf[2] = {(VT *)A.p0, (VT *)A.p1};
    const bool t0 = tid == 0, writer = L == 0 && t0;
    unsigned epoch = 0;

    int row[R];  // -1: none
    VT val[R][W];
    unsigned idx[R][(W + 1) / 2];
    Row r[R], q[R];
    VecN<NC, double> x[R];
    if (t0) S.fail = S.range = 0;
    {
        Row zero;
#pragma unroll
        for (int c = 0; c < NC; ++c) zero.v[c] = (VT)0;
        for (int i = tid; i <= wn; i += BS) pw[i] = zero;
        for (int i = tid; i < nh; i += BS) rh[i] = zero;
        double acc[3 * NC];
#pragma unroll
        for (int k = 0; k < 3 * NC; ++k) acc[k] = 0.0;
        res_residual<NC, VT, false, NW>(A, T0, T1, wave, lane, rbuf, acc);
        if (!res_exchange<3 * NC, NW>(A.sync, S, acc, epoch, A.timeout_ticks, b, nb)) goto timeout;
        if (t0) {
            double sums[3 * NC];
#pragma unroll
            for (int k = 0; k < 3 * NC; ++k) sums[k] = S.sum[k];
            ctl_start<NC>(C, A, sums, writer);
        }
#pragma unroll
        for (int j = 0; j < R; ++j) {
            row[j] = -1;
            q[j] = zero;
            r[j] = zero;
#pragma unroll
            for (int w = 0; w < W; ++w) val[j][w] = (VT)0;
#pragma unroll
            for (int w = 0; w < (W + 1) / 2; ++w) idx[j][w] = (unsigned)wn * 0x10001u;
            const int t = T0 + wave + NW * j;
            if (t >= T1) continue;  // wave-uniform
            const int4 m = A.meta[t];
            const bool has = m.x + lane < m.y;
            const int k0 = A.rs[has ? m.x + lane : m.x];
            const int len = has ? A.rs[m.x + lane + 1] - k0 : 0;
            row[j] = has ? m.x + lane : -1;
            // a lane past its row's nonzeros reads the matrix's last entry
            // and keeps 0 x (the window's zero)
            const int last = A.nnz - 1;
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const int k = min(k0 + w, last);
                VT v;
                if constexpr (MIXED) v = A.val32[k];
                else v = A.val64[k];
                const unsigned pos = w < len ? (unsigned)(A.col[k] - win0) : (unsigned)wn;
                val[j][w] = w < len ? v : (VT)0;
                if (w % 2) idx[j][w / 2] |= pos << 16;
                else idx[j][w / 2] = pos;
                if (w % 5 == 4) __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (!has) continue;
            r[j] = ldv_agent<NC, VT>(rbuf, row[j]);
#pragma unroll
            for (int c = 0; c < NC; ++c) x[j].v[c] = A.x[(size_t)c * A.n + row[j]];
        }
        __syncthreads();
    }
    {
        bool fresh = true;  // rbuf holds r (after a residual), not qbuf the step's q
        int par = 0;
        while (C.any) {
            VT alpha[NC], beta[NC];
            double pend[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                alpha[c] = (VT)C.alpha[c];
                beta[c] = (VT)C.beta[c];
                pend[c] = C.pend[c];
            }
            const bool has_pend = C.has_pend != 0;
            // the window's rows of other blocks: kAhead loads in flight
            constexpr int kAhead = 4;
            const VT *src = fresh ? rbuf : qbuf[par ^ 1];
            for (int base = tid; base < nh; base += kAhead * BS) {
                Row in[kAhead];
#pragma unroll
                for (int u = 0; u < kAhead; ++u) {
                    const int i = min(base + u * BS, nh - 1);
                    in[u] = ldv_agent<NC, VT>(src, i < nl ? win0 + i : R1 + (i - nl));
                }
#pragma unroll
                for (int u = 0; u < kAhead; ++u) {
                    const int i = base + u * BS;
                    if (i >= nh) break;
                    const int slot = i < nl ? i : i + (R1 - R0);
                    Row rn, pn = pw[slot];
                    if (fresh) {
                        rn = in[u];
                    } else {
                        rn = rh[i];
#pragma unroll
                        for (int c = 0; c < NC; ++c)
                            rn.v[c] = fma_t<VT>(-alpha[c], in[u].v[c], rn.v[c]);
                    }
#pragma unroll
                    for (int c = 0; c < NC; ++c) pn.v[c] = fma_t<VT>(beta[c], pn.v[c], rn.v[c]);
                    rh[i] = rn;
                    pw[slot] = pn;
                }
            }
#pragma unroll
            for (int j = 0; j < R; ++j) {
                if (row[j] < 0) continue;
                Row pn = pw[row[j] - win0];
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    if (has_pend)
                        x[j].v[c] = __builtin_fma(x_step(A, pend[c], row[j]), (double)pn.v[c],
                                                  x[j].v[c]);
                    r[j].v[c] = fma_t<VT>(-alpha[c], q[j].v[c], r[j].v[c]);
                    pn.v[c] = fma_t<VT>(beta[c], pn.v[c], r[j].v[c]);
                }
                pw[row[j] - win0] = pn;
            }
            __syncthreads();
            double sums[4 * NC];
#pragma unroll
            for (int k = 0; k < 4 * NC; ++k) sums[k] = 0.0;
#pragma unroll
            for (int j = 0; j < R; ++j) {
                if (T0 + wave + NW * j >= T1) continue;  // wave-uniform
                double s[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) s[c] = 0.0;
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    unsigned word = idx[j][w / 2];
                    VT v = val[j][w];
                    // keeps the widened value and the address out of the
                    // registers across iterations: they would double the
                    // matrix's
                    asm volatile("" : "+v"(word), "+v"(v));
                    const Row pv = pw[w % 2 ? word >> 16 : word & 0xffffu];
#pragma unroll
                    for (int c = 0; c < NC; ++c)
                        s[c] = __builtin_fma((double)v, (double)pv.v[c], s[c]);
                    // five reads in flight: all W of them would not fit
                    if (w % 5 == 4) __builtin_amdgcn_sched_barrier(0);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (row[j] < 0) continue;
                const Row pn = pw[row[j] - win0];
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    q[j].v[c] = (VT)s[c];
                    const double rd = (double)r[j].v[c], qd = (double)q[j].v[c];
                    sums[4 * c] += (double)pn.v[c] * s[c];
                    sums[4 * c + 1] += rd * rd;
                    sums[4 * c + 2] += rd * qd;
                    sums[4 * c + 3] += qd * qd;
                }
                stv_agent<NC, VT>(qbuf[par], row[j], q[j]);
            }
            if (!res_exchange<4 * NC, NW>(A.sync, S, sums, epoch, A.timeout_ticks, b, nb)) goto timeout;
            if (t0) {
#pragma unroll
                for (int k = 0; k < 4 * NC; ++k) sums[k] = S.sum[k];
                ctl_after_phase<NC, MIXED>(C, A, sums);
                if (!C.ru) ctl_end<NC>(C);
            }
            if (!MIXED && tid == 64 && past_range<NC>(S.sum)) S.range = 1;
            __syncthreads();
            fresh = false;
            if constexpr (MIXED) {
                if (C.ru) {
                    // apply the pending x += alpha p_k (FP64), then replace
                    // the recursive residual: r_k := b - A x, alpha := 0
#pragma unroll
                    for (int j = 0; j < R; ++j) {
                        if (row[j] < 0) continue;
                        const Row pn = pw[row[j] - win0];
#pragma unroll
                        for (int c = 0; c < NC; ++c) {
                            x[j].v[c] = __builtin_fma(x_step(A, C.pend[c], row[j]),
                                                      (double)pn.v[c], x[j].v[c]);
                            st_agent(A.x + (size_t)c * A.n + row[j], x[j].v[c]);
                        }
                    }
                    double none[1] = {0.0};
                    if (!res_exchange<1, NW>(A.sync, S, none, epoch, A.timeout_ticks, b, nb))
                        goto timeout;
                    double ra[3 * NC];
#pragma unroll
                    for (int k = 0; k < 3 * NC; ++k) ra[k] = 0.0;
                    res_residual<NC, VT, true, NW>(A, T0, T1, wave, lane, rbuf, ra);
                    if (!res_exchange<3 * NC, NW>(A.sync, S, ra, epoch, A.timeout_ticks, b, nb))
                        goto timeout;
                    if (t0) {
#pragma unroll
                        for (int k = 0; k < 3 * NC; ++k) ra[k] = S.sum[k];
                        ctl_after_update<NC>(C, A, ra);
                        ctl_end<NC>(C);
                    }
#pragma unroll
                    for (int j = 0; j < R; ++j)
                        if (row[j] >= 0) r[j] = ldv_agent<NC, VT>(rbuf, row[j]);
                    __syncthreads();
                    fresh = true;
                }
            }
            if (!C.any) {
                if (C.has_pend) {
#pragma unroll
                    for (int j = 0; j < R; ++j) {
                        if (row[j] < 0) continue;
                        const Row pn = pw[row[j] - win0];
#pragma unroll
                        for (int c = 0; c < NC; ++c)
                            x[j].v[c] = __builtin_fma(x_step(A, C.pend[c], row[j]),
                                                      (double)pn.v[c], x[j].v[c]);
                    }
                }
                break;
            }
            par ^= 1;
        }
    }
    // (the same sums in every block, so the same mark)
    if (MIXED || S.range == 0) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            if (row[j] < 0) continue;
#pragma unroll
            for (int c = 0; c < NC; ++c) A.x[(size_t)c * A.n + row[j]] = x[j].v[c];
        }
    }
    if (writer) {
        ctl_finish<NC>(C, A);
        if (!MIXED && S.range != 0)
            for (int c = 0; c < NC; ++c) A.res[c].status = kCgOutOfRange;
    }
    return;
timeout:
    if (writer) {
        for (int c = 0; c < NC; ++c) A.res[c].status = NSFEM_BARRIER_TIMEOUT;
    }
}

template <int NC, bool MIXED, int W, int R, int NW>
__global__ __launch_bounds__(64 * NW, NW / 4) void k_cg_res(const CgArgs A) {
    extern __shared__ __align__(16) unsigned char smem[];
    cg_resident<NC, MIXED, W, R, NW>(A, blockIdx.x, gridDim.x,
                                     xcd_swizzle(blockIdx.x, gridDim.x), smem);
}

// Many resident solves in one launch (block map as k_cg_batch).
template <int NC, bool MIXED, int W, int R, int NW>
__global__ __launch_bounds__(64 * NW, NW / 4) void k_cg_res_batch(
    const CgArgs *__restrict__ args, const int2 *__restrict__ map) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int2 m = map[blockIdx.x];
    const int inst = __builtin_amdgcn_readfirstlane(m.x);
    const int lb = __builtin_amdgcn_readfirstlane(m.y);
    const CgArgs A = args[inst];
    cg_resident<NC, MIXED, W, R, NW>(A, lb, A.nblocks, lb, smem);
}

// Many independent systems in one persistent launch: block i works for
// instance map[i].x as its block map[i].y of args[instance].nblocks; each
// instance reduces over its own blocks with its own SyncState, and its blocks
// leave the kernel when it converges.
template <int NC, int BS, bool MIXED, typename IT, int WI>
__global__ __launch_bounds__(BS, BS / 256) void k_cg_batch(const CgArgs *__restrict__ args,
                                                           const int2 *__restrict__ map) {
    constexpr int NW = BS / 64;
    __shared__ double prod_raw[NW * (kWaveNnz * NC + (WI == 1 ? 8 : 0))];
    __shared__ double lds[kMaxRed * NW];
    const int2 m = map[blockIdx.x];
    const int inst = __builtin_amdgcn_readfirstlane(m.x);
    const int lb = __builtin_amdgcn_readfirstlane(m.y);
    const CgArgs A = args[inst];
    if constexpr (NC == 1 && MIXED)
        cg_body1<BS, IT, WI>(A, lb, A.nblocks, lb, prod_raw, lds);
    else
        cg_body<NC, BS, MIXED, IT>(A, lb, A.nblocks, lb, prod_raw, lds);
}

constexpr int kCgBlock = 1024;
// One-column mixed solves may run 768-thread blocks: 12 waves per CU with
// 168 VGPRs each instead of 16 with 128, which the tile loop needs to hold
// a prefetched tile without spilling (a scratch reload inside the loop waits
// for every load in flight, the prefetch included).
constexpr int kCgBlockWide = 768;

// Block size of a solve: one-column mixed solves run the wide-register
// blocks unless NSFEM_CG_BLOCK=1024 (read at every solve; measured at the
// 2048^2 cavity, 768 threads with group loads: pressure 95.9 us and v
// diffusion 550 us per iteration against 98.8 / 564 us for 1024 threads
// with one load per nonzero per lane).  The two-column mixed solve was
// slower in 768-thread blocks (mass 1,195 against 1,044 us per iteration).
int cg_block(int nc, bool mixed) {
    if (!(nc == 1 && mixed)) return kCgBlock;
    const char *e = std::getenv("NSFEM_CG_BLOCK");
    return (e && std::atoi(e) == kCgBlock) ? kCgBlock : kCgBlockWide;
}

template <int NC, bool MIXED, typename IT, int WI, int BS>
void cg_launch(Device &d, const CgArgs &args, int grid) {
    void *kargs[] = {(void *)&args};
    NSFEM_HIP(hipLaunchCooperativeKernel((const void *)k_cg<NC, BS, MIXED, IT, WI>, dim3(grid),
                                         dim3(BS), kargs, 0, d.stream));
}
template <int NC, bool MIXED, typename IT, int WI, int BS>
int cg_max_grid(Device &d) {
    int per_cu = 0;
    NSFEM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_cg<NC, BS, MIXED, IT, WI>,
                                                           BS, 0));
    return std::max(1, std::min(per_cu * d.cu_count, kMaxGridBlocks));
}

// Calls f.template run<NC, MIXED, IT, WI>() for the solve's column count,
// precision, column-index width and (one-column mixed solves) items per lane.
template <int WI, typename F>
void cg_dispatch_wi(int nc, bool mixed, bool idx16, F &f) {
    if (nc == 1) {
        if (mixed) {
            if (idx16) f.template run<1, true, int16_t, WI>();
            else f.template run<1, true, int32_t, WI>();
        } else {
            if (idx16) f.template run<1, false, int16_t, kWItems>();
            else f.template run<1, false, int32_t, kWItems>();
        }
    } else {
        if (mixed) {
            if (idx16) f.template run<2, true, int16_t, kWItems>();
            else f.template run<2, true, int32_t, kWItems>();
        } else {
            if (idx16) f.template run<2, false, int16_t, kWItems>();
            else f.template run<2, false, int32_t, kWItems>();
        }
    }
}
// wi 1: the one-column mixed iteration with group loads (16-bit offsets)
template <typename F>
void cg_dispatch(int nc, bool mixed, bool idx16, int wi, F &&f) {
    if (wi == 1 && nc == 1 && mixed && idx16) f.template run<1, true, int16_t, 1>();
    else if (wi <= 4) cg_dispatch_wi<4>(nc, mixed, idx16, f);
    else if (wi <= 7) cg_dispatch_wi<7>(nc, mixed, idx16, f);
    else cg_dispatch_wi<kWItems>(nc, mixed, idx16, f);
}

// Items per lane the one-column mixed iteration needs for a matrix: every
// multi-row wave tile's nonzeros over 64, rounded up to 4, 7 or 8.
int items_per_lane(const Matrix &m) {
    const int need = (m.max_multirow_nz + 63) / 64;
    return need <= 4 ? 4 : need <= 7 ? 7 : kWItems;
}

// Form of the one-column mixed iteration on matrices with 16-bit offsets:
// NSFEM_CG_PHASE = items (one load per nonzero per lane) or groups (8
// nonzeros per lane); without it, groups where `groups_default` (the
// single solves' wide blocks) and the matrix allows them.  Read at every
// solve (comparison runs switch it in one process).
int phase_form(const Matrix &m, bool groups_default) {
    const char *e = std::getenv("NSFEM_CG_PHASE");
    const std::string v = e ? e : "";
    if (v == "items") return -1;
    if (v == "groups" || (v.empty() && groups_default)) return m.groups_ok ? 1 : -1;
    return -1;
}

template <typename IT, int BS, int IB>
void cg_launch_p2(Device &d, const CgArgs &args, int grid) {
    void *kargs[] = {(void *)&args};
    NSFEM_HIP(hipLaunchCooperativeKernel((const void *)k_cg_p2<BS, IT, IB>, dim3(grid), dim3(BS),
                                         kargs, 0, d.stream));
}
template <typename IT, int BS, int IB>
int cg_max_grid_p2(Device &d) {
    int per_cu = 0;
    NSFEM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_cg_p2<BS, IT, IB>, BS, 0));
    return std::max(1, std::min(per_cu * d.cu_count, kMaxGridBlocks));
}
// Calls f.template run<IT, BS, IB>() for the packed two-column iteration's
// block size (768 or 1024) and loads in flight (4 or 8 nonzeros per lane).
template <typename IT, typename F>
void p2_dispatch(int bs, int ib, F &f) {
    if (bs == kCgBlockWide) {
        if (ib == 8) f.template run2<IT, kCgBlockWide, 8>();
        else f.template run2<IT, kCgBlockWide, 4>();
    } else {
        if (ib == 8) f.template run2<IT, kCgBlock, 8>();
        else f.template run2<IT, kCgBlock, 4>();
    }
}

// p2: the two-column mixed solve's packed iteration (k_cg_p2)
struct CgMaxGrid {
    Device &d;
    int out;
    int bs = kCgBlock;
    bool p2 = false;
    int ib = 4;
    template <typename IT, int BS, int IB>
    void run2() {
        out = cg_max_grid_p2<IT, BS, IB>(d);
    }
    template <int NC, bool MX, typename IT, int WI>
    void run() {
        if constexpr (NC == 2 && MX) {
            if (p2) {
                p2_dispatch<IT>(bs, ib, *this);
                return;
            }
        }
        if constexpr (NC == 1 && MX) {
            if (bs == kCgBlockWide) {
                out = cg_max_grid<NC, MX, IT, WI, kCgBlockWide>(d);
                return;
            }
        }
        out = cg_max_grid<NC, MX, IT, WI, kCgBlock>(d);
    }
};
struct CgLaunch {
    Device &d;
    const CgArgs &a;
    int grid;
    int bs = kCgBlock;
    bool p2 = false;
    int ib = 4;
    template <typename IT, int BS, int IB>
    void run2() {
        cg_launch_p2<IT, BS, IB>(d, a, grid);
    }
    template <int NC, bool MX, typename IT, int WI>
    void run() {
        if constexpr (NC == 2 && MX) {
            if (p2) {
                p2_dispatch<IT>(bs, ib, *this);
                return;
            }
        }
        if constexpr (NC == 1 && MX) {
            if (bs == kCgBlockWide) {
                cg_launch<NC, MX, IT, WI, kCgBlockWide>(d, a, grid);
                return;
            }
        }
        cg_launch<NC, MX, IT, WI, kCgBlock>(d, a, grid);
    }
};


// ---- resident solves
// Most nonzeros of a row and most wave tiles of a wave of the resident
// kernels.  168 registers hold short rows and one tile of long ones in one
// column; the kernels of two and three tiles of long rows and of two columns
// spill 14 (two refined columns, one tile) to 310 registers and are still
// ahead of the streaming forms, which read the matrix anew each iteration
// (times above; two FP64 columns of 261,241 P2 rows, 300 spilled: 26.6 us an
// iteration against 50.9).
constexpr int kResRowShort = 8, kResRowLong = 20;
constexpr int res_tiles(bool mixed, int w) { return w == kResRowShort ? 4 : mixed ? 3 : 2; }
// Most LDS of a resident block (160 KB a CU; one block a CU).
constexpr size_t kResLds = 120 * 1024;

// The kernel of a resident solve whose waves own `tiles` wave tiles at most;
// batch: of many solves, with `waves` waves a block (a refined batch: short
// rows and one column only, in kResWaves or kResWavesBatch waves).
template <int NC, bool MIXED, int W, int R>
const void *res_kernel(bool batch, int waves) {
    if (!batch) return (const void *)k_cg_res<NC, MIXED, W, R, kResWaves>;
    if constexpr (MIXED && W == kResRowShort) {
        if (waves == kResWavesBatch)
            return (const void *)k_cg_res_batch<NC, MIXED, W, R, kResWavesBatch>;
    }
    NSFEM_REQUIRE(waves == kResWaves, NSFEM_ERROR, "waves of a resident batch");
    if constexpr (!MIXED || W == kResRowShort)
        return (const void *)k_cg_res_batch<NC, MIXED, W, R, kResWaves>;
    fail(NSFEM_ERROR, "this refined batch streams");
}
template <int NC, bool MIXED, int W>
const void *res_kernel_tiles(bool batch, int waves, int tiles) {
    if (tiles <= 1) return res_kernel<NC, MIXED, W, 1>(batch, waves);
    if (tiles == 2) return res_kernel<NC, MIXED, W, 2>(batch, waves);
    if constexpr (MIXED && W == kResRowShort) {
        // 128 registers: three tiles spill 16, the next kernel's four 58;
        // three is what two tiles a wave come to where the blocks do not
        // divide them evenly
        if (waves == kResWavesBatch && tiles == 3)
            return (const void *)k_cg_res_batch<NC, MIXED, W, 3, kResWavesBatch>;
    }
    return res_kernel<NC, MIXED, W, res_tiles(MIXED, W)>(batch, waves);
}
const void *res_kernel(int nc, bool mixed, int w, int tiles, bool batch, int waves = kResWaves) {
    constexpr int S = kResRowShort, L = kResRowLong;
    if (nc == 2)
        return mixed ? res_kernel_tiles<2, true, L>(batch, waves, tiles)
                     : res_kernel_tiles<2, false, L>(batch, waves, tiles);
    if (w == S)
        return mixed ? res_kernel_tiles<1, true, S>(batch, waves, tiles)
                     : res_kernel_tiles<1, false, S>(batch, waves, tiles);
    return mixed ? res_kernel_tiles<1, true, L>(batch, waves, tiles)
                 : res_kernel_tiles<1, false, L>(batch, waves, tiles);
}

// Allows a kernel the most dynamic LDS of any solve and returns the blocks a
// device holds with this solve's.  (The attribute belongs to the kernel, in
// every thread and device handle: a solve's own amount would lower it between
// another handle's call here and its launch.)
int res_max_grid(Device &d, const void *kernel, int waves, size_t lds) {
    if (lds > 48 * 1024)
        NSFEM_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)kResLds));
    int per_cu = 0;
    NSFEM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 64 * waves, lds));
    return std::min(per_cu * d.cu_count, kResMaxBlocks);
}

// Wave tiles a wave that a resident solve's grid aims at (the quotient is
// rounded down, so some blocks give their waves one more: 65,656 rows come to
// 42 blocks where the first grid without a third tile is 47).  Short rows
// (P1): two, as the grid reductions grow with the blocks (65,656 rows, FP64
// and refined: 4.6 and 5.0 us an iteration on 42 blocks, 4.5 and 4.7 on 47,
// 4.4 and 4.5 on 64, 5.3 and 5.4 on 128, 6.3 and 6.3 on 256).  Long rows
// (P2): one, as a tile's work and the residual passes outweigh them (16,597
// rows, two columns, FP64 and refined: 15.7 and 26.9 us on 16 blocks, 12.7
// and 21.7 on this rule's 31, 9.6 and 15.1 on 64, 12.1 and 18.0 on 256).
int cg_tiles_per_wave(const Matrix &m) { return m.shape.max_nz > kResRowShort ? 1 : 2; }

// Window rows and LDS of a matrix split over `grid` blocks; false when a
// block's tiles, window or LDS go past what the kernel holds.
bool res_fits(const Matrix &m, int nc, bool mixed, int w, int waves, int grid, ResidentPlan &plan) {
    std::vector<int32_t> bt;
    split_tiles(m, grid, bt);
    int64_t cap = 0, halo = 0;
    int tiles = 0;
    for (int b = 0; b < grid; ++b) {
        tiles = std::max(tiles, (bt[b + 1] - bt[b] + waves - 1) / waves);
        if (bt[b + 1] <= bt[b] || tiles > res_tiles(mixed, w)) return false;
        const int64_t r0 = m.host_wtiles[bt[b]], r1 = m.host_wtiles[bt[b + 1]];
        const int64_t w0 = std::max<int64_t>(0, r0 - m.shape.lo);
        const int64_t w1 = std::min<int64_t>(m.rows, r1 + m.shape.hi);
        cap = std::max(cap, w1 - w0);
        halo = std::max(halo, (w1 - w0) - (r1 - r0));
    }
    const size_t bytes = (size_t)(cap + 1 + halo) * nc * (mixed ? sizeof(float) : sizeof(double));
    if (cap >= 65535 || bytes > kResLds) return false;
    plan.ok = true;
    plan.width = w;
    plan.tiles = tiles;
    plan.grid = grid;
    plan.cap = (int)cap;
    plan.lds = bytes;
    return true;
}

// The resident form of a solve on this matrix, or ok = false: rows of at most
// kResRowLong nonzeros, a window that fits the LDS, and a grid, the device's
// blocks at most, that leaves every wave its tiles.  `want` > 0 asks for a
// grid; else cg_tiles_per_wave, more blocks where a wave would get more tiles
// than it holds.
ResidentPlan plan_resident(const Matrix &m, int nc, bool mixed, int want, int max_blocks) {
    ResidentPlan plan;
    if (m.rows != m.cols || m.nnz <= 0 || m.shape.max_nz > kResRowLong) return plan;
    const int w = nc == 1 && m.shape.max_nz <= kResRowShort ? kResRowShort : kResRowLong;
    const int most = std::min(std::min(max_blocks, kResMaxBlocks), m.n_wtiles);
    if (most < 1) return plan;
    if (want > 0) {
        res_fits(m, nc, mixed, w, kResWaves, std::min(want, most), plan);
        return plan;
    }
    int grid = std::max(1, std::min(m.n_wtiles / (cg_tiles_per_wave(m) * kResWaves), most));
    const int room = kResWaves * res_tiles(mixed, w);
    if ((int64_t)room * most < m.n_wtiles) return plan;
    for (int tries = 0; tries < 8 && grid <= most; ++tries) {
        if (res_fits(m, nc, mixed, w, kResWaves, grid, plan)) return plan;
        grid = std::max(grid + 1, std::max((m.n_wtiles + room - 1) / room, grid + grid / 8));
    }
    return plan;
}

// The plan of single solves, kept with the matrix's tiles.
const ResidentPlan &resident_plan(Device &d, Matrix &m, int nc, bool mixed) {
    ResidentPlan &plan = m.res_plan[2 * (nc - 1) + (mixed ? 1 : 0)];
    if (!plan.made) {
        plan = plan_resident(m, nc, mixed, 0, d.cu_count);
        plan.made = true;
    }
    return plan;
}

// Blocks of a streaming solve of `waves` waves each, before the device's
// limit: two wave tiles a wave.  One-column mixed solves of matrices that fit
// the resident form take its grid (a comparison run then has its bits); of
// long rows that do not fit, one tile a wave up to 96 blocks and where two
// need more than the flat reduction takes, as the reduction grows with the
// blocks (microseconds a solve at one and two tiles a wave, mass matrices in
// the reference's node order, 29 to 34 iterations: 16,597 rows 557 and 694,
// 37,062 727 and 735, 65,657 865 and 846, 82,990 1,072 and 962, 102,372 1,170
// and 1,064, 147,220 1,357 and 1,382).
int streaming_blocks(Device &d, Matrix &m, int nc, bool mixed, int waves) {
    const int two = m.n_wtiles / (2 * waves), one = m.n_wtiles / waves;
    if (!(mixed && nc == 1)) return two;
    if (waves == kResWaves) {
        const ResidentPlan &res = resident_plan(d, m, nc, mixed);
        if (res.ok) return res.grid;
    }
    return cg_tiles_per_wave(m) == 1 && (one <= 96 || two > kFlatMax) ? one : two;
}

// Whether a solve may take the resident form: not when a comparison run asks
// for one of the streaming forms (NSFEM_CG_RESIDENT=0, or the form's own
// switches; read at every solve).
bool want_resident(int nc, bool mixed) {
    const char *e = std::getenv("NSFEM_CG_RESIDENT");
    if (e && std::atoi(e) == 0) return false;
    if (!mixed) return true;
    if (nc == 1) return !std::getenv("NSFEM_CG_PHASE") && !std::getenv("NSFEM_CG_BLOCK");
    return !std::getenv("NSFEM_CG_PAIRED") && !std::getenv("NSFEM_CG_P2_BLOCK") &&
           !std::getenv("NSFEM_CG_P2_LOADS");
}

}  // namespace


namespace {
// Device memory one persistent solve works in: six vectors of `vec_bytes`
// (r, p_old, p_new, q or the two packed {r, p, q} states), the grid
// reduction's state, the per-column results and the dot product's scratch.
struct CgWorkspace {
    unsigned char *vectors = nullptr;
    size_t vec_bytes = 0;
    SyncState *sync = nullptr;
    CgColumnResult *res = nullptr;  // [2]
    double *dot_partial = nullptr;  // [kDotBlocks]
    double *scalars = nullptr;      // [2]
};

// true residual ||b_c - A x_c|| for each column (FP64), into host res[c]
void true_residuals(Device &d, Matrix &m, const double *b, const double *x, int nc,
                    double *tmp, const CgWorkspace &ws, double *out) {
    launch_fill(d, nc, 0.0, ws.scalars);
    for (int c = 0; c < nc; ++c) {
        launch_spmv(d, m, x + (size_t)c * m.rows, b + (size_t)c * m.rows, tmp, 1);
        dot_accumulate(d, m.rows, tmp, tmp, ws.scalars + c, ws.dot_partial);
    }
    double h[2] = {0, 0};
    NSFEM_HIP(hipMemcpyAsync(h, ws.scalars, sizeof(double) * nc, hipMemcpyDeviceToHost,
                             d.stream));
    NSFEM_HIP(hipStreamSynchronize(d.stream));
    for (int c = 0; c < nc; ++c) out[c] = std::sqrt(h[c]);
}

// Bytes of one CG vector of a solve (rounded to 256).
size_t cg_vector_bytes(int n, int nc, bool mixed) {
    const size_t vt = mixed ? sizeof(float) : sizeof(double);
    return ((size_t)n * nc * vt + 255) / 256 * 256;
}

// The workspace in the device's own arrays, grown as needed.
CgWorkspace device_workspace(Device &d, int n, int nc, bool mixed) {
    CgWorkspace ws;
    ws.vec_bytes = cg_vector_bytes(n, nc, mixed);
    d.work.ensure(ws.vec_bytes * 6);
    d.sync_mem.ensure(sizeof(SyncState) + 256);
    d.cg_res.ensure(2);
    d.dot_partial.ensure(kDotBlocks);
    d.scalars.ensure(4);
    ws.vectors = d.work.ptr;
    unsigned char *sm = d.sync_mem.ptr;
    ws.sync = reinterpret_cast<SyncState *>(sm + (256 - ((uintptr_t)sm % 256)) % 256);
    ws.res = d.cg_res.ptr;
    ws.dot_partial = d.dot_partial.ptr;
    ws.scalars = d.scalars.ptr;
    return ws;
}
}  // namespace

namespace {

// Tolerances, iteration limits and reliable-update knobs of one solve.
void set_cg_params(const Device &d, const CgRequest &req, int n, CgArgs &a) {
    a.rtol = req.rtol;
    a.atol = req.atol;
    // reliable updates of the mixed solver: when the recursive residual has
    // fallen by rdelta since the last one, or after ru_gap iterations.
    // Measured on the 2048^2 cavity pressure matrix from x0 = 0: forced
    // updates every 1000 iterations cost 26% more iterations, and so does
    // holding updates back for 8 iterations after the last one (the default
    // minimum gap is therefore 0; it saves time only on systems that
    // converge in a few dozen iterations).  Tuning overrides:
    // NSFEM_CG_RDELTA, NSFEM_CG_RU_GAP, NSFEM_CG_RU_MIN_GAP.
    static const double rdelta_env = [] {
        const char *e = std::getenv("NSFEM_CG_RDELTA");
        return e ? std::atof(e) : 0.0;
    }();
    static const int ru_gap_env = [] {
        const char *e = std::getenv("NSFEM_CG_RU_GAP");
        return e ? std::atoi(e) : 0;
    }();
    a.rdelta = rdelta_env > 0.0 && rdelta_env < 1.0 ? rdelta_env : req.reliable_delta;
    a.max_iter = req.max_iter < 0 ? n : req.max_iter;
    a.max_refine = 400;
    static const int ru_min_gap_env = [] {
        const char *e = std::getenv("NSFEM_CG_RU_MIN_GAP");
        return e ? std::atoi(e) : -1;
    }();
    a.ru_gap = ru_gap_env > 0 ? ru_gap_env : (req.ru_gap > 0 ? req.ru_gap : 20000);
    a.ru_min_gap = ru_min_gap_env >= 0 ? ru_min_gap_env : 0;
    a.timeout_ticks = (unsigned long long)d.wall_khz * 1000ull * 20ull;  // 20 s per barrier
    // the flat grid reduction unless NSFEM_CG_FLAT=0 (read at every solve)
    const char *flat = std::getenv("NSFEM_CG_FLAT");
    a.flat = !(flat && std::atoi(flat) == 0);
}

// Packed FP32 {r, p, q} rows of a one-column mixed solve: two copies of 3
// vectors of `vb` bytes (a vector holds n values of the solve's precision).
void set_state_buffers(CgArgs &a, unsigned char *w, size_t vb) {
    a.st[0] = w;
    a.st[1] = w + 3 * vb;
}

// Iteration of two-column mixed solves: the single-reduction iteration
// (k_cg_p2) unless NSFEM_CG_PAIRED=twophase, in its narrow-gather form
// unless NSFEM_CG_PAIRED=packed (read at every solve; comparison runs switch
// it in one process).  Measured on the 2048^2 cavity's mass solve (textbook
// bytes / time): narrow 2,581 (4 loads in flight) and 2,603 GB/s (8),
// packed 2,521, two-phase 2,463.  The batched solves run the two-phase form.
bool paired_packed() {
    const char *e = std::getenv("NSFEM_CG_PAIRED");
    return !(e && std::string(e) == "twophase");
}
// 2: the narrow-gather form, 1: the packed form.
int paired_form() {
    const char *e = std::getenv("NSFEM_CG_PAIRED");
    return (e && std::string(e) == "packed") ? 1 : 2;
}
// Block size of the packed two-column iteration: NSFEM_CG_P2_BLOCK=768 or
// 1024 (read at every solve).
int paired_block() {
    const char *e = std::getenv("NSFEM_CG_P2_BLOCK");
    return (e && std::atoi(e) == kCgBlockWide) ? kCgBlockWide : kCgBlock;
}
// Nonzeros per lane whose loads the two-column iteration keeps in flight
// together: NSFEM_CG_P2_LOADS=4 or 8 (read at every solve); by default 8 for
// the narrow-gather form (one 8-byte gather a nonzero), 4 for the packed
// one (two gathers a nonzero; 8 measured 2,497 against 2,527 GB/s).
int paired_loads(int form) {
    const char *e = std::getenv("NSFEM_CG_P2_LOADS");
    if (e && (std::atoi(e) == 4 || std::atoi(e) == 8)) return std::atoi(e);
    return form == 2 ? 8 : 4;
}

struct CgPass {
    CgColumnResult res[2];
    int iters[2] = {0, 0}, refines[2] = {0, 0};
    double final_res[2] = {0, 0};
    float ms = 0.f;
};

// One persistent-CG solve in the given precision.  The FP64 path ends on the
// recursive residual; the true residual is recomputed and, should rounding
// drift have left it above the tolerance, the solve restarts from the
// current x (at most twice).  `fixed`: a workspace to work in (the
// no-allocation solve), else the device's own arrays.
void cg_pass(Device &d, const CgRequest &req, bool mixed, CgPass &P,
             const CgWorkspace *fixed = nullptr) {
    Matrix &m = *req.m;
    const int n = m.rows, nc = req.ncol;
    if (mixed) ensure_val32(d, m);
    const bool jacobi = mixed && req.jacobi && ensure_jacobi(d, m);
    // 1024 threads per block (16 waves per CU, 128 VGPRs each) for FP64
    // and two-column solves: the loop is bound by gather latency, so waves
    // in flight matter more than registers; 512 threads (8 waves, up to 256
    // VGPRs) was slower on every measured solve.  One-column mixed solves
    // run 768 (cg_block).
    const bool idx16 = m.dcol_ok && want_idx16();
    const bool p2 = nc == 2 && mixed && paired_packed();
    const int bs = p2 ? paired_block() : cg_block(nc, mixed);
    const int form = idx16 && mixed && nc == 1 ? phase_form(m, bs == kCgBlockWide) : -1;
    const int wi = form >= 0 ? form : items_per_lane(m);
    const int ib = p2 ? paired_loads(paired_form()) : 4;
    CgMaxGrid mg{d, 0, bs, p2, ib};
    cg_dispatch(nc, mixed, idx16, wi, mg);
    const int maxg = mg.out;
    int want = req.grid;
    if (want <= 0) {
        // tuning override: NSFEM_CG_GRID=<blocks> (capped by co-residency)
        const char *env = std::getenv("NSFEM_CG_GRID");
        if (env) want = std::atoi(env);
    }
    int grid = want > 0 ? want : streaming_blocks(d, m, nc, mixed, bs / 64);
    grid = std::max(1, std::min(std::min(grid, maxg), std::max(1, m.n_wtiles)));
    ResidentPlan res;
    if (req.resident && want_resident(nc, mixed))
        res = want > 0 ? plan_resident(m, nc, mixed, want, d.cu_count)
                       : resident_plan(d, m, nc, mixed);
    const void *res_fn = nullptr;
    if (res.ok) {
        res_fn = res_kernel(nc, mixed, res.width, res.tiles, false);
        res.ok = res_max_grid(d, res_fn, kResWaves, res.lds) >= res.grid;
        if (res.ok) grid = res.grid;
    }
    const bool verbose = std::getenv("NSFEM_CG_VERBOSE") != nullptr;
    ensure_block_tiles(d, m, grid);

    const CgWorkspace ws = fixed ? *fixed : device_workspace(d, n, nc, mixed);
    const size_t vec_bytes = cg_vector_bytes(n, nc, mixed);
    NSFEM_REQUIRE(vec_bytes <= ws.vec_bytes, NSFEM_ERROR, "CG workspace too small");

    CgArgs a{};
    a.n = n;
    a.nnz = (int)m.nnz;
    a.meta = m.wmeta.ptr;
    a.tiles = m.wtiles.ptr;
    a.block_tiles = m.block_tiles.ptr;
    a.rs = m.row_start.ptr;
    a.col = m.col.ptr;
    a.dcol = m.dcol.ptr;
    a.val64 = m.val.ptr;
    a.val32 = jacobi ? m.jval32.ptr : m.val32.ptr;
    a.scale = jacobi ? m.jscale.ptr : nullptr;
    a.b = req.b;
    a.x = req.x;
    unsigned char *w = ws.vectors;
    a.r = w;
    a.p0 = w + vec_bytes;
    a.p1 = w + 2 * vec_bytes;
    a.q = w + 3 * vec_bytes;
    set_state_buffers(a, w, vec_bytes);
    a.packed2 = p2 ? paired_form() : 0;
    set_cg_params(d, req, n, a);
    a.sync = ws.sync;
    a.res = ws.res;
    a.band_lo = m.shape.lo;
    a.band_hi = m.shape.hi;
    a.win_cap = res.cap;
    const int ngroups = (grid + kGroup - 1) / kGroup;

    for (int attempt = 0; attempt < 3; ++attempt) {
        if (verbose)  // one line per launch, in launch order
            std::fprintf(stderr,
                         "[nsfem] cg launch matrix=%p rows=%d cols=%d wave tiles=%d grid=%d "
                         "maxgrid=%d mixed=%d idx16=%d form=%d block=%d resident=%d attempt=%d\n",
                         (const void *)&m, n, nc, m.n_wtiles, grid, maxg, (int)mixed, (int)idx16,
                         wi, res.ok ? 64 * kResWaves : bs, res.ok ? res.width : 0, attempt);
        NSFEM_HIP(hipEventRecord(d.ev_start, d.stream));
        k_sync_reset<<<(ngroups + 255) / 256, 256, 0, d.stream>>>(a.sync, ngroups,
                                                                  res.ok ? grid : 0);
        NSFEM_HIP(hipGetLastError());
        if (res.ok) {
            void *kargs[] = {(void *)&a};
            NSFEM_HIP(hipLaunchCooperativeKernel(res_fn, dim3(grid), dim3(64 * kResWaves), kargs,
                                                 (unsigned)res.lds, d.stream));
        } else {
            CgLaunch ln{d, a, grid, bs, p2, ib};
            cg_dispatch(nc, mixed, idx16, wi, ln);
        }
        NSFEM_HIP(hipEventRecord(d.ev_stop, d.stream));
        NSFEM_HIP(hipMemcpyAsync(P.res, ws.res, sizeof(CgColumnResult) * nc,
                                 hipMemcpyDeviceToHost, d.stream));
        NSFEM_HIP(hipStreamSynchronize(d.stream));
        float ms = 0.f;
        NSFEM_HIP(hipEventElapsedTime(&ms, d.ev_start, d.ev_stop));
        P.ms += ms;
        if (P.res[0].status == kCgOutOfRange) {
            CgRequest r2 = req;
            r2.resident = false;
            cg_pass(d, r2, mixed, P, fixed);
            return;
        }
        bool drift = false;
        if (!mixed) true_residuals(d, m, req.b, req.x, nc, (double *)a.q, ws, P.final_res);
        for (int c = 0; c < nc; ++c) {
            P.iters[c] += P.res[c].iterations;
            P.refines[c] += P.res[c].refinements;
            if (mixed) P.final_res[c] = P.res[c].last_residual;
            if (P.res[c].status == NSFEM_OK && P.final_res[c] > P.res[c].tolerance * (1.0 + 1e-12))
                drift = true;
            if (P.res[c].status == NSFEM_BARRIER_TIMEOUT)
                fail(NSFEM_BARRIER_TIMEOUT, "CG kernel barrier timed out");
        }
        if (!drift || mixed) break;
    }
}

}  // namespace

namespace {
int run_cg_in(Device &d, const CgRequest &req, nsfem_cg_stats *stats,
              const CgWorkspace *fixed) {
    Matrix &m = *req.m;
    NSFEM_REQUIRE(m.ready, NSFEM_NOT_READY, "matrix slot is empty");
    NSFEM_REQUIRE(m.rows == m.cols, NSFEM_INVALID_ARGUMENT, "CG needs a square matrix");
    NSFEM_REQUIRE(req.ncol == 1 || req.ncol == 2, NSFEM_INVALID_ARGUMENT,
                  "columns must be 1 or 2");
    const bool mixed = req.precision == NSFEM_PRECISION_FP32_REFINED;
    NSFEM_REQUIRE(mixed || req.precision == NSFEM_PRECISION_FP64, NSFEM_INVALID_ARGUMENT,
                  "unknown precision");
    const int nc = req.ncol;
    CgPass P;
    cg_pass(d, req, mixed, P, fixed);
    CgPass F;  // FP64 continuation after an FP32 stagnation
    bool fallback = false;
    if (mixed) {
        for (int c = 0; c < nc; ++c) fallback = fallback || P.res[c].status == NSFEM_STAGNATION;
        if (fallback) {
            CgRequest r2 = req;
            if (r2.max_iter > 0) r2.max_iter = std::max(1, r2.max_iter - std::max(P.iters[0], P.iters[nc - 1]));
            // the same stopping rule: ||b|| (or ||r0||) of the original solve
            r2.rtol = 0.0;
            r2.atol = std::max(P.res[0].tolerance, nc == 2 ? P.res[1].tolerance : 0.0);
            if (nc == 2) r2.atol = std::min(P.res[0].tolerance, P.res[1].tolerance);
            cg_pass(d, r2, false, F, fixed);
        }
    }
    int worst = NSFEM_OK;
    for (int c = 0; c < nc; ++c) {
        const int status = fallback ? F.res[c].status : P.res[c].status;
        if (status != NSFEM_OK && worst == NSFEM_OK) worst = status;
        if (stats) {
            nsfem_cg_stats &s = stats[c];
            s.iterations = P.iters[c] + (fallback ? F.iters[c] : 0);
            s.refinements = P.refines[c] + (fallback ? 1 : 0);
            s.status = status;
            s.columns = nc;
            s.rhs_norm = P.res[c].rhs_norm;
            s.initial_residual = P.res[c].initial_residual;
            s.final_residual = fallback ? F.final_res[c] : P.final_res[c];
            s.tolerance = P.res[c].tolerance;
            s.seconds = (P.ms + (fallback ? F.ms : 0.f)) * 1e-3;
        }
    }
    return worst;
}
}  // namespace

int run_cg(Device &d, const CgRequest &req, nsfem_cg_stats *stats) {
    return run_cg_in(d, req, stats, nullptr);
}

// ------------------------------------------------------ no-allocation CG
// The device memory of the no-allocation solve: one static array per GPU
// (each device the library runs on holds its own copy until the process
// ends).  Host code never uses this name as an address: scratch_init looks
// up the device address once per device handle, and every kernel argument
// and copy uses that address.  Layout: the reduction state, the per-column
// results, the dot product's partials and scalars, then six CG vectors of
// kNoAllocVecBytes (an FP64 system of rows x columns <= kNoAllocMaxValues;
// an FP32 + refinement solve needs the same room for its FP64 fallback).
namespace {
constexpr size_t kNoAllocVecBytes = (size_t)kNoAllocMaxValues * sizeof(double);
constexpr size_t kScratchSync = 0;
constexpr size_t kScratchRes = kScratchSync + (sizeof(SyncState) + 255) / 256 * 256;
constexpr size_t kScratchDot = kScratchRes + 256;
constexpr size_t kScratchScal = kScratchDot + kDotBlocks * sizeof(double);
constexpr size_t kScratchVec = kScratchScal + 256;
constexpr size_t kScratchBytes = kScratchVec + 6 * kNoAllocVecBytes;
static_assert(2 * sizeof(CgColumnResult) <= 256, "results slot");
static_assert(sizeof(SyncState) % 256 == 0, "reduction state alignment");

static __device__ __align__(256) unsigned char scratch[kScratchBytes];
}  // namespace

void scratch_init(Device &d) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
        fail(NSFEM_HIP_ERROR, std::string("hipGetSymbolAddress(scratch): ") +
                                  hipGetErrorString(e));
    d.scratch = static_cast<unsigned char *>(ptr);
}

int run_cg_noalloc(Device &d, const CgRequest &req, nsfem_cg_stats *stats) {
    NSFEM_REQUIRE(d.scratch, NSFEM_NOT_READY, "device scratch not set up");
    NSFEM_REQUIRE(req.m && req.m->ready, NSFEM_NOT_READY, "matrix slot is empty");
    const int64_t values = (int64_t)req.m->rows * req.ncol;
    NSFEM_REQUIRE(values <= kNoAllocMaxValues, NSFEM_INVALID_ARGUMENT,
                  "no-allocation CG: rows x columns = " + std::to_string(values) +
                      " exceeds the scratch capacity of " + std::to_string(kNoAllocMaxValues) +
                      " values; use nsfem_cg_solve");
    NSFEM_REQUIRE(req.precision != NSFEM_PRECISION_FP32_REFINED || req.m->val32.ptr,
                  NSFEM_NOT_READY, "the matrix has no FP32 copy");
    CgWorkspace ws;
    ws.sync = reinterpret_cast<SyncState *>(d.scratch + kScratchSync);
    ws.res = reinterpret_cast<CgColumnResult *>(d.scratch + kScratchRes);
    ws.dot_partial = reinterpret_cast<double *>(d.scratch + kScratchDot);
    ws.scalars = reinterpret_cast<double *>(d.scratch + kScratchScal);
    ws.vectors = d.scratch + kScratchVec;
    ws.vec_bytes = kNoAllocVecBytes;
    return run_cg_in(d, req, stats, &ws);
}

// ------------------------------------------------------------ batched CG
namespace {

template <int NC, bool MIXED, typename IT, int WI>
void cg_batch_launch(Device &d, const CgArgs *args, const int2 *map, int grid) {
    void *kargs[] = {(void *)&args, (void *)&map};
    NSFEM_HIP(hipLaunchCooperativeKernel((const void *)k_cg_batch<NC, kCgBlock, MIXED, IT, WI>,
                                         dim3(grid), dim3(kCgBlock), kargs, 0, d.stream));
}

template <int NC, bool MIXED, typename IT, int WI>
int cg_batch_max_grid(Device &d) {
    int per_cu = 0;
    NSFEM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per_cu, k_cg_batch<NC, kCgBlock, MIXED, IT, WI>, kCgBlock, 0));
    return std::max(1, std::min(per_cu * d.cu_count, kMaxGridBlocks));
}

struct CgBatchMaxGrid {
    Device &d;
    int out;
    template <int NC, bool MX, typename IT, int WI>
    void run() { out = cg_batch_max_grid<NC, MX, IT, WI>(d); }
};
struct CgBatchLaunch {
    Device &d;
    const CgArgs *args;
    const int2 *map;
    int grid;
    template <int NC, bool MX, typename IT, int WI>
    void run() { cg_batch_launch<NC, MX, IT, WI>(d, args, map, grid); }
};

inline size_t round256(size_t b) { return (b + 255) / 256 * 256; }

// Blocks per instance, at most `maxg` in total.  Alone, an instance would get
// one block per 32 wave tiles (`scale` times that, its cap here).  When the
// batch wants more blocks than the device holds, every instance starts with
// one and the rest go, one at a time, to the instance with the largest
// expected time: wave tiles x iterations / blocks, with the iterations of a
// Poisson-type solve growing like the mesh width (tiles^0.5).  So the
// largest system, which needs the most iterations, does not become the
// batch's critical path on a fair share.
std::vector<int> share_blocks(const std::vector<const CgRequest *> &rq, int maxg,
                              const std::vector<int> &want, std::vector<int> nb) {
    const size_t I = rq.size();
    std::vector<double> work(I);
    int64_t total = 0, left = maxg;
    for (size_t i = 0; i < I; ++i) {
        work[i] = std::pow((double)std::max(1, rq[i]->m->n_wtiles), 1.5);
        total += want[i];
        left -= nb[i];
    }
    if (total <= maxg) return want;
    while (left > 0) {
        size_t big = I;
        double worst = -1.0;
        for (size_t i = 0; i < I; ++i) {
            if (nb[i] >= want[i]) continue;
            const double t = work[i] / nb[i];
            if (t > worst) {
                worst = t;
                big = i;
            }
        }
        if (big == I) break;
        ++nb[big];
        --left;
    }
    return nb;
}

std::vector<int> split_blocks(const std::vector<const CgRequest *> &rq, int maxg, int scale) {
    std::vector<int> want(rq.size());
    for (size_t i = 0; i < rq.size(); ++i) {
        const int tiles = std::max(1, rq[i]->m->n_wtiles);
        want[i] = std::min(tiles, std::max(1, tiles * scale / 32));
    }
    return share_blocks(rq, maxg, want, std::vector<int>(rq.size(), 1));
}

// One launch of a batch: its requests' numbers, the blocks of each and, for
// the resident form, what its kernel and windows hold.
struct BatchLaunch {
    std::vector<size_t> which;
    std::vector<int> blocks;
    std::vector<int> cap;
    bool resident = false;
    int width = 0, tiles = 0, waves = 0;
    size_t lds = 0;
};

// Plans of a system in a batch's resident launch, kept with the matrix's tiles
// as a single solve's is: a step plans three or more launches of the same
// matrices, and each plan walks a system's wave tiles.
int batch_kind(int nc, bool mixed, int w, int waves) {
    if (waves == kResWavesBatch) return 4;
    return mixed ? 3 : nc == 2 ? 2 : w == kResRowLong ? 1 : 0;
}
const ResidentPlan &batch_plan(Matrix &m, int nc, bool mixed, int w, int waves, int blocks) {
    ResidentPlan &plan = m.batch_plan[batch_kind(nc, mixed, w, waves)];
    if (!plan.made || plan.asked != blocks) {
        plan = ResidentPlan{};
        res_fits(m, nc, mixed, w, waves, blocks, plan);
        plan.made = true;
        plan.asked = blocks;
    }
    return plan;
}
// On the fewest blocks, at most `most`.
const ResidentPlan &batch_least(Matrix &m, int nc, bool mixed, int w, int waves, int most) {
    ResidentPlan &plan = m.batch_least[batch_kind(nc, mixed, w, waves)];
    if (!plan.made || plan.asked != most) {
        plan = ResidentPlan{};
        const int room = waves * res_tiles(mixed, w);
        int g = (m.n_wtiles + room - 1) / room;
        while (g <= std::min(most, m.n_wtiles) && !res_fits(m, nc, mixed, w, waves, g, plan)) ++g;
        plan.made = true;
        plan.asked = most;
    }
    return plan;
}

// The launches of a batch in the resident form, or none when a system does
// not allow it (refined: two columns and long rows never do).  Systems go
// largest first, so that those of like iteration counts share a launch, each
// with the fewest blocks it fits in; a launch's other blocks go where
// share_blocks sends them, up to a single solve's.
std::vector<BatchLaunch> resident_launches(Device &d, const std::vector<CgRequest> &reqs, int nc,
                                           bool mixed, int scale) {
    std::vector<BatchLaunch> out;
    if (!want_resident(nc, mixed) || (mixed && nc == 2)) return out;
    int w = nc == 1 ? kResRowShort : kResRowLong;
    for (const CgRequest &r : reqs) {
        const Matrix &m = *r.m;
        if (m.nnz <= 0 || m.shape.max_nz > kResRowLong || m.n_wtiles < 1) return out;
        if (m.shape.max_nz > kResRowShort) w = kResRowLong;
    }
    if (mixed && w == kResRowLong) return out;
    const int maxg = res_max_grid(d, res_kernel(nc, mixed, w, res_tiles(mixed, w), true), kResWaves,
                                  kResLds);
    std::vector<size_t> order(reqs.size());
    for (size_t i = 0; i < order.size(); ++i) order[i] = i;
    std::sort(order.begin(), order.end(), [&](size_t a, size_t b) {
        return reqs[a].m->n_wtiles != reqs[b].m->n_wtiles
                   ? reqs[a].m->n_wtiles > reqs[b].m->n_wtiles
                   : a < b;
    });
    std::vector<int> least(reqs.size());
    int used = maxg + 1;
    for (size_t i : order) {
        const ResidentPlan &plan = batch_least(*reqs[i].m, nc, mixed, w, kResWaves, maxg);
        if (!plan.ok) return std::vector<BatchLaunch>();
        const int g = plan.grid;
        least[i] = g;
        if (used + g > maxg) {
            out.emplace_back();
            used = 0;
        }
        used += g;
        out.back().which.push_back(i);
    }
    for (BatchLaunch &l : out) {
        std::vector<const CgRequest *> rq;
        std::vector<int> want, nb;
        for (size_t i : l.which) {
            const Matrix &m = *reqs[i].m;
            rq.push_back(&reqs[i]);
            nb.push_back(least[i]);
            want.push_back(std::max(
                least[i], std::min(m.n_wtiles, scale * m.n_wtiles /
                                                   (cg_tiles_per_wave(m) * kResWaves))));
        }
        l.blocks = share_blocks(rq, maxg, want, nb);
        l.resident = true;
        l.width = w;
        l.waves = kResWaves;
        for (size_t k = 0; k < rq.size(); ++k) {
            const ResidentPlan *plan = &batch_plan(*rq[k]->m, nc, mixed, w, kResWaves, l.blocks[k]);
            if (!plan->ok) {
                plan = &batch_least(*rq[k]->m, nc, mixed, w, kResWaves, maxg);
                l.blocks[k] = plan->grid;
            }
            l.cap.push_back(plan->cap);
            l.tiles = std::max(l.tiles, plan->tiles);
            l.lds = std::max(l.lds, plan->lds);
        }
    }
    return out;
}

// Puts a launch of refined one-column solves, split as the streaming form
// splits it, on the resident form where every system allows it: rows of at
// most kResRowShort nonzeros, windows that fit, and at most kFlatMax blocks
// each (past them the streaming form adds its sums as a tree).  Same blocks,
// same waves, same sums: the iterates are the streaming form's, bit for bit.
// Returns whether it did.  (Two refined columns stream: their two-phase
// iteration has no resident counterpart, and another iteration ends some
// systems a step earlier or later.)  Two steps of 16 refined cavities of 16^2
// to 128^2: 55.5 ms streaming, 24.1 with the pressure solves resident; with
// the velocity's resident too, in the single-reduction iteration, 20.4, but
// the fields moved by up to 6e-4 (inside what solves to 1e-8 leave).
bool batch_resident(Device &d, const std::vector<CgRequest> &reqs, BatchLaunch &l) {
    constexpr int nc = 1, w = kResRowShort;
    constexpr bool mixed = true;
    if (!want_resident(nc, mixed)) return false;
    std::vector<int> cap;
    int tiles = 0, grid = 0;
    size_t lds = 0;
    for (size_t k = 0; k < l.which.size(); ++k) {
        Matrix &m = *reqs[l.which[k]].m;
        if (m.nnz <= 0 || m.shape.max_nz > w || l.blocks[k] > kFlatMax) return false;
        const ResidentPlan &plan = batch_plan(m, nc, mixed, w, kResWavesBatch, l.blocks[k]);
        if (!plan.ok) return false;
        cap.push_back(plan.cap);
        tiles = std::max(tiles, plan.tiles);
        lds = std::max(lds, plan.lds);
        grid += l.blocks[k];
    }
    const void *fn = res_kernel(nc, mixed, w, tiles, true, kResWavesBatch);
    if (grid > res_max_grid(d, fn, kResWavesBatch, lds)) return false;
    l.cap = cap;
    l.resident = true;
    l.width = w;
    l.waves = kResWavesBatch;
    l.tiles = tiles;
    l.lds = lds;
    return true;
}

}  // namespace

int run_cg_batch(Device &d, const std::vector<CgRequest> &reqs, nsfem_cg_stats *stats,
                 int block_scale, double *batch_seconds, bool finish) {
    if (batch_seconds) *batch_seconds = 0.0;
    if (reqs.empty()) return NSFEM_OK;
    const int nc = reqs[0].ncol;
    const bool mixed = reqs[0].precision == NSFEM_PRECISION_FP32_REFINED;
    for (const CgRequest &r : reqs) {
        NSFEM_REQUIRE(r.m && r.m->ready && r.m->rows == r.m->cols, NSFEM_INVALID_ARGUMENT,
                      "batched CG needs square uploaded matrices");
        NSFEM_REQUIRE(r.ncol == nc && (r.precision == NSFEM_PRECISION_FP32_REFINED) == mixed &&
                          (mixed || r.precision == NSFEM_PRECISION_FP64),
                      NSFEM_INVALID_ARGUMENT,
                      "a batch needs one column count and one precision");
        NSFEM_REQUIRE(nc == 1 || nc == 2, NSFEM_INVALID_ARGUMENT, "columns must be 1 or 2");
    }
    bool idx16 = want_idx16();
    int wi = 4;
    std::vector<BatchLaunch> launches;
    if (!mixed) launches = resident_launches(d, reqs, nc, mixed, std::max(1, block_scale));
    if (launches.empty()) {
        // batched launches run 1024-thread blocks: one load per nonzero per
        // lane unless NSFEM_CG_PHASE says otherwise
        int form = mixed && nc == 1 ? phase_form(*reqs[0].m, false) : -1;
        for (const CgRequest &r : reqs) {
            idx16 = idx16 && r.m->dcol_ok;
            if (phase_form(*r.m, false) != form) form = -1;
            wi = std::max(wi, items_per_lane(*r.m));
        }
        if (form >= 0 && idx16) wi = form;
        CgBatchMaxGrid mg{d, 0};
        cg_dispatch(nc, mixed, idx16, wi, mg);
        const int maxg = mg.out;
        // instances beyond the co-resident block count run in further launches
        for (size_t first = 0; first < reqs.size(); first += (size_t)maxg) {
            BatchLaunch l;
            std::vector<const CgRequest *> rq;
            for (size_t i = first; i < std::min(reqs.size(), first + (size_t)maxg); ++i) {
                l.which.push_back(i);
                rq.push_back(&reqs[i]);
            }
            l.blocks = split_blocks(rq, maxg, std::max(1, block_scale));
            l.cap.assign(rq.size(), 0);
            launches.push_back(std::move(l));
        }
        // Refined one-column solves: resident on the streaming form's split
        // (its bits) where that fits.  A batch that wants more blocks than
        // the device has gives its small systems more tiles a wave than the
        // registers hold and takes the resident form's split (other bits, as
        // any change of the batch's split): 64 cavities of 16^2 to 256^2,
        // autotuned, 6.16 batch-steps/s streaming, 11.4 resident.
        if (mixed && nc == 1 && !(launches.size() == 1 && batch_resident(d, reqs, launches[0]))) {
            std::vector<BatchLaunch> own =
                resident_launches(d, reqs, nc, mixed, std::max(1, block_scale));
            if (!own.empty()) launches.swap(own);
        }
    }
    int worst = NSFEM_OK;
    const size_t vt = mixed ? sizeof(float) : sizeof(double);
    for (const BatchLaunch &launch : launches) {
        const size_t I = launch.which.size();
        std::vector<const CgRequest *> rq(I);
        for (size_t i = 0; i < I; ++i) rq[i] = &reqs[launch.which[i]];
        const std::vector<int> &nb = launch.blocks;
        // per-instance memory
        std::vector<size_t> voff(I), vbytes(I);
        size_t work = 0;
        for (size_t i = 0; i < I; ++i) {
            if (mixed) ensure_val32(d, *rq[i]->m);
            ensure_block_tiles(d, *rq[i]->m, nb[i]);
            vbytes[i] = round256((size_t)rq[i]->m->rows * nc * vt);
            voff[i] = work;
            work += 6 * vbytes[i];
        }
        const size_t sync_bytes = round256(sizeof(SyncState));
        d.batch_work.ensure(std::max<size_t>(work, 256));
        d.batch_sync.ensure(sync_bytes * I + 256);
        d.batch_res.ensure(2 * I);
        d.batch_args.ensure(sizeof(CgArgs) * I);
        d.batch_scal.ensure(2 * I);
        unsigned char *sm = d.batch_sync.ptr + (256 - ((uintptr_t)d.batch_sync.ptr % 256)) % 256;
        std::vector<CgArgs> args(I);
        std::vector<int2> map;
        for (size_t i = 0; i < I; ++i) {
            const CgRequest &r = *rq[i];
            Matrix &m = *r.m;
            CgArgs &a = args[i];
            a = CgArgs{};
            a.n = m.rows;
            a.nnz = (int)m.nnz;
            a.meta = m.wmeta.ptr;
            a.tiles = m.wtiles.ptr;
            a.block_tiles = m.block_tiles.ptr;
            a.rs = m.row_start.ptr;
            a.col = m.col.ptr;
            a.dcol = m.dcol.ptr;
            a.val64 = m.val.ptr;
            a.val32 = m.val32.ptr;
            a.b = r.b;
            a.x = r.x;
            unsigned char *w = d.batch_work.ptr + voff[i];
            a.r = w;
            a.p0 = w + vbytes[i];
            a.p1 = w + 2 * vbytes[i];
            a.q = w + 3 * vbytes[i];
            set_state_buffers(a, w, vbytes[i]);
            set_cg_params(d, r, m.rows, a);
            a.sync = reinterpret_cast<SyncState *>(sm + i * sync_bytes);
            a.res = d.batch_res.ptr + 2 * i;
            a.nblocks = nb[i];
            a.band_lo = m.shape.lo;
            a.band_hi = m.shape.hi;
            a.win_cap = launch.cap[i];
            for (int k = 0; k < nb[i]; ++k) map.push_back(make_int2((int)i, k));
        }
        const int grid = (int)map.size();
        if (std::getenv("NSFEM_CG_VERBOSE"))  // one line per launch, in launch order
            std::fprintf(stderr,
                         "[nsfem] cg batch launch instances=%zu cols=%d grid=%d mixed=%d "
                         "resident=%d waves=%d tiles=%d\n",
                         I, nc, grid, (int)mixed, launch.resident ? launch.width : 0,
                         launch.waves, launch.tiles);
        d.batch_map.ensure(map.size());
        NSFEM_HIP(hipMemcpyAsync(d.batch_args.ptr, args.data(), sizeof(CgArgs) * I,
                                 hipMemcpyHostToDevice, d.stream));
        NSFEM_HIP(hipMemcpyAsync(d.batch_map.ptr, map.data(), sizeof(int2) * map.size(),
                                 hipMemcpyHostToDevice, d.stream));
        for (size_t i = 0; i < I; ++i) {
            const int ng = (nb[i] + kGroup - 1) / kGroup;
            k_sync_reset<<<(ng + 255) / 256, 256, 0, d.stream>>>(args[i].sync, ng,
                                                                  launch.resident ? nb[i] : 0);
        }
        NSFEM_HIP(hipGetLastError());
        NSFEM_HIP(hipEventRecord(d.ev_start, d.stream));
        const CgArgs *dargs = reinterpret_cast<const CgArgs *>(d.batch_args.ptr);
        const int2 *dmap = d.batch_map.ptr;
        if (launch.resident) {
            void *kargs[] = {(void *)&dargs, (void *)&dmap};
            const void *fn =
                res_kernel(nc, mixed, launch.width, launch.tiles, true, launch.waves);
            NSFEM_REQUIRE(grid <= res_max_grid(d, fn, launch.waves, launch.lds), NSFEM_ERROR,
                          "batched CG: block split exceeds co-residency");
            NSFEM_HIP(hipLaunchCooperativeKernel(fn, dim3(grid), dim3(64 * launch.waves), kargs,
                                                 (unsigned)launch.lds, d.stream));
        } else {
            CgBatchLaunch ln{d, dargs, dmap, grid};
            cg_dispatch(nc, mixed, idx16, wi, ln);
        }
        NSFEM_HIP(hipEventRecord(d.ev_stop, d.stream));
        // FP64 true residuals of every instance, one host synchronisation
        if (!mixed) {
            launch_fill(d, (int)(nc * I), 0.0, d.batch_scal.ptr);
            for (size_t i = 0; i < I; ++i) {
                const CgRequest &r = *rq[i];
                double *tmp = (double *)args[i].q;  // n * nc doubles of scratch
                for (int c = 0; c < nc; ++c) {
                    const size_t off = (size_t)c * r.m->rows;
                    launch_spmv(d, *r.m, r.x + off, r.b + off, tmp, 1);
                    launch_dot_accumulate(d, r.m->rows, tmp, tmp, d.batch_scal.ptr + nc * i + c);
                }
            }
        }
        std::vector<CgColumnResult> res(2 * I);
        std::vector<double> tres(nc * I, 0.0);
        NSFEM_HIP(hipMemcpyAsync(res.data(), d.batch_res.ptr, sizeof(CgColumnResult) * 2 * I,
                                 hipMemcpyDeviceToHost, d.stream));
        if (!mixed)
            NSFEM_HIP(hipMemcpyAsync(tres.data(), d.batch_scal.ptr, sizeof(double) * nc * I,
                                     hipMemcpyDeviceToHost, d.stream));
        NSFEM_HIP(hipStreamSynchronize(d.stream));
        float ms = 0.f;
        NSFEM_HIP(hipEventElapsedTime(&ms, d.ev_start, d.ev_stop));
        if (batch_seconds) *batch_seconds += ms * 1e-3;
        for (size_t i = 0; i < I; ++i) {
            const CgRequest &r = *rq[i];
            bool redo = false;
            if (res[2 * i].status == kCgOutOfRange) {
                // from the x it came with, in the streaming form
                nsfem_cg_stats *st = stats + 2 * launch.which[i];
                int st2 = NSFEM_BREAKDOWN;
                if (finish) {
                    CgRequest r2 = r;
                    r2.resident = false;
                    st2 = run_cg(d, r2, st);
                    if (batch_seconds) *batch_seconds += st[0].seconds;
                } else {
                    for (int c = 0; c < nc; ++c) {
                        st[c] = nsfem_cg_stats{};
                        st[c].status = st2;
                    }
                }
                if (st2 != NSFEM_OK && worst == NSFEM_OK && finish) worst = st2;
                continue;
            }
            for (int c = 0; c < nc; ++c) {
                const CgColumnResult &cr = res[2 * i + c];
                if (cr.status == NSFEM_BARRIER_TIMEOUT)
                    fail(NSFEM_BARRIER_TIMEOUT, "batched CG kernel barrier timed out");
                const double fin = mixed ? cr.last_residual : std::sqrt(tres[nc * i + c]);
                if (cr.status != NSFEM_OK || fin > cr.tolerance * (1.0 + 1e-12)) redo = true;
                nsfem_cg_stats &st = stats[2 * launch.which[i] + c];
                st.iterations = cr.iterations;
                st.refinements = cr.refinements;
                st.status = cr.status;
                st.columns = nc;
                st.rhs_norm = cr.rhs_norm;
                st.initial_residual = cr.initial_residual;
                st.final_residual = fin;
                st.tolerance = cr.tolerance;
                st.seconds = ms * 1e-3;
            }
            if (redo && finish) {
                // stagnation, the iteration limit or FP64 drift: finish this
                // instance alone from its current x, to its original
                // absolute tolerance
                CgRequest r2 = r;
                r2.rtol = 0.0;
                r2.atol = res[2 * i].tolerance;
                if (nc == 2) r2.atol = std::min(r2.atol, res[2 * i + 1].tolerance);
                if (r2.max_iter > 0)
                    r2.max_iter = std::max(1, r2.max_iter - std::max(res[2 * i].iterations,
                                                                     res[2 * i + nc - 1].iterations));
                nsfem_cg_stats s2[2]{};
                const int st2 = run_cg(d, r2, s2);
                for (int c = 0; c < nc; ++c) {
                    nsfem_cg_stats &st = stats[2 * launch.which[i] + c];
                    st.iterations += s2[c].iterations;
                    st.refinements += s2[c].refinements + 1;
                    st.status = s2[c].status;
                    st.final_residual = s2[c].final_residual;
                    st.seconds += s2[c].seconds;
                }
                if (batch_seconds) *batch_seconds += s2[0].seconds;
                if (st2 != NSFEM_OK && worst == NSFEM_OK) worst = st2;
            }
        }
    }
    return worst;
}

}  // namespace nsfem
