// HIP kernels of the GeMSLR-FGMRES solve path (gfx950, wave64).
//
// Vector blocks are row-interleaved: entry (row i, column c) of an n x nrhs
// block is at [i * nrhs + c]; nrhs is a power of two <= 64 so that a wave
// holds whole rows of columns.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels_trsv.hpp"

namespace pgs {
namespace dev {

constexpr int kWave = 64;

// lane shuffle of a real or complex value
template <typename V>
__device__ __forceinline__ V shfl_xor_v(V v, int m, int width = kWave) { return __shfl_xor(v, m, width); }
template <typename R>
__device__ __forceinline__ cplx<R> shfl_xor_v(cplx<R> v, int m, int width = kWave) {
  return cplx<R>(__shfl_xor(v.re, m, width), __shfl_xor(v.im, m, width));
}

// One step of a sum over lanes: v plus the value of lane ^ M, by lane
// permutes of the vector unit (a ds_bpermute shuffle of a double is two LDS
// round trips).  M = 4 rotates a row of 16 lanes by 4, which is the same once
// the M = 8 step has made the row repeat after 8 lanes: the steps are taken
// from M = 32 down.
template <int M>
__device__ __forceinline__ double lane_step(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)u, hi = (unsigned)(u >> 32);
  if constexpr (M >= 16) {
    auto swap = [](unsigned x) {
      if constexpr (M == 32) return __builtin_amdgcn_permlane32_swap(x, x, false, false);
      else return __builtin_amdgcn_permlane16_swap(x, x, false, false);
    };
    const auto l = swap(lo);
    const auto h = swap(hi);
    const unsigned l0 = l[0], l1 = l[1], h0 = h[0], h1 = h[1];
    return __builtin_bit_cast(double, (unsigned long long)h0 << 32 | l0) +
           __builtin_bit_cast(double, (unsigned long long)h1 << 32 | l1);
  } else {
    constexpr int ctrl = M == 8 ? 0x128 : M == 4 ? 0x124 : M == 2 ? 0x4E : 0xB1;  // row_ror, quad_perm
    const unsigned l = (unsigned)__builtin_amdgcn_mov_dpp((int)lo, ctrl, 0xF, 0xF, true);
    const unsigned h = (unsigned)__builtin_amdgcn_mov_dpp((int)hi, ctrl, 0xF, 0xF, true);
    return v + __builtin_bit_cast(double, (unsigned long long)h << 32 | l);
  }
}
template <int M>
__device__ __forceinline__ float lane_step(float v) {
  const unsigned u = __float_as_uint(v);
  if constexpr (M == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  } else if constexpr (M == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  } else {
    constexpr int ctrl = M == 8 ? 0x128 : M == 4 ? 0x124 : M == 2 ? 0x4E : 0xB1;
    return v + __int_as_float(__builtin_amdgcn_mov_dpp((int)u, ctrl, 0xF, 0xF, true));
  }
}
template <int M, typename R>
__device__ __forceinline__ cplx<R> lane_step(cplx<R> v) {
  return cplx<R>(lane_step<M>(v.re), lane_step<M>(v.im));
}

// Sums each of the K values over the lanes that share lane % nl (nl a power
// of two, at most 64); every lane gets its class's sum.
template <int K, typename V>
__device__ __forceinline__ void lane_class_sums(V (&a)[K], int nl) {
#define PGS_LANE_STEP(M)                                \
  if (M >= nl) {                                        \
    _Pragma("unroll") for (int u = 0; u < K; ++u) a[u] = lane_step<M>(a[u]); \
  }
  PGS_LANE_STEP(32)
  PGS_LANE_STEP(16)
  PGS_LANE_STEP(8)
  PGS_LANE_STEP(4)
  PGS_LANE_STEP(2)
  PGS_LANE_STEP(1)
#undef PGS_LANE_STEP
}
template <typename V>
__device__ __forceinline__ V lane_class_sum(V v, int nl) {
  V a[1] = {v};
  lane_class_sums<1>(a, nl);
  return a[0];
}

// the value of lane `src` (the same in all lanes)
__device__ __forceinline__ double lane_value(double v, int src) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, src);
  const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), src);
  return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}
template <typename R>
__device__ __forceinline__ cplx<R> lane_value(cplx<R> v, int src) {
  return cplx<R>(lane_value(v.re, src), lane_value(v.im, src));
}

template <typename To, typename From>
__device__ __forceinline__ To cvt(From v) { return (To)v; }

// Streaming read of a basis value (non-temporal: each sweep reads a basis
// vector once, and the basis is far larger than the caches).  At 128^3 x 64
// the delayed-CGS2 dots, then with 8-byte loads, went from 0.69 to 0.76 of the
// HBM peak and the update from 0.58 to 0.59; the same loads of q and w and of
// the preconditioned basis in the solution update gained nothing.
__device__ __forceinline__ double ld_stream(const double* p) { return __builtin_nontemporal_load(p); }

// Row and column of element t of a row-interleaved block of nrhs columns.
// Every entry point admits only power-of-two column counts, so a shift and a
// mask replace the 64-bit division (tens of instructions per element in the
// per-element kernels); other counts take the division.
__device__ __forceinline__ int64_t row_of(int64_t t, int nrhs) {
  return (nrhs & (nrhs - 1)) == 0 ? t >> __builtin_ctz((unsigned)nrhs) : t / nrhs;
}
__device__ __forceinline__ int col_of(int64_t t, int nrhs) {
  return (nrhs & (nrhs - 1)) == 0 ? (int)(t & (nrhs - 1)) : (int)(t % nrhs);
}

// ---------------------------------------------------------------------------
// permutations (IntVectorClass::GatherPerm / ScatterRperm,
// ParGeMSLR/SRC/vectors/int_vector.cpp:629-696) fused with a precision change
// ---------------------------------------------------------------------------
// cscale (may be null): a per-column factor applied to the input first (the
// pending normalization of a Krylov vector)
template <typename VI, typename VO>
__global__ void k_gather(int64_t n, int nrhs, const int* __restrict__ perm, const VI* __restrict__ in, VO* __restrict__ out,
                         const double* __restrict__ cscale) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * nrhs) return;
  const int64_t i = row_of(t, nrhs);
  const int c = col_of(t, nrhs);
  VI a = in[(int64_t)perm[i] * nrhs + c];
  if (cscale) a *= VI(cscale[c]);
  out[t] = cvt<VO>(a);
}

// Four consecutive columns of a row per thread (nrhs a multiple of 4, both
// buffers 16-byte aligned): 16-byte and wider accesses instead of one value
// per lane.
template <typename V, int W>
struct alignas(W * sizeof(V) < 16 ? W * sizeof(V) : 16) ColPack {
  V v[W];
};

template <typename VI, typename VO>
__global__ void k_gather4(int64_t n, int nrhs, const int* __restrict__ perm, const VI* __restrict__ in,
                          VO* __restrict__ out, const double* __restrict__ cscale) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t e = 4 * t;
  if (e >= n * nrhs) return;
  const int64_t i = row_of(e, nrhs);
  const int c = col_of(e, nrhs);
  ColPack<VI, 4> a = *reinterpret_cast<const ColPack<VI, 4>*>(in + (int64_t)perm[i] * nrhs + c);
  if (cscale) {
#pragma unroll
    for (int u = 0; u < 4; ++u) a.v[u] *= VI(cscale[c + u]);
  }
  ColPack<VO, 4> b;
#pragma unroll
  for (int u = 0; u < 4; ++u) b.v[u] = cvt<VO>(a.v[u]);
  *reinterpret_cast<ColPack<VO, 4>*>(out + e) = b;
}

template <typename VI, typename VO>
__global__ void k_scatter4(int64_t n, int nrhs, const int* __restrict__ perm, const VI* __restrict__ in,
                           VO* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t e = 4 * t;
  if (e >= n * nrhs) return;
  const int64_t i = row_of(e, nrhs);
  const int c = col_of(e, nrhs);
  const ColPack<VI, 4> a = *reinterpret_cast<const ColPack<VI, 4>*>(in + e);
  ColPack<VO, 4> b;
#pragma unroll
  for (int u = 0; u < 4; ++u) b.v[u] = cvt<VO>(a.v[u]);
  *reinterpret_cast<ColPack<VO, 4>*>(out + (int64_t)perm[i] * nrhs + c) = b;
}

template <typename VI, typename VO>
__global__ void k_scatter(int64_t n, int nrhs, const int* __restrict__ perm, const VI* __restrict__ in, VO* __restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * nrhs) return;
  const int64_t i = row_of(t, nrhs);
  const int c = col_of(t, nrhs);
  out[(int64_t)perm[i] * nrhs + c] = cvt<VO>(in[t]);
}


// ---------------------------------------------------------------------------
// CSR SpMV (CsrMatrixPMatVecHostTemplate, ParGeMSLR/SRC/matrices/
// matrixops.cpp:5139-5330).  mode 0: y = alpha*A*x + beta*y (beta == 0 does
// not read y); mode 1: y = r - A*x.  Accumulation in VACC.
// Single RHS: LPR lanes per row, entries strided over the lanes, DPP/shuffle
// reduction.  Multi RHS: one thread per (row, column) over the row's entries.
// ---------------------------------------------------------------------------
// Workgroups are dealt to the 8 XCDs round-robin; the SpMV kernels renumber
// them so that XCD x takes the contiguous range [x * per, (x + 1) * per) of
// logical workgroups (per = gridDim.x / 8, the grid padded to a multiple of
// 8): the rows of one XCD are contiguous, and the x values their neighbours
// read stay in that XCD's L2.
constexpr int kXcds = 8;

__device__ __forceinline__ int64_t xcd_block() {
  const int64_t per = gridDim.x / kXcds;
  return (int64_t)(blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
}

template <typename VA, typename VX, typename VY, typename VACC, int LPR>
__global__ void k_spmv1(int nrows, const int* __restrict__ ia, const int* __restrict__ ja, const VA* __restrict__ a,
                        const VX* __restrict__ x, VY* __restrict__ y, const VY* __restrict__ r, VACC alpha, VACC beta,
                        int mode) {
  int64_t g = xcd_block() * blockDim.x + threadIdx.x;
  int row = (int)(g / LPR);
  int q = (int)(g % LPR);
  VACC acc = 0;
  if (row < nrows) {
    int k1 = ia[row + 1];
    for (int k = ia[row] + q; k < k1; k += LPR) acc += (VACC)a[k] * (VACC)x[ja[k]];
  }
#pragma unroll
  for (int m = LPR / 2; m > 0; m >>= 1) acc += shfl_xor_v(acc, m, LPR);
  if (row < nrows && q == 0) {
    if (mode == 1) y[row] = cvt<VY>((VACC)r[row] - acc);
    else if (beta == (VACC)0) y[row] = cvt<VY>(alpha * acc);
    else y[row] = cvt<VY>(alpha * acc + beta * (VACC)y[row]);
  }
}

template <typename VA, typename VX, typename VY, typename VACC>
__global__ void k_spmvN(int nrows, int nrhs, const int* __restrict__ ia, const int* __restrict__ ja,
                        const VA* __restrict__ a, const VX* __restrict__ x, VY* __restrict__ y,
                        const VY* __restrict__ r, VACC alpha, VACC beta, int mode) {
  int64_t t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= (int64_t)nrows * nrhs) return;
  const int row = (int)row_of(t, nrhs);
  const int c = col_of(t, nrhs);
  // the element this thread updates is loaded first, in flight with the row's entries
  const VACC y0 = mode == 1 ? (VACC)r[t] : (beta == (VACC)0 ? VACC(0) : (VACC)y[t]);
  VACC acc = 0;
  const int k1 = ia[row + 1];
  // eight entries at a time: their indices and values, then their x gathers,
  // are all in flight before the first multiply-add (summed in entry order)
  for (int k = ia[row]; k < k1; k += 8) {
    int jj[8];
    VACC av[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const bool in = k + u < k1;
      jj[u] = in ? ja[k + u] : 0;
      av[u] = in ? (VACC)a[k + u] : VACC(0);
    }
    VACC xv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) xv[u] = k + u < k1 ? (VACC)x[(int64_t)jj[u] * nrhs + c] : VACC(0);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k + u < k1) acc += av[u] * xv[u];
  }
  if (mode == 1) y[t] = cvt<VY>(y0 - acc);
  else if (beta == (VACC)0) y[t] = cvt<VY>(alpha * acc);
  else y[t] = cvt<VY>(alpha * acc + beta * y0);
}

// CW (4 or 8) consecutive columns per thread (nrhs a multiple of CW, x, y
// and r 16-byte aligned): the row's indices and values are loaded once for
// CW columns and every x gather and y access is 16 bytes or wider; each
// column's sum runs over the entries in the same order as k_spmvN.
template <typename VA, typename VX, typename VY, typename VACC, int CW = 4>
__global__ void k_spmvN4(int nrows, int nrhs, const int* __restrict__ ia, const int* __restrict__ ja,
                         const VA* __restrict__ a, const VX* __restrict__ x, VY* __restrict__ y,
                         const VY* __restrict__ r, VACC alpha, VACC beta, int mode) {
  const int64_t e = CW * (xcd_block() * blockDim.x + threadIdx.x);
  if (e >= (int64_t)nrows * nrhs) return;
  const int row = (int)row_of(e, nrhs);
  const int c = col_of(e, nrhs);
  using PY = ColPack<VY, CW>;
  using PX = ColPack<VX, CW>;
  PY y0;
  if (mode == 1) y0 = *reinterpret_cast<const PY*>(r + e);
  else if (!(beta == (VACC)0)) y0 = *reinterpret_cast<const PY*>(y + e);
  VACC acc[CW];
#pragma unroll
  for (int q = 0; q < CW; ++q) acc[q] = VACC(0);
  const int k1 = ia[row + 1];
  for (int k = ia[row]; k < k1; k += 8) {
    int jj[8];
    VACC av[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const bool in = k + u < k1;
      jj[u] = in ? ja[k + u] : 0;
      av[u] = in ? (VACC)a[k + u] : VACC(0);
    }
    PX xv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k + u < k1) xv[u] = *reinterpret_cast<const PX*>(x + (int64_t)jj[u] * nrhs + c);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k + u < k1) {
#pragma unroll
        for (int q = 0; q < CW; ++q) acc[q] += av[u] * (VACC)xv[u].v[q];
      }
  }
  PY out;
#pragma unroll
  for (int q = 0; q < CW; ++q) {
    if (mode == 1) out.v[q] = cvt<VY>((VACC)y0.v[q] - acc[q]);
    else if (beta == (VACC)0) out.v[q] = cvt<VY>(alpha * acc[q]);
    else out.v[q] = cvt<VY>(alpha * acc[q] + beta * (VACC)y0.v[q]);
  }
  *reinterpret_cast<PY*>(y + e) = out;
}

// (block-diagonal ILU solves: kernels_trsv.hpp)

// ---------------------------------------------------------------------------
// Low-rank correction z += WH (W^H z) (GemslrClass::SolveApplyLowRankLevel,
// ParGeMSLR/SRC/preconditioners/gemslr.cpp:3681-3719).  W, WH row-major m x k.
// Stage 1: per-workgroup partial sums of W^H z for every (j, column);
// stage 2: sum of the partials (fixed order -> deterministic);
// stage 3: z[i, c] += sum_j WH[i, j] t[j, c].
// ---------------------------------------------------------------------------
template <typename V, int NT>
__global__ __launch_bounds__(NT) void k_lr_dot(int m, int k, int nrhs, const V* __restrict__ W,
                                               const V* __restrict__ z, V* __restrict__ part, int rows_per_blk) {
  // thread layout: c = tid % nrhs, row lane = tid / nrhs
  __shared__ V sh[NT];
  const int tid = threadIdx.x;
  const int c = tid % nrhs;
  const int lanes = NT / nrhs;
  const int rl = tid / nrhs;
  const int i0 = blockIdx.x * rows_per_blk;
  const int i1 = min(m, i0 + rows_per_blk);
  for (int j = 0; j < k; ++j) {
    V acc = 0;
    for (int i = i0 + rl; i < i1; i += lanes) acc += sconj(W[(int64_t)i * k + j]) * z[(int64_t)i * nrhs + c];
    sh[tid] = acc;
    __syncthreads();
    for (int s = NT / 2; s >= nrhs; s >>= 1) {
      if (tid < s) sh[tid] += sh[tid + s];
      __syncthreads();
    }
    if (tid < nrhs) part[((int64_t)blockIdx.x * k + j) * nrhs + tid] = sh[tid];
    __syncthreads();
  }
}

// Stage 1 with the k partial sums of an element in registers (KM >= k,
// loops unrolled to KM with the uniform guard j < k): every lane walks the
// elements g = (i, c) of z with a grid stride and adds conj(W[i, j]) * z[i, c] to
// sum j; the sums are then reduced over the lanes of a column and over the
// waves into part[blk * k * nrhs + j * nrhs + c].  Dynamic LDS:
// (NT / 64) * k * nrhs values of V.
template <typename V, int NT, int KM>
__global__ __launch_bounds__(NT) void k_lr_dot_reg(int m, int k, int nrhs, const V* __restrict__ W,
                                                   const V* __restrict__ z, V* __restrict__ part) {
  extern __shared__ unsigned char lr_smem[];
  V* red = reinterpret_cast<V*>(lr_smem);
  const int tid = threadIdx.x;
  V acc[KM];
#pragma unroll
  for (int j = 0; j < KM; ++j) acc[j] = 0;
  const int64_t total = (int64_t)m * nrhs;
  for (int64_t g = (int64_t)blockIdx.x * NT + tid; g < total; g += (int64_t)gridDim.x * NT) {
    const V zv = z[g];
    const V* wr = W + row_of(g, nrhs) * k;
#pragma unroll
    for (int j = 0; j < KM; ++j)
      if (j < k) acc[j] += sconj(wr[j]) * zv;
  }
  const int wid = tid / 64, lane = tid % 64;
  lane_class_sums<KM>(acc, nrhs);
#pragma unroll
  for (int j = 0; j < KM; ++j)
    if (j < k && lane < nrhs) red[(wid * k + j) * nrhs + lane] = acc[j];
  __syncthreads();
  for (int t = tid; t < k * nrhs; t += NT) {
    V s = 0;
    for (int q = 0; q < NT / 64; ++q) s += red[q * k * nrhs + t];
    part[(int64_t)blockIdx.x * k * nrhs + t] = s;
  }
}

template <typename V>
__global__ void k_lr_final(int nblk, int k, int nrhs, const V* __restrict__ part, V* __restrict__ t) {
  // one wave per output, four per workgroup of 256; fixed summation order
  const int g = blockIdx.x * 4 + threadIdx.x / 64;
  const int lane = threadIdx.x % 64;
  if (g >= k * nrhs) return;  // whole wave exits together
  V s = 0;
  for (int b = lane; b < nblk; b += 64) s += part[(int64_t)b * k * nrhs + g];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += shfl_xor_v(s, o);
  if (lane == 0) t[g] = s;
}

// z += WH t with t summed here from the nblk partials of stage 1, by every
// workgroup for itself: while the partials are few (kLrFused values) that costs
// less than the launch that would sum them.  Stage 1 with its lane sums by lane
// permutes and this: 48^3, one FP64 column, rank 16, 20 -> 10.1 us per term in three
// launches -> two.  An apply with one term against the same with the third launch,
// 16^3 to 64^3, 1 to 4 columns: rank 16 up to 3 us less, rank 32 up to 5, rank 3
// with one column 2 us more (there a lane adds up 85 others' sums); 500 x 401, rank
// 16, 2 columns: 4 to 6 us more.  Dynamic LDS: k * nrhs values.
constexpr int kLrFused = 4096;

template <typename V, int NT>
__global__ __launch_bounds__(NT) void k_lr_update_sum(int m, int k, int nrhs, int nblk, const V* __restrict__ WH,
                                                      const V* __restrict__ part, V* __restrict__ z) {
  extern __shared__ unsigned char lu_smem[];
  V* t = reinterpret_cast<V*>(lu_smem);
  __shared__ V red[NT];
  const int no = k * nrhs, tid = threadIdx.x;
  if (no >= NT) {
    for (int o = tid; o < no; o += NT) {
      V s = part[o];
#pragma unroll 4
      for (int b = 1; b < nblk; ++b) s += part[b * no + o];
      t[o] = s;
    }
  } else {
    const int ng = NT / no, g = tid / no, o = tid % no;
    V s = 0;
    if (g < ng) {
#pragma unroll 4
      for (int b = g; b < nblk; b += ng) s += part[b * no + o];
    }
    red[tid] = s;
    __syncthreads();
    if (tid < no) {
      for (int q = 1; q < ng; ++q) s += red[q * no + tid];
      t[tid] = s;
    }
  }
  __syncthreads();
  const int64_t g = (int64_t)blockIdx.x * NT + tid;
  if (g >= (int64_t)m * nrhs) return;
  const int64_t i = row_of(g, nrhs);
  const int c = col_of(g, nrhs);
  V acc = 0;
  for (int j = 0; j < k; ++j) acc += WH[i * k + j] * t[j * nrhs + c];
  z[g] += acc;
}

template <typename V>
__global__ void k_lr_update(int m, int k, int nrhs, const V* __restrict__ WH, const V* __restrict__ t, V* __restrict__ z) {
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= (int64_t)m * nrhs) return;
  const int64_t i = row_of(g, nrhs);
  const int c = col_of(g, nrhs);
  V acc = 0;
  for (int j = 0; j < k; ++j) acc += WH[i * k + j] * t[j * nrhs + c];
  z[g] += acc;
}

// ---------------------------------------------------------------------------
// The same low-rank term on the matrix cores for a block of FP32 columns
// (nrhs = 16 * CT with CT = 1, 2, 4; k <= 16 * KT with KT = 1, 2):
// v_mfma_f32_16x16x4_f32 tiles.  Lane layout of one 16x16x4 product
// D = A B + C: A[i][q] comes from lane i + 16 q, B[q][j] from lane j + 16 q,
// and lane j + 16 r holds D[4 r + e][j] in element e.
// ---------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Stage 1: each wave multiplies W^T (k x its rows) by z (its rows x nrhs)
// four rows per product, with the rank index as the product's rows and the
// columns as its columns; the four waves' tiles are summed in LDS and written
// as the workgroup's partial part[blk * k * nrhs + j * nrhs + c] (summed over
// the workgroups by k_lr_final).  rows_per_wave is a multiple of 4.
template <int KT, int CT>
__global__ __launch_bounds__(256) void k_lr_dot_mfma(int m, int k, int nrhs, const float* __restrict__ W,
                                                     const float* __restrict__ z, float* __restrict__ part,
                                                     int rows_per_wave) {
  __shared__ float red[4][KT * 16][CT * 16];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int jj = lane & 15, q = lane >> 4;
  const int64_t gw = (int64_t)blockIdx.x * 4 + wv;
  const int64_t i_begin = gw * rows_per_wave;
  const int64_t i_end = min((int64_t)m, i_begin + rows_per_wave);
  f32x4 acc[KT][CT];
#pragma unroll
  for (int h = 0; h < KT; ++h)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[h][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nit = i_end > i_begin ? (int)((i_end - i_begin + 3) / 4) : 0;
  for (int it = 0; it < nit; ++it) {
    const int64_t i = i_begin + 4 * it + q;
    const bool ok = i < i_end;
    float a[KT], b[CT];
#pragma unroll
    for (int h = 0; h < KT; ++h) {
      const int j = 16 * h + jj;
      a[h] = (ok && j < k) ? W[i * k + j] : 0.f;
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) b[ct] = ok ? z[i * nrhs + 16 * ct + jj] : 0.f;
#pragma unroll
    for (int h = 0; h < KT; ++h)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) acc[h][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[h], b[ct], acc[h][ct], 0, 0, 0);
  }
#pragma unroll
  for (int h = 0; h < KT; ++h)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int e = 0; e < 4; ++e) red[wv][16 * h + 4 * q + e][16 * ct + jj] = acc[h][ct][e];
  __syncthreads();
  for (int t = threadIdx.x; t < k * nrhs; t += 256) {
    const int j = t / nrhs, c = t % nrhs;
    part[(int64_t)blockIdx.x * k * nrhs + t] = (red[0][j][c] + red[1][j][c]) + (red[2][j][c] + red[3][j][c]);
  }
}

// Stage 3: z[i, c] += sum_j WH[i, j] t[j, c], one 16-row tile per wave.  The
// rank index of product q and operand row p is j = 16 h + 4 p + q, so a lane
// loads WH[i, 16 h + 4 p .. + 3] as one 16-byte vector (k % 4 == 0) and
// feeds its four values to four products; t's operands use the same j.
template <int KT, int CT>
__global__ __launch_bounds__(256) void k_lr_update_mfma(int m, int k, int nrhs, const float* __restrict__ WH,
                                                        const float* __restrict__ t, float* __restrict__ z) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int jj = lane & 15, p = lane >> 4;
  const int64_t i0 = ((int64_t)blockIdx.x * 4 + wv) * 16;
  if (i0 >= m) return;  // whole wave
  float bt[KT][4][CT];
#pragma unroll
  for (int h = 0; h < KT; ++h)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int j = 16 * h + 4 * p + q;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) bt[h][q][ct] = j < k ? t[j * nrhs + 16 * ct + jj] : 0.f;
    }
  const int64_t i = i0 + jj;
  float a[KT][4];
#pragma unroll
  for (int h = 0; h < KT; ++h) {
    const int j0 = 16 * h + 4 * p;
    if ((k & 3) == 0 && i < m && j0 + 3 < k) {
      const float4 v = *reinterpret_cast<const float4*>(WH + i * k + j0);
      a[h][0] = v.x;
      a[h][1] = v.y;
      a[h][2] = v.z;
      a[h][3] = v.w;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) a[h][q] = (i < m && j0 + q < k) ? WH[i * k + j0 + q] : 0.f;
    }
  }
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    f32x4 c;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t r = i0 + 4 * p + e;
      c[e] = r < m ? z[r * nrhs + 16 * ct + jj] : 0.f;
    }
#pragma unroll
    for (int h = 0; h < KT; ++h)
#pragma unroll
      for (int q = 0; q < 4; ++q) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[h][q], bt[h][q][ct], c, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t r = i0 + 4 * p + e;
      if (r < m) z[r * nrhs + 16 * ct + jj] = c[e];
    }
  }
}

// ---------------------------------------------------------------------------
// Krylov kernels (FP64).  A block of p vectors V_j (each n x nrhs) at
// V + j*ldv.  State per column in KState.
// ---------------------------------------------------------------------------
// Delayed CGS2: a tentative basis vector whose squared distance from the
// span of the final ones, q.q - |s|^2, is at most this fraction of q.q is
// taken as dependent (it lies in the span to working precision).
constexpr double kDcgs2DependentTol = 1e-10;

struct KState {
  double normb, tolr, normr, scale;
  int active;   // running in the current cycle
  int status;   // 0 running, 1 converged, 2 breakdown, 3 max iterations, 4 zero rhs/residual,
                // 5 non-finite value (NaN or Inf in b, x0 or the iteration): retired at once
  int iters;    // total inner iterations (FlexGmresClass::_iter)
  int icur;     // inner steps of the current cycle
};

// A column's state for the host: kStateActive while it runs in the current
// cycle, kStateRunning while it may go on in another one.  The kernel that
// settles a step's state writes it for its column straight into host memory.
constexpr int kStateActive = 1, kStateRunning = 2;
__device__ __forceinline__ int state_bits(const KState& s, int maxits) {
  return (s.active ? kStateActive : 0) | (s.status == 0 && s.iters < maxits ? kStateRunning : 0);
}

// The first p - 1 rotations applied to h_0..h_{p-1}: writes the finished
// entries 0..p-2 to `out` (global memory, so that the reads of h and of the
// rotations in LDS need not wait for the writes), returns entry p-1.
template <typename S>
__device__ __forceinline__ S rotate_column(int p, const S* h, const S* cl, const S* sl, S* out) {
  S hi = h[0];
#pragma unroll 4
  for (int j = 1; j < p; ++j) {
    const S hj = h[j], cj = cl[j - 1], sj = sl[j - 1];
    out[j - 1] = sconj(cj) * hi + sj * hj;
    hi = -sj * hi + cj * hj;
  }
  return hi;
}

constexpr int kTailNT = 256;  // threads of the kernels that close a step, one workgroup per column

// Sum of part[b * nrhs + c] over b < nblk in a fixed order (all kTailNT
// threads of a workgroup; red holds one value per wave).
__device__ __forceinline__ double column_sum(int nblk, int nrhs, int c, const double* __restrict__ part, double* red) {
  double t = 0.0;
#pragma unroll 4
  for (int b = threadIdx.x; b < nblk; b += kTailNT) t += part[(int64_t)b * nrhs + c];
  t = lane_class_sum(t, 1);
  if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = t;
  __syncthreads();
  t = red[0];
  for (int k = 1; k < kTailNT / kWave; ++k) t += red[k];
  return t;
}

// partial dot products d[j, c] = sum_rows conj(V_j[r, c]) * w[r, c] for j < p
// (w may be one of the V_j), accumulated in S.  One partial per workgroup.
template <typename VV, typename VW, typename S, int NT>
__global__ __launch_bounds__(NT) void k_multidot(int64_t n, int nrhs, int p, const VV* __restrict__ V, int64_t ldv,
                                                 const VW* __restrict__ w, S* __restrict__ part,
                                                 int64_t rows_per_blk) {
  __shared__ S sh[NT];
  const int tid = threadIdx.x;
  const int c = tid % nrhs;
  const int lanes = NT / nrhs;
  const int rl = tid / nrhs;
  const int64_t i0 = (int64_t)blockIdx.x * rows_per_blk;
  const int64_t i1 = min(n, i0 + rows_per_blk);
  for (int j = 0; j < p; ++j) {
    const VV* vj = V + j * ldv;
    S acc = 0;
    for (int64_t i = i0 + rl; i < i1; i += lanes) acc += sconj((S)vj[i * nrhs + c]) * (S)w[i * nrhs + c];
    // reduce across lanes that share column c
    for (int m = kWave / 2; m >= nrhs; m >>= 1) acc += shfl_xor_v(acc, m);
    const int wid = tid / kWave, lane = tid % kWave;
    if (lane < nrhs) sh[wid * nrhs + lane] = acc;
    __syncthreads();
    if (tid < nrhs) {
      S s = 0;
      for (int q = 0; q < NT / kWave; ++q) s += sh[q * nrhs + tid];
      part[((int64_t)blockIdx.x * p + j) * nrhs + tid] = s;
    }
    __syncthreads();
  }
}

// per-workgroup partial sums of |x[r, c]|^2
template <typename S, int NT>
__global__ __launch_bounds__(NT) void k_colnorm2(int64_t n, int nrhs, const S* __restrict__ x,
                                                 double* __restrict__ part, int64_t rows_per_blk) {
  __shared__ double sh[NT];
  const int tid = threadIdx.x;
  const int c = tid % nrhs;
  const int lanes = NT / nrhs;
  const int64_t i0 = (int64_t)blockIdx.x * rows_per_blk;
  const int64_t i1 = min(n, i0 + rows_per_blk);
  double acc = 0;
  for (int64_t i = i0 + tid / nrhs; i < i1; i += lanes) acc += (double)sabs2(x[i * nrhs + c]);
  for (int m = kWave / 2; m >= nrhs; m >>= 1) acc += __shfl_xor(acc, m);
  const int wid = tid / kWave, lane = tid % kWave;
  if (lane < nrhs) sh[wid * nrhs + lane] = acc;
  __syncthreads();
  if (tid < nrhs) {
    double s = 0;
    for (int q = 0; q < NT / kWave; ++q) s += sh[q * nrhs + tid];
    part[(int64_t)blockIdx.x * nrhs + tid] = s;
  }
}

// out[g] = sum over the nblk partials of output g (one wave per output; the
// partials are summed in a fixed order, so the result does not depend on
// timing).  Grid: ceil(p*nrhs / 4) workgroups of 256 threads.
__global__ __launch_bounds__(256) void k_dot_final_wave(int nblk, int p, int nrhs, const double* __restrict__ part,
                                                        double* __restrict__ out, int accumulate) {
  const int g = blockIdx.x * 4 + threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  const int total = p * nrhs;
  if (g >= total) return;  // whole wave exits together
  double s = 0;
  for (int b = lane; b < nblk; b += kWave) s += part[(int64_t)b * total + g];
#pragma unroll
  for (int m = kWave / 2; m > 0; m >>= 1) s += __shfl_xor(s, m);
  if (lane == 0) out[g] = accumulate ? out[g] + s : s;
}

// w[r, c] -= sum_{j<p} V_j[r, c] * h[j, c]  and, when part != nullptr, the
// per-workgroup partial sums of |w[r, c]|^2 (part[blk * nrhs + c]).  V and w
// hold VV, h and the arithmetic S (VV = S, or float vectors with double
// coefficients).  Dynamic shared memory: p*nrhs values of S, then
// (NT/64)*nrhs doubles.
template <typename VV, typename S, int NT>
__global__ __launch_bounds__(NT) void k_multi_axpy_norm(int64_t n, int nrhs, int p, const VV* __restrict__ V,
                                                        int64_t ldv, const S* __restrict__ h,
                                                        VV* __restrict__ w, double* __restrict__ part) {
  extern __shared__ unsigned char ma_smem[];
  S* hs = reinterpret_cast<S*>(ma_smem);
  double* red = reinterpret_cast<double*>(hs + p * nrhs);
  for (int t = threadIdx.x; t < p * nrhs; t += NT) hs[t] = h[t];
  __syncthreads();
  const int tid = threadIdx.x;
  const int c = tid % nrhs;
  const int64_t per_blk = (n + gridDim.x - 1) / gridDim.x;
  const int64_t i0 = (int64_t)blockIdx.x * per_blk;
  const int64_t i1 = min(n, i0 + per_blk);
  const int lanes = NT / nrhs;
  double sq = 0;
  for (int64_t i = i0 + tid / nrhs; i < i1; i += lanes) {
    const int64_t g = i * nrhs + c;
    S acc = (S)w[g];
    for (int j = 0; j < p; ++j) acc -= (S)V[j * ldv + g] * hs[j * nrhs + c];
    const VV out = (VV)acc;
    w[g] = out;
    sq += (double)sabs2(out);
  }
  if (part == nullptr) return;  // uniform
  for (int m = kWave / 2; m >= nrhs; m >>= 1) sq += __shfl_xor(sq, m);
  const int wid = tid / kWave, lane = tid % kWave;
  if (lane < nrhs) red[wid * nrhs + lane] = sq;
  __syncthreads();
  if (tid < nrhs) {
    double s = 0;
    for (int q = 0; q < NT / kWave; ++q) s += red[q * nrhs + tid];
    part[(int64_t)blockIdx.x * nrhs + tid] = s;
  }
}

// One classical Gram-Schmidt sweep over the basis V_0..V_{p-1} with an
// element's basis values and the partial sums held in registers.  LPE lanes
// share an element (consecutive lanes); lane `sub` of an element holds V_j for
// j = u * LPE + sub, u < pu = ceil(p / LPE) <= PM (compile-time bound; loops
// are unrolled to PM with the wave-uniform guard u < pu, and all loads of an
// element are issued before any is used).  With LPE = 2 and p odd, lane 1
// reads V_p (which must be readable) and gives it weight zero.
//   MODE 0: d[j, c] = sum_rows V_j[r, c] * w[r, c]
//   MODE 1: w -= sum_j V_j h[j, :], then d as in mode 0 with the updated w
//           from the same registers (V is read once for both)
//   MODE 2: w -= sum_j V_j h[j, :], then d[0, c] = sum_rows w[r, c]^2
// The update sums V_j h[j, :] in increasing j within a lane (with LPE = 2 the
// two lanes' sums are added) and subtracts the sum.  Every lane walks the
// elements (blockIdx.x * NT + tid) / LPE + k * gridDim.x * NT / LPE; at the
// end the sums are reduced over the lanes of a column, then over the waves,
// into part[blk * q * nrhs + j * nrhs + c], q = p (modes 0, 1) or 1 (mode 2),
// in a fixed order (deterministic).  Requires nrhs * LPE <= 64.
// Dynamic LDS: (MODE ? p * nrhs : 0) + (NT / 64) * q * nrhs doubles.
template <int NT, int PM, int MODE, int LPE>
__global__ __launch_bounds__(NT) void k_basis_reg(int64_t n, int nrhs, int p, const double* __restrict__ V,
                                                  int64_t ldv, const double* __restrict__ h, double* __restrict__ w,
                                                  double* __restrict__ part) {
  static_assert(MODE != 2 || LPE == 1, "the norm sweep uses one lane per element");
  constexpr int NA = MODE == 2 ? 1 : PM;  // partial sums per lane
  const int q = MODE == 2 ? 1 : p;        // outputs per column
  extern __shared__ double sm[];
  double* hs = sm;
  double* red = sm + (MODE ? p * nrhs : 0);
  const int tid = threadIdx.x;
  if (MODE)
    for (int t = tid; t < p * nrhs; t += NT) hs[t] = h[t];
  __syncthreads();
  const int sub = tid % LPE;
  const int c = (tid / LPE) % nrhs;
  const int pu = (p + LPE - 1) / LPE;
  const double* Vl = V + (int64_t)sub * ldv;
  double acc[NA];
#pragma unroll
  for (int u = 0; u < NA; ++u) acc[u] = 0;
  const int64_t total = n * nrhs;
  const int64_t stride = (int64_t)gridDim.x * (NT / LPE);
  for (int64_t g = ((int64_t)blockIdx.x * NT + tid) / LPE; g < total; g += stride) {
    double wv = w[g];
    double v[PM];
#pragma unroll
    for (int u = 0; u < PM; ++u)
      if (u < pu) v[u] = ld_stream(Vl + (int64_t)(u * LPE) * ldv + g);
    if constexpr (MODE != 0) {
      double sv = 0;
#pragma unroll
      for (int u = 0; u < PM; ++u)
        if (u < pu) {
          const int j = u * LPE + sub;
          sv += v[u] * (j < p ? hs[j * nrhs + c] : 0.0);
        }
      if constexpr (LPE == 2) sv += __shfl_xor(sv, 1);
      wv -= sv;
      if (sub == 0) w[g] = wv;
    }
    if constexpr (MODE == 2) {
      acc[0] += wv * wv;
    } else {
#pragma unroll
      for (int u = 0; u < PM; ++u)
        if (u < pu) acc[u] += v[u] * wv;
    }
  }
  const int wid = tid / kWave, lane = tid % kWave;
#pragma unroll
  for (int u = 0; u < NA; ++u) {
    if (u < (MODE == 2 ? 1 : pu)) {
      const int j = MODE == 2 ? 0 : u * LPE + sub;
      double s = acc[u];
      for (int m = kWave / 2; m >= nrhs * LPE; m >>= 1) s += __shfl_xor(s, m);
      if (lane < nrhs * LPE && j < q) red[(wid * q + j) * nrhs + lane / LPE] = s;
    }
  }
  __syncthreads();
  for (int t = tid; t < q * nrhs; t += NT) {
    double s = 0;
    for (int k = 0; k < NT / kWave; ++k) s += red[k * q * nrhs + t];
    part[(int64_t)blockIdx.x * q * nrhs + t] = s;
  }
}

// ---------------------------------------------------------------------------
// Delayed CGS2 (PGS_ORTH_DCGS2, real bases): the re-orthogonalization of the
// newest basis vector q is done in the next step's sweep, together with the
// first projection of the next vector w, so a step reads the basis twice
// instead of three times.  Basis slots 0..p-1 are final, q is tentative.
// ---------------------------------------------------------------------------

// 16 bytes of consecutive values as one load or store; the address need only
// be aligned for a value
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef f64x2 f64x2_a8 __attribute__((aligned(8)));

__device__ __forceinline__ f64x2 load16(const void* x) { return *reinterpret_cast<const f64x2_a8*>(x); }
__device__ __forceinline__ f64x2 stream16(const void* x) {  // as ld_stream
  return __builtin_nontemporal_load(reinterpret_cast<const f64x2_a8*>(x));
}

// Dots of the basis V_0..V_{p-1} with q and with w (w may be null), in chunks
// of `chunk` <= kDotsChunk vectors (blockIdx.y): per workgroup partials
// part[blockIdx.x * nout * nrhs + o * nrhs + c] for
//   o < p:             V_o . q
//   p <= o < 2 p:      V_{o-p} . w       (w != null)
//   o = 2 p, 2 p + 1:  q . q and q . w   (w != null)
//   o = p:             q . q             (w == null)
// A stream over the basis, bound by HBM.  The waves of a workgroup walk the
// same elements (their reads of q and w meet in the cache of the CU) and
// share out the chunk's vectors: wave k takes j0 + k, j0 + k + NW, ..., at most
// kDotsPM of them, 16 bytes of each per lane (two real values or a complex
// one), and keeps their sums, so that the sums are only reduced over a wave's
// lanes.  ONE: a single real column.
// Before, a lane (or a pair) took 8 bytes of 16 (32) vectors and the waves
// summed up in turn: 96^3 x 16 columns, 17 vectors on average, 440 -> 380 us;
// 128^3, one column 89 -> 66 us; 64^2 rows 10.8 -> 4.6 us; 128^3 x 64 columns
// 4.45 -> 4.6 ms (6 TB/s, the rate of a large read; two vectors a step more
// were read before).  Tried: 128 threads (4.69 ms, 375 us), 512 with 4 or 8
// vectors per wave (5.3 and 4.8 ms, 410 us), 4 KB of a vector per workgroup
// (4.75 ms, 419 us).
// A workgroup walks at most kDotsPieces pieces of 64 lanes where the partials'
// buffer holds more workgroups than one per 256 rows (sweep_blocks): with those
// alone a wide batch of few rows ran on few workgroups, and slower than the
// kernels before (at ten vectors, two or three loads in flight per wave).  Two
// cycles of 10 steps, no preconditioner, 64 complex columns, ms before / with
// one workgroup per 256 rows / now: 16^3 4.56 / 5.90 / 3.02; 28^3 6.00 / 7.31 /
// 4.65; 64 real columns of 24^3 3.93 / 3.51 / 2.14.  16 pieces: 2 % faster at 64
// columns, but past kFixPartials workgroups (a launch more) also at 16; 64: as
// before at 48^3 x 16.
constexpr int kDotsPM = 8;
constexpr int kDotsNT = 256;
constexpr int kDotsPieces = 32;
constexpr int kDotsChunk = kDotsPM * (kDotsNT / kWave);

template <typename S, bool ONE>
__global__ __launch_bounds__(kDotsNT) void k_dcgs2_dots(int64_t n, int nrhs, int p, int chunk, const S* __restrict__ V,
                                                        int64_t ldv, const S* __restrict__ q,
                                                        const S* __restrict__ w, S* __restrict__ part) {
  constexpr int E = 16 / (int)sizeof(S), NW = kDotsNT / kWave, PM = kDotsPM;
  const bool hw = w != nullptr;
  const int lane = threadIdx.x % kWave;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int j0 = blockIdx.y * chunk + wid;  // the wave's first vector
  const int j1 = min(p, (int)(blockIdx.y + 1) * chunk);
  const int pu = j0 < j1 ? (j1 - j0 + NW - 1) / NW : 0;
  const bool own = blockIdx.y == 0 && wid == NW - 1;  // takes q.q and q.w too
  if (pu == 0 && !own) return;
  f64x2 aq[PM], aw[PM], ab[2];
#pragma unroll
  for (int u = 0; u < PM; ++u) aq[u] = aw[u] = f64x2{0.0, 0.0};
  ab[0] = ab[1] = f64x2{0.0, 0.0};
  // acc += conj(x) y for the lane's value or values
  auto add = [](f64x2& acc, f64x2 x, f64x2 y) {
    if constexpr (E == 2) {
      acc += x * y;
    } else {
      acc.x += x.x * y.x + x.y * y.y;
      acc.y += x.x * y.y - x.y * y.x;
    }
  };
  const int64_t total = n * nrhs;
  const int64_t stride = (int64_t)gridDim.x * kWave * E;
  const S* Vw = V + (int64_t)j0 * ldv;
  int64_t g = ((int64_t)blockIdx.x * kWave + lane) * E;
  for (; g + E <= total; g += stride) {
    const f64x2 qv = load16(q + g);
    const f64x2 wv = hw ? load16(w + g) : f64x2{0.0, 0.0};
    f64x2 v[PM];
#pragma unroll
    for (int u = 0; u < PM; ++u)
      if (u < pu) v[u] = stream16(Vw + (int64_t)(u * NW) * ldv + g);
#pragma unroll
    for (int u = 0; u < PM; ++u)
      if (u < pu) {
        add(aq[u], v[u], qv);
        add(aw[u], v[u], wv);
      }
    if (own) {
      add(ab[0], qv, qv);
      add(ab[1], qv, wv);
    }
  }
  if constexpr (ONE) {
    if (g < total) {  // the last value of an odd length
      const double qv = q[g], wv = hw ? w[g] : 0.0;
#pragma unroll
      for (int u = 0; u < PM; ++u)
        if (u < pu) {
          const double v = Vw[(int64_t)(u * NW) * ldv + g];
          aq[u].x += v * qv;
          aw[u].x += v * wv;
        }
      ab[0].x += qv * qv;
      ab[1].x += qv * wv;
    }
  }
  // the rows of the step's table: V.q, then V.w, then q.q and q.w
  const int nl = ONE ? 1 : nrhs / E;  // lanes l and l + nl hold the same columns
  double* out = reinterpret_cast<double*>(part + (int64_t)blockIdx.x * ((hw ? 2 * p : p) + (hw ? 2 : 1)) * nrhs);
  auto put = [&](int row, f64x2 a) {
    if (lane >= nl) return;
    if constexpr (ONE) out[row] = a.x;
    else *reinterpret_cast<f64x2*>(out + ((int64_t)row * (nrhs / E) + lane) * 2) = a;
  };
  auto sum = [&](auto& a) {
    constexpr int K = sizeof(a) / sizeof(a[0]);
    double t[ONE ? K : 2 * K];
#pragma unroll
    for (int u = 0; u < K; ++u) {
      if constexpr (ONE) {
        t[u] = a[u].x + a[u].y;
      } else {
        t[2 * u] = a[u].x;
        t[2 * u + 1] = a[u].y;
      }
    }
    lane_class_sums(t, nl);
#pragma unroll
    for (int u = 0; u < K; ++u) a[u] = ONE ? f64x2{t[u], 0.0} : f64x2{t[ONE ? u : 2 * u], t[ONE ? u : 2 * u + 1]};
  };
  sum(aq);
  if (hw) sum(aw);
#pragma unroll
  for (int u = 0; u < PM; ++u)
    if (u < pu) {
      put(j0 + u * NW, aq[u]);
      if (hw) put(p + j0 + u * NW, aw[u]);
    }
  if (own) {
    sum(ab);
    put(hw ? 2 * p : p, ab[0]);
    if (hw) put(2 * p + 1, ab[1]);
  }
}

// w <- w - sum_{j<p} V_j e_j - e_p q: the projection of w on the final
// basis v_0..v_p, written in terms of the raw basis slots 0..p (q = slot p,
// which stays as it is), with per-workgroup partials of |w|^2 in
// part[blk * nrhs + c].  coef = [e_0..e_{p-1} (p x nrhs) | e_p (nrhs)],
// copied to LDS.
// A stream over p + 2 vectors, bound by HBM: a lane takes 16 bytes of every
// vector (two real values or a complex one), 8 vectors' loads in flight, one
// running sum, so that any p runs at the same occupancy.  Before, a lane held
// all p values of an element (two lanes past 32 vectors, 208 VGPRs, 4.5 TB/s):
// 128^3 x 64 columns, 24 vectors on average, 5.9 -> 5.15 ms (5.5 TB/s with its
// write); 96^3 x 16, 17 vectors, 390 -> 370 us; 32^3 x 4 complex columns,
// 24 vectors, 24 -> 15 us.  ONE: a single column (a lane's two values share
// their coefficients).
template <typename S, int NT, bool ONE>
__global__ __launch_bounds__(NT) void k_dcgs2_update(int64_t n, int nrhs, int p, const S* __restrict__ V,
                                                     int64_t ldv, const S* __restrict__ q, S* __restrict__ w,
                                                     const S* __restrict__ coef, double* __restrict__ part) {
  constexpr int E = 16 / (int)sizeof(S);  // values per lane
  constexpr int U = 8;                    // vectors in flight
  extern __shared__ __align__(16) unsigned char du_raw[];
  const int nc = (p + 1) * nrhs;
  double* red = reinterpret_cast<double*>(du_raw);
  S* cs = reinterpret_cast<S*>(red + (NT / kWave) * nrhs + ((NT / kWave) * nrhs) % 2);
  const int tid = threadIdx.x;
  for (int t = tid; t < nc; t += NT) cs[t] = coef[t];
  __syncthreads();
  const int c = ONE ? 0 : (tid * E) % nrhs;  // the lane's first column (the grid stride keeps it)
  // sum += v * e of vector j
  auto add = [&](f64x2& sum, f64x2 v, int j) {
    if constexpr (E == 1) {
      const S e = cs[j * nrhs + c];
      sum.x += v.x * e.re - v.y * e.im;
      sum.y += v.x * e.im + v.y * e.re;
    } else if constexpr (ONE) {
      sum += v * cs[j];
    } else {
      sum += v * *reinterpret_cast<const f64x2*>(cs + j * nrhs + c);
    }
  };
  f64x2 acc = {0.0, 0.0};
  const int64_t total = n * nrhs;
  const int64_t stride = (int64_t)gridDim.x * NT * E;
  int64_t g = ((int64_t)blockIdx.x * NT + tid) * E;
  for (; g + E <= total; g += stride) {
    f64x2 wv = load16(w + g), sum = {0.0, 0.0}, v[U];
    const f64x2 qv = load16(q + g);
    const S* x = V + g;
    int j = 0;
    for (; j + U <= p; j += U, x += U * ldv) {
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = stream16(x + u * ldv);
#pragma unroll
      for (int u = 0; u < U; ++u) add(sum, v[u], j + u);
    }
#pragma unroll
    for (int u = 0; u < U - 1; ++u)
      if (j + u < p) v[u] = stream16(x + u * ldv);
#pragma unroll
    for (int u = 0; u < U - 1; ++u)
      if (j + u < p) add(sum, v[u], j + u);
    f64x2 gq = {0.0, 0.0};
    add(gq, qv, p);
    wv = wv - sum - gq;
    *reinterpret_cast<f64x2_a8*>(w + g) = wv;
    acc += wv * wv;
  }
  if constexpr (ONE && E == 2) {
    if (g < total) {  // the last value of an odd length
      double sum = 0.0;
      for (int j = 0; j < p; ++j) sum += V[j * ldv + g] * cs[j];
      const double un = w[g] - sum - q[g] * cs[p];
      w[g] = un;
      acc.x += un * un;
    }
  }
  const int wid = tid / kWave, lane = tid % kWave;
  if constexpr (ONE || E == 1) {
    const double s2 = lane_class_sum(acc.x + acc.y, nrhs);
    if (lane < nrhs) red[wid * nrhs + lane] = s2;
  } else {
    double a[2] = {acc.x, acc.y};
    lane_class_sums<2>(a, nrhs / 2);
    if (lane < nrhs / 2) {
      red[wid * nrhs + 2 * lane] = a[0];
      red[wid * nrhs + 2 * lane + 1] = a[1];
    }
  }
  __syncthreads();
  for (int t = tid; t < nrhs; t += NT) {
    double s2 = 0.0;
    for (int k = 0; k < NT / kWave; ++k) s2 += red[k * nrhs + t];
    part[(int64_t)blockIdx.x * nrhs + t] = s2;
  }
}

// One launch of modified Gram-Schmidt: w -= vp h with h = vp^H w summed here
// from nprev partials (a row of nrhs values each; none: w stays), then partials
// of vn^H w, or, without vn, of ||w||^2 (doubles), one row of nrhs values per
// workgroup in part.  h is kept in hout (may be null).  A step against i vectors
// is i + 1 of these, each reading w, vp and vn and writing w, where a dot, its
// sum and an update took three launches per vector and read w once more: 48^3,
// one column, 11.2 -> 4.5 us per vector; 128^3, 20 steps,
// 1 column 7.2 -> 4.8 ms, 16 columns 66 -> 54.  Every workgroup adds up all partials
// itself, which costs less than a launch up to kMgsPartials values.
// A workgroup takes at most kMgsPieces pieces of 256 lanes (sweep_blocks, as the
// delayed-CGS2 dots): two cycles of 30 steps, 64 complex columns, ms as three
// launches / with one workgroup per 256 rows / now: 16^3 30.7 / 37.0 / 12.4; 24^3
// 47.1 / 52.4 / 20.7; 64 real columns of 24^3 33.9 / 21.5 / 12.7.  4 pieces are as
// fast, 16 and 32 slower (24^3: 24.0 and 33.4).
// ONE: a single real column.
constexpr int kMgsNT = 256;
constexpr int kMgsPartials = 4096;
constexpr int kMgsPieces = 8;

template <typename S, bool ONE>
__global__ __launch_bounds__(kMgsNT) void k_mgs_step(int64_t n, int nrhs, int nprev, const S* __restrict__ prev,
                                                     S* __restrict__ hout, const S* __restrict__ vp,
                                                     const S* __restrict__ vn, S* __restrict__ w,
                                                     S* __restrict__ part) {
  constexpr int E = 16 / (int)sizeof(S), NW = kMgsNT / kWave;
  __shared__ S red[NW][64];
  __shared__ S hs[64];
  const int tid = threadIdx.x, lane = tid % kWave, wid = tid / kWave;
  if (nprev > 0) {
    S t = S(0.0);
#pragma unroll 4
    for (int b = row_of(tid, nrhs); b < nprev; b += kMgsNT / nrhs) t += prev[b * nrhs + col_of(tid, nrhs)];
    t = lane_class_sum(t, nrhs);
    if (lane < nrhs) red[wid][lane] = t;
    __syncthreads();
    if (tid < nrhs) {
      for (int k = 1; k < NW; ++k) t += red[k][tid];
      hs[tid] = t;
      if (hout && blockIdx.x == 0) hout[tid] = t;
    }
    __syncthreads();
  }
  const int c = ONE ? 0 : (tid * E) % nrhs;  // the lane's first column (the grid stride keeps it)
  f64x2 h = {0.0, 0.0};
  if (nprev > 0) {
    if constexpr (ONE) h = f64x2{hs[0], hs[0]};
    else h = *reinterpret_cast<const f64x2_a8*>(&hs[c]);
  }
  f64x2 acc = {0.0, 0.0};
  const int64_t total = n * nrhs;
  const int64_t stride = (int64_t)gridDim.x * kMgsNT * E;
  int64_t g = ((int64_t)blockIdx.x * kMgsNT + tid) * E;
  for (; g + E <= total; g += stride) {
    f64x2 wv = load16(w + g);
    const f64x2 nv = vn ? load16(vn + g) : f64x2{0.0, 0.0};
    if (nprev > 0) {
      const f64x2 pv = load16(vp + g);
      if constexpr (E == 2) {
        wv -= pv * h;
      } else {
        wv.x -= pv.x * h.x - pv.y * h.y;
        wv.y -= pv.x * h.y + pv.y * h.x;
      }
      *reinterpret_cast<f64x2_a8*>(w + g) = wv;
    }
    const f64x2 x = vn ? nv : wv;
    if constexpr (E == 2) {
      acc += x * wv;
    } else {
      acc.x += x.x * wv.x + x.y * wv.y;
      acc.y += x.x * wv.y - x.y * wv.x;
    }
  }
  if constexpr (ONE) {
    if (g < total) {  // the last value of an odd length
      double wv = w[g];
      if (nprev > 0) w[g] = wv = wv - vp[g] * hs[0];
      acc.x += (vn ? vn[g] : wv) * wv;
    }
  }
  __syncthreads();
  if constexpr (E == 1) {
    const S t = lane_class_sum(S(acc.x, acc.y), nrhs);
    if (lane < nrhs) red[wid][lane] = t;
  } else if constexpr (ONE) {
    const double t = lane_class_sum(acc.x + acc.y, 1);
    if (lane == 0) red[wid][0] = t;
  } else {
    double a[2] = {acc.x, acc.y};
    lane_class_sums<2>(a, nrhs / 2);
    if (lane < nrhs / 2) {
      red[wid][2 * lane] = a[0];
      red[wid][2 * lane + 1] = a[1];
    }
  }
  __syncthreads();
  if (tid < nrhs) {
    S t = red[0][tid];
    for (int k = 1; k < NW; ++k) t += red[k][tid];
    if (vn) part[(int64_t)blockIdx.x * nrhs + tid] = t;
    else reinterpret_cast<double*>(part)[(int64_t)blockIdx.x * nrhs + tid] = sreal(t);
  }
}

// Per column (one workgroup, blockIdx.x = column), after the
// dots of step p.  The basis slots hold raw vectors: slot j < p is step j's
// first projection as k_dcgs2_update left it, and the final (orthonormal)
// basis is v_j = sum_{i<=j} slot_i R[i, j], R upper triangular (row-major,
// (m+1) x (m+1) per column); slot p = q still waits for its scale sg
// (vscale).  From the raw dots d = [slot_j^H q (p) | slot_j^H w (p) | q.q |
// q.w] (final pass: [slot_j^H q | q.q]):
//   s_j = v_j^H (sg q) = sg sum_{i<=j} conj(R[i, j]) d_i,  a_j = v_j^H w alike;
// then q's norm nu = sqrt(sg^2 q.q - |s|^2), the correction of the tentative
// Hessenberg column p-1 (H[0..p-1, p-1] += H[p, p-1] s; H[p, p-1] *= nu) and
// its Givens update as k_givens (convergence test, cycle end); then (not
// final) H[0..p-1, p] = a, H[p, p] = c_p = (sg q.w - s^H a) / nu.  The final
// v_p = (sg q - sum_j v_j s_j) / nu is R's column p: R[i, p] = -(R s)_i / nu,
// R[p, p] = sg / nu; and w - sum_{j<p} v_j a_j - c_p v_p = w - sum_{i<=p}
// slot_i e_i with e_i = (R (a - gm s))_i for i < p, e_p = sg gm, gm = c_p / nu:
// coef = [e_0..e_p] (rows of nrhs) for k_dcgs2_update, zero for columns that
// are not active.  p = 0: q is the exact v0 (nu = 1, no column to finalize).
// With nblk > 0, d holds nblk partial tables of the dots (part of
// k_dcgs2_dots), summed here in a fixed order.  flag (final pass, may be
// null): the column's state for the host (state_bits).
// Lanes take the basis indices, waves share the sums; only the Givens
// recurrence runs on one lane, from LDS (it was one lane reading memory all
// through: 10 -> 6.6 us at 15 vectors, 21 -> 9 at 24, 29 -> 14 at 24 complex
// ones, and the launch that summed the partials is gone).
// Dynamic LDS: fix_lds(p, NT) values of S.
__host__ __device__ inline int fix_lds(int p, int nt) { return (2 * p + 2) * (1 + nt / kWave) + 5 * p + 1; }

template <typename S, int NT>
__global__ __launch_bounds__(NT) void k_dcgs2_fix(int nrhs, int m, int p, int maxits, int final_pass, int nblk,
                                                  const S* __restrict__ d, S* __restrict__ H, S* __restrict__ cs,
                                                  S* __restrict__ sn, S* __restrict__ rs, KState* __restrict__ st,
                                                  S* __restrict__ coef, const double* __restrict__ vscale,
                                                  S* __restrict__ R, int* __restrict__ flag) {
  constexpr int NW = NT / kWave;
  extern __shared__ unsigned char fx_raw[];
  S* dt = reinterpret_cast<S*>(fx_raw);  // the dot table, later [s_j | a_j]
  S* red = dt + 2 * p + 2;               // NW rows of sums
  S* cl = red + NW * (2 * p + 2);        // earlier rotations
  S* sl = cl + p;
  S* h = sl + p;    // the tentative Hessenberg column, p + 1 values
  S* sv = h + p + 1;
  S* av = sv + p;
  __shared__ int go_sh;
  __shared__ double in_sh;
  __shared__ S gm_sh;
  const int c = blockIdx.x;
  const int tid = threadIdx.x, lane = tid % kWave, wid = tid / kWave;
  const int64_t ldr = m + 1;
  S* Rc = R + (int64_t)c * ldr * ldr;
  S* Hc = H + (int64_t)c * (m + 1) * m;
  S* csc = cs + (int64_t)c * m;
  S* snc = sn + (int64_t)c * m;
  const int col = p - 1;
  const double sg = vscale ? vscale[c] : 1.0;
  KState s = st[c];
  bool go = s.active != 0;  // the same in every thread
  if (go) {
    const int no = final_pass ? p + 1 : 2 * p + 2;
    if (nblk > 0) {
      for (int o = lane; o < no; o += kWave) {
        S acc = S(0.0);
#pragma unroll 8
        for (int b = wid; b < nblk; b += NW) acc += d[((int64_t)b * no + o) * nrhs + c];
        red[wid * no + o] = acc;
      }
      __syncthreads();
      for (int o = tid; o < no; o += NT) {
        S acc = red[o];
        for (int k = 1; k < NW; ++k) acc += red[k * no + o];
        dt[o] = acc;
      }
    } else {
      for (int o = tid; o < no; o += NT) dt[o] = d[(int64_t)o * nrhs + c];
    }
    for (int j = tid; j + 1 < p; j += NT) {
      cl[j] = csc[j];
      sl[j] = snc[j];
    }
    if (p > 0)
      for (int j = tid; j <= p; j += NT) h[j] = Hc[j + col * (m + 1)];
    __syncthreads();
    // s and a on the final basis (lanes over j, rows of R read along j, the
    // rows dealt to the waves)
    for (int j = lane; j < p; j += kWave) {
      S ts = S(0.0), ta = S(0.0);
#pragma unroll 4
      for (int i = wid; i <= j; i += NW) {
        const S r = sconj(Rc[i * ldr + j]);
        ts += r * dt[i];
        if (!final_pass) ta += r * dt[p + i];
      }
      red[wid * 2 * p + j] = ts;
      red[wid * 2 * p + p + j] = ta;
    }
    __syncthreads();
    for (int j = tid; j < p; j += NT) {
      S ts = red[j], ta = red[p + j];
      for (int k = 1; k < NW; ++k) {
        ts += red[k * 2 * p + j];
        ta += red[k * 2 * p + p + j];
      }
      sv[j] = S(sg) * ts;
      av[j] = ta;
    }
    __syncthreads();
  }
  // d rows: slot_j^H q (j < p), then slot_j^H w (j < p), then q.q, q.w
  // (final: slot_j^H q, q.q)
  double qq = 0.0, nu = 1.0, ss = 0.0;
  S qw = S(0.0), sa = S(0.0);
  if (go) {
    qq = sg * sg * (double)sreal(final_pass ? dt[p] : dt[2 * p]);
    if (!final_pass) qw = S(sg) * dt[2 * p + 1];
    for (int j = lane; j < p; j += kWave) {
      ss += (double)sabs2(sv[j]);
      if (!final_pass) sa += sconj(sv[j]) * av[j];
    }
    ss = lane_class_sum(ss, 1);
    sa = lane_class_sum(sa, 1);
    nu = p > 0 ? sqrt(fmax(qq - ss, 0.0)) : 1.0;
    if (p > 0) {
      const S hq = h[p];
      __syncthreads();
      for (int j = tid; j < p; j += NT) h[j] += hq * sv[j];
      if (tid == 0) h[p] = hq * S(nu);
      __syncthreads();
    }
  }
  if (tid == 0) {
    // the column's scalar part; returns whether w gets coefficients
    auto scalar_part = [&]() -> bool {
      if (!go) return false;
      const double eps = 2.220446049250313e-16;
      auto retire = [&](int status) {
        s.status = status;
        s.active = 0;
        s.scale = 0.0;
        st[c] = s;
      };
      if (!isfinite(qq) || !isfinite(sabs_d(qw))) {
        retire(5);
        return false;
      }
      // the tentative v_p lies in the span of v_0..v_{p-1} to working
      // precision when q.q - |s|^2 cancels (|s| = 1 - 5e-11 and closer): nu
      // and the final v_p = (q - V s) / nu are then rounding noise, so the
      // column's cycle ends with Hessenberg column p - 1 (whose subdiagonal
      // nu * h is negligible there, a lucky breakdown) and restarts from its
      // true residual instead of continuing on a basis vector that is not
      // orthogonal
      if (p > 0) {
        if (!isfinite(ss)) {
          retire(5);
          return false;
        }
        const bool dependent = !(qq - ss > kDcgs2DependentTol * qq);
        // Givens update of column col, as k_givens (fgmres.hpp:428-461)
        S* rsc = rs + (int64_t)c * (m + 1);
        S* hc = Hc + (int64_t)col * (m + 1);
        s.iters += 1;
        s.icur = p;
        const S hii = rotate_column(p, h, cl, sl, hc);
        const S hii1 = h[p];
        hc[p] = hii1;
        const double g = sqrt((double)sabs2(hii) + (double)sabs2(hii1));
        if (!isfinite(g)) {
          retire(5);
          return false;
        }
        if (fabs(g) < eps) {  // breakdown: the reference leaves x untouched (fgmres.hpp:440-443)
          retire(2);
          return false;
        }
        const S cn = hii / S(g), sn1 = hii1 / S(g);
        const S r0 = rsc[p - 1];
        csc[p - 1] = cn;
        snc[p - 1] = sn1;
        rsc[p] = -sn1 * r0;
        rsc[p - 1] = sconj(cn) * r0;
        hc[p - 1] = sconj(cn) * hii + sn1 * hii1;
        s.normr = sabs_d(-sn1 * r0);
        if (s.normr <= s.tolr) {
          s.status = 1;
          s.active = 0;
        } else if (p >= m || s.iters >= maxits || dependent) {
          s.active = 0;  // cycle ends for this column
        }
        st[c] = s;
        if (!s.active) return false;
      }
      if (final_pass) return false;
      const double in = nu > 0.0 ? 1.0 / nu : 0.0;
      // coefficient of w on the final v_p: (q - V s)^H w / nu = (q.w - s^H a) / nu
      const S cp = (qw - sa) * S(in);
      Hc[p + (int64_t)p * (m + 1)] = cp;
      in_sh = in;
      gm_sh = cp * S(in);
      return true;
    };
    go_sh = scalar_part() ? 1 : 0;
    if (flag) flag[c] = state_bits(s, maxits);
  }
  if (final_pass) return;
  __syncthreads();
  if (!go_sh) {
    for (int j = tid; j <= p; j += NT) coef[(int64_t)j * nrhs + c] = S(0.0);
    return;
  }
  const double in = in_sh;
  const S gm = gm_sh;
  for (int j = tid; j < p; j += NT) Hc[j + (int64_t)p * (m + 1)] = av[j];
  // R's column p and the update's coefficients (16 lanes to a row of R)
  for (int i0 = 0; i0 < p; i0 += NT / 16) {
    const int i = i0 + tid / 16;
    S rsv = S(0.0), rg = S(0.0);
    if (i < p) {
#pragma unroll 4
      for (int j = i + tid % 16; j < p; j += 16) {
        const S r = Rc[i * ldr + j];
        rsv += r * sv[j];
        rg += r * (av[j] - gm * sv[j]);
      }
    }
    rsv = lane_step<1>(lane_step<2>(lane_step<4>(lane_step<8>(rsv))));
    rg = lane_step<1>(lane_step<2>(lane_step<4>(lane_step<8>(rg))));
    if (i < p && tid % 16 == 0) {
      Rc[i * ldr + p] = -rsv * S(in);
      coef[(int64_t)i * nrhs + c] = rg;
    }
  }
  if (tid == 0) {
    Rc[p * ldr + p] = S(sg * in);
    coef[(int64_t)p * nrhs + c] = S(sg) * gm;
  }
}

// After k_dcgs2_update of step p, per column (blockIdx.x): ||w|| from the
// nblk partials of ||w||^2, the tentative H[p+1, p] = ||w|| and the scale that
// normalizes w (zero for columns that are not active); the column's state for
// the host in flag.
template <typename S>
__global__ __launch_bounds__(kTailNT) void k_dcgs2_norm(int nblk, int nrhs, int m, int p, int maxits,
                                                        const double* __restrict__ part, S* __restrict__ H,
                                                        KState* __restrict__ st, double* __restrict__ vscale,
                                                        int* __restrict__ flag) {
  __shared__ double red[kTailNT / kWave];
  const int c = blockIdx.x;
  const double t2 = column_sum(nblk, nrhs, c, part, red);
  if (threadIdx.x != 0) return;
  KState s = st[c];
  if (!s.active) {
    s.scale = 0.0;
  } else if (!isfinite(t2)) {
    s.status = 5;
    s.active = 0;
    s.scale = 0.0;
  } else {
    const double t = sqrt(t2);
    H[(int64_t)c * (m + 1) * m + (p + 1) + p * (m + 1)] = S(t);
    s.scale = t > 0.0 ? 1.0 / t : 0.0;
  }
  st[c] = s;
  vscale[c] = s.scale;  // w stays as it is; its readers apply the scale
  if (flag) flag[c] = state_bits(s, maxits);
}

// v[r, c] *= s[c]   (s from KState.scale)
template <typename S>
__global__ void k_scale_cols(int64_t n, int nrhs, const KState* __restrict__ st, S* __restrict__ v) {
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n * nrhs) return;
  v[g] *= S(st[col_of(g, nrhs)].scale);
}

// FGMRES start (fgmres.hpp:318-359): normb, normr from squared norms.
__global__ void k_fgmres_init(int nrhs, const double* __restrict__ nb2, const double* __restrict__ nr2, double tol,
                              int absolute, int maxits, KState* __restrict__ st,
                              double* __restrict__ x_zero_flag, int* __restrict__ flag) {
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nrhs) return;
  const double eps = 2.220446049250313e-16;
  KState s;
  s.normb = sqrt(nb2[c]);
  s.normr = sqrt(nr2[c]);
  s.tolr = absolute ? tol : tol * s.normb;
  s.scale = 0.0;
  s.iters = 0;
  s.icur = 0;
  s.active = 0;
  s.status = 0;
  x_zero_flag[c] = 0.0;
  if (!isfinite(s.normb) || !isfinite(s.normr)) {  // NaN or Inf in b or x0: x stays as given
    s.status = 5;
  } else if (s.normb < eps) {  // zero right-hand side: x = 0 (fgmres.hpp:321-328)
    s.status = 4;
    x_zero_flag[c] = 1.0;
  } else if (s.normr < eps) {  // initial guess already exact (fgmres.hpp:341-348)
    s.status = 4;
  } else {
    s.active = 1;
  }
  st[c] = s;
  if (flag) flag[c] = state_bits(s, maxits);
}

// x[r, c] = 0 where flag[c] != 0
template <typename S>
__global__ void k_zero_cols(int64_t n, int nrhs, const double* __restrict__ flag, S* __restrict__ x) {
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n * nrhs) return;
  if (flag[col_of(g, nrhs)] != 0.0) x[g] = S(0.0);
}

// Start of a restart cycle (fgmres.hpp:382-386): rs[0] = normr, v0 /= normr.
template <typename S>
__global__ void k_cycle_start(int nrhs, int m, KState* __restrict__ st, S* __restrict__ rs,
                              double* __restrict__ vscale = nullptr) {
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nrhs) return;
  if (vscale) vscale[c] = 1.0;  // v0 is normalized in place
  KState s = st[c];
  if (s.status == 0) {
    s.active = 1;
    s.icur = 0;
    rs[(int64_t)c * (m + 1)] = S(s.normr);
    s.scale = 1.0 / s.normr;
  } else {
    s.active = 0;
    s.scale = 0.0;
  }
  st[c] = s;
}

// Hessenberg column + Givens update for inner step i (1-based), fgmres.hpp:424-461
// (complex: c = h_ii / gamma and s = h_i+1,i / gamma, rotations applied with
// conj(c) as the reference does).  hcol[j*nrhs + c], j <= i-1 : orthogonalization
// coefficients (plus those of hadd, a second projection pass, when not null);
// ||w||^2 from nblk partials.  One workgroup per column: the column and the
// earlier rotations go through LDS, one lane runs the recurrence; the
// column's state for the host in flag (may be null).
// Dynamic LDS: 3 i values of S.
template <typename S>
__global__ __launch_bounds__(kTailNT) void k_givens(int nblk, int nrhs, int m, int i, int maxits,
                                                    const S* __restrict__ hcol, const S* __restrict__ hadd,
                                                    const double* __restrict__ part, S* __restrict__ H,
                                                    S* __restrict__ cs, S* __restrict__ sn, S* __restrict__ rs,
                                                    KState* __restrict__ st, int* __restrict__ flag) {
  extern __shared__ unsigned char gv_raw[];
  S* h = reinterpret_cast<S*>(gv_raw);
  S* cl = h + i;
  S* sl = cl + i;
  __shared__ double red[kTailNT / kWave];
  const int c = blockIdx.x;
  S* csc = cs + (int64_t)c * m;
  S* snc = sn + (int64_t)c * m;
  for (int j = threadIdx.x; j < i; j += kTailNT) {
    h[j] = hadd ? hcol[j * nrhs + c] + hadd[j * nrhs + c] : hcol[j * nrhs + c];
    if (j + 1 < i) {
      cl[j] = csc[j];
      sl[j] = snc[j];
    }
  }
  const double t = sqrt(column_sum(nblk, nrhs, c, part, red));  // its barrier also covers h, cl, sl
  if (threadIdx.x != 0) return;
  KState s = st[c];
  auto settle = [&](int status, int active, double scale) {
    s.status = status;
    s.active = active;
    s.scale = scale;
    st[c] = s;
    if (flag) flag[c] = state_bits(s, maxits);
  };
  if (!s.active) {
    settle(s.status, 0, 0.0);
    return;
  }
  const double eps = 2.220446049250313e-16;
  S* rsc = rs + (int64_t)c * (m + 1);
  S* hc = H + (int64_t)c * (m + 1) * m + (int64_t)(i - 1) * (m + 1);
  s.iters += 1;
  s.icur = i;
  const S hii = rotate_column(i, h, cl, sl, hc);
  const S hii1 = S(t);
  hc[i] = hii1;
  const double gam = sqrt((double)sabs2(hii) + (double)sabs2(hii1));
  if (!isfinite(gam) || !isfinite(t)) {  // NaN or Inf from the apply or the matrix product
    settle(5, 0, 0.0);
    return;
  }
  if (fabs(gam) < eps) {  // breakdown: the reference leaves x untouched (fgmres.hpp:440-443)
    settle(2, 0, 0.0);
    return;
  }
  const S cn = hii / S(gam), sn1 = hii1 / S(gam);
  const S r0 = rsc[i - 1];
  csc[i - 1] = cn;
  snc[i - 1] = sn1;
  rsc[i] = -sn1 * r0;
  rsc[i - 1] = sconj(cn) * r0;
  hc[i - 1] = sconj(cn) * hii + sn1 * hii1;
  s.normr = sabs_d(-sn1 * r0);
  const double scale = (t > 0.0) ? 1.0 / t : 0.0;
  if (s.normr <= s.tolr) settle(1, 0, scale);
  else settle(s.status, i >= m || s.iters >= maxits ? 0 : s.active, scale);  // the cycle may end for this column
}

// Back substitution on the triangularized H (fgmres.hpp:471-480); coef[j*nrhs+c].
// One wave per column; lane j of round r holds y_{64 r + j}, and each solved
// value is taken out of the rest by the column of H that it multiplies (one
// lane reading H along its rows took 62 us for 30 vectors and 268 for 50
// complex ones, now 9 and 30).  m < 128.
template <typename S>
__global__ __launch_bounds__(kWave) void k_backsolve(int nrhs, int m, const S* __restrict__ H,
                                                     const S* __restrict__ rs, const KState* __restrict__ st,
                                                     S* __restrict__ coef, int* __restrict__ upd) {
  const int c = blockIdx.x;
  const int lane = threadIdx.x;
  const KState s = st[c];
  const bool use = !(s.status == 2 || s.status == 4 || s.status == 5 || s.icur == 0);
  const int i = use ? s.icur : 0;
  if (lane == 0) upd[c] = use ? 1 : 0;
  const S* Hc = H + (int64_t)c * (m + 1) * m;
  const S* rsc = rs + (int64_t)c * (m + 1);
  S y[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) y[r] = r * kWave + lane < i ? rsc[r * kWave + lane] : S(0.0);
#pragma unroll
  for (int r = 1; r >= 0; --r) {
#pragma unroll 4
    for (int k = min(i, (r + 1) * kWave) - 1; k >= r * kWave; --k) {
      const S* hk = Hc + (int64_t)k * (m + 1);
      const S yk = lane_value(y[r], k % kWave) / hk[k];
      const int row = r * kWave + lane;
      if (row == k) y[r] = yk;
      else if (row < k) y[r] -= hk[row] * yk;
      if (r == 1) y[0] -= hk[lane] * yk;
    }
  }
#pragma unroll
  for (int r = 0; r < 2; ++r)
    if (r * kWave + lane < m) coef[(r * kWave + lane) * nrhs + c] = y[r];
}

// x[r, c] += sum_j coef[j, c] * Z_j[r, c] for columns with upd[c], summed
// in S, x stored as VX (dynamic shared memory: p*nrhs values of S)
template <typename VZ, typename S, typename VX = S>
__global__ void k_update_x(int64_t n, int nrhs, int p, const VZ* __restrict__ Z, int64_t ldz,
                           const S* __restrict__ coef, const int* __restrict__ upd, VX* __restrict__ x) {
  extern __shared__ unsigned char ux_smem[];
  S* cs = reinterpret_cast<S*>(ux_smem);
  for (int t = threadIdx.x; t < p * nrhs; t += blockDim.x) cs[t] = coef[t];
  __syncthreads();
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n * nrhs) return;
  const int c = col_of(g, nrhs);
  if (!upd[c]) return;
  S acc = (S)x[g];
  for (int j = 0; j < p; ++j) acc += cs[j * nrhs + c] * (S)Z[j * ldz + g];
  x[g] = (VX)acc;
}

// x[t] = 0 for t < m (a kernel rather than a memset: launches may be
// captured into graphs)
template <typename V>
__global__ void k_fill_zero(int64_t m, V* __restrict__ x) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < m) x[t] = V(0.0);
}

// copy v (double) into z (VZ) : identity preconditioner
template <typename S, typename VZ>
__global__ void k_copy_conv(int64_t m, const S* __restrict__ in, VZ* __restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < m) out[t] = (VZ)in[t];
}

// z[r, c] = v[r, c] * cscale[c] : identity preconditioner on a Krylov vector
// whose normalization is pending
template <typename S, typename VZ>
__global__ void k_copy_scale_cols(int64_t n, int nrhs, const double* __restrict__ cscale, const S* __restrict__ in,
                                  VZ* __restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n * nrhs) out[t] = (VZ)(in[t] * S(cscale[col_of(t, nrhs)]));
}

// ---------------------------------------------------------------------------
// single-vector operations of SequentialVectorClass on the device
// (Axpy / Scale / Fill / Dot, ParGeMSLR/SRC/vectors/sequential_vector.cpp:
// 706-732, 1037-1172; vectorops.cpp:93-146, 633-680)
// ---------------------------------------------------------------------------
template <typename S>
__global__ void k_vec_axpy(int64_t n, S alpha, const S* __restrict__ x, S* __restrict__ y) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] += alpha * x[i];
}

template <typename S>
__global__ void k_vec_scale(int64_t n, S alpha, S* __restrict__ x) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    x[i] *= alpha;
}

template <typename S>
__global__ void k_vec_fill(int64_t n, S v, S* __restrict__ x) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    x[i] = v;
}

// Per-workgroup partials of sum_i conj(x_i) y_i: part[blk * 2] (real part),
// part[blk * 2 + 1] (imaginary part, 0 for real values); summed in a fixed
// order by k_dot_final_wave with p = 2.  256 threads.
template <typename S>
__global__ __launch_bounds__(256) void k_vec_dot(int64_t n, const S* __restrict__ x, const S* __restrict__ y,
                                                 double* __restrict__ part) {
  __shared__ double red[2][4];
  double re = 0.0, im = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const S t = sconj(x[i]) * y[i];
    if constexpr (scalar_traits<S>::is_complex) {
      re += t.re;
      im += t.im;
    } else {
      re += t;
    }
  }
#pragma unroll
  for (int m = kWave / 2; m > 0; m >>= 1) {
    re += __shfl_xor(re, m);
    im += __shfl_xor(im, m);
  }
  const int wv = threadIdx.x / kWave;
  if (threadIdx.x % kWave == 0) {
    red[0][wv] = re;
    red[1][wv] = im;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    const double* r = red[threadIdx.x];
    part[(int64_t)blockIdx.x * 2 + threadIdx.x] = (r[0] + r[1]) + (r[2] + r[3]);
  }
}

}  // namespace dev
}  // namespace pgs
