// Block-diagonal ILU solve x = U^{-1} L^{-1} rhs for one GeMSLR level
// (IluClass::SolveHost, ParGeMSLR/SRC/preconditioners/ilu.cpp:3752-3783):
// L unit lower (strict part stored), U strictly upper, Dinv = 1/pivots.
//
// Layout (built on the host by trsv_pack): per diagonal block a sequence of
// steps (level sets, L sweep then U sweep); step s is
//   desc[s] = {row_off, ent_off, nrows, width}   (block-relative offsets)
//   ent[ent_off + t * width + j] = (column, value) of slot j of row t
//   ri[row_off + t]              = (row, 1/pivot)   (1/pivot used on U steps)
// Padded slots hold (0, 0).  x is first loaded with rhs and both sweeps run in
// place, so padded slots only ever read finite values.  The pipelined kernels
// let a lane read slot q + e * LPR of its row unclamped: past the row's width
// that is a padded or a neighbouring entry (a valid column) or, at the end of
// the block, a zero from an out-of-range buffer load, and its weight is
// replaced by zero.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "../host/ring_pack.hpp"

namespace pgs {
namespace dev {

// Complex value of the device path: (re, im), arithmetic as in std::complex.
template <typename R>
struct alignas(2 * sizeof(R)) cplx {
  R re, im;
  cplx() = default;
  __host__ __device__ constexpr cplx(R r) : re(r), im(0) {}
  __host__ __device__ constexpr cplx(R r, R i) : re(r), im(i) {}
  template <typename Q>
  __host__ __device__ explicit constexpr cplx(const cplx<Q>& o) : re((R)o.re), im((R)o.im) {}
  __host__ __device__ cplx& operator+=(const cplx& o) { re += o.re; im += o.im; return *this; }
  __host__ __device__ cplx& operator-=(const cplx& o) { re -= o.re; im -= o.im; return *this; }
  __host__ __device__ cplx& operator*=(const cplx& o) {
    const R r = re * o.re - im * o.im;
    im = re * o.im + im * o.re;
    re = r;
    return *this;
  }
  __host__ __device__ cplx& operator/=(const cplx& o) {
    const R d = o.re * o.re + o.im * o.im;
    const R r = (re * o.re + im * o.im) / d;
    im = (im * o.re - re * o.im) / d;
    re = r;
    return *this;
  }
};
template <typename R> __host__ __device__ inline cplx<R> operator+(cplx<R> a, const cplx<R>& b) { return a += b; }
template <typename R> __host__ __device__ inline cplx<R> operator-(cplx<R> a, const cplx<R>& b) { return a -= b; }
template <typename R> __host__ __device__ inline cplx<R> operator*(cplx<R> a, const cplx<R>& b) { return a *= b; }
template <typename R> __host__ __device__ inline cplx<R> operator/(cplx<R> a, const cplx<R>& b) { return a /= b; }
template <typename R> __host__ __device__ inline cplx<R> operator-(const cplx<R>& a) { return cplx<R>(-a.re, -a.im); }
template <typename R> __host__ __device__ inline bool operator==(const cplx<R>& a, const cplx<R>& b) {
  return a.re == b.re && a.im == b.im;
}

// Scalar traits: real type, conjugate, squared magnitude.
template <typename V> struct scalar_traits { using real = V; static constexpr bool is_complex = false; };
template <typename R> struct scalar_traits<cplx<R>> { using real = R; static constexpr bool is_complex = true; };
template <typename V> __host__ __device__ inline V sconj(const V& v) { return v; }
template <typename R> __host__ __device__ inline cplx<R> sconj(const cplx<R>& v) { return cplx<R>(v.re, -v.im); }
template <typename V> __host__ __device__ inline V sabs2(const V& v) { return v * v; }
template <typename R> __host__ __device__ inline R sabs2(const cplx<R>& v) { return v.re * v.re + v.im * v.im; }
template <typename V> __host__ __device__ inline double sabs_d(const V& v) { return fabs((double)v); }
template <typename R> __host__ __device__ inline double sabs_d(const cplx<R>& v) {
  return sqrt((double)v.re * v.re + (double)v.im * v.im);
}
template <typename V> __host__ __device__ inline V sreal(const V& v) { return v; }
template <typename R> __host__ __device__ inline R sreal(const cplx<R>& v) { return v.re; }

template <typename V>
struct alignas(8) TPair;
template <>
struct alignas(8) TPair<float> {
  int col;
  float val;
};
template <>
struct alignas(16) TPair<double> {  // value first: a 12-byte load takes (value, column)
  double val;
  int col;
  int pad;
};
template <>
struct alignas(16) TPair<cplx<float>> {
  cplx<float> val;
  int col;
  int pad;
};
template <>
struct alignas(16) TPair<cplx<double>> {
  cplx<double> val;
  int col;
  int pad[3];
};

constexpr int kBufferRsrcWord3 = 0x00020000;  // gfx9 raw buffer: 32-bit dwords, no swizzle

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, kBufferRsrcWord3);
}

// Buffer loads: reads outside [0, bytes) of the resource return zeros.
__device__ __forceinline__ int4 bload_i4(__amdgpu_buffer_rsrc_t r, int off) {
  auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
  return make_int4((int)v[0], (int)v[1], (int)v[2], (int)v[3]);
}
__device__ __forceinline__ TPair<float> bload_pair(__amdgpu_buffer_rsrc_t r, int off, float) {
  auto v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
  TPair<float> p;
  p.col = (int)v[0];
  p.val = __uint_as_float(v[1]);
  return p;
}
__device__ __forceinline__ TPair<double> bload_pair(__amdgpu_buffer_rsrc_t r, int off, double) {
  auto v = __builtin_amdgcn_raw_buffer_load_b96(r, off, 0, 0);
  TPair<double> p;
  p.val = __hiloint2double((int)v[1], (int)v[0]);
  p.col = (int)v[2];
  p.pad = 0;
  return p;
}
// Sum over the 4 lanes of a quad with DPP quad permutations (xor 1, xor 2).
__device__ __forceinline__ float quad_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
  return v;
}
__device__ __forceinline__ double quad_perm_f64(double v, int ctrl_sel) {
  int lo = __double2loint(v), hi = __double2hiint(v);
  if (ctrl_sel == 1) {
    lo = __builtin_amdgcn_mov_dpp(lo, 0xB1, 0xF, 0xF, true);
    hi = __builtin_amdgcn_mov_dpp(hi, 0xB1, 0xF, 0xF, true);
  } else {
    lo = __builtin_amdgcn_mov_dpp(lo, 0x4E, 0xF, 0xF, true);
    hi = __builtin_amdgcn_mov_dpp(hi, 0x4E, 0xF, 0xF, true);
  }
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double quad_sum(double v) {
  v += quad_perm_f64(v, 1);
  v += quad_perm_f64(v, 2);
  return v;
}
// Sum over lane pairs (xor 1).
__device__ __forceinline__ float pair_sum(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
}
__device__ __forceinline__ double pair_sum(double v) { return v + quad_perm_f64(v, 1); }
// The value of the lane q ^ 1 / q ^ 2 of the same quad.
__device__ __forceinline__ float dpp_xor1(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
}
__device__ __forceinline__ float dpp_xor2(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
}
__device__ __forceinline__ double dpp_xor1(double v) { return quad_perm_f64(v, 1); }
__device__ __forceinline__ double dpp_xor2(double v) { return quad_perm_f64(v, 2); }
template <typename R>
__device__ __forceinline__ cplx<R> dpp_xor1(cplx<R> v) { return cplx<R>(dpp_xor1(v.re), dpp_xor1(v.im)); }
template <typename R>
__device__ __forceinline__ cplx<R> dpp_xor2(cplx<R> v) { return cplx<R>(dpp_xor2(v.re), dpp_xor2(v.im)); }
template <typename R>
__device__ __forceinline__ cplx<R> quad_sum(cplx<R> v) { return cplx<R>(quad_sum(v.re), quad_sum(v.im)); }

// Direct kernel: any width, nrhs columns (row-interleaved); one thread per
// (row of the step, column), plain loads.  Used for levels whose rows are too
// wide for the pipelined kernel.
template <typename V, int NT>
__global__ __launch_bounds__(NT) void k_trsv_direct(const int* __restrict__ blk_row0, const int* __restrict__ blk_step,
                                                    const int* __restrict__ blk_stepU,
                                                    const int64_t* __restrict__ blk_ent0,
                                                    const int64_t* __restrict__ blk_ri0, const int4* __restrict__ desc,
                                                    const TPair<V>* __restrict__ ent, const TPair<V>* __restrict__ ri,
                                                    const V* __restrict__ rhs, V* __restrict__ x, int nrhs) {
  const int b = blockIdx.x;
  const int r0 = blk_row0[b], nb = blk_row0[b + 1] - r0;
  const int tid = threadIdx.x;
  const V* rb = rhs + (int64_t)r0 * nrhs;
  V* xb = x + (int64_t)r0 * nrhs;
  const TPair<V>* eb = ent + blk_ent0[b];
  const TPair<V>* rib = ri + blk_ri0[b];
  for (int i = tid; i < nb * nrhs; i += NT) xb[i] = rb[i];
  __syncthreads();
  const int s0 = blk_step[b], sU = blk_stepU[b], s1 = blk_step[b + 1];
  for (int s = s0; s < s1; ++s) {
    const int4 d = desc[s];
    const bool upper = (s >= sU);
    const int items = d.z * nrhs;
    for (int it = tid; it < items; it += NT) {
      const int t = it / nrhs;
      const int c = it - t * nrhs;
      const TPair<V> rr = rib[d.x + t];
      V acc = xb[(int64_t)rr.col * nrhs + c];
      for (int j = 0; j < d.w; ++j) {
        const TPair<V> p = eb[d.y + t * d.w + j];
        acc -= p.val * xb[(int64_t)p.col * nrhs + c];
      }
      if (upper) acc *= rr.val;
      xb[(int64_t)rr.col * nrhs + c] = acc;
    }
    __syncthreads();
  }
}

// Pipelined kernel: one workgroup per (diagonal block, RHS column); grid
// index = column * nblocks + block, so all columns of a block are dispatched
// to the same XCD (round-robin over 8 XCDs when nblocks % 8 == 0) and share
// its L2 copy of the factors.  A step is solved by LPR lanes per row with EPL
// slots per lane (steps are at most NT/LPR rows and LPR*EPL slots wide).  The
// slots, row pairs and descriptors of the next D steps are in flight while
// the current step runs; every load is unconditional (buffer loads, indices
// clamped into the step) so the hardware wait counters advance in order and
// only the data of the current step is waited for.
// XLDS: the block's column of x lives in LDS (else in global memory).
template <typename V, bool XLDS, int NT, int LPR, int EPL, int D>
__global__ __launch_bounds__(NT) void k_trsv_pipe(int nblocks, const int* __restrict__ blk_row0,
                                                  const int* __restrict__ blk_step, const int* __restrict__ blk_stepU,
                                                  const int64_t* __restrict__ blk_ent0,
                                                  const int64_t* __restrict__ blk_ri0, const int4* __restrict__ desc,
                                                  const TPair<V>* __restrict__ ent, const TPair<V>* __restrict__ ri,
                                                  const V* __restrict__ rhs, V* __restrict__ x, int nrhs) {
  extern __shared__ unsigned char smem_raw[];
  const int b = blockIdx.x % nblocks;
  const int c = blockIdx.x / nblocks;
  const int r0 = blk_row0[b], nb = blk_row0[b + 1] - r0;
  const int sbeg = blk_step[b], send = blk_step[b + 1], sU = blk_stepU[b];
  const int64_t e0 = blk_ent0[b], e1 = blk_ent0[b + 1];
  const int64_t q0 = blk_ri0[b], q1 = blk_ri0[b + 1];
  const __amdgpu_buffer_rsrc_t rs_ent = make_rsrc(ent + e0, (e1 - e0) * (int64_t)sizeof(TPair<V>));
  const __amdgpu_buffer_rsrc_t rs_ri = make_rsrc(ri + q0, (q1 - q0) * (int64_t)sizeof(TPair<V>));
  const __amdgpu_buffer_rsrc_t rs_desc = make_rsrc(desc + sbeg, (int64_t)(send - sbeg) * 16);
  const int tid = threadIdx.x;
  const int q = tid % LPR;
  const int t0 = tid / LPR;
  V* xg = x + (int64_t)r0 * nrhs + c;
  V* xs = XLDS ? reinterpret_cast<V*>(smem_raw) : nullptr;

  TPair<V> pe[D][EPL];
  TPair<V> pr[D];
  int4 dd[D];  // descriptor of the step held by stage k
  int4 dn[D];  // descriptor of the step stage k loads next
  constexpr int PS = (int)sizeof(TPair<V>);

#define PGS_LOAD_STAGE(K, DESC)                                                 \
  do {                                                                          \
    const int4 d_ = (DESC);                                                     \
    dd[K] = d_;                                                                 \
    const int tt_ = min(t0, max(d_.z - 1, 0));                                  \
    pr[K] = bload_pair(rs_ri, (d_.x + tt_) * PS, V(0));                         \
    const int eb_ = (d_.y + tt_ * d_.w + q) * PS;                               \
    _Pragma("unroll") for (int e_ = 0; e_ < EPL; ++e_)                          \
      pe[K][e_] = bload_pair(rs_ent, eb_ + e_ * LPR * PS, V(0));                \
  } while (0)

#pragma unroll
  for (int k = 0; k < D; ++k) {
    PGS_LOAD_STAGE(k, bload_i4(rs_desc, k * 16));
    dn[k] = bload_i4(rs_desc, (k + D) * 16);
  }
  // block column <- rhs column
  const V* rb = rhs + (int64_t)r0 * nrhs + c;
  if (XLDS) {
    for (int i = tid; i < nb; i += NT) xs[i] = rb[(int64_t)i * nrhs];
  } else {
    for (int i = tid; i < nb; i += NT) xg[(int64_t)i * nrhs] = rb[(int64_t)i * nrhs];
  }
  __syncthreads();
  for (int base = sbeg; base < send; base += D) {
#pragma unroll
    for (int k = 0; k < D; ++k) {
      const int s = base + k;
      const int4 d = dd[k];
      // gather first (all slots, columns are always in range), then mask the values
      const int row = pr[k].col;
      const V xrow = XLDS ? xs[row] : xg[(int64_t)row * nrhs];
      V xv[EPL];
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        const int cj = pe[k][e].col;
        xv[e] = XLDS ? xs[cj] : xg[(int64_t)cj * nrhs];
      }
      V acc = 0;
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        const V w = (q + e * LPR < d.w) ? pe[k][e].val : (V)0;
        acc += w * xv[e];
      }
      if constexpr (LPR == 4) {
        acc = quad_sum(acc);
      } else if constexpr (LPR == 2) {
        acc = pair_sum(acc);
      } else {
#pragma unroll
        for (int m = LPR / 2; m > 0; m >>= 1) acc += __shfl_xor(acc, m, LPR);
      }
      const V dv = pr[k].val;
      if (s < send && q == 0 && t0 < d.z) {
        V v = xrow - acc;
        if (s >= sU) v *= dv;
        if (XLDS) xs[row] = v;
        else xg[(int64_t)row * nrhs] = v;
      }
      if constexpr (XLDS) {
        // the stage registers are free again: start the loads of step s + D
        // before waiting at the barrier (the barrier only waits for LDS)
        PGS_LOAD_STAGE(k, dn[k]);
        dn[k] = bload_i4(rs_desc, (s - sbeg + 2 * D) * 16);
        __syncthreads();
      } else {
        // x lives in global memory: the barrier's release fence waits for all
        // outstanding vector memory operations, so issue the loads after it
        __syncthreads();
        PGS_LOAD_STAGE(k, dn[k]);
        dn[k] = bload_i4(rs_desc, (s - sbeg + 2 * D) * 16);
      }
    }
  }
#undef PGS_LOAD_STAGE
  if (XLDS) {
    for (int i = tid; i < nb; i += NT) xg[(int64_t)i * nrhs] = xs[i];
  }
}

// Ring kernel: one workgroup per (diagonal block, C = CG * NG right-hand-side
// columns); grid index = group * nblocks + block (all groups of a block on one
// XCD, as above).  The packed columns are ring slots: the value of the row
// stored at position p lives in LDS slot p % rows (CG values per slot, one ring
// per column group) from its step until its last reader, so the LDS footprint
// is the sweep window, not the block.  The L sweep reads rhs and writes y to x in
// global memory; the U sweep reads y back from x and overwrites it with the
// solution (a row's y is read before that row is written).
//
// What bounds it: a block is a chain of dependent steps (3,350 at 128^3), and a
// step is LDS gathers -> multiply-adds -> quad reduction -> LDS write -> barrier,
// about 230 clocks of latency, plus the instructions around it at 4 to 6 clocks
// each, since a SIMD issues one instruction of a wave at a time.  So the work is
// split over waves, one per SIMD for one column: NH * NG solving waves (NH = 2:
// the rows 0-15 and 16-31 of a step, NH = 1: half steps of at most 16 rows; NG
// groups of CG columns) do nothing but the chain, NH waves copy the factor
// records to LDS and one the right-hand sides, K steps ahead and straight from
// memory to LDS.  Four lanes solve a row with five entries each; lane q of a row
// finalizes columns q, q + 4, ...  When every wave did everything (5 entry loads, a
// row pair, a descriptor and a right-hand side per step: about 51 instructions
// for one FP32 column, 69 for FP64, against 35 and 42 in a solving wave now),
// level 0 took, us per launch at 128^3, FP32 / FP64, before -> now: 1 column 652 /
// 970 -> 495 / 664; 8 columns 740 / 1013 -> 599 / 803; 64 columns 1586 / 3699 ->
// 1452 / 2887; 64^3, 1 column: 219 / 255 -> 129 / 146; 1023 x 1021, 8 columns: 790 /
// 1020 -> 506 / 596.  With the loading waves idle the solving waves alone take
// 415 / 482 (128^3, 1 column) and 112 / 128 (64^3): LDS serves both.
template <typename V, int CG>
struct alignas(CG * sizeof(V) < 16 ? CG * sizeof(V) : 16) RingRow {
  V v[CG];
};

// A ring row read through its LDS byte address.  The ring kernel has no
// static LDS, so its dynamic LDS starts at address 0 (checked on the host
// when the kernels are set up): the address is the slot's byte offset.
template <typename T>
__device__ __forceinline__ T lds_read(unsigned addr) {
  constexpr int N = (int)sizeof(T) / 4;
  if constexpr (N == 1) {
    return __builtin_bit_cast(T, *reinterpret_cast<const __attribute__((address_space(3))) unsigned*>((size_t)addr));
  } else {
    using W = unsigned __attribute__((ext_vector_type(N)));
    return __builtin_bit_cast(T, *reinterpret_cast<const __attribute__((address_space(3))) W*>((size_t)addr));
  }
}

// Buffer stores (vector memory): writes outside the resource are dropped.
__device__ __forceinline__ void bstore_val(__amdgpu_buffer_rsrc_t r, int off, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, off, 0, 0);
}
__device__ __forceinline__ void bstore_val(__amdgpu_buffer_rsrc_t r, int off, double v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(__attribute__((ext_vector_type(2))) unsigned, v), r, off, 0, 0);
}
__device__ __forceinline__ void bstore_val(__amdgpu_buffer_rsrc_t r, int off, cplx<float> v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(__attribute__((ext_vector_type(2))) unsigned, v), r, off, 0, 0);
}
__device__ __forceinline__ void bstore_val(__amdgpu_buffer_rsrc_t r, int off, cplx<double> v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned, v), r, off, 0, 0);
}

// Two consecutive values in one buffer access (8-byte and smaller values).
template <typename V>
__device__ __forceinline__ void bstore_val2(__amdgpu_buffer_rsrc_t r, int off, const RingRow<V, 2>& o) {
  static_assert(sizeof(V) <= 8, "two values in one access");
  if constexpr (sizeof(V) == 4)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(__attribute__((ext_vector_type(2))) unsigned, o), r, off, 0, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned, o), r, off, 0, 0);
}

// An empty asm that takes a value as read and rewritten: the value must have
// arrived, and it counts as produced here rather than by its load.
__device__ __forceinline__ void pin_reg(int& v) { __asm__ __volatile__("" : "+v"(v)); }

// The records of the factor entries are laid out by ring_pack.hpp: a lane's five
// values and five ring slots, in pieces.
template <typename V>
struct LaneRec {
  V val[5];
  unsigned s01, s23, s4;
};

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// LDS byte address of a ring row: base + slot * RS with the slot in the low or
// high half of w, one instruction.
template <int RS, bool HIGH>
__device__ __forceinline__ unsigned slot_addr(unsigned w, unsigned base) {
  unsigned a;
  if constexpr (HIGH) __asm__("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(a) : "v"(w), "s"(RS), "v"(base));
  else __asm__("v_mad_u32_u16 %0, %1, %2, %3" : "=v"(a) : "v"(w), "s"(RS), "v"(base));
  return a;
}

// A value written through its LDS byte address.
template <typename T>
__device__ __forceinline__ void lds_write(unsigned addr, const T& v) {
  constexpr int N = (int)sizeof(T) / 4;
  if constexpr (N == 1) {
    *reinterpret_cast<__attribute__((address_space(3))) unsigned*>((size_t)addr) = __builtin_bit_cast(unsigned, v);
  } else {
    using W = unsigned __attribute__((ext_vector_type(N)));
    *reinterpret_cast<__attribute__((address_space(3))) W*>((size_t)addr) = __builtin_bit_cast(W, v);
  }
}

// Pieces of a lane's record: loads (and direct-to-LDS copies) per wave and step.
template <typename V>
constexpr int ring_pieces() {
  return sizeof(V) == 4 ? 2 : sizeof(V) == 8 ? 4 : 6;
}
// Bytes of one wave's records in LDS: piece i at i * 1024, 16 bytes per lane (the
// last piece of 8-byte values: 4).
template <typename V>
constexpr int ring_stage_bytes() {
  return 16 * ring_row_bytes<V>();
}

// A right-hand side row of C values in pieces that direct-to-LDS copies can move
// (4 or 16 bytes per lane): U bytes each, ND copies for the 16 NH rows of a step.
template <typename V, int C, int NH>
struct RingRhs {
  static constexpr int row = C * (int)sizeof(V);
  static constexpr int U = row < 16 ? 4 : 16;
  static constexpr int ND = (16 * NH * row / U + 63) / 64;
};

// LDS of the ring kernel in bytes, by offset: NG rings of CG columns (each with
// its dummy row), then K stages of {records of 16 NH rows; 32 pairs (ring slot
// times sizeof(V), row id); 32 pivots; the rows' right-hand sides}.  A copy moves
// a piece of every lane, so a part holds at least 64 pieces.
template <typename V, int CG, int NG, int NH>
struct RingLds {
  using R = RingRhs<V, CG * NG, NH>;
  static constexpr int rec = NH * ring_stage_bytes<V>();
  static constexpr int info = 64 * 4, piv = 64 * (sizeof(V) == 16 ? 16 : 4), rhs = R::ND * 64 * R::U;
  static constexpr int stage = rec + info + piv + rhs;
  __host__ __device__ static int ring(int rows) { return ((rows + 1) * CG * (int)sizeof(V) + 15) & ~15; }
  __host__ __device__ static int bytes(int rows, int K) { return NG * ring(rows) + K * stage; }
};

// Hand-over of the stages.  A stage's reads are issued a step ahead (take).  With
// two waves per group of columns (NH = 2) a step ends with all LDS work done,
// since the waves read each other's ring rows; the stage taken in a step is free
// at its end.  With one wave per group (NH = 1) no other wave reads its ring: LDS
// serves a wave's accesses in order, so a step ends at once, without waiting for
// its ring write or for the reads of the next step's stage.  That stage is free
// a step later, when its values have been used: the loading waves run one step
// later ("late": K - 1 steps ahead, K - 3 in flight), and the solving waves need
// K > 4 stages (with 4 only one copy would be in flight: 96^3, 64 columns, 830 ->
// 1040 us).  One column, FP64: 64^3 171 -> 150 us, 1023x1021 570 -> 520.
template <int NH, int K>
constexpr bool ring_late() { return NH == 1 && K > 4; }

// Sweep of a wave that moves records: those of the group of rows HC of each step
// (the first or the second 16).  Between the barriers of steps s - 1 and s it
// starts the copy of the records of step s + K (late: s + K - 1) into a stage that
// the solving waves have done with, and waits until those of step s + 2 have
// arrived.  The first of these waves also moves the ring slots and row ids, the
// last the pivots: issuing the copies is what the loading waves spend their time
// on, and the slowest of them sets the step (one wave for both groups, with all
// row data on its neighbour: level 0 at 128^3, 1 column, 664 us in FP64 where the
// solving waves alone take 482).
template <typename V, int K, int CG, int NG, int NH, int HC, bool UPPER>
__device__ __forceinline__ void ring_copy_sweep(int nsteps, const int* pos, int rows, int dummy,
                                                __amdgpu_buffer_rsrc_t rs_ent, __amdgpu_buffer_rsrc_t rs_info,
                                                __amdgpu_buffer_rsrc_t rs_dinv) {
  constexpr int RB = ring_row_bytes<V>(), PB = ring_stage_bytes<V>(), NP = ring_pieces<V>();
  using L = RingLds<V, CG, NG, NH>;
  static_assert(2 * K + 2 <= 64, "step boundaries of a pass and its look-ahead in one register");
  constexpr int late = ring_late<NH, K>() ? 1 : 0;
  // the copies of the K - 2 steps after s + 2 (late: K - 3)
  constexpr bool kInfo = HC == 0, kPiv = UPPER && HC == NH - 1;
  constexpr int kWait = K > 2 ? (K - 2 - late) * (NP + (kInfo ? 1 : 0) + (kPiv ? 1 : 0)) : 0;
  static_assert(kWait <= 60, "outstanding copies");
  const int lane = threadIdx.x & 63;
  const unsigned stage0 = (unsigned)(NG * L::ring(rows));
  const __amdgpu_buffer_rsrc_t rs_pos = make_rsrc(pos, (int64_t)(nsteps + 1) * 4);
  int pv = (int)__builtin_amdgcn_raw_buffer_load_b32(rs_pos, min(lane, nsteps) * 4, 0, 0);
  const int l16 = lane * 16;
  auto copy_group = [&](unsigned a, int p, int n) {
    // lanes past a group's rows copy zeros (no memory traffic)
    using LP = __attribute__((address_space(3))) void*;
    const bool in = lane < 4 * n;
    const int vo16 = in ? l16 : kRingOut;
    const int base = p * RB, pc = n * 64;
    constexpr int N16 = sizeof(V) == 8 ? 3 : NP;
#pragma unroll
    for (int j = 0; j < N16; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_ent, (LP)(size_t)(a + j * 1024), 16, vo16, base + j * pc, 0, 0);
    if constexpr (sizeof(V) == 8)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_ent, (LP)(size_t)(a + 3 * 1024), 4, in ? lane * 4 : kRingOut, base + 3 * pc,
                                               0, 0);
  };
  auto copy_step = [&](int stage, int i) {  // step i of the pass
    const int p0 = __builtin_amdgcn_readlane(pv, i), n = __builtin_amdgcn_readlane(pv, i + 1) - p0;
    const int n0 = min(n, kRingGroup);
    const unsigned a = stage0 + stage * L::stage;
    if constexpr (HC == 0) copy_group(a, p0, n0);
    else copy_group(a + PB, p0 + n0, n - n0);
    // lanes past the step's rows copy the dummy row's pair and no pivot
    using LP = __attribute__((address_space(3))) void*;
    if constexpr (kInfo)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_info, (LP)(size_t)(a + L::rec), 4,
                                               lane < 2 * n ? lane * 4 : dummy - p0 * 8 + (lane & 1) * 4, p0 * 8, 0, 0);
    if constexpr (kPiv) {
      if constexpr (sizeof(V) == 16)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_dinv, (LP)(size_t)(a + L::rec + L::info), 16,
                                                 lane < n ? l16 : kRingOut, p0 * 16, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_dinv, (LP)(size_t)(a + L::rec + L::info), 4,
                                                 lane < n * ((int)sizeof(V) / 4) ? lane * 4 : kRingOut,
                                                 p0 * (int)sizeof(V), 0, 0);
    }
  };
#pragma unroll
  for (int k = 0; k < K - late; ++k) copy_step(k, k);
  __builtin_amdgcn_sched_barrier(0);
  __asm__ __volatile__("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  // the solving waves take step 0 here, before its stage is used again
  if constexpr (!late) __builtin_amdgcn_s_barrier();
  __asm__ __volatile__("" ::: "memory");
  for (int base = 0; base < nsteps; base += K) {
    const int pvn = (int)__builtin_amdgcn_raw_buffer_load_b32(rs_pos, min(base + K + lane, nsteps) * 4, 0, 0);
#pragma unroll
    for (int kk = 0; kk < K; ++kk) {
      copy_step((kk + K - late) % K, kk + K - late);
      __builtin_amdgcn_sched_barrier(0);
      __asm__ __volatile__("s_waitcnt vmcnt(%0)" ::"n"(kWait) : "memory");
      __builtin_amdgcn_s_barrier();
      __asm__ __volatile__("" ::: "memory");
    }
    pv = pvn;
  }
  // nothing may still be on its way to LDS when the stages are used again or
  // the workgroup ends
  __asm__ __volatile__("s_waitcnt vmcnt(0)" ::: "memory");
}

// Sweep of the wave that moves the right-hand sides, as ring_copy_sweep the
// records; the row ids that their addresses need are loaded K steps before them.
template <typename V, int K, int CG, int NG, int NH>
__device__ __forceinline__ void ring_row_sweep(int nsteps, const int* pos, int rows, int nrhs, int c0,
                                               __amdgpu_buffer_rsrc_t rs_info, __amdgpu_buffer_rsrc_t rs_src) {
  constexpr int VS = (int)sizeof(V);
  using L = RingLds<V, CG, NG, NH>;
  using R = typename L::R;
  constexpr int ND = R::ND, U = R::U;
  constexpr int OPS = 2 * ND;
  constexpr int late = ring_late<NH, K>() ? 1 : 0;
  constexpr int kWait = K > 2 ? (K - 2 - late) * OPS : 0;
  static_assert(kWait <= 60, "outstanding loads");
  static_assert(3 * K + 2 <= 64, "step boundaries of a pass and its look-ahead in one register");
  const int lane = threadIdx.x & 63;
  const int csh = __builtin_ctz((unsigned)nrhs);
  const unsigned stage0 = (unsigned)(NG * L::ring(rows));
  using LP = __attribute__((address_space(3))) void*;
  int rl[ND], rb[ND];  // this lane's row of the step and byte of the row, per copy
#pragma unroll
  for (int j = 0; j < ND; ++j) {
    rl[j] = (j * 64 + lane) * U / R::row;
    rb[j] = c0 * VS + (j * 64 + lane) * U % R::row;
  }
  int rowr[K][ND];

  const __amdgpu_buffer_rsrc_t rs_pos = make_rsrc(pos, (int64_t)(nsteps + 1) * 4);
  int pv = (int)__builtin_amdgcn_raw_buffer_load_b32(rs_pos, min(lane, nsteps) * 4, 0, 0);
  auto bnd = [&](int i) { return __builtin_amdgcn_readlane(pv, i); };
  auto load_row = [&](int k, int i) {
    const int p = bnd(i), n = bnd(i + 1) - p;
#pragma unroll
    for (int j = 0; j < ND; ++j)
      rowr[k][j] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs_info, rl[j] < n ? rl[j] * 8 + 4 : kRingOut, p * 8, 0);
  };
  // right-hand sides of step i of the pass into stage k, their row ids in
  // rowr[k]; lanes past the step's rows copy zeros (no memory traffic)
  auto copy_step = [&](int k, int i) {
    const int p = bnd(i), n = bnd(i + 1) - p;
    const unsigned a = stage0 + k * L::stage + L::rec;
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      const int o = (int)((unsigned)rowr[k][j] << csh) * VS + rb[j];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_src, (LP)(size_t)(a + L::info + L::piv + j * 64 * U), U,
                                               rl[j] < n ? o : kRingOut, 0, 0, 0);
    }
  };
#pragma unroll
  for (int k = 0; k < K; ++k) load_row(k, k);
#pragma unroll
  for (int k = 0; k < K - late; ++k) copy_step(k, k);
#pragma unroll
  for (int k = 0; k < K - late; ++k) load_row(k, K + k);
  // The compiler gives the loop's first steps the load waits of the worst
  // path into them.  Taking the prologue's registers as redefined here (one
  // wait for its loads, once per sweep) leaves the loop the waits of its own
  // back edge.
  __builtin_amdgcn_sched_barrier(0);
  __asm__ __volatile__("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int k = 0; k < K; ++k)
#pragma unroll
    for (int j = 0; j < ND; ++j) pin_reg(rowr[k][j]);
  __builtin_amdgcn_s_barrier();
  // the solving waves take step 0 here, before its stage is used again
  if constexpr (!late) __builtin_amdgcn_s_barrier();
  __asm__ __volatile__("" ::: "memory");
  for (int base = 0; base < nsteps; base += K) {
    const int pvn = (int)__builtin_amdgcn_raw_buffer_load_b32(rs_pos, min(base + K + lane, nsteps) * 4, 0, 0);
#pragma unroll
    for (int kk = 0; kk < K; ++kk) {
      copy_step((kk + K - late) % K, kk + K - late);
      load_row((kk + K - late) % K, kk + 2 * K - late);
      __builtin_amdgcn_sched_barrier(0);
      __asm__ __volatile__("s_waitcnt vmcnt(%0)" ::"n"(kWait) : "memory");
      __builtin_amdgcn_s_barrier();
      __asm__ __volatile__("" ::: "memory");
    }
    pv = pvn;
  }
  __asm__ __volatile__("s_waitcnt vmcnt(0)" ::: "memory");
}

// Sweep of the solving waves: wave g * NH + h of group g of CG columns takes
// rows 16 h .. 16 h + 15 of each step (NH = 2), or all of a half step's (NH = 1).
template <typename V, int K, int CG, int NG, int NH, bool UPPER>
__device__ __forceinline__ void ring_solve_sweep(int h, int g, int nsteps, int rows, int nrhs, int c0,
                                                 __amdgpu_buffer_rsrc_t rs_dst) {
  constexpr int VS = (int)sizeof(V);
  constexpr int PB = ring_stage_bytes<V>();
  using L = RingLds<V, CG, NG, NH>;
  constexpr int NCL = CG == 8 ? 2 : 1;  // columns finalized per lane: adjacent ones, one access for both
  static_assert(CG == 1 || CG == 2 || CG == 4 || (CG == 8 && VS == 4), "columns per group");
  // Left alone, the compiler moves reads of the next step's stage before the last
  // gathers and their waits into the sum.  Holding it back: 64^3, 8 / 64 FP32
  // columns 169 -> 160 and 274 -> 253 us; 128^3, 1 column 516 -> 498; but with
  // several columns and two waves per group up to 3 % slower.
  constexpr bool kOrder = NH == 1 || CG == 1;
  const int lane = threadIdx.x & 63;
  const int q = lane % 4;
  const int t = 16 * h + lane / 4;                      // this lane's row of the step
  const int cq = CG == 8 ? 2 * q : q % CG;              // after the reduction the lane holds column cq (and cq + 1 of 8)
  const unsigned gat = g * (unsigned)L::ring(rows);     // this group's ring
  const unsigned wad = gat + cq * VS;                   // this lane's column of its row 0
  const int cl = g * CG + cq;
  const int sh = __builtin_ctz((unsigned)nrhs * (unsigned)VS);
  const unsigned coff = (unsigned)((c0 + cl) * VS);
  const unsigned ring_end = NG * (unsigned)L::ring(rows);
  const unsigned st_a = ring_end + h * PB + lane * 16;
  const unsigned st_x = ring_end + h * PB + 3 * 1024 + lane * 4;
  const unsigned info_a = ring_end + L::rec + t * 8;
  const unsigned piv_a = ring_end + L::rec + L::info + t * VS;
  const unsigned rhs_a = ring_end + L::rec + L::info + L::piv + (t * CG * NG + cl) * VS;

  LaneRec<V> rec;
  u32x2 info;
  V xin[NCL], dv = V(0);
  auto take = [&](int stage) {  // the records and row data of a step
    const unsigned a = st_a + stage * L::stage;
    if constexpr (sizeof(V) == 4) {
      const u32x4 v0 = lds_read<u32x4>(a), v1 = lds_read<u32x4>(a + 1024);
#pragma unroll
      for (int e = 0; e < 4; ++e) rec.val[e] = __uint_as_float(v0[e]);
      rec.val[4] = __uint_as_float(v1[0]);
      rec.s01 = v1[1];
      rec.s23 = v1[2];
      rec.s4 = v1[3];
    } else if constexpr (sizeof(V) == 8) {
      const u32x4 v0 = lds_read<u32x4>(a), v1 = lds_read<u32x4>(a + 1024), v2 = lds_read<u32x4>(a + 2048);
      rec.s4 = lds_read<unsigned>(st_x + stage * L::stage);
      rec.val[0] = __builtin_bit_cast(V, u32x2{v0[0], v0[1]});
      rec.val[1] = __builtin_bit_cast(V, u32x2{v0[2], v0[3]});
      rec.val[2] = __builtin_bit_cast(V, u32x2{v1[0], v1[1]});
      rec.val[3] = __builtin_bit_cast(V, u32x2{v1[2], v1[3]});
      rec.val[4] = __builtin_bit_cast(V, u32x2{v2[0], v2[1]});
      rec.s01 = v2[2];
      rec.s23 = v2[3];
    } else {
#pragma unroll
      for (int e = 0; e < 5; ++e) rec.val[e] = __builtin_bit_cast(V, lds_read<u32x4>(a + e * 1024));
      const u32x4 x = lds_read<u32x4>(a + 5 * 1024);
      rec.s01 = x[0];
      rec.s23 = x[1];
      rec.s4 = x[2];
    }
    const unsigned d = stage * L::stage;
    info = lds_read<u32x2>(info_a + d);
    if constexpr (NCL == 2) {
      const RingRow<V, 2> r = lds_read<RingRow<V, 2>>(rhs_a + d);
      xin[0] = r.v[0];
      xin[1] = r.v[1];
    } else {
      xin[0] = lds_read<V>(rhs_a + d);
    }
    if constexpr (UPPER) dv = lds_read<V>(piv_a + d);
  };

  __syncthreads();  // the loading waves have filled the first stages
  take(0);
  if constexpr (!ring_late<NH, K>()) __syncthreads();  // step 0 is taken: its stage may be used again
  for (int base = 0; base < nsteps; base += K) {
#pragma unroll
    for (int kk = 0; kk < K; ++kk) {
      const unsigned sa[5] = {slot_addr<CG * VS, false>(rec.s01, gat), slot_addr<CG * VS, true>(rec.s01, gat),
                              slot_addr<CG * VS, false>(rec.s23, gat), slot_addr<CG * VS, true>(rec.s23, gat),
                              slot_addr<CG * VS, false>(rec.s4, gat)};
      RingRow<V, CG> xv[5];
      V wgt[5];
#pragma unroll
      for (int e = 0; e < 5; ++e) {
        xv[e] = lds_read<RingRow<V, CG>>(sa[e]);
        wgt[e] = rec.val[e];  // padded slots weigh zero
      }
      const unsigned wa = CG * NG == 1 ? info[0] : info[0] * CG + wad;
      const int off = (int)((info[1] << sh) + coff);
      V x0[NCL];
#pragma unroll
      for (int j = 0; j < NCL; ++j) x0[j] = xin[j];
      const V d0 = dv;
      // the next step's records and row data follow the gathers in the LDS queue
      if constexpr (kOrder) __builtin_amdgcn_sched_barrier(0);
      take((kk + 1) % K);
      V acc[CG];
#pragma unroll
      for (int c = 0; c < CG; ++c) acc[c] = 0;
#pragma unroll
      for (int e = 0; e < 5; ++e) {
#pragma unroll
        for (int c = 0; c < CG; ++c) acc[c] += wgt[e] * xv[e].v[c];
      }
      // nothing that waits for the reads after the gathers comes before this
      if constexpr (kOrder) __builtin_amdgcn_sched_barrier(0);
      // sum over the row's lanes, scattered so that lane q ends with column q % CG
      // (with 8 columns: columns 2q and 2q + 1)
      V a[NCL];
      if constexpr (CG == 8) {
        // xor 2: keep columns 0-3 (q bit 1 clear) or 4-7, send the other half
        const bool b0 = q & 1, b1 = q & 2;
        V hh[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) hh[c] = (b1 ? acc[c + 4] : acc[c]) + dpp_xor2(b1 ? acc[c] : acc[c + 4]);
        // xor 1: keep columns 0-1 of the half (q bit 0 clear) or 2-3
#pragma unroll
        for (int c = 0; c < 2; ++c) a[c] = (b0 ? hh[c + 2] : hh[c]) + dpp_xor1(b0 ? hh[c] : hh[c + 2]);
      } else if constexpr (CG == 4) {
        // xor 1: keep columns with bit 0 = q bit 0, send the other two
        const bool b0 = q & 1, b1 = q & 2;
        const V k0 = (b0 ? acc[1] : acc[0]) + dpp_xor1(b0 ? acc[0] : acc[1]);
        const V k1 = (b0 ? acc[3] : acc[2]) + dpp_xor1(b0 ? acc[2] : acc[3]);
        // xor 2: keep the pair with bit 1 = q bit 1
        a[0] = (b1 ? k1 : k0) + dpp_xor2(b1 ? k0 : k1);
      } else if constexpr (CG == 2) {
        const bool b0 = q & 1;
        const V k0 = (b0 ? acc[1] : acc[0]) + dpp_xor1(b0 ? acc[0] : acc[1]);
        a[0] = k0 + dpp_xor2(k0);
      } else {
        a[0] = quad_sum(acc[0]);
      }
      // with fewer than four columns several lanes hold and write the same
      // value; lanes past the step's rows write the dummy ring row and past
      // the buffer's range (dropped): no branch
      if constexpr (NCL == 2) {
        RingRow<V, 2> o;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          o.v[j] = x0[j] - a[j];
          if (UPPER) o.v[j] *= d0;
        }
        lds_write(wa, o);
        bstore_val2<V>(rs_dst, off, o);
      } else {
        V v = x0[0] - a[0];
        if (UPPER) v *= d0;
        lds_write(wa, v);
        bstore_val(rs_dst, off, v);
      }
      if constexpr (ring_late<NH, K>()) {
        __asm__ __volatile__("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __asm__ __volatile__("" ::: "memory");
      } else {
        __syncthreads();
      }
    }
  }
}

// pos: per block b the boundaries of its steps (blk_step[b + 1] - blk_step[b] + 1
// values from blk_step[b] + b; the first of them is 0, sU's the block's
// rows).  info, dinv: per position the pair (ring slot times sizeof(V),
// block-local row id) from ring_info0, the dummy row's pair after the block's
// own, and 1/pivot from blk_ri0[b]; ent: the block's records, from blk_ri0[b] *
// ring_row_bytes<V>().
template <typename V, int K, int CG, int NG, int NH>
__global__ __launch_bounds__(64 * (NH * NG + NH + 1)) void k_trsv_ring(
    int nblocks, int rows, const int* __restrict__ blk_row0, const int* __restrict__ blk_step,
    const int* __restrict__ blk_stepU, const int64_t* __restrict__ blk_ri0, const int* __restrict__ pos,
    const unsigned char* __restrict__ ent, const RingInfo* __restrict__ info, const V* __restrict__ dinv,
    const V* __restrict__ rhs, V* __restrict__ x, int nrhs) {
  extern __shared__ unsigned char smem_raw[];
  const int b = blockIdx.x % nblocks;
  const int c0 = (blockIdx.x / nblocks) * CG * NG;
  const int r0 = blk_row0[b], nb = blk_row0[b + 1] - r0;
  const int sbeg = blk_step[b], send = blk_step[b + 1], sU = blk_stepU[b];
  const int64_t q0 = blk_ri0[b], np = blk_ri0[b + 1] - q0;
  const int* pb = pos + sbeg + b;
  const int64_t vbytes = (int64_t)nb * nrhs * (int64_t)sizeof(V);
  V* xb = x + (int64_t)r0 * nrhs;
  const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(xb, vbytes);
  const __amdgpu_buffer_rsrc_t rs_info = make_rsrc(info + ring_info0(q0, b), (np + 1) * 8);
  // rings, dummy rows and stages start as zeros: a record that is not there reads
  // slot 0 with weight zero
  uint4* lds4 = reinterpret_cast<uint4*>(smem_raw);
  for (int i = threadIdx.x; i < RingLds<V, CG, NG, NH>::bytes(rows, K) / 16; i += 64 * (NH * NG + NH + 1)) lds4[i] = uint4{0, 0, 0, 0};
  __syncthreads();
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (w < NH * NG) {
    const int h = NH == 1 ? 0 : w % 2, g = NG == 1 ? 0 : w / NH;
    ring_solve_sweep<V, K, CG, NG, NH, false>(h, g, sU - sbeg, rows, nrhs, c0, rs_x);
    // y of every row has reached memory before the row data's wave reads it back (a
    // barrier alone orders LDS, not one wave's stores before another's copies)
    __asm__ __volatile__("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    ring_solve_sweep<V, K, CG, NG, NH, true>(h, g, send - sU, rows, nrhs, c0, rs_x);
  } else if (w < NH * NG + NH) {
    const __amdgpu_buffer_rsrc_t rs_ent = make_rsrc(ent + q0 * ring_row_bytes<V>(), np * ring_row_bytes<V>());
    const __amdgpu_buffer_rsrc_t rs_dinv = make_rsrc(dinv + q0, np * (int64_t)sizeof(V));
    const int dummy = (int)(np * 8);
    auto copies = [&](auto hc) {
      constexpr int HC = decltype(hc)::value;
      ring_copy_sweep<V, K, CG, NG, NH, HC, false>(sU - sbeg, pb, rows, dummy, rs_ent, rs_info, rs_dinv);
      __syncthreads();
      ring_copy_sweep<V, K, CG, NG, NH, HC, true>(send - sU, pb + (sU - sbeg), rows, dummy, rs_ent, rs_info, rs_dinv);
    };
    if (NH == 1 || w == NH * NG) copies(std::integral_constant<int, 0>());
    else copies(std::integral_constant<int, NH - 1>());
  } else {
    ring_row_sweep<V, K, CG, NG, NH>(sU - sbeg, pb, rows, nrhs, c0, rs_info, make_rsrc(rhs + (int64_t)r0 * nrhs, vbytes));
    __syncthreads();
    ring_row_sweep<V, K, CG, NG, NH>(send - sU, pb + (sU - sbeg), rows, nrhs, c0, rs_info, rs_x);
  }
}

}  // namespace dev
}  // namespace pgs
