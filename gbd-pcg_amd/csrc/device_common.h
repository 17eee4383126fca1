// Device helpers shared by the PCG kernels: exchange words, global-pointer
// casts and DPP-based cross-lane reductions (gfx950 / GFX9 DPP).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "internal.h"

namespace gbdpcg {

// ---------------------------------------------------------------------------
// exchange words
// ---------------------------------------------------------------------------

// Global-address-space view of a generic pointer: accesses compile to global_*
// instead of flat_* (flat operations also count against the LDS wait counter).
template <typename T>
using gptr_t = __attribute__((address_space(1))) T *;
template <typename T>
__device__ __forceinline__ gptr_t<T> gptr(T *p) {
  return (gptr_t<T>)p;
}
template <typename T>
__device__ __forceinline__ gptr_t<const T> gptr(const T *p) {
  return (gptr_t<const T>)p;
}

__device__ __forceinline__ void xstore(uint64_t *p, uint32_t payload, uint32_t epoch) {
  const uint64_t w = ((uint64_t)epoch << 32) | (uint64_t)payload;
  __hip_atomic_store(gptr(p), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Same word with a workgroup-scope store: it completes in the XCD's shared L2
// (the CU's L1 is write-through) instead of being written through to memory, and
// the device-scope polls below, which skip the L1, find it there.  Only valid
// when the writer and every reader of the word run on the same XCD; the kernels
// check that at run time (xcc_id) before using it.
__device__ __forceinline__ void xstore_xcd(uint64_t *p, uint32_t payload, uint32_t epoch) {
  const uint64_t w = ((uint64_t)epoch << 32) | (uint64_t)payload;
  __hip_atomic_store(gptr(p), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ void xstore_sel(uint64_t *p, uint32_t payload, uint32_t epoch, bool xcd) {
  if (xcd)
    xstore_xcd(p, payload, epoch);
  else
    xstore(p, payload, epoch);
}

// XCD (accelerator complex die) this wave runs on: hardware register XCC_ID,
// bits [3:0].
__device__ __forceinline__ uint32_t xcc_id() { return (uint32_t)__builtin_amdgcn_s_getreg((3 << 11) | 20) & 0xFu; }

// A value every lane holds identically, moved to a scalar register: later
// arithmetic on it can use SGPR operands and branches on it become scalar.
__device__ __forceinline__ float uniform(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ double uniform(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffll));
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

__device__ __forceinline__ uint64_t xload(uint64_t *p) {
  return __hip_atomic_load(gptr(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Spins until *p carries `epoch`; returns false when the spin bound is reached.
__device__ __forceinline__ bool xwait(uint64_t *p, uint32_t epoch, uint32_t &payload) {
  for (uint32_t spin = 0; spin < kSpinLimit; ++spin) {
    const uint64_t w = xload(p);
    if ((uint32_t)(w >> 32) == epoch) {
      payload = (uint32_t)w;
      return true;
    }
  }
  return false;
}

// Fused multiply-add in the precision of T (__builtin_fma on floats would
// promote to double).
__device__ __forceinline__ float fmaT(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmaT(double a, double b, double c) { return __builtin_fma(a, b, c); }

// Single-word wait for words that usually land before the caller looks (edge
// values): polls with a short sleep to keep the polling traffic low.
__device__ __forceinline__ bool xwait_lazy(uint64_t *p, uint32_t epoch, uint32_t &payload) {
  for (uint32_t spin = 0; spin < kSpinLimit; ++spin) {
    const uint64_t w = xload(p);
    if ((uint32_t)(w >> 32) == epoch) {
      payload = (uint32_t)w;
      return true;
    }
    __builtin_amdgcn_s_sleep(4);
  }
  return false;
}

// Waits until the NW consecutive words at p all carry `epoch` (one group of
// loads per poll).
template <int NW>
__device__ __forceinline__ bool xwait_words(uint64_t *p, uint32_t epoch, uint32_t (&out)[NW]) {
  for (uint32_t spin = 0; spin < kSpinLimit; ++spin) {
    uint64_t A[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) A[i] = xload(p + i);
    bool ok = true;
#pragma unroll
    for (int i = 0; i < NW; ++i) ok = ok && (uint32_t)(A[i] >> 32) == epoch;
    if (ok) {
#pragma unroll
      for (int i = 0; i < NW; ++i) out[i] = (uint32_t)A[i];
      return true;
    }
  }
  return false;
}


// a / b for the scalar recurrences.  FP32: hardware reciprocal (1 ulp) and one
// residual correction of the quotient, about 1 ulp in all (no denormal-mode
// switches, unlike the IEEE sequence, and four dependent operations instead of
// ten).  Meaningful for finite non-zero b only: callers test b and discard the
// quotient otherwise.
template <typename T>
__device__ __forceinline__ T qdiv(T a, T b) {
  if constexpr (sizeof(T) == 4) {
    const float r = __builtin_amdgcn_rcpf(b);
    const float q = a * r;
    const float res = __builtin_fmaf(-b, q, a);
    return __builtin_fmaf(res, r, q);
  } else {
    return a / b;
  }
}

template <typename T>
__device__ __forceinline__ uint32_t payload_word(T v, int q) {
  if constexpr (sizeof(T) == 4) {
    return __float_as_uint(v);
  } else {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    return q == 0 ? (uint32_t)b : (uint32_t)(b >> 32);
  }
}

// ---------------------------------------------------------------------------
// reductions (deterministic: the same data give bit-identical sums in every
// lane, wave and workgroup)
// ---------------------------------------------------------------------------

// Cross-lane moves use DPP (a VALU operand modifier, a few cycles) rather than
// __shfl_xor, which lowers to ds_bpermute and costs an LDS round trip per step.
// Every control used has a source lane for each lane: there is no previous value to
// set up, and FP32 additions take the move as their operand.  GFX9 DPP controls:
constexpr int kDppQuadXor1 = 0xB1;  // quad_perm [1,0,3,2]
constexpr int kDppQuadXor2 = 0x4E;  // quad_perm [2,3,0,1]
constexpr int kDppRowRor4 = 0x124, kDppRowRor8 = 0x128;  // rotations of rows of 16 lanes

// Value of `v` from the lane selected by CTRL.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo));
}

// Two values exchanged across halves of the wave (W 32: the upper half of a with
// the lower of b) or neighbouring rows of 16 lanes (W 16: a's odd rows with b's
// even ones).  Afterwards a + b holds, in the lower half (in the even rows), the
// sums of a's halves (rows) and in the others those of b: two values folded into
// one by one instruction per 32 bits and an addition.
template <int W>
__device__ __forceinline__ void swap_lanes(uint32_t &a, uint32_t &b) {
  if constexpr (W == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  }
}
template <int W>
__device__ __forceinline__ void swap_lanes(float &a, float &b) {
  uint32_t x = __float_as_uint(a), y = __float_as_uint(b);
  swap_lanes<W>(x, y);
  a = __uint_as_float(x);
  b = __uint_as_float(y);
}
template <int W>
__device__ __forceinline__ void swap_lanes(double &a, double &b) {
  const uint64_t u = (uint64_t)__double_as_longlong(a), v = (uint64_t)__double_as_longlong(b);
  uint32_t xl = (uint32_t)u, xh = (uint32_t)(u >> 32), yl = (uint32_t)v, yh = (uint32_t)(v >> 32);
  swap_lanes<W>(xl, yl);
  swap_lanes<W>(xh, yh);
  a = __longlong_as_double((long long)(((uint64_t)xh << 32) | xl));
  b = __longlong_as_double((long long)(((uint64_t)yh << 32) | yl));
}
template <int W, typename T>
__device__ __forceinline__ T fold(T a, T b) {
  swap_lanes<W>(a, b);
  return a + b;
}

// Value of lane l (a constant), uniform.
__device__ __forceinline__ float read_lane(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double read_lane(double v, int l) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Sums over each row of 16 lanes, in all of them (not the same bits in each: take
// the row's first lane).
template <typename T>
__device__ __forceinline__ T row_sum(T v) {
  v += dpp<kDppQuadXor1>(v);
  v += dpp<kDppQuadXor2>(v);
  v += dpp<kDppRowRor4>(v);
  v += dpp<kDppRowRor8>(v);
  return v;
}

// Three sums over the 64 lanes of a wave (all lanes active): sum l in lane 16 l.  A
// fixed tree: identical inputs give identical bits in every wave.  The iteration of
// FP64 systems of n = 28 is bound by VALU issue, a fifth of which six separate scans
// took (three instructions per 32 bits and step); folded, six sums take 39
// instructions instead of 276, three in FP32 11 instead of 57.
template <typename T>
__device__ __forceinline__ T wave_sums(T s0, T s1, T s2) {
  return row_sum(fold<16>(fold<32>(s0, s2), fold<32>(s1, s1)));
}

// The same for the even and the odd lanes by themselves: sum l of the even lanes in
// lane 16 l, of the odd ones in lane 16 l + 1.
template <typename T>
__device__ __forceinline__ T wave_sums_parity(T s0, T s1, T s2) {
  T v = fold<16>(fold<32>(s0, s2), fold<32>(s1, s1));
  v += dpp<kDppQuadXor2>(v);
  v += dpp<kDppRowRor4>(v);
  v += dpp<kDppRowRor8>(v);
  return v;
}

// Six such sums: sums 0..3 in lanes 16 l, sum 4 in lane 1, sum 5 in lane 33.
template <typename T>
__device__ __forceinline__ T wave_sums(T s0, T s1, T s2, T s3, T s4, T s5) {
  const T a = fold<16>(fold<32>(s0, s2), fold<32>(s1, s3));
  const T h = fold<32>(s4, s5), b = fold<16>(h, h);
  const bool odd = (threadIdx.x & 1) != 0;  // even lanes go on with a, odd ones with b
  T v = (odd ? b : a) + dpp<kDppQuadXor1>(odd ? a : b);
  v += dpp<kDppQuadXor2>(v);
  v += dpp<kDppRowRor4>(v);
  v += dpp<kDppRowRor8>(v);
  return v;
}
// Index of the sum that this lane holds after wave_sums of COUNT values, or -1.
template <int COUNT>
__device__ __forceinline__ int wave_sums_slot() {
  const int l = (int)threadIdx.x & 63;
  if constexpr (COUNT == 3) return (l & 15) == 0 && l < 48 ? l >> 4 : -1;
  return (l & 15) == 0 ? l >> 4 : (l & 31) == 1 ? 4 + (l >> 5) : -1;
}

// Sum over the 64 lanes of a wave (all lanes active), in every lane.
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  v = fold<32>(v, v);
  return read_lane(row_sum(fold<16>(v, v)), 0);
}

// Three such sums.
template <typename T>
__device__ __forceinline__ void wave_sum3(T &a, T &b, T &c) {
  const T v = wave_sums(a, b, c);
  a = read_lane(v, 0);
  b = read_lane(v, 16);
  c = read_lane(v, 32);
}

// Sum over each aligned group of 4 lanes; all 4 lanes get the same bits.
template <typename T>
__device__ __forceinline__ T quad_sum(T v) {
  v += dpp<kDppQuadXor2>(v);
  v += dpp<kDppQuadXor1>(v);
  return v;
}

}  // namespace gbdpcg
