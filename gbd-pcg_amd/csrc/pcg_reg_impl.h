// Register-resident PCG kernels for gfx950: the latency path (templates,
// instantiated in pcg_reg_kernel.hip (fused recurrence, column chunks),
// pcg_reg_ref_kernel.hip (reference recurrence), pcg_rowcast_kernel.hip (row
// broadcast), pcg_pair_kernel_f32/_f64.hip (forward + adjoint together) and
// pcg_any_*.hip (any stateSize up to 32, systems of one workgroup)).
//
// Same method and exchange protocol as pcg_kernel.hip, with every block row a
// workgroup owns held in registers instead of LDS.  FUSED: the single-reduction
// (Chronopoulos-Gear) form, described below; reference form
// (include/pcg.cuh:118-208): two exchanges per iteration, the first carrying
// p'v and the edge knots of v = S p, the second r'z and r'r only (z = Pinv r is
// formed on one ghost knot each side from the resident ghost rows of Pinv, so
// p needs no halo).  Fused form:
//   * LPR lanes (reg_lpr: 2 for most sizes, 1 for n <= 2 and for the n = 28
//     layouts that hold whole rows) share one matrix row; each lane keeps a
//     CW-column chunk of that row of Pinv (rows of the owned knots plus one
//     ghost knot each side) and of S (owned knots) in VGPRs for the whole
//     solve, loaded from HBM once.  Row-broadcast layout (BC): one lane per row,
//     16 lanes per knot, whole rows, the vector window broadcast by DPP;
//   * per iteration: one pass u = Pinv r (owned + ghost rows), one pass w = S u
//     (owned rows), then one cross-workgroup exchange carrying (r'u, w'u, r'r)
//     and the two edge knots of w each side;
//   * the lanes that produce an edge value publish it themselves, and the
//     wave that polls the scalars also reduces them (DPP), so an iteration has
//     four workgroup barriers and one exchange.
// LDS holds only ghost-extended vectors (a few KB), so several workgroups fit a
// CU when the batched path uses this kernel.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"
#include "internal.h"

namespace gbdpcg {

namespace {
// threadIdx.x through an empty asm: index arithmetic derived from it is then
// recomputed where it is used instead of being hoisted to the kernel entry and
// kept live (in VGPRs) across the whole solve.
__device__ __forceinline__ int opaque_tid() {
  int t = (int)threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

struct RegOut {
  int iters, status;
  double eta, rr;
};

// Sum over the waves of a workgroup of partial l (stride S per wave), as a
// pairwise tree in a fixed order: three dependent adds for eight waves instead
// of seven.
template <int NW, int S, typename T>
__device__ __forceinline__ T waves_total(const T *wsum, int l) {
  if constexpr (NW == 1) {
    return wsum[l];
  } else {
    return waves_total<NW / 2, S>(wsum, l) + waves_total<NW - NW / 2, S>(wsum + (NW / 2) * S, l);
  }
}

// stateSize of an item: a constant (RT false), or read from the system.
template <int NS, bool RT>
struct StateSize {
  static constexpr int n = NS;
  __device__ __forceinline__ void set_n(int) {}
};
template <int NS>
struct StateSize<NS, true> {
  int n;
  __device__ __forceinline__ void set_n(int v) { n = v; }
};

// Status of one exchange within the item (all threads agree after a gather).
// BC: row-broadcast layout (one lane per matrix row, 16 lanes per knot, every
// lane holding its whole row of 3n columns).
// LP > 0: any stateSize n <= NS with padded_n(n) == NS (a multiple of 4), LP
// lanes per row.  Vectors and chunks have the compile-time stride NS, so the
// matvecs are those of a fixed size; lanes, records and HBM offsets follow n.
// ALONE: the system's only rank, with no ghost rows and no exchange.
template <typename T, int NS, int NT, bool BC = false, int LP = 0, bool ALONE = false>
struct RegItem : StateSize<NS, (LP > 0)> {
  static constexpr bool RT = LP > 0;
  using StateSize<NS, RT>::n;
  static constexpr int nP = (int)padded_n(NS);
  static_assert(!RT || (nP == NS && !BC), "runtime stateSizes: column chunks, NS a multiple of 4");
  static constexpr int LPR = BC ? 1 : RT ? LP : (int)reg_lpr(NS, NT, (int)sizeof(T));  // lanes per matrix row
  static constexpr int CW = BC ? 3 * NS : (int)reg_chunk(NS, LPR);           // columns per lane
  static constexpr int WPV = (int)(sizeof(T) / 4);
  static constexpr int NWAVES = NT / 64;
  // Tiled rows (tile_dot): TL lanes share two rows, each with TW columns of every
  // block of both; MW values per lane and matrix.
  static constexpr bool TILED = !BC && !RT && NS == 28 && NT == 256;
  static constexpr int TL = 2 * LPR, TW = TILED ? NS / TL : 1;
  static constexpr int MW = TILED ? 6 * TW : CW;

  // geometry
  int N, G, rank, a, b, K, VL;
  uint64_t *slots;
  uint32_t base, seq;
  double tol;
  bool rel;
  bool xcd;     // every rank on this workgroup's XCD: exchange stores stay in L2
  bool xcd_ok;  // the system allows XCD-local stores (KF_NOXCD clear)
  // lane roles
  int q, c, m, row, kg;
  int i;  // tiled rows: number of the lane in its group
  bool act_u, act_w, owner, ghost;
  int gpos;
  // LDS
  T *rv, *uv, *wv, *xv, *lv, *wsum, *tot;
  T only[3];  // ALONE on one wave: its sums
  int *ctl;

  __device__ __forceinline__ uint64_t *rec(int type, int g) const {
    return slots + (size_t)(type * G + g) * rec_words((uint32_t)n, WPV);
  }

  // Owner lanes publish their value into the edge slots of the current exchange
  // (value kRecScalars + e*n + row for own knot a+e, kRecScalars + 2n + e*n + row
  // for own knot b-1-e).  A lane has at most two such slots (K >= 2), slot_lo for
  // its left-edge role and slot_hi for its right-edge one, each -1 when absent and
  // tagged with its depth e in bit 16 (edge = 1 publishes depth 0 only).
  int slot_lo, slot_hi;

  __device__ __forceinline__ void set_edge_slots() {
    const int kl = m - 1;
    slot_lo = -1;
    slot_hi = -1;
    if (!owner) return;
    if (kl < 2) slot_lo = (kRecScalars + kl * n + row) | (kl << 16);
    const int e = K - 1 - kl;
    if (e < 2) slot_hi = (kRecScalars + 2 * n + e * n + row) | (e << 16);
  }

  // voff: 0 for the first edge block of a record, 4n for the second (paired
  // solves publish the edges of two vectors per exchange).
  template <bool XCD>
  __device__ __forceinline__ void store_edges(uint64_t *r, T val, int edge, uint32_t epoch, int voff) const {
    const int lim = edge << 16;
    if (slot_lo >= 0 && slot_lo < lim) {
#pragma unroll
      for (int qq = 0; qq < WPV; ++qq) {
        uint64_t *p = r + ((slot_lo & 0xFFFF) + voff) * WPV + qq;
        if constexpr (XCD) xstore_xcd(p, payload_word(val, qq), epoch); else xstore(p, payload_word(val, qq), epoch);
      }
    }
    if (slot_hi >= 0 && slot_hi < lim) {
#pragma unroll
      for (int qq = 0; qq < WPV; ++qq) {
        uint64_t *p = r + ((slot_hi & 0xFFFF) + voff) * WPV + qq;
        if constexpr (XCD) xstore_xcd(p, payload_word(val, qq), epoch); else xstore(p, payload_word(val, qq), epoch);
      }
    }
  }

  __device__ __forceinline__ void publish_edge(T val, int edge, int voff = 0) const {
    if (ALONE || G == 1) return;
    const uint32_t epoch = base + seq;
    uint64_t *r = rec((int)(seq & 1u), rank);
    if (xcd)
      store_edges<true>(r, val, edge, epoch, voff);
    else
      store_edges<false>(r, val, edge, epoch, voff);
  }

  // Workgroup totals of three per-lane partials (DPP per wave, then the waves in
  // order by thread 0), published as this rank's three scalars; with one
  // workgroup they go straight to tot.  One barrier.  With `placement`, the
  // second and third scalars are replaced by x and x^2, x = 1 + this XCD's id,
  // so that after the gather every rank can tell (identically) whether all ranks
  // share one XCD: G * sum(x^2) == sum(x)^2 exactly when all x are equal.
  // ALONE: the waves' sums only, which only_totals adds up.
  __device__ __forceinline__ void reduce_publish(T s0, T s1, T s2, bool placement = false) {
    const T sums = wave_sums(s0, s1, s2);
    if constexpr (ALONE && NWAVES == 1) {
      only[0] = read_lane(sums, 0);
      only[1] = read_lane(sums, 16);
      only[2] = read_lane(sums, 32);
      return;
    }
    const int slot = wave_sums_slot<3>();
    if (slot >= 0) wsum[(threadIdx.x >> 6) * 3 + slot] = sums;
    if constexpr (ALONE) return;
    __syncthreads();
    // lanes 0..2 of wave 0: scalar l summed over the waves in order, published
    const int l = threadIdx.x;
    if (l >= 3) return;
    T tv = waves_total<NWAVES, 3>(wsum, l);
    if (G == 1) {
      tot[l] = tv;
      return;
    }
    if (placement && l > 0) {
      const T x = (T)(1 + xcc_id());
      tv = l == 1 ? x : x * x;
    }
    const uint32_t epoch = base + seq;
    uint64_t *r = rec((int)(seq & 1u), rank);
#pragma unroll
    for (int qq = 0; qq < WPV; ++qq) xstore_sel(r + l * WPV + qq, payload_word(tv, qq), epoch, xcd);
  }

  // ALONE: every wave adds up the waves' sums itself, in waves_total's order: one
  // LDS round trip and one barrier (through wave 0 and tot, a second of each).
  // Waves that were not launched left theirs zero.
  // The next reduction writes the same sums: settle() stands between the two
  // where the solve has no barrier of its own.
  __device__ __forceinline__ void settle() const {
    if constexpr (ALONE) __syncthreads();
  }
  __device__ __forceinline__ void only_totals(T &t0, T &t1, T &t2) const {
    __syncthreads();
    if constexpr (NWAVES == 1) {
      t0 = only[0];
      t1 = only[1];
      t2 = only[2];
    } else {
      const int l = (int)threadIdx.x & 3;
      const T v = waves_total<NWAVES, 3>(wsum, l < 3 ? l : 0);
      t0 = read_lane(v, 0);
      t1 = read_lane(v, 1);
      t2 = read_lane(v, 2);
    }
  }

  static __device__ __forceinline__ T word_value(const uint32_t *w, int v) {
    if constexpr (WPV == 1) {
      return __uint_as_float(w[v]);
    } else {
      return __longlong_as_double((long long)(((uint64_t)w[2 * v + 1] << 32) | w[2 * v]));
    }
  }

  // Source word and LDS destination of edge entry i (payload word i of the
  // neighbours' edge knots, left neighbour's first) of edge block voff.
  __device__ __forceinline__ void edge_slot(int i, int nleft, int type, int voff, T *vec, uint64_t *&src,
                                            uint32_t *&dst) const {
    if (i < nleft) {  // left neighbour's right edge: knot a-1-e = local 1-e
      const int vi = i / WPV, qq = i - vi * WPV;
      const int e = vi >= n ? 1 : 0, rr = vi - e * n;
      src = rec(type, rank - 1) + (kRecScalars + voff + 2 * n + e * n + rr) * WPV + qq;
      dst = reinterpret_cast<uint32_t *>(vec + (1 - e) * nP + rr) + qq;
    } else {  // right neighbour's left edge: knot b+e = local K+2+e
      const int ii = i - nleft;
      const int vi = ii / WPV, qq = ii - vi * WPV;
      const int e = vi >= n ? 1 : 0, rr = vi - e * n;
      src = rec(type, rank + 1) + (kRecScalars + voff + e * n + rr) * WPV + qq;
      dst = reinterpret_cast<uint32_t *>(vec + (K + 2 + e) * nP + rr) + qq;
    }
  }

  // One-wave workgroups: lane t polls rank t's three totals and edge entries t
  // and t + 64 in one spin loop (one round trip when everything has landed);
  // ranks beyond 64 are polled afterwards.  Sums as the multi-wave gather does.
  __device__ __forceinline__ bool gather_one_wave(T *vec, int edge, uint32_t epoch, int type, int t) {
    constexpr int NW = 3 * WPV;
    const int en = edge * n * WPV;
    const int nleft = rank > 0 ? en : 0;
    const int ne = nleft + (rank < G - 1 ? en : 0);  // <= 4 * 16 * 2 = 128
    uint64_t *src0 = nullptr, *src1 = nullptr;
    uint32_t *dst0 = nullptr, *dst1 = nullptr;
    if (t < ne) edge_slot(t, nleft, type, 0, vec, src0, dst0);
    if (t + 64 < ne) edge_slot(t + 64, nleft, type, 0, vec, src1, dst1);
    bool need_s = t < G, need0 = src0 != nullptr, need1 = src1 != nullptr;
    uint32_t wv_[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) wv_[i] = 0;
    uint32_t v0 = 0, v1 = 0;
    for (uint32_t spin = 0; spin < kSpinLimit && (need_s || need0 || need1); ++spin) {
      if (need_s) {
        uint64_t A[NW];
        uint64_t *p = rec(type, t);
#pragma unroll
        for (int i = 0; i < NW; ++i) A[i] = xload(p + i);
        bool all = true;
#pragma unroll
        for (int i = 0; i < NW; ++i) all = all && (uint32_t)(A[i] >> 32) == epoch;
        if (all) {
#pragma unroll
          for (int i = 0; i < NW; ++i) wv_[i] = (uint32_t)A[i];
          need_s = false;
        }
      }
      if (need0) {
        const uint64_t w = xload(src0);
        if ((uint32_t)(w >> 32) == epoch) {
          v0 = (uint32_t)w;
          need0 = false;
        }
      }
      if (need1) {
        const uint64_t w = xload(src1);
        if ((uint32_t)(w >> 32) == epoch) {
          v1 = (uint32_t)w;
          need1 = false;
        }
      }
    }
    bool ok = !(need_s || need0 || need1);
    if (src0 && !need0) *dst0 = v0;
    if (src1 && !need1) *dst1 = v1;
    T acc0 = 0, acc1 = 0, acc2 = 0;
    if (t < G && !need_s) {
      acc0 = word_value(wv_, 0);
      acc1 = word_value(wv_, 1);
      acc2 = word_value(wv_, 2);
    }
    for (int g = t + 64; g < G; g += 64) {
      uint32_t w2[NW];
      if (!xwait_words<NW>(rec(type, g), epoch, w2)) {
        ok = false;
        break;
      }
      acc0 += word_value(w2, 0);
      acc1 += word_value(w2, 1);
      acc2 += word_value(w2, 2);
    }
    const T sums = wave_sums(acc0, acc1, acc2);
    const int slot = wave_sums_slot<3>();
    if (slot >= 0) tot[slot] = sums;
    return ok;
  }

  // Polls the current exchange.  Wave 0 gathers every rank's wave totals and
  // reduces them (waves in order, then ranks by a fixed DPP tree) into tot; the
  // other waves copy the neighbours' `edge` edge knots into the ghost knots of
  // `vec` (one-wave workgroups: gather_one_wave).  Ends with a barrier after
  // which t0..t2 hold the totals in every thread; returns false (uniformly) if
  // a wait hit its bound.
  __device__ __forceinline__ bool gather(T *vec, int edge, T &t0, T &t1, T &t2) {
    if constexpr (ALONE) {
      only_totals(t0, t1, t2);
      return true;
    }
    if (G == 1) {
      __syncthreads();
      t0 = uniform(tot[0]);
      t1 = uniform(tot[1]);
      t2 = uniform(tot[2]);
      ++seq;
      return true;
    }
    const uint32_t epoch = base + seq;
    const int type = (int)(seq & 1u);
    bool ok = true;
    const int t = opaque_tid();
    if constexpr (NT == 64) {
      ok = gather_one_wave(vec, edge, epoch, type, t);
    } else if (t < 64) {
      constexpr int NW = 3 * WPV;
      T acc0 = 0, acc1 = 0, acc2 = 0;
      for (int g = t; g < G; g += 64) {
        uint32_t wv_[NW];
        if (!xwait_words<NW>(rec(type, g), epoch, wv_)) {
          ok = false;
          break;
        }
        acc0 += word_value(wv_, 0);
        acc1 += word_value(wv_, 1);
        acc2 += word_value(wv_, 2);
      }
      const T sums = wave_sums(acc0, acc1, acc2);
      const int slot = wave_sums_slot<3>();
      if (slot >= 0) tot[slot] = sums;
    } else {
      const int en = edge * n * WPV;
      const int nleft = rank > 0 ? en : 0;
      const int nright = rank < G - 1 ? en : 0;
      for (int i = t - 64; i < nleft + nright; i += NT - 64) {
        uint64_t *src;
        uint32_t *dst;
        edge_slot(i, nleft, type, 0, vec, src, dst);
        uint32_t val = 0;
        if (xcd ? xwait(src, epoch, val) : xwait_lazy(src, epoch, val)) {
          *dst = val;
        } else {
          ok = false;
          break;
        }
      }
    }
    if (!ok) ctl[0] = 1;
    __syncthreads();
    ++seq;
    t0 = uniform(tot[0]);
    t1 = uniform(tot[1]);
    t2 = uniform(tot[2]);
    return __builtin_amdgcn_readfirstlane(ctl[0]) == 0;
  }

  // Paired solves: six workgroup totals (the first three for vector A, the last
  // three for B; each scalar reduced exactly as reduce_publish reduces it),
  // wsum holding 6 per wave.  Lanes 0..5 publish.  placement as in
  // reduce_publish, for scalars 1 and 2.
  __device__ __forceinline__ void reduce_publish6(T s0, T s1, T s2, T s3, T s4, T s5, bool placement = false) {
    const T sums = wave_sums(s0, s1, s2, s3, s4, s5);
    const int slot = wave_sums_slot<6>();
    if (slot >= 0) wsum[(threadIdx.x >> 6) * 6 + slot] = sums;
    publish6(placement);
  }
  // The same with side A's partials on even lanes and side B's on odd ones.
  __device__ __forceinline__ void reduce_publish_sides(T s0, T s1, T s2, bool placement = false) {
    const T sums = wave_sums_parity(s0, s1, s2);
    const int l = (int)threadIdx.x & 63;
    if ((l & 15) < 2 && l < 48) wsum[(threadIdx.x >> 6) * 6 + (l & 1) * 3 + (l >> 4)] = sums;
    publish6(placement);
  }
  __device__ __forceinline__ void publish6(bool placement) {
    __syncthreads();
    const int l = threadIdx.x;
    if (l >= 6) return;
    T tv = waves_total<NWAVES, 6>(wsum, l);
    if (G == 1) {
      tot[l] = tv;
      return;
    }
    if (placement && (l == 1 || l == 2)) {
      const T x = (T)(1 + xcc_id());
      tv = l == 1 ? x : x * x;
    }
    const uint32_t epoch = base + seq;
    uint64_t *r = rec((int)(seq & 1u), rank);
#pragma unroll
    for (int qq = 0; qq < WPV; ++qq) xstore_sel(r + l * WPV + qq, payload_word(tv, qq), epoch, xcd);
  }

  // gather for paired solves: six totals, and the neighbours' `edge` edge knots
  // of vA (first edge block) and vB (second) into their ghost knots.
  __device__ __forceinline__ bool gather_pair(T *vA, T *vB, int edge, T (&tt)[6]) {
    const bool ok = gather6(vA, vB, edge);
#pragma unroll
    for (int l = 0; l < 6; ++l) tt[l] = uniform(tot[l]);
    return ok;
  }
  // The same, each lane taking its side's three totals.
  __device__ __forceinline__ bool gather_sides(T *vA, T *vB, int edge, int side, T (&tt)[3]) {
    const bool ok = gather6(vA, vB, edge);
#pragma unroll
    for (int l = 0; l < 3; ++l) tt[l] = tot[side * 3 + l];
    return ok;
  }
  __device__ __forceinline__ bool gather6(T *vA, T *vB, int edge) {
    if (G == 1) {
      __syncthreads();
      ++seq;
      return true;
    }
    const uint32_t epoch = base + seq;
    const int type = (int)(seq & 1u);
    bool ok = true;
    const int t = opaque_tid();
    if (t < 64) {
      constexpr int NW = 6 * WPV;
      T acc[6] = {0, 0, 0, 0, 0, 0};
      for (int g = t; g < G; g += 64) {
        uint32_t wv_[NW];
        if (!xwait_words<NW>(rec(type, g), epoch, wv_)) {
          ok = false;
          break;
        }
#pragma unroll
        for (int l = 0; l < 6; ++l) acc[l] += word_value(wv_, l);
      }
      const T sums = wave_sums(acc[0], acc[1], acc[2], acc[3], acc[4], acc[5]);
      const int slot = wave_sums_slot<6>();
      if (slot >= 0) tot[slot] = sums;
    } else {
      const int en = edge * n * WPV;
      const int nleft = rank > 0 ? en : 0;
      const int nright = rank < G - 1 ? en : 0;
      const int per = nleft + nright;
      for (int i = t - 64; i < 2 * per; i += NT - 64) {
        const int v = i >= per ? 1 : 0;
        const int iv = i - v * per;
        uint64_t *src;
        uint32_t *dst;
        edge_slot(iv, nleft, type, v * 4 * n, v ? vB : vA, src, dst);
        uint32_t val = 0;
        if (xcd ? xwait(src, epoch, val) : xwait_lazy(src, epoch, val)) {
          *dst = val;
        } else {
          ok = false;
          break;
        }
      }
    }
    if (!ok) ctl[0] = 1;
    __syncthreads();
    ++seq;
    return __builtin_amdgcn_readfirstlane(ctl[0]) == 0;
  }
};

// Four accumulator chains (the FMA latency, not the issue rate, bounds a short
// dot product), summed in a fixed order.
template <typename T, int CW>
__device__ __forceinline__ T chunk_dot(const T (&mat)[CW], const T *__restrict__ x) {
  T a0 = 0, a1 = 0, a2 = 0, a3 = 0;
#pragma unroll
  for (int j = 0; j < CW; j += 4) {
    if constexpr (sizeof(T) == 4) {
      const float4 xv = *reinterpret_cast<const float4 *>(x + j);
      a0 = __builtin_fmaf(mat[j + 0], xv.x, a0);
      a1 = __builtin_fmaf(mat[j + 1], xv.y, a1);
      a2 = __builtin_fmaf(mat[j + 2], xv.z, a2);
      a3 = __builtin_fmaf(mat[j + 3], xv.w, a3);
    } else {
      const double2 x0 = *reinterpret_cast<const double2 *>(x + j);
      const double2 x1 = *reinterpret_cast<const double2 *>(x + j + 2);
      a0 = fmaT(mat[j + 0], x0.x, a0);
      a1 = fmaT(mat[j + 1], x0.y, a1);
      a2 = fmaT(mat[j + 2], x1.x, a2);
      a3 = fmaT(mat[j + 3], x1.y, a3);
    }
  }
  return (a0 + a1) + (a2 + a3);
}

// The paired kernels' FP32 instances held to 128 VGPRs keep their Pinv chunks in
// LDS rather than in registers (see pair_pinv_lds): float4 block b of lane t's
// chunk sits at float4 index b * NT + t, so a wave's 16-byte reads of one block
// are contiguous and conflict-free.  Two dot products (the two sides of a
// paired solve) share each matrix read; each side's four accumulator chains
// follow chunk_dot's order, so the bits are those of chunk_dot.
template <int CW, int NT>
__device__ __forceinline__ void chunk_dot2_lds(const float *__restrict__ plds, int tid, const float *__restrict__ xa,
                                               const float *__restrict__ xb, float &ya, float &yb) {
  float a0 = 0, a1 = 0, a2 = 0, a3 = 0, b0 = 0, b1 = 0, b2 = 0, b3 = 0;
#pragma unroll
  for (int j = 0; j < CW; j += 4) {
    const float4 mv = *reinterpret_cast<const float4 *>(plds + ((size_t)(j / 4) * NT + tid) * 4);
    const float4 u = *reinterpret_cast<const float4 *>(xa + j);
    const float4 v = *reinterpret_cast<const float4 *>(xb + j);
    a0 = __builtin_fmaf(mv.x, u.x, a0);
    a1 = __builtin_fmaf(mv.y, u.y, a1);
    a2 = __builtin_fmaf(mv.z, u.z, a2);
    a3 = __builtin_fmaf(mv.w, u.w, a3);
    b0 = __builtin_fmaf(mv.x, v.x, b0);
    b1 = __builtin_fmaf(mv.y, v.y, b1);
    b2 = __builtin_fmaf(mv.z, v.z, b2);
    b3 = __builtin_fmaf(mv.w, v.w, b3);
  }
  ya = (a0 + a1) + (a2 + a3);
  yb = (b0 + b1) + (b2 + b3);
}

// Sum over the LPR lanes sharing one matrix row; all of them get the same bits.
template <int LPR, typename T>
__device__ __forceinline__ T group_sum(T v) {
  if constexpr (LPR == 2) {
    v += dpp<kDppQuadXor1>(v);
  } else if constexpr (LPR == 4) {
    v = quad_sum(v);
  }
  return v;
}

// Element at a uniform element offset from A plus a per-lane one (32-bit byte
// offsets against a scalar base: one scalar addition and one load).
template <typename V, typename T>
__device__ __forceinline__ V load_at(const T *A, uint32_t uniform_off, uint32_t lane_off) {
  const auto *col = reinterpret_cast<const __attribute__((address_space(1))) unsigned char *>(gptr(A + uniform_off));
  return *reinterpret_cast<const __attribute__((address_space(1))) V *>(col + lane_off * (uint32_t)sizeof(T));
}

// Lane offsets of the three blocks of block row kg at `row` (a lane without the
// block is sent to the diagonal block of its own or of the first knot, so that
// every load is in bounds and none reads the padding) and whether each is absent.
struct BlockRow {
  uint32_t off[3];
  bool absent[3];
};
__device__ __forceinline__ BlockRow block_row(int kg, int row, int N, bool active, int n) {
  BlockRow b;
  const uint32_t nn = (uint32_t)(n * n);
  const bool ok = active && kg >= 0 && kg < N;
  b.absent[0] = !(ok && kg > 0);
  b.absent[1] = !ok;
  b.absent[2] = !(ok && kg < N - 1);
  b.off[1] = ok ? (uint32_t)kg * 3u * nn + nn + (uint32_t)row : nn;
  b.off[0] = b.absent[0] ? b.off[1] : b.off[1] - nn;
  b.off[2] = b.absent[2] ? b.off[1] : b.off[1] + nn;
  return b;
}

// Chunk c1 (0 or 1) of CW columns of a padded row (NS columns per block, stateSize
// n <= NS, NS - n < 4, a constant or known at run time only).  Few instructions per element matter: the set-up is
// straight-line code that runs once, at the rate at which it is fetched.  Set-up
// (max_iter = 0) with one lane per row, against a select of offset and value per
// element: FP32 n = 32 N = 16 8.9 us (16.9), n = 20 N = 20 7.2 (10.4), FP64 n = 13 N = 16
// 7.3 (9.0).  The two chunks of a row differ by a lane offset that depends on the
// pair of blocks they are in, of which a row has few (n = 24 N = 100 13.3, 14.6);
// columns that may be padding are tested in scalar code.
template <typename T, int NS, int CW>
__device__ __forceinline__ void load_chunk(T (&dst)[CW], const T *__restrict__ A, int kg, int row, bool c1, int N,
                                               bool active, int n) {
  static_assert(3 * NS <= 2 * CW, "at most two chunks per row");
  // opaque copy: keeps the lane offsets below from being hoisted out of the batched
  // item loop (they would stay live, in registers, for the whole solve)
  asm volatile("" : "+v"(row));
  const BlockRow b = block_row(kg, row, N, active, n);
#pragma unroll
  for (int j = 0; j < CW; ++j) {
    const int s0 = j / NS, k0 = j % NS;
    if constexpr (CW >= 3 * NS) {  // one lane per row
      if (s0 > 2) {
        dst[j] = (T)0;
        continue;
      }
      T v = 0;
      if (k0 < NS - 3 || k0 < n) v = load_at<T>(A, (uint32_t)(k0 * n), b.off[s0]);
      dst[j] = b.absent[s0] ? (T)0 : v;
    } else {
      const int s1 = (CW + j) / NS, k1 = (CW + j) % NS;
      const bool sure = k0 < NS - 3 && k1 < NS - 3 && s1 < 3;
      if (sure) {
        const int d = k1 - k0;  // the same for every column of the pair of blocks
        const uint32_t lane = d >= 0 ? (c1 ? b.off[s1] + (uint32_t)(d * n) : b.off[s0])
                                     : (c1 ? b.off[s1] : b.off[s0] + (uint32_t)(-d * n));
        const T v = load_at<T>(A, (uint32_t)((d >= 0 ? k0 : k1) * n), lane);
        dst[j] = (c1 ? b.absent[s1] : b.absent[s0]) ? (T)0 : v;
      } else {
        const bool v0 = k0 < n, v1 = s1 < 3 && k1 < n;  // uniform
        T v = 0;
        bool no = true;
        if (v0 || v1) {
          const int t1 = s1 < 3 ? s1 : 2;
          const uint32_t lane = c1 ? (v1 ? b.off[t1] + (uint32_t)(k1 * n) : b.off[1])
                                   : (v0 ? b.off[s0] + (uint32_t)(k0 * n) : b.off[1]);
          v = load_at<T>(A, 0u, lane);
          no = c1 ? (!v1 || b.absent[t1]) : (!v0 || b.absent[s0]);
        }
        dst[j] = no ? (T)0 : v;
      }
    }
  }
}

// Rows `row` and `row` + 1 (when second) of block row kg, whole: adjacent in the
// column-major blocks, so one 8-byte load serves both (4-byte aligned when n is
// odd).  A lane with one row takes it from the upper half of the pair before it.
// Set-up of n = 14 N = 64 11.4 us, of n = 8 N = 100 6.7 (row by row, with selects: 21.5
// and 20.7).
template <int NS>
__device__ __forceinline__ void load_two_rows(float (&a)[3 * NS], float (&b)[3 * NS], const float *__restrict__ A,
                                              int kg, int row, int N, bool active, bool second, int n) {
  typedef float pair_t __attribute__((ext_vector_type(2), aligned(4)));
  const bool last = active && !second;
  const BlockRow r = block_row(kg, last ? row - 1 : row, N, active, n);
#pragma unroll
  for (int j = 0; j < 3 * NS; ++j) {
    const int s = j / NS, k = j % NS;
    pair_t v = {0.f, 0.f};
    if (k < NS - 3 || k < n) v = load_at<pair_t>(A, (uint32_t)(k * n), r.off[s]);
    a[j] = r.absent[s] ? 0.f : last ? v.y : v.x;
    b[j] = (r.absent[s] || last) ? 0.f : v.y;
  }
}

// The same in guarded loads, for the n = 28 instances of 512 threads, whose registers
// leave no room for the masks and offsets above (their batches reload every item's
// matrices: FP64 forward + adjoint of 32 systems of N = 512, no iterations, 405 us
// against 426).  One lane per row: the guards are uniform over each block.
template <typename T, int NS, int CW>
__device__ __forceinline__ void load_guarded(T (&dst)[CW], const T *__restrict__ A, int kg, int row, int c, int N,
                                             bool active) {
  constexpr int n = NS, nP = (int)padded_n(NS);
  int cl = c, rl = row;
  asm volatile("" : "+v"(cl), "+v"(rl));
  if constexpr (CW == 3 * nP) {
    const bool rowok = active && kg >= 0 && kg < N;
#pragma unroll
    for (int s3 = 0; s3 < 3; ++s3) {
      if (rowok && !(kg == 0 && s3 == 0) && !(kg == N - 1 && s3 == 2)) {
#pragma unroll
        for (int cc = 0; cc < nP; ++cc)
          dst[s3 * nP + cc] = cc < n ? gptr(A)[(size_t)kg * 3 * n * n + (size_t)(s3 * n + cc) * n + rl] : (T)0;
      } else {
#pragma unroll
        for (int cc = 0; cc < nP; ++cc) dst[s3 * nP + cc] = (T)0;
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < CW; ++j) {
      const int col = cl * CW + j;
      const int seg = col / nP, cc = col - seg * nP;
      T v = 0;
      if (active && kg >= 0 && kg < N && seg < 3 && cc < n && !(kg == 0 && seg == 0) && !(kg == N - 1 && seg == 2))
        v = gptr(A)[(size_t)kg * 3 * n * n + (size_t)(seg * n + cc) * n + rl];
      dst[j] = v;
    }
  }
}

// A fixed size's chunk of either kind.
template <typename T, int NS, int NT, int CW>
__device__ __forceinline__ void load_fixed(T (&dst)[CW], const T *__restrict__ A, int kg, int row, int c, int N,
                                           bool active) {
  if constexpr (NS == 28 && NT == 512)
    load_guarded<T, NS, CW>(dst, A, kg, row, c, N, active);
  else
    load_chunk<T, (int)padded_n(NS), CW>(dst, A, kg, row, c != 0, N, active, NS);
}

// Tiled rows.  A vector window read from LDS costs as many cycles as the bytes it
// hands to the lanes, broadcast or not, and two matrix rows of a knot want the same
// window: so the TL lanes that hold two rows (LPR each) do not take a row's columns
// each, but TW columns of every block of both rows, and each reads half the window
// that its own row would need.  Two partial sums per lane are then added up across
// the lanes by DPP, one row to each half of the group.  Value (s TW + j) 2 + r of a
// lane is row r, column j of its columns in block s.  For n = 28 at 256 threads (single
// solves), per iteration: FP64 N = 100 3.45 -> 2.79 us, FP32 N = 64 1.73 -> 1.61; n = 6 to
// 14 and the instances of 512 threads, which VALU issue bounds, gain nothing by it.

// Columns j of this lane (number i of its group), block s, of rows r0 and r0 + 1 of
// block row kg: adjacent in the column-major blocks, so one load serves both rows
// (aligned to T only).  Branch-free as load_chunk: a scalar offset per column, a
// lane offset per block.
template <typename T, int NS, int TL, int TW>
__device__ __forceinline__ void load_tile(T (&dst)[6 * TW], const T *__restrict__ A, int kg, int r0, int i, int N,
                                          bool active) {
  typedef T pair_t __attribute__((ext_vector_type(2), aligned(sizeof(T))));
  constexpr int n = NS;
  static_assert(n % TL == 0 && TW == n / TL, "tiles without padded columns");
  int il = i;
  asm volatile("" : "+v"(il));
  const BlockRow b = block_row(kg, r0, N, active, n);
  const uint32_t col0 = (uint32_t)(il * TW * n);
#pragma unroll
  for (int s = 0; s < 3; ++s) {
#pragma unroll
    for (int j = 0; j < TW; ++j) {
      const pair_t v = load_at<pair_t>(A, (uint32_t)(j * n), b.off[s] + col0);
      dst[(s * TW + j) * 2] = b.absent[s] ? (T)0 : v.x;
      dst[(s * TW + j) * 2 + 1] = b.absent[s] ? (T)0 : v.y;
    }
  }
}

// TW consecutive vector entries from LDS, in the widest reads their alignment
// (a multiple of TW values from a 16-byte boundary) allows.
template <typename T, int TW>
__device__ __forceinline__ void read_window(const T *__restrict__ x, T (&o)[TW]) {
  constexpr int V = (TW * (int)sizeof(T)) % 16 == 0 ? 16 / (int)sizeof(T) : (TW * (int)sizeof(T)) % 8 == 0 ? 8 / (int)sizeof(T) : 1;
  typedef T vec_t __attribute__((ext_vector_type(V)));
#pragma unroll
  for (int j = 0; j < TW; j += V) {
    const vec_t v = *reinterpret_cast<const vec_t *>(x + j);
#pragma unroll
    for (int k = 0; k < V; ++k) o[j + k] = v[k];
  }
}

// A lane's partial sums of its two rows over its columns of the window at x (the
// lane's first column; blocks nP apart): two accumulator chains per row.
template <typename T, int TW, int nP>
__device__ __forceinline__ void tile_dot(const T (&mat)[6 * TW], const T *__restrict__ x, T &ya, T &yb) {
  T a0 = 0, a1 = 0, b0 = 0, b1 = 0;
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    T xs[TW];
    read_window<T, TW>(x + s * nP, xs);
#pragma unroll
    for (int j = 0; j < TW; ++j) {
      const int e = s * TW + j;
      if (e % 2 == 0) {
        a0 = fmaT(mat[2 * e], xs[j], a0);
        b0 = fmaT(mat[2 * e + 1], xs[j], b0);
      } else {
        a1 = fmaT(mat[2 * e], xs[j], a1);
        b1 = fmaT(mat[2 * e + 1], xs[j], b1);
      }
    }
  }
  ya = a0 + a1;
  yb = b0 + b1;
}

// Adds a group's partial sums up: the lanes of its first half get row a's total, the
// others row b's, the same bits in every lane of a row.
template <int TL, typename T>
__device__ __forceinline__ T tile_sum(T ya, T yb, int i) {
  const bool upper = i >= TL / 2;
  const T keep = upper ? yb : ya, send = upper ? ya : yb;
  if constexpr (TL == 2) {
    return keep + dpp<kDppQuadXor1>(send);
  } else {
    const T v = keep + dpp<kDppQuadXor2>(send);
    return v + dpp<kDppQuadXor1>(v);
  }
}

// Row-broadcast layout: the whole row `row` of block row kg (3n values, block
// column s, column k at index s*n + k).
template <typename T, int NS, bool GUARDED = false>
__device__ __forceinline__ void load_row(T (&dst)[3 * NS], const T *__restrict__ A, int kg, int row, int N,
                                         bool active) {
  constexpr int n = NS;
  int rl = row;
  asm volatile("" : "+v"(rl));
  if constexpr (GUARDED) {
#pragma unroll
    for (int j = 0; j < 3 * n; ++j) {
      const int seg = j / n;
      T v = 0;
      if (active && kg >= 0 && kg < N && !(kg == 0 && seg == 0) && !(kg == N - 1 && seg == 2))
        v = gptr(A)[(size_t)kg * 3 * n * n + (size_t)j * n + rl];
      dst[j] = v;
    }
    return;
  }
  // branch-free, as load_chunk
  const BlockRow b = block_row(kg, rl, N, active, n);
#pragma unroll
  for (int j = 0; j < 3 * n; ++j) {
    const int s = j / n, k = j % n;
    const T v = load_at<T>(A, (uint32_t)(k * n), b.off[s]);
    dst[j] = b.absent[s] ? (T)0 : v;
  }
}

// a0/a1 += m[k] * (x of lane k of this lane's 16-lane row), k = 0..NS-1, on
// alternate accumulators.  DPP row_newbcast:k hands every lane of a row the
// value of its lane k, so one VALU op does one multiply-add with no LDS traffic.
// The compiler does not fold a broadcast into an accumulating FMA by itself,
// hence the asm; each block opens with s_nop 4, the 5 wait states a DPP read
// needs after a VALU write of EXEC (2 after a VALU write of its source VGPR).
#define GBDPCG_RC(OP, k, a, mi) OP " %" #a ", %2, %" #mi " row_newbcast:" #k " row_mask:0xf bank_mask:0xf\n\t"
#define GBDPCG_RC12(OP)                                                                                     \
  GBDPCG_RC(OP, 0, 0, 3) GBDPCG_RC(OP, 1, 1, 4) GBDPCG_RC(OP, 2, 0, 5) GBDPCG_RC(OP, 3, 1, 6)                \
  GBDPCG_RC(OP, 4, 0, 7) GBDPCG_RC(OP, 5, 1, 8) GBDPCG_RC(OP, 6, 0, 9) GBDPCG_RC(OP, 7, 1, 10)               \
  GBDPCG_RC(OP, 8, 0, 11) GBDPCG_RC(OP, 9, 1, 12) GBDPCG_RC(OP, 10, 0, 13) GBDPCG_RC(OP, 11, 1, 14)
#define GBDPCG_RC14(OP) GBDPCG_RC12(OP) GBDPCG_RC(OP, 12, 0, 15) GBDPCG_RC(OP, 13, 1, 16)
#define GBDPCG_M12(m) "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "v"(m[4]), "v"(m[5]), "v"(m[6]), \
    "v"(m[7]), "v"(m[8]), "v"(m[9]), "v"(m[10]), "v"(m[11])
#define GBDPCG_M14(m) GBDPCG_M12(m), "v"(m[12]), "v"(m[13])

template <typename T, int NS>
struct RowCast;
template <>
struct RowCast<float, 14> {
  static __device__ __forceinline__ void fma(float &a0, float &a1, float x, const float *m) {
    asm("s_nop 4\n\t" GBDPCG_RC14("v_fmac_f32_dpp") : "+v"(a0), "+v"(a1) : "v"(x), GBDPCG_M14(m));
  }
};
template <>
struct RowCast<float, 12> {
  static __device__ __forceinline__ void fma(float &a0, float &a1, float x, const float *m) {
    asm("s_nop 4\n\t" GBDPCG_RC12("v_fmac_f32_dpp") : "+v"(a0), "+v"(a1) : "v"(x), GBDPCG_M12(m));
  }
};
template <>
struct RowCast<double, 14> {
  static __device__ __forceinline__ void fma(double &a0, double &a1, double x, const double *m) {
    asm("s_nop 4\n\t" GBDPCG_RC14("v_fmac_f64_dpp") : "+v"(a0), "+v"(a1) : "v"(x), GBDPCG_M14(m));
  }
};
template <>
struct RowCast<double, 12> {
  static __device__ __forceinline__ void fma(double &a0, double &a1, double x, const double *m) {
    asm("s_nop 4\n\t" GBDPCG_RC12("v_fmac_f64_dpp") : "+v"(a0), "+v"(a1) : "v"(x), GBDPCG_M12(m));
  }
};
#undef GBDPCG_RC
#undef GBDPCG_RC12
#undef GBDPCG_RC14
#undef GBDPCG_M12
#undef GBDPCG_M14

// y = row . (xa | xb | xc), x* the lane's entries of three consecutive knots;
// four accumulator chains summed in a fixed order.
template <typename T, int NS>
__device__ __forceinline__ T rowcast_dot(const T (&mat)[3 * NS], T xa, T xb, T xc) {
  T a0 = 0, a1 = 0, a2 = 0, a3 = 0;
  RowCast<T, NS>::fma(a0, a1, xa, mat);
  RowCast<T, NS>::fma(a2, a3, xb, mat + NS);
  RowCast<T, NS>::fma(a0, a1, xc, mat + 2 * NS);
  return (a0 + a1) + (a2 + a3);
}

__device__ __forceinline__ bool finite_d(double v) { return __builtin_isfinite(v); }
__device__ __forceinline__ bool finite_t(float v) { return __builtin_isfinite(v); }
__device__ __forceinline__ bool finite_t(double v) { return __builtin_isfinite(v); }


// One matvec row pass: this lane's row of a resident block row times the vector
// window of knots m-1..m+1 (local knots m..m+2) of `vec`; 0 on inactive lanes.
// chunk_mv: each lane holding columns of its own row; row_mv: as reg_item holds it.
template <typename T, int NS, int NT, bool BC, int LP, bool ALONE, int CW>
__device__ __forceinline__ T chunk_mv(const RegItem<T, NS, NT, BC, LP, ALONE> &it, const T (&mat)[CW], const T *vec,
                                      bool act) {
  using R = RegItem<T, NS, NT, BC, LP, ALONE>;
  if constexpr (BC) {
    // every lane of the 16-lane row takes part in the broadcasts; lanes past the
    // window read (and discard) the last knot's entries
    const int mm = it.m < it.K + 1 ? it.m : it.K + 1;
    const T *v = vec + mm * R::nP + it.row;
    const T y = rowcast_dot<T, NS>(mat, v[0], v[R::nP], v[2 * R::nP]);
    return act ? y : (T)0;
  } else {
    T y = act ? chunk_dot<T, CW>(mat, vec + it.m * R::nP + it.c * CW) : (T)0;
    return group_sum<R::LPR>(y);
  }
}

template <typename T, int NS, int NT, bool BC, int LP, bool ALONE, int MW>
__device__ __forceinline__ T row_mv(const RegItem<T, NS, NT, BC, LP, ALONE> &it, const T (&mat)[MW], const T *vec,
                                    bool act) {
  using R = RegItem<T, NS, NT, BC, LP, ALONE>;
  if constexpr (R::TILED) {
    T ya = 0, yb = 0;
    if (act) tile_dot<T, R::TW, R::nP>(mat, vec + it.m * R::nP + it.i * R::TW, ya, yb);
    return tile_sum<R::TL>(ya, yb, it.i);
  } else {
    return chunk_mv(it, mat, vec, act);
  }
}

// Whether a paired instance keeps its Pinv chunks in LDS: the FP32 column-chunk
// instances of 2 < n <= 14 at 512 threads, held to 128 VGPRs so that two workgroups
// share a CU (with the chunks in registers they spill ~100 B per lane).  The
// host sizes LDS with the same rule (reg_lds_bytes).
__host__ __device__ constexpr bool pair_pinv_lds(size_t tsize, int nt, bool bc, int ns) {
  return tsize == 4 && nt == 512 && !bc && ns > 2 && ns <= 14;
}

// Whether a paired instance keeps its S chunks in LDS: FP64 rows of n = 28 at
// 512 threads (two lanes per row, two waves per SIMD; with both matrices in
// registers a lane would need ~290 registers).  Slots for the owned rows only:
// pair_s_slots(nt, n) lanes (two ghost knots' lanes fewer than the workgroup).
// Such an instance runs paired items only (plans of forward + adjoint systems).
// The host sizes LDS with the same rules (reg_lds_bytes).
__host__ __device__ constexpr bool pair_s_lds(size_t tsize, int nt, bool bc, int ns) {
  return tsize == 8 && nt == 512 && !bc && ns == 28;
}
__host__ __device__ constexpr int pair_s_slots(int nt, int ns) { return nt - 2 * 2 * ns; }

// Paired items on two lanes per row: a quad holds two rows, each lane W columns of the
// padded row (a quarter, rounded up to an even number) of both, value 2 j + r being
// row r, column j.  So a lane reads a quarter of each side's window and not half:
// those reads bound the iteration once VALU issue does not.  Per iteration, against a
// chunk of its own row per lane: FP64 n = 28, one knot range without exchange, 2.50 us
// (2.67), FP64 n = 12 N = 100 x100 7.68 (8.53), FP32 n = 14 N = 128 x64 2.46 (2.57).  Where a
// lane's columns are not whole 16-byte reads (FP32 n = 6 and 12) the chunks stay: n = 12
// N = 100 x100 4.65 us, 4.80 in quads.
template <int NS>
constexpr int quad_cols() {
  return 2 * ((3 * (int)padded_n(NS) + 7) / 8);
}
template <typename T, int NS>
constexpr bool in_quads() {
  return quad_cols<NS>() * (int)sizeof(T) % 16 == 0;
}

// Loads them, both rows (r0, r0 + 1: adjacent in memory) at once; lane i of the quad.
// Guarded loads for n = 28, as load_guarded, branch-free otherwise.
template <typename T, int NS>
__device__ __forceinline__ void load_quad(T (&dst)[2 * quad_cols<NS>()], const T *__restrict__ A, int kg, int r0,
                                          int i, int N, bool active) {
  typedef T pair_t __attribute__((ext_vector_type(2), aligned(sizeof(T))));
  constexpr int n = NS, nP = (int)padded_n(NS), W = quad_cols<NS>();
  int il = i, rl = r0;
  asm volatile("" : "+v"(il), "+v"(rl));
  const bool rowok = active && kg >= 0 && kg < N;
  const uint32_t base = rowok ? (uint32_t)kg * (uint32_t)(3 * n * n) + (uint32_t)rl : 0u;
#pragma unroll
  for (int j = 0; j < W; ++j) {
    const int col = il * W + j, seg = col / nP, cc = col - seg * nP;
    const bool ok = rowok && seg < 3 && cc < n && !(kg == 0 && seg == 0) && !(kg == N - 1 && seg == 2);
    pair_t v = {0, 0};
    if constexpr (NS > 14) {
      if (ok) v = load_at<pair_t>(A, 0u, base + (uint32_t)((seg * n + cc) * n));
      dst[2 * j] = v.x;
      dst[2 * j + 1] = v.y;
    } else {
      v = load_at<pair_t>(A, 0u, ok ? base + (uint32_t)((seg * n + cc) * n) : 0u);
      dst[2 * j] = ok ? v.x : (T)0;
      dst[2 * j + 1] = ok ? v.y : (T)0;
    }
  }
}

// A lane's columns of both rows times both sides' windows (xa, xb: its first column),
// from registers or from its slot `idx` in LDS (SL > 0: 16-byte block b at block index
// b * SL + idx, so a wave's reads of one block are contiguous): ya, yb are the partial
// products of rows 0 and 1.
template <int SL, typename T, int W, int MW>
__device__ __forceinline__ void quad_dot2(const T (&mat)[MW], const T *__restrict__ lds, int idx,
                                          const T *__restrict__ xa, const T *__restrict__ xb, T (&ya)[2], T (&yb)[2]) {
  constexpr int V = 16 / (int)sizeof(T);
  static_assert(W % V == 0, "whole 16-byte reads");
  typedef T block_t __attribute__((ext_vector_type(V)));
  T a[2][2] = {{0, 0}, {0, 0}}, b[2][2] = {{0, 0}, {0, 0}};
  block_t mv = {};
#pragma unroll
  for (int j0 = 0; j0 < W; j0 += V) {
    const block_t u = *reinterpret_cast<const block_t *>(xa + j0), v = *reinterpret_cast<const block_t *>(xb + j0);
#pragma unroll
    for (int jj = 0; jj < V; ++jj) {
      const int j = j0 + jj;
      if constexpr (SL > 0) {
        if (2 * j % V == 0) mv = *reinterpret_cast<const block_t *>(lds + ((size_t)(2 * j / V) * SL + idx) * V);
      }
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        T e;
        if constexpr (SL > 0) e = mv[2 * j % V + r]; else e = mat[2 * j + r];
        a[r][j % 2] = fmaT(e, u[jj], a[r][j % 2]);
        b[r][j % 2] = fmaT(e, v[jj], b[r][j % 2]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    ya[r] = a[r][0] + a[r][1];
    yb[r] = b[r][0] + b[r][1];
  }
}

// A matrix times both sides' vectors: partial products of the lanes that share a row (a
// quad: two rows) added up by DPP, so that the even lane of each row ends with its
// product for side A and the odd one for side B.
template <int SL, typename T, int NS, int NT, int MW>
__device__ __forceinline__ T sides_mv(const RegItem<T, NS, NT> &it, const T (&mat)[MW], const T *lds, int idx,
                                      const T *va, const T *vb, bool act) {
  using R = RegItem<T, NS, NT>;
  static_assert(R::LPR == 2 && NS % 2 == 0, "two lanes per row, rows in pairs");
  T a[2] = {0, 0}, b[2] = {0, 0};
  if constexpr (!in_quads<T, NS>()) {
    if (act) {
      const int off = it.m * R::nP + it.c * R::CW;
      if constexpr (SL > 0) {
        chunk_dot2_lds<R::CW, SL>(lds, idx, va + off, vb + off, a[0], b[0]);
      } else {
        a[0] = chunk_dot<T, R::CW>(mat, va + off);
        b[0] = chunk_dot<T, R::CW>(mat, vb + off);
      }
    }
  } else if (act) {
    const int off = it.m * R::nP + it.i * quad_cols<NS>();
    quad_dot2<SL, T, quad_cols<NS>()>(mat, lds, idx, va + off, vb + off, a, b);
  }
  const bool odd = it.c != 0;
  if constexpr (!in_quads<T, NS>()) return (odd ? b[0] : a[0]) + dpp<kDppQuadXor1>(odd ? a[0] : b[0]);
  const bool upper = it.i >= 2;
  const T pa = (upper ? a[1] : a[0]) + dpp<kDppQuadXor2>(upper ? a[0] : a[1]);
  const T pb = (upper ? b[1] : b[0]) + dpp<kDppQuadXor2>(upper ? b[0] : b[1]);
  return (odd ? pb : pa) + dpp<kDppQuadXor1>(odd ? pa : pb);
}

// g_S block rows of a rank's owned knots a..a+K-1 (paired items): -1/2 (gg_k lam_j^T +
// lam_k gg_j^T) for j in {k-1, k, k+1}, zero outside the system.  gg and lam are
// the ghost-extended windows in LDS (knot a-1+i at (i+1) nP).  V consecutive rows
// of one block column are contiguous in the cbtd layout, so each thread forms V
// of them and stores them at once (16 bytes where n and gS's alignment allow).
template <typename T, int NS, int NT>
__device__ __forceinline__ void write_gS(T *gS, const T *gg, const T *lam, int a, int K, int N) {
  constexpr int n = NS, nP = (int)padded_n(NS), bs = 3 * NS * NS;
  constexpr int VM = (int)(16 / sizeof(T));
  constexpr int V = n % VM == 0 ? VM : (n % 2 == 0 ? 2 : 1);
  typedef T vec_t __attribute__((ext_vector_type(V)));
  const bool vec_ok = V > 1 && ((uintptr_t)gS & (V * sizeof(T) - 1)) == 0;
  const int step = vec_ok ? V : 1;
  for (int e = opaque_tid() * step; e < K * bs; e += NT * step) {
    const int kl = e / bs;
    const int wq = e - kl * bs;
    const int col = wq / n;
    const int rr_ = wq - col * n;
    const int seg = col / n;
    const int cc = col - seg * n;
    const int k = a + kl;
    const int j = k - 1 + seg;
    const bool in = j >= 0 && j < N;
    const int lk = (kl + 2) * nP, lj = (kl + 1 + seg) * nP;
    const T lj_v = in ? lam[lj + cc] : (T)0, gj_v = in ? gg[lj + cc] : (T)0;
    if (vec_ok) {
      vec_t out;
#pragma unroll
      for (int v = 0; v < V; ++v) out[v] = in ? (T)-0.5 * (gg[lk + rr_ + v] * lj_v + lam[lk + rr_ + v] * gj_v) : (T)0;
      *reinterpret_cast<__attribute__((address_space(1))) vec_t *>(gptr(gS) + (size_t)a * bs + e) = out;
    } else {
      gptr(gS)[(size_t)a * bs + e] = in ? (T)-0.5 * (gg[lk + rr_] * lj_v + lam[lk + rr_] * gj_v) : (T)0;
    }
  }
}

// write_gS for a stateSize known at run time only, V consecutive rows per thread and
// step (2 for even n).  One workgroup writes a whole system's g_S, so the cost is
// instructions per element: the place of the next one is stepped, not divided out
// (FP32 n = 14 N = 64, adjoint alone: 78 -> 63 us).
template <typename T, int nP, int V>
__device__ __forceinline__ void write_gS_steps(T *gS, const T *gg, const T *lam, int n, int a, int K, int N,
                                               int threads) {
  typedef T vec_t __attribute__((ext_vector_type(V), aligned(sizeof(T))));
  const int cols = 3 * n, bs = cols * n, step = threads * V;
  const int dr = step % n, dcol = (step / n) % cols, dk = step / bs;
  int e = opaque_tid() * V;
  int k = e / bs, col = (e - k * bs) / n, r = e - k * bs - col * n;
  for (; e < K * bs; e += step) {
    const int seg = (col >= n) + (col >= 2 * n), cc = col - seg * n;
    const int j = a + k - 1 + seg;
    const int lk = (k + 2) * nP + r, lj = (k + 1 + seg) * nP + cc;
    const bool in = j >= 0 && j < N;
    const T lj_v = in ? lam[lj] : (T)0, gj_v = in ? gg[lj] : (T)0;
    vec_t out;
#pragma unroll
    for (int v = 0; v < V; ++v) out[v] = in ? (T)-0.5 * (gg[lk + v] * lj_v + lam[lk + v] * gj_v) : (T)0;
    *reinterpret_cast<__attribute__((address_space(1))) vec_t *>(gptr(gS) + (size_t)a * bs + e) = out;
    r += dr;
    col += dcol;
    k += dk;
    if (r >= n) {
      r -= n;
      ++col;
    }
    if (col >= cols) {
      col -= cols;
      ++k;
    }
  }
}
template <typename T, int nP>
__device__ __forceinline__ void write_gS_any(T *gS, const T *gg, const T *lam, int n, int a, int K, int N,
                                             int threads) {
  if (n & 1)
    write_gS_steps<T, nP, 1>(gS, gg, lam, n, a, K, N, threads);
  else
    write_gS_steps<T, nP, 2>(gS, gg, lam, n, a, K, N, threads);
}

// PRE: the set-up's HBM reads (initial guess window, first right-hand side)
// issued together with the matrix chunks, one round trip instead of three (off
// for the one-pass items of the paired kernel, whose 128-VGPR allocation spills
// differently, and runs its batches slower, with it; the paired item issues its
// own set-up reads together).
// BF: row broadcast of n <= 14 loads its rows branch-free (load_row); the runtime-n
// instances, short of registers, keep the guarded loads there.  Column chunks are
// loaded branch-free in any case, but for n = 28 at 512 threads (load_fixed).
// LP: lanes per row of the runtime-stateSize items, ALONE: a system's only rank
// (RegItem).
template <typename T, int NS, int NT, bool FUSED, bool BC = false, bool PRE = true, bool BF = PRE, int LP = 0,
          bool ALONE = false>
__device__ __forceinline__ void reg_item(const KSys &d, uint32_t rank, T *lds) {
  using R = RegItem<T, NS, NT, BC, LP, ALONE>;
  constexpr int nP = R::nP, CW = R::CW;
  R it;
  it.set_n((int)d.n);
  const int n = it.n;
  // a single solve's only workgroup is launched with the waves its rows need
  const int stride = ALONE ? (int)blockDim.x : NT;
  it.N = (int)d.N;
  it.G = ALONE ? 1 : (int)d.G;
  it.rank = ALONE ? 0 : (int)rank;
  it.a = ALONE ? 0 : (int)knot_begin(rank, d.G, d.N);
  it.b = ALONE ? it.N : (int)knot_begin(rank + 1, d.G, d.N);
  it.K = it.b - it.a;
  const int K = it.K;
  it.VL = (K + 4) * nP + (BC ? 16 : R::LPR * CW);
  it.slots = d.slots;
  it.tol = d.tol;
  it.rel = (d.flags & KF_REL) != 0;
  it.xcd = false;
  it.xcd_ok = (d.flags & KF_NOXCD) == 0;
  // lane roles (from an opaque thread index: recomputed per item rather than
  // hoisted out of the batched item loop)
  const int t = opaque_tid();
  it.q = t / R::LPR;
  it.c = t % R::LPR;
  it.i = t & (R::TL - 1);
  if constexpr (BC) {
    it.m = t >> 4;
    it.row = t & 15;
  } else {
    const int ln = ALONE ? (int)alone_lanes((uint32_t)n, d.N, R::LPR, NT, sizeof(T)) : n;
    it.m = it.q / ln;
    it.row = it.q - it.m * ln;
    // no neighbours: no lanes for ghost rows (a lone item of an any-size instance so
    // holds two knots more; the planner gives a fixed size no more than with neighbours)
    if (ALONE || (!R::RT && it.G == 1)) ++it.m;
  }
  it.kg = it.a - 1 + it.m;
  it.act_u = it.m < K + 2 && (!(BC || ALONE) || it.row < n);
  it.act_w = it.m >= 1 && it.m <= K && (!(BC || ALONE) || it.row < n);
  it.owner = it.act_w && it.c == 0;
  it.ghost = it.c == R::LPR - 1 && it.q < 4 * n && !ALONE && (R::RT || it.G > 1);
  if (!ALONE) it.set_edge_slots();
  {
    const int gk = it.q / n, gr = it.q - (it.q / n) * n;  // ghost element q: knot slot 0..3
    const int gj = gk < 2 ? gk : K + gk;                  // local knots 0, 1, K+2, K+3
    it.gpos = gj * nP + gr;
  }
  // LDS carve-up
  it.rv = lds;
  it.uv = it.rv + it.VL;
  it.wv = it.uv + it.VL;
  it.xv = it.wv + it.VL;
  it.lv = it.xv + it.VL;
  it.wsum = it.lv + it.VL;
  it.tot = it.wsum + 3 * R::NWAVES;
  it.ctl = reinterpret_cast<int *>(it.tot + 4);
  const int total = (int)(it.tot + 4 - lds);

  const int m = it.m, row = it.row, c = it.c, kg = it.kg;
  const int own_pos = (m + 1) * nP + row;  // local knot of own row kl = m - 1 is m + 1

  if (!ALONE && t == 0) {
    const uint32_t ea = (uint32_t)(xload(it.rec(0, it.rank)) >> 32);
    const uint32_t eb = (uint32_t)(xload(it.rec(1, it.rank)) >> 32);
    uint32_t base = (ea > eb ? ea : eb) + 1u;
    if (base > 0xFFF00000u) base = 1u;
    it.ctl[0] = 0;
    it.ctl[1] = (int)base;
  }
  for (int i = opaque_tid(); i < total; i += stride) lds[i] = (T)0;

  const bool fwd = (d.flags & KF_FWD) != 0;
  const bool adj = (d.flags & KF_ADJ) != 0;
  // every HBM read of the set-up in one round trip (PRE): the initial guess
  // window (own + one ghost knot each side; one per thread, the rest after the
  // barrier) and the first right-hand side,
  // issued with the matrix chunks
  const T *lam0 = static_cast<const T *>(d.lambda);
  const int wl = (K + 2) * n;
  T lam_pre = 0;
  int lam_pos = -1;
  if constexpr (PRE) {
    const int i = opaque_tid();
    if (i < wl) {
      const int jj = i / n, e = i - jj * n;
      const int k = it.a - 1 + jj;
      if (k >= 0 && k < it.N) {
        lam_pre = gptr(lam0)[(size_t)k * n + e];
        lam_pos = (jj + 1) * nP + e;
      }
    }
  }
  T b_pre = 0;
  if constexpr (PRE) {
    if (it.owner) b_pre = gptr(static_cast<const T *>(fwd ? d.gamma : d.glambda))[(size_t)kg * n + row];
  }

  // matrix chunks straight from HBM into registers
  T mM[R::MW], mS[R::MW];
  // row broadcast: branch-free loads on the single-solve instances; guarded ones
  // leave fewer live masks, which the paired and runtime-n instances need more
  constexpr bool kGuarded = !(BF && NS <= 14);
  // S first: loads complete in issue order, so the first product r = b - S x
  // (and the first exchange) can start while the Pinv chunks are in flight
  if constexpr (BC) {
    load_row<T, NS, kGuarded>(mS, static_cast<const T *>(d.S), kg, row, it.N, it.act_w);
    load_row<T, NS, kGuarded>(mM, static_cast<const T *>(d.Pinv), kg, row, it.N, it.act_u);
  } else if constexpr (R::RT) {
    load_chunk<T, nP, CW>(mS, static_cast<const T *>(d.S), kg, row, c != 0, it.N, it.act_w, n);
    load_chunk<T, nP, CW>(mM, static_cast<const T *>(d.Pinv), kg, row, c != 0, it.N, it.act_u, n);
  } else if constexpr (R::TILED) {
    const int r0 = row - it.i / R::LPR;
    load_tile<T, NS, R::TL, R::TW>(mS, static_cast<const T *>(d.S), kg, r0, it.i, it.N, it.act_w);
    load_tile<T, NS, R::TL, R::TW>(mM, static_cast<const T *>(d.Pinv), kg, r0, it.i, it.N, it.act_u);
  } else {
    load_fixed<T, NS, NT, CW>(mS, static_cast<const T *>(d.S), kg, row, c, it.N, it.act_w);
    load_fixed<T, NS, NT, CW>(mM, static_cast<const T *>(d.Pinv), kg, row, c, it.N, it.act_u);
  }
  __syncthreads();
  it.base = ALONE ? 0u : (uint32_t)it.ctl[1];
  it.seq = 0;
  {
    T *dst = fwd ? it.xv : it.lv;
    if (lam_pos >= 0) dst[lam_pos] = lam_pre;
    for (int i = opaque_tid() + (PRE ? stride : 0); i < wl; i += stride) {
      const int jj = i / n, e = i - jj * n;
      const int k = it.a - 1 + jj;
      if (k >= 0 && k < it.N) dst[(jj + 1) * nP + e] = gptr(lam0)[(size_t)k * n + e];
    }
  }
  __syncthreads();

  RegOut fo{0, GBDPCG_CONVERGED, 0.0, 0.0}, ao{0, GBDPCG_CONVERGED, 0.0, 0.0};
  bool timed_out = false;
  for (int pass = fwd ? 0 : 1; pass <= (adj ? 1 : 0); ++pass) {
    RegOut out{0, GBDPCG_MAX_ITER, 0.0, 0.0};
    if (pass == 1) {
      // adjoint: lambda (own + ghosts) was left in xv by the forward pass, or
      // loaded into lv above; keep it in lv and restart from x = 0
      if (fwd) {
        for (int i = opaque_tid(); i < it.VL; i += stride) it.lv[i] = it.xv[i];
      }
      for (int i = opaque_tid(); i < it.VL; i += stride) it.xv[i] = (T)0;
      __syncthreads();
    }
    // with PRE the first pass's right-hand side was read with the set-up
    const T *rhs = static_cast<const T *>(pass == 0 ? d.gamma : d.glambda);
    T x_i = 0, b_i = 0;
    if (it.owner) {
      x_i = it.xv[own_pos];
      b_i = PRE && (pass == 0) == fwd ? b_pre : gptr(rhs)[(size_t)kg * n + row];
    }
    // r = rhs - S x (own rows)
    T r_i;
    {
      T y = row_mv(it, mS, it.xv, it.act_w);
      r_i = it.owner ? b_i - y : (T)0;  // zero on the other lanes for good: only w'u needs a select
    }
    if (it.owner) it.rv[own_pos] = r_i;
    it.publish_edge(r_i, 2);
    it.reduce_publish(it.owner ? b_i * b_i : (T)0, (T)0, (T)0, true);
    T gg, sx, sxx;
    if (!it.gather(it.rv, 2, gg, sx, sxx)) {
      out.status = GBDPCG_TIMED_OUT;
      timed_out = true;
      if (pass == 0) fo = out; else ao = out;
      break;
    }
    // the sums are of small integers, exact in T; compare in double
    // (uniform by construction; readfirstlane lets the compiler branch on it in
    // scalar code)
    if constexpr (!ALONE)
      it.xcd = __builtin_amdgcn_readfirstlane(
                 (int)(it.xcd_ok && it.G > 1 && (double)sx * (double)sx == (double)it.G * (double)sxx)) != 0;
    // exit threshold: |r'z| < tol (reference) or r'r <= tol^2 rhs'rhs
    const double thr = it.rel ? it.tol * it.tol * (double)gg : it.tol;
    T r_g = it.ghost ? it.rv[it.gpos] : (T)0;
    if constexpr (!FUSED) {
      // reference recurrence.  z = Pinv r on own and one ghost knot each side,
      // p = z, eta = r'z
      T z_i, p_i, eta, rr;
      {
        z_i = row_mv(it, mM, it.rv, it.act_u);
        it.settle();
        p_i = z_i;
        if (it.act_u && c == 0) it.uv[(m + 1) * nP + row] = p_i;  // uv holds p
        const T rz = r_i * z_i;
        const T r2 = r_i * r_i;
        it.reduce_publish(rz, (T)0, r2);
        T unused;
        if (!it.gather(it.wv, 0, eta, unused, rr)) {
          out.status = GBDPCG_TIMED_OUT;
          timed_out = true;
          if (pass == 0) fo = out; else ao = out;
          break;
        }
        out.eta = (double)eta;
        out.rr = (double)rr;
        bool stop = false;
        if (!finite_t(eta) || !finite_t(rr)) {
          out.status = GBDPCG_NONFINITE;
          stop = true;
        } else if (eta == (T)0) {
          out.status = rr == (T)0 ? GBDPCG_CONVERGED : GBDPCG_BREAKDOWN;
          stop = true;
        }
        if (stop) {
          out.iters = 0;
          goto finish;
        }
        it.settle();
      }
      {
        uint32_t iter = 0;
        const uint32_t max_iter = d.max_iter;
        while (iter < max_iter) {
          // v = S p (own rows); alpha = eta / p'v.  The exchange also carries the
          // two edge knots of v each side: the ghost lanes' r needs them.
          T v_i;
          {
            v_i = row_mv(it, mS, it.uv, it.act_w);
          }
          it.publish_edge(v_i, 2);
          it.reduce_publish(it.owner ? p_i * v_i : (T)0, (T)0, (T)0);
          T pv, u1, u2;
          if (!it.gather(it.wv, 2, pv, u1, u2)) {
            out.status = GBDPCG_TIMED_OUT;
            timed_out = true;
            break;
          }
          const T v_g = it.ghost ? it.wv[it.gpos] : (T)0;
          if (pv == (T)0 || !finite_t(pv)) {
            out.status = pv == (T)0 ? GBDPCG_BREAKDOWN : GBDPCG_NONFINITE;
            break;
          }
          const T alpha = qdiv(eta, pv);
          // lambda += alpha p ; r -= alpha v (own rows, and the ghost lanes' r)
          if (it.owner) {
            x_i = fmaT(alpha, p_i, x_i);
            r_i = fmaT(-alpha, v_i, r_i);
            it.rv[own_pos] = r_i;
          }
          if (it.ghost) {
            r_g = fmaT(-alpha, v_g, r_g);
            it.rv[it.gpos] = r_g;
          }
          __syncthreads();
          // z = Pinv r (own + ghost rows) ; eta' = r'z ; exit test
          {
            z_i = row_mv(it, mM, it.rv, it.act_u);
          }
          const T rz = r_i * z_i;
          const T r2 = r_i * r_i;
          it.reduce_publish(rz, (T)0, r2);
          T eta_new, u3;
          if (!it.gather(it.wv, 0, eta_new, u3, rr)) {
            out.status = GBDPCG_TIMED_OUT;
            timed_out = true;
            break;
          }
          ++iter;
          out.eta = (double)eta_new;
          out.rr = (double)rr;
          if (it.rel ? ((double)rr <= thr) : (__builtin_fabs((double)eta_new) < thr)) {
            out.status = GBDPCG_CONVERGED;
            break;
          }
          if (!finite_t(eta_new)) {
            out.status = GBDPCG_NONFINITE;
            break;
          }
          // p = z + beta p on own and ghost knots
          const T beta = qdiv(eta_new, eta);
          eta = eta_new;
          p_i = fmaT(beta, p_i, z_i);
          if (it.act_u && c == 0) it.uv[(m + 1) * nP + row] = p_i;
          __syncthreads();
        }
        out.iters = (int)iter;
      }
    } else {
      // u = Pinv r (own + ghost rows), w = S u (own rows)
      T u_i, w_i;
      T p_i, s_i, s_g;
      T eta, alpha, rr;
      {
        u_i = row_mv(it, mM, it.rv, it.act_u);
        if (it.act_u && c == 0) it.uv[(m + 1) * nP + row] = u_i;
        __syncthreads();
        w_i = row_mv(it, mS, it.uv, it.act_w);
        it.publish_edge(w_i, 2);
        const T rz = r_i * u_i;
        const T wu = it.owner ? w_i * u_i : (T)0;
        const T r2 = r_i * r_i;
        it.reduce_publish(rz, wu, r2);
        T delta;
        if (!it.gather(it.wv, 2, eta, delta, rr)) {
          out.status = GBDPCG_TIMED_OUT;
          timed_out = true;
          if (pass == 0) fo = out; else ao = out;
          break;
        }
        p_i = u_i;
        s_i = w_i;
        s_g = it.ghost ? it.wv[it.gpos] : (T)0;
        alpha = delta != (T)0 ? eta / delta : (T)0;
        out.eta = (double)eta;
        out.rr = (double)rr;
        bool stop = false;
        if (!finite_d((double)eta) || !finite_d((double)rr)) {
          out.status = GBDPCG_NONFINITE;
          stop = true;
        } else if (eta == (T)0) {
          out.status = rr == (T)0 ? GBDPCG_CONVERGED : GBDPCG_BREAKDOWN;
          stop = true;
        } else if (delta == (T)0 || !finite_d((double)alpha)) {
          out.status = GBDPCG_BREAKDOWN;
          stop = true;
        }
        if (stop) {
          out.iters = 0;
          goto finish;
        }
      }
      {
        uint32_t iter = 0;
        const uint32_t max_iter = d.max_iter;
        T last_eta = eta, last_rr = rr;  // of the last exchange (uniform)
        while (iter < max_iter) {
          // x += alpha p ; r -= alpha s  (own in registers, ghosts by the ghost lanes)
          if (it.owner) {
            x_i = fmaT(alpha, p_i, x_i);
            r_i = fmaT(-alpha, s_i, r_i);
            it.rv[own_pos] = r_i;
          }
          if (it.ghost) {
            r_g = fmaT(-alpha, s_g, r_g);
            it.rv[it.gpos] = r_g;
          }
          __syncthreads();
          u_i = row_mv(it, mM, it.rv, it.act_u);
          if (it.act_u && c == 0) it.uv[(m + 1) * nP + row] = u_i;
          __syncthreads();
          w_i = row_mv(it, mS, it.uv, it.act_w);
          it.publish_edge(w_i, 2);
          const T rz = r_i * u_i;
          const T wu = it.owner ? w_i * u_i : (T)0;
          const T r2 = r_i * r_i;
          it.reduce_publish(rz, wu, r2);
          T eta_new, delta_new;
          if (!it.gather(it.wv, 2, eta_new, delta_new, rr)) {
            out.status = GBDPCG_TIMED_OUT;
            timed_out = true;
            break;
          }
          // ghost lanes: the neighbour's w, read now so the LDS latency overlaps the
          // scalar recurrence below
          const T w_g = it.ghost ? it.wv[it.gpos] : (T)0;
          ++iter;
          last_eta = eta_new;
          last_rr = rr;
          // the stop tests and the next coefficients are independent: all are
          // computed first, then one branch (a shorter dependency chain; the
          // coefficients of a stopping iteration are discarded).  beta and
          // eta'/alpha: two divisions in flight at once.
          const bool conv = it.rel ? ((double)rr <= thr) : (__builtin_fabs((double)eta_new) < thr);
          const bool nonfin = !finite_t(eta_new);
          const T beta = qdiv(eta_new, eta);
          const T den = delta_new - beta * qdiv(eta_new, alpha);
          const bool brk = den == (T)0 || !finite_t(den);
          const T alpha_new = qdiv(eta_new, den);
          if (conv || nonfin || brk) {
            out.status = conv ? GBDPCG_CONVERGED : nonfin ? GBDPCG_NONFINITE : GBDPCG_BREAKDOWN;
            break;
          }
          alpha = alpha_new;
          eta = eta_new;
          p_i = fmaT(beta, p_i, u_i);
          s_i = fmaT(beta, s_i, w_i);
          if (it.ghost) s_g = fmaT(beta, s_g, w_g);
        }
        out.iters = (int)iter;
        out.eta = (double)last_eta;
        out.rr = (double)last_rr;
      }
    }
  finish:
    if (pass == 0) fo = out; else ao = out;
    if (timed_out) break;
    // solution: own knots to HBM; for the adjoint, also its edge knots to the
    // neighbours (g_S needs lambda and g_gamma one knot beyond the owned range)
    {
      T *dst = static_cast<T *>(pass == 0 ? d.lambda : d.ggamma);
      if (it.owner) gptr(dst)[(size_t)kg * n + row] = x_i;
    }
    if (adj) {
      if (it.owner) it.xv[own_pos] = x_i;
      it.settle();
      it.publish_edge(x_i, 1);
      it.reduce_publish((T)0, (T)0, (T)0);
      T z0, z1, z2;
      if (!it.gather(it.xv, 1, z0, z1, z2)) {
        timed_out = true;
        if (pass == 0) fo.status = GBDPCG_TIMED_OUT; else ao.status = GBDPCG_TIMED_OUT;
        break;
      }
    }
    if (pass == 1 && R::RT) {
      write_gS_any<T, nP>(static_cast<T *>(d.gS), it.xv, it.lv, n, it.a, K, it.N, stride);
    } else if (pass == 1) {
      // g_S block rows of the own knots: -1/2 (gg_k lam_j^T + lam_k gg_j^T), j in {k-1,k,k+1}
      // (one element per thread and step: the vectorised write_gS costs this
      // item two VGPRs, and with them the 512-thread FP32 n = 14 instance's
      // second workgroup per CU)
      const int bs = 3 * n * n;
      T *gS = static_cast<T *>(d.gS);
      for (int e = opaque_tid(); e < K * bs; e += stride) {
        const int kl = e / bs;
        const int wq = e - kl * bs;
        const int col = wq / n;
        const int rr_ = wq - col * n;
        const int seg = col / n;
        const int cc = col - seg * n;
        const int k = it.a + kl;
        const int j = k - 1 + seg;
        T val = 0;
        if (j >= 0 && j < it.N) {
          const int lk = (kl + 2) * nP, lj = (kl + 1 + seg) * nP;
          val = (T)-0.5 * (it.xv[lk + rr_] * it.lv[lj + cc] + it.lv[lk + rr_] * it.xv[lj + cc]);
        }
        gptr(gS)[(size_t)it.a * bs + e] = val;
      }
    }
    __syncthreads();
  }
  if (rank == 0 && t == 0 && d.result != nullptr) {
    gbdpcg_result res;
    res.iters = fo.iters;
    res.status = fo.status;
    res.adj_iters = ao.iters;
    res.adj_status = ao.status;
    res.eta = fo.eta;
    res.rr = fo.rr;
    res.adj_eta = ao.eta;
    res.adj_rr = ao.rr;
    *d.result = res;
  }
  if (timed_out && t == 0 && d.err != nullptr)
    __hip_atomic_store(d.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Two rows per lane: FP32 systems of one workgroup (stateSize n <= NS as in
// RegItem) too large for a lane per row.  Lane (m, h) holds rows 2h and 2h + 1 of
// knot m - 1, so a vector window read from LDS serves two rows: the iteration is
// bound by those reads and the multiply-adds (two waves per SIMD), still without
// an exchange.  Per iteration, fused / reference form, against several ranks:
// n = 12 N = 64 1.09 / 1.27 us (1.36 / 2.23), n = 14 N = 64 1.21 / 1.41 (1.40 /
// 2.32), n = 13 N = 50 1.22 / 1.39 (1.63 / 2.37), n = 8 N = 128 0.95 / 1.14 (1.50 /
// 2.28).
template <int NS, int NT>
struct TwoRows {
  static constexpr int nP = NS, CW = 3 * NS, NWAVES = NT / 64;
  int n, N, m, row;        // row: the first of the lane's rows
  bool act, second;        // the lane has rows; it has both (odd n: the last lane of a knot has one)
  float *wsum;

  // y = the lane's two rows times the window of knots m-1..m+1 of vec
  __device__ __forceinline__ void mv(const float (&a)[CW], const float (&b)[CW], const float *vec, float &ya,
                                     float &yb) const {
    float a0 = 0, a1 = 0, a2 = 0, a3 = 0, b0 = 0, b1 = 0, b2 = 0, b3 = 0;
    if (act) {
      const float *x = vec + m * nP;
#pragma unroll
      for (int j = 0; j < CW; j += 4) {
        const float4 xv = *reinterpret_cast<const float4 *>(x + j);
        a0 = __builtin_fmaf(a[j + 0], xv.x, a0);
        b0 = __builtin_fmaf(b[j + 0], xv.x, b0);
        a1 = __builtin_fmaf(a[j + 1], xv.y, a1);
        b1 = __builtin_fmaf(b[j + 1], xv.y, b1);
        a2 = __builtin_fmaf(a[j + 2], xv.z, a2);
        b2 = __builtin_fmaf(b[j + 2], xv.z, b2);
        a3 = __builtin_fmaf(a[j + 3], xv.w, a3);
        b3 = __builtin_fmaf(b[j + 3], xv.w, b3);
      }
    }
    ya = (a0 + a1) + (a2 + a3);
    yb = (b0 + b1) + (b2 + b3);
  }

  __device__ __forceinline__ void put(float *vec, float ya, float yb) const {
    if (act) *reinterpret_cast<float2 *>(vec + (m + 1) * nP + row) = make_float2(ya, yb);
  }

  // Workgroup totals in every wave; the caller has a barrier between two calls.
  __device__ __forceinline__ void totals(float &s0, float &s1, float &s2) const {
    const float sums = wave_sums(s0, s1, s2);
    const int slot = wave_sums_slot<3>();
    if (slot >= 0) wsum[(threadIdx.x >> 6) * 3 + slot] = sums;
    __syncthreads();
    const int l = (int)threadIdx.x & 3;
    const float v = waves_total<NWAVES, 3>(wsum, l < 3 ? l : 0);
    s0 = read_lane(v, 0);
    s1 = read_lane(v, 1);
    s2 = read_lane(v, 2);
  }
};

template <int NS, int NT, bool FUSED>
__device__ __forceinline__ void two_rows_item(const KSys &d, float *lds) {
  using R = TwoRows<NS, NT>;
  constexpr int nP = R::nP, CW = R::CW;
  R it;
  const int n = (int)d.n, N = (int)d.N, stride = (int)blockDim.x;
  it.n = n;
  it.N = N;
  const int VL = (N + 4) * nP + CW;
  float *rv = lds, *uv = rv + VL, *xv = uv + VL, *lv = xv + VL;
  it.wsum = lv + VL;
  const int total = 4 * VL + 3 * R::NWAVES;
  const int t = opaque_tid();
  {
    const int half = (int)two_rows_lanes((uint32_t)n, d.N, NT), k = t / half;
    it.m = k + 1;
    it.row = 2 * (t - k * half);
    it.act = k < N && it.row < n;
    it.second = it.act && it.row + 1 < n;
  }
  const int kg = it.m - 1;
  const bool fwd = (d.flags & KF_FWD) != 0, adj = (d.flags & KF_ADJ) != 0, rel = (d.flags & KF_REL) != 0;
  for (int i = opaque_tid(); i < total; i += stride) lds[i] = 0.f;

  // one HBM round trip: right-hand side, guess and matrices together
  const float *lam0 = static_cast<const float *>(d.lambda);
  auto rhs_at = [&](const void *p, float &a, float &b) {
    const float *v = static_cast<const float *>(p) + (size_t)kg * n + it.row;
    a = it.act ? gptr(v)[0] : 0.f;
    b = it.second ? gptr(v)[1] : 0.f;
  };
  float xa, xb, ba, bb;
  rhs_at(lam0, xa, xb);
  rhs_at(fwd ? d.gamma : d.glambda, ba, bb);
  float sa[CW], sb[CW], pa[CW], pb[CW];
  load_two_rows<NS>(sa, sb, static_cast<const float *>(d.S), kg, it.row, N, it.act, it.second, n);
  load_two_rows<NS>(pa, pb, static_cast<const float *>(d.Pinv), kg, it.row, N, it.act, it.second, n);
  __syncthreads();
  it.put(fwd ? xv : lv, xa, xb);
  __syncthreads();

  RegOut fo{0, GBDPCG_CONVERGED, 0.0, 0.0}, ao{0, GBDPCG_CONVERGED, 0.0, 0.0};
  for (int pass = fwd ? 0 : 1; pass <= (adj ? 1 : 0); ++pass) {
    RegOut out{0, GBDPCG_MAX_ITER, 0.0, 0.0};
    if (pass == 1) {
      // lambda stays in lv; the adjoint starts from x = 0
      if (fwd) {
        it.put(lv, xa, xb);
        rhs_at(d.glambda, ba, bb);
      }
      xa = xb = 0.f;
      it.put(xv, 0.f, 0.f);
      __syncthreads();
    }
    float ra, rb;
    it.mv(sa, sb, xv, ra, rb);
    ra = ba - ra;
    rb = bb - rb;
    it.put(rv, ra, rb);
    float gg = ba * ba + bb * bb, z0 = 0, z1 = 0;
    it.totals(gg, z0, z1);
    const double thr = rel ? d.tol * d.tol * (double)gg : d.tol;
    // u = Pinv r (the reference form's z)
    float ua, ub;
    it.mv(pa, pb, rv, ua, ub);
    it.put(uv, ua, ub);
    __syncthreads();
    float eta = ra * ua + rb * ub, delta = 0, rr = ra * ra + rb * rb, wa = 0, wb = 0;
    if constexpr (FUSED) {
      it.mv(sa, sb, uv, wa, wb);
      delta = wa * ua + wb * ub;
    }
    it.totals(eta, delta, rr);
    // p = u (reference form: held in uv as well); s = w
    float qa = ua, qb = ub, va = wa, vb = wb;
    float alpha = FUSED && delta != 0.f ? eta / delta : 0.f;
    out.eta = (double)eta;
    out.rr = (double)rr;
    bool run = d.max_iter > 0;
    if (!finite_t(eta) || !finite_t(rr)) {
      out.status = GBDPCG_NONFINITE;
      run = false;
    } else if (eta == 0.f) {
      out.status = rr == 0.f ? GBDPCG_CONVERGED : GBDPCG_BREAKDOWN;
      run = false;
    } else if (FUSED && (delta == 0.f || !finite_t(alpha))) {
      out.status = GBDPCG_BREAKDOWN;
      run = false;
    }
    uint32_t iter = 0;
    __syncthreads();  // totals above before those of the loop
    while (run) {
      if constexpr (FUSED) {
        xa = fmaT(alpha, qa, xa);
        xb = fmaT(alpha, qb, xb);
        ra = fmaT(-alpha, va, ra);
        rb = fmaT(-alpha, vb, rb);
        it.put(rv, ra, rb);
        __syncthreads();
        it.mv(pa, pb, rv, ua, ub);
        it.put(uv, ua, ub);
        __syncthreads();
        it.mv(sa, sb, uv, wa, wb);
        float eta_new = ra * ua + rb * ub, delta_new = wa * ua + wb * ub;
        rr = ra * ra + rb * rb;
        it.totals(eta_new, delta_new, rr);
        ++iter;
        out.eta = (double)eta_new;
        out.rr = (double)rr;
        const bool conv = rel ? ((double)rr <= thr) : (__builtin_fabs((double)eta_new) < thr);
        const bool nonfin = !finite_t(eta_new);
        const float beta = qdiv(eta_new, eta);
        const float den = delta_new - beta * qdiv(eta_new, alpha);
        const bool brk = den == 0.f || !finite_t(den);
        const float alpha_new = qdiv(eta_new, den);
        if (conv || nonfin || brk) {
          out.status = conv ? GBDPCG_CONVERGED : nonfin ? GBDPCG_NONFINITE : GBDPCG_BREAKDOWN;
          break;
        }
        alpha = alpha_new;
        eta = eta_new;
        qa = fmaT(beta, qa, ua);
        qb = fmaT(beta, qb, ub);
        va = fmaT(beta, va, wa);
        vb = fmaT(beta, vb, wb);
      } else {
        it.mv(sa, sb, uv, va, vb);
        float pv = qa * va + qb * vb, y1 = 0, y2 = 0;
        it.totals(pv, y1, y2);
        if (pv == 0.f || !finite_t(pv)) {
          out.status = pv == 0.f ? GBDPCG_BREAKDOWN : GBDPCG_NONFINITE;
          break;
        }
        alpha = qdiv(eta, pv);
        xa = fmaT(alpha, qa, xa);
        xb = fmaT(alpha, qb, xb);
        ra = fmaT(-alpha, va, ra);
        rb = fmaT(-alpha, vb, rb);
        it.put(rv, ra, rb);
        __syncthreads();
        it.mv(pa, pb, rv, ua, ub);
        float eta_new = ra * ua + rb * ub, y3 = 0;
        rr = ra * ra + rb * rb;
        it.totals(eta_new, y3, rr);
        ++iter;
        out.eta = (double)eta_new;
        out.rr = (double)rr;
        if (rel ? ((double)rr <= thr) : (__builtin_fabs((double)eta_new) < thr)) {
          out.status = GBDPCG_CONVERGED;
          break;
        }
        if (!finite_t(eta_new)) {
          out.status = GBDPCG_NONFINITE;
          break;
        }
        const float beta = qdiv(eta_new, eta);
        eta = eta_new;
        qa = fmaT(beta, qa, ua);
        qb = fmaT(beta, qb, ub);
        it.put(uv, qa, qb);
        __syncthreads();
      }
      run = iter < d.max_iter;
    }
    out.iters = (int)iter;
    if (pass == 0) fo = out; else ao = out;
    float *dst = static_cast<float *>(pass == 0 ? d.lambda : d.ggamma) + (size_t)kg * n + it.row;
    if (it.act) gptr(dst)[0] = xa;
    if (it.second) gptr(dst)[1] = xb;
    if (pass == 1) {
      it.put(xv, xa, xb);
      __syncthreads();
      write_gS_any<float, nP>(static_cast<float *>(d.gS), xv, lv, n, 0, N, N, stride);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0 && d.result != nullptr) {
    gbdpcg_result res;
    res.iters = fo.iters;
    res.status = fo.status;
    res.adj_iters = ao.iters;
    res.adj_status = ao.status;
    res.eta = fo.eta;
    res.rr = fo.rr;
    res.adj_eta = ao.eta;
    res.adj_rr = ao.rr;
    *d.result = res;
  }
}

// Forward and adjoint solves of one system iterated together (fused recurrence;
// both flags set).  The two solves share S and Pinv and are independent until
// g_S is formed, so each iteration runs the two right-hand sides (A: gamma,
// from lambda0; B: g_lambda, from 0) through the same resident matrices and one
// exchange carrying both sets of scalars and edges.  Each side performs the
// operations of its own solve in reg_item, in the row broadcast in the same order (the
// same bits); chunks and lone items of reg_item group the lanes of a sum otherwise.  A
// side stops on its own exit test; the other then goes on with both sides' products
// formed and the stopped one's discarded.
template <typename T, int NS, int NT, bool BC>
__device__ __forceinline__ void reg_item_pair(const KSys &d, uint32_t rank, T *lds) {
  using R = RegItem<T, NS, NT, BC>;
  constexpr int n = R::n, nP = R::nP, CW = R::CW;
  R it;
  it.N = (int)d.N;
  it.G = (int)d.G;
  it.rank = (int)rank;
  it.a = (int)knot_begin(rank, d.G, d.N);
  it.b = (int)knot_begin(rank + 1, d.G, d.N);
  it.K = it.b - it.a;
  const int K = it.K;
  it.VL = (K + 4) * nP + (BC ? 16 : R::LPR * CW);
  it.slots = d.slots;
  it.tol = d.tol;
  it.rel = (d.flags & KF_REL) != 0;
  it.xcd = false;
  it.xcd_ok = (d.flags & KF_NOXCD) == 0;
  const int t = opaque_tid();
  it.q = t / R::LPR;
  it.c = t % R::LPR;
  it.i = t & (R::TL - 1);
  if constexpr (BC) {
    it.m = t >> 4;
    it.row = t & 15;
  } else {
    it.m = it.q / n;
    it.row = it.q - it.m * n;
  }
  it.kg = it.a - 1 + it.m;
  it.act_u = it.m < K + 2 && (!BC || it.row < n);
  it.act_w = it.m >= 1 && it.m <= K && (!BC || it.row < n);
  it.owner = it.act_w && it.c == 0;
  it.ghost = it.c == R::LPR - 1 && it.q < 4 * n;
  it.set_edge_slots();
  {
    const int gk = it.q / n, gr = it.q - (it.q / n) * n;
    const int gj = gk < 2 ? gk : K + gk;
    it.gpos = gj * nP + gr;
  }
  // LDS: r, u, w of each side, lambda and g_gamma windows, 6 partials per wave
  T *rA = lds, *uA = rA + it.VL, *wA = uA + it.VL;
  T *rB = wA + it.VL, *uB = rB + it.VL, *wB = uB + it.VL;
  it.xv = wB + it.VL;  // lambda0 window, later g_gamma with ghosts
  it.lv = it.xv + it.VL;  // lambda with ghosts (for g_S)
  it.rv = rA;
  it.uv = uA;
  it.wv = wA;
  it.wsum = it.lv + it.VL;
  it.tot = it.wsum + 6 * R::NWAVES;
  it.ctl = reinterpret_cast<int *>(it.tot + 8);
  const int total = (int)(it.tot + 8 - lds);

  const int m = it.m, row = it.row, c = it.c, kg = it.kg;
  const int own_pos = (m + 1) * nP + row;
  constexpr int VB = 4 * n;  // second edge block

  if (t == 0) {
    const uint32_t ea = (uint32_t)(xload(it.rec(0, it.rank)) >> 32);
    const uint32_t eb = (uint32_t)(xload(it.rec(1, it.rank)) >> 32);
    uint32_t base = (ea > eb ? ea : eb) + 1u;
    if (base > 0xFFF00000u) base = 1u;
    it.ctl[0] = 0;
    it.ctl[1] = (int)base;
  }
  for (int i = opaque_tid(); i < total; i += NT) lds[i] = (T)0;

  // the set-up's vector reads (initial guess window: (K + 2) n <= NT values, one
  // per thread; both right-hand sides of the owned rows) issued with the matrix
  // chunks: one HBM round trip instead of three
  const T *lam0 = static_cast<const T *>(d.lambda);
  const int wl = (K + 2) * n;
  T lam_pre = 0, bA = 0, bB = 0;
  int lam_pos = -1;
  {
    const int i = opaque_tid();
    if (i < wl) {
      const int jj = i / n, e = i - jj * n;
      const int k = it.a - 1 + jj;
      if (k >= 0 && k < it.N) {
        lam_pre = gptr(lam0)[(size_t)k * n + e];
        lam_pos = (jj + 1) * nP + e;
      }
    }
    if (it.owner) {
      bA = gptr(static_cast<const T *>(d.gamma))[(size_t)kg * n + row];
      bB = gptr(static_cast<const T *>(d.glambda))[(size_t)kg * n + row];
    }
  }

  T mM[CW], mS[CW];
  if constexpr (BC) {
    load_row<T, NS, true>(mM, static_cast<const T *>(d.Pinv), kg, row, it.N, it.act_u);
    load_row<T, NS, true>(mS, static_cast<const T *>(d.S), kg, row, it.N, it.act_w);
  } else {
    load_fixed<T, NS, NT, CW>(mM, static_cast<const T *>(d.Pinv), kg, row, c, it.N, it.act_u);
    load_fixed<T, NS, NT, CW>(mS, static_cast<const T *>(d.S), kg, row, c, it.N, it.act_w);
  }
  __syncthreads();
  it.base = (uint32_t)it.ctl[1];
  it.seq = 0;
  if (lam_pos >= 0) it.xv[lam_pos] = lam_pre;
  for (int i = opaque_tid() + NT; i < wl; i += NT) {
    const int jj = i / n, e = i - jj * n;
    const int k = it.a - 1 + jj;
    if (k >= 0 && k < it.N) it.xv[(jj + 1) * nP + e] = gptr(lam0)[(size_t)k * n + e];
  }
  __syncthreads();

  RegOut fo{0, GBDPCG_MAX_ITER, 0.0, 0.0}, ao{0, GBDPCG_MAX_ITER, 0.0, 0.0};
  bool timed_out = false;
  T xA = 0, xB = 0;
  if (it.owner) xA = it.xv[own_pos];
  // r = rhs - S x (B starts from x = 0: r = g_lambda)
  T rA_i;
  rA_i = bA - chunk_mv(it, mS, it.xv, it.act_w);
  if (!it.owner) rA_i = (T)0;  // and stays so: only w'u needs a select below
  T rB_i = bB;
  if (it.owner) {
    rA[own_pos] = rA_i;
    rB[own_pos] = rB_i;
  }
  it.publish_edge(rA_i, 2);
  it.publish_edge(rB_i, 2, VB);
  T tt[6];
  it.reduce_publish6(it.owner ? bA * bA : (T)0, (T)0, (T)0, it.owner ? bB * bB : (T)0, (T)0, (T)0, true);
  bool runA = true, runB = true;
  double thrA = 0.0, thrB = 0.0;
  T rgA = 0, rgB = 0;
  T pA = 0, sA = 0, sgA = 0, etaA = 0, alphaA = 0;
  T pB = 0, sB = 0, sgB = 0, etaB = 0, alphaB = 0;
  T uA_i = 0, wA_i = 0, uB_i = 0, wB_i = 0;
  uint32_t iterA = 0, iterB = 0;
  const uint32_t max_iter = d.max_iter;
  if (!it.gather_pair(rA, rB, 2, tt)) {
    timed_out = true;
  } else {
    it.xcd = __builtin_amdgcn_readfirstlane(
                 (int)(it.xcd_ok && it.G > 1 && (double)tt[1] * (double)tt[1] == (double)it.G * (double)tt[2])) != 0;
    thrA = uniform(it.rel ? it.tol * it.tol * (double)tt[0] : it.tol);
    thrB = uniform(it.rel ? it.tol * it.tol * (double)tt[3] : it.tol);
    rgA = it.ghost ? rA[it.gpos] : (T)0;
    rgB = it.ghost ? rB[it.gpos] : (T)0;
    // first u = Pinv r, w = S u of both sides
    uA_i = chunk_mv(it, mM, rA, it.act_u);
    uB_i = chunk_mv(it, mM, rB, it.act_u);
    if (it.act_u && c == 0) {
      uA[(m + 1) * nP + row] = uA_i;
      uB[(m + 1) * nP + row] = uB_i;
    }
    __syncthreads();
    wA_i = chunk_mv(it, mS, uA, it.act_w);
    wB_i = chunk_mv(it, mS, uB, it.act_w);
    it.publish_edge(wA_i, 2);
    it.publish_edge(wB_i, 2, VB);
    it.reduce_publish6(rA_i * uA_i, it.owner ? wA_i * uA_i : (T)0, rA_i * rA_i,
                       rB_i * uB_i, it.owner ? wB_i * uB_i : (T)0, rB_i * rB_i);
    if (!it.gather_pair(wA, wB, 2, tt)) timed_out = true;
  }
  // initial checks of each side (as in reg_item)
  // last r'z and r'r of each side (uniform, kept as T; widened at the end)
  T lastA[2] = {0, 0}, lastB[2] = {0, 0};
  auto first = [&](RegOut &out, bool &run, T eta, T delta, T rr, T w_i, T u_i, T *wv, T &p, T &s_, T &sg, T &et,
                   T &alpha, T (&last)[2]) {
    p = u_i;
    s_ = w_i;
    sg = it.ghost ? wv[it.gpos] : (T)0;
    et = eta;
    alpha = uniform(delta != (T)0 ? eta / delta : (T)0);
    last[0] = eta;
    last[1] = rr;
    bool stop = false;
    if (!finite_d((double)eta) || !finite_d((double)rr)) {
      out.status = GBDPCG_NONFINITE;
      stop = true;
    } else if (eta == (T)0) {
      out.status = rr == (T)0 ? GBDPCG_CONVERGED : GBDPCG_BREAKDOWN;
      stop = true;
    } else if (delta == (T)0 || !finite_d((double)alpha)) {
      out.status = GBDPCG_BREAKDOWN;
      stop = true;
    }
    if (stop) run = false;
    if (max_iter == 0) run = false;
  };
  if (!timed_out) {
    first(fo, runA, tt[0], tt[1], tt[2], wA_i, uA_i, wA, pA, sA, sgA, etaA, alphaA, lastA);
    first(ao, runB, tt[3], tt[4], tt[5], wB_i, uB_i, wB, pB, sB, sgB, etaB, alphaB, lastB);
  } else {
    runA = runB = false;
  }
  // The scalar step of one side after an exchange, as in reg_item: candidates
  // first (both sides in straight-line code, so their dependency chains
  // overlap), then committed for a running side only.
  struct Cand {
    bool conv, nonfin, brk;
    T alpha, p, s, sg;
  };
  auto cand = [&](double thr, T eta_new, T delta_new, T rr, T w_i, T u_i, T w_g, T p, T s_, T sg, T eta,
                  T alpha) -> Cand {
    Cand c;
    c.conv = it.rel ? ((double)rr <= thr) : (__builtin_fabs((double)eta_new) < thr);
    c.nonfin = !finite_t(eta_new);
    const T beta = qdiv(eta_new, eta);
    const T den = delta_new - beta * qdiv(eta_new, alpha);
    c.brk = den == (T)0 || !finite_t(den);
    c.alpha = uniform(qdiv(eta_new, den));
    c.p = fmaT(beta, p, u_i);
    c.s = fmaT(beta, s_, w_i);
    c.sg = fmaT(beta, sg, w_g);
    return c;
  };
  // returns whether the side keeps running
  auto commit = [&](const Cand &c, RegOut &out, uint32_t &iter, T eta_new, T rr, T &p, T &s_, T &sg, T &eta,
                    T &alpha, T (&last)[2]) -> bool {
    ++iter;
    last[0] = eta_new;
    last[1] = rr;
    if (c.conv) {
      out.status = GBDPCG_CONVERGED;
      return false;
    }
    if (c.nonfin) {
      out.status = GBDPCG_NONFINITE;
      return false;
    }
    if (c.brk) {
      out.status = GBDPCG_BREAKDOWN;
      return false;
    }
    alpha = c.alpha;
    eta = eta_new;
    p = c.p;
    s_ = c.s;
    if (it.ghost) sg = c.sg;
    return iter < max_iter;
  };
  // Both sides' vector work runs every iteration (a stopped side's results are
  // discarded and its state is frozen), so that the compiler can interleave the
  // two sides' matvecs, reductions and scalar chains.
  while (runA || runB) {
    if (it.owner) {
      const T xa = fmaT(alphaA, pA, xA), ra = fmaT(-alphaA, sA, rA_i);
      const T xb = fmaT(alphaB, pB, xB), rb = fmaT(-alphaB, sB, rB_i);
      if (runA) {
        xA = xa;
        rA_i = ra;
      }
      if (runB) {
        xB = xb;
        rB_i = rb;
      }
      rA[own_pos] = rA_i;
      rB[own_pos] = rB_i;
    }
    if (it.ghost) {
      const T ga = fmaT(-alphaA, sgA, rgA), gb = fmaT(-alphaB, sgB, rgB);
      if (runA) rgA = ga;
      if (runB) rgB = gb;
      rA[it.gpos] = rgA;
      rB[it.gpos] = rgB;
    }
    __syncthreads();
    uA_i = chunk_mv(it, mM, rA, it.act_u);
    uB_i = chunk_mv(it, mM, rB, it.act_u);
    if (it.act_u && c == 0) {
      uA[(m + 1) * nP + row] = uA_i;
      uB[(m + 1) * nP + row] = uB_i;
    }
    __syncthreads();
    wA_i = chunk_mv(it, mS, uA, it.act_w);
    wB_i = chunk_mv(it, mS, uB, it.act_w);
    // both edge blocks every exchange (a stopped side's are stale and unused):
    // the neighbours' gather waits for every slot of the current epoch
    it.publish_edge(wA_i, 2);
    it.publish_edge(wB_i, 2, VB);
    it.reduce_publish6(rA_i * uA_i, it.owner ? wA_i * uA_i : (T)0, rA_i * rA_i,
                       rB_i * uB_i, it.owner ? wB_i * uB_i : (T)0, rB_i * rB_i);
    if (!it.gather_pair(wA, wB, 2, tt)) {
      timed_out = true;
      break;
    }
    const T wgA = it.ghost ? wA[it.gpos] : (T)0;
    const T wgB = it.ghost ? wB[it.gpos] : (T)0;
    const Cand cA = cand(thrA, tt[0], tt[1], tt[2], wA_i, uA_i, wgA, pA, sA, sgA, etaA, alphaA);
    const Cand cB = cand(thrB, tt[3], tt[4], tt[5], wB_i, uB_i, wgB, pB, sB, sgB, etaB, alphaB);
    if (runA) runA = commit(cA, fo, iterA, tt[0], tt[2], pA, sA, sgA, etaA, alphaA, lastA);
    if (runB) runB = commit(cB, ao, iterB, tt[3], tt[5], pB, sB, sgB, etaB, alphaB, lastB);
  }
  fo.iters = (int)iterA;
  ao.iters = (int)iterB;
  fo.eta = (double)lastA[0];
  fo.rr = (double)lastA[1];
  ao.eta = (double)lastB[0];
  ao.rr = (double)lastB[1];
  if (timed_out) {
    fo.status = GBDPCG_TIMED_OUT;
    ao.status = GBDPCG_TIMED_OUT;
  } else {
    // lambda and g_gamma to HBM and, with one ghost knot each side, to LDS
    if (it.owner) {
      gptr(static_cast<T *>(d.lambda))[(size_t)kg * n + row] = xA;
      gptr(static_cast<T *>(d.ggamma))[(size_t)kg * n + row] = xB;
      it.lv[own_pos] = xA;
      it.xv[own_pos] = xB;
    }
    it.publish_edge(xB, 1);
    it.publish_edge(xA, 1, VB);
    it.reduce_publish6((T)0, (T)0, (T)0, (T)0, (T)0, (T)0);
    if (!it.gather_pair(it.xv, it.lv, 1, tt)) {
      timed_out = true;
      fo.status = GBDPCG_TIMED_OUT;
      ao.status = GBDPCG_TIMED_OUT;
    } else {
      write_gS<T, NS, NT>(static_cast<T *>(d.gS), it.xv, it.lv, it.a, K, it.N);
    }
  }
  __syncthreads();
  if (rank == 0 && t == 0 && d.result != nullptr) {
    gbdpcg_result res;
    res.iters = fo.iters;
    res.status = fo.status;
    res.adj_iters = ao.iters;
    res.adj_status = ao.status;
    res.eta = fo.eta;
    res.rr = fo.rr;
    res.adj_eta = ao.eta;
    res.adj_rr = ao.rr;
    *d.result = res;
  }
  if (timed_out && t == 0 && d.err != nullptr)
    __hip_atomic_store(d.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The same for two lanes per row: the even lane of a row works for side A, the odd
// one for side B.  Both take part in both sides' products (sides_mv); everything else
// of an iteration, which VALU issue bounds, is one instruction stream for the two
// sides: the vector updates, the reductions (three sums over the lanes of one parity
// each), the divisions and exit tests.  Each side runs the recurrence of its own
// solve; the sums of a row (quads) and of a wave come together in another order than
// reg_item's.  Against both sides in every lane, per iteration: 64 systems of n = 14
// N = 128 FP32 2.59 us (3.00), FP64 5.58 (6.53), one knot range of n = 28 FP64 without
// exchange 2.66 (3.20), all rounds of 32 systems of n = 28 N = 512 60.8 (65.6).
template <typename T, int NS, int NT>
__device__ __forceinline__ void reg_item_sides(const KSys &d, uint32_t rank, T *lds) {
  using R = RegItem<T, NS, NT>;
  constexpr int n = R::n, nP = R::nP, CW = R::CW;
  // matrix chunks in LDS ahead of the vectors: Pinv for the instances held to 128
  // VGPRs, S for the FP64 n = 28 instance at 512 threads (whose vectors need only 8
  // values of read-ahead)
  constexpr bool PLDS = pair_pinv_lds(sizeof(T), NT, false, NS), SLDS = pair_s_lds(sizeof(T), NT, false, NS);
  constexpr int SLP = PLDS ? NT : 0, SLS = SLDS ? pair_s_slots(NT, NS) : 0;
  T *mlds = lds;
  lds += (size_t)(SLP + SLS) * CW;
  R it;
  it.N = (int)d.N;
  it.G = (int)d.G;
  it.rank = (int)rank;
  it.a = (int)knot_begin(rank, d.G, d.N);
  it.b = (int)knot_begin(rank + 1, d.G, d.N);
  it.K = it.b - it.a;
  const int K = it.K;
  it.VL = (K + 4) * nP + (SLDS ? 8 : R::LPR * CW);
  it.slots = d.slots;
  it.tol = d.tol;
  it.rel = (d.flags & KF_REL) != 0;
  it.xcd = false;
  it.xcd_ok = (d.flags & KF_NOXCD) == 0;
  const int t = opaque_tid();
  it.q = t / R::LPR;
  it.c = t % R::LPR;
  it.i = t & 3;
  it.m = it.q / n;
  it.row = it.q - it.m * n;
  it.kg = it.a - 1 + it.m;
  it.act_u = it.m < K + 2;
  it.act_w = it.m >= 1 && it.m <= K;
  it.owner = it.act_w;
  it.ghost = it.q < 4 * n;
  it.set_edge_slots();
  {
    const int gk = it.q / n, gr = it.q - (it.q / n) * n;
    const int gj = gk < 2 ? gk : K + gk;
    it.gpos = gj * nP + gr;
  }
  // LDS: r, u, w of each side, lambda and g_gamma windows, 6 partials per wave
  T *rA = lds, *uA = rA + it.VL, *wA = uA + it.VL;
  const int vb = 3 * it.VL;  // from a vector of side A to that of side B
  it.xv = rA + 2 * vb;       // lambda0 window, later g_gamma with ghosts
  it.lv = it.xv + it.VL;     // lambda with ghosts (for g_S)
  it.wsum = it.lv + it.VL;
  it.tot = it.wsum + 6 * R::NWAVES;
  it.ctl = reinterpret_cast<int *>(it.tot + 8);
  const int total = (int)(it.tot + 8 - lds);

  const int m = it.m, row = it.row, c = it.c, kg = it.kg;
  const int own_pos = (m + 1) * nP + row;
  const int edge_off = c * 4 * n;  // this side's edge block
  T *rv = rA + c * vb, *uv = uA + c * vb, *wv = wA + c * vb;

  if (t == 0) {
    const uint32_t ea = (uint32_t)(xload(it.rec(0, it.rank)) >> 32);
    const uint32_t eb = (uint32_t)(xload(it.rec(1, it.rank)) >> 32);
    uint32_t base = (ea > eb ? ea : eb) + 1u;
    if (base > 0xFFF00000u) base = 1u;
    it.ctl[0] = 0;
    it.ctl[1] = (int)base;
  }
  for (int i = opaque_tid(); i < total; i += NT) lds[i] = (T)0;

  // the set-up's vector reads (initial guess window: (K + 2) n <= NT values, one
  // per thread; the side's right-hand side) issued with the matrix chunks
  const T *lam0 = static_cast<const T *>(d.lambda);
  const int wl = (K + 2) * n;
  T lam_pre = 0, b_i = 0;
  int lam_pos = -1;
  {
    const int i = opaque_tid();
    if (i < wl) {
      const int jj = i / n, e = i - jj * n;
      const int k = it.a - 1 + jj;
      if (k >= 0 && k < it.N) {
        lam_pre = gptr(lam0)[(size_t)k * n + e];
        lam_pos = (jj + 1) * nP + e;
      }
    }
    if (it.owner) b_i = gptr(static_cast<const T *>(c ? d.glambda : d.gamma))[(size_t)kg * n + row];
  }

  // a matrix kept in LDS goes there through registers (no barrier: a lane reads its
  // own values only)
  constexpr int MW = in_quads<T, NS>() ? 2 * quad_cols<NS>() : CW, V = 16 / (int)sizeof(T);
  static_assert(MW <= CW && MW % V == 0, "LDS slots of CW values, whole blocks");
  typedef T block_t __attribute__((ext_vector_type(V)));
  const int sslot = t - R::LPR * n;  // S: no slots for the ghost knots' lanes
  T mM[PLDS ? 1 : MW], mS[SLDS ? 1 : MW];
  auto to_lds = [&](const T(&v)[MW], int slots, int slot) {
#pragma unroll
    for (int j = 0; j < MW; j += V) {
      block_t e;
#pragma unroll
      for (int k = 0; k < V; ++k) e[k] = v[j + k];
      *reinterpret_cast<block_t *>(mlds + ((size_t)(j / V) * slots + slot) * V) = e;
    }
  };
  auto load = [&](T(&v)[MW], const void *mat, bool active) {
    if constexpr (in_quads<T, NS>())
      load_quad<T, NS>(v, static_cast<const T *>(mat), kg, row - (it.i >> 1), it.i, it.N, active);
    else
      load_fixed<T, NS, NT, CW>(v, static_cast<const T *>(mat), kg, row, c, it.N, active);
  };
  if constexpr (SLDS) {
    T tmp[MW];
    load(tmp, d.S, it.act_w);
    if (it.act_w) to_lds(tmp, SLS, sslot);
  }
  if constexpr (PLDS) {
    T tmp[MW];
    load(tmp, d.Pinv, it.act_u);
    to_lds(tmp, SLP, t);
  } else {
    load(mM, d.Pinv, it.act_u);
  }
  if constexpr (!SLDS) load(mS, d.S, it.act_w);
  __syncthreads();
  it.base = (uint32_t)it.ctl[1];
  it.seq = 0;
  if (lam_pos >= 0) it.xv[lam_pos] = lam_pre;
  for (int i = opaque_tid() + NT; i < wl; i += NT) {
    const int jj = i / n, e = i - jj * n;
    const int k = it.a - 1 + jj;
    if (k >= 0 && k < it.N) it.xv[(jj + 1) * nP + e] = gptr(lam0)[(size_t)k * n + e];
  }
  __syncthreads();

  RegOut out{0, GBDPCG_MAX_ITER, 0.0, 0.0};
  bool timed_out = false, run = true;
  T x_i = it.owner && c == 0 ? it.xv[own_pos] : (T)0;
  // r = rhs - S x (side B starts from x = 0: r = g_lambda); zero on lanes without an
  // own row, where it stays zero: only w'u needs a select below
  T r_i;
  {
    const T y = sides_mv<SLS>(it, mS, mlds, sslot, it.xv, it.xv, it.act_w);
    r_i = !it.owner ? (T)0 : c ? b_i : b_i - y;
  }
  if (it.owner) rv[own_pos] = r_i;
  it.publish_edge(r_i, 2, edge_off);
  it.reduce_publish_sides(it.owner ? b_i * b_i : (T)0, (T)0, (T)0, true);
  T tt[3];
  double thr = 0.0;
  T r_g = 0, p_i = 0, s_i = 0, s_g = 0, eta = 0, alpha = 0, u_i = 0, w_i = 0;
  T last_eta = 0, last_rr = 0;
  uint32_t iter = 0;
  const uint32_t max_iter = d.max_iter;
  if (!it.gather_sides(rA, rA + vb, 2, c, tt)) {
    timed_out = true;
  } else {
    // placement sums: side A's second and third
    const double sx = (double)uniform(it.tot[1]), sxx = (double)uniform(it.tot[2]);
    it.xcd = __builtin_amdgcn_readfirstlane((int)(it.xcd_ok && it.G > 1 && sx * sx == (double)it.G * sxx)) != 0;
    thr = it.rel ? it.tol * it.tol * (double)tt[0] : it.tol;
    r_g = it.ghost ? rv[it.gpos] : (T)0;
    u_i = sides_mv<SLP>(it, mM, mlds, t, rA, rA + vb, it.act_u);
    if (it.act_u) uv[own_pos] = u_i;
    __syncthreads();
    w_i = sides_mv<SLS>(it, mS, mlds, sslot, uA, uA + vb, it.act_w);
    it.publish_edge(w_i, 2, edge_off);
    it.reduce_publish_sides(r_i * u_i, it.owner ? w_i * u_i : (T)0, r_i * r_i);
    if (!it.gather_sides(wA, wA + vb, 2, c, tt)) timed_out = true;
  }
  if (!timed_out) {
    // initial checks (as in reg_item)
    const T delta = tt[1], rr = tt[2];
    eta = tt[0];
    p_i = u_i;
    s_i = w_i;
    s_g = it.ghost ? wv[it.gpos] : (T)0;
    alpha = delta != (T)0 ? eta / delta : (T)0;
    last_eta = eta;
    last_rr = rr;
    if (!finite_d((double)eta) || !finite_d((double)rr)) {
      out.status = GBDPCG_NONFINITE;
      run = false;
    } else if (eta == (T)0) {
      out.status = rr == (T)0 ? GBDPCG_CONVERGED : GBDPCG_BREAKDOWN;
      run = false;
    } else if (delta == (T)0 || !finite_d((double)alpha)) {
      out.status = GBDPCG_BREAKDOWN;
      run = false;
    }
    if (max_iter == 0) run = false;
  } else {
    run = false;
  }
  // A stopped side's lanes hold their state and go on forming (unused) products for
  // the exchange.  Every wave has lanes of both sides, so all of them, and all ranks,
  // leave the loop together.
  while (__builtin_amdgcn_ballot_w64(run) != 0) {
    if (run) {
      if (it.owner) {
        x_i = fmaT(alpha, p_i, x_i);
        r_i = fmaT(-alpha, s_i, r_i);
      }
      if (it.ghost) r_g = fmaT(-alpha, s_g, r_g);
    }
    if (it.owner) rv[own_pos] = r_i;
    if (it.ghost) rv[it.gpos] = r_g;
    __syncthreads();
    u_i = sides_mv<SLP>(it, mM, mlds, t, rA, rA + vb, it.act_u);
    if (it.act_u) uv[own_pos] = u_i;
    __syncthreads();
    w_i = sides_mv<SLS>(it, mS, mlds, sslot, uA, uA + vb, it.act_w);
    // a stopped side's edges are stale and unused: the neighbours' gather waits for
    // every slot of the current epoch
    it.publish_edge(w_i, 2, edge_off);
    it.reduce_publish_sides(r_i * u_i, it.owner ? w_i * u_i : (T)0, r_i * r_i);
    if (!it.gather_sides(wA, wA + vb, 2, c, tt)) {
      timed_out = true;
      break;
    }
    const T w_g = it.ghost ? wv[it.gpos] : (T)0;
    // as in reg_item: stop tests and next coefficients first, then one branch
    const T eta_new = tt[0], rr = tt[2];
    const bool conv = it.rel ? ((double)rr <= thr) : (__builtin_fabs((double)eta_new) < thr);
    const bool nonfin = !finite_t(eta_new);
    const T beta = qdiv(eta_new, eta);
    const T den = tt[1] - beta * qdiv(eta_new, alpha);
    const bool brk = den == (T)0 || !finite_t(den);
    const T alpha_new = qdiv(eta_new, den);
    if (run) {
      ++iter;
      last_eta = eta_new;
      last_rr = rr;
      if (conv || nonfin || brk) {
        out.status = conv ? GBDPCG_CONVERGED : nonfin ? GBDPCG_NONFINITE : GBDPCG_BREAKDOWN;
        run = false;
      } else {
        alpha = alpha_new;
        eta = eta_new;
        p_i = fmaT(beta, p_i, u_i);
        s_i = fmaT(beta, s_i, w_i);
        s_g = fmaT(beta, s_g, w_g);
        run = iter < max_iter;
      }
    }
  }
  if (!timed_out) {
    // lambda and g_gamma to HBM and, with one ghost knot each side, to LDS
    if (it.owner) {
      gptr(static_cast<T *>(c ? d.ggamma : d.lambda))[(size_t)kg * n + row] = x_i;
      (c ? it.xv : it.lv)[own_pos] = x_i;
    }
    it.publish_edge(x_i, 1, c ? 0 : 4 * n);
    it.reduce_publish_sides((T)0, (T)0, (T)0);
    if (!it.gather_sides(it.xv, it.lv, 1, c, tt))
      timed_out = true;
    else
      write_gS<T, NS, NT>(static_cast<T *>(d.gS), it.xv, it.lv, it.a, K, it.N);
  }
  if (timed_out) out.status = GBDPCG_TIMED_OUT;
  __syncthreads();
  if (t < 64) {
    // side A's outcome is in lane 0, side B's in lane 1
    const int status = out.status, iters = (int)iter;
    gbdpcg_result res;
    res.iters = __builtin_amdgcn_readlane(iters, 0);
    res.status = __builtin_amdgcn_readlane(status, 0);
    res.adj_iters = __builtin_amdgcn_readlane(iters, 1);
    res.adj_status = __builtin_amdgcn_readlane(status, 1);
    res.eta = (double)read_lane(last_eta, 0);
    res.rr = (double)read_lane(last_rr, 0);
    res.adj_eta = (double)read_lane(last_eta, 1);
    res.adj_rr = (double)read_lane(last_rr, 1);
    if (rank == 0 && t == 0 && d.result != nullptr) *d.result = res;
  }
  if (timed_out && t == 0 && d.err != nullptr)
    __hip_atomic_store(d.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

// NS > 0: the kernel is specialised for stateSize NS.  NS == -1: runtime dispatch
// over the specialised sizes up to 14 (FP64 batches that mix them).
template <typename T, int NS, int NT, bool FUSED, bool BC>
__device__ __forceinline__ void reg_dispatch(const KSys &d, uint32_t rank, T *lds) {
  if constexpr (NS > 0) {
    reg_item<T, NS, NT, FUSED, BC>(d, rank, lds);
  } else if constexpr (BC) {
    switch (d.n) {
      case 12: reg_item<T, 12, NT, FUSED, true, true, false>(d, rank, lds); break;
      case 14: reg_item<T, 14, NT, FUSED, true, true, false>(d, rank, lds); break;
      default: break;  // the planner only admits the sizes above
    }
  } else {
    switch (d.n) {
      case 2: reg_item<T, 2, NT, FUSED, false, true, false>(d, rank, lds); break;
      case 6: reg_item<T, 6, NT, FUSED, false, true, false>(d, rank, lds); break;
      case 12: reg_item<T, 12, NT, FUSED, false, true, false>(d, rank, lds); break;
      case 14: reg_item<T, 14, NT, FUSED, false, true, false>(d, rank, lds); break;
      default: break;  // the planner only admits the sizes above
    }
  }
}

// Single system (systems == nullptr): workgroup b is rank b/stride when
// b % stride == 0.  Batched: items[round * gridDim.x + b] as in pcg_kernel.
template <typename T, int NS, int NT, bool FUSED, bool BC>
__device__ __forceinline__ void reg_entry(const KSys &one, const KSys *__restrict__ systems,
                                          const uint32_t *__restrict__ items, uint32_t rounds, uint32_t stride) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  T *lds = reinterpret_cast<T *>(lds_raw);
  if (systems == nullptr) {
    if (blockIdx.x % stride) return;
    const uint32_t rank = blockIdx.x / stride;
    if (rank >= one.G) return;
    reg_dispatch<T, NS, NT, FUSED, BC>(one, rank, lds);
    return;
  }
  for (uint32_t rd = 0; rd < rounds; ++rd) {
    const uint32_t item = items[(size_t)rd * gridDim.x + blockIdx.x];
    if (item == kNoItem) continue;
    __syncthreads();
    const KSys d = systems[item >> 12];
    reg_dispatch<T, NS, NT, FUSED, BC>(d, item & 0xFFFu, lds);
  }
}

// Waves per SIMD the column-chunk kernel is compiled for: the FP32 instances
// for rows of n <= 14 at 512 threads are held to 128 VGPRs, so that two workgroups
// share a CU in batch plans and long single solves (the planners count on it).
template <typename T, int NS, int NT>
constexpr int reg_waves_per_eu() {
  return (sizeof(T) == 4 && NT == 512 && NS <= 14) ? 4 : 1;
}

// Register-resident rows, reg_lpr(n) lanes per row, column chunks.
template <typename T, int NS, int NT, bool FUSED>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(reg_waves_per_eu<T, NS, NT>())))
pcg_reg_kernel(KSys one, const KSys *__restrict__ systems,
                                                     const uint32_t *__restrict__ items, uint32_t rounds,
                                                     uint32_t stride) {
  reg_entry<T, NS, NT, FUSED, false>(one, systems, items, rounds, stride);
}

// Register-resident rows, row-broadcast layout (n in {12, 14}): one lane per row,
// 16 lanes per knot, the vector window broadcast within each 16-lane row by DPP.
template <typename T, int NS, int NT, bool FUSED>
__global__ void __launch_bounds__(NT) pcg_rowcast_kernel(KSys one, const KSys *__restrict__ systems,
                                                         const uint32_t *__restrict__ items, uint32_t rounds,
                                                         uint32_t stride) {
  reg_entry<T, NS, NT, FUSED, true>(one, systems, items, rounds, stride);
}

// Paired forward + adjoint items (fused recurrence, both flags set) go to
// reg_item_sides or reg_item_pair, every other item to reg_item.
template <typename T, int NS, int NT, bool BC>
__device__ __forceinline__ void pair_item(const KSys &d, uint32_t rank, T *lds) {
  if ((d.flags & (KF_FWD | KF_ADJ)) == (KF_FWD | KF_ADJ) && (d.flags & KF_FUSED)) {
    if constexpr (!BC && RegItem<T, NS, NT>::LPR == 2)
      reg_item_sides<T, NS, NT>(d, rank, lds);
    else
      reg_item_pair<T, NS, NT, BC>(d, rank, lds);
  } else if constexpr (pair_s_lds(sizeof(T), NT, BC, NS)) {
    // instances with S in LDS run paired items only (plans route no other item
    // to them): flag the launch rather than skip the item silently
    if (threadIdx.x == 0 && d.err != nullptr) __hip_atomic_store(d.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  } else {
    reg_item<T, NS, NT, true, BC, false>(d, rank, lds);
  }
}

template <typename T, int NS, int NT, bool BC>
__device__ __forceinline__ void pair_dispatch(const KSys &d, uint32_t rank, T *lds) {
  if constexpr (NS > 0) {
    pair_item<T, NS, NT, BC>(d, rank, lds);
  } else if constexpr (BC) {
    switch (d.n) {
      case 12: pair_item<T, 12, NT, true>(d, rank, lds); break;
      case 14: pair_item<T, 14, NT, true>(d, rank, lds); break;
      default: break;
    }
  } else {
    switch (d.n) {  // runtime-n paired plans hold rows of n <= 14 only
      case 2: pair_item<T, 2, NT, false>(d, rank, lds); break;
      case 6: pair_item<T, 6, NT, false>(d, rank, lds); break;
      case 12: pair_item<T, 12, NT, false>(d, rank, lds); break;
      case 14: pair_item<T, 14, NT, false>(d, rank, lds); break;
      default: break;
    }
  }
}

// Waves per SIMD the paired kernel is compiled for: FP32 column-chunk rows of
// n <= 14 (and the runtime-n instance, which holds those sizes only) at 512
// threads are held to 128 VGPRs, so that two workgroups share a
// CU (a batch of 64 systems of N = 128 then runs in one round); the compiler
// spills what does not fit.
template <typename T, int NS, int NT, bool BC>
constexpr int pair_waves_per_eu() {
  return (sizeof(T) == 4 && NT == 512 && !BC && NS <= 14) ? 4 : 1;
}

// Forward + adjoint solves iterated together (see reg_item_pair); same launch
// interface as pcg_reg_kernel.
template <typename T, int NS, int NT, bool BC>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(pair_waves_per_eu<T, NS, NT, BC>())))
pcg_pair_kernel(KSys one, const KSys *__restrict__ systems,
                                                      const uint32_t *__restrict__ items, uint32_t rounds,
                                                      uint32_t stride) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  T *lds = reinterpret_cast<T *>(lds_raw);
  if (systems == nullptr) {
    if (blockIdx.x % stride) return;
    const uint32_t rank = blockIdx.x / stride;
    if (rank >= one.G) return;
    pair_dispatch<T, NS, NT, BC>(one, rank, lds);
    return;
  }
  for (uint32_t rd = 0; rd < rounds; ++rd) {
    const uint32_t item = items[(size_t)rd * gridDim.x + blockIdx.x];
    if (item == kNoItem) continue;
    __syncthreads();
    const KSys d = systems[item >> 12];
    pair_dispatch<T, NS, NT, BC>(d, item & 0xFFFu, lds);
  }
}

// Any stateSize up to 32: an item runs as the class of its padded size (n
// rounded up to 4), any_lpr lanes per row.  Bound by the same chain of on-chip
// latencies as the fixed sizes; a class costs the multiply-adds and registers of
// its padding only.  Against the LDS-resident kernel, which ran these sizes (one
// solve on several workgroups, microseconds per iteration): n = 13 N = 50 FP32 reference form 2.35
// (4.1), fused 1.61 (2.9), FP64 3.31 (4.2) and 2.15 (3.2); n = 24 N = 60 FP32
// 2.65 (4.1) and 1.78 (3.5); a batch of 96 systems of ten sizes n <= 31, FP32
// reference form, 135 us (1,081).  SET names the classes one kernel
// holds and with them its registers: the tiny and narrow ones serve systems of
// n <= 8 and n <= 16, the wide one larger ones, kAnyAll batches of mixed sizes.
template <typename T, int NT, bool FUSED, int SET, bool ALONE>
__device__ __forceinline__ void any_class(const KSys &d, uint32_t rank, T *lds) {
  constexpr int LP = any_lpr(SET, (int)sizeof(T));
  constexpr bool kLow = SET != kAnyWide, kMid = SET != kAnyTiny && SET != kAnyWide,
                 kHigh = SET == kAnyWide || SET == kAnyAll;
  switch (padded_n(d.n)) {
    case 4: if constexpr (kLow) reg_item<T, 4, NT, FUSED, false, true, true, LP, ALONE>(d, rank, lds); break;
    case 8: if constexpr (kLow) reg_item<T, 8, NT, FUSED, false, true, true, LP, ALONE>(d, rank, lds); break;
    case 12: if constexpr (kMid) reg_item<T, 12, NT, FUSED, false, true, true, LP, ALONE>(d, rank, lds); break;
    case 16: if constexpr (kMid) reg_item<T, 16, NT, FUSED, false, true, true, LP, ALONE>(d, rank, lds); break;
    case 20: if constexpr (kHigh) reg_item<T, 20, NT, FUSED, false, true, true, LP, ALONE>(d, rank, lds); break;
    case 24: if constexpr (kHigh) reg_item<T, 24, NT, FUSED, false, true, true, LP, ALONE>(d, rank, lds); break;
    case 28: if constexpr (kHigh) reg_item<T, 28, NT, FUSED, false, true, true, LP, ALONE>(d, rank, lds); break;
    case 32: if constexpr (kHigh) reg_item<T, 32, NT, FUSED, false, true, true, LP, ALONE>(d, rank, lds); break;
    default: break;  // the planner only admits the sizes above
  }
}

// Instances that hold systems of one workgroup, of several, or both (internal.h).
template <typename T, int NT, bool FUSED, int SET>
__device__ __forceinline__ void any_dispatch(const KSys &d, uint32_t rank, T *lds) {
  if constexpr (SET == kAnyLong && sizeof(T) == 4) {
    switch (padded_n(d.n)) {
      case 4: two_rows_item<4, NT, FUSED>(d, lds); break;
      case 8: two_rows_item<8, NT, FUSED>(d, lds); break;
      case 12: two_rows_item<12, NT, FUSED>(d, lds); break;
      case 16: two_rows_item<16, NT, FUSED>(d, lds); break;
      default: break;
    }
  } else if constexpr (!any_alone(SET)) {
    any_class<T, NT, FUSED, SET, false>(d, rank, lds);
  } else if constexpr (SET == kAnyTiny || SET == kAnyLong) {
    any_class<T, NT, FUSED, SET, true>(d, rank, lds);
  } else if (d.G == 1) {
    any_class<T, NT, FUSED, SET, true>(d, rank, lds);
  } else {
    any_class<T, NT, FUSED, SET, false>(d, rank, lds);
  }
}

// Waves per SIMD: kAnyRows is held to three (FP32) or two (FP64) workgroups of 256
// threads per CU.
template <typename T, int SET>
constexpr int any_waves_per_eu() {
  return SET == kAnyRows ? (sizeof(T) == 4 ? 3 : 2) : 1;
}

template <typename T, int NT, bool FUSED, int SET>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(any_waves_per_eu<T, SET>())))
pcg_any_kernel(KSys one, const KSys *__restrict__ systems, const uint32_t *__restrict__ items, uint32_t rounds,
               uint32_t stride) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  T *lds = reinterpret_cast<T *>(lds_raw);
  if (systems == nullptr) {
    if (blockIdx.x % stride) return;
    const uint32_t rank = blockIdx.x / stride;
    if (rank >= one.G) return;
    any_dispatch<T, NT, FUSED, SET>(one, rank, lds);
    return;
  }
  for (uint32_t rd = 0; rd < rounds; ++rd) {
    const uint32_t item = items[(size_t)rd * gridDim.x + blockIdx.x];
    if (item == kNoItem) continue;
    __syncthreads();
    const KSys d = systems[item >> 12];
    any_dispatch<T, NT, FUSED, SET>(d, item & 0xFFFu, lds);
  }
}

}  // namespace gbdpcg
