// Slabs of a matrix from global memory to LDS, two in flight in registers while one is used:
// the operand loader and the loop of the small-tile products (gemm_tile.hpp), the exact
// column sums beside them and the row reductions (ops.hip).
//
// A slab is T rows (or columns) of KS = 4096 / T k-values, 16 KiB, four float4 per thread of a
// 256-thread block whatever T is.  Every load in the loop is unconditional: addresses past
// the matrix are clamped into it, and what lies past the k range becomes `fill` when the slab
// is stored to LDS.  A loop without branches around loads keeps the waits exact (the wait
// before an LDS store leaves the next slab's loads in flight) and the code short, which
// matters for launches of a few microseconds.
//
// Matrices need no alignment beyond their floats' own (UA): the hardware takes 16-byte loads
// at 4-byte addresses.  In a row-major ("mn-fast") matrix a group of four columns may then
// run past the row's end into the next row, whose values only feed columns that are never
// stored; only in the very last row is it moved back to the matrix's end and shifted into
// place, as is the last group of a k-fast row when K is not a multiple of 4.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace orca_hip {
namespace {

// Native 4-float vector: copies stay SSA values (HIP's float4 struct copies
// lower to memcpy, which can pin a register stage in scratch).
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef floatx4 floatx4_u __attribute__((aligned(4)));

// The four floats that start d places into v (d = 0 .. 3; the rest is don't care).
__device__ __forceinline__ floatx4 shift_down(floatx4 v, int d) {
  floatx4 x;
  x.x = d == 0 ? v.x : d == 1 ? v.y : d == 2 ? v.z : v.w;
  x.y = d == 0 ? v.y : d == 1 ? v.z : v.w;
  x.z = d == 0 ? v.z : v.w;
  x.w = v.w;
  return x;
}

template <int T, bool KFAST, bool UA>
struct TileOperand {
  static constexpr int KS = 4096 / T;                 // k-values per slab
  static constexpr int PITCH = KS + 4;                // floats per k-fast LDS row
  static constexpr int GAP = T < 32 ? T : 32;         // mn-fast: extra floats per 16 rows, so the k groups of a
                                                      // fragment read lie in different banks
  static constexpr int FLOATS = KFAST ? T * PITCH : KS * T + (KS / 16) * GAP;
  static constexpr int RSTEP = 1024 / T;              // mn-fast: k rows between a thread's float4s

  const char* base;   // uniform
  uint32_t voff[4];   // byte offsets of this thread's float4s (k-fast: without the k part)
  uint32_t limit;     // mn-fast: the largest byte offset a load may have
  uint32_t step;      // mn-fast: bytes per slab
  int k0;             // this thread's k in slab 0 (mn-fast: of its first float4)
  int K, kend;        // k-values of the operand; end of this block's range
  int dlast;          // mn-fast: places the last row's group is moved back

  static __device__ __forceinline__ int mn_off(int k) { return k * T + (k >> 4) * GAP; }

  // Rows and column groups past `lim` (M or N) become the last valid one.
  __device__ __forceinline__ void init(const float* src, int64_t ld, int row0, int lim, int kb, int kend_, int K_) {
    const int tid = threadIdx.x;
    base = reinterpret_cast<const char*>(src);
    K = K_;
    kend = kend_;
    if (KFAST) {
      k0 = kb + (tid % (KS / 4)) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        voff[j] = (uint32_t)((int64_t)min(row0 + (tid + 256 * j) / (KS / 4), lim - 1) * ld * 4);
    } else {
      const int c = min(row0 + (tid % (T / 4)) * 4, (lim - 1) & ~3);
      k0 = kb + tid / (T / 4);
      dlast = UA ? max(0, c + 4 - lim) : 0;
      limit = (uint32_t)(((int64_t)(K - 1) * ld + c - dlast) * 4);
      step = (uint32_t)(KS * ld * 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) voff[j] = (uint32_t)(((int64_t)(k0 + RSTEP * j) * ld + c) * 4);
    }
  }
  __device__ __forceinline__ void load(int t, floatx4 (&r)[4]) const {
    const uint32_t kc = KFAST ? (uint32_t)min(k0 + t * KS, K - 4) * 4u : 0u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t off = KFAST ? voff[j] + kc : min(voff[j] + (uint32_t)t * step, limit);
      if (UA)
        r[j] = *reinterpret_cast<const floatx4_u*>(base + off);
      else
        r[j] = *reinterpret_cast<const floatx4*>(base + off);
    }
  }
  // Slab t from registers to LDS.  LAST: it may be the block's last slab, `fill` from
  // kend on (and, UA, shifted where its load was moved back into the operand).
  template <bool LAST>
  __device__ __forceinline__ void store(int t, const floatx4 (&r)[4], float* __restrict__ s, float fill = 0.0f) const {
    const int tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      floatx4 v = r[j];
      if (KFAST) {
        const int k = k0 + t * KS;
        if (LAST && UA) {
          v = shift_down(v, max(0, k - (K - 4)));
          v.x = k < kend ? v.x : fill;
          v.y = k + 1 < kend ? v.y : fill;
          v.z = k + 2 < kend ? v.z : fill;
          v.w = k + 3 < kend ? v.w : fill;
        } else if (LAST) {
          v = k < kend ? v : floatx4{fill, fill, fill, fill};
        }
        const int idx = tid + 256 * j;
        *reinterpret_cast<floatx4*>(s + idx / (KS / 4) * PITCH + idx % (KS / 4) * 4) = v;
      } else {
        const int k = k0 + t * KS + RSTEP * j;
        if (LAST && UA) v = shift_down(v, k == K - 1 ? dlast : 0);
        if (LAST) v = k < kend ? v : floatx4{fill, fill, fill, fill};
        *reinterpret_cast<floatx4*>(s + mn_off(tid / (T / 4) + RSTEP * j) + tid % (T / 4) * 4) = v;
      }
    }
  }
  // The HS k-values from kc on (kc % 16 + HS <= 16) of row (or column) `row`.
  template <int HS>
  static __device__ __forceinline__ void frag(const float* __restrict__ s, int row, int kc, float (&f)[HS]) {
    if (KFAST) {
      const float* p = s + row * PITCH + kc;
#pragma unroll
      for (int q = 0; q < HS / 4; ++q) {
        const floatx4 v = *reinterpret_cast<const floatx4*>(p + 4 * q);
        f[4 * q] = v.x;
        f[4 * q + 1] = v.y;
        f[4 * q + 2] = v.z;
        f[4 * q + 3] = v.w;
      }
    } else {
      const float* p = s + mn_off(kc) + row;
#pragma unroll
      for (int q = 0; q < HS; ++q) f[q] = p[q * T];
    }
  }
};

// Slabs 0 .. n - 1 through two register stages and two LDS buffers: while slab t is
// used, slab t + 1 moves from its stage to the other buffer and slab t + 3's loads go
// into that stage (slab t + 2's are in flight in the other one).
//   load(t, stage), store(t, stage, buffer, last) with stage, buffer and last as
//   integral constants; begin(): slab 0 is in buffer 0; use(t, buffer, mid, more) calls
//   mid() where it wants the store and the loads issued and, if more, the block's
//   barrier after which slab t + 1 is in the other buffer.
// The loop's own slabs are never the last ones: their stores go unchecked, and every
// load in it is unconditional (a load behind a branch would make the next store wait
// for every load in flight).
// ONE: there is one slab (and one buffer).
template <bool ONE, class Load, class Store, class Begin, class Use>
__device__ __forceinline__ void slab_pipeline(int n, Load load, Store store, Begin begin, Use use) {
  constexpr std::integral_constant<int, 0> S0;
  constexpr std::integral_constant<int, 1> S1;
  constexpr std::false_type MID;
  constexpr std::true_type LAST;
  if constexpr (ONE) {
    load(0, S0);
    store(0, S0, S0, LAST);
    __syncthreads();
    begin();
    use(0, S0, []() {}, false, MID);
    return;
  }
  if (n > 2) {
    load(0, S0);
    load(1, S1);
    store(0, S0, S0, MID);
    load(2, S0);
  } else {
    load(0, S0);
    if (n > 1) load(1, S1);
    store(0, S0, S0, LAST);
  }
  __syncthreads();
  begin();
  int t = 0;
  for (; t + 4 < n; t += 2) {
    use(t, S0, [&]() {
      store(t + 1, S1, S1, MID);
      load(t + 3, S1);
    }, true, LAST);
    use(t + 1, S1, [&]() {
      store(t + 2, S0, S0, MID);
      load(t + 4, S0);
    }, true, LAST);
  }
  // 1 .. 4 slabs left: t + 1 and t + 2 are in flight, t + 3 is not loaded yet
  use(t, S0, [&]() {
    if (t + 1 < n) store(t + 1, S1, S1, LAST);
    if (t + 3 < n) load(t + 3, S1);
  }, t + 1 < n, MID);
  if (t + 1 >= n) return;
  use(t + 1, S1, [&]() {
    if (t + 2 < n) store(t + 2, S0, S0, LAST);
  }, t + 2 < n, MID);
  if (t + 2 >= n) return;
  use(t + 2, S0, [&]() {
    if (t + 3 < n) store(t + 3, S1, S1, LAST);
  }, t + 3 < n, MID);
  if (t + 3 >= n) return;
  use(t + 3, S1, []() {}, false, MID);
}

}  // namespace
}  // namespace orca_hip
