#pragma once

#include "spk_fft_core.hpp"

namespace spk {

// ---------------------------------------------------------------------------
// Transforms of the resident kernels: T = N/8 threads per line, 8 values each,
// two thread mappings.  In the coalesced mapping (line tid % TT, t = tid / TT)
// a wavefront covers all lines of the band: the mapping of the Phi loads and
// stores.  In the private mapping the threads of one line (N <= 512), or of
// the even or the odd samples of one line (N = 1024: the first three stages
// are two independent 512-point transforms, the last radix-2 stage combines
// them), lie in one wavefront, so their LDS exchanges need no workgroup
// barrier and the two wavefronts of a SIMD overlap one's exchanges with the
// other's butterflies.  A phase loads coalesced, runs its first transform into
// the private mapping, its pointwise work there, and its second transform back
// into the coalesced one: 3 barriers at 1024 and 2 below instead of 6 and 4.
// Butterflies, twiddles and their order are stage_butterflies', so values are
// the pass kernels' bit for bit.  A thread's twiddles do not change during a
// launch and stay in registers.  LEAN (128 registers per thread, four
// wavefronts per SIMD) reads them from the table in LDS at each stage and
// makes both private exchanges in one region.
//
// The CPU test suite runs this code too, a host thread for each of a
// workgroup's (tests/emu/line_emu.cpp, which defines threadIdx, __syncthreads
// and wave_lds_order).
// ---------------------------------------------------------------------------
// orders a wavefront's LDS writes before its reads (the hardware keeps a
// wavefront's LDS accesses in order)
#if defined(__HIPCC__)
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
#else
void wave_lds_order();
#endif

template <int N, int TT, bool LEAN = false>
struct LineFft {
  static constexpr int E = 8, T = N / E;
  static constexpr bool SPLIT = T > 64;              // even and odd samples apart
  static constexpr int TW = SPLIT ? 64 : T;          // lanes of a sub-transform
  static constexpr int M = E * TW;                   // its length
  static constexpr int SUBS = N * TT / M;            // sub-transforms of a workgroup
  using P = RadixPlan<M, E>;
  static constexpr int S = P::kStages;               // 2 or 3: 8, 8[, 8 or less]
  static_assert(T <= 128 && S >= 2 && S <= 3, "64 <= N <= 1024");
  // LDS: a chunk of each region per sub-transform (c32 slots)
  static constexpr int CHA = M + M / 8 + 2;          // e -> e + e / 8
  static constexpr int CHB = S == 3 && !LEAN ? M + M / 8 : 0;   // e -> e + 8 (e / 64)
  static constexpr int HALF = M / 2 + 16;            // even, then odd values
  static constexpr int CHC = SPLIT ? 2 * HALF : 0;
  static constexpr int LDS = SUBS * (CHA + CHB + CHC);

  int cb, ct;     // coalesced mapping: line, t
  int pb, pt;     // private mapping: line, natural t (values pt + i T)
  int sub, l;     // sub-transform and lane in it
  c32* a0;        // coalesced thread's first slot of the first exchange
  c32* a;         // private chunks
  c32* b;
  c32* c;
  c32* cline;     // region C of this line
  const c32* fa;  // coalesced thread's read base of the last exchange
  const c32* table;               // the staged twiddle table
  static constexpr int REG = LEAN ? 0 : 1;
  c32 w1[REG ? 7 : 1];                      // stage 1
  c32 w2[REG && S == 3 ? 7 : 1];            // stage 2 (entries by butterfly, then value)
  c32 w3[REG && SPLIT ? 4 : 1], w3c[REG && SPLIT ? 4 : 1], w2c[REG && !SPLIT && S == 3 ? 7 : 1];
  c32 w1c[REG && S == 2 ? 7 : 1];

  template <int ST>
  static __device__ __forceinline__ void load_tw(c32* w, const c32* twl, int t) {
    // entries of stage ST for the butterflies t + q T of a thread
    constexpr int R = plan_radix(N, E, ST), NS = RadixPlan<N, E>::span(ST), Q = E / R;
    constexpr int STEP = ST == RadixPlan<N, E>::kStages - 1 ? T : TW;
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int r = 1; r < R; ++r)
        w[q * (R - 1) + r - 1] =
            twl[staged_tw_offset(N, E, ST) + ((t + q * STEP) & (NS - 1)) * (R - 1) + r - 1];
  }
  // stage ST with its twiddles: those of registers w, or the table's for t
  template <int ST, bool INV>
  __device__ __forceinline__ void stage(c32 (&x)[E], const c32* w, int t) const {
    constexpr int R = plan_radix(N, E, ST);
    if constexpr (LEAN) {
      c32 u[(E / R) * (R - 1)];
      load_tw<ST>(u, table, t);
      butterflies<R, INV>(x, u);
    } else {
      butterflies<R, INV>(x, w);
    }
  }
  __device__ __forceinline__ void init(c32* lds, const c32* twl) {
    const int tid = threadIdx.x;
    cb = tid % TT;
    ct = tid / TT;
    sub = tid / TW;
    l = tid % TW;
    pb = SPLIT ? sub / 2 : sub;
    pt = SPLIT ? 2 * l + (sub & 1) : l;
    a = lds + sub * CHA;
    table = twl;
    b = LEAN ? a : lds + SUBS * CHA + sub * CHB;
    c = lds + SUBS * (CHA + CHB) + sub * CHC;
    cline = lds + SUBS * (CHA + CHB) + 2 * pb * CHC;
    const int csub = SPLIT ? 2 * cb + (ct & 1) : cb, cl = SPLIT ? ct >> 1 : ct;
    a0 = lds + csub * CHA + 9 * cl;
    if constexpr (SPLIT) fa = lds + 2 * cb * CHA;
    else if constexpr (S == 3) fa = LEAN ? lds + cb * CHA : lds + SUBS * CHA + cb * CHB;
    else fa = lds + cb * CHA;
    if constexpr (LEAN) return;
    load_tw<1>(w1, twl, l);
    if constexpr (S == 3) load_tw<2>(w2, twl, l);
    if constexpr (SPLIT) {
      load_tw<3>(w3, twl, pt);
      load_tw<3>(w3c, twl, ct);
    } else if constexpr (S == 3) {
      load_tw<2>(w2c, twl, ct);
    } else {
      load_tw<1>(w1c, twl, ct);
    }
  }
  // butterflies of a stage of radix R on the thread's registers
  template <int R, bool INV>
  static __device__ __forceinline__ void butterflies(c32 (&x)[E], const c32* w) {
    constexpr int Q = E / R;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      c32 v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = x[q + r * Q];
      if (w) {
#pragma unroll
        for (int r = 1; r < R; ++r) v[r] = twiddle<INV>(v[r], w[q * (R - 1) + r - 1]);
      }
      dft<R, INV>(v);
#pragma unroll
      for (int r = 0; r < R; ++r) x[q + r * Q] = v[r];
    }
  }
  __device__ __forceinline__ void put_a(const c32 (&x)[E], c32* p) const {
#pragma unroll
    for (int r = 0; r < E; ++r) p[r] = x[r];
  }
  __device__ __forceinline__ void get_a(c32 (&x)[E]) const {
    const c32* p = a + l + (l >> 3);
#pragma unroll
    for (int q = 0; q < E; ++q) x[q] = p[q * (TW + TW / 8)];
  }
  // slot of value e = t + q step of a B chunk
  static __device__ __forceinline__ int slot_b(int e) { return e + 8 * (e >> 6); }
  __device__ __forceinline__ void put_b(const c32 (&x)[E]) const {
    c32* p = b + 72 * (l >> 3) + (l & 7);   // (l / 8) 64 + l % 8 + 8 r
#pragma unroll
    for (int r = 0; r < E; ++r) p[8 * r] = x[r];
  }
  __device__ __forceinline__ void get_b(c32 (&x)[E]) const {
#pragma unroll
    for (int q = 0; q < E; ++q) x[q] = b[slot_b(l + q * TW)];
  }
  // stages 1 .. of the sub-transform in the private mapping, after the first
  // exchange; last = false leaves out the final stage of the plan below 1024
  template <bool INV>
  __device__ __forceinline__ void middle(c32 (&x)[E]) {
    get_a(x);
    stage<1, INV>(x, w1, l);
    if constexpr (S == 3) {
      if constexpr (LEAN) wave_lds_order();   // a chunk is read before it is written
      put_b(x);
      wave_lds_order();
      get_b(x);
      stage<2, INV>(x, w2, l);
    }
  }
  // coalesced values ct + i T of line cb -> transform at pt + i T of line pb
  template <bool INV>
  __device__ __forceinline__ void to_private(c32 (&x)[E]) {
    butterflies<8, INV>(x, nullptr);
    put_a(x, a0);
    __syncthreads();
    middle<INV>(x);
    if constexpr (SPLIT) {
#pragma unroll
      for (int r = 0; r < E; ++r) c[(l & 1) * HALF + (l >> 1) + 32 * r] = x[r];   // l + 64 r
      __syncthreads();
      const c32* p = cline + (pt & 1) * HALF + l;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        x[q] = p[64 * q];
        x[q + 4] = p[CHC + 64 * q];
      }
      stage<3, INV>(x, w3, pt);
    }
  }
  // values pt + i T of line pb -> the same values at ct + i T of line cb
  template <class HOOK>
  __device__ __forceinline__ void spread(c32 (&x)[E], HOOK before_barrier) {
    // slot of value v of a line: its chunks of region A one after the other
    auto slot = [](int line, int v) {
      return (SPLIT ? 2 * line + v / M : line) * CHA + v % M + (v % M) / 8;
    };
    c32* base = a - sub * CHA;
#pragma unroll
    for (int i = 0; i < E; ++i) base[slot(pb, pt + i * T)] = x[i];
    before_barrier();
    __syncthreads();
#pragma unroll
    for (int i = 0; i < E; ++i) x[i] = base[slot(cb, ct + i * T)];
  }
  // values pt + i T of line pb -> transform at ct + i T of line cb
  template <bool INV, class HOOK>
  __device__ __forceinline__ void to_coalesced(c32 (&x)[E], HOOK before_barrier) {
    butterflies<8, INV>(x, nullptr);
    put_a(x, a + 9 * l);
    if constexpr (SPLIT) {
      wave_lds_order();
      middle<INV>(x);
      c32* p = a + l + (l >> 3);
#pragma unroll
      for (int r = 0; r < E; ++r) p[72 * r] = x[r];   // l + 64 r
      before_barrier();
      __syncthreads();
      const c32* g = fa + ct + (ct >> 3);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        x[q] = g[144 * q];
        x[q + 4] = g[CHA + 144 * q];
      }
      stage<3, INV>(x, w3c, ct);
    } else if constexpr (S == 3) {
      wave_lds_order();
      get_a(x);
      stage<1, INV>(x, w1, l);
      if constexpr (LEAN) wave_lds_order();   // a chunk is read before it is written
      put_b(x);
      before_barrier();
      __syncthreads();
#pragma unroll
      for (int q = 0; q < E; ++q) x[q] = fa[slot_b(ct + q * T)];
      stage<2, INV>(x, w2c, ct);
    } else {
      before_barrier();
      __syncthreads();
      const c32* g = fa + ct + (ct >> 3);
#pragma unroll
      for (int q = 0; q < E; ++q) x[q] = g[q * (T + T / 8)];
      stage<1, INV>(x, w1c, ct);
    }
  }
};

}  // namespace spk
