// gfx950 (CDNA4) kernels of the DBD SpGEMM path: C = A * B, CSR, int64 row pointers,
// int32 column indices, FP32 or FP64 values.
//
// Reference kernels replaced (S/ = dbd/for_small_datasets/src/ of the reference):
//   calculate_UpperBound  S/preProc.cu:170-179   -> k_row_products (no atomics, int64)
//   rowproduct_* + merge  S/computeGPU.cu:135-329 -> k_symbolic_hash, k_numeric_wave[_fast],
//                                                   k_numeric_block, k_*_long
//   collect               S/computeGPU.cu:331-341 -> not needed: exact offsets come from the
//                                                   symbolic pass, numeric writes in place.
// Differences on purpose: first touch is detected by a key compare-and-swap (the reference
// tests |acc| < 1e-4, S/computeGPU.cu:311-312), A's values are not truncated to int
// (S/computeGPU.cu:140), columns are emitted sorted, and every count is 64-bit.
//
// Layout of work: rows are binned by a per-row key (symbolic: min(P_i, ncols); numeric:
// nnz_i). Each bin has a kernel shape (T hash slots in LDS, NT threads per row, G lanes per
// A entry). Rows above the largest LDS table go to window kernels that sweep the row's
// column range in LDS-sized windows with one cursor per A entry.
#include "kernels.h"

#include <algorithm>
#include <climits>
#include <utility>
#include <mutex>
#include <map>

namespace dbd {

constexpr int kEmpty = -1;

// ------------------------------------------------------------------------------------
// wave / group primitives
// ------------------------------------------------------------------------------------
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Wait until no vector memory operation of this wave is outstanding (s_waitcnt vmcnt(0); the
// other counters at their maximum). Placed at the end of rarely taken branches that issue
// loads, so the compiler's count of outstanding loads on the common path stays exact.
__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// 64-bit readlane of a wave-uniform lane index.
__device__ __forceinline__ int64_t readlane64(int64_t v, int lane) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)v >> 32), lane);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// A "group" is NT threads that own one row. NT <= 64: a (sub-)wave, synchronised with
// wave_sync (several groups per workgroup). NT > 64: the whole workgroup (__syncthreads).
template <int NT>
__device__ __forceinline__ void gsync() {
  if constexpr (NT <= 64)
    wave_sync();
  else
    __syncthreads();
}

struct OpMin {
  template <typename T>
  __device__ T operator()(T a, T b) const { return a < b ? a : b; }
};
struct OpMax {
  template <typename T>
  __device__ T operator()(T a, T b) const { return a > b ? a : b; }
};
struct OpOr {
  __device__ int operator()(int a, int b) const { return a | b; }
};
struct OpAdd {
  template <typename T>
  __device__ T operator()(T a, T b) const { return a + b; }
};

// Lane move within the wave by DPP control word, of a 4- or 8-byte value; lanes without a source
// keep `old`.
template <int CTRL, int ROWS = 0xF, int BANKS = 0xF, typename T>
__device__ __forceinline__ T dpp_mov(T old, T x) {
  if constexpr (sizeof(T) == 4) {
    return (T)__builtin_amdgcn_update_dpp((int)old, (int)x, CTRL, ROWS, BANKS, false);
  } else {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)(uint64_t)old, (int)(uint32_t)(uint64_t)x,
                                                              CTRL, ROWS, BANKS, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)((uint64_t)old >> 32),
                                                              (int)(uint32_t)((uint64_t)x >> 32), CTRL, ROWS, BANKS, false);
    return (T)(((uint64_t)hi << 32) | lo);
  }
}

template <int CTRL>
__device__ __forceinline__ double dpp_mov(double old, double x) {
  return __longlong_as_double(dpp_mov<CTRL>(__double_as_longlong(old), __double_as_longlong(x)));
}

template <typename T>
__device__ __forceinline__ T read_lane(T x, int lane) {
  if constexpr (sizeof(T) == 4)
    return (T)__builtin_amdgcn_readlane((int)x, lane);
  else
    return (T)readlane64((int64_t)x, lane);
}

// Whole-wave reduction of an integer without LDS: DPP within rows of 16 lanes (quad swaps, half
// mirror, mirror), then the four row results through readlane. All 64 lanes must be active.
template <typename T, typename Op>
__device__ __forceinline__ T wave_reduce_dpp(T x, Op op) {
  x = op(x, dpp_mov<0xB1>(x, x));   // quad_perm [1,0,3,2]
  x = op(x, dpp_mov<0x4E>(x, x));   // quad_perm [2,3,0,1]
  x = op(x, dpp_mov<0x141>(x, x));  // row_half_mirror
  x = op(x, dpp_mov<0x140>(x, x));  // row_mirror
  return op(op(read_lane(x, 0), read_lane(x, 16)), op(read_lane(x, 32), read_lane(x, 48)));
}

// Inclusive prefix sum over the wave with DPP: shifts of 1-3, 4 and 8 lanes inside each row of
// 16 lanes, then the row totals through the row broadcasts of lanes 15 and 31. All 64 lanes
// must be active.
template <typename T>
__device__ __forceinline__ T wave_incl_scan_dpp(T x) {
  T s = x + dpp_mov<0x111>(T(0), x);              // row_shr:1
  s += dpp_mov<0x112>(T(0), x);                   // row_shr:2
  s += dpp_mov<0x113>(T(0), x);                   // row_shr:3
  s += dpp_mov<0x114, 0xF, 0xE>(T(0), s);         // row_shr:4, lanes 4-15
  s += dpp_mov<0x118, 0xF, 0xC>(T(0), s);         // row_shr:8, lanes 8-15
  s += dpp_mov<0x142, 0xA, 0xF>(T(0), s);         // row_bcast:15 -> rows 1, 3
  s += dpp_mov<0x143, 0xC, 0xF>(T(0), s);         // row_bcast:31 -> rows 2, 3
  return s;
}

template <int NT>
struct Group {
  static_assert(NT >= 64, "whole waves");
  static constexpr int NW = NT / 64;

  template <typename T, typename Op>
  __device__ static T reduce(T v, Op op, T* sc) {
    v = wave_reduce_dpp(v, op);
    if constexpr (NT > 64) {
      const int t = threadIdx.x % NT;
      if ((t & 63) == 0) sc[t >> 6] = v;
      __syncthreads();
      v = sc[0];
#pragma unroll
      for (int i = 1; i < NW; ++i) v = op(v, sc[i]);
      __syncthreads();
    }
    return v;
  }

  // Exclusive prefix of v over the group; total returned through `total`.
  template <typename T>
  __device__ static T exscan(T v, T& total, T* sc) {
    const int t = threadIdx.x % NT;
    const T x = wave_incl_scan_dpp(v);
    if constexpr (NT <= 64) {
      total = read_lane(x, 63);
      return x - v;
    } else {
      const int lane = t & 63, wid = t >> 6;
      if (lane == 63) sc[wid] = x;
      __syncthreads();
      T pre = 0, tot = 0;
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        T s = sc[i];
        if (i < wid) pre += s;
        tot += s;
      }
      __syncthreads();
      total = tot;
      return pre + x - v;
    }
  }
};

// Mask of the G lanes (within this wave) that share this lane's subgroup.
template <int G>
__device__ __forceinline__ uint64_t subgroup_mask() {
  if constexpr (G >= 64) {
    return ~0ull;
  } else {
    const int first = (threadIdx.x & 63) & ~(G - 1);
    return ((1ull << G) - 1ull) << first;
  }
}

// Fibonacci hashing of a column into a power-of-two table.
template <int T>
__device__ __forceinline__ uint32_t hslot(int c) {
  constexpr int LOG = __builtin_ctz(T);
  return ((uint32_t)c * 2654435761u) >> (32 - LOG);
}

// Insert key c; returns 1 if this call created the entry, 0 if it was present, -1 if the
// table is full (cannot happen when the planner sized it; checked anyway, never spins).
template <int T>
__device__ __forceinline__ int hash_insert_key(int* hk, int c) {
  uint32_t h = hslot<T>(c);
#pragma unroll 1
  for (int probe = 0; probe < T; ++probe) {
    // compare-and-swap first: at load <= 1/2 most probes find the slot empty or holding c
    const int old = atomicCAS(hk + h, kEmpty, c);
    if (old == kEmpty) return 1;
    if (old == c) return 0;
    h = (h + 1) & (T - 1);
  }
  return -1;
}

template <typename V>
__device__ __forceinline__ void lds_add(V* p, V v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Insert-or-accumulate (c, v). Returns false only if the table is full.
template <int T, typename V>
__device__ __forceinline__ bool hash_insert_add(int* hk, V* hv, int c, V v) {
  uint32_t h = hslot<T>(c);
#pragma unroll 1
  for (int probe = 0; probe < T; ++probe) {
    const int old = atomicCAS(hk + h, kEmpty, c);
    if (old == kEmpty || old == c) {
      lds_add(hv + h, v);
      return true;
    }
    h = (h + 1) & (T - 1);
  }
  return false;
}

// Product sink of the hash kernels: tracks the column range, inserts keys (and accumulates
// values when VALS). With BATCH, batch() issues the first probe of all U products before
// looking at any result (U LDS compare-and-swaps in flight together); collisions then continue
// probing. Without it the products are inserted one after another. Sums are FP64 for FP32 products
// too: ds_add_f32 takes 194 clocks a wave, ds_add_f64 9 to 21.
template <int T, typename V, bool VALS, bool BATCH = true>
struct HashSink {
  int* K;
  double* H;
  int cmin = INT_MAX, cmax = -1, created = 0, bad = 0;
  __device__ __forceinline__ void probe_from(uint32_t h, int c, V v) {
#pragma unroll 1
    for (int probe = 1; probe < T; ++probe) {
      h = (h + 1) & (T - 1);
      const int old = atomicCAS(K + h, kEmpty, c);
      if (old == kEmpty || old == c) {
        created += (old == kEmpty);
        if (VALS) lds_add(H + h, (double)v);
        return;
      }
    }
    bad = 1;
  }
  template <int U>
  __device__ __forceinline__ void batch(const int (&c)[U], const V (&v)[U]) {
    if constexpr (!BATCH) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (c[u] >= 0) one(c[u], v[u]);
      return;
    }
    uint32_t h[U];
    int old[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      h[u] = hslot<T>(c[u]);
      old[u] = (c[u] >= 0) ? atomicCAS(K + h[u], kEmpty, c[u]) : 0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (c[u] < 0) continue;
      cmin = min(cmin, c[u]);
      cmax = max(cmax, c[u]);
      if (old[u] == kEmpty || old[u] == c[u]) {
        created += (old[u] == kEmpty);
        if (VALS) lds_add(H + h[u], (double)v[u]);
      } else {
        probe_from(h[u], c[u], v[u]);
      }
    }
  }
  __device__ __forceinline__ void one(int c, V v) {
    cmin = min(cmin, c);
    cmax = max(cmax, c);
    const uint32_t h = hslot<T>(c);
    const int old = atomicCAS(K + h, kEmpty, c);
    if (old == kEmpty || old == c) {
      created += (old == kEmpty);
      if (VALS) lds_add(H + h, (double)v);
    } else {
      probe_from(h, c, v);
    }
  }
};

// Lookup of a key known to be present; returns slot or -1.
template <int T>
__device__ __forceinline__ int hash_find(const int* hk, int c) {
  uint32_t h = hslot<T>(c);
#pragma unroll 1
  for (int probe = 0; probe < T; ++probe) {
    int cur = hk[h];
    if (cur == c) return (int)h;
    if (cur == kEmpty) return -1;
    h = (h + 1) & (T - 1);
  }
  return -1;
}

// Slots a lane owns in a one-wave row table of T slots (T/64 per lane): 16-byte chunks
// t, t + 64, ... (fewer slots per lane: the slots t*IPT ..), so a wide LDS access of the whole
// wave covers one contiguous block and hits every bank once.
template <int T>
__device__ __forceinline__ int slot_of(int t, int q) {
  constexpr int IPT = T / 64;
  constexpr int CW = IPT < 4 ? IPT : 4;
  return CW * ((q / CW) * 64 + t) + q % CW;
}

// Clear a one-wave row table (keys to kEmpty, values to 0) with contiguous 16-byte stores.
template <int T, typename V>
__device__ __forceinline__ void clear_table(int t, int* K, V* H) {
  if constexpr (T >= 256) {
#pragma unroll
    for (int c = 0; c < T / 256; ++c) reinterpret_cast<int4*>(K)[c * 64 + t] = make_int4(kEmpty, kEmpty, kEmpty, kEmpty);
  } else {
#pragma unroll
    for (int q = 0; q < T / 64; ++q) K[q * 64 + t] = kEmpty;
  }
  if (H) {
    constexpr int CH = T * (int)sizeof(V) / 16;  // 16-byte chunks of values
#pragma unroll
    for (int c = t; c < CH; c += 64) reinterpret_cast<int4*>(H)[c] = make_int4(0, 0, 0, 0);
  }
}

// Element-parallel walk over the spans of up to 64 entries, one per lane of a wave (`len` elements at
// `start`): extra(rank) stores what else the elements need of this lane's entry, at its rank among
// the entries with elements, and body(at, j) takes U elements per lane, element u of them at
// position at[u], of the entry of rank j[u] (at[u] < 0: none). The owner of a flattened element is
// not searched: the entries set a bit where their elements begin (bit S - 1 for the entry that
// starts at S >= 1, in words of 64 elements), and an element's owner is the number of bits before it,
// one mbcnt on a mask that readlane makes wave-uniform (a bisection over 64 starts costs 6
// dependent LDS reads per element). l: LDS of this wave's own. With w0 and wstep several waves that
// hold the same entries share the elements, U words at a time.
constexpr int kSpanWords = 32;
template <typename I>
struct SpanLdsT {  // I: holds positions in B
  I tb[64];
  unsigned long long wm[kSpanWords];
};
using SpanLds = SpanLdsT<int64_t>;
struct SpanKeep {  // for a second walk over the same spans: span_words(lane, *this, 0, ..) if T fits kSpanWords
  int T = 0, ex = 0;
  unsigned long long m = 0ull;
};
template <int U, typename I, typename F>
__device__ __forceinline__ void span_words(int lane, const SpanKeep& k, int g0, const SpanLdsT<I>& l, F&& body, int w0,
                                           int wstep) {
  const int words = min(kSpanWords, (k.T - g0 + 63) >> 6);
  for (int w = w0; w < words; w += wstep) {
    int64_t at[U];
    int j[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int wu = min(w + u, 63);
      const uint64_t mw = (uint64_t)readlane64((int64_t)k.m, wu);
      const int f = g0 + 64 * (w + u) + lane;
      const bool ok = w + u < words && f < k.T;
      const int o = __builtin_amdgcn_readlane(k.ex, wu) +
                    __builtin_amdgcn_mbcnt_hi((uint32_t)(mw >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mw, 0));
      j[u] = w + u < words ? o : 0;  // past the last element: its owner again
      at[u] = ok ? l.tb[j[u]] + (I)f : -1;
    }
    body(at, j);
  }
}
template <int U, typename I, typename X, typename F>
__device__ __forceinline__ SpanKeep walk_spans(int lane, int len, int64_t start, SpanLdsT<I>& l, X&& extra, F&& body,
                                               int w0 = 0, int wstep = U) {
  SpanKeep k;
  const uint64_t live = __builtin_amdgcn_ballot_w64(len > 0);
  if (!live) return k;
  const int incl = wave_incl_scan_dpp(len);
  const int S = incl - len;
  k.T = __builtin_amdgcn_readlane(incl, 63);
  if (len > 0) {
    const int r = __builtin_amdgcn_mbcnt_hi((uint32_t)(live >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)live, 0));
    l.tb[r] = (I)(start - S);
    extra(r);
  }
  for (int g0 = 0; g0 < k.T; g0 += 64 * kSpanWords) {  // wave-uniform
    if (lane < kSpanWords) l.wm[lane] = 0ull;
    wave_sync();
    const int b = S - 1 - g0;
    if (len > 0 && S > 0 && b >= 0 && b < 64 * kSpanWords) atomicOr(&l.wm[b >> 6], 1ull << (b & 63));
    wave_sync();
    k.m = lane < kSpanWords ? l.wm[lane] : 0ull;
    const int pc = __popcll(k.m);
    const int before = __popcll(__builtin_amdgcn_ballot_w64(len > 0 && S > 0 && b < 0));
    k.ex = before + wave_incl_scan_dpp(pc) - pc;
    span_words<U>(lane, k, g0, l, body, w0, wstep);
  }
  wave_sync();  // the tables are rewritten by the wave's next entries
  return k;
}

// Descriptor of the A entry a lane holds: start and length of the selected B row, A's value.
template <typename V>
struct ADesc {
  int64_t b0;
  int len;
  V va;
};

// f(std::integral_constant<int, i>) for i = 0 .. N-1, unrolled at compile time (for indices
// that must be immediates, such as DPP lane selects).
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Which A entry of a 64-entry chunk a lane holds. With G = 16 the layout is transposed: lane
// 16r + j holds entry 4j + r, so in step S (entries 16S .. 16S+15) subgroup r's u-th entry,
// 16S + 4u + r, sits in lane 4S + u of the subgroup's own row of 16 lanes and reaches all of
// the row through one DPP row broadcast (no LDS traffic). With G = 64 lane e holds entry e and
// the wave takes it with readlane.
template <int G>
__device__ __forceinline__ int desc_slot(int lane) {
  static_assert(G == 16 || G == 64, "walk widths");
  return G == 16 ? 4 * (lane & 15) + (lane >> 4) : lane;
}

// Field of the entry at broadcast index J (G = 16: lane J of each row; G = 64: lane e) to all
// lanes that walk it.
template <int G, int J>
__device__ __forceinline__ int ebcast(int x, int e) {
  if constexpr (G == 16)
    return __builtin_amdgcn_update_dpp(0, x, 0x150 + J, 0xF, 0xF, false);  // row_newbcast:J
  else
    return __builtin_amdgcn_readlane(x, e);
}
template <int G, int J>
__device__ __forceinline__ int64_t ebcast64(int64_t x, int e) {
  const uint32_t lo = (uint32_t)ebcast<G, J>((int)(uint32_t)x, e);
  const uint32_t hi = (uint32_t)ebcast<G, J>((int)(uint32_t)((uint64_t)x >> 32), e);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}
template <int G, int J>
__device__ __forceinline__ double ebcastv(double x, int e) {
  return __longlong_as_double(ebcast64<G, J>(__double_as_longlong(x), e));
}
template <int G, int J>
__device__ __forceinline__ float ebcastv(float x, int e) {
  return __int_as_float(ebcast<G, J>(__float_as_int(x), e));
}

// Lane `lane` loads the descriptor of A entry base + desc_slot(lane). These loads cover the
// chunk's entries in A's order (coalesced). Lanes past a1 load entry a1 - 1 instead, and the
// values are kept raw: the consumers (gather_step, consume_step) take only entries below the
// chunk's count. Unconditional loads keep the compiler's in-order count of outstanding loads
// exact (a branch around a load, or a select on its result right after it, makes the wave wait
// for the load at that point). a1 >= 1 for every row that reaches a kernel (such rows have
// products).
template <int G, bool WITHV, typename V>
__device__ __forceinline__ ADesc<V> load_desc(int64_t base, int64_t a1, int lane, const int64_t* __restrict__ bstart,
                                              const int32_t* __restrict__ blen, const V* __restrict__ Aval) {
  const int64_t j = base + desc_slot<G>(lane);
  const int64_t jj = j < a1 ? j : (a1 > 0 ? a1 - 1 : 0);
  ADesc<V> d;
  d.b0 = bstart[jj];
  d.len = blen[jj];
  d.va = WITHV ? Aval[jj] : V(0);
  return d;
}

// One gather step over a chunk of A entries: the wave's 64/G subgroups take U entries each
// (G = 16: step S, entries 16S .. 16S+15; G = 64: entries e0 .. e0+U-1) and issue the U B-row
// gathers (the first G entries of each B row). Only the loaded columns and B values are kept;
// they are masked and multiplied when the step is consumed.
template <int U, typename V>
struct Step {
  int c[U];   // B columns as loaded (masked when consumed)
  V bv[U];    // B values as loaded
};

// index of entry u of this lane's subgroup in the step
template <int G, int S>
__device__ __forceinline__ int step_entry(int e0, int u, int sg) {
  return G == 16 ? 16 * S + 4 * u + sg : e0 + u;
}

template <int G, int U, bool WITHV, typename V, int S = 0>
__device__ __forceinline__ void gather_step(Step<U, V>& st, int lane, int e0, int cnt, const ADesc<V>& d,
                                            const int32_t* __restrict__ Bidx, const V* __restrict__ Bval) {
  static_assert(G == 64 || U == 4, "with G = 16 a step is 4 subgroups x 4 entries");
  const int sg = lane / G, lg = lane % G;
  // unconditional loads: lanes past the B row re-read its last entry, entries without a B row
  // read entry 0 (B has entries whenever a row reaches a kernel). The loaded values are kept
  // raw: masking them here would make the wave wait for the loads right away.
  static_for<U>([&](auto uc) {
    constexpr int u = decltype(uc)::value;
    const int e = step_entry<G, S>(e0, u, sg);
    const int er = min(e0 + u, 63);
    const int64_t pb = ebcast64<G, 4 * S + (u & 3)>(d.b0, er);
    const int lv = ebcast<G, 4 * S + (u & 3)>(d.len, er);
    const int pl = e < cnt ? lv : 0;
    const int64_t at = pl > 0 ? pb + min(lg, pl - 1) : 0;
    st.c[u] = Bidx[at];
    st.bv[u] = WITHV ? Bval[at] : V(0);
  });
}

// Hand a gathered step to the sink: f.batch(c[U], v[U]) for the first G entries of each B row (c < 0
// marks no product), v = A_ik * B_kj. What B rows longer than G have left is walk_tails'.
template <int G, int U, bool WITHV, typename V, typename F, int S = 0>
__device__ __forceinline__ void consume_step(const Step<U, V>& st, int lane, int e0, int cnt, const ADesc<V>& d, F& f) {
  const int sg = lane / G, lg = lane % G;
  int c[U];
  V v[U];
  static_for<U>([&](auto uc) {
    constexpr int u = decltype(uc)::value;
    const int e = step_entry<G, S>(e0, u, sg);
    const int er = min(e0 + u, 63);
    const int lv = ebcast<G, 4 * S + (u & 3)>(d.len, er);
    V pv = V(0);
    if constexpr (WITHV) pv = ebcastv<G, 4 * S + (u & 3)>(d.va, er);
    const bool has = e < cnt && lg < lv;
    c[u] = has ? st.c[u] : -1;
    v[u] = (WITHV && has) ? pv * st.bv[u] : V(0);
  });
  f.template batch<U>(c, v);
}

// LDS of one wave for walk_flat: the spans' tables and A's values by rank.
template <typename V, bool WITHV>
struct FlatLds {
  SpanLds sp;
  V va[WITHV ? 64 : 1];
};

// The products of one entry per lane (`len` elements of its B row from `start` on, A's value va),
// element-parallel over the wave.
template <int U, bool WITHV, typename V, typename F>
__device__ __forceinline__ void walk_flat(int lane, int len, int64_t start, V va, const int32_t* __restrict__ Bidx,
                                          const V* __restrict__ Bval, FlatLds<V, WITHV>& l, F& f, int w0 = 0,
                                          int wstep = U) {
  walk_spans<U>(lane, len, start, l.sp,
                [&](int r) {
                  if (WITHV) l.va[r] = va;
                },
                [&](const int64_t (&at)[U], const int (&j)[U]) {
                  int c[U];
                  V v[U];
#pragma unroll
                  for (int u = 0; u < U; ++u) {
                    const int64_t p = at[u] < 0 ? 0 : at[u];
                    c[u] = Bidx[p];
                    v[u] = WITHV ? l.va[WITHV ? j[u] : 0] * Bval[p] : V(0);
                  }
#pragma unroll
                  for (int u = 0; u < U; ++u) c[u] = at[u] < 0 ? -1 : c[u];
                  f.template batch<U>(c, v);
                },
                w0, wstep);
}

// The rest of the B rows longer than G of one chunk's entries. One by one, G lanes each, they were a
// chain of dependent loads: half of the time of rows whose B rows average 33 entries.
template <int G, int U, bool WITHV, typename V, typename F>
__device__ __forceinline__ void walk_tails(int lane, int cnt, const ADesc<V>& d, const int32_t* __restrict__ Bidx,
                                           const V* __restrict__ Bval, FlatLds<V, WITHV>& l, F& f) {
  const int len = desc_slot<G>(lane) < cnt ? max(d.len - G, 0) : 0;
  if (!__builtin_amdgcn_ballot_w64(len > 0)) return;
  walk_flat<U, WITHV>(lane, len, d.b0 + G, d.va, Bidx, Bval, l, f);
  wait_vmem();
}

template <int G, int U, bool WITHV, typename V, typename F, int S>
__device__ __forceinline__ void walk_step(int lane, int e0, int cnt, const ADesc<V>& d,
                                          const int32_t* __restrict__ Bidx, const V* __restrict__ Bval, F& f) {
  Step<U, V> st;
  gather_step<G, U, WITHV, V, S>(st, lane, e0, cnt, d, Bidx, Bval);
  consume_step<G, U, WITHV, V, F, S>(st, lane, e0, cnt, d, f);
}

// All products of `cnt` (<= 64) A entries of one chunk, from entry `from` on (a multiple of a
// step). Control flow around the broadcasts is wave-uniform.
template <int G, int U, bool WITHV, typename V, typename F>
__device__ __forceinline__ void walk_chunk(int lane, int cnt, const ADesc<V>& d, const int32_t* __restrict__ Bidx,
                                           const V* __restrict__ Bval, F& f, int from = 0) {
  if constexpr (G == 16) {  // steps are compile-time (their broadcast lanes are DPP immediates)
    if (from <= 0 && 0 < cnt) walk_step<G, U, WITHV, V, F, 0>(lane, 0, cnt, d, Bidx, Bval, f);
    if (from <= 16 && 16 < cnt) walk_step<G, U, WITHV, V, F, 1>(lane, 16, cnt, d, Bidx, Bval, f);
    if (from <= 32 && 32 < cnt) walk_step<G, U, WITHV, V, F, 2>(lane, 32, cnt, d, Bidx, Bval, f);
    if (from <= 48 && 48 < cnt) walk_step<G, U, WITHV, V, F, 3>(lane, 48, cnt, d, Bidx, Bval, f);
  } else {
    for (int e0 = from; e0 < cnt; e0 += U) walk_step<G, U, WITHV, V, F, 0>(lane, e0, cnt, d, Bidx, Bval, f);
  }
}

// All products of one row for a group of NT >= 64 threads: wave w handles A entries
// a0 + 64w, a0 + 64w + NT, ...; `first` holds the descriptors of the wave's first chunk when
// the caller prefetched them.
template <int NT, int G, int U, bool WITHV, typename V, typename F>
__device__ __forceinline__ void for_row_products_pre(int t, int64_t a0, int64_t a1, const ADesc<V>& first,
                                                     const int64_t* __restrict__ bstart,
                                                     const int32_t* __restrict__ blen, const V* __restrict__ Aval,
                                                     const int32_t* __restrict__ Bidx, const V* __restrict__ Bval,
                                                     FlatLds<V, WITHV>& l, F& f, const Step<U, V>* step0 = nullptr) {
  static_assert(NT >= 64, "wave-level walk");
  constexpr int STEP = G == 16 ? 16 : U;  // entries per step
  const int lane = t & 63, wv = t >> 6;
  int64_t base = a0 + 64 * wv;
  if (base < a1) {
    const int cnt = (int)min((int64_t)64, a1 - base);
    int from = 0;
    if (step0) {  // the caller already issued the first step's gathers
      consume_step<G, U, WITHV, V, F, 0>(*step0, lane, 0, cnt, first, f);
      from = STEP;
    }
    if (from < cnt) {
      walk_chunk<G, U, WITHV, V>(lane, cnt, first, Bidx, Bval, f, from);
      if (step0) wait_vmem();
    }
    walk_tails<G, U, WITHV>(lane, cnt, first, Bidx, Bval, l, f);
  }
  if (base + NT < a1) {
    for (base += NT; base < a1; base += NT) {
      const ADesc<V> d = load_desc<G, WITHV, V>(base, a1, lane, bstart, blen, Aval);
      const int cnt = (int)min((int64_t)64, a1 - base);
      walk_chunk<G, U, WITHV, V>(lane, cnt, d, Bidx, Bval, f);
      walk_tails<G, U, WITHV>(lane, cnt, d, Bidx, Bval, l, f);
    }
    if (step0) wait_vmem();
  }
}

// All products of one row for a workgroup of NT > 64 threads. G = 16: 16 lanes per B row, 64 entries
// per wave. G = 64: element-parallel; a row of up to 64 entries is every wave's, which share its
// elements (dealt 64 entries per wave such a row was one wave's work), a row of more is dealt entry
// by entry over the waves.
template <int NT, int G, int U, bool WITHV, typename V, typename F>
__device__ __forceinline__ void for_row_products(int t, int64_t a0, int64_t a1, const int64_t* __restrict__ bstart,
                                                 const int32_t* __restrict__ blen, const V* __restrict__ Aval,
                                                 const int32_t* __restrict__ Bidx, const V* __restrict__ Bval,
                                                 FlatLds<V, WITHV>& l, F& f) {
  if constexpr (G == 64) {
    constexpr int NW = NT / 64;
    const int lane = t & 63, wv = t >> 6;
    const bool shared = a1 - a0 <= 64;  // uniform
    for (int64_t base = a0; base < a1; base += NT) {
      const int64_t ka = base + (shared ? lane : wv + NW * lane);
      int len = 0;
      int64_t start = 0;
      V va = V(0);
      if (ka < a1) {
        len = blen[ka];
        start = bstart[ka];
        va = WITHV ? Aval[ka] : V(0);
      }
      walk_flat<U, WITHV>(lane, len, start, va, Bidx, Bval, l, f, shared ? wv * U : 0, shared ? NW * U : U);
    }
  } else {
    const ADesc<V> first = load_desc<G, WITHV, V>(a0 + 64 * (t >> 6), a1, t & 63, bstart, blen, Aval);
    for_row_products_pre<NT, G, U, WITHV, V>(t, a0, a1, first, bstart, blen, Aval, Bidx, Bval, l, f);
  }
}

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own L2). When the grid
// is a multiple of 8, virtual block ids are regrouped so that consecutive ids (consecutive bin
// slots, i.e. nearby rows) run on the same XCD.
__device__ __forceinline__ int64_t xcd_block() {
  const uint32_t b = blockIdx.x, n = gridDim.x;
  if (n % 8 != 0) return b;
  return (int64_t)(b % 8) * (n / 8) + b / 8;
}

// Rows handled by one wave, software-pipelined. The wave's rows are the bin slots s0, s0 +
// stride, ...; their ids and row pointers are loaded 64 rows at a time with vector loads (lane
// L holds row L of the batch) and read out with readlane, so no scalar loads are outstanding
// while the wave waits on LDS (scalar loads and LDS share one counter). The next row's A
// descriptors are issued at the top of each iteration and its first B gathers after the
// current row's products are in LDS, so each wait is for loads issued a good while earlier.
template <int G, bool WITHV, typename V>
struct RowPipe {
  int64_t slot, stride, end;   // slot of the current row (wave-uniform)
  int kb;                      // batch index of the next row (wave-uniform)
  int bR;                      // batch: row ids (per lane)
  int64_t bA0, bA1, bC0, bC1;  // batch: row pointers (per lane)
  int row, row1;               // current / next row (wave-uniform)
  int64_t a0, a1, c0, c1;      // current row: A range and output range
  int64_t na0, na1, nc0, nc1;  // next row
  ADesc<V> d, nd;              // descriptors of the current / next row
  bool more;                   // a next row exists

  __device__ __forceinline__ void load_batch(int64_t s0, int lane, const int32_t* __restrict__ rows,
                                             const int64_t* __restrict__ Aptr, const int64_t* __restrict__ Cptr) {
    int64_t ls = s0 + (int64_t)lane * stride;
    if (ls >= end) ls = end - 1;  // past the bin: repeat its last row (never used)
    const int r = rows[ls];
    bR = r;
    bA0 = Aptr[r];
    bA1 = Aptr[r + 1];
    if (Cptr) {
      bC0 = Cptr[r];
      bC1 = Cptr[r + 1];
    } else {
      bC0 = bC1 = 0;
    }
  }
  __device__ __forceinline__ void extract(int j, int& r, int64_t& x0, int64_t& x1, int64_t& y0, int64_t& y1) const {
    r = __builtin_amdgcn_readlane(bR, j);
    x0 = readlane64(bA0, j);
    x1 = readlane64(bA1, j);
    y0 = readlane64(bC0, j);
    y1 = readlane64(bC1, j);
  }
  __device__ __forceinline__ void start(int64_t s0, int64_t st, int64_t e, const int32_t* __restrict__ rows,
                                        const int64_t* __restrict__ Aptr, const int64_t* __restrict__ Cptr, int lane,
                                        const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
                                        const V* __restrict__ Aval) {
    slot = s0;
    stride = st;
    end = e;
    load_batch(s0, lane, rows, Aptr, Cptr);
    kb = 0;
    extract(0, row, a0, a1, c0, c1);
    d = load_desc<G, WITHV, V>(a0, a1, lane, bstart, blen, Aval);
  }
  // top of an iteration: pointers (a new batch every 64 rows) and descriptors of the next row;
  // past the last row the current row is repeated, so the loads stay unconditional
  __device__ __forceinline__ void prefetch(int lane, const int32_t* __restrict__ rows,
                                           const int64_t* __restrict__ Aptr, const int64_t* __restrict__ Cptr,
                                           const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
                                           const V* __restrict__ Aval) {
    more = slot + stride < end;
    if (more) {
      ++kb;
      if (kb == 64) {
        load_batch(slot + stride, lane, rows, Aptr, Cptr);
        kb = 0;
        wait_vmem();
      }
    }
    extract(kb, row1, na0, na1, nc0, nc1);
    nd = load_desc<G, WITHV, V>(na0, na1, lane, bstart, blen, Aval);
  }
  __device__ __forceinline__ bool advance() {
    if (!more) return false;
    slot += stride;
    row = row1;
    a0 = na0;
    a1 = na1;
    c0 = nc0;
    c1 = nc1;
    d = nd;
    return true;
  }
};

// Error bits written to the device error word.
constexpr int kErrTableFull = 1;
constexpr int kErrCountMismatch = 2;
constexpr int kErrWindow = 4;
constexpr int kErrMissingKey = 8;
constexpr int kErrCapacity = 16;  // output larger than the capacity the caller provided

// ------------------------------------------------------------------------------------
// fills, scan, gathers
// ------------------------------------------------------------------------------------
template <typename T>
__global__ void k_fill(T* __restrict__ p, int64_t n, T v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

static int fill_grid(int64_t n) {
  int64_t g = (n + 255) / 256;
  if (g > 65536) g = 65536;
  if (g < 1) g = 1;
  return (int)g;
}

void launch_fill_i64(int64_t* p, int64_t n, int64_t v, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill<int64_t>, dim3(fill_grid(n)), dim3(256), 0, s, p, n, v);
}
void launch_fill_i32(int32_t* p, int64_t n, int32_t v, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill<int32_t>, dim3(fill_grid(n)), dim3(256), 0, s, p, n, v);
}
void launch_fill_bytes0(void* p, int64_t nbytes, hipStream_t s) {
  // callers pass 4-byte multiples (value arrays, counters)
  launch_fill_i32((int32_t*)p, nbytes / 4, 0, s);
}

// Reduce-then-scan over tiles of 4096 int64 (256 threads x 16 items). No look-back and no
// memsets: safe to capture in a hipGraph and replay.
constexpr int kScanThreads = 256;
constexpr int kScanItems = 16;
constexpr int64_t kScanTile = kScanThreads * kScanItems;

int64_t scan_tmp_elems(int64_t n) { return (n + kScanTile - 1) / kScanTile + 2; }

__global__ __launch_bounds__(kScanThreads) void k_scan_reduce(const int64_t* __restrict__ in, int64_t n,
                                                              int64_t* __restrict__ part) {
  __shared__ int64_t sc[kScanThreads / 64];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
  int64_t s = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    int64_t j = base + i;
    if (j < n) s += in[j];
  }
  s = Group<kScanThreads>::reduce(s, OpAdd(), sc);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// Single workgroup: exclusive scan of part[0..nb) in place; part[nb] = total.
__global__ __launch_bounds__(1024) void k_scan_partials(int64_t* __restrict__ part, int64_t nb) {
  __shared__ int64_t sc[16];
  int64_t carry = 0;
  for (int64_t base = 0; base < nb; base += 1024) {
    int64_t j = base + threadIdx.x;
    int64_t v = (j < nb) ? part[j] : 0;
    int64_t tot;
    int64_t ex = Group<1024>::exscan(v, tot, sc);
    if (j < nb) part[j] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) part[nb] = carry;
}

__global__ __launch_bounds__(kScanThreads) void k_scan_apply(const int64_t* in, int64_t* out, int64_t n,
                                                             const int64_t* __restrict__ part, int64_t nb) {
  __shared__ int64_t sc[kScanThreads / 64];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
  int64_t loc[kScanItems];
  int64_t s = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    int64_t j = base + i;
    loc[i] = (j < n) ? in[j] : 0;
    s += loc[i];
  }
  int64_t tot;
  int64_t pre = Group<kScanThreads>::exscan(s, tot, sc) + part[blockIdx.x];
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    int64_t j = base + i;
    if (j < n) out[j] = pre;
    pre += loc[i];
  }
  if (blockIdx.x == nb - 1 && threadIdx.x == 0) out[n] = part[nb];
}

// One workgroup, 16 items a thread at a time: one launch instead of three up to kScanOne items, where a
// launch costs more than the idle CUs (16,384 items: 5 us against 3 x 4 us and two gaps).
constexpr int64_t kScanOne = 32768;
__global__ __launch_bounds__(1024) void k_scan_one(const int64_t* in, int64_t* out, int64_t n) {
  __shared__ int64_t sc[16];
  int64_t carry = 0;
  for (int64_t b = 0; b < n; b += 1024 * kScanItems) {  // uniform
    const int64_t base = b + (int64_t)threadIdx.x * kScanItems;
    int64_t loc[kScanItems], sum = 0, tot;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
      loc[i] = base + i < n ? in[base + i] : 0;
      sum += loc[i];
    }
    int64_t pre = carry + Group<1024>::exscan(sum, tot, sc);
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
      if (base + i < n) out[base + i] = pre;
      pre += loc[i];
    }
    carry += tot;
  }
  if (threadIdx.x == 0) out[n] = carry;
}

void launch_exclusive_scan(const int64_t* in, int64_t* out, int64_t n, int64_t* tmp, hipStream_t s) {
  if (n <= 0) {
    launch_fill_i64(out, 1, 0, s);
    return;
  }
  if (n <= kScanOne) {
    hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(1024), 0, s, in, out, n);
    return;
  }
  const int64_t nb = (n + kScanTile - 1) / kScanTile;
  hipLaunchKernelGGL(k_scan_reduce, dim3((unsigned)nb), dim3(kScanThreads), 0, s, in, n, tmp);
  hipLaunchKernelGGL(k_scan_partials, dim3(1), dim3(1024), 0, s, tmp, nb);
  hipLaunchKernelGGL(k_scan_apply, dim3((unsigned)nb), dim3(kScanThreads), 0, s, in, out, n, tmp, nb);
}

// Output capacity check inside a captured pipeline: when the exact output size (*total) exceeds
// the caller's capacity, flag it and empty every bin range (offs[0 .. n)), so the kernels that
// follow drain nothing and write nothing.
__global__ void k_capacity_guard(const int64_t* __restrict__ total, int64_t cap, int64_t* __restrict__ offs, int64_t n,
                                 int* __restrict__ err) {
  if (*total <= cap) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(err, kErrCapacity);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    offs[i] = 0;
}

void launch_capacity_guard(const int64_t* total, int64_t cap, int64_t* offs, int64_t n, int* err, hipStream_t s) {
  hipLaunchKernelGGL(k_capacity_guard, dim3(fill_grid(n)), dim3(256), 0, s, total, cap, offs, n, err);
}

// ------------------------------------------------------------------------------------
// row analysis: P_i = sum over A_i of B row lengths
// ------------------------------------------------------------------------------------
// The work is split by nonzeros of A, not by rows: a workgroup takes kRpTile consecutive nonzeros,
// writes their descriptors coalesced, scans their B row lengths in LDS and reads every row's sum
// off the prefix at its ends. Rows that cross a tile add their parts atomically (P starts at 0). A
// row of any length costs the same per nonzero; with 16 lanes per row the longest row of an
// R-MAT 20 sample kept one subgroup busy for the whole 1.11 ms of the launch (0.012 ms now), and
// the analysis of a batch of 32 skewed members (1.0e7 nonzeros) took 1.39 ms (0.068 ms now).
// On 3.2e7 nonzeros with random columns both take 0.52 ms: there the gathers of B's row pointer
// bound it, one 128-byte line each.
constexpr int kRpThreads = 256;
constexpr int kRpItems = 8;
constexpr int kRpTile = kRpThreads * kRpItems;
constexpr int64_t kRpRowWalk = 4096;  // rows per tile up to which the rows are walked (see below)

int64_t row_tiles(int64_t nnz) { return (nnz + kRpTile - 1) / kRpTile; }

// Clears P, nnz and the error word, and notes the row that holds the first nonzero of every tile
// (tile_row[number of tiles] = the row of the last nonzero). The nonzeros are those the row
// pointer covers, [Aptr[0], Aptr[nr]): a device view may be a run of rows of a larger matrix.
__global__ __launch_bounds__(256) void k_row_init(int64_t nr, const int64_t* __restrict__ Aptr,
                                                  int64_t* __restrict__ P, int64_t* __restrict__ nnz,
                                                  int32_t* __restrict__ tile_row, int* __restrict__ err) {
  if (err && blockIdx.x == 0 && threadIdx.x == 0) *err = 0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nr; i += (int64_t)gridDim.x * 256) {
    P[i] = 0;
    nnz[i] = 0;
    const int64_t a0 = Aptr[i], a1 = Aptr[i + 1];
    if (a1 <= a0) continue;
    const int64_t first = Aptr[0], end = Aptr[nr];
    for (int64_t q = (a0 - first + kRpTile - 1) / kRpTile; first + q * kRpTile < a1; ++q) tile_row[q] = (int32_t)i;
    if (a1 == end) tile_row[(end - first + kRpTile - 1) / kRpTile] = (int32_t)i;
  }
}

__global__ __launch_bounds__(kRpThreads) void k_row_products(int64_t nr, const int64_t* __restrict__ Aptr,
                                                             const int32_t* __restrict__ Aidx,
                                                             const int64_t* __restrict__ Bptr,
                                                             int64_t* __restrict__ P, int64_t* __restrict__ bstart,
                                                             int32_t* __restrict__ blen,
                                                             const int32_t* __restrict__ tile_row) {
  __shared__ int len[kRpTile];
  __shared__ int64_t pre[kRpTile + 1];
  __shared__ int64_t sc[kRpThreads / 64];
  const int t = threadIdx.x;
  const int64_t base = Aptr[0] + (int64_t)blockIdx.x * kRpTile;
  const int64_t left = Aptr[nr] - base;
  if (left <= 0) return;  // uniform: the grid covers the index array, the rows may end before it
  const int n = (int)min((int64_t)kRpTile, left);
  const int64_t r0 = tile_row[blockIdx.x], r1 = tile_row[blockIdx.x + 1];
  int k[kRpItems];
#pragma unroll
  for (int q = 0; q < kRpItems; ++q) k[q] = Aidx[base + min(t + q * kRpThreads, n - 1)];
  int64_t b0[kRpItems], b1[kRpItems];
#pragma unroll
  for (int q = 0; q < kRpItems; ++q) {
    b0[q] = Bptr[k[q]];
    b1[q] = Bptr[k[q] + 1];
  }
#pragma unroll
  for (int q = 0; q < kRpItems; ++q) {
    const int j = t + q * kRpThreads;
    const int l = j < n ? (int)(b1[q] - b0[q]) : 0;
    len[j] = l;
    if (j < n) {
      bstart[base + j] = b0[q];
      blen[base + j] = l;
    }
  }
  __syncthreads();
  int64_t loc[kRpItems], sum = 0, tot;
#pragma unroll
  for (int q = 0; q < kRpItems; ++q) {
    loc[q] = sum;
    sum += len[t * kRpItems + q];
  }
  const int64_t ex = Group<kRpThreads>::exscan(sum, tot, sc);
#pragma unroll
  for (int q = 0; q < kRpItems; ++q) pre[t * kRpItems + q] = ex + loc[q];
  if (t == 0) pre[kRpTile] = tot;
  __syncthreads();
  if (r1 - r0 < kRpRowWalk) {  // uniform
    for (int64_t r = r0 + t; r <= r1; r += kRpThreads) {
      const int64_t a0 = Aptr[r], a1 = Aptr[r + 1];
      const int s0 = (int)max(a0 - base, (int64_t)0), s1 = (int)min(a1 - base, (int64_t)n);
      if (s1 <= s0) continue;
      const int64_t v = pre[s1] - pre[s0];
      if (a0 >= base && a1 <= base + n)
        P[r] = v;
      else
        atomicAdd((unsigned long long*)&P[r], (unsigned long long)v);
    }
    return;
  }
  // a tile over thousands of rows, most of them empty: every thread finds the rows of its own
  // nonzeros by bisection instead
  int j = t * kRpItems;
  const int jend = min(j + kRpItems, n);
  while (j < jend) {
    int64_t lo = r0, hi = r1;  // the row with Aptr[row] <= base + j < Aptr[row + 1]
    while (lo < hi) {
      const int64_t m = (lo + hi) >> 1;
      if (Aptr[m + 1] > base + j) hi = m;
      else lo = m + 1;
    }
    const int je = (int)min(Aptr[lo + 1] - base, (int64_t)jend);
    atomicAdd((unsigned long long*)&P[lo], (unsigned long long)(pre[je] - pre[j]));
    j = max(je, j + 1);
  }
}

void launch_row_products(const Mat& A, const Mat& B, int64_t* P, int64_t* nnz, int64_t* bstart, int32_t* blen,
                         int32_t* tile_row, int* err, hipStream_t s) {
  hipLaunchKernelGGL(k_row_init, dim3(fill_grid(A.nrows)), dim3(256), 0, s, A.nrows, A.ptr, P, nnz, tile_row, err);
  if (A.nrows <= 0 || A.nnz <= 0) return;
  hipLaunchKernelGGL(k_row_products, dim3((unsigned)row_tiles(A.nnz)), dim3(kRpThreads), 0, s, A.nrows, A.ptr, A.idx,
                     B.ptr, P, bstart, blen, tile_row);
}

// ------------------------------------------------------------------------------------
// band index of the long B rows (for the long-row window kernels)
// ------------------------------------------------------------------------------------
// B rows of at least `minlen` entries ("heavy" rows) get a slot; for each, the position (from the
// row's start) of its first entry at or past every multiple of 4096 columns, over nb1 entries,
// the last of which (past every column) holds the row's length. A long-row window of aligned
// columns then reads its exact element range from two entries instead of walking the row.
__global__ void k_heavy_flag(const int64_t* __restrict__ Bptr, int64_t nrows, int64_t minlen, int64_t* __restrict__ flag) {
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < nrows; k += (int64_t)gridDim.x * blockDim.x)
    flag[k] = (Bptr[k + 1] - Bptr[k]) >= minlen ? 1 : 0;
}

__global__ void k_heavy_slot(const int64_t* __restrict__ flag_scan, const int64_t* __restrict__ Bptr, int64_t nrows,
                             int64_t minlen, int32_t* __restrict__ slot, int32_t* __restrict__ slot_row) {
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < nrows; k += (int64_t)gridDim.x * blockDim.x) {
    const bool heavy = (Bptr[k + 1] - Bptr[k]) >= minlen;
    const int32_t sl = (int32_t)flag_scan[k];
    slot[k] = heavy ? sl : -1;
    if (heavy) slot_row[sl] = (int32_t)k;
  }
}

// One workgroup per heavy row: entry q of band position b is written by the element that opens
// band b (the first element whose band is >= b), bands past the last element by the tail.
__global__ __launch_bounds__(256) void k_band_index(const int32_t* __restrict__ slot_row, int64_t nslots,
                                                    const int64_t* __restrict__ Bptr, const int32_t* __restrict__ Bidx,
                                                    int64_t nb1, int32_t* __restrict__ band) {
  for (int64_t sl = blockIdx.x; sl < nslots; sl += gridDim.x) {
    const int k = slot_row[sl];
    const int64_t b0 = Bptr[k];
    const int32_t L = (int32_t)(Bptr[k + 1] - b0);
    int32_t* out = band + sl * nb1;
    for (int32_t q = threadIdx.x; q < L; q += blockDim.x) {
      const int bq = Bidx[b0 + q] >> kBandShift;
      const int bp = q > 0 ? (Bidx[b0 + q - 1] >> kBandShift) : -1;
      for (int b = bp + 1; b <= bq; ++b) out[b] = q;
    }
    const int blast = L > 0 ? (Bidx[b0 + L - 1] >> kBandShift) : -1;
    for (int64_t b = blast + 1 + threadIdx.x; b < nb1; b += blockDim.x) out[b] = L;
  }
}

// hist[j] = number of B rows with at least 2^j entries, j = 0 .. 31 (hist zeroed by the caller)
__global__ void k_len_hist(const int64_t* __restrict__ Bptr, int64_t nrows, int64_t* __restrict__ hist) {
  __shared__ int h[32];
  if (threadIdx.x < 32) h[threadIdx.x] = 0;
  __syncthreads();
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < nrows; k += (int64_t)gridDim.x * blockDim.x) {
    const int64_t L = Bptr[k + 1] - Bptr[k];
    if (L > 0) atomicAdd(&h[63 - __clzll((unsigned long long)L)], 1);  // floor(log2 L)
  }
  __syncthreads();
  if (threadIdx.x < 32) {
    int64_t c = 0;
    for (int j = threadIdx.x; j < 32; ++j) c += h[j];  // rows with floor(log2 L) >= threadIdx.x
    if (c) atomicAdd((unsigned long long*)&hist[threadIdx.x], (unsigned long long)c);
  }
}

void launch_len_hist(const int64_t* Bptr, int64_t nrows, int64_t* hist, hipStream_t s) {
  launch_fill_i64(hist, 32, 0, s);
  if (nrows <= 0) return;
  int64_t g = (nrows + 255) / 256;
  if (g > 1024) g = 1024;
  hipLaunchKernelGGL(k_len_hist, dim3((unsigned)g), dim3(256), 0, s, Bptr, nrows, hist);
}

int64_t band_count(int64_t ncols) {
  const int64_t nb = (ncols + (1 << kBandShift) - 1) >> kBandShift;
  return (nb + kBandPad - 1) / kBandPad * kBandPad + 1;
}

void launch_heavy_slots(const int64_t* Bptr, int64_t nrows, int64_t minlen, int64_t* flag, int64_t* tmp,
                        int32_t* slot, int32_t* slot_row, hipStream_t s) {
  if (nrows <= 0) return;
  hipLaunchKernelGGL(k_heavy_flag, dim3(fill_grid(nrows)), dim3(256), 0, s, Bptr, nrows, minlen, flag);
  launch_exclusive_scan(flag, flag, nrows, tmp, s);
  hipLaunchKernelGGL(k_heavy_slot, dim3(fill_grid(nrows)), dim3(256), 0, s, flag, Bptr, nrows, minlen, slot, slot_row);
}

void launch_band_index(const int32_t* slot_row, int64_t nslots, const int64_t* Bptr, const int32_t* Bidx, int64_t nb1,
                       int32_t* band, hipStream_t s) {
  if (nslots <= 0) return;
  const int64_t g = nslots < 65536 ? nslots : 65536;
  hipLaunchKernelGGL(k_band_index, dim3((unsigned)g), dim3(256), 0, s, slot_row, nslots, Bptr, Bidx, nb1, band);
}

// ------------------------------------------------------------------------------------
// binning: stable counting sort of row ids by category
// ------------------------------------------------------------------------------------
constexpr int kBinTile = 256;
int64_t bin_tiles(int64_t n) { return (n + kBinTile - 1) / kBinTile; }

// The limits past the last category are INT64_MAX, so no branch and no load depends on the key.
__device__ __forceinline__ int category_of(int64_t k, const CatTable& ct) {
  int c = 0;
#pragma unroll
  for (int x = 0; x < kMaxCats; ++x) c += k > ct.lim[x];
  return c;
}

// Category of row i: by key. Numeric tables end with the long category (limit INT64_MAX, so no
// key goes past it) and the hub category; with hub_slot, a long row that has a hub slot (a
// symbolic long row that hub_row picks, whose columns per range the symbolic pass counted) is a
// hub row. Without hub_slot the hub category stays empty.
__device__ __forceinline__ int row_category(int64_t k, const CatTable& ct, const int32_t* __restrict__ hub_slot,
                                            int64_t i) {
  const int c = category_of(k, ct);
  if (hub_slot && c == ct.n - 2 && hub_slot[i] >= 0) return ct.n - 1;
  return c;
}

// The tiles' category counts (cat-major) and, behind them, the tiles' sums of the keys: one scan turns
// them into the bins' offsets and the prefix of the keys.
__global__ __launch_bounds__(kBinTile) void k_bin_count(const int64_t* __restrict__ key, int64_t n, int64_t cap,
                                                        CatTable ct, int64_t* __restrict__ counts, int64_t nwg,
                                                        const int32_t* __restrict__ hub_slot,
                                                        int* __restrict__ many) {
  __shared__ int hist[kMaxCats];
  __shared__ int64_t sc[kBinTile / 64];
  if (threadIdx.x < kMaxCats) hist[threadIdx.x] = 0;
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * kBinTile + threadIdx.x;
  const int64_t k = i < n ? key[i] : 0;
  if (i < n) {
    const int c = row_category(min(k, cap), ct, hub_slot, i);
    atomicAdd(&hist[c], 1);
    if (hub_slot && c == ct.n - 1 && (hub_slot[i] & kHubMany)) atomicAdd(many, 1);
  }
  const int64_t sum = Group<kBinTile>::reduce(k, OpAdd(), sc);  // also: the counts are complete
  if ((int)threadIdx.x < ct.n) counts[(int64_t)threadIdx.x * nwg + blockIdx.x] = hist[threadIdx.x];
  if (threadIdx.x == 0) counts[(int64_t)ct.n * nwg + blockIdx.x] = sum;
}

// What the host reads after a binning, in pinned memory: categories' offsets, error word (with the
// count beside it), and the keys' sums up to the start of each block of `bt` tiles (the last one: all).
__device__ __forceinline__ void bin_report(const BinOut& o, int64_t tile, int64_t nwg, int ncat, const int64_t* offs,
                                           int64_t key_sum, int64_t key_all) {
  if (!o.host) return;
  const int t = threadIdx.x;
  if (tile == 0) {
    if (t <= ncat) o.host->tot[t] = offs[(int64_t)t * nwg];
    if (t < 2) o.host->err[t] = o.err[t];
    if (t == 0) o.host->blk[(nwg + o.bt - 1) / o.bt] = key_all;
  }
  if (t == 0 && tile % o.bt == 0) o.host->blk[tile / o.bt] = key_sum;
}

__global__ __launch_bounds__(kBinTile) void k_bin_scatter(const int64_t* __restrict__ key, int64_t n, int64_t cap,
                                                          CatTable ct, const int64_t* __restrict__ offs, int64_t nwg,
                                                          int32_t* __restrict__ rows,
                                                          const int32_t* __restrict__ hub_slot, BinOut o) {
  __shared__ int wc[kBinTile / 64][kMaxCats];
  __shared__ int64_t sc[kBinTile / 64];
  const int64_t i = (int64_t)blockIdx.x * kBinTile + threadIdx.x;
  const int64_t k = i < n ? key[i] : 0;
  const int c = i < n ? row_category(min(k, cap), ct, hub_slot, i) : -1;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  int rank = 0;
  for (int cc = 0; cc < ct.n; ++cc) {
    const uint64_t b = __ballot(c == cc);
    if (c == cc) rank = __popcll(b & lt);
    if (lane == 0) wc[wid][cc] = __popcll(b);
  }
  __syncthreads();
  if (c >= 0) {
    for (int w = 0; w < wid; ++w) rank += wc[w][c];
    rows[offs[(int64_t)c * nwg + blockIdx.x] + rank] = (int32_t)i;
  }
  const int64_t* kp = offs + (int64_t)ct.n * nwg;  // keys' prefix by tile, behind the number of rows
  const int64_t before = kp[blockIdx.x] - kp[0];
  if (o.ptr) {
    int64_t tot;
    const int64_t at = before + Group<kBinTile>::exscan(k, tot, sc);
    if (i < n) {
      o.ptr[i] = at;
      if (o.ptr2) o.ptr2[i] = at;
      if (i == n - 1) {
        o.ptr[n] = at + k;
        if (o.ptr2) o.ptr2[n] = at + k;
      }
    }
  }
  bin_report(o, blockIdx.x, nwg, ct.n, offs, before, kp[nwg] - kp[0]);
}

// Both binning kernels and the scan between them in one launch of one workgroup, for up to 64 tiles:
// chunk of 64 rows q * 16 + wave is lane-parallel in its wave, the counts of all chunks and the
// keys' sums are scanned in LDS.
constexpr int kBinOneTiles = 64;
__global__ __launch_bounds__(1024) void k_bin_one(const int64_t* __restrict__ key, int64_t n, int64_t cap, CatTable ct,
                                                  int64_t* __restrict__ offs, int64_t nwg, int32_t* __restrict__ rows,
                                                  const int32_t* __restrict__ hub_slot, int* __restrict__ many, BinOut o) {
  constexpr int CH = kBinOneTiles * kBinTile / 64;  // chunks of 64 rows
  constexpr int Q = CH / 16;                        // per wave
  __shared__ int cc[kMaxCats * CH];                 // rows by (category, chunk), then their places
  __shared__ int64_t ks[CH];                        // keys by chunk, then their prefix
  __shared__ int64_t sc[16];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int nch = (int)((n + 63) / 64);
  int64_t k[Q];
  int c[Q], rank[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int64_t i = (int64_t)(q * 16 + wv) * 64 + lane;
    k[q] = i < n ? key[i] : 0;
  }
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int ch = q * 16 + wv;
    const int64_t i = (int64_t)ch * 64 + lane;
    if (ch >= nch) continue;  // wave-uniform
    c[q] = i < n ? row_category(min(k[q], cap), ct, hub_slot, i) : -1;
    rank[q] = 0;
    int cnt = 0;  // lane x: rows of category x
    for (int x = 0; x < ct.n; ++x) {
      const uint64_t b = __builtin_amdgcn_ballot_w64(c[q] == x);
      if (c[q] == x) rank[q] = __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0));
      cnt = lane == x ? (int)__popcll(b) : cnt;
    }
    if (lane < ct.n) cc[lane * nch + ch] = cnt;
    if (hub_slot && c[q] == ct.n - 1 && (hub_slot[i] & kHubMany)) atomicAdd(many, 1);
    int64_t tot;
    const int64_t ex = Group<64>::exscan(k[q], tot, sc);
    if (lane == 0) ks[ch] = tot;
    k[q] = ex;  // within the chunk, from here on
  }
  __syncthreads();
  int64_t carry = 0, tot;
  for (int b = 0; b < ct.n * nch; b += 1024) {  // uniform
    const int v = b + t < ct.n * nch ? cc[b + t] : 0;
    const int64_t ex = carry + Group<1024>::exscan((int64_t)v, tot, sc);
    if (b + t < ct.n * nch) cc[b + t] = (int)ex;
    carry += tot;
  }
  const int64_t kv = t < nch ? ks[t] : 0;
  const int64_t kex = Group<1024>::exscan(kv, tot, sc);
  if (t < nch) ks[t] = kex;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int ch = q * 16 + wv;
    const int64_t i = (int64_t)ch * 64 + lane;
    if (i >= n) continue;
    rows[cc[c[q] * nch + ch] + rank[q]] = (int32_t)i;
    if (o.ptr) {
      const int64_t at = ks[ch] + k[q];
      o.ptr[i] = at;
      if (o.ptr2) o.ptr2[i] = at;
    }
  }
  if (o.ptr && t == 0) {
    o.ptr[n] = tot;
    if (o.ptr2) o.ptr2[n] = tot;
  }
  // the offsets as the launches by tile leave them
  for (int x = t; x < ct.n * (int)nwg; x += 1024) offs[x] = cc[(x / (int)nwg) * nch + 4 * (x % (int)nwg)];
  for (int x = t; x <= (int)nwg; x += 1024) offs[(int64_t)ct.n * nwg + x] = n + (x < (int)nwg ? ks[4 * x] : tot);
  if (!o.host) return;
  if (t < ct.n) o.host->tot[t] = cc[t * nch];
  if (t == ct.n) o.host->tot[t] = n;
  if (t < 2) o.host->err[t] = o.err[t];
  const int nb = (int)((nwg + o.bt - 1) / o.bt);
  for (int b = t; b <= nb; b += 1024) o.host->blk[b] = b < nb ? ks[4 * b * o.bt] : tot;
}

void launch_bin(const int64_t* key, int64_t n, int64_t cap, const CatTable& ct, int64_t* counts, int64_t* offs,
                int64_t* tmp, int32_t* rows, const BinOut& o, hipStream_t s, const int32_t* hub_slot, int* many) {
  const int64_t nwg = bin_tiles(n);
  if (nwg == 0) {
    launch_fill_i64(offs, 1, 0, s);
    if (o.ptr) launch_fill_i64(o.ptr, 1, 0, s);
    if (o.ptr2) launch_fill_i64(o.ptr2, 1, 0, s);
    return;
  }
  if (nwg <= kBinOneTiles) {
    hipLaunchKernelGGL(k_bin_one, dim3(1), dim3(1024), 0, s, key, n, cap, ct, offs, nwg, rows, hub_slot, many, o);
    return;
  }
  hipLaunchKernelGGL(k_bin_count, dim3((unsigned)nwg), dim3(kBinTile), 0, s, key, n, cap, ct, counts, nwg, hub_slot,
                     many);
  launch_exclusive_scan(counts, offs, (ct.n + 1) * nwg, tmp, s);
  hipLaunchKernelGGL(k_bin_scatter, dim3((unsigned)nwg), dim3(kBinTile), 0, s, key, n, cap, ct, offs, nwg, rows,
                     hub_slot, o);
}

// The error word and the count beside it to the host's copy.
__global__ void k_report_err(const int* __restrict__ err, HostReport* host) {
  if (threadIdx.x < 2) host->err[threadIdx.x] = err[threadIdx.x];
}
void launch_report_err(const int* err, HostReport* host, hipStream_t s) {
  hipLaunchKernelGGL(k_report_err, dim3(1), dim3(64), 0, s, err, host);
}

// ------------------------------------------------------------------------------------
// symbolic: nnz_i by LDS hash of keys
// ------------------------------------------------------------------------------------
template <int NT>
constexpr int wg_of() { return NT <= 64 ? 256 : NT; }

// One-wave rows: 7 waves per SIMD (72 VGPRs); a seventh of the waves fewer is 6 % of the pass on
// 2,000,000 rows of 256 products.
template <int T, int NT, int G>
__global__ __launch_bounds__(wg_of<NT>()) __attribute__((amdgpu_waves_per_eu(NT == 64 ? 7 : 1))) void k_symbolic_hash(
    const int32_t* __restrict__ rows, const int64_t* __restrict__ pbeg, const int64_t* __restrict__ pend,
    const int64_t* __restrict__ Aptr, const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
    const int32_t* __restrict__ Bidx, int64_t* __restrict__ nnz, int* __restrict__ err) {
  constexpr int WG = wg_of<NT>();
  constexpr int GPB = WG / NT;
  static_assert(NT % G == 0 && T % NT == 0, "shape");
  __shared__ int hk[GPB][T];
  __shared__ int sc[GPB][NT > 64 ? NT / 64 : 1];
  __shared__ FlatLds<float, false> fl[WG / 64];
  const int t = threadIdx.x % NT;
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x / NT);  // wave-uniform: keep row state scalar
  FlatLds<float, false>& wl = fl[__builtin_amdgcn_readfirstlane(threadIdx.x / 64)];
  int* K = hk[g];
  const int64_t beg = *pbeg, end = *pend;
  if constexpr (NT == 64) {
    const int64_t s0 = beg + xcd_block() * GPB + g;
    if (s0 >= end) return;
    RowPipe<G, false, float> rp;
    rp.start(s0, (int64_t)gridDim.x * GPB, end, rows, Aptr, nullptr, t, bstart, blen, (const float*)nullptr);
    Step<4, float> st0;  // first gather step of the current row, issued during the previous row
    gather_step<G, 4, false, float>(st0, t, 0, (int)min((int64_t)64, rp.a1 - rp.a0), rp.d, Bidx,
                                    (const float*)nullptr);
    // row counts are collected one row per lane and written 64 rows at a time; error bits of
    // all rows are reported once after the loop
    int crow = 0, ccnt = 0, jn = 0, flags = 0;
    for (;;) {
      rp.prefetch(t, rows, Aptr, nullptr, bstart, blen, (const float*)nullptr);
      clear_table<T, float>(t, K, nullptr);
      wave_sync();
      HashSink<T, float, false, false> sk{K, nullptr};
      for_row_products_pre<64, G, 4, false, float>(t, rp.a0, rp.a1, rp.d, bstart, blen, (const float*)nullptr, Bidx,
                                                   (const float*)nullptr, wl, sk, &st0);
      // the next row's first gathers (past the last row: the current row again, unused)
      gather_step<G, 4, false, float>(st0, t, 0, (int)min((int64_t)64, rp.na1 - rp.na0), rp.nd, Bidx,
                                      (const float*)nullptr);
      const int cnt = wave_reduce_dpp(sk.created, OpAdd());
      flags |= sk.bad ? kErrTableFull : 0;
      crow = (t == jn) ? rp.row : crow;
      ccnt = (t == jn) ? cnt : ccnt;
      ++jn;
      if (jn == 64 || !rp.more) {
        if (t < jn) nnz[crow] = ccnt;
        jn = 0;
      }
      wave_sync();
      if (!rp.advance()) break;
    }
    flags = wave_reduce_dpp(flags, OpOr());
    if (t == 0 && flags) atomicOr(err, flags);
    return;
  }
  for (int64_t slot = beg + (int64_t)blockIdx.x * GPB + g; slot < end; slot += (int64_t)gridDim.x * GPB) {
    const int row = rows[slot];
#pragma unroll
    for (int s = t; s < T; s += NT) K[s] = kEmpty;
    gsync<NT>();
    const int64_t a0 = Aptr[row], a1 = Aptr[row + 1];
    HashSink<T, float, false, false> sk{K, nullptr};
    for_row_products<NT, G, 4, false, float>(t, a0, a1, bstart, blen, (const float*)nullptr, Bidx,
                                             (const float*)nullptr, wl, sk);
    const int cnt = Group<NT>::reduce(sk.created, OpAdd(), sc[g]);
    const int bad = Group<NT>::reduce(sk.bad, OpMax(), sc[g]);
    if (t == 0) {
      nnz[row] = cnt;
      if (bad) atomicOr(err, kErrTableFull);
    }
    gsync<NT>();
  }
}

// ------------------------------------------------------------------------------------
// several short rows per wave
// ------------------------------------------------------------------------------------
// A wave per row leaves most lanes idle on rows of a few products, and pays the table clears, the
// ranking and every wait once per row. Rows of up to 256 table slots share a wave instead: 512 / T
// rows, T / 8 lanes and T slots each, eight slots a lane. The rows' A entries (a lane each) are
// flattened together (walk_spans), so one gather covers all of the wave's rows; inserts go to the
// row's own part of the table; the ranking (as wave_rank_keys) runs in all rows at once, its scans
// within the row's lanes. Bound by the chain row id - row pointers - descriptors - gathers, which
// 20 waves a CU and up to 8 rows a wave hide. Where: kMultiRows.
constexpr int kMultiSlots = 512;

// Reduction and inclusive prefix sum within groups of L = 8, 16 or 32 lanes.
template <int L, typename Op>
__device__ __forceinline__ int lanes_reduce(int x, Op op) {
  x = op(x, dpp_mov<0xB1>(x, x));
  x = op(x, dpp_mov<0x4E>(x, x));
  x = op(x, dpp_mov<0x141>(x, x));
  if constexpr (L >= 16) x = op(x, dpp_mov<0x140>(x, x));
  if constexpr (L >= 32) x = op(x, __shfl_xor(x, 16));
  return x;
}
template <int L>
__device__ __forceinline__ int lanes_incl_scan(int x, int l) {
  int y = dpp_mov<0x111>(0, x);
  x += l >= 1 ? y : 0;
  y = dpp_mov<0x112>(0, x);
  x += l >= 2 ? y : 0;
  y = dpp_mov<0x114>(0, x);
  x += l >= 4 ? y : 0;
  if constexpr (L >= 16) {
    y = dpp_mov<0x118>(0, x);
    x += (l & 15) >= 8 ? y : 0;
  }
  if constexpr (L >= 32) x += dpp_mov<0x142, 0xA, 0xF>(0, x);
  return x;
}

// LDS of one wave: the rows' tables, and per rank of walk_spans A's value and the row's table.
template <typename V, bool WITHV>
struct MultiLds {
  __align__(16) int K[kMultiSlots];
  __align__(16) double H[WITHV ? kMultiSlots : 2];
  SpanLds sp;
  V va[WITHV ? 64 : 1];
  int tab[64];
};

// Inserts the products of the wave's rows: lane l holds entries e, e + L, .. < a1 of its row, whose
// table starts at K[tab]. Returns a non-zero value in some lane if a table is full.
template <int T, bool WITHV, typename V>
__device__ __forceinline__ int multi_insert(int lane, int64_t e, int64_t a1, int tab, MultiLds<V, WITHV>& m,
                                            const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
                                            const V* __restrict__ Aval, const int32_t* __restrict__ Bidx,
                                            const V* __restrict__ Bval) {
  constexpr int L = T / 8, U = 4;
  int bad = 0;
  while (__builtin_amdgcn_ballot_w64(e < a1)) {  // wave-uniform
    int len = 0;
    int64_t start = 0;
    V va = V(0);
    if (e < a1) {
      len = blen[e];
      start = bstart[e];
      if (WITHV) va = Aval[e];
    }
    walk_spans<U>(lane, len, start, m.sp,
                  [&](int r) {
                    if (WITHV) m.va[r] = va;
                    m.tab[r] = tab;
                  },
                  [&](const int64_t (&at)[U], const int (&j)[U]) {
                    int c[U], old[U];
                    V b[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                      const int64_t p = at[u] < 0 ? 0 : at[u];
                      c[u] = Bidx[p];
                      b[u] = WITHV ? Bval[p] : V(0);
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u)
                      old[u] = at[u] < 0 ? 0 : atomicCAS(&m.K[m.tab[j[u]] + hslot<T>(c[u])], kEmpty, c[u]);
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                      if (at[u] < 0) continue;
                      const int tb = m.tab[j[u]];
                      uint32_t h = hslot<T>(c[u]);
                      int o = old[u], probe = 0;
                      while (o != kEmpty && o != c[u] && probe < T) {
                        h = (h + 1) & (T - 1);
                        o = atomicCAS(&m.K[tb + h], kEmpty, c[u]);
                        ++probe;
                      }
                      if (probe == T) bad = 1;
                      else if (WITHV) lds_add(&m.H[tb + h], (double)m.va[WITHV ? j[u] : 0] * (double)b[u]);
                    }
                  });
    e += L;
  }
  return bad;
}

template <int T>
__global__ __launch_bounds__(256) void k_symbolic_multi(
    const int32_t* __restrict__ rows, const int64_t* __restrict__ pbeg, const int64_t* __restrict__ pend,
    const int64_t* __restrict__ Aptr, const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
    const int32_t* __restrict__ Bidx, int64_t* __restrict__ nnz, int* __restrict__ err) {
  constexpr int R = kMultiSlots / T, L = 64 / R;
  __shared__ MultiLds<float, false> lds[4];
  const int lane = threadIdx.x & 63, g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  MultiLds<float, false>& m = lds[g];
  const int rl = lane / L, l = lane % L;
  const int64_t beg = *pbeg, end = *pend;
  int bad = 0;
  for (int64_t s0 = beg + (xcd_block() * 4 + g) * R; s0 < end; s0 += (int64_t)gridDim.x * 4 * R) {  // wave-uniform
    const bool have = s0 + rl < end;
    const int row = rows[have ? s0 + rl : s0];
    const int64_t a0 = Aptr[row], a1 = have ? Aptr[row + 1] : a0;
    int4* K4 = reinterpret_cast<int4*>(m.K);
    K4[lane] = K4[lane + 64] = make_int4(kEmpty, kEmpty, kEmpty, kEmpty);
    wave_sync();
    bad |= multi_insert<T, false, float>(lane, a0 + l, a1, rl * T, m, bstart, blen, nullptr, Bidx, nullptr);
    wave_sync();
    const int4 x = K4[2 * lane], y = K4[2 * lane + 1];  // this lane's eight slots of its row's table
    int cnt = (x.x != kEmpty) + (x.y != kEmpty) + (x.z != kEmpty) + (x.w != kEmpty) + (y.x != kEmpty) +
              (y.y != kEmpty) + (y.z != kEmpty) + (y.w != kEmpty);
    cnt = lanes_reduce<L>(cnt, OpAdd());
    if (have && l == 0) nnz[row] = cnt;
    wave_sync();
  }
  if (__builtin_amdgcn_ballot_w64(bad) && lane == 0) atomicOr(err, kErrTableFull);
}

template <typename V, int T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void k_numeric_multi(
    const int32_t* __restrict__ rows, const int64_t* __restrict__ pbeg, const int64_t* __restrict__ pend,
    const int64_t* __restrict__ Aptr, const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
    const V* __restrict__ Aval, const int32_t* __restrict__ Bidx, const V* __restrict__ Bval,
    const int64_t* __restrict__ Cptr, int64_t cbase, int32_t* __restrict__ Cidx, V* __restrict__ Cval,
    int* __restrict__ err) {
  constexpr int R = kMultiSlots / T, L = 64 / R;
  constexpr int NB = T / 2 - 1;  // buckets of a row; the counter behind them ends up as the total
  __shared__ MultiLds<V, true> lds[4];
  const int lane = threadIdx.x & 63, g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  MultiLds<V, true>& m = lds[g];
  const int rl = lane / L, l = lane % L;
  int* K = m.K + rl * T;        // this row's table, then its bucket counters, then its ranked keys
  int* perm = K + T / 2;        // keys by bucket, then the ranked keys' slots
  double* H = m.H + rl * T;
  const int64_t beg = *pbeg, end = *pend;
  int flags = 0;
  for (int64_t s0 = beg + (xcd_block() * 4 + g) * R; s0 < end; s0 += (int64_t)gridDim.x * 4 * R) {  // wave-uniform
    const bool have = s0 + rl < end;
    const int row = rows[have ? s0 + rl : s0];
    const int64_t a0 = Aptr[row], a1 = have ? Aptr[row + 1] : a0;
    const int64_t c0 = Cptr[row] - cbase;
    const int nexp = have ? (int)(Cptr[row + 1] - Cptr[row]) : 0;  // at most T / 2
    int4* K4 = reinterpret_cast<int4*>(m.K);
    K4[lane] = K4[lane + 64] = make_int4(kEmpty, kEmpty, kEmpty, kEmpty);
#pragma unroll
    for (int q = 0; q < 4; ++q) reinterpret_cast<int4*>(m.H)[lane + 64 * q] = make_int4(0, 0, 0, 0);
    wave_sync();
    if (multi_insert<T, true, V>(lane, a0 + l, a1, rl * T, m, bstart, blen, Aval, Bidx, Bval)) flags |= kErrTableFull;
    wave_sync();
    int kk[8], bi[8];
    {
      const int4 x = K4[2 * lane], y = K4[2 * lane + 1];
      kk[0] = x.x, kk[1] = x.y, kk[2] = x.z, kk[3] = x.w, kk[4] = y.x, kk[5] = y.y, kk[6] = y.z, kk[7] = y.w;
    }
    int cmin = INT_MAX, cmax = -1;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      cmin = kk[q] != kEmpty ? min(cmin, kk[q]) : cmin;
      cmax = max(cmax, kk[q]);
    }
    cmin = lanes_reduce<L>(cmin, OpMin());
    cmax = lanes_reduce<L>(cmax, OpMax());
    wave_sync();
    // ---- bucket counts and their prefix ----
    reinterpret_cast<int4*>(K)[l] = make_int4(0, 0, 0, 0);
    const uint32_t range = (uint32_t)(cmax - cmin) + 1u;
    const bool direct = range <= (uint32_t)NB;
    const uint32_t mul = direct ? 0u : (uint32_t)((float)NB * 4294967296.0f / (float)range * 0.99999f);
    wave_sync();
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      bi[q] = 0;
      if (kk[q] != kEmpty) {
        const uint32_t x = (uint32_t)(kk[q] - cmin);
        const int b = direct ? (int)x : (int)__umulhi(x, mul);
        bi[q] = b | (atomicAdd(&K[b], 1) << 16);
      }
    }
    wave_sync();
    {
      const int4 x = reinterpret_cast<int4*>(K)[l];
      const int sum = x.x + x.y + x.z + x.w;
      const int p = lanes_incl_scan<L>(sum, l) - sum;
      wave_sync();
      reinterpret_cast<int4*>(K)[l] = make_int4(p, p + x.x, p + x.x + x.y, p + x.x + x.y + x.z);
    }
    wave_sync();
    // ---- keys by bucket, ranks within the buckets ----
    const int n = K[NB];
    int sl[8];  // start | length << 16
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      sl[q] = 0;
      if (kk[q] != kEmpty) {
        const int b = bi[q] & 0xFFFF;
        const int b0 = K[b], b1 = min(K[b + 1], T / 2);
        sl[q] = b0 | (max(b1 - b0, 0) << 16);
      }
    }
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (kk[q] != kEmpty) {
        const int pos = (sl[q] & 0xFFFF) + (bi[q] >> 16);
        if (pos < T / 2) perm[pos] = kk[q];
      }
    wave_sync();
    int rk[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) rk[q] = kk[q] != kEmpty ? (sl[q] & 0xFFFF) : T;
    for (int j = 0;; ++j) {
      bool more = false;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int len = sl[q] >> 16;
        if (len > 1 && j < len) rk[q] += (perm[(sl[q] & 0xFFFF) + j] < kk[q]);
        more |= (len > 1 && j + 1 < len);
      }
      if (!__builtin_amdgcn_ballot_w64(more)) break;
    }
    wave_sync();
    // ---- key at its rank, slot beside it; stores ----
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (rk[q] < T / 2) {
        K[rk[q]] = kk[q];
        perm[rk[q]] = 8 * l + q;
      }
    wave_sync();
    flags |= (n != nexp) ? kErrCountMismatch : 0;
    const int nw = min(n, nexp);
    for (int k = l; k < nw; k += L) {
      Cidx[c0 + k] = K[k];
      Cval[c0 + k] = (V)H[perm[k]];
    }
    wave_sync();
  }
  flags = wave_reduce_dpp(flags, OpOr());
  if (lane == 0 && flags) atomicOr(err, flags);
}

// Per-row records of the banded long-row windows, 16 bytes each (the workspace holds 16 bytes per
// A nonzero): an entry with a banded B row (start of its B row, its slot, its index in the row),
// and one without (position from its B row's start, index in the row, next column, entries left).
struct HRec {
  int64_t b0;
  int32_t slot;
  int32_t e;
};
struct LRec {
  int32_t prel;
  int32_t e;
  int32_t nc;
  int32_t rem;
};
static_assert(sizeof(HRec) == 16 && sizeof(LRec) == 16, "records share the 16-byte workspace slots");

// Cursor of one A entry of a long row in a column sweep: position in B and entries left of
// its B row, and the column at that position (INT_MAX when the row is exhausted).
struct LongState {
  int64_t p;
  int nc;
  int rem;
};

// Lanes per A entry for a long row of nA entries in a group of NT threads: as many as divide
// the group evenly over the entries (a power of two from 4 to 64).
template <int NT>
__device__ __forceinline__ int long_lanes(int64_t nA) {
  int g = 64;
  while (g > 4 && (int64_t)(NT / g) < nA) g >>= 1;
  return g;
}


// Span walks (long-row windows, symbolic and numeric): elements per window of an A entry whose B
// row has no band index entry; the window ends before the first element such a span leaves out.
// 64 (measured against 16 and 256): B rows shorter than the band index's smallest banded length
// rarely cut a window, and a span re-reads at most 64 elements.
constexpr int kSpanCap = 64;
constexpr int kSymSpanEntries = 64;  // symbolic span walks: rows of up to one wave of entries

// Rows too long for an LDS table: sweep the row's columns in windows of W bits.
// With B's band index, rows of up to kSymSpanEntries entries walk
// element-parallel: every active entry's element span in the window (banded B rows: up to the
// band boundary at or past the window end; other B rows: at most kSpanCap elements, the
// window then ending before the first element left out) is flattened by a scan in wave 0, each
// thread of the workgroup takes U elements at a time, and the entry state (B row start and
// length, elements consumed, next column, band slot) lives in LDS. (A workgroup-wide version for
// rows of up to NT entries measured slower than the cursor walks below: its scans cost more
// barriers per window than the walks' chains.)
// Otherwise one cursor per A entry (16 bytes per A nonzero, so a row's workspace lies beside its
// entries for every kernel that uses it) walks its sorted B
// row, whose extent comes from the row analysis' descriptors; an entry with more elements in the
// window than one step of G continues UL steps at a time, their loads issued together.
template <int NT, int W, int G>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(8))) void k_symbolic_long(
    const int32_t* __restrict__ rows, const int64_t* __restrict__ pbeg, const int64_t* __restrict__ pend,
    const int64_t* __restrict__ Aptr, const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
    const int32_t* __restrict__ Bidx, int64_t* __restrict__ nnz, int64_t* __restrict__ cursor,
    int* __restrict__ err, const int32_t* __restrict__ hub_slot, const int32_t* __restrict__ Aidx, const int32_t* __restrict__ hslot, const int32_t* __restrict__ band,
    int64_t nb1) {
  constexpr int NWORD = W / 32;
  constexpr int WPT = NWORD / NT;
  constexpr int UL = 8;
  constexpr int U = 4;
  static_assert(NWORD % NT == 0 && NT % 64 == 0, "shape");
  __shared__ uint32_t bm[NWORD];
  __shared__ int sc[NT / 64 > 0 ? NT / 64 : 1];
  __shared__ long long scl[NT / 64 > 0 ? NT / 64 : 1];
  // span-walk entry state and window tables (entry e in slot e)
  __shared__ int64_t eB0[kSymSpanEntries];
  __shared__ int eL[kSymSpanEntries], eP[kSymSpanEntries], eNC[kSymSpanEntries], eSL[kSymSpanEntries];
  __shared__ int sS[kSymSpanEntries], sN[kSymSpanEntries];
  __shared__ int s_T, s_lo;
  __shared__ long long s_hi;
  const int t = threadIdx.x, lg = t % G, lane = t & 63;
  const int64_t beg = *pbeg, end = *pend;
  for (int64_t slot = beg + blockIdx.x; slot < end; slot += gridDim.x) {
    const int row = rows[slot];
    if (hub_slot && hub_slot[row] >= 0) continue;  // uniform: k_hub_count counts the hub rows
    const int64_t a0 = Aptr[row], a1 = Aptr[row + 1];
#pragma unroll
    for (int q = 0; q < WPT; ++q) bm[t + q * NT] = 0u;
    const int nA = (int)min(a1 - a0, (int64_t)kSymSpanEntries + 1);
    if (band != nullptr && nA <= kSymSpanEntries) {  // uniform
      // ================= span walks (entries in slots 0 .. nA - 1, wave 0) =================
      long long prow_l = 0;
      if (t < nA) {
        const int64_t ka = a0 + t;
        const int64_t b0 = bstart[ka];
        const int L = blen[ka];
        eB0[t] = b0;
        eL[t] = L;
        eP[t] = 0;
        eSL[t] = hslot[Aidx[ka]];
        eNC[t] = L > 0 ? Bidx[b0] : INT_MAX;
        prow_l = L;
      }
      if (t < 64) {
        const int m = wave_reduce_dpp(t < nA ? eNC[t] : INT_MAX, OpMin());
        if (t == 0) s_lo = m;
      }
      const long long prow = Group<NT>::reduce(prow_l, OpAdd(), scl);  // also orders the writes
      int lo = s_lo;
      long long count = 0;
      long long windows = 0;
      while (lo != INT_MAX) {
        // ---- the active entries' element spans; the window ends before any element a capped
        // span leaves out ----
        if (t < 64) {
          const int64_t hi0 = min((int64_t)lo + W, (int64_t)INT_MAX);
          int len = 0, clip = INT_MAX;
          if (t < nA && (int64_t)eNC[t] < hi0) {
            const int p = eP[t], L = eL[t], sl = eSL[t];
            int q;
            if (sl >= 0) {
              q = band[(int64_t)sl * nb1 + min((hi0 + (1 << kBandShift) - 1) >> kBandShift, nb1 - 1)];
            } else {
              q = min(L, p + kSpanCap);
              if (q < L) clip = Bidx[eB0[t] + q];
            }
            len = q - p;
          }
          const int cm = wave_reduce_dpp(clip, OpMin());
          const int incl = wave_incl_scan_dpp(len);
          if (t < nA) {
            sS[t] = incl - len;
            sN[t] = 0;
          }
          if (t == 63) {
            s_T = incl;
            s_hi = min(hi0, (int64_t)cm);
          }
        }
        __syncthreads();
        const int T = s_T;
        const int64_t hi = s_hi;
        // ---- presence bits, element-parallel ----
        for (int f0 = 0; f0 < T; f0 += NT * U) {  // uniform
          int c[U], jj[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int f = f0 + u * NT + t;
            int j = 0;  // the last entry with sS[j] <= f
#pragma unroll
            for (int step = kSymSpanEntries / 2; step >= 1; step >>= 1)
              if (j + step < nA && sS[j + step] <= f) j += step;
            jj[u] = j;
            const int64_t at = f < T ? eB0[j] + eP[j] + (f - sS[j]) : 0;  // lanes past T: unused read
            c[u] = Bidx[at];
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int f = f0 + u * NT + t;
            const int j = jj[u];
            const bool in = f < T && (int64_t)c[u] < hi;
            if (in) {
              const int o = c[u] - lo;
              atomicOr(&bm[o >> 5], 1u << (o & 31));
            }
            // an entry's elements below hi are a prefix of its span: the last such lane of each
            // wave records its length
            const int jn = __shfl_down(j, 1);
            const int inn = __shfl_down((int)in, 1);
            if (in && (lane == 63 || !inn || jn != j)) atomicMax(&sN[j], f - sS[j] + 1);
          }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < WPT; ++q) {
          count += __popc(bm[t + q * NT]);
          bm[t + q * NT] = 0u;
        }
        // ---- cursors advance past the window; the next window starts at the smallest next column ----
        if (t < 64) {
          int nl = INT_MAX;
          if (t < nA) {
            const int took = sN[t];
            nl = eNC[t];
            if (took > 0) {
              const int p = eP[t] + took;
              eP[t] = p;
              nl = p < eL[t] ? Bidx[eB0[t] + p] : INT_MAX;
              eNC[t] = nl;
            }
          }
          const int m = wave_reduce_dpp(nl, OpMin());
          if (t == 0) s_lo = m;
        }
        __syncthreads();  // also: the bitmap is clear
        lo = s_lo;
        if (++windows > prow) {  // uniform: no progress; reported, the row's count is not trusted
          if (t == 0) atomicOr(err, kErrWindow);
          break;
        }
      }
      count = Group<NT>::reduce(count, OpAdd(), scl);
      if (t == 0) nnz[row] = count;
      __syncthreads();
      continue;
    }
    int lo_l = INT_MAX;
    long long prow_l = 0;
    for (int64_t ka = a0 + t; ka < a1; ka += NT) {
      const int64_t b0 = bstart[ka];
      cursor[2 * ka] = b0;
      prow_l += blen[ka];
      if (blen[ka] > 0) lo_l = min(lo_l, Bidx[b0]);
    }
    // every window takes at least the element at its first column, so a row of P_i products
    // needs at most P_i windows; more would mean a walk that stopped making progress
    const long long prow = Group<NT>::reduce(prow_l, OpAdd(), scl);
    int lo = Group<NT>::reduce(lo_l, OpMin(), sc);  // also orders the cursor writes
    long long count = 0;
    long long windows = 0;
    while (lo != INT_MAX) {
      const int64_t hi = min((int64_t)lo + W, (int64_t)INT_MAX);  // INT_MAX: past the B row
      for (int64_t ka = a0 + t / G; ka < a1; ka += NT / G) {
        int64_t p = cursor[2 * ka];
        const int64_t b1 = bstart[ka] + blen[ka];
        int nin;
        {
          const int64_t q = p + lg;
          const int c = (q < b1) ? Bidx[q] : INT_MAX;
          const bool in = (int64_t)c < hi;
          if (in) {
            const int o = c - lo;
            atomicOr(&bm[o >> 5], 1u << (o & 31));
          }
          nin = __popcll(__ballot(in) & subgroup_mask<G>());
          p += nin;
        }
        // B rows with more elements in the window than one step: UL steps at a time. p grows by
        // G per full step and never passes b1 on this path, so the walk ends within len / G steps
        // whatever the sentinel column past the row compares as.
        while (nin == G && p < b1) {  // subgroup-uniform
          int cc[UL];
#pragma unroll
          for (int k = 0; k < UL; ++k) {
            const int64_t q = p + k * G + lg;
            cc[k] = (q < b1) ? Bidx[q] : INT_MAX;
          }
#pragma unroll
          for (int k = 0; k < UL; ++k) {
            if (nin == G) {
              const bool in = (int64_t)cc[k] < hi;
              if (in) {
                const int o = cc[k] - lo;
                atomicOr(&bm[o >> 5], 1u << (o & 31));
              }
              nin = __popcll(__ballot(in) & subgroup_mask<G>());
              p += nin;
            }
          }
        }
        if (lg == 0) cursor[2 * ka] = p;
      }
      __syncthreads();
      long long pc = 0;
#pragma unroll
      for (int q = 0; q < WPT; ++q) {
        const int wq = __popc(bm[t + q * NT]);
        pc += wq;
        bm[t + q * NT] = 0u;
      }
      count += pc;
      int nl = INT_MAX;
      for (int64_t ka = a0 + t; ka < a1; ka += NT) {
        const int64_t p = cursor[2 * ka];
        if (p < bstart[ka] + blen[ka]) nl = min(nl, Bidx[p]);
      }
      lo = Group<NT>::reduce(nl, OpMin(), sc);
      if (++windows > prow) {  // uniform: no progress; reported, the row's count is not trusted
        if (t == 0) atomicOr(err, kErrWindow);
        break;
      }
    }
    count = Group<NT>::reduce(count, OpAdd(), scl);
    if (t == 0) nnz[row] = count;
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------
// hub rows: long rows computed in column ranges
// ------------------------------------------------------------------------------------
// A window kernel sweeps its row with one workgroup, window after window, and visits the row's A
// entries in every window: one round trip to memory after another, on one CU, however many are
// idle. Hub rows are cut into ranges of kHubRange columns instead, a workgroup per (row, range)
// that accumulates in LDS, so a heavy row spreads over the GPU and no product needs a global
// atomic:
//   - k_hub_split lists each row's entries by kind, 16 bytes each beside the row's A entries: those
//     whose B row is in the band index (a range's element span is two index entries) from the
//     front, the others (short B rows) from the back; and the row's first and last column;
//   - k_hub_count counts the columns of every range (bitmap windows of one or several ranges), for
//     nnz_i and, scanned, the ranges' output offsets;
//   - over more than kHubWhole ranges the short B rows' products, (column, a_ik * b_kj), are
//     bucketed per (row, range) by k_hub_bucket; over fewer each range reads the short rows whole
//     and keeps its part (a short row's few cache lines cost less than writing and reading 12
//     bytes per product);
//   - k_hub_range accumulates a range and emits it in column order at its offset.
// Which rows: hub_row (kernels.h). Sums of a column may associate differently from run to run (the
// order of LDS atomics), within the usual rounding bound.
constexpr int kHubRangeBands = kHubRange >> kBandShift;
constexpr int kHubSplitNT = 256;
constexpr int kHubSplitPer = 4;
constexpr int kHubChunk = kHubSplitNT * kHubSplitPer;  // entries of a row per k_hub_split workgroup
constexpr int kHubBucketChunk = 512;                   // short entries of a row per k_hub_bucket workgroup
constexpr int kHubWhole = 8;

// The kinds of entries as k_hub_split lists them: start of the B row, its band slot or (short) its
// length, index in the A row.
struct HubRec {
  int64_t b0;
  int32_t s;
  int32_t e;
};
static_assert(sizeof(HubRec) == 16, "records share the 16-byte workspace slots");

// Per hub row: workgroups that split it (none for a row that is not long: only after a captured
// pipeline's operands changed structure), and its counters and column span cleared; also the
// number of rows of many entries that the numeric binning counts.
__global__ void k_hub_chunks(const int32_t* __restrict__ hub_rows, int64_t n, const int64_t* __restrict__ Aptr,
                             const int64_t* __restrict__ P, int64_t ncols, int64_t key_lim, int64_t* __restrict__ cnt,
                             int32_t* __restrict__ hcnt, int32_t* __restrict__ lcnt, int32_t* __restrict__ span,
                             int64_t* __restrict__ nnz, int* __restrict__ many) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *many = 0;
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x) {
    const int r = hub_rows[j];
    const bool is_long = min(P[r], ncols) > key_lim;
    cnt[j] = is_long ? (Aptr[r + 1] - Aptr[r] + kHubChunk - 1) / kHubChunk : 0;
    if (is_long) nnz[r] = 0;  // k_hub_count adds the ranges' columns up
    hcnt[j] = lcnt[j] = 0;
    span[2 * j] = INT_MAX;
    span[2 * j + 1] = -1;
  }
}

// The list entry whose chunks hold chunk q (off: exclusive scan of the chunk counts, n + 1 entries).
__device__ __forceinline__ int64_t chunk_owner(const int64_t* __restrict__ off, int64_t n, int64_t q) {
  int64_t lo = 0, hi = n - 1;
  while (lo < hi) {
    const int64_t m = (lo + hi + 1) >> 1;
    if (off[m] <= q) lo = m;
    else hi = m - 1;
  }
  return lo;
}

__global__ __launch_bounds__(kHubSplitNT) void k_hub_split(
    const int32_t* __restrict__ hub_rows, int64_t n, const int64_t* __restrict__ coff, const int64_t* __restrict__ Aptr,
    const int32_t* __restrict__ Aidx, const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
    const int32_t* __restrict__ Bidx, const int32_t* __restrict__ hslot, HubRec* __restrict__ recs,
    int32_t* __restrict__ hcnt, int32_t* __restrict__ lcnt, int32_t* __restrict__ span) {
  __shared__ int s_n[2], s_base[2];
  const int64_t q = blockIdx.x;
  if (q >= coff[n]) return;  // the grid is a bound
  const int64_t j = chunk_owner(coff, n, q);
  const int row = hub_rows[j];
  const int64_t a0 = Aptr[row], nA = Aptr[row + 1] - a0, e0 = (q - coff[j]) * kHubChunk;
  const int t = threadIdx.x, lane = t & 63;
  if (t < 2) s_n[t] = 0;
  __syncthreads();
  HubRec rec[kHubSplitPer];
  int kind[kHubSplitPer], pos[kHubSplitPer];  // 0: banded, 1: short, -1: no product
  int cmin = INT_MAX, cmax = -1;
#pragma unroll
  for (int i = 0; i < kHubSplitPer; ++i) {
    const int64_t e = e0 + t + i * kHubSplitNT;
    kind[i] = -1;
    if (e < nA) {
      const int64_t ka = a0 + e;
      const int L = blen[ka];
      const int sl = hslot[Aidx[ka]];
      if (L > 0) {
        kind[i] = sl >= 0 ? 0 : 1;
        rec[i] = HubRec{bstart[ka], sl >= 0 ? sl : L, (int)e};
        cmin = min(cmin, Bidx[rec[i].b0]);
        cmax = max(cmax, Bidx[rec[i].b0 + L - 1]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kHubSplitPer; ++i) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint64_t b = __builtin_amdgcn_ballot_w64(kind[i] == k);
      int at = 0;
      if (lane == 0) at = atomicAdd(&s_n[k], (int)__popcll(b));
      at = __builtin_amdgcn_readfirstlane(at);
      if (kind[i] == k) pos[i] = at + __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0));
    }
  }
  __syncthreads();
  if (t == 0) s_base[0] = atomicAdd(&hcnt[j], s_n[0]);
  if (t == 1) s_base[1] = atomicAdd(&lcnt[j], s_n[1]);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kHubSplitPer; ++i) {
    if (kind[i] == 0) recs[a0 + s_base[0] + pos[i]] = rec[i];
    if (kind[i] == 1) recs[a0 + nA - 1 - (s_base[1] + pos[i])] = rec[i];
  }
  cmin = wave_reduce_dpp(cmin, OpMin());
  cmax = wave_reduce_dpp(cmax, OpMax());
  if (lane == 0 && cmax >= 0) {
    atomicMin(&span[2 * j], cmin);
    atomicMax(&span[2 * j + 1], cmax);
  }
}

// A row whose windows of `wide` ranges would hold more than 1/kHubFine of all products each: it is
// counted range by range.
constexpr int kHubFine = 1024;
__device__ __forceinline__ bool hub_fine(int64_t P, int nrng, int wide, int64_t products) {
  return P / ((nrng + wide - 1) / wide) > products / kHubFine;
}

// Columns per range of the hub rows: a workgroup per (row, window of SW ranges), presence bits in
// LDS. rng_cnt[slot * nrng + range] receives the counts (0 beforehand), nnz[row] their sum. The wide
// instance (fewer visits of the entries) leaves out the fine rows, the FINE one takes them from
// their list: with windows of 131,072 columns alone the heaviest row of an R-MAT 20 sample would be
// 8 workgroups' work while the other rows of the launch are long done. Windows of 16 ranges (16 KB
// of bits) keep four workgroups on a CU; over many ranges and rows (hub_wide) the visits of the
// entries and of the short rows, once per window, cost more than that, and 64 ranges are taken
// (R-MAT 22: 0.84 s of symbolic pass with 16, 0.73 s with 64).
template <int NT, int SW, bool FINE>
__global__ __launch_bounds__(NT) void k_hub_count(
    const int32_t* __restrict__ hub_rows, const int32_t* __restrict__ fine, int nwin, int nrng,
    const int64_t* __restrict__ Aptr,
    const int32_t* __restrict__ Bidx, const HubRec* __restrict__ recs, const int32_t* __restrict__ hcnt,
    const int32_t* __restrict__ lcnt, const int32_t* __restrict__ span, const int32_t* __restrict__ band, int64_t nb1,
    const int32_t* __restrict__ hub_slot, int32_t* __restrict__ rng_cnt, int64_t* __restrict__ nnz) {
  constexpr int W = SW * kHubRange;
  constexpr int NWORD = W / 32;
  constexpr int WPT = NWORD > NT ? NWORD / NT : 1;  // bitmap words per thread, in one range
  constexpr int RT = kHubRange / 32 / WPT;          // threads that count one range
  constexpr int U = 4;
  constexpr int RL = RT < 32 ? RT : 32;             // of them, lanes that add up before the LDS add
  static_assert(NT % 64 == 0 && (NWORD % NT == 0 || NT % NWORD == 0) && RT >= 1, "a thread's words lie in one range");
  __shared__ __align__(16) uint32_t bm[NWORD];
  __shared__ SpanLds sl[NT / 64];
  __shared__ int rc[SW];
  const int t = threadIdx.x, lane = t & 63;
  const int64_t i = blockIdx.x / nwin;
  const int w = (int)(blockIdx.x - i * nwin);
  const int64_t j = FINE ? fine[i] : i;
  const int row = hub_rows[j];
  const int64_t lo = (int64_t)w * W, hi = lo + W;
  if (span[2 * j + 1] < lo || span[2 * j] >= hi) return;
  if (!FINE && (hub_slot[row] & kHubFineBit)) return;
  const int64_t a0 = Aptr[row], a1 = Aptr[row + 1];
  const int nH = hcnt[j], nL = lcnt[j];
  for (int q = t; q < NWORD; q += NT) bm[q] = 0u;
  if (t < SW) rc[t] = 0;
  __syncthreads();
  const int64_t w0 = lo >> kBandShift, w1 = min(hi >> kBandShift, nb1 - 1);
  for (int e0 = 0; e0 < nH; e0 += NT) {  // uniform; strided, so heavy neighbours spread over the waves
    const int e = e0 + (t >> 6) + (NT / 64) * lane;
    int len = 0;
    int64_t start = 0;
    if (e < nH) {
      const HubRec r = recs[a0 + e];
      const int32_t* bd = band + (int64_t)r.s * nb1;
      const int s0 = bd[w0];
      len = bd[w1] - s0;
      start = r.b0 + s0;
    }
    walk_spans<U>(lane, len, start, sl[t >> 6], [](int) {},
                  [&](const int64_t (&at)[U], const int (&)[U]) {
                    int c[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) c[u] = Bidx[at[u] < 0 ? 0 : at[u]];
#pragma unroll
                    for (int u = 0; u < U; ++u)
                      if (at[u] >= 0) {
                        const int o = (int)(c[u] - lo);
                        atomicOr(&bm[o >> 5], 1u << (o & 31));
                      }
                  });
  }
  for (int e0 = 0; e0 < nL; e0 += NT) {  // short rows whole
    const int e = e0 + t;
    const HubRec r = e < nL ? recs[a1 - 1 - e] : HubRec{0, 0, 0};
    walk_spans<U>(lane, r.s, r.b0, sl[t >> 6], [](int) {},
                  [&](const int64_t (&at)[U], const int (&)[U]) {
                    int c[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) c[u] = Bidx[at[u] < 0 ? 0 : at[u]];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                      const int64_t o = c[u] - lo;
                      if (at[u] >= 0 && o >= 0 && o < W) atomicOr(&bm[o >> 5], 1u << (o & 31));
                    }
                  });
  }
  __syncthreads();
  int pc = 0;
#pragma unroll
  for (int q = 0; q < WPT; ++q) pc += t * WPT < NWORD ? __popc(bm[t * WPT + q]) : 0;
#pragma unroll
  for (int o = RL / 2; o > 0; o >>= 1) pc += __shfl_xor(pc, o);
  if ((lane & (RL - 1)) == 0 && pc) atomicAdd(&rc[t / RT], pc);
  __syncthreads();
  if (t < SW) {
    const int r = w * SW + t;
    if (r < nrng && rc[t]) {
      rng_cnt[j * nrng + r] = rc[t];
      atomicAdd((unsigned long long*)&nnz[row], (unsigned long long)rc[t]);
    }
  }
}

// Workgroups per listed row for its short entries.
__global__ void k_hub_bucket_chunks(const int32_t* __restrict__ rows, int64_t n, const int32_t* __restrict__ hub_slot,
                                    const int32_t* __restrict__ lcnt, int64_t* __restrict__ cnt) {
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x) {
    const int hs = hub_slot[rows[j]];
    cnt[j] = hs >= 0 ? (lcnt[hs & kHubSlotMask] + kHubBucketChunk - 1) / kHubBucketChunk : 0;
  }
}

// Products of the short entries per (row, range). WRITE = false adds their counts to scnt (0
// beforehand). WRITE = true puts them into the buckets at soff, the scan of scnt: a workgroup
// counts its own, takes its places off scnt (which runs down to 0), and writes.
template <typename V, bool WRITE>
__global__ __launch_bounds__(256) void k_hub_bucket(
    const int32_t* __restrict__ rows, int64_t n, const int64_t* __restrict__ coff, const int64_t* __restrict__ Aptr,
    const V* __restrict__ Aval, const int32_t* __restrict__ Bidx, const V* __restrict__ Bval,
    const HubRec* __restrict__ recs, const int32_t* __restrict__ hub_slot, const int32_t* __restrict__ lcnt, int nrng,
    int64_t* __restrict__ scnt, const int64_t* __restrict__ soff, int32_t* __restrict__ scol, V* __restrict__ sval,
    const int* __restrict__ err) {
  constexpr int NT = 256, U = 4;
  extern __shared__ unsigned long long lc[];  // nrng counts, then places
  __shared__ SpanLds sl[NT / 64];
  __shared__ V tva[NT];
  if (WRITE && (*err & kErrCapacity)) return;  // the buckets (or C) are smaller than this structure needs
  const int64_t q = blockIdx.x;
  if (q >= coff[n]) return;  // the grid is a bound
  const int64_t j = chunk_owner(coff, n, q);
  const int row = rows[j], hs = hub_slot[row] & kHubSlotMask;
  const int t = threadIdx.x, lane = t & 63;
  const int64_t a0 = Aptr[row], a1 = Aptr[row + 1];
  const int l0 = (int)(q - coff[j]) * kHubBucketChunk, l1 = min(l0 + kHubBucketChunk, lcnt[hs]);
  for (int r = t; r < nrng; r += NT) lc[r] = 0ull;
  __syncthreads();
  for (int e0 = l0; e0 < l1; e0 += NT) {
    const HubRec r = e0 + t < l1 ? recs[a1 - 1 - (e0 + t)] : HubRec{0, 0, 0};
    walk_spans<U>(lane, r.s, r.b0, sl[t >> 6], [](int) {},
                  [&](const int64_t (&at)[U], const int (&)[U]) {
                    int c[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) c[u] = Bidx[at[u] < 0 ? 0 : at[u]];
#pragma unroll
                    for (int u = 0; u < U; ++u)
                      if (at[u] >= 0) atomicAdd(&lc[c[u] >> kHubRangeShift], 1ull);
                  });
  }
  __syncthreads();
  for (int r = t; r < nrng; r += NT) {
    const unsigned long long c = lc[r];
    if (!c) continue;
    unsigned long long* g = (unsigned long long*)&scnt[j * nrng + r];
    if (WRITE) lc[r] = (unsigned long long)soff[j * nrng + r] + atomicAdd(g, 0ull - c) - c;
    else atomicAdd(g, c);
  }
  if (!WRITE) return;
  __syncthreads();
  V* wva = tva + (t & ~63);
  for (int e0 = l0; e0 < l1; e0 += NT) {
    const HubRec r = e0 + t < l1 ? recs[a1 - 1 - (e0 + t)] : HubRec{0, 0, 0};
    const V va = e0 + t < l1 ? Aval[a0 + r.e] : V(0);
    walk_spans<U>(lane, r.s, r.b0, sl[t >> 6], [&](int k) { wva[k] = va; },
                  [&](const int64_t (&at)[U], const int (&jj)[U]) {
                    int c[U];
                    V p[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                      const int64_t x = at[u] < 0 ? 0 : at[u];
                      c[u] = Bidx[x];
                      p[u] = wva[jj[u]] * Bval[x];
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u)
                      if (at[u] >= 0) {
                        const int64_t pos = (int64_t)atomicAdd(&lc[c[u] >> kHubRangeShift], 1ull);
                        scol[pos] = c[u];
                        sval[pos] = p[u];
                      }
                  });
  }
}

// What a range workgroup needs to know of its row, in one 32-byte load: A entries [a0, a1), where the
// row's output starts, banded and short entries.
struct HubRow {
  int64_t a0, a1, out;
  int32_t nH, nL;
};
static_assert(sizeof(HubRow) == 32, "one load");

// One (row, range) item per workgroup: the range's values, emitted from info.out + roff[item] -
// roff[first item of the row] on, with roff[item + 1] - roff[item] columns expected. soff null: no
// buckets, the short rows are read here.
//
// Bound by the latency of an item's chain (row, records, band ends, gathers, stores), so two
// workgroups share a CU (80 KB of LDS each), with all of its 32 waves as long as positions in B fit 32
// bits (the walks' tables; with 64 bits half the waves: R-MAT 16 1.80 ms against 1.61, samples of R-MAT
// 20 rows 4.42 against 3.97), and nothing else is kept in LDS: a column is present
// when its sum is no longer -0.0, the initial value, which no sum reaches (products of -0.0 are
// made +0.0 first), so there is no bitmap to OR (127 clocks a wave for 64 neighbouring columns) and
// a thread emits the sums it reads. The sums are FP64 for FP32 operands too: ds_add_f32 takes 194
// clocks a wave, ds_add_f64 9 to 21 (and the rounding is better).
template <typename V, int NT, typename I>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(NT / 128))) void k_hub_range(
    const HubRow* __restrict__ info, int nrng, const V* __restrict__ Aval, const int32_t* __restrict__ Bidx,
    const V* __restrict__ Bval, const int32_t* __restrict__ band, int64_t nb1, const HubRec* __restrict__ recs,
    const int64_t* __restrict__ soff, const int32_t* __restrict__ scol, const V* __restrict__ sval,
    const int64_t* __restrict__ roff, int32_t* __restrict__ Cidx, V* __restrict__ Cval, int* __restrict__ err) {
  constexpr int NW = NT / 64;
  constexpr int U = 4;
  constexpr int PT = kHubRange / NT;  // columns per thread
  static_assert(NT % 64 == 0 && kHubRange % NT == 0 && PT * NW <= 128, "shape");
  __shared__ __align__(16) double dv[kHubRange];
  __shared__ SpanLdsT<I> sl[NW];
  __shared__ double tva[NT];
  int* wcnt = reinterpret_cast<int*>(tva);  // 128, once the walks are done
  const int64_t item = blockIdx.x;
  const int64_t j = item / nrng;
  const int64_t r0 = roff[item], nexp = roff[item + 1] - r0, rfirst = roff[j * nrng];
  const HubRow row = info[j];
  // a range without columns (by the symbolic count) holds no product: nothing to add or emit
  if (nexp == 0) return;
  if (*err & kErrCapacity) return;  // the buckets or C are smaller than this structure needs
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int64_t c0 = (item - j * nrng) << kHubRangeShift;
  const int64_t w0 = c0 >> kBandShift;
  const int64_t w1 = min(w0 + kHubRangeBands, nb1 - 1);
  double* wva = tva + (t & ~63);
#pragma unroll
  for (int q = 0; q < PT / 2; ++q) reinterpret_cast<double2*>(dv)[t + q * NT] = make_double2(-0.0, -0.0);
  __syncthreads();
  auto add = [&](int o, double p) { lds_add(&dv[o], p + 0.0); };  // -0.0 + 0.0 is +0.0
  // products of the banded entries in this range: chunks of NT entries, each wave taking 64 of
  // them, strided, so the heaviest (which lie together) spread over the waves
  for (int e0 = 0; e0 < row.nH; e0 += NT) {  // uniform
    const int e = e0 + wv + NW * lane;
    int len = 0;
    int64_t start = 0;
    double va = 0.0;
    if (e < row.nH) {
      const HubRec q = recs[row.a0 + e];
      const int32_t* bd = band + (int64_t)q.s * nb1;
      const int s0 = bd[w0];
      len = bd[w1] - s0;
      start = q.b0 + s0;
      va = (double)Aval[row.a0 + q.e];
    }
    walk_spans<U>(lane, len, start, sl[wv], [&](int k) { wva[k] = va; },
                  [&](const int64_t (&at)[U], const int (&jj)[U]) {
                    int c[U];
                    V b[U];
                    double av[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                      const int64_t p = at[u] < 0 ? 0 : at[u];
                      c[u] = Bidx[p];
                      b[u] = Bval[p];
                      av[u] = wva[jj[u]];
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u)
                      if (at[u] >= 0) add((int)(c[u] - c0), av[u] * (double)b[u]);
                  });
  }
  // products of the short entries: the range's bucket, or its part of the rows themselves
  if (soff) {
    const int64_t q1 = soff[item + 1];
    for (int64_t q = soff[item] + t; q < q1; q += NT) add((int)(scol[q] - c0), (double)sval[q]);
  } else {
    for (int e0 = 0; e0 < row.nL; e0 += NT) {  // uniform
      const int e = e0 + wv + NW * lane;
      const HubRec q = e < row.nL ? recs[row.a1 - 1 - e] : HubRec{0, 0, 0};
      const double va = e < row.nL ? (double)Aval[row.a0 + q.e] : 0.0;
      walk_spans<U>(lane, q.s, q.b0, sl[wv], [&](int k) { wva[k] = va; },
                    [&](const int64_t (&at)[U], const int (&jj)[U]) {
                      int c[U];
                      V b[U];
                      double av[U];
#pragma unroll
                      for (int u = 0; u < U; ++u) {
                        const int64_t p = at[u] < 0 ? 0 : at[u];
                        c[u] = Bidx[p];
                        b[u] = Bval[p];
                        av[u] = wva[jj[u]];
                      }
#pragma unroll
                      for (int u = 0; u < U; ++u) {
                        const int64_t o = c[u] - c0;
                        if (at[u] >= 0 && o >= 0 && o < kHubRange) add((int)o, av[u] * (double)b[u]);
                      }
                    });
    }
  }
  __syncthreads();
  // emission, a lane per column: a wave's stores lie side by side
  double v[PT];
  uint64_t m[PT];
#pragma unroll
  for (int q = 0; q < PT; ++q) {
    v[q] = dv[t + q * NT];
    m[q] = __builtin_amdgcn_ballot_w64(__double_as_longlong(v[q]) != (long long)0x8000000000000000ull);
    if (lane == 0) wcnt[q * NW + wv] = __popcll(m[q]);
  }
  __syncthreads();
  if (wv == 0) {  // exclusive scan of the 128 counts in place; the total goes to flags
    const int x0 = 2 * lane < PT * NW ? wcnt[2 * lane] : 0, x1 = 2 * lane + 1 < PT * NW ? wcnt[2 * lane + 1] : 0;
    const int incl = wave_incl_scan_dpp(x0 + x1);
    wcnt[2 * lane] = incl - x0 - x1;
    wcnt[2 * lane + 1] = incl - x1;
    if (lane == 63 && (int64_t)incl != nexp) atomicOr(err, kErrWindow);
  }
  __syncthreads();
  const int64_t out = row.out + r0 - rfirst;
#pragma unroll
  for (int q = 0; q < PT; ++q) {
    const int k = wcnt[q * NW + wv] + __builtin_amdgcn_mbcnt_hi((uint32_t)(m[q] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m[q], 0));
    if ((m[q] >> lane & 1ull) && k < nexp) {
      Cidx[out + k] = (int)(c0 + t + q * NT);
      Cval[out + k] = (V)v[q];
    }
  }
}

// ------------------------------------------------------------------------------------
// numeric: accumulate in an LDS hash, sort by a monotone bucket map + in-bucket rank,
// emit coalesced
// ------------------------------------------------------------------------------------
// Rank distinct keys held in registers (IPT per lane, kEmpty = none, at most T/2 in all) in
// column order, using the T ints at K (free for the call) for the bucket counters (lower half)
// and the bucket permutation (upper half). The bucket map b(x) = floor(x * mul / 2^32),
// x = c - cmin (or b = x when the column range fits the buckets) is monotone, so a key's rank is
// the start of its bucket plus the number of smaller keys in the bucket; mul only has to keep b
// below NB, so it is formed in single precision and rounded down. LDS reads of all keys are
// issued before their results are used. rk[q] = rank of kk[q], -1 if empty. Returns the number
// of keys (more than T/2 means a table was overfilled; ranks are then not exact and the caller
// reports it).
template <int T, int IPT>
__device__ __forceinline__ int wave_rank_keys(int t, int* K, int cmin, int cmax, const int (&kk)[IPT],
                                              int (&rk)[IPT]) {
  constexpr int H2 = T / 2;
  constexpr int NB = H2 - 1;           // buckets; BC[NB] receives the total
  constexpr int PER = (H2 + 63) / 64;  // counters per lane in the scan
  static_assert(NB < 65536 && T <= 65536, "bucket and in-bucket index share one int");
  const uint32_t range = (uint32_t)(cmax - cmin) + 1u;
  const bool direct = range <= (uint32_t)NB;
  const uint32_t mul =
      direct ? 0u : (uint32_t)((float)NB * 4294967296.0f / (float)range * 0.99999f);
  int* BC = K;
  int* perm = K + H2;
#pragma unroll
  for (int q = 0; q < PER; ++q)
    if (t * PER + q < H2) BC[t * PER + q] = 0;
  wave_sync();
  int bi[IPT];  // bucket | (arrival order in the bucket) << 16
#pragma unroll
  for (int q = 0; q < IPT; ++q) {
    const uint32_t x = (uint32_t)(kk[q] - cmin);
    const int b = direct ? (int)x : (int)__umulhi(x, mul);
    bi[q] = b;
    if (kk[q] != kEmpty) bi[q] = b | (atomicAdd(&BC[b], 1) << 16);
  }
  wave_sync();
  int total;
  {
    int loc[PER];
    int sum = 0;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int i = t * PER + q;
      loc[q] = (i < NB) ? BC[i] : 0;
      sum += loc[q];
    }
    const int incl = wave_incl_scan_dpp(sum);
    total = __builtin_amdgcn_readlane(incl, 63);
    int pre = incl - sum;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int i = t * PER + q;
      if (i < NB) BC[i] = pre;
      pre += loc[q];
    }
    if (t == 0) BC[NB] = total;
  }
  wave_sync();
  // bucket start and length of every live slot (reads first, then the permutation writes)
  int sl[IPT];  // start | length << 16
#pragma unroll
  for (int q = 0; q < IPT; ++q) {
    sl[q] = 0;
    if (kk[q] != kEmpty) {
      const int b = bi[q] & 0xFFFF;
      const int s0 = BC[b], s1 = min(BC[b + 1], H2);
      sl[q] = s0 | (max(s1 - s0, 0) << 16);
    }
  }
#pragma unroll
  for (int q = 0; q < IPT; ++q)
    if (kk[q] != kEmpty) {
      const int pos = (sl[q] & 0xFFFF) + (bi[q] >> 16);
      if (pos < H2) perm[pos] = kk[q];
    }
  wave_sync();
  // in-bucket rank: only buckets holding more than one key need comparisons; position j of
  // every such bucket is read for all slots at once
#pragma unroll
  for (int q = 0; q < IPT; ++q) rk[q] = (kk[q] != kEmpty) ? (sl[q] & 0xFFFF) : -1;
  for (int j = 0;; ++j) {
    bool more = false;
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
      const int len = sl[q] >> 16;
      if (len > 1 && j < len) rk[q] += (perm[(sl[q] & 0xFFFF) + j] < kk[q]);
      more |= (len > 1 && j + 1 < len);
    }
    if (!__builtin_amdgcn_ballot_w64(more)) break;
  }
  return total;
}

// Sort the live entries of a group's row table (T slots, NT > 64 threads, at most T/2 live)
// by column and write them to Cidx/Cval[0 .. min(n, limit)); returns n. Buckets by the
// monotone map b(c) = floor((c - cmin) * NB / range), NB = T/2 counters in BC (NB + 1 ints),
// then the rank inside a bucket by comparison. The table's key and value LDS are reused.
// Leaves the table (K, H) unspecified and BC dirty; the caller clears them.
template <typename V, int T, int NT>
__device__ __forceinline__ int block_rank_emit(int t, int* K, double* H, int* BC, int* sc, int cmin, int cmax,
                                               int32_t* __restrict__ Cidx, V* __restrict__ Cval, int64_t limit) {
  constexpr int IPT = T / NT;
  constexpr int NB = T / 2;
  constexpr int PER = (NB + NT - 1) / NT;
  for (int s2 = t; s2 <= NB; s2 += NT) BC[s2] = 0;
  gsync<NT>();
  const uint32_t range = (uint32_t)(cmax - cmin) + 1u;
  const uint64_t mul = ((uint64_t)NB << 32) / (uint64_t)range;
  int ik[IPT], ib[IPT], io[IPT];
  double iv[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const int s2 = t + j * NT;
    const int key = K[s2];
    ik[j] = key;
    iv[j] = H[s2];
    ib[j] = 0;
    io[j] = 0;
    if (key != kEmpty) {
      const int b = (int)(((uint64_t)(uint32_t)(key - cmin) * mul) >> 32);
      ib[j] = b;
      io[j] = atomicAdd(&BC[b], 1);
    }
  }
  gsync<NT>();
  {  // exclusive scan of bucket counts, PER contiguous buckets per thread
    int loc[PER];
    int sum = 0;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int i = t * PER + q;
      loc[q] = (i < NB) ? BC[i] : 0;
      sum += loc[q];
    }
    int total;
    int pre = Group<NT>::exscan(sum, total, sc);
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int i = t * PER + q;
      if (i < NB) BC[i] = pre;
      pre += loc[q];
    }
    if (t == 0) BC[NB] = total;
  }
  gsync<NT>();
  int* perm = K;  // the table keys are in registers now; reuse their LDS
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (ik[j] != kEmpty) perm[BC[ib[j]] + io[j]] = ik[j];
  gsync<NT>();
  int rk[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    rk[j] = 0;
    if (ik[j] != kEmpty) {
      const int s0 = BC[ib[j]], s1 = BC[ib[j] + 1];
      int r = s0;
      for (int m = s0; m < s1; ++m) r += (perm[m] < ik[j]);
      rk[j] = r;
    }
  }
  gsync<NT>();
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (ik[j] != kEmpty) {
      K[rk[j]] = ik[j];
      H[rk[j]] = iv[j];
    }
  gsync<NT>();
  const int n = BC[NB];
  const int nw = (int)min((int64_t)n, limit);
  for (int m = t; m < nw; m += NT) {
    Cidx[m] = K[m];
    Cval[m] = (V)H[m];
  }
  gsync<NT>();
  return n;
}

template <typename V, int T, int NT, int G, bool FAST = false>
__device__ __forceinline__ void numeric_hash_body(
    const int32_t* __restrict__ rows, const int64_t* __restrict__ pbeg, const int64_t* __restrict__ pend,
    const int64_t* __restrict__ Aptr, const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
    const V* __restrict__ Aval, const int32_t* __restrict__ Bidx, const V* __restrict__ Bval,
    const int64_t* __restrict__ Cptr, int64_t cbase, int32_t* __restrict__ Cidx, V* __restrict__ Cval,
    int* __restrict__ err) {
  constexpr int WG = wg_of<NT>();
  constexpr int GPB = WG / NT;
  constexpr int IPT = T / NT;  // table slots per thread
  static_assert(NT % G == 0 && T % NT == 0, "shape");
  constexpr bool WAVE = (NT == 64);
  constexpr int NB = T / 2;  // buckets (workgroup path)
  __shared__ int hk[GPB][T];
  __shared__ double hv[GPB][T];
  __shared__ int bc[GPB][WAVE ? 1 : NB + 1];
  __shared__ int sc[GPB][NT > 64 ? NT / 64 : 1];
  __shared__ FlatLds<V, true> fl[WG / 64];
  const int t = threadIdx.x % NT;
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x / NT);  // wave-uniform
  FlatLds<V, true>& wl = fl[__builtin_amdgcn_readfirstlane(threadIdx.x / 64)];
  int* K = hk[g];
  double* H = hv[g];
  const int64_t beg = *pbeg, end = *pend;
  if constexpr (WAVE) {
    // one wave per row, rows software-pipelined (RowPipe); the table is ranked by
    // wave_rank_keys while the next row's descriptors are in flight
    const int64_t s0 = beg + xcd_block() * GPB + g;
    if (s0 >= end) return;
    RowPipe<G, true, V> rp;
    rp.start(s0, (int64_t)gridDim.x * GPB, end, rows, Aptr, Cptr, t, bstart, blen, Aval);
    Step<4, V> st0;  // first gather step of the current row, issued during the previous row
    gather_step<G, 4, true, V>(st0, t, 0, (int)min((int64_t)64, rp.a1 - rp.a0), rp.d, Bidx, Bval);
    int flags = 0;   // error bits of all rows of this wave, reported once after the loop
    constexpr int STEP = G == 16 ? 16 : 4;  // A entries covered by the first gather step
    for (;;) {
      rp.prefetch(t, rows, Aptr, Cptr, bstart, blen, Aval);
      // Rows whose products are all distinct (P_i equals the symbolic count nnz_i) and are all
      // in the first gather step (at most STEP A entries, B rows of at most G entries) skip the
      // hash table: their products are ranked straight from registers.
      bool fast = false;
      if (FAST && rp.a1 - rp.a0 <= STEP) {
        const bool inrow = desc_slot<G>(t) < rp.a1 - rp.a0;
        const bool longb = __builtin_amdgcn_ballot_w64(inrow && rp.d.len > G) != 0;
        const int P = wave_reduce_dpp(inrow ? min(rp.d.len, G + 1) : 0, OpAdd());
        fast = !longb && (int64_t)P == rp.c1 - rp.c0 && P <= T / 2;
      }
      if (fast) {
        const int64_t nA = rp.a1 - rp.a0;
        const int64_t nexp = rp.c1 - rp.c0;
        const int sg = t / G, lg = t % G;
        const int cnt = (int)nA;
        int kc[4], rk[4];
        V kv[4];
        int lmin = INT_MAX, lmax = -1;
        static_for<4>([&](auto uc) {
          constexpr int u = decltype(uc)::value;
          const int e = step_entry<G, 0>(0, u, sg);
          const int lv = ebcast<G, u>(rp.d.len, u);
          const V pv = ebcastv<G, u>(rp.d.va, u);
          const bool has = e < cnt && lg < lv;
          kc[u] = has ? st0.c[u] : kEmpty;
          kv[u] = pv * st0.bv[u];
          lmin = has ? min(lmin, kc[u]) : lmin;
          lmax = has ? max(lmax, kc[u]) : lmax;
        });
        // the next row's first gathers, in flight while this row is ranked and stored
        gather_step<G, 4, true, V>(st0, t, 0, (int)min((int64_t)64, rp.na1 - rp.na0), rp.nd, Bidx, Bval);
        const int cmin = wave_reduce_dpp(lmin, OpMin());
        const int cmax = wave_reduce_dpp(lmax, OpMax());
        const int n = wave_rank_keys<T, 4>(t, K, cmin, cmax, kc, rk);
        flags |= ((int64_t)n != nexp) ? kErrCountMismatch : 0;
        wave_sync();
        V* S = reinterpret_cast<V*>(H);  // products as they are: nothing is added up
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (rk[u] >= 0) {
            K[rk[u]] = kc[u];
            S[rk[u]] = kv[u];
          }
        wave_sync();
        // fixed-count unconditional coalesced stores, as below
        const int64_t o0 = rp.c0 - cbase;
        const int nw = (int)min((int64_t)n, nexp);
        int32_t* di = nw > 0 ? Cidx + o0 : (int32_t*)(err + 4);
        V* dv = nw > 0 ? Cval + o0 : (V*)(err + 8);
        const int last = max(nw, 1) - 1;
#pragma unroll
        for (int j = 0; j < (T / 2 + 63) / 64; ++j) {
          const int m = min(t + 64 * j, last);
          const int key = K[m];
          const V val = S[m];
          di[m] = key;
          dv[m] = val;
        }
        wave_sync();
        if (!rp.advance()) break;
        continue;
      }
      clear_table<T, double>(t, K, H);
      wave_sync();
      HashSink<T, V, true> sk{K, H};
      for_row_products_pre<64, G, 4, true, V>(t, rp.a0, rp.a1, rp.d, bstart, blen, Aval, Bidx, Bval, wl, sk, &st0);
      // the next row's first gathers (past the last row: the current row again, unused); they
      // are in flight while this row is ranked and stored
      gather_step<G, 4, true, V>(st0, t, 0, (int)min((int64_t)64, rp.na1 - rp.na0), rp.nd, Bidx, Bval);
      wave_sync();
      const int cmin = wave_reduce_dpp(sk.cmin, OpMin());
      const int cmax = wave_reduce_dpp(sk.cmax, OpMax());
      int kk[IPT], rk[IPT];
#pragma unroll
      for (int q = 0; q < IPT; ++q) kk[q] = K[slot_of<T>(t, q)];
      wave_sync();
      const int n = wave_rank_keys<T, IPT>(t, K, cmin, cmax, kk, rk);
      const int64_t o0 = rp.c0 - cbase;
      const int64_t nexp = rp.c1 - rp.c0;
      flags |= (sk.bad || n > T / 2) ? kErrTableFull : 0;
      flags |= ((int64_t)n != nexp) ? kErrCountMismatch : 0;
      // stage the ranked row in the (now free) key table: key at its rank, source slot at
      // T/2 + rank; the values stay in their hash slots
      wave_sync();
#pragma unroll
      for (int q = 0; q < IPT; ++q)
        if (rk[q] >= 0 && rk[q] < T / 2) {
          K[rk[q]] = kk[q];
          K[T / 2 + rk[q]] = slot_of<T>(t, q);
        }
      wave_sync();
      // a fixed number of unconditional, coalesced stores: lanes past the row's end repeat its
      // last element (same address, same data). Unconditional stores keep the compiler's count
      // of outstanding memory operations exact, so waiting for the next row's gathers never
      // waits for these stores. A row that came out empty (only after an inconsistency, which
      // is reported) writes to the sink behind the error word instead of the output.
      const int nw = (int)min((int64_t)min(n, T / 2), nexp);
      int32_t* di = nw > 0 ? Cidx + o0 : (int32_t*)(err + 4);
      V* dv = nw > 0 ? Cval + o0 : (V*)(err + 8);
      const int last = max(nw, 1) - 1;
#pragma unroll
      for (int j = 0; j < (T / 2 + 63) / 64; ++j) {
        const int m = min(t + 64 * j, last);
        const int key = K[m];
        const V val = (V)H[K[T / 2 + m] & (T - 1)];
        di[m] = key;
        dv[m] = val;
      }
      wave_sync();
      if (!rp.advance()) break;
    }
    flags = wave_reduce_dpp(flags, OpOr());
    if (t == 0 && flags) atomicOr(err, flags);
    return;
  } else {
    int* BC = bc[g];
    for (int64_t slot = beg + (int64_t)blockIdx.x * GPB + g; slot < end; slot += (int64_t)gridDim.x * GPB) {
      const int row = rows[slot];
#pragma unroll
      for (int s2 = t; s2 < T; s2 += NT) {
        K[s2] = kEmpty;
        H[s2] = 0.0;
      }
      gsync<NT>();
      const int64_t a0 = Aptr[row], a1 = Aptr[row + 1];
      HashSink<T, V, true> sk{K, H};
      for_row_products<NT, G, 4, true, V>(t, a0, a1, bstart, blen, Aval, Bidx, Bval, wl, sk);
      gsync<NT>();
      const int cmin = Group<NT>::reduce(sk.cmin, OpMin(), sc[g]);
      const int cmax = Group<NT>::reduce(sk.cmax, OpMax(), sc[g]);
      int bad = sk.bad;
      const int64_t o0 = Cptr[row] - cbase;
      const int64_t nexp = Cptr[row + 1] - Cptr[row];
      const int n = block_rank_emit<V, T, NT>(t, K, H, BC, sc[g], cmin, cmax, Cidx + o0, Cval + o0, nexp);
      bad = Group<NT>::reduce(bad, OpMax(), sc[g]);
      if (t == 0) {
        if (bad) atomicOr(err, kErrTableFull);
        if ((int64_t)n != nexp) atomicOr(err, kErrCountMismatch);
      }
      gsync<NT>();
    }
  }
}

// Occupancy target of the one-wave-per-row numeric kernel (waves per SIMD); the compiler fits
// its registers to it. The workgroup-per-row shapes are limited by LDS instead. The variant with
// the register path for rows of distinct products needs more registers: 4 waves per SIMD.
#ifndef DBD_NUMERIC_WAVES_PER_EU
#define DBD_NUMERIC_WAVES_PER_EU 5
#endif
#ifndef DBD_NUMERIC_FAST_WAVES_PER_EU
#define DBD_NUMERIC_FAST_WAVES_PER_EU 4
#endif

#define DBD_NUMERIC_ARGS                                                                                     \
  const int32_t *__restrict__ rows, const int64_t *__restrict__ pbeg, const int64_t *__restrict__ pend,     \
      const int64_t *__restrict__ Aptr, const int64_t *__restrict__ bstart, const int32_t *__restrict__ blen, \
      const V *__restrict__ Aval, const int32_t *__restrict__ Bidx, const V *__restrict__ Bval,              \
      const int64_t *__restrict__ Cptr, int64_t cbase, int32_t *__restrict__ Cidx, V *__restrict__ Cval,      \
      int *__restrict__ err

template <typename V, int T, int NT, int G>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DBD_NUMERIC_WAVES_PER_EU))) void
k_numeric_wave(DBD_NUMERIC_ARGS) {
  numeric_hash_body<V, T, NT, G>(rows, pbeg, pend, Aptr, bstart, blen, Aval, Bidx, Bval, Cptr, cbase, Cidx, Cval,
                                 err);
}

// Same rows, with the register path for rows whose products are all distinct (chosen when the
// problem has few duplicate products).
template <typename V, int T, int NT, int G>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DBD_NUMERIC_FAST_WAVES_PER_EU))) void
k_numeric_wave_fast(DBD_NUMERIC_ARGS) {
  numeric_hash_body<V, T, NT, G, true>(rows, pbeg, pend, Aptr, bstart, blen, Aval, Bidx, Bval, Cptr, cbase, Cidx,
                                       Cval, err);
}

template <typename V, int T, int NT, int G>
__global__ __launch_bounds__(NT) void k_numeric_block(DBD_NUMERIC_ARGS) {
  numeric_hash_body<V, T, NT, G>(rows, pbeg, pend, Aptr, bstart, blen, Aval, Bidx, Bval, Cptr, cbase, Cidx, Cval,
                                 err);
}

// Rows of a few thousand columns and more, without a hash table or a sort: a column's place among the
// row's columns comes from a bitmap. One workgroup per row, in windows of the row's columns:
//   - up to VC columns wide: the products are added at their column (a column is present when its sum
//     is no longer -0.0, as in k_hub_range);
//   - up to BW columns wide, holding at most VC products or entries of C: a walk over the window's
//     products sets presence bits, their prefix gives every column its rank, and a second walk adds
//     the products at the ranks.
// A row no wider than such a window is one window, its B rows walked whole. Wider rows read B's band
// index (BANDS), whose ends give every long B row's part of a window and the products per band, by
// which a window is as many bands, up to 16, as the values fit (one band always does); the products
// of B rows without an index row (short ones) stay in registers, up to four a thread. Without the
// index: windows of VC columns, the B rows read whole in each.
//
// The walks are element-parallel (walk_spans); rows of up to 64 entries are every wave's, which share
// the elements, others are dealt over the waves. Bound by the chains of a window (band ends, gathers,
// barriers): 52 KB of LDS let three workgroups of 8 waves share a CU, for which a few registers spill
// (two workgroups without spills: 5.25 ms against 4.93 on 8,190 rows of R-MAT 20). Measured against
// the windows of k_numeric_long and the tables of 4096 slots and more, all rows of a pass: R-MAT 20
// rows 7.10 -> 4.93 ms, R-MAT 16 1.76 -> 1.02 ms, a batch of 32 1.81 -> 1.16 ms, 100 skewed rows over
// 6007 columns 0.54 -> 0.15 ms.
template <typename V, int NT, int VC, int BW, bool BANDS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(6))) void k_numeric_rank(
    const int32_t* __restrict__ rows, const int64_t* __restrict__ pbeg, const int64_t* __restrict__ pend,
    const int64_t* __restrict__ Aptr, const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
    const V* __restrict__ Aval, const int32_t* __restrict__ Bidx, const V* __restrict__ Bval,
    const int64_t* __restrict__ Cptr, int64_t cbase, int32_t* __restrict__ Cidx, V* __restrict__ Cval,
    int* __restrict__ err, const int32_t* __restrict__ Aidx, const int32_t* __restrict__ hslot,
    const int32_t* __restrict__ band, int64_t nb1) {
  constexpr int NW = NT / 64, U = 4, NWORD = BW / 64, WPT = NWORD / NT, PT = VC / NT;
  constexpr int WB = BW / VC, CB = BANDS ? 256 : 1;  // bands of a window at most; bands counted at a time
  struct WaveLds {
    SpanLds sp;
    double va[64];
  };
  static_assert(WPT == 2 && NWORD == 2 * NT && PT * NW == 64 && VC == 1 << kBandShift && WB == 16, "shape");
  static_assert(VC * 2 <= NW * (int)sizeof(WaveLds) && BW <= 65536, "the columns' list lies in the walks' LDS");
  __shared__ __align__(16) double dv[VC];
  __shared__ unsigned long long bm[NWORD];
  __shared__ uint16_t pre[NWORD / 2];
  __shared__ WaveLds wls[NW];
  __shared__ int wcnt[64], cnt[CB];
  int(*red)[NW] = reinterpret_cast<int(*)[NW]>(wcnt);
  uint16_t* off = reinterpret_cast<uint16_t*>(wls);
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  WaveLds& wl = wls[wv];
  for (int q = t; q < VC; q += NT) dv[q] = -0.0;
  for (int q = t; q < NWORD; q += NT) bm[q] = 0ull;
  __syncthreads();
  const int64_t beg = *pbeg, end = *pend;
  int flags = 0;
  for (int64_t slot = beg + blockIdx.x; slot < end; slot += gridDim.x) {
    const int row = rows[slot];
    const int64_t a0 = Aptr[row], nA = Aptr[row + 1] - a0;
    const int64_t out = Cptr[row] - cbase, nexp = Cptr[row + 1] - Cptr[row];
    const bool shared = nA <= 64;  // uniform
    const int w0s = shared ? wv * U : 0, wstep = shared ? NW * U : U;
    // an entry: start and length of its B row, A's value, its band index row (or null)
    struct Entry {
      int64_t b;
      int L;
      double a;
      const int32_t* bd;
    };
    auto load = [&](int64_t e) {
      Entry x{0, 0, 0.0, nullptr};
      if (e < nA) {
        const int64_t ka = a0 + e;
        x.b = bstart[ka];
        x.L = blen[ka];
        x.a = (double)Aval[ka];
        if constexpr (BANDS) {
          const int sl = hslot[Aidx[ka]];
          if (sl >= 0) x.bd = band + (int64_t)sl * nb1;
        }
      }
      return x;
    };
    const int el = shared ? lane : wv + NW * lane;  // entry of this lane in each NT entries
    const Entry e1 = load(el);
    int cmin = INT_MAX, cmax = -1;
    for (int64_t e0 = 0; e0 < nA; e0 += NT) {  // uniform
      const Entry x = e0 ? load(e0 + el) : e1;
      if (x.L > 0) {
        cmin = min(cmin, Bidx[x.b]);
        cmax = max(cmax, Bidx[x.b + x.L - 1]);
      }
    }
    cmin = wave_reduce_dpp(cmin, OpMin());
    cmax = wave_reduce_dpp(cmax, OpMax());
    if (!shared) {
      if (lane == 0) red[0][wv] = cmin, red[1][wv] = cmax;
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        cmin = min(cmin, red[0][i]);
        cmax = max(cmax, red[1][i]);
      }
    }
    const int64_t width = (int64_t)cmax - cmin;
    bool rank = width >= VC;                                  // uniform, of the current window
    const bool banded = BANDS && rank && !(width < BW && nexp <= VC);
    if (!BANDS && nexp > VC) rank = false;  // windows of VC columns
    int64_t lo = banded ? (int64_t)cmin & ~(int64_t)(VC - 1) : cmin;
    int lim = rank ? BW : VC;  // columns of the window
    // banded rows: products of the B rows without an index row
    int sc[U] = {-1, -1, -1, -1};
    double sv[U] = {0.0, 0.0, 0.0, 0.0};
    bool sreg = false;
    if (banded && nA <= NT) {  // uniform
      const int len = e1.bd ? 0 : e1.L;
      sreg = wave_reduce_dpp(min(len, 1 << 20), OpAdd()) <= 64 * wstep;
      if (sreg)
        walk_spans<U>(lane, len, e1.b, wl.sp, [&](int r) { wl.va[r] = e1.a; },
                      [&](const int64_t (&at)[U], const int (&j)[U]) {
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                          const int64_t p = at[u] < 0 ? 0 : at[u];
                          sc[u] = at[u] < 0 ? -1 : Bidx[p];
                          sv[u] = wl.va[j[u]] * (double)Bval[p];
                        }
                      },
                      w0s, wstep);
    }
    int64_t w1 = 0;                 // banded: the band past the window
    int s0 = 0, s1 = 0;             // and the first entry's span in it
    SpanKeep keep;                  // of the last walk, if it can be repeated
    // the window's products, for the bodies below
    auto walk = [&](auto&& body) {
      for (int64_t e0 = 0; e0 < nA; e0 += NT) {  // uniform
        Entry x = e1;
        int f0 = s0, f1 = s1;
        if (e0) {
          x = load(e0 + el);
          if (banded && x.bd) {
            f0 = x.bd[lo >> kBandShift];
            f1 = x.bd[w1];
          }
        }
        int len = x.L;
        int64_t start = x.b;
        if (banded) {
          len = x.bd ? f1 - f0 : sreg ? 0 : x.L;
          start += x.bd ? f0 : 0;
        }
        keep = walk_spans<U>(lane, len, start, wl.sp, [&](int r) { wl.va[r] = x.a; }, body, w0s, wstep);
      }
    };
    auto walk_again = [&](auto&& body) {
      if (nA <= NT && keep.T <= 64 * kSpanWords) span_words<U>(lane, keep, 0, wl.sp, body, w0s, wstep);
      else walk(body);
    };
    int64_t done = 0, cb = -CB;  // first of the counted bands
    while (lo <= cmax) {  // uniform; lo grows by at least VC
      if constexpr (BANDS) if (banded) {
        const int64_t b0 = lo >> kBandShift;
        if (b0 + WB > cb + CB) {
          // ---- products per band of bands [cb, cb + CB), by entries (band ends are read a wave at a time) ----
          cb = b0;
          __syncthreads();
          if (t < CB) cnt[t] = 0;
          __syncthreads();
          int c[CB / 64];
#pragma unroll
          for (int q = 0; q < CB / 64; ++q) c[q] = 0;
          for (int64_t e0 = 0; e0 < nA; e0 += NT) {  // uniform
            const Entry x = e0 ? load(e0 + el) : e1;
            uint64_t has = __builtin_amdgcn_ballot_w64(x.bd != nullptr);
            if (shared) has &= 0x0101010101010101ull << wv;  // the waves hold the same entries
            while (has) {  // wave-uniform
              const int l = __builtin_ctzll(has);
              has &= has - 1;
              const int32_t* bd = reinterpret_cast<const int32_t*>(readlane64(reinterpret_cast<int64_t>(x.bd), l));
#pragma unroll
              for (int q = 0; q < CB / 64; ++q) {
                const int64_t b = cb + 64 * q + lane;
                c[q] += bd[min(b + 1, nb1 - 1)] - bd[min(b, nb1 - 1)];
              }
            }
#pragma unroll
            for (int q = 0; q < CB / 64; ++q) c[q] = min(c[q], 1 << 24);  // of millions of entries
            if (!sreg)
              walk_spans<U>(lane, x.bd ? 0 : x.L, x.b, wl.sp, [](int) {},
                            [&](const int64_t (&at)[U], const int (&)[U]) {
#pragma unroll
                              for (int u = 0; u < U; ++u) {
                                const int64_t b = (Bidx[at[u] < 0 ? 0 : at[u]] >> kBandShift) - cb;
                                if (at[u] >= 0 && b >= 0 && b < CB) atomicAdd(&cnt[b], 1);
                              }
                            },
                            w0s, wstep);
          }
#pragma unroll
          for (int q = 0; q < CB / 64; ++q)
            if (c[q]) atomicAdd(&cnt[64 * q + lane], c[q]);
          if (sreg) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const int64_t b = (sc[u] >> kBandShift) - cb;
              if (sc[u] >= 0 && b >= 0 && b < CB) atomicAdd(&cnt[b], 1);
            }
          }
          __syncthreads();
        }
        // ---- the window: as many bands as the values fit ----
        const int x = lane < WB ? min(cnt[b0 - cb + lane], VC + 1) : VC + 1;
        const int incl = wave_incl_scan_dpp(x);
        const int nb = max((int)__popcll(__builtin_amdgcn_ballot_w64(incl <= VC)), 1);
        lim = nb << kBandShift;
        if (__builtin_amdgcn_readlane(incl, nb - 1) == 0) {
          lo += lim;
          continue;
        }
        rank = nb > 1;
        w1 = min(b0 + nb, nb1 - 1);
        if (e1.bd) {
          s0 = e1.bd[b0];
          s1 = e1.bd[w1];
        }
      }
      const int lo32 = (int)lo;
      if (!rank) {
        // ================= products at their columns =================
        walk([&](const int64_t (&at)[U], const int (&j)[U]) {
          int c[U];
          V b[U];
          double av[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int64_t p = at[u] < 0 ? 0 : at[u];
            c[u] = Bidx[p];
            b[u] = Bval[p];
            av[u] = wl.va[j[u]];
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const uint32_t o = (uint32_t)(c[u] - lo32);
            if (at[u] >= 0 && o < (uint32_t)VC) lds_add(&dv[o], av[u] * (double)b[u] + 0.0);
          }
        });
        if (sreg) {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const uint32_t o = (uint32_t)(sc[u] - lo32);
            if (o < (uint32_t)VC) lds_add(&dv[o], sv[u] + 0.0);
          }
        }
        __syncthreads();
        double v[PT];
        uint64_t m[PT];
#pragma unroll
        for (int q = 0; q < PT; ++q) {
          v[q] = dv[t + q * NT];
          m[q] = __builtin_amdgcn_ballot_w64(__double_as_longlong(v[q]) != (long long)0x8000000000000000ull);
          dv[t + q * NT] = -0.0;
          if (lane == 0) wcnt[q * NW + wv] = __popcll(m[q]);
        }
        __syncthreads();
        const int x = wcnt[lane];
        const int incl = wave_incl_scan_dpp(x);
#pragma unroll
        for (int q = 0; q < PT; ++q) {
          const int64_t k = done + __builtin_amdgcn_readlane(incl - x, q * NW + wv) +
                            __builtin_amdgcn_mbcnt_hi((uint32_t)(m[q] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m[q], 0));
          if ((m[q] >> lane & 1ull) && k < nexp) {
            Cidx[out + k] = lo32 + t + q * NT;
            Cval[out + k] = (V)v[q];
          }
        }
        done += __builtin_amdgcn_readlane(incl, 63);
      } else {
        // ================= presence, ranks, products at their ranks =================
        uint32_t* bm32 = reinterpret_cast<uint32_t*>(bm);
        walk([&](const int64_t (&at)[U], const int (&)[U]) {
          int c[U];
#pragma unroll
          for (int u = 0; u < U; ++u) c[u] = Bidx[at[u] < 0 ? 0 : at[u]];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const uint32_t o = (uint32_t)(c[u] - lo32);
            if (at[u] >= 0 && o < (uint32_t)lim) atomicOr(&bm32[o >> 5], 1u << (o & 31));
          }
        });
        if (sreg) {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const uint32_t o = (uint32_t)(sc[u] - lo32);
            if (o < (uint32_t)lim) atomicOr(&bm32[o >> 5], 1u << (o & 31));
          }
        }
        __syncthreads();
        unsigned long long wd[WPT];
        int n = 0;
#pragma unroll
        for (int q = 0; q < WPT; ++q) {
          wd[q] = bm[t * WPT + q];
          n += __popcll(wd[q]);
        }
        const int incl = wave_incl_scan_dpp(n);
        if (lane == 63) wcnt[wv] = incl;
        __syncthreads();
        int base = incl - n, tot = 0;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
          const int x = wcnt[i];
          base += i < wv ? x : 0;
          tot += x;
        }
        pre[t] = (uint16_t)base;
        __syncthreads();
        auto add = [&](uint32_t o, double p) {
          const int w = o >> 6;
          const unsigned long long below = w & 1 ? bm[w - 1] : 0ull;
          const uint32_t r = (uint32_t)pre[w >> 1] + (uint32_t)__popcll(below) +
                             (uint32_t)__popcll(bm[w] & ((1ull << (o & 63)) - 1ull));
          if (r < (uint32_t)VC) lds_add(&dv[r], p + 0.0);
        };
        walk_again([&](const int64_t (&at)[U], const int (&j)[U]) {
          int c[U];
          V b[U];
          double av[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int64_t p = at[u] < 0 ? 0 : at[u];
            c[u] = Bidx[p];
            b[u] = Bval[p];
            av[u] = wl.va[j[u]];
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const uint32_t o = (uint32_t)(c[u] - lo32);
            if (at[u] >= 0 && o < (uint32_t)lim) add(o, av[u] * (double)b[u]);
          }
        });
        if (sreg) {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const uint32_t o = (uint32_t)(sc[u] - lo32);
            if (o < (uint32_t)lim) add(o, sv[u]);
          }
        }
        __syncthreads();
        // values as they lie, columns through a list in LDS (the walks are done with it)
        const int nw = (int)min((int64_t)min(tot, VC), max(nexp - done, (int64_t)0));
        {
          int r = base;
#pragma unroll
          for (int q = 0; q < WPT; ++q) {
            unsigned long long m = wd[q];
            while (m) {
              const int b = __ffsll(m) - 1;
              m &= m - 1ull;
              if (r < VC) off[r] = (uint16_t)(64 * (t * WPT + q) + b);
              ++r;
            }
            bm[t * WPT + q] = 0ull;
          }
        }
        for (int i = t; i < min(tot, VC); i += NT) {
          if (i < nw) Cval[out + done + i] = (V)dv[i];
          dv[i] = -0.0;
        }
        __syncthreads();
        for (int i = t; i < nw; i += NT) Cidx[out + done + i] = lo32 + off[i];
        done += tot;
        __syncthreads();  // the list is in the walks' LDS
      }
      lo += lim;
    }
    __syncthreads();
    flags |= done != nexp ? kErrCountMismatch : 0;
  }
  if (flags && lane == 0) atomicOr(err, flags);
}

// Long rows, any column range: the row's columns are swept in windows [lo, hi); a window starts
// at the smallest next column over the row's A entries, so empty column ranges are skipped, and
// every window's output is produced in column order (no sort).
//
// Rows of up to kSpanMax entries (with B's band index; without it, rows whose entries each have
// a subgroup of G lanes, nA <= NT/G) take windows of up to BW columns, with two walks over the
// window's products:
//   1. presence: every B column in the window sets its bit in an LDS bitmap (span walks: every
//      thread takes U elements of the flattened spans per step; cursor walks: each A entry's
//      subgroup counts its elements in the window, U loads per lane in flight);
//   2. values: the bitmap's word prefixes give every column its rank among the window's
//      columns, and A_ik * B_kj is added at that rank in an LDS value array of VC entries.
// The values are then stored as they lie (coalesced) and the columns read off the bitmap. When
// more than VC columns are present the window is cut at the VC-th column (the values walk stops
// there, the next window starts at it) and the next window is narrowed to the width that held
// VC columns; windows widen again (doubling up to BW) when they fit. Between the two cursor walks
// an active entry keeps -1 - count in its `nc` field.
//
// Rows of more entries take dense windows of VC columns in one walk (values added at column -
// lo, presence bits beside them): banded windows (below) when their entries fit the registers,
// else cursor windows, each A entry walked by a subgroup from a cursor (LongState: position,
// remaining, next column), 4 lanes per entry (8 when an entry averages 4 or more elements
// per window over the row's column span), 4 entries per subgroup in flight, a B row with more elements
// in the window than one step continuing UL steps at a time (loads issued together); an entry
// whose next column lies beyond the window costs one state read per window. Their cursors are in
// LDS (sharing the word-prefix space) up to kOldStates entries, else in the workspace `state`
// (16 bytes per A nonzero). Both paths leave the value array and the bitmap clear.
constexpr int kNumLongStates = 512;
constexpr int kSpanMax = 256;  // span-walk windows: A entries per row at most (one per thread)


template <typename V, int NT, int BW, int VC>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(3))) void k_numeric_long(
    const int32_t* __restrict__ rows, const int64_t* __restrict__ pbeg, const int64_t* __restrict__ pend,
    const int64_t* __restrict__ Aptr, const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
    const V* __restrict__ Aval, const int32_t* __restrict__ Bidx, const V* __restrict__ Bval,
    const int64_t* __restrict__ Cptr, int64_t cbase, int32_t* __restrict__ Cidx, V* __restrict__ Cval,
    LongState* __restrict__ state, int* __restrict__ err, const int32_t* __restrict__ Aidx,
    const int32_t* __restrict__ hslot, const int32_t* __restrict__ band, int64_t nb1) {
  constexpr int NWORD = BW / 32;
  constexpr int WPT = NWORD / NT;  // bitmap words per thread
  constexpr int OWORD = VC / 32;   // bitmap words of a dense window
  constexpr int NW = NT / 64;
  constexpr int U = 4;             // loads per lane in flight per walk step
  constexpr int UL = 8;            // dense windows: steps of G elements loaded together on a long B row
  constexpr int DVB = VC * (int)sizeof(V);
  constexpr int kOldStates = (NWORD * 2 + kNumLongStates * 16) / 16;
  static_assert(NWORD % NT == 0 && NT % 64 == 0 && VC < 65535 && OWORD <= NT, "shape");
  __shared__ __align__(16) unsigned char lds[DVB + NWORD * 4 + NWORD * 2 + kNumLongStates * 16];
  V* dv = reinterpret_cast<V*>(lds);
  uint32_t* bm = reinterpret_cast<uint32_t*>(lds + DVB);
  uint16_t* pre = reinterpret_cast<uint16_t*>(lds + DVB + NWORD * 4);  // exclusive prefix per word
  LongState* stl = reinterpret_cast<LongState*>(lds + DVB + NWORD * 4 + NWORD * 2);
  LongState* ostl = reinterpret_cast<LongState*>(lds + DVB + NWORD * 4);
  __shared__ int red[NW], red_cnt[NW];
  __shared__ long long redl[NW];
  __shared__ long long s_hi1, s_hi2;
  __shared__ int s_nh, s_nl;
  static_assert(2 * NT * (8 + (int)sizeof(V) + 4) <= NWORD * 2 + kNumLongStates * 16,
                "banded windows: range tables exceed the LDS they share");
  static_assert(kSpanMax <= NT && kSpanMax % 64 == 0 && kSpanMax * (16 + (int)sizeof(V)) <= kNumLongStates * 16,
                "span walks: one entry per thread, tables within the state LDS");
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  for (int q = t; q < NWORD; q += NT) bm[q] = 0u;
  for (int q = t; q < VC; q += NT) dv[q] = V(0);
  __syncthreads();
  auto block_min = [&](int x) {  // all threads; ends with a barrier
    const int m = wave_reduce_dpp(x, OpMin());
    if (lane == 0) red[wv] = m;
    __syncthreads();
    int r = red[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) r = min(r, red[i]);
    __syncthreads();
    return r;
  };
  int flags = 0;
  const int64_t beg = *pbeg, end = *pend;
  for (int64_t slot = beg + blockIdx.x; slot < end; slot += gridDim.x) {
    const int row = rows[slot];
    const int64_t a0 = Aptr[row], a1 = Aptr[row + 1], nA = a1 - a0;
    const int64_t c1 = Cptr[row + 1] - cbase;
    int64_t out = Cptr[row] - cbase;
    int G = long_lanes<NT>(nA);
    int NSG = NT / G, sg = t / G, lg = t & (G - 1), sgbase = lane & ~(G - 1);
    uint64_t submask = (G == 64 ? ~0ull : ((1ull << G) - 1ull)) << sgbase;
    const bool spans = band != nullptr && nA <= kSpanMax;  // uniform
    if (spans || nA <= NSG) {
      // ================= two walks per window of up to BW columns =================
      // With B's band index the walks are element-parallel over the workgroup: every active
      // entry's element span in the window (banded B rows: up to the band boundary at or past the
      // window end; other B rows: at most kSpanCap elements, the window ending before the first
      // element left out) is flattened by a scan and each thread takes U elements at a time, so
      // an entry with many elements in the window costs no chain of dependent steps. The entry
      // state (B row start and length, elements consumed, next column) is in the registers of
      // thread e (rows of up to kSpanMax entries). Without the index (rows of up to NT / G
      // entries) each entry's subgroup walks it from a cursor in LDS.
      LongState* st = stl;
      int* hS = reinterpret_cast<int*>(lds + DVB + NWORD * 4 + NWORD * 2);  // span starts
      int* np = hS + kSpanMax;                                               // consumed in walk 2
      int64_t* hb0 = reinterpret_cast<int64_t*>(np + kSpanMax);             // span start positions
      V* hva = reinterpret_cast<V*>(hb0 + kSpanMax);                         // A values
      int64_t eb0 = 0;
      int eL = 0, ep = 0, enc = INT_MAX;
      V eva = V(0);
      const int32_t* ebd = nullptr;
      int lmin = INT_MAX;
      long long psum = 0;
      if (spans) {
        if (t < nA) {
          const int64_t ka = a0 + t;
          eb0 = bstart[ka];
          eL = blen[ka];
          eva = Aval[ka];
          const int sl = hslot[Aidx[ka]];
          ebd = sl >= 0 ? band + (int64_t)sl * nb1 : nullptr;
          enc = eL > 0 ? Bidx[eb0] : INT_MAX;
          lmin = enc;
          psum = eL;
        }
      } else {
        for (int64_t e = t; e < nA; e += NT) {
          LongState x;
          x.p = bstart[a0 + e];
          x.rem = blen[a0 + e];
          x.nc = x.rem > 0 ? Bidx[x.p] : INT_MAX;
          st[e] = x;
          lmin = min(lmin, x.nc);
          psum += x.rem;
        }
      }
      // flattened element f of the window belongs to entry j, the last with hS[j] <= f (f < T)
      auto span_owner = [&](int f) {
        int j = 0;
#pragma unroll
        for (int step = kSpanMax / 2; step >= 1; step >>= 1)
          if (j + step < nA && hS[j + step] <= f) j += step;
        return j;
      };
      // a window always takes the element at its first column: at most P_i windows per row
      const long long prow = Group<NT>::reduce(psum, OpAdd(), redl);
      int lo = block_min(lmin);  // also orders the state writes before the walks
      int64_t width = BW;
      long long windows = 0;
      while (lo != INT_MAX) {
        int64_t hi1 = min((int64_t)lo + width, (int64_t)INT_MAX);  // INT_MAX: exhausted entry
        int T = 0;
        if (spans) {
          // ---- the active entries' element spans; the window ends before any element a
          // capped span leaves out ----
          int len = 0, clip = INT_MAX;
          if (t < nA && (int64_t)enc < hi1) {
            int q;
            if (ebd != nullptr) {
              q = ebd[min((hi1 + (1 << kBandShift) - 1) >> kBandShift, nb1 - 1)];
            } else {
              q = min(eL, ep + kSpanCap);
              if (q < eL) clip = Bidx[eb0 + q];
            }
            len = q - ep;
          }
          if (nA <= 64) {  // uniform: wave 0 holds every entry
            if (wv == 0) {
              const int cm = wave_reduce_dpp(clip, OpMin());
              const int incl = wave_incl_scan_dpp(len);
              if (lane < nA) hS[lane] = incl - len;
              if (lane == 63) {
                s_nh = incl;
                s_hi1 = min(hi1, (int64_t)cm);
              }
            }
          } else {
            int tot;
            const int pre0 = Group<NT>::exscan(len, tot, red_cnt);
            const int cm = Group<NT>::reduce(clip, OpMin(), red);
            if (t < nA) hS[t] = pre0;
            if (t == 0) {
              s_nh = tot;
              s_hi1 = min(hi1, (int64_t)cm);
            }
          }
          if (t < nA) {
            hb0[t] = eb0 + ep;
            hva[t] = eva;
            np[t] = 0;
          }
          __syncthreads();
          T = s_nh;
          hi1 = s_hi1;
          // ---- walk 1: presence bits of [lo, hi1), element-parallel ----
          for (int f0 = 0; f0 < T; f0 += NT * U) {  // uniform
            int c[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const int f = f0 + u * NT + t;
              const int j = span_owner(f);
              const int64_t at = f < T ? hb0[j] + (f - hS[j]) : 0;  // lanes past T: unused read
              c[u] = Bidx[at];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
              if (f0 + u * NT + t < T && (int64_t)c[u] < hi1) {
                const int o = c[u] - lo;
                atomicOr(&bm[o >> 5], 1u << (o & 31));
              }
            }
          }
        } else {
        // ---- walk 1: presence bits of [lo, hi1), per-entry counts ----
        for (int64_t e = sg; e < nA; e += NSG) {  // subgroup-uniform
          LongState x = st[e];
          if ((int64_t)x.nc < hi1) {
            int64_t p = x.p;
            int rem = x.rem, cnt = 0;
            for (;;) {
              int c[U];
#pragma unroll
              for (int u = 0; u < U; ++u) {
                const int k = u * G + lg;
                const int64_t at = rem > 0 ? p + min(k, rem - 1) : 0;
                const int cv = Bidx[at];
                c[u] = k < rem ? cv : INT_MAX;
              }
              int nin = 0;
#pragma unroll
              for (int u = 0; u < U; ++u) {
                const bool in = (int64_t)c[u] < hi1;
                if (in) {
                  const int o = c[u] - lo;
                  atomicOr(&bm[o >> 5], 1u << (o & 31));
                }
                nin += __popcll(__ballot(in) & submask);
              }
              cnt += nin;
              if (nin < U * G || rem <= U * G) break;  // rem shrinks every step: bounded walk
              p += U * G;
              rem -= U * G;
            }
            if (lg == 0) {
              x.nc = -1 - cnt;
              st[e] = x;
            }
          }
        }
        }
        __syncthreads();
        // ---- word prefixes, and the cut when more than VC columns are present ----
        uint32_t wd[WPT];
        int wp[WPT];
        int cnts = 0;
#pragma unroll
        for (int q = 0; q < WPT; ++q) {
          wd[q] = bm[t * WPT + q];
          cnts += __popc(wd[q]);
        }
        const int incl = wave_incl_scan_dpp(cnts);
        if (lane == 63) red_cnt[wv] = incl;
        __syncthreads();
        int base = 0, tot = 0;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
          const int ci = red_cnt[i];
          base += i < wv ? ci : 0;
          tot += ci;
        }
        base += incl - cnts;
        {
          int run = base;
#pragma unroll
          for (int q = 0; q < WPT; ++q) {
            wp[q] = run;
            pre[t * WPT + q] = (uint16_t)min(run, 65535);
            run += __popc(wd[q]);
          }
        }
        if (tot <= VC) {
          if (t == 0) s_hi2 = hi1;
        } else {
#pragma unroll
          for (int q = 0; q < WPT; ++q) {
            const int pc = __popc(wd[q]);
            if (wp[q] <= VC && VC < wp[q] + pc) {  // the VC-th set bit (from 0) is in this word
              uint32_t w = wd[q];
              for (int j = 0; j < VC - wp[q]; ++j) w &= w - 1u;
              s_hi2 = (int64_t)lo + 32 * (t * WPT + q) + (__ffs(w) - 1);
            }
          }
        }
        __syncthreads();
        const int64_t hi2 = s_hi2;
        const int nw = min(tot, VC);
        lmin = INT_MAX;
        if (spans) {
          // ---- walk 2: values of [lo, hi2) at their ranks, element-parallel; each entry's
          // elements below hi2 are a prefix of its span, whose length the last such lane of
          // every wave records ----
          for (int f0 = 0; f0 < T; f0 += NT * U) {  // uniform
            int c[U], jj[U];
            V b[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const int f = f0 + u * NT + t;
              jj[u] = span_owner(f);
              const int64_t at = f < T ? hb0[jj[u]] + (f - hS[jj[u]]) : 0;
              c[u] = Bidx[at];
              b[u] = Bval[at];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const int f = f0 + u * NT + t;
              const int j = jj[u];
              const bool in = f < T && (int64_t)c[u] < hi2;
              if (in) {
                const int o = c[u] - lo;
                const int w = o >> 5;
                const int r = (int)pre[w] + __popc(bm[w] & ((1u << (o & 31)) - 1u));
                lds_add(&dv[r], hva[j] * b[u]);
              }
              const int jn = __shfl_down(j, 1);
              const int inn = __shfl_down((int)in, 1);
              if (in && (lane == 63 || !inn || jn != j)) atomicMax(&np[j], f - hS[j] + 1);
            }
          }
          __syncthreads();  // np complete
          if (t < nA) {
            const int took = np[t];
            if (took > 0) {
              ep += took;
              enc = ep < eL ? Bidx[eb0 + ep] : INT_MAX;
            }
            lmin = enc;
          }
        } else {
        // ---- walk 2: values of [lo, hi2) at their ranks; cursors advance to hi2 ----
        for (int64_t e = sg; e < nA; e += NSG) {  // subgroup-uniform
          LongState x = st[e];
          if (x.nc < 0) {
            const int cnt = -1 - x.nc;
            const int n = min(cnt + 1, x.rem);  // the window's elements and the one after it
            const V va = Aval[a0 + e];
            int nin2 = 0, nxt = INT_MAX;
            for (int k0 = 0; k0 < n; k0 += U * G) {
              int c[U];
              V b[U];
#pragma unroll
              for (int u = 0; u < U; ++u) {
                const int k = k0 + u * G + lg;
                const int64_t at = x.p + min(k, n - 1);
                c[u] = Bidx[at];
                b[u] = Bval[at];
              }
#pragma unroll
              for (int u = 0; u < U; ++u) {
                const int k = k0 + u * G + lg;
                const bool valid = k < n;
                const bool in = valid && (int64_t)c[u] < hi2;
                if (in) {
                  const int o = c[u] - lo;
                  const int w = o >> 5;
                  const int r = (int)pre[w] + __popc(bm[w] & ((1u << (o & 31)) - 1u));
                  lds_add(&dv[r], va * b[u]);
                }
                if (valid && !in) nxt = min(nxt, c[u]);
                nin2 += __popcll(__ballot(in) & submask);
              }
            }
#pragma unroll
            for (int o = 1; o < 64; o <<= 1)
              if (o < G) nxt = min(nxt, __shfl_xor(nxt, o));
            x.p += nin2;
            x.rem -= nin2;
            x.nc = x.rem > 0 ? nxt : INT_MAX;
            if (lg == 0) st[e] = x;
          }
          lmin = min(lmin, x.nc);
        }
        }
        __syncthreads();
        // ---- emit: values as they lie, columns from the bitmap; both left clear ----
        for (int i = t; i < nw; i += NT) {
          if (out + i < c1) Cval[out + i] = dv[i];
          else flags |= kErrWindow;
          dv[i] = V(0);
        }
#pragma unroll
        for (int q = 0; q < WPT; ++q) {
          const int w = t * WPT + q;
          const int64_t cb = (int64_t)lo + 32 * w;
          uint32_t bits = wd[q];
          if (cb >= hi2) bits = 0u;
          else if (cb + 32 > hi2) bits &= (1u << (int)(hi2 - cb)) - 1u;
          int64_t pos = out + wp[q];
          while (bits) {
            const int bb = __ffs(bits) - 1;
            bits &= bits - 1u;
            if (pos < c1) Cidx[pos] = (int)(cb + bb);
            else flags |= kErrWindow;
            ++pos;
          }
          bm[w] = 0u;
        }
        out += nw;
        // the width that held VC columns when cut, else twice the last width
        width = tot > VC ? max((int64_t)64, hi2 - lo) : min((int64_t)BW, 2 * width);
        lo = block_min(lmin);  // also: the clears are done before the next walk 1
        if (++windows > prow) {  // uniform: no progress (reported; the row's output is not trusted)
          flags |= kErrWindow;
          break;
        }
      }
    } else {
      bool banded_done = false;  // uniform
      if (band != nullptr) {
      // ================= banded dense windows =================
      // Windows are aligned blocks of VC columns. An entry whose B row is banded knows the exact
      // range of its elements in each window from the band index; the window's elements of all
      // banded entries are gathered element-parallel over the workgroup, one per lane. The other
      // entries (B rows below the banding threshold) keep a cursor, one lane each, four elements
      // per load. Per-entry state stays in registers (up to KE banded and KE other entries per
      // thread), and each window's element loads are issued together with the next window's band
      // end and next column, so a window costs one dependent round trip to memory. Rows with more
      // entries of either kind take the cursor windows below.
      constexpr int LOGVC = __builtin_ctz(VC);
      constexpr int BPW = VC >> kBandShift;  // bands per window
      constexpr int KE = 2;
      HRec* hrec = reinterpret_cast<HRec*>(state + a0);
      LRec* lrec = reinterpret_cast<LRec*>(state + a0);
      // chunk arrays in the word-prefix and state LDS of the other paths, which both rewrite it
      // before use (the bitmap words past the dense window's must stay clear for the two walks)
      unsigned char* reg = lds + DVB + NWORD * 4;
      int64_t* hb0 = reinterpret_cast<int64_t*>(reg);                        // KE * NT
      V* hva = reinterpret_cast<V*>(reg + KE * NT * 8);                      // KE * NT
      int* hS = reinterpret_cast<int*>(reg + KE * NT * (8 + (int)sizeof(V)));  // KE * NT
      if (t == 0) s_nh = s_nl = 0;
      __syncthreads();
      int lmin = INT_MAX, lmax = -1;
      long long psum = 0;
      for (int64_t e = t; e < nA; e += NT) {
        const int64_t ka = a0 + e;
        const int L = blen[ka];
        if (L <= 0) continue;
        const int64_t b0 = bstart[ka];
        const int sl = hslot[Aidx[ka]];
        const int cf = Bidx[b0], cl = Bidx[b0 + L - 1];
        lmin = min(lmin, cf);
        lmax = max(lmax, cl);
        psum += L;
        if (sl >= 0) {
          const int h = atomicAdd(&s_nh, 1);
          hrec[h] = HRec{b0, sl, (int)e};
        } else {
          const int l = atomicAdd(&s_nl, 1);
          lrec[nA - 1 - l] = LRec{0, (int)e, cf, L};
        }
      }
      psum = Group<NT>::reduce(psum, OpAdd(), redl);
      lmax = Group<NT>::reduce(lmax, OpMax(), red_cnt);
      lmin = Group<NT>::reduce(lmin, OpMin(), red_cnt);  // the reductions also order the record writes
      const int nH = s_nh, nL = s_nl;
      if (nH <= KE * NT && nL <= KE * NT) {  // uniform
        banded_done = true;
        int w = lmin == INT_MAX ? 1 : (lmin >> LOGVC);
        const int wl = lmin == INT_MAX ? 0 : (lmax >> LOGVC);
        // banded entries k * NT + t: B row start, A value, band row, length, range [s, s1) of the
        // current window, its end one window on (s1n) and the column after the window (nxc)
        int64_t hbr[KE];
        V hv[KE];
        const int32_t* hbi[KE];
        int hL[KE], hs[KE], hs1[KE], hs1n[KE], hnx[KE];
        // other entries: B row start, A value, position, entries left, column at the position
        int64_t lb0[KE];
        V lva[KE];
        int lp[KE], lrem[KE], lnc[KE];
#pragma unroll
        for (int k = 0; k < KE; ++k) {
          const int h = k * NT + t;
          hL[k] = 0;
          hs[k] = hs1[k] = hs1n[k] = 0;
          hnx[k] = INT_MAX;
          hbr[k] = 0;
          hv[k] = V(0);
          hbi[k] = band;
          if (h < nH) {
            const HRec r = hrec[h];
            hbr[k] = r.b0;
            hv[k] = Aval[a0 + r.e];
            hbi[k] = band + (int64_t)r.slot * nb1;
            hL[k] = hbi[k][nb1 - 1];
            hs[k] = hbi[k][w * BPW];
            hs1[k] = hbi[k][(w + 1) * BPW];
          }
          lrem[k] = 0;
          lnc[k] = INT_MAX;
          lp[k] = 0;
          lb0[k] = 0;
          lva[k] = V(0);
          if (h < nL) {
            const LRec r = lrec[nA - 1 - h];
            lb0[k] = bstart[a0 + r.e];
            lva[k] = Aval[a0 + r.e];
            lrem[k] = r.rem;
            lnc[k] = r.nc;
          }
        }
        long long windows = 0;  // every window holds an element: at most psum windows
        while (w <= wl) {
          const int lo = w << LOGVC;
          const int64_t hi = (int64_t)lo + VC;
          // ---- ranges of the banded entries: exclusive scan of their counts ----
          int csum = 0;
#pragma unroll
          for (int k = 0; k < KE; ++k) csum += hs1[k] - hs[k];
          const int incl = wave_incl_scan_dpp(csum);
          if (lane == 63) red_cnt[wv] = incl;
          __syncthreads();
          int base = 0, T = 0;
#pragma unroll
          for (int i = 0; i < NW; ++i) {
            const int ci = red_cnt[i];
            base += i < wv ? ci : 0;
            T += ci;
          }
          {
            int run = base + incl - csum;  // entries k * NT + t: this thread's entries in order
#pragma unroll
            for (int k = 0; k < KE; ++k) {
              hS[t * KE + k] = run;
              hb0[t * KE + k] = hbr[k] + hs[k];
              hva[t * KE + k] = hv[k];
              run += hs1[k] - hs[k];
            }
          }
          // ---- next window's band ends and the columns after this window (loads in flight
          // with this window's gathers) ----
#pragma unroll
          for (int k = 0; k < KE; ++k) {
            hs1n[k] = hs1[k];
            hnx[k] = INT_MAX;
            if (hs1[k] < hL[k]) {
              hs1n[k] = hbi[k][min((w + 2) * BPW, (int)nb1 - 1)];
              hnx[k] = Bidx[hbr[k] + hs1[k]];
            }
          }
          // ---- other entries: first four elements of those with one in this window ----
          int lc[KE][4];
          V lbv[KE][4];
#pragma unroll
          for (int k = 0; k < KE; ++k) {
            const bool act = lrem[k] > 0 && (int64_t)lnc[k] < hi;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const int64_t at = act ? lb0[k] + lp[k] + min(q, lrem[k] - 1) : 0;
              lc[k][q] = Bidx[at];
              lbv[k][q] = Bval[at];
            }
          }
          __syncthreads();  // the range table is complete
          // ---- banded elements: element f belongs to the table entry j with hS[j] <= f < hS[j + 1]
          // (entries in thread-major order: thread t's KE entries are t * KE .. t * KE + KE - 1) ----
          constexpr int NE = KE * NT;
          for (int f0 = 0; f0 < T; f0 += NT * U) {  // uniform
            int col[U];
            V bv[U], va[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const int f = f0 + u * NT + t;
              int j = 0;
#pragma unroll
              for (int step = NE / 2; step >= 1; step >>= 1)
                if (hS[j + step] <= f) j += step;  // hS is non-decreasing; entries past nH hold T
              const int64_t at = f < T ? hb0[j] + (f - hS[j]) : 0;  // lanes past T: unused read
              col[u] = Bidx[at];
              bv[u] = Bval[at];
              va[u] = hva[j];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
              if (f0 + u * NT + t < T) {
                const int o = col[u] - lo;
                lds_add(&dv[o], va[u] * bv[u]);
                atomicOr(&bm[o >> 5], 1u << (o & 31));
              }
            }
          }
          // ---- other entries: accumulate the loaded elements, continue a run longer than four ----
#pragma unroll
          for (int k = 0; k < KE; ++k) {
            if (lrem[k] > 0 && (int64_t)lnc[k] < hi) {
              int took = 0;
              bool stop = false;
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                if (!stop) {
                  if (q < lrem[k] && (int64_t)lc[k][q] < hi) {
                    const int o = lc[k][q] - lo;
                    lds_add(&dv[o], lva[k] * lbv[k][q]);
                    atomicOr(&bm[o >> 5], 1u << (o & 31));
                    ++took;
                  } else {
                    stop = true;
                  }
                }
              }
              int nc = (took < 4 && took < lrem[k]) ? lc[k][took] : INT_MAX;
              lp[k] += took;
              lrem[k] -= took;
              while (!stop && lrem[k] > 0) {  // rem shrinks every round that continues
                int cc[4];
                V bb[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                  const int64_t at = lb0[k] + lp[k] + min(q, lrem[k] - 1);
                  cc[q] = Bidx[at];
                  bb[q] = Bval[at];
                }
                took = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                  if (!stop) {
                    if (q < lrem[k] && (int64_t)cc[q] < hi) {
                      const int o = cc[q] - lo;
                      lds_add(&dv[o], lva[k] * bb[q]);
                      atomicOr(&bm[o >> 5], 1u << (o & 31));
                      ++took;
                    } else {
                      stop = true;
                      if (q < lrem[k]) nc = cc[q];
                    }
                  }
                }
                lp[k] += took;
                lrem[k] -= took;
              }
              lnc[k] = lrem[k] > 0 ? nc : INT_MAX;
            }
          }
          // the next window: the smallest next column over all entries
          int nxt = INT_MAX;
#pragma unroll
          for (int k = 0; k < KE; ++k) {
            nxt = min(nxt, hnx[k]);
            if (lrem[k] > 0) nxt = min(nxt, lnc[k]);
          }
          __syncthreads();  // the window's products are in LDS
          // emit in column order: one bitmap word per thread, positions by a group scan
          uint32_t wd = t < OWORD ? bm[t] : 0u;
          const int cntw = __popc(wd);
          const int inclw = wave_incl_scan_dpp(cntw);
          const int wm = wave_reduce_dpp(nxt, OpMin());
          if (lane == 63) red_cnt[wv] = inclw;
          if (lane == 0) red[wv] = wm;
          __syncthreads();
          int basew = 0, tot = 0, nlo = INT_MAX;
#pragma unroll
          for (int i = 0; i < NW; ++i) {
            const int ci = red_cnt[i];
            basew += i < wv ? ci : 0;
            tot += ci;
            nlo = min(nlo, red[i]);
          }
          if (wd) {
            int64_t pos = out + basew + inclw - cntw;
            bm[t] = 0u;
            while (wd) {
              const int bb = __ffs(wd) - 1;
              wd &= wd - 1u;
              const int o = t * 32 + bb;
              if (pos < c1) {
                Cidx[pos] = lo + o;
                Cval[pos] = dv[o];
              } else {
                flags |= kErrWindow;
              }
              dv[o] = V(0);
              ++pos;
            }
          }
          out += tot;
          // every next column lies past this window, so the loop moves on; the banded ranges
          // advance: a skipped window holds none of their elements, so the next start is this
          // end, and the next end is the prefetched one unless windows were skipped
          const int wn = nlo == INT_MAX ? wl + 1 : (nlo >> LOGVC);
#pragma unroll
          for (int k = 0; k < KE; ++k) {
            hs[k] = hs1[k];
            hs1[k] = (wn == w + 1 || hs1[k] >= hL[k]) ? hs1n[k] : hbi[k][min((wn + 1) * BPW, (int)nb1 - 1)];
          }
          w = wn;
          __syncthreads();  // cleared before the next window's products; reduction slots free
          if (++windows > psum) {  // uniform: no progress (reported; the row's output is not trusted)
            flags |= kErrWindow;
            break;
          }
        }
      }
      }
      if (!banded_done) {
      // ================= dense windows of VC columns, one walk =================
      LongState* st = nA <= kOldStates ? ostl : state + a0;
      int lmin = INT_MAX, lmax = -1;
      long long psum = 0;
      for (int64_t e = t; e < nA; e += NT) {
        LongState x;
        x.p = bstart[a0 + e];
        x.rem = blen[a0 + e];
        x.nc = x.rem > 0 ? Bidx[x.p] : INT_MAX;
        if (x.rem > 0) lmax = max(lmax, Bidx[x.p + x.rem - 1]);
        st[e] = x;
        lmin = min(lmin, x.nc);
        psum += x.rem;
      }
      // 8 lanes per entry when an entry averages 4 or more elements per window (its B row long
      // next to the number of VC-column windows the row's column span takes), else 4
      psum = Group<NT>::reduce(psum, OpAdd(), redl);
      const int cmax = Group<NT>::reduce(lmax, OpMax(), red_cnt);
      const int cmin = Group<NT>::reduce(lmin, OpMin(), red_cnt);
      const double span = cmax >= cmin ? (double)cmax - (double)cmin + 1.0 : 1.0;
      if ((double)psum * VC >= 4.0 * (double)nA * span) {
        G = 8;
        NSG = NT / G;
        sg = t / G;
        lg = t & (G - 1);
        sgbase = lane & ~(G - 1);
        submask = ((1ull << G) - 1ull) << sgbase;
      }
      int lo = cmin;  // the reductions above also ordered the state writes before the walk
      long long windows = 0;  // at most psum windows (each takes the element at its first column)
      while (lo != INT_MAX) {
        const int64_t hi = min((int64_t)lo + VC, (int64_t)INT_MAX);  // INT_MAX: exhausted entry
        lmin = INT_MAX;
        // 4 entries per subgroup at a time: their first loads are issued together
        for (int64_t e0 = sg; e0 < nA; e0 += (int64_t)NSG * 4) {  // subgroup-uniform
          LongState x[4];
          int c[4];
          V bv[4], va[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int64_t e = e0 + (int64_t)u * NSG;
            if (e < nA) x[u] = st[e];
            else x[u] = LongState{0, INT_MAX, 0};
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            c[u] = INT_MAX;
            bv[u] = V(0);
            va[u] = V(0);
            if (x[u].nc < hi) {  // subgroup-uniform
              const int64_t at = x[u].rem > 0 ? x[u].p + min(lg, x[u].rem - 1) : 0;
              const int cv = Bidx[at];
              bv[u] = Bval[at];
              va[u] = Aval[a0 + e0 + (int64_t)u * NSG];
              c[u] = lg < x[u].rem ? cv : INT_MAX;
            }
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if (x[u].nc < hi) {
              // the first G elements were loaded above; a B row with more in the window (a long
              // B row) continues UL steps of G at a time, their loads issued together
              bool done = false;
              {
                const int cu = c[u];
                const bool in = cu != INT_MAX && (int64_t)cu < hi;  // INT_MAX: B row exhausted
                if (in) {
                  const int o = cu - lo;
                  lds_add(&dv[o], va[u] * bv[u]);
                  atomicOr(&bm[o >> 5], 1u << (o & 31));
                }
                const int nin = __popcll(__ballot(in) & submask);
                if (nin < G) {
                  x[u].nc = __shfl(cu, sgbase + nin);
                  x[u].p += nin;
                  x[u].rem -= nin;
                  done = true;
                } else {
                  x[u].p += G;
                  x[u].rem -= G;
                }
              }
              // bounded: every pass either ends (fewer than G in the window) or takes G elements
              // off rem, and with rem <= 0 every lane holds the INT_MAX sentinel, which is
              // excluded explicitly, so the pass ends
              while (!done) {  // subgroup-uniform
                int cc[UL];
                V bb[UL];
#pragma unroll
                for (int k = 0; k < UL; ++k) {
                  const int kk = k * G + lg;
                  const int64_t at = x[u].rem > 0 ? x[u].p + min(kk, x[u].rem - 1) : 0;
                  const int cv = Bidx[at];
                  bb[k] = Bval[at];
                  cc[k] = kk < x[u].rem ? cv : INT_MAX;
                }
#pragma unroll
                for (int k = 0; k < UL; ++k) {
                  if (!done) {
                    const bool in = cc[k] != INT_MAX && (int64_t)cc[k] < hi;
                    if (in) {
                      const int o = cc[k] - lo;
                      lds_add(&dv[o], va[u] * bb[k]);
                      atomicOr(&bm[o >> 5], 1u << (o & 31));
                    }
                    const int nin = __popcll(__ballot(in) & submask);
                    if (nin < G) {
                      x[u].nc = __shfl(cc[k], sgbase + nin);
                      x[u].p += nin;
                      x[u].rem -= nin;
                      done = true;
                    } else {
                      x[u].p += G;
                      x[u].rem -= G;
                    }
                  }
                }
              }
              if (lg == 0) st[e0 + (int64_t)u * NSG] = x[u];
            }
            lmin = min(lmin, x[u].nc);
          }
        }
        __syncthreads();  // the window's products are in LDS
        // emit in column order: one bitmap word per thread, positions by a group scan
        uint32_t w = t < OWORD ? bm[t] : 0u;
        const int cnt = __popc(w);
        const int incl = wave_incl_scan_dpp(cnt);
        const int wm = wave_reduce_dpp(lmin, OpMin());
        if (lane == 63) red_cnt[wv] = incl;
        if (lane == 0) red[wv] = wm;
        __syncthreads();
        int base = 0, tot = 0, nlo = INT_MAX;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
          const int ci = red_cnt[i];
          base += i < wv ? ci : 0;
          tot += ci;
          nlo = min(nlo, red[i]);
        }
        if (w) {
          int64_t pos = out + base + incl - cnt;
          bm[t] = 0u;
          while (w) {
            const int bb = __ffs(w) - 1;
            w &= w - 1u;
            const int o = t * 32 + bb;
            if (pos < c1) {
              Cidx[pos] = lo + o;
              Cval[pos] = dv[o];
            } else {
              flags |= kErrWindow;
            }
            dv[o] = V(0);
            ++pos;
          }
        }
        out += tot;
        lo = nlo;
        __syncthreads();  // cleared before the next window's products; reduction slots free
        if (++windows > psum) {  // uniform: no progress (reported; the row's output is not trusted)
          flags |= kErrWindow;
          break;
        }
      }
      }
    }
    if (out != c1) flags |= kErrWindow;
  }
  flags = wave_reduce_dpp(flags, OpOr());
  if (lane == 0 && flags) atomicOr(err, flags);
}

// ------------------------------------------------------------------------------------
// backward: dA_ik = sum_j dC_ij B_kj ; dB_kj += A_ik dC_ij  (pattern of C from forward)
// ------------------------------------------------------------------------------------
// FP32 sums of dB over many products: every add rounds at the size of the sum so far, and thousands
// of rows meet in the values of a graph's hub rows (R-MAT 16: 400 products a value on average, a
// relative error of 1.1e-6 to 1.6e-6 with the order of the rows). From kDbPartsFrom products per
// value on, workgroup b adds into part b % kDbParts of a workspace instead, and the parts are added
// up in FP64: 2.1e-7 at the same speed. The parts go by XCD as the workgroups do.
constexpr int kDbParts = 8;
constexpr int64_t kDbPartsFrom = 32;
__global__ void k_db_sum(const float* __restrict__ part, int64_t n, float* __restrict__ dB) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    double x = 0.0;
#pragma unroll
    for (int q = 0; q < kDbParts; ++q) x += (double)part[q * n + i];
    dB[i] = (float)((double)dB[i] + x);
  }
}
size_t db_part_bytes(int dtype, int64_t products, int64_t nnzB) {
  return dtype == 0 && nnzB > 0 && products / nnzB >= kDbPartsFrom ? (size_t)kDbParts * 4 * (size_t)nnzB : 0;
}
void launch_db_sum(const void* part, int64_t n, void* dB, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_db_sum, dim3(fill_grid(n)), dim3(256), 0, s, (const float*)part, n, (float*)dB);
}

// LDS of one wave: the spans' tables, and per rank A's value and the sum of dA's products.
template <typename V>
struct BwdLds {
  SpanLds sp;
  V va[64];
  double acc[64];
};

// The products of one entry per lane (entry ka, `len` elements of its B row from `start` on, A's value
// va), element-parallel: find(c, g) looks the column up (1: g = dC_ij, 0: not this window's, -1: not in
// C's row), A_ik * dC_ij is added into dB and dC_ij * B_kj into the entry's sum, which goes to dA
// atomically (other waves and windows hold the rest of it; dA is 0 beforehand).
template <int U, typename V, typename F>
__device__ __forceinline__ void walk_bwd(int lane, int len, int64_t start, int64_t ka, V va, BwdLds<V>& l,
                                         const int32_t* __restrict__ Bidx, const V* __restrict__ Bval,
                                         V* __restrict__ dA, V* __restrict__ dB, int& bad, F&& find, int w0 = 0,
                                         int wstep = U) {
  int mine = -1;
  l.acc[lane] = 0.0;
  walk_spans<U>(lane, len, start, l.sp,
                [&](int r) {
                  l.va[r] = va;
                  mine = r;
                },
                [&](const int64_t (&at)[U], const int (&j)[U]) {
                  int c[U];
                  V b[U];
#pragma unroll
                  for (int u = 0; u < U; ++u) {
                    const int64_t p = at[u] < 0 ? 0 : at[u];
                    c[u] = Bidx[p];
                    b[u] = Bval[p];
                  }
#pragma unroll
                  for (int u = 0; u < U; ++u) {
                    V g = V(0);
                    const int ok = at[u] < 0 ? 0 : find(c[u], g);
                    if (ok < 0) bad = 1;
                    if (dB && ok > 0) atomicAdd(&dB[at[u]], l.va[j[u]] * g);
                    // lanes of one entry add into one sum, and LDS takes such adds lane after lane: a
                    // row of 16 lanes that is all one entry's (owners do not decrease along the lanes)
                    // adds up by DPP first
                    double x = ok > 0 ? (double)g * (double)b[u] : 0.0;
                    if (dpp_mov<0x150>(0, j[u]) == dpp_mov<0x15F>(0, j[u])) {  // row-uniform
                      x += dpp_mov<0xB1>(x, x);
                      x += dpp_mov<0x4E>(x, x);
                      x += dpp_mov<0x141>(x, x);
                      x += dpp_mov<0x140>(x, x);
                      if ((lane & 15) == 0) lds_add(&l.acc[j[u]], x);
                    } else if (ok > 0) {
                      lds_add(&l.acc[j[u]], x);
                    }
                  }
                },
                w0, wstep);
  wave_sync();
  if (dA && mine >= 0) atomicAdd(&dA[ka], (V)l.acc[mine]);
  wave_sync();  // the sums are rewritten by the wave's next entries
}

// Per C row: dC_i goes into an LDS table keyed by column; then the products of the row's entries are
// walked as in the forward kernels (rows of up to 64 entries by all waves together) and looked up.
// Bound by the atomics into dB: 266 G/s on neighbouring entries on this GPU (170 G/s in runs of 16).
// Walked 16 lanes per B row with 64 entries a wave, rows of 2049-4096 columns at R-MAT 16 took
// 1.98 ms, 0.49 now (an LDS add per product alone: 0.55).
template <typename V, int T, int NT>
__global__ __launch_bounds__(wg_of<NT>()) void k_backward_hash(
    const int32_t* __restrict__ rows, const int64_t* __restrict__ pbeg, const int64_t* __restrict__ pend,
    const int64_t* __restrict__ Aptr, const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
    const V* __restrict__ Aval, const int32_t* __restrict__ Bidx, const V* __restrict__ Bval,
    const int64_t* __restrict__ Cptr, const int32_t* __restrict__ Cidx, const V* __restrict__ dC,
    V* __restrict__ dA, V* __restrict__ dB, int64_t db_stride, int* __restrict__ err) {
  constexpr int WG = wg_of<NT>();
  constexpr int GPB = WG / NT;
  constexpr int NW = NT / 64;
  constexpr int U = 4;
  static_assert(NT % 64 == 0 && T % NT == 0, "shape");
  __shared__ int hk[GPB][T];
  __shared__ V hv[GPB][T];
  __shared__ BwdLds<V> bl[WG / 64];
  __shared__ int sc[GPB][NT > 64 ? NT / 64 : 1];
  if (dB) dB += (blockIdx.x % kDbParts) * db_stride;
  const int t = threadIdx.x % NT;
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
  const int lane = t & 63, wv = t >> 6;
  BwdLds<V>& l = bl[__builtin_amdgcn_readfirstlane(threadIdx.x / 64)];
  int* K = hk[g];
  V* H = hv[g];
  const int64_t beg = *pbeg, end = *pend;
  for (int64_t slot = beg + (int64_t)blockIdx.x * GPB + g; slot < end; slot += (int64_t)gridDim.x * GPB) {
    const int row = rows[slot];
#pragma unroll
    for (int s = t; s < T; s += NT) K[s] = kEmpty;
    gsync<NT>();
    const int64_t c0 = Cptr[row], c1 = Cptr[row + 1];
    int bad = 0;
    for (int64_t m = c0 + t; m < c1; m += NT) {
      const int c = Cidx[m];
      uint32_t h = hslot<T>(c);
      // keys of a C row are unique: claim the first free slot
      for (int probe = 0; probe < T; ++probe) {
        if (atomicCAS(K + h, kEmpty, c) == kEmpty) {
          H[h] = dC[m];
          break;
        }
        h = (h + 1) & (T - 1);
      }
    }
    gsync<NT>();
    const int64_t a0 = Aptr[row], a1 = Aptr[row + 1];
    const bool shared = NW > 1 && a1 - a0 <= 64;  // uniform
    for (int64_t base = a0; base < a1; base += NT) {
      const int64_t ka = base + (shared ? lane : wv + NW * lane);
      const bool have = ka < a1;
      walk_bwd<U>(lane, have ? blen[ka] : 0, have ? bstart[ka] : 0, ka, have ? Aval[ka] : V(0), l, Bidx, Bval, dA, dB, bad,
                  [&](int c, V& gv) {
                    const int s = hash_find<T>(K, c);
                    if (s < 0) return -1;  // C does not belong to these operands
                    gv = H[s];
                    return 1;
                  },
                  shared ? wv * U : 0, shared ? NW * U : U);
    }
    bad = Group<NT>::reduce(bad, OpMax(), sc[g]);
    if (t == 0 && bad) atomicOr(err, kErrMissingKey);
    gsync<NT>();
  }
}

// Rows of thousands of columns of a B of at most BW columns: C's row as a bitmap with its prefix, which
// turns a product's column into its rank, and the row's part of dC by rank, VC values at a time (the
// products are walked once for each). Bound by the atomics into dB, behind the chain bitmap - prefix -
// value of a lookup: two workgroups of 8 waves share a CU (79 KB of LDS). At R-MAT 16, FP32, the 3,900
// rows of more than 4096 columns that are no hub rows 1.64 (k_backward_long) -> 0.49 ms, those of
// 1025-4096 0.60 (k_backward_hash) -> 0.4 ms. any_order: C's row may list its columns in any order, as in
// the tables (the windows of k_backward_long take them in order only).
template <typename V, int NT, int VC, int BW>
__global__ __launch_bounds__(NT) void k_backward_rank(
    const int32_t* __restrict__ rows, const int64_t* __restrict__ pbeg, const int64_t* __restrict__ pend,
    const int64_t* __restrict__ Aptr, const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
    const V* __restrict__ Aval, const int32_t* __restrict__ Bidx, const V* __restrict__ Bval,
    const int64_t* __restrict__ Cptr, const int32_t* __restrict__ Cidx, const V* __restrict__ dC,
    V* __restrict__ dA, V* __restrict__ dB, int64_t db_stride, int* __restrict__ err, bool any_order) {
  constexpr int NW = NT / 64, U = 4, NWORD = BW / 64;
  static_assert(NWORD == 2 * NT, "two words a thread");
  __shared__ V val[VC];
  __shared__ unsigned long long bm[NWORD];
  __shared__ uint16_t pre[NT];
  __shared__ BwdLds<V> bl[NW];
  __shared__ int sc[NW];
  if (dB) dB += (blockIdx.x % kDbParts) * db_stride;
  uint32_t* bm32 = reinterpret_cast<uint32_t*>(bm);
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t beg = *pbeg, end = *pend;
  int bad = 0;
  for (int64_t slot = beg + blockIdx.x; slot < end; slot += gridDim.x) {
    const int row = rows[slot];
    const int64_t a0 = Aptr[row], a1 = Aptr[row + 1], c0 = Cptr[row];
    const int n = (int)min(Cptr[row + 1] - c0, (int64_t)BW);
    bm[2 * t] = bm[2 * t + 1] = 0ull;
    __syncthreads();
    int falls = 0;
    for (int m = t; m < n; m += NT) {
      const uint32_t c = (uint32_t)Cidx[c0 + m];
      if (c < (uint32_t)BW) atomicOr(&bm32[c >> 5], 1u << (c & 31));
      else bad = 1;
      if (any_order && m > 0) falls |= (uint32_t)Cidx[c0 + m - 1] >= c;
    }
    const bool rises = !__syncthreads_or(falls);  // the columns, so an entry's place is its rank
    int total;
    const int mine = __popcll(bm[2 * t]) + __popcll(bm[2 * t + 1]);
    pre[t] = (uint16_t)Group<NT>::exscan(mine, total, sc);  // below 65536: of all columns one lies behind
    if (total != n) bad = 1;
    __syncthreads();
    // rank of a column, -1 if C's row does not have it
    auto rank = [&](int col) -> int {
      const uint32_t c = (uint32_t)col;
      if (c >= (uint32_t)BW) return -1;
      const int w = c >> 6;
      const unsigned long long x = bm[w], y = w & 1 ? bm[w - 1] : 0ull;
      if (!(x >> (c & 63) & 1ull)) return -1;
      return (int)pre[w >> 1] + __popcll(y) + __popcll(x & ((1ull << (c & 63)) - 1ull));
    };
    const bool shared = a1 - a0 <= 64;  // uniform
    for (int m0 = 0; m0 < n; m0 += VC) {  // uniform
      const int nv = min(VC, n - m0);
      if (rises) {
        for (int m = t; m < nv; m += NT) val[m] = dC[c0 + m0 + m];
      } else {
        for (int m = t; m < n; m += NT) {
          const uint32_t r = (uint32_t)(rank(Cidx[c0 + m]) - m0);
          if (r < (uint32_t)nv) val[r] = dC[c0 + m];
        }
      }
      __syncthreads();
      for (int64_t base = a0; base < a1; base += NT) {
        const int64_t ka = base + (shared ? lane : wv + NW * lane);
        const bool have = ka < a1;
        walk_bwd<U>(lane, have ? blen[ka] : 0, have ? bstart[ka] : 0, ka, have ? Aval[ka] : V(0), bl[wv], Bidx, Bval, dA, dB,
                    bad,
                    [&](int c, V& g) {
                      const int r = rank(c);
                      if (r < 0) return -1;
                      if ((uint32_t)(r - m0) >= (uint32_t)nv) return 0;
                      g = val[r - m0];
                      return 1;
                    },
                    shared ? wv * U : 0, shared ? NW * U : U);
      }
      __syncthreads();
    }
  }
  if (__builtin_amdgcn_ballot_w64(bad) && lane == 0) atomicOr(err, kErrMissingKey);
}

// Hub rows in column windows of SR ranges, a workgroup per (row, window): the window's part of C's
// row (found by the symbolic pass's range counts) lies densely in LDS, and the entries are read as in
// k_hub_range; the short ones whole in every window, so few windows are wanted (hub_backward_ranges).
// The 5,900 heaviest rows at R-MAT 16, FP32: 2.96 ms (4.73 with an LDS add per product, whose lanes
// mostly share an entry; 2.6 of it without any), of which the atomics into dB take 1 ms.
__device__ __forceinline__ float absent(float) { return __int_as_float(0x7fc0dead); }
__device__ __forceinline__ double absent(double) { return __longlong_as_double(0x7ff8dead00000000ll); }
__device__ __forceinline__ bool is_absent(float x) { return __float_as_int(x) == 0x7fc0dead; }
__device__ __forceinline__ bool is_absent(double x) { return __double_as_longlong(x) == 0x7ff8dead00000000ll; }

template <typename V, int NT, int SR>
__global__ __launch_bounds__(NT) void k_hub_backward(
    const HubRow* __restrict__ info, int nrng, int nwin, const V* __restrict__ Aval, const int32_t* __restrict__ Bidx,
    const V* __restrict__ Bval, const int32_t* __restrict__ band, int64_t nb1, const HubRec* __restrict__ recs,
    const int64_t* __restrict__ roff, const int32_t* __restrict__ Cidx, const V* __restrict__ dC, V* __restrict__ dA,
    V* __restrict__ dB, int64_t db_stride, int* __restrict__ err) {
  constexpr int W = SR * kHubRange;
  constexpr int NW = NT / 64;
  constexpr int U = 4;
  static_assert(W % NT == 0, "shape");
  __shared__ V dv[W];
  __shared__ BwdLds<V> bl[NW];
  if (dB) dB += (blockIdx.x % kDbParts) * db_stride;
  const int64_t j = blockIdx.x / nwin;
  const int w = (int)(blockIdx.x - j * nwin);
  const int64_t* ro = roff + j * nrng;
  const int64_t o0 = ro[w * SR] - ro[0], o1 = ro[min(w * SR + SR, nrng)] - ro[0];
  const HubRow row = info[j];
  if (o1 == o0) return;  // no column, so no product
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int64_t c0 = (int64_t)w * W;
  int bad = 0;
#pragma unroll 4
  for (int q = t; q < W; q += NT) dv[q] = absent(V(0));
  __syncthreads();
  for (int64_t m = o0 + t; m < o1; m += NT) {
    const int64_t o = Cidx[row.out + m] - c0;
    if (o >= 0 && o < W) dv[o] = dC[row.out + m];
    else bad = 1;
  }
  __syncthreads();
  const int64_t w0 = c0 >> kBandShift, w1 = min((c0 + W) >> kBandShift, nb1 - 1);
  for (int e0 = 0; e0 < row.nH; e0 += NT) {  // uniform
    const int e = e0 + wv + NW * lane;
    int len = 0;
    int64_t start = 0, ka = 0;
    V va = V(0);
    if (e < row.nH) {
      const HubRec q = recs[row.a0 + e];
      const int32_t* bd = band + (int64_t)q.s * nb1;
      const int s0 = bd[w0];
      len = bd[w1] - s0;
      start = q.b0 + s0;
      ka = row.a0 + q.e;
      va = Aval[ka];
    }
    walk_bwd<U>(lane, len, start, ka, va, bl[wv], Bidx, Bval, dA, dB, bad, [&](int c, V& g) {
      g = dv[c - c0];
      return is_absent(g) ? -1 : 1;
    });
  }
  for (int e0 = 0; e0 < row.nL; e0 += NT) {  // uniform
    const int e = e0 + wv + NW * lane;
    const HubRec q = e < row.nL ? recs[row.a1 - 1 - e] : HubRec{0, 0, 0};
    const int64_t ka = row.a0 + q.e;
    walk_bwd<U>(lane, q.s, q.b0, ka, e < row.nL ? Aval[ka] : V(0), bl[wv], Bidx, Bval, dA, dB, bad, [&](int c, V& g) {
      const int64_t o = c - c0;
      if (o < 0 || o >= W) return 0;
      g = dv[o];
      return is_absent(g) ? -1 : 1;
    });
  }
  if (__builtin_amdgcn_ballot_w64(bad) && lane == 0) atomicOr(err, kErrMissingKey);
}

// Long rows: dC's row values are scattered into a dense LDS window (the C row is sorted, so
// windows follow it); B cursors advance per window; dA accumulates across windows.
template <typename V, int NT, int W, int G>
__global__ __launch_bounds__(NT) void k_backward_long(
    const int32_t* __restrict__ rows, const int64_t* __restrict__ pbeg, const int64_t* __restrict__ pend,
    const int64_t* __restrict__ Aptr, const int32_t* __restrict__ Aidx, const V* __restrict__ Aval,
    const int64_t* __restrict__ Bptr, const int32_t* __restrict__ Bidx, const V* __restrict__ Bval,
    const int64_t* __restrict__ Cptr, const int32_t* __restrict__ Cidx, const V* __restrict__ dC,
    V* __restrict__ dA, V* __restrict__ dB, int64_t db_stride, int64_t* __restrict__ cursor, int* __restrict__ err) {
  __shared__ V dv[W];
  __shared__ int sc[NT / 64];
  __shared__ long long scl[NT / 64];
  if (dB) dB += (blockIdx.x % kDbParts) * db_stride;
  const int t = threadIdx.x;
  const int64_t beg = *pbeg, end = *pend;
  // rows from the end of the range: callers put the heaviest rows last
  for (int64_t s2 = beg + blockIdx.x; s2 < end; s2 += gridDim.x) {
    const int row = rows[end - 1 - (s2 - beg)];
    const int64_t a0 = Aptr[row], a1 = Aptr[row + 1];
    const int64_t c0 = Cptr[row], c1 = Cptr[row + 1];
    for (int64_t ka = a0 + t; ka < a1; ka += NT) {
      cursor[2 * ka] = Bptr[Aidx[ka]];
      if (dA) dA[ka] = V(0);
    }
    int64_t cc = c0;
    __syncthreads();
    int bad = 0;
    while (cc < c1) {
      const int lo = Cidx[cc];
      const int64_t hi = min((int64_t)lo + W, (int64_t)INT_MAX);  // INT_MAX: past the B row
      // C entries of this window: [cc, ce)
      // a window holds at most W distinct columns, so entries past cc + W are outside it
      long long ce_l = min((long long)c1, (long long)(cc + W));
      for (int64_t m = cc + t; m < c1 && m < cc + W; m += NT) {
        const int c = Cidx[m];
        if ((int64_t)c < hi) {
          dv[c - lo] = dC[m];
        } else {
          ce_l = min(ce_l, (long long)m);
        }
      }
      const int64_t ce = Group<NT>::reduce(ce_l, OpMin(), scl);
      for (int64_t ka = a0 + t / G; ka < a1; ka += NT / G) {
        const int k = Aidx[ka];
        const V va = Aval[ka];
        int64_t p = cursor[2 * ka];
        const int64_t b1 = Bptr[k + 1];
        V acc = V(0);
        // one step of G, then (a long B row) UL steps at a time with their loads issued together
        int nin = G;
        for (int first = 1; nin == G && p < b1; first = 0) {  // subgroup-uniform
          constexpr int UL = 4;
          int cc[UL];
          V bb[UL];
          const int ns = first ? 1 : UL;
#pragma unroll
          for (int k = 0; k < UL; ++k) {
            const int64_t q = p + k * G + (t % G);
            const bool ok = k < ns && q < b1;
            cc[k] = ok ? Bidx[q] : INT_MAX;
            bb[k] = ok ? Bval[q] : V(0);
          }
#pragma unroll
          for (int k = 0; k < UL; ++k) {
            if (k < ns && nin == G) {
              const int64_t q = p + (t % G);
              const int c = cc[k];
              const bool in = (int64_t)c < hi;
              if (in && c >= lo) {
                const V gv = dv[c - lo];
                acc += gv * bb[k];
                if (dB) atomicAdd(&dB[q], va * gv);
              } else if (in) {
                bad = 1;  // product column absent from C's row: C does not belong to these operands
              }
              nin = __popcll(__ballot(in) & subgroup_mask<G>());
              p += nin;
            }
          }
        }
#pragma unroll
        for (int o = G / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, G);
        if ((t % G) == 0) {
          cursor[2 * ka] = p;
          if (dA) dA[ka] += acc;
        }
      }
      __syncthreads();
      // clear the window entries that were set
      for (int64_t m = cc + t; m < ce; m += NT) dv[Cidx[m] - lo] = V(0);
      if (ce <= cc) bad = 1;
      cc = (ce > cc) ? ce : c1;
      __syncthreads();
    }
    // every B entry reached must have been covered by a window
    for (int64_t ka = a0 + t; ka < a1; ka += NT)
      if (cursor[2 * ka] != Bptr[Aidx[ka] + 1]) bad = 1;
    bad = Group<NT>::reduce(bad, OpMax(), sc);
    if (t == 0 && bad) atomicOr(err, kErrMissingKey);
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------
// dispatch tables
// ------------------------------------------------------------------------------------
static int device_cus() {
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev] = n;
  }
  return cus[dev];
}

// Workgroups of kernel f (block threads) resident on one CU, from the occupancy calculator.
static int resident_blocks(const void* f, int block) {
  static std::mutex mu;
  static std::map<std::pair<const void*, int>, int> cache;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = 0;
  std::lock_guard<std::mutex> lk(mu);
  const auto key = std::make_pair(f, block * 64 + dev);
  auto it = cache.find(key);
  if (it != cache.end()) return it->second;
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, f, block, 0) != hipSuccess || n < 1) n = 4;
  cache[key] = n;
  return n;
}

// Grid of a row kernel: for persistent launches (`grid` given) as many workgroups as are resident at
// once where the kernel is named (two per CU, whatever the shape, left most of a CU idle: a batch of 32
// 5.69 ms, 5.03 so), else `grid`; otherwise one group per row. The
// one-wave-per-row kernels (gpb > 1) walk many rows per wave, their row pipeline amortising
// over them: their grid is capped at what is resident at once, so no second, partly filled
// round of workgroups follows the first (all workgroups get equal row counts).
static int grid_for(int64_t nrows, int gpb, int grid, const void* f = nullptr, int block = 256) {
  int64_t g = (nrows + gpb - 1) / gpb;
  if (grid > 0)
    return f ? (int)std::max<int64_t>(std::min<int64_t>(g, (int64_t)device_cus() * resident_blocks(f, block)), 1) : grid;
  if (gpb > 1 && f) g = std::min<int64_t>(g, (int64_t)device_cus() * resident_blocks(f, block));
  if (g > 1048576) g = 1048576;
  if (g < 1) g = 1;
  return (int)g;
}

// Rows of a category from which several share a wave: up to there every row can have a wave of its own
// at once (256 CUs, 20 waves each), whose chain is shorter (1,000 rows of 62: 8 us against 14). From
// there on, per launch: 1,200,000 rows of up to 32 columns 0.70 -> 0.26 ms, batch members' rows of up
// to 64 / 128 columns 52 -> 36 / 67 -> 50 us. Rows of distinct products past 32 columns keep the
// register path of k_numeric_wave_fast (20,000 rows of up to 64 columns: 26 us against 40).
constexpr int64_t kMultiRows = 8192;

constexpr int kLongNT = 256;
constexpr int kSymLongW = 131072;  // bits per symbolic window (16 KB bitmap)
#ifndef DBD_NUM_LONG_BW
#define DBD_NUM_LONG_BW 65536
#endif
constexpr int kNumLongBW = DBD_NUM_LONG_BW;  // columns per numeric window (bitmap + word prefixes)
constexpr int kNumLongVC64 = 4096;  // FP64 values per window (32 KB; with 8 KB of cursors: 3 workgroups per CU)
constexpr int kNumLongVC32 = 8192;  // FP32 values per window (32 KB)
constexpr int kBwdLongW64 = 8192;
constexpr int kBwdLongW32 = 16384;
constexpr int kLongG = 16;

#define DBD_SHAPES(X, G) \
  X(64, 64, G)           \
  X(128, 64, G)          \
  X(256, 64, G)          \
  X(512, 64, G)          \
  X(1024, 128, G)        \
  X(2048, 256, G)        \
  X(4096, 512, G)        \
  X(8192, 1024, G)

int symbolic_groups_per_wg(const KernelShape& k) {
  if (k.T <= 0) return 1;  // long and hub rows: one workgroup per row
  return k.NT <= 64 ? 256 / k.NT : 1;
}

// Threads per row of the symbolic tables from 1024 slots on. Many rows: one wave up to 2048 slots, 256
// and 512 threads for 4096 and 8192 (waiting on the barriers and clearing the table are most of what a
// row costs, and more rows share a CU). Few rows, which leave CUs idle: the widest workgroups, whose
// chains are shorter. Per launch, wide -> narrow: 300,007 rows of 297 products 569 -> 326 us, 99,000
// rows of 1024-2048 332 -> 254 us, 3,200 of 2048-4096 31 -> 20 us; a few hundred to 2000 rows of each
// of a web graph 24 -> 65 us in all.
constexpr int64_t kFewWaveRows = 8192, kFewGroupRows = 1024;
static KernelShape symbolic_shape(KernelShape k, int64_t nrows) {
  if (k.NT == 64 && nrows <= kFewWaveRows && (k.T == 1024 || k.T == 2048)) return {k.T, k.T / 8, 64};
  if (k.NT == k.T / 16 && nrows <= kFewGroupRows && (k.T == 4096 || k.T == 8192)) return {k.T, k.T / 8, k.G};
  return k;
}

void launch_symbolic(const KernelShape& table_shape, const int32_t* rows, const int64_t* pbeg, const int64_t* pend,
                     int64_t nrows_hint, int grid, const Mat& A, const Mat& B, int64_t* nnz, int64_t* cursor,
                     int* err, hipStream_t s, const int32_t* hub_slot) {
  const KernelShape k = symbolic_shape(table_shape, nrows_hint);
  const int gpb = symbolic_groups_per_wg(k);
  if (k.T == 0) {
    const dim3 gr(grid_for(nrows_hint, gpb, grid));
    hipLaunchKernelGGL((k_symbolic_long<1024, kSymLongW, kLongG>), gr, dim3(1024), 0, s, rows, pbeg, pend, A.ptr,
                       A.bstart, A.blen, B.idx, nnz, cursor, err, hub_slot, A.idx, B.hslot, B.band, B.nb1);
    return;
  }
#define M(T_)                                                                                                    \
  if (k.T == T_ && k.NT == 64 && k.G == 16 && nrows_hint > kMultiRows) {                                       \
    const dim3 gr(grid_for(nrows_hint, 4 * (kMultiSlots / T_), grid, (const void*)k_symbolic_multi<T_>, 256)); \
    hipLaunchKernelGGL((k_symbolic_multi<T_>), gr, dim3(256), 0, s, rows, pbeg, pend, A.ptr, A.bstart, A.blen, \
                       B.idx, nnz, err);                                                                        \
    return;                                                                                                     \
  }
  M(64)
  M(128)
  M(256)
#undef M
#define X(T_, NT_, G_)                                                                                         \
  if (k.T == T_ && k.NT == NT_ && k.G == G_) {                                                               \
    const dim3 gr(grid_for(nrows_hint, gpb, grid, (const void*)k_symbolic_hash<T_, NT_, G_>, wg_of<NT_>())); \
    hipLaunchKernelGGL((k_symbolic_hash<T_, NT_, G_>), gr, dim3(wg_of<NT_>()), 0, s, rows, pbeg, pend, A.ptr, \
                       A.bstart, A.blen, B.idx, nnz, err);                                                   \
    return;                                                                                                   \
  }
  DBD_SHAPES(X, 16)
  DBD_SHAPES(X, 64)
  X(16384, 1024, 16)
  X(16384, 1024, 64)
  X(1024, 64, 16)
  X(1024, 64, 64)
  X(2048, 64, 16)
  X(2048, 64, 64)
  X(4096, 256, 16)
  X(4096, 256, 64)
  X(8192, 512, 16)
  X(8192, 512, 64)
#undef X
}

// k_numeric_rank takes the rows of the long category and of the tables from kRankSlots on where its
// windows are few: B no wider than a window of ranks (long rows without a band index: 16 windows of
// values), or B's band index leaving only short rows out. Long rows without a band index, one
// allocation-free product of skewed rows against the cursor windows of k_numeric_long: 6007 columns
// 0.80 -> 0.43 ms, 20,011 columns 2.0 -> 1.07 ms, 59,999 columns 70 -> 35 ms.
constexpr int kRankNT = 512, kRankVC = 4096, kRankBW = 65536, kRankSlots = 4096;
static bool rank_rows(const Mat& B) {
  return B.band ? B.band_min <= kRankShort : B.ncols <= kRankBW;
}

template <typename V>
static void launch_numeric_t(const KernelShape& k, const int32_t* rows, const int64_t* pbeg, const int64_t* pend,
                             int64_t nrows_hint, int grid, const Mat& A, const Mat& B, const int64_t* Cptr,
                             int64_t cbase, int32_t* Cidx, V* Cval, int64_t* cursor, int* err, hipStream_t s,
                             bool distinct) {
  const int gpb = symbolic_groups_per_wg(k);
  const V* Av = (const V*)A.val;
  const V* Bv = (const V*)B.val;
  const bool is_long = k.T == 0 || k.T == kHubShape;
  if ((is_long || k.T >= kRankSlots) && rank_rows(B)) {
    auto run = [&](auto* kernel) {
      const dim3 gr(grid_for(nrows_hint, 1, grid, (const void*)kernel, kRankNT));
      hipLaunchKernelGGL(kernel, gr, dim3(kRankNT), 0, s, rows, pbeg, pend, A.ptr, A.bstart, A.blen, Av, B.idx, Bv, Cptr,
                         cbase, Cidx, Cval, err, A.idx, B.hslot, B.band, B.nb1);
    };
    if (B.band && (is_long || B.ncols > kRankBW)) run(k_numeric_rank<V, kRankNT, kRankVC, kRankBW, true>);
    else run(k_numeric_rank<V, kRankNT, kRankVC, kRankBW, false>);
    return;
  }
  if (is_long) {  // hub rows reach here only when the range kernels cannot run
    const dim3 gr(grid_for(nrows_hint, gpb, grid));
    constexpr int VC = sizeof(V) == 8 ? kNumLongVC64 : kNumLongVC32;
    hipLaunchKernelGGL((k_numeric_long<V, kLongNT, kNumLongBW, VC>), gr, dim3(kLongNT), 0, s, rows, pbeg, pend, A.ptr,
                       A.bstart, A.blen, Av, B.idx, Bv, Cptr, cbase, Cidx, Cval, (LongState*)cursor, err, A.idx,
                       B.hslot, B.band, B.nb1);
    return;
  }
#define M(T_)                                                                                                    \
  if (k.T == T_ && k.NT == 64 && k.G == 16 && nrows_hint > kMultiRows && (T_ == 64 || !distinct)) {            \
    const dim3 gr(grid_for(nrows_hint, 4 * (kMultiSlots / T_), grid, (const void*)k_numeric_multi<V, T_>, 256)); \
    hipLaunchKernelGGL((k_numeric_multi<V, T_>), gr, dim3(256), 0, s, rows, pbeg, pend, A.ptr, A.bstart, A.blen, \
                       Av, B.idx, Bv, Cptr, cbase, Cidx, Cval, err);                                            \
    return;                                                                                                     \
  }
  M(64)
  M(128)
  M(256)
#undef M
#define X(T_, NT_, G_)                                                                                           \
  if (k.T == T_ && k.NT == NT_ && k.G == G_) {                                                                 \
    if constexpr (NT_ == 64) {                                                                                 \
      if (distinct) {                                                                                          \
        const dim3 gr(grid_for(nrows_hint, gpb, grid, (const void*)k_numeric_wave_fast<V, T_, NT_, G_>, 256)); \
        hipLaunchKernelGGL((k_numeric_wave_fast<V, T_, NT_, G_>), gr, dim3(256), 0, s, rows, pbeg, pend,       \
                           A.ptr, A.bstart, A.blen, Av, B.idx, Bv, Cptr, cbase, Cidx, Cval, err);             \
      } else {                                                                                                 \
        const dim3 gr(grid_for(nrows_hint, gpb, grid, (const void*)k_numeric_wave<V, T_, NT_, G_>, 256));      \
        hipLaunchKernelGGL((k_numeric_wave<V, T_, NT_, G_>), gr, dim3(256), 0, s, rows, pbeg, pend, A.ptr,     \
                           A.bstart, A.blen, Av, B.idx, Bv, Cptr, cbase, Cidx, Cval, err);                    \
      }                                                                                                        \
    } else {                                                                                                    \
      const dim3 gr(grid_for(nrows_hint, gpb, grid, (const void*)k_numeric_block<V, T_, NT_, G_>, NT_));       \
      hipLaunchKernelGGL((k_numeric_block<V, T_, NT_, G_>), gr, dim3(NT_), 0, s, rows, pbeg, pend, A.ptr,      \
                         A.bstart, A.blen, Av, B.idx, Bv, Cptr, cbase, Cidx, Cval, err);                      \
    }                                                                                                           \
    return;                                                                                                     \
  }
  DBD_SHAPES(X, 16)
  DBD_SHAPES(X, 64)
#undef X
}

void launch_numeric(int dtype, const KernelShape& k, const int32_t* rows, const int64_t* pbeg, const int64_t* pend,
                    int64_t nrows_hint, int grid, const Mat& A, const Mat& B, const int64_t* Cptr, int64_t cbase,
                    int32_t* Cidx, void* Cval, int64_t* cursor, int* err, hipStream_t s, bool distinct) {
  if (dtype == 1)
    launch_numeric_t<double>(k, rows, pbeg, pend, nrows_hint, grid, A, B, Cptr, cbase, Cidx, (double*)Cval, cursor,
                             err, s, distinct);
  else
    launch_numeric_t<float>(k, rows, pbeg, pend, nrows_hint, grid, A, B, Cptr, cbase, Cidx, (float*)Cval, cursor,
                            err, s, distinct);
}

int hub_ranges(int64_t ncols) { return (int)((ncols + kHubRange - 1) >> kHubRangeShift); }
bool hub_buckets_used(int64_t ncols) { return hub_ranges(ncols) > kHubWhole; }

// A wave per long row. The rule counts the ranges between the row's first and last column, over at
// most kHubEntries of its entries (rows of more are hub rows anyway).
__global__ __launch_bounds__(256) void k_hub_flags(const int32_t* __restrict__ rows, int64_t n,
                                                   const int64_t* __restrict__ Aptr, const int64_t* __restrict__ P,
                                                   const int64_t* __restrict__ bstart, const int32_t* __restrict__ blen,
                                                   const int32_t* __restrict__ Bidx, int64_t per_range, int wide,
                                                   int64_t products, int64_t* __restrict__ flag) {
  const int lane = threadIdx.x & 63;
  for (int64_t j = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); j < n; j += (int64_t)gridDim.x * 4) {
    const int r = rows[j];
    const int64_t a0 = Aptr[r], nA = Aptr[r + 1] - a0, p = P[r];
    const int m = (int)min(nA, kHubEntries);
    int cmin = INT_MAX, cmax = -1;
    for (int e = lane; e < m; e += 64) {
      const int64_t ka = a0 + e * nA / m;
      const int L = blen[ka];
      if (L <= 0) continue;
      cmin = min(cmin, Bidx[bstart[ka]]);
      cmax = max(cmax, Bidx[bstart[ka] + L - 1]);
    }
    cmin = wave_reduce_dpp(cmin, OpMin());
    cmax = wave_reduce_dpp(cmax, OpMax());
    if (lane == 0) {
      const int nrng = cmax >= cmin ? (cmax >> kHubRangeShift) - (cmin >> kHubRangeShift) + 1 : 1;
      const bool hub = hub_row(nA, p, nrng, per_range);
      const bool fine = hub && hub_fine(p, nrng, wide, products);
      flag[j] = (hub ? 1 : 0) + (fine ? kHubFineOne : 0);
    }
  }
}

__global__ void k_hub_slots(const int32_t* __restrict__ rows, int64_t n, const int64_t* __restrict__ flag,
                            const int64_t* __restrict__ pos, const int64_t* __restrict__ Aptr,
                            int32_t* __restrict__ hub_slot, int32_t* __restrict__ hub_rows, int32_t* __restrict__ fine) {
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x) {
    if (!flag[j]) continue;
    const int r = rows[j];
    const int32_t sl = (int32_t)(pos[j] & (kHubFineOne - 1));
    const bool is_fine = flag[j] >= kHubFineOne;
    hub_slot[r] = sl | (Aptr[r + 1] - Aptr[r] > kHubEntries ? kHubMany : 0) | (is_fine ? kHubFineBit : 0);
    hub_rows[sl] = r;
    if (is_fine) fine[pos[j] >> kHubFineShift] = sl;
  }
}

__global__ void k_hub_gather_counts(const int32_t* __restrict__ rows, int64_t n, int nrng,
                                    const int32_t* __restrict__ hub_slot, const int32_t* __restrict__ hcnt,
                                    const int32_t* __restrict__ lcnt, const int32_t* __restrict__ rng_cnt,
                                    const int64_t* __restrict__ Aptr, const int64_t* __restrict__ Cptr, int64_t cbase,
                                    int64_t* __restrict__ rcnt, HubRow* __restrict__ info) {
  const int64_t items = n * nrng;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < items; q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t j = q / nrng;
    const int r = (int)(q - j * nrng);
    const int row = rows[j], hs = hub_slot[row];
    // a row without a slot (only if a captured pipeline's operands changed structure) has none
    rcnt[q] = hs >= 0 ? rng_cnt[(int64_t)(hs & kHubSlotMask) * nrng + r] : 0;
    if (r == 0)
      info[j] = HubRow{Aptr[row], Aptr[row + 1], Cptr[row] - cbase, hs >= 0 ? hcnt[hs & kHubSlotMask] : 0,
                       hs >= 0 ? lcnt[hs & kHubSlotMask] : 0};
  }
}

void launch_hub_flags(const int32_t* rows, int64_t n, const Mat& A, const Mat& B, const int64_t* P, int64_t per_range,
                      int wide, int64_t products, int64_t* flag, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_hub_flags, dim3(fill_grid(64 * n)), dim3(256), 0, s, rows, n, A.ptr, P, A.bstart, A.blen, B.idx,
                     per_range, wide, products, flag);
}
void launch_hub_slots(const int32_t* rows, int64_t n, const Mat& A, const int64_t* flag, const int64_t* pos,
                      const HubWork& h, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_hub_slots, dim3(fill_grid(n)), dim3(256), 0, s, rows, n, flag, pos, A.ptr, h.slot, h.rows, h.fine);
}
void launch_hub_gather_counts(const HubWork& h, const int32_t* rows, int64_t n, const Mat& A, const Mat& B,
                              const int64_t* Cptr, int64_t cbase, int64_t* rcnt, hipStream_t s) {
  if (n <= 0) return;
  const int nrng = hub_ranges(B.ncols);
  hipLaunchKernelGGL(k_hub_gather_counts, dim3(fill_grid(n * nrng)), dim3(256), 0, s, rows, n, nrng, h.slot, h.hcnt,
                     h.lcnt, h.rng_cnt, A.ptr, Cptr, cbase, rcnt, (HubRow*)h.info);
}

void launch_hub_split(const HubWork& h, const Mat& A, const Mat& B, const int64_t* P, int64_t key_lim, int64_t* nnz,
                      int* many, hipStream_t s) {
  if (h.n <= 0) return;
  hipLaunchKernelGGL(k_hub_chunks, dim3(fill_grid(h.n)), dim3(256), 0, s, h.rows, h.n, A.ptr, P, B.ncols, key_lim,
                     h.coff, h.hcnt, h.lcnt, h.span, nnz, many);
  launch_exclusive_scan(h.coff, h.coff, h.n, h.tmp, s);
  // every row has at most one partly filled chunk
  hipLaunchKernelGGL(k_hub_split, dim3((unsigned)(A.nnz / kHubChunk + h.n)), dim3(kHubSplitNT), 0, s, h.rows, h.n,
                     h.coff, A.ptr, A.idx, A.bstart, A.blen, B.idx, B.hslot, (HubRec*)h.recs, h.hcnt, h.lcnt, h.span);
}

// Launches of n rows x nwin windows in groups of fewer than 2^32 work-items: go(first row, rows).
template <typename F>
static void row_groups(int64_t n, int nwin, int nt, F&& go) {
  const int64_t per = std::max<int64_t>(1, (((int64_t)1 << 32) / nt - 1) / nwin);
  for (int64_t j0 = 0; j0 < n; j0 += per) go(j0, std::min(per, n - j0));
}

int hub_wide(int64_t ncols, int64_t nlong) { return hub_ranges(ncols) > 64 && nlong >= 8192 ? 64 : 16; }

template <int SW>
static void launch_hub_count_wide(const HubWork& h, const Mat& A, const Mat& B, int64_t* nnz, hipStream_t s) {
  constexpr int NT = 512;
  const int nrng = hub_ranges(B.ncols), nwin = (nrng + SW - 1) / SW;
  row_groups(h.n, nwin, NT, [&](int64_t j0, int64_t nj) {
    hipLaunchKernelGGL((k_hub_count<NT, SW, false>), dim3((unsigned)(nj * nwin)), dim3(NT), 0, s, h.rows + j0, nullptr,
                       nwin, nrng, A.ptr, B.idx, (const HubRec*)h.recs, h.hcnt + j0, h.lcnt + j0, h.span + 2 * j0,
                       B.band, B.nb1, h.slot, h.rng_cnt + j0 * nrng, nnz);
  });
}

void launch_hub_count(const HubWork& h, const Mat& A, const Mat& B, int64_t* nnz, hipStream_t s) {
  if (h.n <= 0) return;
  constexpr int NTF = 1024;
  const int nrng = hub_ranges(B.ncols);
  launch_fill_i32(h.rng_cnt, h.n * nrng, 0, s);
  if (h.nfine < h.n) {
    if (h.wide == 64) launch_hub_count_wide<64>(h, A, B, nnz, s);
    else launch_hub_count_wide<16>(h, A, B, nnz, s);
  }
  row_groups(h.nfine, nrng, NTF, [&](int64_t j0, int64_t nj) {
    hipLaunchKernelGGL((k_hub_count<NTF, 1, true>), dim3((unsigned)(nj * nrng)), dim3(NTF), 0, s, h.rows, h.fine + j0,
                       nrng, nrng, A.ptr, B.idx, (const HubRec*)h.recs, h.hcnt, h.lcnt, h.span, B.band, B.nb1, h.slot,
                       h.rng_cnt, nnz);
  });
}

// Bucket capacity check of the hub path inside a captured pipeline: more short products than the
// buckets hold flags the capacity bit, on which the bucket and range kernels write nothing.
__global__ void k_hub_guard(const int64_t* __restrict__ total, int64_t cap, int* __restrict__ err) {
  if (*total > cap) atomicOr(err, kErrCapacity);
}

void launch_hub_guard(const int64_t* total, int64_t cap, int* err, hipStream_t s) {
  hipLaunchKernelGGL(k_hub_guard, dim3(1), dim3(1), 0, s, total, cap, err);
}

template <typename V>
static void launch_hub_bucket_t(bool write, const HubWork& h, const int32_t* rows, int64_t n, const Mat& A, const Mat& B,
                                int64_t* scnt, const int64_t* soff, int32_t* scol, V* sval, const int* err,
                                hipStream_t s) {
  const int nrng = hub_ranges(B.ncols);
  const size_t lds = (size_t)nrng * sizeof(unsigned long long);
  const dim3 gr((unsigned)(A.nnz / kHubBucketChunk + n));  // a row has at most one partly filled chunk
  const V *Av = (const V*)A.val, *Bv = (const V*)B.val;
  if (write)
    hipLaunchKernelGGL((k_hub_bucket<V, true>), gr, dim3(256), lds, s, rows, n, h.boff, A.ptr, Av, B.idx, Bv,
                       (const HubRec*)h.recs, h.slot, h.lcnt, nrng, scnt, soff, scol, sval, err);
  else
    hipLaunchKernelGGL((k_hub_bucket<V, false>), gr, dim3(256), lds, s, rows, n, h.boff, A.ptr, Av, B.idx, Bv,
                       (const HubRec*)h.recs, h.slot, h.lcnt, nrng, scnt, soff, scol, sval, err);
}

void launch_hub_bucket_count(const HubWork& h, const int32_t* rows, int64_t n, const Mat& A, const Mat& B,
                             int64_t* scnt, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_hub_bucket_chunks, dim3(fill_grid(n)), dim3(256), 0, s, rows, n, h.slot, h.lcnt, h.boff);
  launch_exclusive_scan(h.boff, h.boff, n, h.tmp, s);
  launch_fill_i64(scnt, n * hub_ranges(B.ncols), 0, s);
  launch_hub_bucket_t<float>(false, h, rows, n, A, B, scnt, nullptr, nullptr, nullptr, nullptr, s);
}

void launch_hub_bucket_fill(int dtype, const HubWork& h, const int32_t* rows, int64_t n, const Mat& A, const Mat& B,
                            int64_t* scnt, const int64_t* soff, int32_t* scol, void* sval, const int* err,
                            hipStream_t s) {
  if (n <= 0) return;
  if (dtype == 1)
    launch_hub_bucket_t<double>(true, h, rows, n, A, B, scnt, soff, scol, (double*)sval, err, s);
  else
    launch_hub_bucket_t<float>(true, h, rows, n, A, B, scnt, soff, scol, (float*)sval, err, s);
}

// One workgroup per (row, range) item, rows in groups with their slices of the per-row and per-item
// arrays.
template <typename V>
static void launch_hub_range_t(const HubWork& h, int64_t nh, const Mat& A, const Mat& B, const int64_t* soff,
                               const int32_t* scol, const V* sval, const int64_t* roff, int32_t* Cidx, V* Cval, int* err,
                               hipStream_t s) {
  const int nrng = hub_ranges(B.ncols);
  auto run = [&](auto* kernel, int NT) {
    row_groups(nh, nrng, NT, [&](int64_t j0, int64_t nj) {
      const int64_t i0 = j0 * nrng;
      hipLaunchKernelGGL(kernel, dim3((unsigned)(nj * nrng)), dim3(NT), 0, s, (const HubRow*)h.info + j0, nrng,
                         (const V*)A.val, B.idx, (const V*)B.val, B.band, B.nb1, (const HubRec*)h.recs,
                         soff ? soff + i0 : nullptr, scol, sval, roff + i0, Cidx, Cval, err);
    });
  };
  if (B.nnz <= INT32_MAX) run(k_hub_range<V, 1024, int32_t>, 1024);
  else run(k_hub_range<V, 512, int64_t>, 512);
}

void launch_hub_range(int dtype, const HubWork& h, int64_t nh, const Mat& A, const Mat& B, const int64_t* soff,
                      const int32_t* scol, const void* sval, const int64_t* roff, int32_t* Cidx, void* Cval, int* err,
                      hipStream_t s) {
  if (nh <= 0) return;
  if (dtype == 1)
    launch_hub_range_t<double>(h, nh, A, B, soff, scol, (const double*)sval, roff, Cidx, (double*)Cval, err, s);
  else
    launch_hub_range_t<float>(h, nh, A, B, soff, scol, (const float*)sval, roff, Cidx, (float*)Cval, err, s);
}

template <typename V>
static void launch_backward_t(const KernelShape& k, const int32_t* rows, const int64_t* pbeg, const int64_t* pend,
                              int64_t nrows_hint, int grid, const Mat& A, const Mat& B, const int64_t* Cptr,
                              const int32_t* Cidx, const V* dC, V* dA, V* dB, int64_t db_stride, int64_t* cursor, int* err,
                              hipStream_t s) {
  const int gpb = symbolic_groups_per_wg(k);
  const V* Av = (const V*)A.val;
  const V* Bv = (const V*)B.val;
  if ((k.T == 0 || k.T >= kRankSlots) && B.ncols <= kRankBW) {  // figures: k_backward_rank
    constexpr int VC = 57344 / sizeof(V);
    hipLaunchKernelGGL((k_backward_rank<V, kRankNT, VC, kRankBW>), dim3(grid_for(nrows_hint, 1, grid)), dim3(kRankNT), 0, s,
                       rows, pbeg, pend, A.ptr, A.bstart, A.blen, Av, B.idx, Bv, Cptr, Cidx, dC, dA, dB, db_stride, err, k.T != 0);
    return;
  }
  if (k.T == 0 || k.T == kHubShape) {  // long and hub rows: windows over the C row
    const dim3 gr(grid_for(nrows_hint, gpb, grid));
    constexpr int W = sizeof(V) == 8 ? kBwdLongW64 : kBwdLongW32;
    hipLaunchKernelGGL((k_backward_long<V, kLongNT, W, kLongG>), gr, dim3(kLongNT), 0, s, rows, pbeg, pend, A.ptr,
                       A.idx, Av, B.ptr, B.idx, Bv, Cptr, Cidx, dC, dA, dB, db_stride, cursor, err);
    return;
  }
#define X(T_, NT_)                                                                                              \
  if (k.T == T_ && k.NT == NT_) {                                                                               \
    const dim3 gr(grid_for(nrows_hint, gpb, grid, (const void*)k_backward_hash<V, T_, NT_>, wg_of<NT_>()));     \
    hipLaunchKernelGGL((k_backward_hash<V, T_, NT_>), gr, dim3(wg_of<NT_>()), 0, s, rows, pbeg, pend, A.ptr,    \
                       A.bstart, A.blen, Av, B.idx, Bv, Cptr, Cidx, dC, dA, dB, db_stride, err);                           \
    return;                                                                                                     \
  }
  X(64, 64)
  X(128, 64)
  X(256, 64)
  X(512, 64)
  X(1024, 128)
  X(2048, 256)
  X(4096, 512)
  X(8192, 1024)
#undef X
}

void launch_backward(int dtype, const KernelShape& k, const int32_t* rows, const int64_t* pbeg, const int64_t* pend,
                     int64_t nrows_hint, int grid, const Mat& A, const Mat& B, const int64_t* Cptr,
                     const int32_t* Cidx, const void* dC, void* dA, void* dB, int64_t db_stride, int64_t* cursor, int* err,
                     hipStream_t s) {
  if (dtype == 1)
    launch_backward_t<double>(k, rows, pbeg, pend, nrows_hint, grid, A, B, Cptr, Cidx, (const double*)dC,
                              (double*)dA, (double*)dB, db_stride, cursor, err, s);
  else
    launch_backward_t<float>(k, rows, pbeg, pend, nrows_hint, grid, A, B, Cptr, Cidx, (const float*)dC,
                             (float*)dA, (float*)dB, db_stride, cursor, err, s);
}

// Ranges per window of the hub rows' backward kernel for B of this width, 0: the window kernel takes
// them. Up to kHubWhole ranges one (FP64: two workgroups per CU); beyond, all of a CU's LDS, as long
// as no more than 16 windows read the short entries (R-MAT 18: 8 windows FP32, 16 FP64).
int hub_backward_ranges(int dtype, int64_t ncols) {
  const int nrng = hub_ranges(ncols), big = dtype == 1 ? 2 : 4;
  return nrng <= kHubWhole ? 1 : (nrng + big - 1) / big <= 16 ? big : 0;
}

template <typename V, int NT, int SR>
static void launch_hub_backward_t(const HubWork& h, int64_t n, const Mat& A, const Mat& B, const int64_t* roff,
                                  const int32_t* Cidx, const V* dC, V* dA, V* dB, int64_t db_stride, int* err,
                                  hipStream_t s) {
  const int nrng = hub_ranges(B.ncols), nwin = (nrng + SR - 1) / SR;
  row_groups(n, nwin, NT, [&](int64_t j0, int64_t nj) {
    hipLaunchKernelGGL((k_hub_backward<V, NT, SR>), dim3((unsigned)(nj * nwin)), dim3(NT), 0, s, (const HubRow*)h.info + j0,
                       nrng, nwin, (const V*)A.val, B.idx, (const V*)B.val, B.band, B.nb1, (const HubRec*)h.recs,
                       roff + j0 * nrng, Cidx, dC, dA, dB, db_stride, err);
  });
}

void launch_hub_backward(int dtype, const HubWork& h, int64_t n, const Mat& A, const Mat& B, const int64_t* roff,
                         const int32_t* Cidx, const void* dC, void* dA, void* dB, int64_t db_stride, int* err,
                         hipStream_t s) {
  if (n <= 0) return;
  const bool one = hub_backward_ranges(dtype, B.ncols) == 1;
  if (dtype == 1) {
    if (one)
      launch_hub_backward_t<double, 512, 1>(h, n, A, B, roff, Cidx, (const double*)dC, (double*)dA, (double*)dB, db_stride,
                                             err, s);
    else
      launch_hub_backward_t<double, 1024, 2>(h, n, A, B, roff, Cidx, (const double*)dC, (double*)dA, (double*)dB, db_stride,
                                             err, s);
  } else {
    if (one)
      launch_hub_backward_t<float, 512, 1>(h, n, A, B, roff, Cidx, (const float*)dC, (float*)dA, (float*)dB, db_stride, err,
                                            s);
    else
      launch_hub_backward_t<float, 1024, 4>(h, n, A, B, roff, Cidx, (const float*)dC, (float*)dA, (float*)dB, db_stride, err,
                                            s);
  }
}

bool shape_available(int phase, const KernelShape& k) {
  if (k.T == 0 || k.T == kHubShape) return true;
  if (k.G != 16 && k.G != 64) return false;
  if (k.G > k.NT) return false;
  const int T = k.T, NT = k.NT;
  const bool base = (T == 64 && NT == 64) || (T == 128 && NT == 64) || (T == 256 && NT == 64) ||
                    (T == 512 && NT == 64) || (T == 1024 && NT == 128) || (T == 2048 && NT == 256) ||
                    (T == 4096 && NT == 512) || (T == 8192 && NT == 1024);
  if (base) return true;
  return phase == 0 && ((T == 16384 && NT == 1024) || (T == 8192 && NT == 512) || (T == 4096 && NT == 256) ||
                        (T == 2048 && NT == 64) || (T == 1024 && NT == 64));
}

}  // namespace dbd
