// Wave64 helpers shared by the graph kernels.
#pragma once
#include <hip/hip_runtime.h>
#include "gdb_discovery.hpp"

namespace gdb {

__device__ __forceinline__ int lane_id() { return (int)__lane_id(); }

// Value of `v` in lane `src` (wave-uniform) for every lane: a scalar read of
// the register, no LDS round trip.
__device__ __forceinline__ int bcast(int v, int src) { return __builtin_amdgcn_readlane(v, src); }

// Wave-wide max over the active lanes, by DPP row shifts (no LDS round
// trips), from the device library.
extern "C" __device__ int __ockl_wfred_max_i32(int);
__device__ __forceinline__ int wave_max(int v) { return __ockl_wfred_max_i32(v); }

__device__ __forceinline__ float shfl_xor(float x, int o) { return __shfl_xor(x, o, 64); }
__device__ __forceinline__ int shfl_xor(int x, int o) { return __shfl_xor(x, o, 64); }
__device__ __forceinline__ unsigned shfl_xor(unsigned x, int o) {
  return (unsigned)__shfl_xor((int)x, o, 64);
}
__device__ __forceinline__ unsigned long long shfl_xor(unsigned long long x, int o) {
  return __shfl_xor(x, o, 64);
}

// Global-address-space accessors.  Graph arrays reach the kernels through
// structs, so the compiler sees generic pointers and emits flat instructions,
// whose waits also cover LDS traffic; these keep the accesses global_*.
template <typename T>
__device__ __forceinline__ T ldg(const T* p) {
  return *(const __attribute__((address_space(1))) T*)p;
}
__device__ __forceinline__ int ld_rlx_g(const int* p) {  // agent scope, relaxed
  return __hip_atomic_load((const __attribute__((address_space(1))) int*)p, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned atomic_min_g(unsigned* p, unsigned v) {
  return __hip_atomic_fetch_min((__attribute__((address_space(1))) unsigned*)p, v, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long atomic_min_g(unsigned long long* p, unsigned long long v) {
  return __hip_atomic_fetch_min((__attribute__((address_space(1))) unsigned long long*)p, v, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int atomic_or_g(int* p, int v) {
  return __hip_atomic_fetch_or((__attribute__((address_space(1))) int*)p, v, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int atomic_max_g(int* p, int v) {
  return __hip_atomic_fetch_max((__attribute__((address_space(1))) int*)p, v, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned atomic_cas_g(unsigned* p, unsigned expected, unsigned desired) {
  __hip_atomic_compare_exchange_strong((__attribute__((address_space(1))) unsigned*)p, &expected, desired,
                                       __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return expected;
}
__device__ __forceinline__ int atomic_cas_g(int* p, int expected, int desired) {
  __hip_atomic_compare_exchange_strong((__attribute__((address_space(1))) int*)p, &expected, desired,
                                       __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return expected;
}

struct MaxFound {  // running max plus "at least one candidate seen"
  float mx;
  int found;
};
__device__ __forceinline__ MaxFound shfl_xor(MaxFound x, int o) {
  return MaxFound{__shfl_xor(x.mx, o, 64), __shfl_xor(x.found, o, 64)};
}
struct MaxAt {  // running max and the candidate holding it (at = -1: none seen)
  float mx;
  int at;
};
__device__ __forceinline__ MaxAt shfl_xor(MaxAt x, int o) {
  return MaxAt{__shfl_xor(x.mx, o, 64), __shfl_xor(x.at, o, 64)};
}

// Thread / wave cooperative reduction over the edge ranges [b, e) held by
// the lanes of one wave.  Lanes whose range is at most `serial_limit` edges
// walk it alone; longer ranges are walked by the whole wave (64 consecutive
// edges per step, coalesced) and reduced with xor-shuffles.  `edge(k)` maps
// an edge index to a value, `red` combines two values.  All 64 lanes must
// call this (wave-uniform control flow).
template <typename T, typename EdgeFn, typename RedFn>
__device__ __forceinline__ T wave_coop_reduce(bool active, int b, int e, T identity, EdgeFn edge,
                                              RedFn red, int serial_limit) {
  T acc = identity;
  const bool heavy = active && (e - b) > serial_limit;
  // Unrolled so that the loads of several edges are in flight together.
  if (active && !heavy) {
#pragma unroll 4
    for (int k = b; k < e; ++k) acc = red(acc, edge(k));
  }
  unsigned long long mask = __ballot(heavy);
  const int lane = lane_id();
  while (mask) {
    const int leader = __ffsll((long long)mask) - 1;
    const int lb = bcast(b, leader);
    const int le = bcast(e, leader);
    T part = identity;
#pragma unroll 4
    for (int k = lb + lane; k < le; k += 64) part = red(part, edge(k));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) part = red(part, shfl_xor(part, off));
    if (lane == leader) acc = part;
    mask &= mask - 1;
  }
  return acc;
}

// Thread / wave cooperative walk over the edge ranges [b, e) of the lanes of
// one wave, calling fn(k, valid, payload) in wave-uniform steps so that fn
// may use wave collectives (ballot-based queue pushes).  `payload` is the
// value the range's owner lane passed in (for example its vertex's distance):
// a lane walking another lane's range sees the owner's payload.  Short ranges
// are walked by their own lane (trip count = the longest short range in the
// wave); long ranges by all 64 lanes, 64 consecutive edges per step.  Lanes
// without an edge in a step get valid = false.
template <typename F>
__device__ __forceinline__ void wave_coop_foreach(bool active, int b, int e, unsigned payload, F fn,
                                                  int serial_limit) {
  const bool heavy = active && (e - b) > serial_limit;
  int len = (active && !heavy) ? (e - b) : 0;
  const int maxlen = wave_max(len);
  for (int t = 0; t < maxlen; ++t) fn(b + t, t < len, payload);
  unsigned long long mask = __ballot(heavy);
  const int lane = lane_id();
  while (mask) {
    const int leader = __ffsll((long long)mask) - 1;
    const int lb = bcast(b, leader);
    const int le = bcast(e, leader);
    const unsigned lp = (unsigned)bcast((int)payload, leader);
    for (int base = lb; base < le; base += 64) fn(base + lane, base + lane < le, lp);
    mask &= mask - 1;
  }
}

// Wave cooperative "some edge k in [b, e) has pred(k)" with early exit:
// short ranges are scanned by their own lane up to the first hit, long ones
// by the whole wave, 64 consecutive edges per step, up to the first step
// with a hit.  All 64 lanes must call it.
template <typename P>
__device__ __forceinline__ bool wave_coop_any(bool active, int b, int e, P pred, int serial_limit) {
  const bool heavy = active && (e - b) > serial_limit;
  bool found = false;
  if (active && !heavy)
    for (int k = b; k < e; ++k)
      if (pred(k)) {
        found = true;
        break;
      }
  unsigned long long mask = __ballot(heavy);
  const int lane = lane_id();
  while (mask) {
    const int leader = __ffsll((long long)mask) - 1;
    const int lb = bcast(b, leader);
    const int le = bcast(e, leader);
    bool hit = false;
    for (int base = lb; base < le; base += 64) {
      const bool h = base + lane < le && pred(base + lane);
      if (__ballot(h) != 0ull) {
        hit = true;
        break;
      }
    }
    if (lane == leader) found = hit;
    mask &= mask - 1;
  }
  return found;
}

// Appends `item` for every lane with push == true to queue[*tail ...]:
// one atomic per wave.  Returns nothing; all 64 lanes must call it.
__device__ __forceinline__ void wave_push(bool push, int item, int* queue, int* tail) {
  const unsigned long long m = __ballot(push);
  if (m == 0ull) return;
  const int lane = lane_id();
  int base = 0;
  if (lane == __ffsll((long long)m) - 1) base = fadd_rlx(tail, __popcll(m));
  base = bcast(base, __ffsll((long long)m) - 1);
  if (push) queue[base + __popcll(m & ((1ull << lane) - 1ull))] = item;
}

// Appends the items of N push slots of every lane with one atomic per wave.
template <int N>
__device__ __forceinline__ void wave_push_n(const bool (&push)[N], const int (&item)[N], int* queue,
                                            int* tail) {
  unsigned long long m[N];
  int cnt = 0;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    m[j] = __ballot(push[j]);
    cnt += __popcll(m[j]);
  }
  if (cnt == 0) return;
  const int lane = lane_id();
  int base = 0;
  if (lane == 0) base = fadd_rlx(tail, cnt);
  base = bcast(base, 0);
  const unsigned long long lt = (1ull << lane) - 1ull;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (push[j]) queue[base + __popcll(m[j] & lt)] = item[j];
    base += __popcll(m[j]);
  }
}

// Queue pushes staged in LDS.  One returning atomic on a queue's size per wave
// step serialises at about 8 ns each; a group that stages its pushes reserves
// space for a batch of them at once.  wave_stage_n appends the items of N push
// slots of every lane to the stage (what does not fit goes straight to the
// queue); group_flush, called by all threads of the group, moves the staged items
// to the queue when more than `above` wait.  It holds two to three barriers of the
// group: a loop calls it between its trips, and once at its end.
struct PushStage {
  int* items;  // LDS, `cap` entries
  int* count;  // LDS, zeroed before the first use
  int* base;   // LDS
  int cap;
};
template <int N>
__device__ __forceinline__ void wave_stage_n(const PushStage& st, bool (&push)[N], const int (&item)[N], int* queue,
                                             int* tail) {
  unsigned long long m[N];
  int cnt = 0;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    m[j] = __ballot(push[j]);
    cnt += __popcll(m[j]);
  }
  if (cnt == 0) return;
  const int lane = lane_id();
  int base = 0;
  if (lane == 0) base = atomicAdd(st.count, cnt);
  base = bcast(base, 0);
  const bool full = base + cnt > st.cap;
  const unsigned long long lt = (1ull << lane) - 1ull;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int pos = base + __popcll(m[j] & lt);
    if (push[j] && pos < st.cap) {
      st.items[pos] = item[j];
      push[j] = false;
    }
    base += __popcll(m[j]);
  }
  if (full) wave_push_n<N>(push, item, queue, tail);
}
// With `row`, the edges of the moved vertices are added to *sum (LDS) while the
// queue's reply is on its way.
__device__ __forceinline__ void group_flush(const PushStage& st, int above, int* queue, int* tail, const int* row,
                                            int* sum) {
  __syncthreads();
  const int c = *st.count < st.cap ? *st.count : st.cap;
  if (c <= above) {
    __syncthreads();  // every wave has read the count before the next push
    return;
  }
  int at = 0;
  if (threadIdx.x == 0) at = fadd_rlx(tail, c);
  if (row) {
    int d = 0;
    for (int i = threadIdx.x; i < c; i += blockDim.x) d += row[st.items[i] + 1] - row[st.items[i]];
    for (int off = 32; off > 0; off >>= 1) d += __shfl_xor(d, off, 64);
    if (lane_id() == 0 && d) atomicAdd(sum, d);
  }
  if (threadIdx.x == 0) *st.base = at;
  __syncthreads();
  if (threadIdx.x == 0) *st.count = 0;
  for (int i = threadIdx.x; i < c; i += blockDim.x) queue[*st.base + i] = st.items[i];
  __syncthreads();
}

// Traversal steps with more edges out of their queue than this mark what they reach
// by plain stores and collect it in a sweep over all vertices; steps with fewer
// claim each vertex by an atomic.  Claims bound the large steps: plain loads stay
// stale until the next barrier, so nearly every edge to a vertex not reached before
// the step sends one, up to 20 ps each.  A sweep costs a barrier and a few bytes
// per vertex, about 10 us and n / 0.5 ns.  (Lines from 50000 + n / 8 to 400000 + n /
// 12 measured within 3% of each other in BFS and BC.)
__host__ __device__ inline int sweep_line(int n) { return 100000 + n / 16; }

// Wave-wide OR of a predicate.
__device__ __forceinline__ bool wave_any(bool p) { return __ballot(p) != 0ull; }

// Whether a lane has any edge slot in a walk step (lanes without one can
// skip the step's loads).
template <int N>
__device__ __forceinline__ bool any_slot(const bool (&ok)[N]) {
  bool a = false;
#pragma unroll
  for (int j = 0; j < N; ++j) a |= ok[j];
  return a;
}

// Chunked cooperative walk over the edge ranges [b, e) of the lanes of one
// wave: step(ok, kk) handles N edge slots of the calling lane at once (slot j
// is edge kk[j] when ok[j]) and returns the lane's contribution; it is called
// in wave-uniform steps, so it may use wave collectives, and it should issue
// the slots' loads and atomics branch-free, all loads before any use, so that
// the N slots cost one chain of memory round trips.  Short ranges are walked
// by their own lane N edges per step; long ranges by the whole wave, N x 64
// consecutive edges per step (slot j of lane i takes edge base + i + 64 j, so
// each slot's loads are coalesced), and reduced into the owner lane.  Ranges of at
// most 16 N edges, still long, are walked four at a time, 16 lanes each: one such
// row on the whole wave leaves most slots empty and costs the same chain of trips
// (BC on directed R-MAT 15 0.45 -> 0.40 ms, on R-MAT 22 23.4 -> 21.7; pull SSSP R-MAT
// 16 0.44 -> 0.41; BFS R-MAT 20 0.42 -> 0.40; MST R-MAT 18 0.59 -> 0.575).  Which way a
// range is walked depends on its length alone, and so does the order of its sum.
// As wave_walk_n, but step(ok, kk, owner) also gets the `payload` of the
// range's owner lane (for a long row walked by the whole wave, the leader's
// payload on every lane).  SHORT: the caller's ranges are all short, and the long
// walks' code and registers stay out (colouring by rounds, R-MAT 19: 305 ms, 323 with
// them).
template <int N, bool SHORT = false, typename T, typename Step, typename R>
__device__ __forceinline__ T wave_walk_np(bool active, int b, int e, int payload, T identity, Step step, R red,
                                          int serial_limit) {
  const bool heavy = active && (e - b) > serial_limit;
  const int len = (active && !heavy) ? (e - b) : 0;
  const int maxlen = wave_max(len);
  T acc = identity;
  for (int c = 0; c < maxlen; c += N) {
    bool ok[N];
    int kk[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      ok[j] = c + j < len;
      kk[j] = b + c + j;
    }
    acc = red(acc, step(ok, kk, payload));
  }
  if constexpr (SHORT) return acc;
  const int lane = lane_id();
  const bool mid = heavy && (e - b) <= 16 * N;
  unsigned long long mask = __ballot(mid);
  while (mask) {
    int owner[4];  // the owners of this trip's ranges, -1 none
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      owner[q] = mask ? __ffsll((long long)mask) - 1 : -1;
      mask &= mask - 1;
    }
    const int mine = lane < 32 ? (lane < 16 ? owner[0] : owner[1]) : (lane < 48 ? owner[2] : owner[3]);
    const int from = mine < 0 ? 0 : mine;
    const int lb = __shfl(b, from, 64), le = __shfl(e, from, 64), lp = __shfl(payload, from, 64);
    bool ok[N];
    int kk[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      kk[j] = lb + (lane & 15) + 16 * j;
      ok[j] = mine >= 0 && kk[j] < le;
    }
    T part = red(identity, step(ok, kk, lp));
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) part = red(part, shfl_xor(part, off));
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      T x = (lane >> 4) == q ? part : identity;
      x = red(x, shfl_xor(x, 16));
      x = red(x, shfl_xor(x, 32));
      if (lane == owner[q]) acc = x;
    }
  }
  mask = __ballot(heavy && !mid);
  while (mask) {
    const int leader = __ffsll((long long)mask) - 1;
    const int lb = bcast(b, leader);
    const int le = bcast(e, leader);
    const int lp = bcast(payload, leader);
    T part = identity;
    for (int base = lb; base < le; base += 64 * N) {
      bool ok[N];
      int kk[N];
#pragma unroll
      for (int j = 0; j < N; ++j) {
        kk[j] = base + lane + 64 * j;
        ok[j] = kk[j] < le;
      }
      part = red(part, step(ok, kk, lp));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) part = red(part, shfl_xor(part, off));
    if (lane == leader) acc = part;
    mask &= mask - 1;
  }
  return acc;
}

// Chunked cooperative "some edge of [b, e) has pred" with early exit:
// step(ok, kk, owner) tests N edge slots of the calling lane at once (the
// same slot layout and payload as wave_walk_np) and returns whether one of
// them hit.  A lane walks the first serial_limit edges of its own range, long or
// short, and stops at its first step with a hit: most ranges end there (in MIS,
// nine of ten within eight edges, whatever their length).  What is left of a
// long one is walked by the whole wave up to the first step in which some lane
// hit.  All 64 lanes must call it.
template <int N, typename Step>
__device__ __forceinline__ bool wave_walk_any(bool active, int b, int e, int payload, Step step,
                                              int serial_limit) {
  const bool is_long = active && (e - b) > serial_limit;
  const int len = !active ? 0 : is_long ? serial_limit : e - b;
  bool found = false;
  for (int c = 0; __ballot(c < len && !found) != 0ull; c += N) {
    bool ok[N];
    int kk[N];
    const bool live = c < len && !found;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      ok[j] = live && c + j < len;
      kk[j] = b + c + j;
    }
    found |= step(ok, kk, payload);
  }
  b += serial_limit;
  unsigned long long mask = __ballot(is_long && !found);
  const int lane = lane_id();
  while (mask) {
    const int leader = __ffsll((long long)mask) - 1;
    const int lb = bcast(b, leader);
    const int le = bcast(e, leader);
    const int lp = bcast(payload, leader);
    bool hit = false;
    for (int base = lb; base < le; base += 64 * N) {
      bool ok[N];
      int kk[N];
#pragma unroll
      for (int j = 0; j < N; ++j) {
        kk[j] = base + lane + 64 * j;
        ok[j] = kk[j] < le;
      }
      if (__ballot(step(ok, kk, lp)) != 0ull) {
        hit = true;
        break;
      }
    }
    if (lane == leader) found = hit;
    mask &= mask - 1;
  }
  return found;
}

template <int N, bool SHORT = false, typename T, typename Step, typename R>
__device__ __forceinline__ T wave_walk_n(bool active, int b, int e, T identity, Step step, R red,
                                         int serial_limit) {
  return wave_walk_np<N, SHORT>(
      active, b, e, 0, identity, [&](const bool (&ok)[N], const int (&kk)[N], int) { return step(ok, kk); }, red,
      serial_limit);
}

// Uniform-trip grid-stride loop over [0, n): every thread of a group runs
// the same number of iterations (i may be >= n in the last one), so the body
// may use wave- and group-wide collectives.
#define GDB_FOR_UNIFORM(i, valid, start, stride, n)                             \
  for (long long _base = (long long)(start) - (long long)threadIdx.x;           \
       _base < (long long)(n); _base += (long long)(stride))                      \
    for (int _once = 1, i = (int)(_base + threadIdx.x),                          \
             valid = (_base + (long long)threadIdx.x) < (long long)(n);          \
         _once; _once = 0)

// The same trips over the items [0, n), dealt to the waves 2^SH at a time
// (SH 0 to 6) instead of 64 at a time, in another order for each of a wave's
// shares.  A wave walks its long rows one after the other, so neighbouring
// items are better spread: in a queue shorter than the grid some waves would
// walk 64 rows and the others none, and in a skewed graph long rows are
// neighbours, or, as in an R-MAT graph, share low bits of their ids (dealt in
// a fixed order, a wave would get all of one residue).  Measured: R-MAT 22 BC
// of 16 sources 86 -> 33 ms, R-MAT 18 SSSP 1.4 -> 0.97 (queues); R-MAT 18 MST
// 0.93 -> 0.63, R-MAT 16 pull SSSP 0.69 -> 0.43 (all vertices, where a fixed
// order gained nothing).  SH = 6 keeps a wave's 64 items together: short rows,
// whose words it then reads in one line.
__device__ __forceinline__ long long spread_item(int start, int stride, int sh) {
  if (sh == 6) return start;  // what the rest comes to, without its division
  const unsigned waves = (unsigned)stride >> 6, l = (unsigned)lane_id(), share = l >> sh;
  const unsigned turn = (waves * 5u / 8u) | 1u;
  return (((long long)share * waves + ((unsigned)start / 64u + share * turn) % waves) << sh) + (l & ((1u << sh) - 1u));
}
#define GDB_FOR_SPREAD(i, valid, start, stride, n, SH)                          \
  for (long long _base = 0, _at = gdb::spread_item((start), (stride), (SH)); _base < (long long)(n); \
       _base += (long long)(stride))                                            \
    for (int _once = 1, i = (int)(_base + _at), valid = _base + _at < (long long)(n); _once; _once = 0)
// SH of a loop over all vertices of a graph of n vertices and m edges: one by
// one where rows are long enough to be walked by waves (four or eight at a time
// measured 2 to 25% slower on R-MAT graphs), 64 together where they are short
// (2^20-vertex grid MST 1.16 ms against 1.44).
__host__ __device__ inline int spread_rows(int n, long long m) { return m >= 8LL * n ? 0 : 6; }
// The same for a step over `items` queued vertices.  Where all rows are short (`even`:
// six edges a vertex at most, no row of more than kEvenRow) a wave takes 16 neighbours
// in a step of up to 1024, and 64 in one of up to 256: the fewer groups have work, the
// fewer come late to the barrier.  One by one against this: BFS of a 100^2 grid of
// shuffled ids 0.84 -> 0.76 ms, BC of it, 11 sources, 6.6 -> 5.8.  Longer steps fill the
// waves one by one (64 always: SSSP of a shuffled 500^2 grid 7.9 -> 13.4 ms), and so do
// rows of eight edges (SSSP of G(3000) of degree 8 216 us, 228 by 16).
constexpr int kEvenRow = 64;
__host__ __device__ inline bool even_rows(int n, long long m, bool long_row) { return m <= 6LL * n && !long_row; }
__host__ __device__ inline int spread_queue(bool even, int items) { return !even || items > 1024 ? 0 : items <= 256 ? 6 : 4; }
// Whether such a step pushes straight to the queue.  Its pushes are few, and the
// barriers of the group that staging takes (group_flush) cost more than their atomics:
// BFS of a shuffled 500^2 grid 5.0 -> 4.3 ms (512 items: 4.8), of a 100^2 grid 0.75 ->
// 0.70; BC of the 300^2 grid 10.8 -> 10.3.
__host__ __device__ inline bool push_directly(bool even, int items) { return even && items <= 1024; }

}  // namespace gdb
