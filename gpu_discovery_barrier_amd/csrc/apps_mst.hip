// Minimum spanning forest (Boruvka) on the discovery protocol.
//
// Reference: lonestar mst (code/experiments/lonestar_gpu_opencl/apps/mst):
// per round every component finds its lightest cross-component edge
// (dfindelemin, dfindelemin2, verify_min_elem in kernel/mst_common.cl) and
// the chosen edges unify components (dfindcompmintwo, mst_port_kernel.cl,
// with discovery barriers inside a uniform-trip loop); the host repeats
// rounds while the component count falls (mst_port.cpp:203-313) and prints
// weight, components and edges.
//
// Here one persistent kernel runs every round.  A component's choice is the
// smallest key (weight, id of the component on the other side) over its
// cross edges, one 64-bit atomic min per vertex or wave.  With that order the
// choices form no cycle but pairs: in a longer cycle all weights are equal
// (each is at most the next), the component t that the cycle's smallest id s
// chose has s among its own lightest targets, so t chose s, and the cycle is
// the pair {s, t}.  The smaller id of a pair stays a root and the edge is
// counted once.  Per round, three barriers:
//   1  every vertex: smallest key of its cross edges -> best[comp]
//   2  every root with a choice: adds the edge's weight and points at the
//      other side; of a pair that chose each other the smaller id stays
//   3  every vertex follows parents to its new root (path halving)
// The weight of a minimum spanning forest is unique, so it and the
// component and edge counts are compared exactly.
//
// What bounds it: gathers of the neighbours' components, one walk of the
// edges per round.  Rows are walked kSlots edges per lane step, by their lane
// up to kSerialLimit edges, by a wave up to kLongRow, and longer ones in
// pieces of kLongRow edges spread over all waves (a skewed graph's longest row
// has as many edges as a thousand others); a vertex or piece without a cross
// edge never gets one again and is left out of later rounds.  R-MAT 18 (7.6 M
// edges, longest row 25 k): 0.58 ms (one lane walking each row twice per
// round, six barriers: 46.4 ms; vertices 64 at a time: 0.93).  Walking the rows of a wave as one list, with
// the minima in LDS, took 1.07 ms: the search for each edge's row costs more
// than the steps it saves.
#include <cstring>
#include "graph_common.hpp"
#include "runtime.hpp"

namespace {

typedef unsigned long long u64;
constexpr u64 kNoKey = ~0ull;
constexpr unsigned kNoW = 0xffffffffu;  // an edge of this weight is never chosen
constexpr int kSerialLimit = 16;
constexpr int kSlots = 4;
constexpr int kLongRow = 1024;

// Root of component c: follows parent pointers, halving the path (a pointer
// is only ever replaced by one of its ancestors, so racing walkers agree).
__device__ __forceinline__ int find_root(int* parent, int c, int n) {
  for (int guard = 0; guard < n; ++guard) {
    const int p = parent[c];
    if (p == c || (unsigned)p >= (unsigned)n) return c;
    const int gp = parent[p];
    if ((unsigned)gp < (unsigned)n && gp != p) parent[c] = gp;
    c = p;
  }
  return c;
}

// Lowers best[c] to key for every lane that holds one.  Lanes of the first
// such lane's component (all of them, once one component spans most of the
// graph) share one atomic; a key that is not below the current value sends
// none.
__device__ __forceinline__ void lower_best(u64* best, bool has, int c, u64 key) {
  const u64 mask = __ballot(has);
  if (!mask) return;
  const int leader = __ffsll((long long)mask) - 1;
  const bool same = has && c == gdb::bcast(c, leader);
  u64 k = same ? key : kNoKey;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const u64 o = __shfl_xor(k, off, 64);
    k = o < k ? o : k;
  }
  if (same) {
    has = gdb::lane_id() == leader;
    key = k;
  }
  if (has && key < __hip_atomic_load(&best[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    gdb::atomic_min_g(&best[c], key);
}

template <int WGS>
__global__ __launch_bounds__(WGS) void k_mst(gdb_kernel_ctx_t* ctx, const int* __restrict__ row,
                                             const int* __restrict__ col, const unsigned* __restrict__ w,
                                             int n, int* comp, int* parent, u64* best, unsigned char* dead,
                                             int2* pieces, int piece_cap, int* npieces, int* flags, u64* total,
                                             int* out) {
  DISCOVERY_PROTOCOL(ctx);
  const int tid = p_get_global_id(ctx, &local_ctx);
  const int stride = p_get_global_size(ctx, &local_ctx);
  const int lane = gdb::lane_id();
  const int wave = tid >> 6, nwaves = stride >> 6;
  const int spare = (int)((unsigned)tid % (unsigned)n);
  const int sh = gdb::spread_rows(n, row[n]);
  int rounds = 0, nbar = 0;
  u64 wsum = 0;
  int added = 0;
  for (int v = tid; v < n; v += stride) {
    comp[v] = v;
    parent[v] = v;
    best[v] = kNoKey;
    dead[v] = 0;
    const int b = row[v], e = row[v + 1];
    if (e - b > kLongRow) {
      const int k = (e - b + kLongRow - 1) / kLongRow;
      const int at = gdb::fadd_rlx(npieces, k);
      for (int j = 0; j < k && at + j < piece_cap; ++j) pieces[at + j] = make_int2(v, b + j * kLongRow);
    }
  }
  if (!discovery_barrier(ctx, &local_ctx)) return;
  ++nbar;
  const int np = min(gdb::ld_rlx(npieces), piece_cap);
  for (;;) {
    if (tid == 0) gdb::st_rlx(&flags[(rounds + 1) % 3], 0);
    const bool first = rounds == 0;  // every vertex is its own component
    auto step = [&](const bool (&ok)[kSlots], const int (&kk)[kSlots], int cv) -> u64 {
      if (!gdb::any_slot(ok)) return kNoKey;  // no slot: no loads
      int u[kSlots], cu[kSlots];
      unsigned wk[kSlots];
#pragma unroll
      for (int j = 0; j < kSlots; ++j) {
        const int k = ok[j] ? kk[j] : 0;  // edge 0 exists here
        u[j] = gdb::ldg(col + k);
        wk[j] = gdb::ldg(w + k);
      }
#pragma unroll
      for (int j = 0; j < kSlots; ++j) {
        const bool in = ok[j] && (unsigned)u[j] < (unsigned)n;
        if (!in) wk[j] = kNoW;
        cu[j] = first ? u[j] : gdb::ldg(comp + (in ? u[j] : spare));
      }
      u64 key = kNoKey;
#pragma unroll
      for (int j = 0; j < kSlots; ++j) {
        const u64 k = ((u64)wk[j] << 32) | (unsigned)cu[j];
        if (wk[j] != kNoW && cu[j] != cv && k < key) key = k;
      }
      return key;
    };
    auto least = [](u64 a, u64 c) { return a < c ? a : c; };
    // 1: rows of up to kLongRow edges, then the pieces of the longer ones.
    GDB_FOR_SPREAD(v, valid, tid, stride, n, sh) {
      int b = 0, e = 0, cv = 0;
      if (valid && !dead[v]) {
        cv = comp[v];
        b = row[v];
        e = row[v + 1];
        if (e - b > kLongRow) b = e;
      }
      const u64 key = gdb::wave_walk_np<kSlots>(e > b, b, e, cv, kNoKey, step, least, kSerialLimit);
      const bool has = key != kNoKey && (unsigned)cv < (unsigned)n;
      if (e > b && !has) dead[v] = 1;
      if (first) {
        if (has) best[v] = key;  // v's own word
      } else {
        lower_best(best, has, cv, key);
      }
    }
    for (int i = wave; i < np; i += nwaves) {
      const int2 pc = pieces[i];
      if (pc.x < 0) continue;  // no cross edge left
      const int e = min(row[pc.x + 1], pc.y + kLongRow), cv = comp[pc.x];
      u64 key = kNoKey;
      for (int base = pc.y; base < e; base += 64 * kSlots) {
        bool ok[kSlots];
        int kk[kSlots];
#pragma unroll
        for (int j = 0; j < kSlots; ++j) {
          kk[j] = base + lane + 64 * j;
          ok[j] = kk[j] < e;
        }
        key = least(key, step(ok, kk, cv));
      }
      if (__ballot(key != kNoKey) == 0) {
        if (lane == 0) pieces[i].x = -1;
      } else if ((unsigned)cv < (unsigned)n) {
        lower_best(best, key != kNoKey, cv, key);
      }
    }
    if (!discovery_barrier(ctx, &local_ctx)) return;
    ++nbar;
    // 2
    bool progress = false;
    for (int c = tid; c < n; c += stride) {
      if (comp[c] != c) continue;
      const u64 k = best[c];
      if (k == kNoKey) continue;
      const int p = (int)(unsigned)k;
      if ((unsigned)p >= (unsigned)n) continue;
      if (best[p] != kNoKey && (int)(unsigned)best[p] == c && c < p) continue;  // the pair's root; p counts the edge
      parent[c] = p;
      wsum += k >> 32;
      ++added;
      progress = true;
    }
    if (gdb::wave_any(progress) && lane == 0) gdb::st_rlx(&flags[rounds % 3], 1);
    if (!discovery_barrier(ctx, &local_ctx)) return;
    ++nbar;
    // 3
    for (int v = tid; v < n; v += stride) {
      const int c = comp[v];
      if (best[v] != kNoKey) best[v] = kNoKey;
      if ((unsigned)c < (unsigned)n) {
        const int r = find_root(parent, c, n);
        if (r != c) comp[v] = r;
      }
    }
    if (!discovery_barrier(ctx, &local_ctx)) return;
    ++nbar;
    ++rounds;
    if (gdb::ld_rlx(&flags[(rounds - 1) % 3]) == 0) break;
    if (rounds > 64) {  // each round at least halves the components with a cross edge
      gdb::set_error(ctx, GDB_ERR_QUEUE_OVERFLOW);
      break;
    }
  }
  // Totals: one atomic per wave.
  u64 ws = wsum;
  int ad = added, roots = 0;
  for (int v = tid; v < n; v += stride) roots += comp[v] == v;
  for (int off = 32; off > 0; off >>= 1) {
    ws += __shfl_xor(ws, off, 64);
    ad += __shfl_xor(ad, off, 64);
    roots += __shfl_xor(roots, off, 64);
  }
  if (lane == 0) {
    if (ws) atomicAdd(total, ws);
    if (ad) atomicAdd(&out[2], ad);
    if (roots) atomicAdd(&out[3], roots);
  }
  if (tid == 0) {
    out[0] = rounds;
    out[1] = nbar;
  }
}

}  // namespace

using namespace gdbrt;

extern "C" int gdb_mst(gdb_ctx* ctx, int n, int m, const int* row, const int* col, const unsigned* w,
                       unsigned long long* weight, int* edges, int* components, const gdb_opts* opts,
                       gdb_stats* stats) {
  if (!ctx || n < 0 || m < 0 || (n > 0 && !row) || (m > 0 && (!col || !w))) return GDB_E_INVALID;
  gdb_opts o{};
  if (opts) o = *opts;
  gdbrt::apply_tuning("mst", n, &o);
  const int wgs = default_wgs(&o);
  gdb_stats st{};
  if (n == 0) {
    if (weight) *weight = 0;
    if (edges) *edges = 0;
    if (components) *components = 0;
    if (stats) *stats = st;
    return GDB_SUCCESS;
  }
  // Each row longer than kLongRow has at most 2 * edges / kLongRow pieces.
  const int piece_cap = 2 * (m / kLongRow) + 1;
  const size_t bytes = carve_bytes<int>(n) * 2 + carve_bytes<u64>(n) + carve_bytes<unsigned char>(n) +
                       carve_bytes<int2>(piece_cap) + carve_bytes<int>(32) + carve_bytes<u64>(1);
  int rc = ensure_workspace(ctx, bytes);
  if (rc) return rc;
  Carve cv(ctx->ws);
  int* comp = cv.take<int>(n);
  int* parent = cv.take<int>(n);
  u64* best = cv.take<u64>(n);
  unsigned char* dead = cv.take<unsigned char>(n);
  int2* pieces = cv.take<int2>(piece_cap);
  int* flags = cv.take<int>(32);
  u64* total = cv.take<u64>(1);
  int* out = flags + 8;
  int* npieces = flags + 16;
  const int nwords = (int)((int*)(total + 1) - flags);  // flags and total are neighbours in the workspace
  rc = prepare_launch(ctx, flags, nwords);
  if (rc) return rc;
  rc = gdb_dispatch_wgs(wgs, [&](auto W) -> int {
    constexpr int WG = decltype(W)::value;
    int groups = 0;
    int r2 = launch_groups(ctx, (const void*)k_mst<WG>, &o, row_walk_items(n, m, wgs), &groups);
    if (r2) return r2;
    r2 = timer_start(ctx);
    if (r2) return r2;
    hipLaunchKernelGGL(k_mst<WG>, dim3(groups), dim3(WG), 0, ctx->stream, ctx->d, row, col, w, n, comp, parent,
                       best, dead, pieces, piece_cap, npieces, flags, total, out);
    GDB_HIP(hipGetLastError());
    return finish_launch(ctx, &st.kernel_ms, flags, nwords);
  });
  if (rc) return rc;
  const int* hout = collected_words(ctx) + 8;
  unsigned long long hw = 0;
  memcpy(&hw, collected_words(ctx) + nwords - 2, sizeof(hw));
  st.rounds = hout[0];
  st.barriers = hout[1];
  st.launches = 1;
  st.work_edges = (long long)m * hout[0];
  st.work_items = (long long)n * hout[0];
  st.participating = collected_participating(ctx);
  rc = collected_error(ctx);
  if (weight) *weight = hw;
  if (edges) *edges = hout[2];
  if (components) *components = hout[3];
  if (stats) *stats = st;
  return rc;
}
