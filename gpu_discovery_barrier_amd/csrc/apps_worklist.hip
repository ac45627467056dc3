// Lonestar data-driven worklist BFS and SSSP on the discovery protocol.
//
// BFS (code/experiments/lonestar_gpu_opencl/apps/bfs/): dist = MYINFINITY
// (1e9) everywhere, dist[source] = 0 (bfs_port.cpp:112-121); iteration 0
// pushes the source; iteration i pops every worklist item and, for each
// out-edge, sets an unvisited destination to dist = i and pushes it
// (processedge2, bfs_common.cl:73-90); the loop runs while the input
// worklist is non-empty (bfs_port_kernel.cl:173-189).
// SSSP (apps/sssp/): processedge2 relaxes alt = dist[src] + w with
// atomic_min and pushes the destination when alt improved it
// (sssp_common.cl:58-81).  Both converge to exact levels / distances.
//
// Queues hold each vertex at most once per iteration: BFS claims a vertex
// with a compare-and-swap on dist (or sweeps, below), SSSP stamps it with the
// iteration number;
// a queue therefore never exceeds n entries (the reference sizes them by the
// edge count and does not bounds-check pushes, worklist_cl.h:60-62).
//
// Schedules:
//   plain persistent - drelax2's loop: process, barrier, swap and reset the
//                      output index, barrier (two barriers per iteration);
//                      a thread walks its item's edges.
//   tuned persistent - one barrier per iteration (queue tails rotate over
//                      three slots so the reset of the next-next tail needs
//                      no barrier); rows are walked by lanes, waves or in
//                      pieces; pushes are staged in LDS; BFS iterations with
//                      many edges mark vertices and collect them in a sweep.
//                      With the launch shape left open, a sparse graph whose
//                      vertex ids follow locality takes the batched engine's
//                      owner-partitioned ranges instead (solve_if_local).
//   relaunch         - one launch per iteration with a host loop reading the
//                      output size (the non-persistent schedule).
#include <algorithm>
#include <cstring>
#include <mutex>
#include "graph_common.hpp"
#include "runtime.hpp"

// Scratch of gdb_sssp_worklist_noalloc: the stamp array and both queues
// (3 x n ints) plus flags and work counters, for n up to 2^22 vertices.
// Each device that loads the library holds its own copy until the process
// ends.  Host code never passes `scratch` itself to a kernel: its device
// address comes from hipGetSymbolAddress (resolve_noalloc_scratch).
#define GDB_NOALLOC_SCRATCH_BYTES ((size_t)3 * (4u << 22) + 4096)
static __device__ __align__(256) unsigned char scratch[GDB_NOALLOC_SCRATCH_BYTES];

namespace gdbrt {

int resolve_noalloc_scratch(gdb_ctx* ctx) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static void* addr[kMaxDevices] = {};
  if (ctx->device < 0 || ctx->device >= kMaxDevices) return GDB_E_INVALID;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[ctx->device]) {
    int cur = -1;
    GDB_HIP(hipGetDevice(&cur));
    if (cur != ctx->device) GDB_HIP(hipSetDevice(ctx->device));
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != ctx->device) GDB_HIP(hipSetDevice(cur));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)", __FILE__, __LINE__);
    addr[ctx->device] = p;
  }
  ctx->noalloc_scratch = addr[ctx->device];
  return GDB_SUCCESS;
}

}  // namespace gdbrt

namespace {

constexpr unsigned kInf = 1000000000u;  // bfs_common.cl:35
constexpr int kSerialLimit = 16;
constexpr int kChunk = 4;  // edge slots a lane handles per step in the tuned kernel

// Relaxes edge k out of v (distance dv).  Returns whether dst must be pushed.
template <bool WEIGHTED>
__device__ __forceinline__ bool relax_edge(const int* __restrict__ col, const int* __restrict__ w,
                                           unsigned* dist, int* stamp, int k, unsigned dv, int iter,
                                           int n, int* dst_out) {
  const int dst = col[k];
  *dst_out = dst;
  if ((unsigned)dst >= (unsigned)n) return false;
  if (!WEIGHTED) {
    if (dist[dst] != kInf) return false;
    return atomicCAS(&dist[dst], kInf, (unsigned)iter) == kInf;
  } else {
    const unsigned wt = (unsigned)w[k];
    if (wt >= kInf) return false;
    const unsigned alt = dv + wt;
    if (alt >= dist[dst]) return false;
    const unsigned old = atomicMin(&dist[dst], alt);
    if (alt >= old) return false;
    return atomicExch(&stamp[dst], iter) != iter;
  }
}

template <int WGS, bool WEIGHTED>
__global__ __launch_bounds__(WGS) void k_wl_plain(gdb_kernel_ctx_t* ctx, const int* __restrict__ row,
                                                  const int* __restrict__ col,
                                                  const int* __restrict__ w, unsigned* dist,
                                                  int* stamp, int* q0, int* q1, int* idx, int n,
                                                  int* out) {
  DISCOVERY_PROTOCOL(ctx);
  const int tid = p_get_global_id(ctx, &local_ctx);
  const int threads = p_get_global_size(ctx, &local_ctx);
  int* in = q0;
  int* outq = q1;
  int* in_idx = &idx[0];
  int* out_idx = &idx[1];
  int iteration = 1, nbar = 0;
  while (gdb::ld_rlx(in_idx) > 0) {
    const int nin = gdb::ld_rlx(in_idx);
    if (nin > n) {  // a queue never holds more than n entries
      gdb::set_error(ctx, GDB_ERR_QUEUE_OVERFLOW);
      break;
    }
    GDB_FOR_UNIFORM(i, valid, tid, threads, nin) {
      int v = -1;
      if (valid) {
        v = in[i];
        if ((unsigned)v >= (unsigned)n) {
          gdb::set_error(ctx, GDB_ERR_QUEUE_OVERFLOW);
          valid = 0;
        }
      }
      const int b = valid ? row[v] : 0, e = valid ? row[v + 1] : 0;
      const unsigned dv = valid ? dist[v] : 0u;
      int maxlen = e - b;
      for (int off = 32; off > 0; off >>= 1) {
        const int o = __shfl_xor(maxlen, off, 64);
        maxlen = o > maxlen ? o : maxlen;
      }
      for (int t = 0; t < maxlen; ++t) {
        int dst = 0;
        const bool push =
            (b + t < e) && relax_edge<WEIGHTED>(col, w, dist, stamp, b + t, dv, iteration, n, &dst);
        gdb::wave_push(push, dst, outq, out_idx);
      }
    }
    if (!discovery_barrier(ctx, &local_ctx)) return;
    ++nbar;
    int* t = in;
    in = outq;
    outq = t;
    int* ti = in_idx;
    in_idx = out_idx;
    out_idx = ti;
    if (tid == 0) gdb::st_rlx(out_idx, 0);
    ++iteration;
    if (!discovery_barrier(ctx, &local_ctx)) return;  // bfs_port_kernel.cl:187-188
    ++nbar;
  }
  if (tid == 0) {
    out[0] = iteration - 1;
    out[1] = nbar;
  }
}

// Tuned persistent schedule.  What bounded it on skewed graphs was not the
// edges but two serial points: one returning atomic on the queue's size per
// wave step (about 8 ns each on one word, 0.5 M of them on R-MAT 20), and the
// longest row, walked by one wave.  Pushes therefore collect in LDS and a group
// reserves queue space for a batch of them at once; a row longer than kLongRow
// is cut into pieces that all waves share in a second phase of the iteration
// (one more barrier, only in iterations with such a row).  R-MAT 20 BFS: 4.3
// ms -> 0.88 with 256 groups of 256 (2.0 with 64), 0.64 with 512-thread groups and
// the queue's items dealt to the waves; R-MAT 18 SSSP: 4.0 -> 1.43 -> 0.86.
constexpr int kLongRow = 1024;

// BFS iterations with many edges (gdb::sweep_line) set a byte per vertex by plain
// stores, all of the same value, which later edges of the same XCD see; then all
// waves sweep the bytes, give the newly marked vertices their level and queue them.
// R-MAT 20: 0.65 -> 0.42 ms, 17: 0.217 -> 0.203, 12: unchanged.  A bit per vertex
// claimed by OR, as a denser filter in place of dist, was slower: 1.16 ms.

// SPARSE: at most six edges a vertex, where rows may be even (gdb::even_rows); the others
// do without that code.
template <int WGS, bool WEIGHTED, bool SPARSE>
__global__ __launch_bounds__(WGS) void k_wl_tuned(gdb_kernel_ctx_t* ctx, const int* __restrict__ row,
                                                  const int* __restrict__ col,
                                                  const int* __restrict__ w, unsigned* dist,
                                                  int* stamp, int* q0, int* q1, int* tails, int n,
                                                  int4* pieces, int piece_cap, const int* long_row,
                                                  long long* work, int* out) {
  DISCOVERY_PROTOCOL(ctx);
  constexpr int kStage = 8 * WGS;  // pushes of this group awaiting queue space
  __shared__ int s_q[kStage], s_n, s_base, s_deg;
  const gdb::PushStage stage{s_q, &s_n, &s_base, kStage};
  const int tid = p_get_global_id(ctx, &local_ctx);
  const int threads = p_get_global_size(ctx, &local_ctx);
  const int lane = gdb::lane_id(), wave = tid >> 6, nwaves = threads >> 6;
  const int spare = n > 0 ? (int)((unsigned)tid % (unsigned)n) : 0;
  int* const piece_counts = tails + 3;  // rotating, like the tails
  int* const edge_counts = tails + 12;  // BFS: edges of the queued vertices, rotating too
  unsigned char* const mark = (unsigned char*)stamp;  // BFS: a byte per vertex, set once it is reached
  const int sweep_from = gdb::sweep_line(n);
  const bool may_sweep = !WEIGHTED && row[n] > sweep_from;
  const bool even = SPARSE && gdb::even_rows(n, row[n], *long_row != 0);
  // Moves staged vertices to the queue; BFS adds up their edges.
  auto flush = [&](int above, int* queue, int* tail) {
    gdb::group_flush(stage, above, queue, tail, may_sweep ? row : nullptr, &s_deg);
  };
  int iteration = 1, nbar = 0;
  long long items = 0, edges = 0;
  int nin = gdb::ld_rlx(&tails[1]);
  if (threadIdx.x == 0) s_n = s_deg = 0;
  __syncthreads();
  int ne = may_sweep && nin > 0 ? row[q0[0] + 1] - row[q0[0]] : 0;
  while (nin > 0) {
    if (nin > n) {
      gdb::set_error(ctx, GDB_ERR_QUEUE_OVERFLOW);
      break;
    }
    const int* in = (iteration & 1) ? q0 : q1;
    int* outq = (iteration & 1) ? q1 : q0;
    int* out_tail = &tails[(iteration + 1) % 3];
    int* npieces = &piece_counts[iteration % 3];
    int* out_edges = &edge_counts[(iteration + 1) % 3];
    const bool sweep = may_sweep && ne > sweep_from;
    const bool direct = !sweep && gdb::push_directly(even, nin);  // its edges are not counted: no sweep follows
    if (tid == 0) {
      gdb::st_rlx(&tails[(iteration + 2) % 3], 0);
      gdb::st_rlx(&piece_counts[(iteration + 1) % 3], 0);
      gdb::st_rlx(&edge_counts[(iteration + 2) % 3], 0);
    }
    items += nin;
    auto flush_edges = [&]() {
      if (may_sweep && threadIdx.x == 0 && s_deg) {
        gdb::fadd_rlx(out_edges, s_deg);
        s_deg = 0;
      }
    };
    // kChunk edges per lane step (long rows: the whole wave, carrying the
    // row owner's distance): the column and weight loads, then the
    // targets' distances (BFS: their marks), then atomics only where a candidate improves
    // (lanes with none send no atomic), then the once-per-iteration stamps
    // of the improved targets, then the pushes.  Unused slots read edge
    // 0 and this thread's spare vertex, so that the slots stay branch-free.
    auto step = [&](const bool (&ok)[kChunk], const int (&kk)[kChunk], int pd) -> int {
      const unsigned src = (unsigned)pd;
      int dst[kChunk];
      bool push[kChunk];
#pragma unroll
      for (int j = 0; j < kChunk; ++j) {
        dst[j] = -1;
        push[j] = false;
      }
      if (gdb::any_slot(ok)) {
        unsigned wt[kChunk], cur[kChunk];
        bool act[kChunk], need[kChunk];
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
          const int e0 = ok[j] ? kk[j] : 0;  // edge 0 exists here
          dst[j] = gdb::ldg(col + e0);
          wt[j] = WEIGHTED ? (unsigned)gdb::ldg(w + e0) : 1u;
        }
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
          act[j] = ok[j] && (unsigned)dst[j] < (unsigned)n && wt[j] < kInf;
          if (!ok[j]) dst[j] = -1;
          cur[j] = WEIGHTED ? gdb::ldg(dist + (act[j] ? dst[j] : spare)) : (unsigned)gdb::ldg(mark + (act[j] ? dst[j] : spare));
        }
        // A stale distance is never below the current one, so it can
        // only let a needless atomic through.
        bool any_need = false;
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
          need[j] = act[j] && (WEIGHTED ? src + wt[j] < cur[j] : cur[j] == 0u);
          any_need |= need[j];
        }
        if (sweep) {
#pragma unroll
          for (int j = 0; j < kChunk; ++j)
            if (need[j]) mark[dst[j]] = 1;
        } else if (any_need) {
          unsigned old[kChunk];
          bool imp[kChunk], any_imp = false;
#pragma unroll
          for (int j = 0; j < kChunk; ++j) {
            unsigned* dp = &dist[need[j] ? dst[j] : spare];
            old[j] = WEIGHTED ? gdb::atomic_min_g(dp, need[j] ? src + wt[j] : ~0u)
                              : gdb::atomic_cas_g(dp, need[j] ? kInf : ~0u, need[j] ? (unsigned)iteration : ~0u);
          }
#pragma unroll
          for (int j = 0; j < kChunk; ++j) {
            imp[j] = need[j] && (WEIGHTED ? src + wt[j] < old[j] : old[j] == kInf);
            any_imp |= imp[j];
          }
          if (!WEIGHTED) {
#pragma unroll
            for (int j = 0; j < kChunk; ++j) {
              push[j] = imp[j];
              if (imp[j]) mark[dst[j]] = 1;
            }
          } else if (any_imp) {
            // Stamps only grow (iteration numbers): the first to raise
            // one to this iteration queues the target.
            int sp[kChunk];
#pragma unroll
            for (int j = 0; j < kChunk; ++j)
              sp[j] = gdb::atomic_max_g(&stamp[imp[j] ? dst[j] : spare], imp[j] ? iteration : INT_MIN);
#pragma unroll
            for (int j = 0; j < kChunk; ++j) push[j] = imp[j] && sp[j] < iteration;
          }
        }
      }
      if (direct) gdb::wave_push_n<kChunk>(push, dst, outq, out_tail);
      else if (!sweep) gdb::wave_stage_n<kChunk>(stage, push, dst, outq, out_tail);
      return 0;
    };
    auto any = [](int a, int c) { return a | c; };
    long long left = nin;
    GDB_FOR_SPREAD(i, valid, tid, threads, nin, gdb::spread_queue(even, nin)) {
      int v = -1, b = 0, e = 0;
      unsigned dv = 0;
      if (valid) {
        v = in[i];
        if ((unsigned)v >= (unsigned)n) valid = 0;
      }
      if (valid) {
        b = row[v];
        e = row[v + 1];
        if (WEIGHTED) dv = dist[v];
        edges += e - b;
        if (e - b > kLongRow) {
          const int k = (e - b + kLongRow - 1) / kLongRow;
          const int at = gdb::fadd_rlx(npieces, k);
          for (int j = 0; j < k && at + j < piece_cap; ++j, b += kLongRow)
            pieces[at + j] = make_int4(b, min(e, b + kLongRow), (int)dv, 0);
          valid = b < e;  // the part the list has no room for is walked here
        }
      }
      gdb::wave_walk_np<kChunk>(valid != 0, b, e, (int)dv, 0, step, any, kSerialLimit);
      left -= threads;
      if (left > 0) flush(kStage / 2, outq, out_tail);
    }
    if (!direct) flush(0, outq, out_tail);
    flush_edges();
    if (!discovery_barrier(ctx, &local_ctx)) return;
    ++nbar;
    // The words that say what comes next, in one trip: usually the next iteration.
    const int pieces_out = gdb::ld_rlx(npieces), queued = gdb::ld_rlx(out_tail);
    const int queued_edges = may_sweep ? gdb::ld_rlx(out_edges) : 0;
    const int np = min(pieces_out, piece_cap);
    if (np > 0) {
      for (int p0 = 0; p0 < np; p0 += nwaves) {  // the same trips in every wave
        const int p = p0 + wave;
        const int4 pc = p < np ? pieces[p] : make_int4(0, 0, 0, 0);
        for (int base = pc.x; base < pc.y; base += 64 * kChunk) {
          bool ok[kChunk];
          int kk[kChunk];
#pragma unroll
          for (int j = 0; j < kChunk; ++j) {
            kk[j] = base + lane + 64 * j;
            ok[j] = kk[j] < pc.y;
          }
          step(ok, kk, pc.z);
        }
        if (!direct && p0 + nwaves < np) flush(kStage / 2, outq, out_tail);
      }
      if (!direct) flush(0, outq, out_tail);
      flush_edges();
      if (!discovery_barrier(ctx, &local_ctx)) return;
      ++nbar;
    }
    if (sweep) {
      for (long long p0 = 0; p0 < n; p0 += (long long)kChunk * threads) {
        bool push[kChunk];
        int v[kChunk];
        unsigned mk[kChunk], dv[kChunk];
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
          const long long i = p0 + (long long)j * threads + tid;
          push[j] = i < n;
          v[j] = (int)i;
          mk[j] = gdb::ldg(mark + (push[j] ? v[j] : spare));
          dv[j] = gdb::ldg(dist + (push[j] ? v[j] : spare));
        }
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
          push[j] = push[j] && mk[j] != 0 && dv[j] == kInf;
          if (push[j]) dist[v[j]] = (unsigned)iteration;
        }
        gdb::wave_stage_n<kChunk>(stage, push, v, outq, out_tail);
        if (p0 + (long long)kChunk * threads < n) flush(kStage / 2, outq, out_tail);
      }
      flush(0, outq, out_tail);
      flush_edges();
      if (!discovery_barrier(ctx, &local_ctx)) return;
      ++nbar;
    }
    nin = queued;
    ne = queued_edges;
    if (np > 0 || sweep) {
      nin = gdb::ld_rlx(out_tail);
      if (may_sweep) ne = gdb::ld_rlx(out_edges);
    }
    ++iteration;
  }
  // Edges examined, summed over threads (one atomic per wave).
  for (int off = 32; off > 0; off >>= 1) edges += __shfl_xor(edges, off, 64);
  if (lane == 0 && edges) atomicAdd((unsigned long long*)&work[1], (unsigned long long)edges);
  if (tid == 0) {
    out[0] = iteration - 1;
    out[1] = nbar;
    work[0] = items;
  }
}

// Relaunch schedule: one iteration per launch.  tails rotate as above.
template <bool WEIGHTED>
__global__ void k_wl_step(const int* __restrict__ row, const int* __restrict__ col,
                          const int* __restrict__ w, unsigned* dist, int* stamp, int* q0, int* q1,
                          int* tails, int n, int iteration, int* active) {
  // active[0] counts non-empty iterations; active[1] is a sticky done flag
  // raised by the first launch that finds an empty input.
  if (active[1]) return;
  int nin = tails[iteration % 3];
  if (nin > n) nin = n;
  if (nin == 0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) active[1] = 1;
    return;
  }
  const int* in = (iteration & 1) ? q0 : q1;
  int* outq = (iteration & 1) ? q1 : q0;
  int* out_tail = &tails[(iteration + 1) % 3];
  const int gid = blockIdx.x * blockDim.x + threadIdx.x;
  if (gid == 0) {
    tails[(iteration + 2) % 3] = 0;
    atomicAdd(active, 1);
  }
  const int stride = gridDim.x * blockDim.x;
  GDB_FOR_UNIFORM(i, valid, gid, stride, nin) {
    int v = -1, b = 0, e = 0;
    unsigned dv = 0;
    if (valid) {
      v = in[i];
      if ((unsigned)v >= (unsigned)n) valid = 0;
    }
    if (valid) {
      b = row[v];
      e = row[v + 1];
      if (WEIGHTED) dv = dist[v];
    }
    gdb::wave_coop_foreach(
        valid != 0, b, e, dv,
        [&](int k, bool ok, unsigned src_dist) {
          int dst = 0;
          const bool push =
              ok && relax_edge<WEIGHTED>(col, w, dist, stamp, k, src_dist, iteration, n, &dst);
          gdb::wave_push(push, dst, outq, out_tail);
        },
        kSerialLimit);
  }
}

// *long_row (0 before): whether a row has more than kEvenRow edges (row null: not asked).
__global__ void k_wl_init(const int* __restrict__ row, unsigned* dist, int* stamp, int* q0, int* q1, int* flags,
                          int* long_row, int n, int src, bool bytes) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && row && row[i + 1] - row[i] > gdb::kEvenRow) *long_row = 1;
  if (i < n) {  // initialize (bfs_common.cl:64-71) + dist[source] = 0
    dist[i] = i == src ? 0u : kInf;
    stamp[i] = bytes && i == src >> 2 ? 1 << 8 * (src & 3) : 0;  // bytes: the source is marked
  }
  if (i < 32) flags[i] = 0;
  if (i == 0) {  // iteration 0: push the source (bfs_port_kernel.cl:130-137)
    q0[0] = src;
    q1[0] = src;
    flags[0] = 1;  // plain: input index
    flags[4 + 1] = 1;  // tuned / relaunch: tails[1] = input size of iteration 1
  }
}

// dverifysolution (bfs_common.cl:43-60, sssp_common.cl:41-56).
__global__ void k_verify(const int* __restrict__ row, const int* __restrict__ col,
                         const int* __restrict__ w, const unsigned* dist, int n,
                         unsigned long long* nerr) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= n) return;
  unsigned long long bad = 0;
  for (int k = row[u]; k < row[u + 1]; ++k) {
    const int v = col[k];
    const unsigned wt = w ? (unsigned)w[k] : 1u;
    if (wt > 0 && dist[u] + wt < dist[v]) ++bad;
  }
  if (bad) atomicAdd(nerr, bad);
}

// ---- local graphs: the owner-partitioned solve --------------------------------
// A sample of the graph's edges: how many, how far apart their ends are (hist[b]:
// |u - v| < 2^b and not less than 2^(b-1)), and the sum of their weights.
struct Locality {
  int hist[32];
  int edges;
  int pad;
  unsigned long long wsum;
};
constexpr int kSampleVertices = 8192, kSampleEdges = 8;  // evenly spaced vertices, edges of each (a row's
                                                         // long ones may be its last)

__global__ __launch_bounds__(256) void k_locality(const int* __restrict__ row, const int* __restrict__ col,
                                                  const int* __restrict__ w, int n, Locality* out) {
  __shared__ int s_hist[32];
  if (threadIdx.x < 32) s_hist[threadIdx.x] = 0;
  __syncthreads();
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int count = n < kSampleVertices ? n : kSampleVertices;
  int edges = 0;
  unsigned long long ws = 0;
  if (i < count) {
    const int v = (int)((long long)i * n / count);
    const int b = row[v], e = min(row[v + 1], b + kSampleEdges);
    for (int k = b; k < e; ++k) {
      const int u = col[k];
      if ((unsigned)u >= (unsigned)n) continue;  // as the solvers, which skip such an edge
      const int d = abs(u - v);
      atomicAdd(&s_hist[d == 0 ? 0 : 32 - __clz(d)], 1);
      ++edges;
      if (w) ws += min((unsigned)w[k], kInf);
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    edges += __shfl_xor(edges, off, 64);
    ws += __shfl_xor(ws, off, 64);
  }
  if (gdb::lane_id() == 0 && edges) {
    atomicAdd(&out->edges, edges);
    if (w) atomicAdd(&out->wsum, ws);
  }
  __syncthreads();
  if (threadIdx.x < 32 && s_hist[threadIdx.x]) atomicAdd(&out->hist[threadIdx.x], s_hist[threadIdx.x]);
}

// Largest finite distance plus one: the iterations of a BFS worklist.
__global__ void k_levels(const unsigned* __restrict__ dist, int n, int* out) {
  int m = 0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    if (dist[i] < kInf) m = max(m, (int)dist[i] + 1);
  m = gdb::wave_max(m);
  if (gdb::lane_id() == 0 && m > gdb::ld_rlx(out)) atomicMax(out, m);  // 10 ns each on one word
}

// Solves a sparse local graph (grids, meshes, road networks) by the batched
// engine's owner-partitioned ranges: such a graph has thousands of short
// iterations, and there a hop inside a range costs an LDS round instead of
// an inter-group barrier.  *done is false when the graph is none; st then holds the
// device time and launches of finding out.
//
// The rule: at most kLocalDegree edges per vertex (denser graphs, the sample's
// cost not spent on them, are skewed or random in use, and a slot record holds
// four edges), and 99.5% of the sampled edges (SSSP: 98.5%) shorter than half a range:
// more long ones cut the iterations short and leave the ranges crossing each
// other (grids of 128^2 to 1024^2 with 0.5, 1 and 1.8% of random edges, against the
// queues: BFS .93 to .67, 1.38 to .90 and 1.54 to 1.23 of the time, SSSP .74 to
// .37, 1.08 to .61 and 1.23 to .73).  Ranges
// of kLocalRange vertices, one group each (1024^2 grid: 64 ranges 4.63 ms,
// 128 4.92, 256 6.0; 128^2: 1 to 8 within 10%), at most one per CU.  SSSP
// bands of 96 mean weights (24 to 200 measured, within 15%).  1024^2 grid:
// SSSP 33.4 ms with iteration queues, 4.7 here; BFS 13.7 and 2.7; a 64^2 grid
// 0.57 and 0.20, 0.46 and 0.15.
constexpr int kLocalDegree = 6, kLocalRange = 12288, kLocalBand = 96;
constexpr int kLocalNearBfs = 995, kLocalNearSssp = 985;  // of a thousand edges
constexpr int kLocalRangeMax = 30000;  // distances, marks, queues and boundary list of a range fit a CU's LDS

template <bool WEIGHTED>
int solve_if_local(gdb_ctx* ctx, int n, int m, const int* row, const int* col, const int* w, int source,
                   unsigned* dist, gdb_stats* st, bool* done) {
  using namespace gdbrt;
  *done = false;
  if (ctx->xcd_active >= 0 || (long long)m > (long long)kLocalDegree * n || m < n / 2) return GDB_SUCCESS;
  int rc = ensure_workspace(ctx, sizeof(Locality));
  if (rc) return rc;
  Locality* d = (Locality*)ctx->ws;
  constexpr int kWords = sizeof(Locality) / sizeof(int);
  rc = prepare_launch(ctx, (int*)d, kWords);
  if (!rc) rc = timer_start(ctx);
  if (rc) return rc;
  hipLaunchKernelGGL(k_locality, dim3(kSampleVertices / 256), dim3(256), 0, ctx->stream, row, col,
                     WEIGHTED ? w : nullptr, n, d);
  GDB_HIP(hipGetLastError());
  Locality h;
  double ms = 0;
  rc = finish_launch(ctx, &ms, d, kWords);
  if (rc) return rc;
  st->kernel_ms += ms;
  ++st->launches;
  memcpy(&h, collected_words(ctx), sizeof(h));
  if (h.edges == 0) return GDB_SUCCESS;
  const int G = std::max(1, std::min(ctx->num_cus, (n + kLocalRange - 1) / kLocalRange));
  const int range = (n + G - 1) / G;
  long long near = 0;
  for (int b = 0; b < 31 && (1LL << b) <= range / 2; ++b) near += h.hist[b];
  if (near * 1000 < (WEIGHTED ? kLocalNearSssp : kLocalNearBfs) * (long long)h.edges || range > kLocalRangeMax)
    return GDB_SUCCESS;
  gdb_task t{};
  t.algo = WEIGHTED ? GDB_TASK_SSSP : GDB_TASK_BFS;
  t.n = n;
  t.m = m;
  t.row = row;
  t.col = col;
  t.w = w;
  t.source = source;
  t.out = dist;
  t.delta = WEIGHTED ? (int)std::min<unsigned long long>(kInf, 1 + kLocalBand * h.wsum / (unsigned)h.edges) : 0;
  t.owned = 1;
  gdb_opts o{};
  o.wgs = 1024;
  o.groups = G;
  o.barrier = -1;
  gdb_stats solve{};
  rc = gdb_batch_solve(ctx, &t, 1, G, &o, &solve);
  // A range without work waits for the others as long as the solve takes, a queue
  // iteration's barrier never that long: under a short wait bound the queues may
  // still finish.  (The context has been reset.)
  solve.kernel_ms += st->kernel_ms;
  solve.launches += st->launches;
  if (rc == GDB_E_TIMEOUT || t.rounds == 0) {  // or no group took part
    st->kernel_ms = solve.kernel_ms;
    st->launches = solve.launches;
    return rc == GDB_E_TIMEOUT ? GDB_SUCCESS : rc;
  }
  *st = solve;
  if (rc) return rc;
  if (!WEIGHTED) {
    int* levels = (int*)ctx->ws;
    rc = prepare_launch(ctx, levels, 1);
    if (!rc) rc = timer_start(ctx);
    if (rc) return rc;
    hipLaunchKernelGGL(k_levels, dim3(std::min(256, (n + 255) / 256)), dim3(256), 0, ctx->stream, dist, n, levels);
    GDB_HIP(hipGetLastError());
    rc = finish_launch(ctx, &ms, levels, 1);
    if (rc) return rc;
    st->kernel_ms += ms;
    ++st->launches;
    st->rounds = collected_words(ctx)[0];
  }
  *done = true;
  return GDB_SUCCESS;
}

// `fixed_ws`: a caller-provided device buffer of `fixed_bytes` bytes that
// replaces the context's grow-only workspace (no allocation), or nullptr.
template <bool WEIGHTED>
int run_worklist(gdb_ctx* ctx, int n, int m, const int* row, const int* col, const int* w, int source,
                 unsigned* dist, const gdb_opts* opts, gdb_stats* stats, void* fixed_ws = nullptr,
                 size_t fixed_bytes = 0) {
  using namespace gdbrt;
  if (!ctx || n < 0 || m < 0 || (n > 0 && (!row || !dist)) || (m > 0 && !col) ||
      (WEIGHTED && m > 0 && !w) || (n > 0 && (source < 0 || source >= n)))
    return GDB_E_INVALID;
  gdb_opts o{};
  if (opts) o = *opts;
  if (o.variant == GDB_VARIANT_TUNED && o.schedule == GDB_SCHED_PERSISTENT) {
    // A sparse graph's BFS that solve_if_local declines may have a thousand short
    // iterations: a row of its own, with fewer groups to meet in each (a shuffled 500^2
    // grid: 6.6 ms with 128 groups, 5.2 with 64, 4.3 with 32; G(400000) of degree 4 0.27,
    // 0.27 and 0.32).
    if (WEIGHTED || (long long)m > (long long)kLocalDegree * n || !gdbrt::apply_tuning("bfs_wl_sparse", n, &o))
      gdbrt::apply_tuning(WEIGHTED ? "sssp_wl" : "bfs_wl", n, &o);
  }
  const int wgs = default_wgs(&o);
  gdb_stats st{};
  if (n == 0) {
    if (stats) *stats = st;
    return GDB_SUCCESS;
  }
  if (opts && opts->wgs == 0 && opts->groups == 0 && o.variant == GDB_VARIANT_TUNED &&
      o.schedule == GDB_SCHED_PERSISTENT && !fixed_ws) {
    bool done = false;
    const int lrc = solve_if_local<WEIGHTED>(ctx, n, m, row, col, w, source, dist, &st, &done);
    if (lrc || done) {
      if (stats) *stats = st;
      return lrc;
    }
  }
  const gdb_stats tried = st;  // what the attempt took
  const bool tuned_wl = o.variant == GDB_VARIANT_TUNED && o.schedule != GDB_SCHED_RELAUNCH;
  // A row longer than kLongRow has at most 2 * edges / kLongRow pieces.
  int piece_cap = tuned_wl ? (int)(2LL * m / kLongRow) + 1 : 0;
  size_t bytes = carve_bytes<int>(n) * 3 + carve_bytes<int>(32) + carve_bytes<long long>(3);
  if (fixed_ws) {  // the list takes what the caller's buffer has left
    if (bytes > fixed_bytes) return GDB_E_SCRATCH;
    piece_cap = (int)std::min<size_t>(piece_cap, (fixed_bytes - bytes) / sizeof(int4) & ~(size_t)15);
  }
  bytes += carve_bytes<int4>(piece_cap);
  void* base = fixed_ws;
  int rc = GDB_SUCCESS;
  if (base) {
    if (bytes > fixed_bytes) return GDB_E_SCRATCH;
  } else {
    rc = ensure_workspace(ctx, bytes);
    if (rc) return rc;
    base = ctx->ws;
  }
  Carve cv(base);
  int* stamp = cv.take<int>(n);
  int* q0 = cv.take<int>(n);
  int* q1 = cv.take<int>(n);
  int* flags = cv.take<int>(32);
  long long* work = cv.take<long long>(3);
  int4* pieces = cv.take<int4>(piece_cap);
  int* tails = flags + 4;
  int* out = flags + 12;
  int* long_row = (int*)(work + 2);
  rc = prepare_launch(ctx, (int*)work, 5);
  if (rc) return rc;
  hipLaunchKernelGGL(k_wl_init, dim3((n + 255) / 256), dim3(256), 0, ctx->stream,
                     gdb::even_rows(n, m, false) ? row : nullptr, dist, stamp, q0, q1, flags, long_row, n, source,
                     !WEIGHTED);
  GDB_HIP(hipGetLastError());

  if (o.schedule == GDB_SCHED_RELAUNCH) {
    const int check = o.relaunch_check > 1 ? o.relaunch_check : 1;
    int grid = (n + wgs - 1) / wgs;
    if (grid > 4096) grid = 4096;
    int* active = flags + 14;
    rc = timer_start(ctx);
    if (rc) return rc;
    int it = 0;
    for (;;) {
      for (int k = 0; k < check; ++k) {
        ++it;
        hipLaunchKernelGGL(k_wl_step<WEIGHTED>, dim3(grid), dim3(wgs), 0, ctx->stream, row, col, w,
                           dist, stamp, q0, q1, tails, n, it, active);
        st.launches += 1;
      }
      GDB_HIP(hipGetLastError());
      GDB_HIP(hipMemcpyAsync(ctx->h_flag, tails, 3 * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
      GDB_HIP(hipStreamSynchronize(ctx->stream));
      if (ctx->h_flag[(it + 1) % 3] == 0 || ctx->h_flag[it % 3] == 0) break;
      if (it > n + 2) return GDB_E_TIMEOUT;
    }
    rc = timer_stop(ctx, &st.kernel_ms);
    if (rc) return rc;
    int act = 0;
    GDB_HIP(hipMemcpy(&act, active, sizeof(int), hipMemcpyDeviceToHost));
    st.rounds = act;
    st.participating = grid;
  } else {
    const bool tuned = o.variant == GDB_VARIANT_TUNED;
    const int nwords = (int)((int*)(work + 2) - flags);  // flags and work are neighbours in the workspace
    rc = gdb_dispatch_wgs(wgs, [&](auto W) -> int {
      constexpr int WG = decltype(W)::value;
      const bool sparse = gdb::even_rows(n, m, false);
      const void* kern = !tuned   ? (const void*)k_wl_plain<WG, WEIGHTED>
                         : sparse ? (const void*)k_wl_tuned<WG, WEIGHTED, true>
                                  : (const void*)k_wl_tuned<WG, WEIGHTED, false>;
      int groups = 0;
      int r2 = launch_groups(ctx, kern, &o, tuned ? row_walk_items(n, m, wgs) : n, &groups);
      if (r2) return r2;
      r2 = timer_start(ctx);
      if (r2) return r2;
      if (tuned && sparse)
        hipLaunchKernelGGL((k_wl_tuned<WG, WEIGHTED, true>), dim3(groups), dim3(WG), 0, ctx->stream, ctx->d,
                           row, col, w, dist, stamp, q0, q1, tails, n, pieces, piece_cap,
                           long_row, work, out);
      else if (tuned)
        hipLaunchKernelGGL((k_wl_tuned<WG, WEIGHTED, false>), dim3(groups), dim3(WG), 0, ctx->stream, ctx->d,
                           row, col, w, dist, stamp, q0, q1, tails, n, pieces, piece_cap,
                           long_row, work, out);
      else
        hipLaunchKernelGGL((k_wl_plain<WG, WEIGHTED>), dim3(groups), dim3(WG), 0, ctx->stream, ctx->d,
                           row, col, w, dist, stamp, q0, q1, flags, n, out);
      GDB_HIP(hipGetLastError());
      return finish_launch(ctx, &st.kernel_ms, flags, nwords);
    });
    if (rc) return rc;
    st.kernel_ms += tried.kernel_ms;
    st.launches = 1 + tried.launches;
    const int* h = collected_words(ctx);
    st.rounds = h[out - flags];
    st.barriers = h[out + 1 - flags];
    if (tuned) {
      long long hw[2];
      memcpy(hw, h + nwords - 4, sizeof(hw));
      st.work_items = hw[0];
      st.work_edges = hw[1];
    }
    st.participating = collected_participating(ctx);
  }
  rc = o.schedule == GDB_SCHED_RELAUNCH ? check_device_error(ctx) : collected_error(ctx);
  if (stats) *stats = st;
  return rc;
}

}  // namespace

extern "C" int gdb_bfs_worklist(gdb_ctx* ctx, int n, int m, const int* row, const int* col, int source,
                                unsigned* dist, const gdb_opts* opts, gdb_stats* stats) {
  return run_worklist<false>(ctx, n, m, row, col, nullptr, source, dist, opts, stats);
}

extern "C" int gdb_sssp_worklist(gdb_ctx* ctx, int n, int m, const int* row, const int* col,
                                 const int* w, int source, unsigned* dist, const gdb_opts* opts,
                                 gdb_stats* stats) {
  return run_worklist<true>(ctx, n, m, row, col, w, source, dist, opts, stats);
}

extern "C" int gdb_sssp_worklist_noalloc(gdb_ctx* ctx, int n, int m, const int* row, const int* col,
                                         const int* w, int source, unsigned* dist, const gdb_opts* opts,
                                         gdb_stats* stats) {
  if (!ctx) return GDB_E_INVALID;
  if (!ctx->noalloc_scratch) return GDB_E_INVALID;  // resolved by gdb_ctx_create
  if (n > GDB_NOALLOC_MAX_N) return GDB_E_SCRATCH;
  return run_worklist<true>(ctx, n, m, row, col, w, source, dist, opts, stats, ctx->noalloc_scratch,
                            GDB_NOALLOC_SCRATCH_BYTES);
}

extern "C" int gdb_verify_distances(gdb_ctx* ctx, int n, int m, const int* row, const int* col,
                                    const int* w, const unsigned* dist, long long* nerr) {
  using namespace gdbrt;
  if (!ctx || !nerr || n < 0 || m < 0 || (n > 0 && (!row || !dist)) || (m > 0 && !col))
    return GDB_E_INVALID;
  *nerr = 0;
  if (n == 0) return GDB_SUCCESS;
  int rc = ensure_workspace(ctx, 256);
  if (rc) return rc;
  unsigned long long* d_err = (unsigned long long*)ctx->ws;
  rc = fill_i32(ctx, (int*)d_err, 0, 2);
  if (rc) return rc;
  hipLaunchKernelGGL(k_verify, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, row, col, w, dist, n,
                     d_err);
  GDB_HIP(hipGetLastError());
  unsigned long long h = 0;
  GDB_HIP(hipMemcpyAsync(&h, d_err, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
  GDB_HIP(hipStreamSynchronize(ctx->stream));
  *nerr = (long long)h;
  return GDB_SUCCESS;
}
