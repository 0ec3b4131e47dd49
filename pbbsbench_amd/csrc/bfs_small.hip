// Single-source BFS of a small graph by one workgroup, the whole run in one
// launch: parents, depths and the queue of reached vertices live in LDS, so a
// level costs a few LDS round trips and one read of its rows instead of a
// launch, and claims are LDS atomics.  Levels run top-down:
// parent[v] = max{u in F_k : (u,v) in E} by atomicMax, guarded by
// depth[v] > k as in the level kernels (deterministicBFS/BFS.C:59-74); the
// claim that returns -1 appends v to the queue, whose tail is F_{k+1}.
//
// A level takes its frontier kSmallBlock vertices at a time and their edges
// kPer per thread at a time: every vertex marks its first edge of the step, and
// a running maximum over the marks gives each edge its vertex, so hub rows
// spread over the workgroup.  (A binary search per edge over the degree sums
// made ten LDS reads of it.)  What bounds a run are its steps' waits, two
// gathers and four barriers each: a call to device memory on rMat of 2^12
// vertices, 53K edges takes 54 us (69 with a launch per level), on a torus of
// 12^3 52 (156).  Eight edges a thread halve the steps of a wide level and
// lengthen the narrow ones: 5 and 19% more.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bfs_device.hpp"
#include "device_util.hpp"

namespace pbbs {

namespace {

constexpr uint16_t kFar = 0xffff;   // not reached (a depth is below n <= kSmallMaxN)
constexpr int kPer = 4;             // edges a thread takes together (its marks are 8-byte words)
static_assert(kSmallMaxN < kFar, "depths and ids fit 16 bits");

template <typename OffT>
__global__ __launch_bounds__(kSmallBlock) void bfs_small_kernel(
    const BfsSmallJob* __restrict__ jobs, BfsSmallJob one) {
  __shared__ int32_t parent[kSmallMaxN];
  __shared__ uint16_t depth[kSmallMaxN];
  __shared__ uint16_t queue[kSmallMaxN];   // reached vertices, level by level
  __shared__ uint32_t base[kSmallBlock];   // per vertex of the chunk: row start - first edge
  __shared__ alignas(16) uint16_t mark[kPer * kSmallBlock];   // vertex + 1 at its first edge
  __shared__ uint32_t wsum[kSmallBlock / kWave];
  __shared__ int32_t sink[kSmallBlock];
  __shared__ unsigned tail;
  const BfsSmallJob job = jobs ? jobs[blockIdx.x] : one;
  const gptr<const OffT> off = glob((const OffT*)job.off);
  const gptr<const int32_t> adj = glob(job.adj);
  constexpr unsigned kWaves = kSmallBlock / kWave;
  const int t = threadIdx.x, n = job.n;
  const int w = __builtin_amdgcn_readfirstlane(t / kWave);
  const unsigned lane = __lane_id();
  for (int i = t; i < n; i += kSmallBlock) {
    parent[i] = -1;
    depth[i] = kFar;
  }
  sink[t] = 0;
  __syncthreads();
  if (t == 0) {
    parent[job.source] = job.source;
    depth[job.source] = 0;
    queue[0] = (uint16_t)job.source;
    tail = 1;
  }
  __syncthreads();
  unsigned head = 0, end = 1;
  int k = 0, levels = 0;
  unsigned long long edges = 0;
  for (; head < end; ++k) {
    unsigned long long level_edges = 0;
    for (unsigned c = head; c < end; c += kSmallBlock) {
      uint32_t deg = 0, lo = 0;
      if (c + t < end) {
        const int v = queue[c + t];
        const OffT o = off[v];
        deg = (uint32_t)(off[v + 1] - o);
        lo = (uint32_t)o;   // m < 2^32
      }
      const uint32_t x = wave_inclusive_sum_dpp(deg);
      if (lane == kWave - 1) wsum[w] = x;
      __syncthreads();
      // the wavefronts' sums, one per lane of the first row, scanned
      const uint32_t ws = wave_inclusive_sum_dpp(lane < kWaves ? wsum[lane] : 0u);
      const uint32_t E = __builtin_amdgcn_readlane(ws, kWave - 1);   // the chunk's edges
      const uint32_t first =                                         // this vertex's first
          x - deg + (w ? __builtin_amdgcn_readlane(ws, w - 1) : 0u);
      base[t] = lo - first;
      level_edges += E;
      for (uint32_t e0 = 0; e0 < E; e0 += kPer * kSmallBlock) {
#pragma unroll
        for (int q = 0; q < kPer / 4; ++q) reinterpret_cast<uint64_t*>(mark + kPer * t)[q] = 0;
        __syncthreads();   // wsum is free again too
        if (deg) {
          if (first >= e0) {
            if (first - e0 < (uint32_t)(kPer * kSmallBlock)) mark[first - e0] = (uint16_t)(t + 1);
          } else if (e0 - first < deg) {
            mark[0] = (uint16_t)(t + 1);
          }
        }
        __syncthreads();
        uint64_t mk[kPer / 4];
#pragma unroll
        for (int q = 0; q < kPer / 4; ++q)
          mk[q] = reinterpret_cast<const uint64_t*>(mark + kPer * t)[q];
        unsigned idx[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
          idx[j] = (unsigned)(mk[j / 4] >> (16 * (j % 4)) & 0xffff);
          if (j) idx[j] = max(idx[j], idx[j - 1]);
        }
        const unsigned run = wave_inclusive_max_dpp(idx[kPer - 1]);
        if (lane == kWave - 1) wsum[w] = run;
        __syncthreads();
        const unsigned wm = wave_inclusive_max_dpp(lane < kWaves ? wsum[lane] : 0u);
        const unsigned ahead = max(dpp_u32<kWaveShr1, 0xf>(run, 0u),
                                   w ? (unsigned)__builtin_amdgcn_readlane(wm, w - 1) : 0u);
        int v[kPer], u[kPer], d[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
          idx[j] = max(max(idx[j], ahead), 1u) - 1u;
          const uint32_t e = e0 + (uint32_t)(kPer * t + j);
          v[j] = e < E ? adj[base[idx[j]] + e] : -1;
        }
#pragma unroll
        for (int j = 0; j < kPer; ++j) u[j] = queue[c + idx[j]];
#pragma unroll
        for (int j = 0; j < kPer; ++j) d[j] = depth[v[j] < 0 ? job.source : v[j]];
        // every lane makes every atomic, idle ones on a word of their own: a
        // conditional one waits for its result before the next is made
        int old[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j)   // the source's depth is 0: idle lanes claim nothing
          old[j] = atomicMax(d[j] > k ? &parent[v[j]] : &sink[t], u[j]);
        unsigned long long fresh[kPer];
        unsigned total = 0;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
          const bool f = d[j] > k && old[j] == -1;
          if (f) depth[v[j]] = (uint16_t)(k + 1);
          fresh[j] = __ballot(f);
          total += (unsigned)__popcll(fresh[j]);
        }
        if (total) {   // one append a wavefront
          unsigned at = 0;
          if (lane == 0) at = atomicAdd(&tail, total);
          at = __shfl(at, 0);
#pragma unroll
          for (int j = 0; j < kPer; ++j) {
            if (fresh[j] >> lane & 1)
              queue[at + __builtin_amdgcn_mbcnt_hi(
                             (unsigned)(fresh[j] >> 32),
                             __builtin_amdgcn_mbcnt_lo((unsigned)fresh[j], 0u))] = (uint16_t)v[j];
            at += (unsigned)__popcll(fresh[j]);
          }
        }
      }
      __syncthreads();   // base and wsum are free again; the level's claims are in
    }
    edges += level_edges;
    levels += level_edges != 0;
    head = end;
    end = tail;
    __syncthreads();   // everybody has read tail
  }
  for (int i = t; i < n; i += kSmallBlock) {
    if (job.parent) job.parent[i] = parent[i];
    if (job.depth) job.depth[i] = depth[i] == kFar ? n : depth[i];
  }
  if (t == 0) {
    BfsState* h = job.host_state;
    h->reached = end;
    h->edges_reached = edges;
    h->max_depth = k - 1;
    h->td_levels = levels;
    h->bu_levels = 0;
    job.host_status[1] = levels;
    job.host_status[0] = 1;
  }
}

}  // namespace

// jobs: device array of njobs jobs, one workgroup each, or null: the job `one`.
template <typename OffT>
hipError_t launch_bfs_small(const BfsSmallJob* jobs, int njobs, const BfsSmallJob& one,
                            hipStream_t stream) {
  hipLaunchKernelGGL(bfs_small_kernel<OffT>, dim3(jobs ? njobs : 1), dim3(kSmallBlock), 0, stream,
                     jobs, one);
  return hipGetLastError();
}

template hipError_t launch_bfs_small<uint32_t>(const BfsSmallJob*, int, const BfsSmallJob&,
                                               hipStream_t);
template hipError_t launch_bfs_small<int64_t>(const BfsSmallJob*, int, const BfsSmallJob&,
                                              hipStream_t);

}  // namespace pbbs
