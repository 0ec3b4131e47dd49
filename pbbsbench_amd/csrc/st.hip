// Spanning forest of an edge array: the forest PBBS's incrementalST returns
// (benchmarks/spanningForest/incrementalST/ST.C:35-71), which is the forest
// its speculative_for round schedule (common/speculative_for.h:30-100, with
// granularity 100) produces.  That schedule decides the answer: edges that
// share a round reserve and commit against the union-find state of the
// rounds before, so a later edge of the round can join the forest where a
// serial pass would have taken an earlier one.  The GPU therefore runs the
// same schedule, round by round, with every round's work spread over the
// device:
//   reserve  the schedule's size rule on the round before (halve above 20%
//            failures, double below 10%), then each iterate i of the round
//            (the failed ones of the round before first, in order, then the
//            next unprocessed edges) finds the roots u < v of its ends and
//            write-mins i into R[v];
//   commit   an iterate still holding R[v] links v under u (parents[v] = u;
//            roots are always their tree's smallest vertex, so links go from
//            larger to smaller ids and never close a cycle); the iterates
//            that reserved and lost, in order, form the front of the next
//            round.
// The forest is R's reserved entries in vertex order (ST.C:67-69).  The
// schedule's control words live in device memory, so rounds are launched
// without the host reading anything between them.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <climits>

#include "bfs_device.hpp"

namespace pbbs {

namespace {

__device__ __forceinline__ unsigned lanes_below(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// Roots of J vertices per thread (algorithm/union_find.h:36-52): -1 marks a
// root; a walk points each visited vertex at its grandparent.  Finds run only
// in the reserve kernel, where no link happens, so every pointer it reads or
// writes is an ancestor and a stale read is still one.  The loads of all J are
// issued together: the parent of every vertex, then every grandparent (most
// walks end there), then the rest of the long walks one by one.  x[j] < 0
// marks an idle slot.
template <int J>
__device__ __forceinline__ void st_find_many(int32_t* parents, int32_t (&x)[J]) {
  int32_t p[J], g[J];
#pragma unroll
  for (int j = 0; j < J; ++j) p[j] = parents[x[j] < 0 ? 0 : x[j]];
#pragma unroll
  for (int j = 0; j < J; ++j) g[j] = parents[p[j] < 0 ? 0 : p[j]];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    if (x[j] < 0 || p[j] < 0) continue;   // idle, or x is a root
    int32_t i = x[j], q = p[j], gq = g[j];
    while (gq >= 0) {
      parents[i] = gq;
      i = q;
      q = gq;
      gq = parents[q];
    }
    x[j] = q;
  }
}

// Contiguous share of [0, size) for workgroup b of g, in whole workgroup tiles.
__device__ __forceinline__ void st_share(long long size, long long& lo, long long& hi) {
  const long long tiles = (size + kBlock - 1) / kBlock;
  const long long per = (tiles + gridDim.x - 1) / gridDim.x * kBlock;
  lo = (long long)blockIdx.x * per;
  hi = lo + per < size ? lo + per : size;
}

// Order-preserving positions of the kept entries of a J x kBlock step (entry
// j * kBlock + threadIdx.x): pos[j] among them, and their number.  wcnt holds
// J * kWavesPerBlock counts; the workgroup meets twice.
template <int J>
__device__ __forceinline__ unsigned st_order(const bool (&keep)[J], unsigned (&pos)[J],
                                             unsigned* wcnt) {
  const unsigned w = threadIdx.x / kWave;
  unsigned long long m[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    m[j] = __ballot(keep[j]);
    if (__lane_id() == 0) wcnt[j * kWavesPerBlock + w] = (unsigned)__popcll(m[j]);
  }
  __syncthreads();
  unsigned run = 0;
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int k = 0; k < kWavesPerBlock; ++k) {
      if (k == (int)w) pos[j] = run + lanes_below(m[j]);
      run += wcnt[j * kWavesPerBlock + k];
    }
  __syncthreads();   // wcnt is free again
  return run;
}

__global__ __launch_bounds__(kBlock) void st_init_kernel(StArgs a) {
  const long long tid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long nth = (long long)gridDim.x * blockDim.x;
  for (long long v = tid; v < a.n; v += nth) {
    a.parents[v] = -1;
    a.R[v] = UINT_MAX;
  }
  if (tid == 0) {
    StCtl& c = *a.ctl;
    StSlot z{};
    z.rounds = -1;            // the first round's kernel makes it 0
    z.cur = a.max_round / 4;
    z.finished = a.m == 0;
    c.slot[0] = c.slot[1] = z;
    c.rounds = 0;
    c.count = 0;
    c.error = 0;
    c.filter = 0;
    __threadfence_system();
    __hip_atomic_store(&a.host_status[1], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&a.host_status[0], z.finished, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// The edges both of whose ends lie in one large tree are most of a run's
// edges once that tree has formed, and they drop out of their round with no
// effect.  This kernel writes the vertices of the tree to a bitmap: 2 MB at
// 2^24 vertices, which each XCD's L2 holds, where the two finds such an edge
// costs read a 128-byte line each from the 64 MB parents.  Trees only grow,
// so the bitmap stays true, if not complete, until it is written again.  It
// also points every vertex at its root.
//
// The tree is the most frequent root of 256 sampled edge ends not yet
// processed; below an eighth of them there is no such tree, and the bitmap is
// left alone.  Every workgroup samples the same edges and no link happens
// here, so all of them take the same decision.
__global__ __launch_bounds__(kBlock) void st_tree_kernel(StArgs a, int par) {
  __shared__ int32_t roots[kBlock];
  __shared__ unsigned long long best[kWavesPerBlock];
  const StSlot c = a.ctl->slot[par];
  if (c.finished) return;
  const unsigned t = threadIdx.x;
  {
    const unsigned long long left = (unsigned long long)(a.m - c.done);
    const unsigned long long h = (unsigned long long)(t + 1) * 0x9E3779B97F4A7C15ull;
    const int32_t x = a.eu[c.done + (long long)((h >> 32) * left >> 32)];
    int32_t r = -1;
    if ((uint32_t)x < (uint32_t)a.n) {
      r = x;
      for (int32_t p = a.parents[r]; p >= 0; p = a.parents[r]) r = p;
    }
    roots[t] = r;
  }
  __syncthreads();
  unsigned long long mine = 0;   // votes, then the root
  for (int j = 0; j < kBlock; ++j) mine += roots[j] == roots[t];
  mine = roots[t] < 0 ? 0 : mine << 32 | (unsigned)roots[t];
  for (int d = 32; d >= 1; d >>= 1) {
    const unsigned long long o = __shfl_xor(mine, d);
    mine = o > mine ? o : mine;
  }
  if (__lane_id() == 0) best[t / kWave] = mine;
  __syncthreads();
  for (int j = 0; j < kWavesPerBlock; ++j) mine = best[j] > mine ? best[j] : mine;
  if ((mine >> 32) < kBlock / 8) return;
  const int32_t tree = (int32_t)(unsigned)mine;
  if (blockIdx.x == 0 && t == 0) a.ctl->filter = 1;
  constexpr int kU = 4;
  const long long nwords = (a.n + 63) / 64;
  const long long W = (long long)gridDim.x * kWavesPerBlock;
  for (long long w0 = ((long long)blockIdx.x * kWavesPerBlock + t / kWave) * kU; w0 < nwords;
       w0 += W * kU) {
    int32_t p[kU], g[kU];
#pragma unroll
    for (int j = 0; j < kU; ++j) {
      const long long v = (w0 + j) * 64 + __lane_id();
      p[j] = v < a.n ? a.parents[v] : -1;
    }
#pragma unroll
    for (int j = 0; j < kU; ++j) g[j] = a.parents[p[j] < 0 ? 0 : p[j]];
#pragma unroll
    for (int j = 0; j < kU; ++j) {
      const long long v = (w0 + j) * 64 + __lane_id();
      int32_t r = p[j] < 0 ? (int32_t)v : p[j];
      if (p[j] >= 0 && g[j] >= 0) {
        r = g[j];
        for (int32_t q = a.parents[r]; q >= 0; q = a.parents[r]) r = q;
        a.parents[v] = r;
      }
      const unsigned long long in = __ballot(v < a.n && r == tree);
      if (__lane_id() == 0 && w0 + j < nwords) a.tree_bits[w0 + j] = in;
    }
  }
}

// One round's reservations, and first the bookkeeping of the round before
// (speculative_for.h:78-95), which every workgroup works out for itself from
// that round's per-tile counts of losers; workgroup 0 writes it to the other
// slot for the kernels after this one.
//
// The round's iterates are cut into tiles of a.tile, one workgroup each: the
// losers of the round before, in order (their tiles' lists end to end), then
// the next edge ids.  A step takes J x kBlock of them: the edges in the large
// tree drop out by the bitmap, the rest are compacted in LDS (so finds run on
// full wavefronts), find their roots and reserve; those whose ends differ go
// to the tile's list, in order.  J iterates per thread keep 2J loads in flight.
// Bound by random accesses while most edges take finds (a 128-byte line of
// parents each); once the bitmap holds the tree, by its lookups in the L2 and
// the chain of dependent loads (about 22 us a launch however few edges are
// left).  190.6M shuffled RMAT edges on 2^24 vertices, 111 rounds: 75-100 us a
// round without the bitmap; with it, 95 us before round 8, 45 at round 30 and
// 30 from round 60 on, 4.4 ms a forest against 7.9 (the forest: 10.9 -> 5.8
// ms, with the commit, schedule and pack launches in one: 2.7 -> 0.95 ms).
// A pass that filtered the edges two rounds ahead, on workgroups of their own
// beside the rounds, took 6.3 ms: the filter's lookups cost the same there.
template <int J>
__global__ __launch_bounds__(kBlock) void st_reserve_kernel(StArgs a, int par) {
  constexpr int kPer = kStMaxTiles / kBlock;
  __shared__ unsigned pre[kStMaxTiles + 1];
  __shared__ uint32_t lid[J * kBlock];
  __shared__ int32_t lu[J * kBlock], lv[J * kBlock];
  __shared__ unsigned wcnt[J * kWavesPerBlock];
  const unsigned t = threadIdx.x;
  unsigned cnt[kPer];   // loaded with the slot, not after it
#pragma unroll
  for (int j = 0; j < kPer; ++j) cnt[j] = a.lost[t * kPer + j];
  const StSlot p = a.ctl->slot[par];
  const bool filter = a.ctl->filter != 0;
  if (p.finished) {
    if (blockIdx.x == 0 && t == 0) a.ctl->slot[par ^ 1].finished = 1;
    return;
  }
  {
    const long long tiles = (p.size + a.tile - 1) / a.tile;
    unsigned mine = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      if ((int)t * kPer + j >= tiles) cnt[j] = 0;   // left by a larger round, or by no round
      mine += cnt[j];
    }
    unsigned x = mine;
    for (int d = 1; d < kWave; d <<= 1) {
      const unsigned y = __shfl_up(x, d);
      if (__lane_id() >= (unsigned)d) x += y;
    }
    if (__lane_id() == kWave - 1) wcnt[t / kWave] = x;
    __syncthreads();
    x -= mine;
    for (int j = 0; j < (int)(t / kWave); ++j) x += wcnt[j];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      pre[t * kPer + j] = x;
      x += cnt[j];
    }
    if (t == kBlock - 1) pre[kStMaxTiles] = x;
    __syncthreads();
  }
  StSlot c;
  c.nkeep = pre[kStMaxTiles];
  c.done = p.done + p.size - c.nkeep;
  c.cur = p.cur;
  const float share = (float)c.nkeep / (float)p.size;   // NaN before round 0: no change
  if (share > .2) {
    long long lo = a.max_round / 64 + 1;
    if (c.nkeep > lo) lo = c.nkeep;
    c.cur = c.cur / 2 > lo ? c.cur / 2 : lo;
  } else if (share < .1) {
    c.cur = c.cur * 2 < a.max_round ? c.cur * 2 : a.max_round;
  }
  c.rounds = p.rounds + 1;
  c.size = c.cur < a.m - c.done ? c.cur : a.m - c.done;
  const bool over = c.done >= a.m;
  const bool gave_up = !over && c.rounds > a.max_tries;   // size 0 never moves
  c.finished = over || gave_up;
  c.pad = 0;
  if (blockIdx.x == 0 && t == 0) {
    a.ctl->slot[par ^ 1] = c;
    a.ctl->rounds = c.rounds;
    if (gave_up) atomicOr(&a.ctl->error, 2);
    __threadfence_system();
    __hip_atomic_store(&a.host_status[1], (int32_t)c.rounds, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
    if (c.finished)
      __hip_atomic_store(&a.host_status[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if (c.finished) return;
  const uint32_t* bits = reinterpret_cast<const uint32_t*>(a.tree_bits);
  const long long tiles = (c.size + a.tile - 1) / a.tile;
  for (long long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const long long i0 = tile * a.tile;
    const long long i1 = i0 + a.tile < c.size ? i0 + a.tile : c.size;
    unsigned nout = 0;
    for (long long base = i0; base < i1; base += J * kBlock) {
      uint32_t id[J];
      int32_t u[J], v[J];
      bool keep[J];
      unsigned pos[J];
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const long long i = base + j * kBlock + t;
        keep[j] = i < i1;
        id[j] = keep[j] ? (uint32_t)(c.done + i) : 0u;
        if (i < c.nkeep && keep[j]) {   // a loser: the tile whose list holds it
          int lo = 0, hi = kStMaxTiles;   // pre[lo] <= i < pre[hi]
          while (hi - lo > 1) {
            const int mid = (lo + hi) / 2;
            if (pre[mid] <= (unsigned)i) lo = mid;
            else hi = mid;
          }
          id[j] = a.hold[lo * a.tile + (i - pre[lo])];
        }
      }
#pragma unroll
      for (int j = 0; j < J; ++j) {
        u[j] = a.eu[id[j]];
        v[j] = a.ev[id[j]];
      }
#pragma unroll
      for (int j = 0; j < J; ++j) {
        if (keep[j] && ((uint32_t)u[j] >= (uint32_t)a.n || (uint32_t)v[j] >= (uint32_t)a.n)) {
          // an end outside [0, n): the run reports it and its forest is not
          // used; the edge takes no part (it is never read as a vertex)
          keep[j] = false;
          atomicOr(&a.ctl->error, 1);
        }
        if (!keep[j]) u[j] = v[j] = 0;
      }
      if (filter) {
        uint32_t bu[J], bv[J];
#pragma unroll
        for (int j = 0; j < J; ++j) {
          bu[j] = bits[(uint32_t)u[j] >> 5];
          bv[j] = bits[(uint32_t)v[j] >> 5];
        }
#pragma unroll
        for (int j = 0; j < J; ++j)
          keep[j] = keep[j] && !((bu[j] >> (u[j] & 31)) & (bv[j] >> (v[j] & 31)) & 1u);
      }
      const unsigned total = st_order<J>(keep, pos, wcnt);
#pragma unroll
      for (int j = 0; j < J; ++j)
        if (keep[j]) {
          lid[pos[j]] = id[j];
          lu[pos[j]] = u[j];
          lv[pos[j]] = v[j];
        }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const unsigned s = j * kBlock + t;
        keep[j] = s < total;
        id[j] = keep[j] ? lid[s] : 0u;
        u[j] = keep[j] ? lu[s] : -1;
        v[j] = keep[j] ? lv[s] : -1;
      }
      st_find_many<J>(a.parents, u);
      st_find_many<J>(a.parents, v);
#pragma unroll
      for (int j = 0; j < J; ++j) {
        keep[j] = u[j] != v[j];   // idle slots hold -1 twice
        if (u[j] > v[j]) {
          const int32_t x = u[j];
          u[j] = v[j];
          v[j] = x;
        }
        if (keep[j]) atomicMin(&a.R[v[j]], id[j]);
      }
      const unsigned kept = st_order<J>(keep, pos, wcnt);   // also frees the LDS lists
#pragma unroll
      for (int j = 0; j < J; ++j)
        if (keep[j]) {
          const long long o = i0 + nout + pos[j];
          a.I[o] = id[j];
          a.su[o] = u[j];
          a.sv[o] = v[j];
        }
      nout += kept;
    }
    if (t == 0) a.cand[tile] = nout;
  }
}

// Commit: an iterate still holding R[v] links v under u; the others of the
// tile's list, in order, form the tile's part of the next round's front.
__global__ __launch_bounds__(kBlock) void st_commit_kernel(StArgs a, int par) {
  constexpr int J = 2;
  __shared__ unsigned wcnt[J * kWavesPerBlock];
  const StSlot c = a.ctl->slot[par ^ 1];
  if (c.finished) return;
  const long long tiles = (c.size + a.tile - 1) / a.tile;
  for (long long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const long long i0 = tile * a.tile;
    const unsigned n = a.cand[tile];
    unsigned nl = 0;
    for (unsigned base = 0; base < n; base += J * kBlock) {
      uint32_t id[J], r[J];
      int32_t v[J];
      bool lose[J];
      unsigned pos[J];
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const unsigned s = base + j * kBlock + threadIdx.x;
        lose[j] = s < n;
        id[j] = lose[j] ? a.I[i0 + s] : 0u;
        v[j] = lose[j] ? a.sv[i0 + s] : 0;
      }
#pragma unroll
      for (int j = 0; j < J; ++j) r[j] = a.R[v[j]];
#pragma unroll
      for (int j = 0; j < J; ++j)
        if (lose[j] && r[j] == id[j]) {
          a.parents[v[j]] = a.su[i0 + base + j * kBlock + threadIdx.x];
          lose[j] = false;
        }
      const unsigned lost = st_order<J>(lose, pos, wcnt);
#pragma unroll
      for (int j = 0; j < J; ++j)
        if (lose[j]) a.hold[i0 + nl + pos[j]] = id[j];
      nl += lost;
    }
    if (threadIdx.x == 0) a.lost[tile] = nl;
  }
}

// The ndST contract (spanningForest/ndST/ST.C): any spanning forest.  One
// pass over the edges: an edge finds the roots u < v of its ends and, if it
// is the first to claim hooks[u] (compare-and-swap from free), links u under
// v; a lost claim or a stale root means finding again.  Links go from the
// smaller root to the larger, so no cycle forms; each root is hooked once.
// Finds here run beside links, so they read parents at agent scope (not a
// stale L1 copy).  A claim lost to an edge whose link is not yet visible is
// retried; kAnyTries bounds that wait, and running out marks the run as
// failed (error bit 4) rather than spinning on.
constexpr int kAnyTries = 1 << 16;

__device__ __forceinline__ int32_t ld_parent(const int32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int32_t st_find_any(int32_t* parents, int32_t i) {
  int32_t p = ld_parent(&parents[i]);
  if (p < 0) return i;
  int32_t gp = ld_parent(&parents[p]);
  while (gp >= 0) {
    __hip_atomic_store(&parents[i], gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    i = p;
    p = gp;
    gp = ld_parent(&parents[p]);
  }
  return p;
}

__global__ __launch_bounds__(kBlock) void st_any_kernel(StArgs a) {
  const long long tid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long nth = (long long)gridDim.x * blockDim.x;
  uint32_t* hooks = a.R;
  for (long long i = tid; i < a.m; i += nth) {
    int32_t u = a.eu[i], v = a.ev[i];
    if ((uint32_t)u >= (uint32_t)a.n || (uint32_t)v >= (uint32_t)a.n) {
      atomicOr(&a.ctl->error, 1);
      continue;
    }
    // The retry loop runs while any lane of the wavefront still retries, and
    // a winning lane links inside it.  With a per-lane exit the compiler may
    // move the link store to the loop's exit, which the wavefront reaches
    // only when every lane is done: a lane waiting for that link would then
    // never see it.
    bool active = true;
    int t = 0;
    while (__ballot(active)) {
      if (active) {
        u = st_find_any(a.parents, u);
        v = st_find_any(a.parents, v);
        if (u == v) {
          active = false;
        } else {
          if (u > v) {
            const int32_t x = u;
            u = v;
            v = x;
          }
          if (__hip_atomic_load(&hooks[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                  UINT_MAX &&
              atomicCAS(&hooks[u], UINT_MAX, (uint32_t)i) == UINT_MAX) {
            __hip_atomic_store(&a.parents[u], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            active = false;
          } else if (++t == kAnyTries) {
            atomicOr(&a.ctl->error, 4);
            active = false;
          }
        }
      }
    }
  }
}

// filter_map of R (ST.C:67-69): per-workgroup counts of reserved entries, one
// workgroup's scan of them, then the ordered writes.
__global__ __launch_bounds__(kBlock) void st_out_count_kernel(StArgs a) {
  __shared__ unsigned wsum[kWavesPerBlock];
  long long lo, hi;
  st_share(a.n, lo, hi);
  unsigned cnt = 0;
  for (long long v = lo + threadIdx.x; v < hi; v += kBlock) cnt += a.R[v] != UINT_MAX;
  for (int d = 32; d >= 1; d >>= 1) cnt += __shfl_xor(cnt, d);
  if (__lane_id() == 0) wsum[threadIdx.x / kWave] = cnt;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned t = 0;
    for (int w = 0; w < kWavesPerBlock; ++w) t += wsum[w];
    a.blk[blockIdx.x] = t;
  }
}

__global__ __launch_bounds__(1024) void st_out_scan_kernel(StArgs a, int groups) {
  __shared__ unsigned long long part[1024 / kWave];
  const int t = threadIdx.x;
  unsigned long long mine = 0;
  for (int j = 0; j < kStScanPer; ++j) {
    const int g = t * kStScanPer + j;
    if (g < groups) mine += a.blk[g];
  }
  unsigned long long x = mine;
  const unsigned lane = __lane_id();
  for (int d = 1; d < kWave; d <<= 1) {
    const unsigned long long y = __shfl_up(x, d);
    if (lane >= (unsigned)d) x += y;
  }
  if (lane == kWave - 1) part[t / kWave] = x;
  __syncthreads();
  if (t < kWave) {
    unsigned long long y = t < 1024 / kWave ? part[t] : 0;
    for (int d = 1; d < kWave; d <<= 1) {
      const unsigned long long z = __shfl_up(y, d);
      if (lane >= (unsigned)d) y += z;
    }
    if (t < 1024 / kWave) part[t] = y;
  }
  __syncthreads();
  unsigned long long run = x - mine + (t >= kWave ? part[t / kWave - 1] : 0);
  for (int j = 0; j < kStScanPer; ++j) {
    const int g = t * kStScanPer + j;
    if (g < groups) {
      const unsigned long long cg = a.blk[g];
      a.blk[g] = (unsigned)run;
      run += cg;
    }
  }
  if (t == 1023) a.ctl->count = (long long)run;
}

__global__ __launch_bounds__(kBlock) void st_out_write_kernel(StArgs a, int32_t* forest) {
  __shared__ unsigned wcnt[kWavesPerBlock];
  long long lo, hi;
  st_share(a.n, lo, hi);
  unsigned base = a.blk[blockIdx.x];
  const unsigned lane = __lane_id(), w = threadIdx.x / kWave;
  for (long long t0 = lo; t0 < hi; t0 += kBlock) {
    const long long v = t0 + threadIdx.x;
    const uint32_t r = v < hi ? a.R[v] : UINT_MAX;
    const bool k = r != UINT_MAX;
    const unsigned long long m = __ballot(k);
    if (lane == 0) wcnt[w] = (unsigned)__popcll(m);
    __syncthreads();
    unsigned before = 0, total = 0;
    for (int j = 0; j < kWavesPerBlock; ++j) {
      before += j < (int)w ? wcnt[j] : 0;
      total += wcnt[j];
    }
    if (k) forest[base + before + lanes_below(m)] = (int32_t)r;
    base += total;
    __syncthreads();
  }
}

}  // namespace

hipError_t launch_st_init(const StArgs& a, int grid, hipStream_t stream) {
  hipLaunchKernelGGL(st_init_kernel, dim3(grid), dim3(kBlock), 0, stream, a);
  return hipGetLastError();
}

// One round of the schedule: two launches, each a no-op once the run is over.
// Round r reads slot r & 1.
hipError_t launch_st_round(const StArgs& a, long long round, int grid, hipStream_t stream) {
  if (grid < 1 || grid > kStMaxTiles) return hipErrorInvalidValue;
  const int par = (int)(round & 1);
  if (a.step == 8)
    hipLaunchKernelGGL(st_reserve_kernel<8>, dim3(grid), dim3(kBlock), 0, stream, a, par);
  else if (a.step == 4)
    hipLaunchKernelGGL(st_reserve_kernel<4>, dim3(grid), dim3(kBlock), 0, stream, a, par);
  else
    hipLaunchKernelGGL(st_reserve_kernel<1>, dim3(grid), dim3(kBlock), 0, stream, a, par);
  hipLaunchKernelGGL(st_commit_kernel, dim3(grid), dim3(kBlock), 0, stream, a, par);
  return hipGetLastError();
}

// The bitmap of the large tree as round r is about to find it.
hipError_t launch_st_tree(const StArgs& a, long long round, int grid, hipStream_t stream) {
  hipLaunchKernelGGL(st_tree_kernel, dim3(grid), dim3(kBlock), 0, stream, a, (int)(round & 1));
  return hipGetLastError();
}

hipError_t launch_st_any(const StArgs& a, int grid, hipStream_t stream) {
  hipLaunchKernelGGL(st_any_kernel, dim3(grid), dim3(kBlock), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_st_output(const StArgs& a, int32_t* forest, int grid, hipStream_t stream) {
  if (grid < 1 || grid > kStMaxGroups) return hipErrorInvalidValue;
  hipLaunchKernelGGL(st_out_count_kernel, dim3(grid), dim3(kBlock), 0, stream, a);
  hipLaunchKernelGGL(st_out_scan_kernel, dim3(1), dim3(1024), 0, stream, a, grid);
  hipLaunchKernelGGL(st_out_write_kernel, dim3(grid), dim3(kBlock), 0, stream, a, forest);
  return hipGetLastError();
}

}  // namespace pbbs
