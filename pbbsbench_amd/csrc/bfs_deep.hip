// Single-source BFS of deep graphs with short rows (every row at most
// kDeepMaxRow entries, symmetric): all levels in one persistent launch that
// meets every few levels, not every level, then one pass for the parents.
//
// What bounds a deep graph's level is latency: a few hundred vertices per
// CU, a chain of dependent round trips, and the meeting of all workgroups.
// So each workgroup holds its part of the frontier in LDS and expands it
// several levels on its own before it meets the others.  Depths are claimed
// with atomicMin, which keeps that exact:
//   * The workgroups start a superstep with F_k split among them and every
//     depth up to k final.  In phase j (0, 1, ...) each expands what it
//     claimed in phase j - 1, claiming neighbours at k + j + 1.  A vertex of
//     F_{k+1} has a neighbour in F_k, so somebody lowers it to k + 1 in phase
//     0, and whoever did expands it in phase 1; by induction every vertex of
//     F_{k+j} is lowered to its depth in phase j - 1 and expanded in phase j.
//   * A workgroup that runs ahead may first claim a vertex at too large a
//     depth; the true claim lowers it later in the superstep, and its stale
//     copy in the first claimer's list only costs the time to expand it.
// Parents need the final depths: parent[v] = the largest neighbour with depth
// depth[v] - 1 (deterministicBFS/BFS.C:65-74), one pass over the rows once
// the levels are done.
//
// Nothing is written back or dropped from the L2 at a meeting: depths move by
// device-scope atomics and loads, the lists that change hands by device-scope
// stores and loads, and everything else is constant.  The meeting itself is
// one 8-byte word per workgroup, {superstep, levels advanced, entries}: each
// workgroup stores its own and polls all of them, so the wait also delivers
// the counts the next split needs.  Words and lists alternate between two
// sets; a workgroup writes a set again only after all have met once more, by
// when nobody reads it.
//
// 216^3 torus, 325 levels: 6.05 ms with a grid barrier every level (18.6 us a
// level), 1.56 ms so: 4.5 us a level, parents 87 us.  Two workgroups per CU
// against one: 2.43 and 2.72 ms (before `seen` replaced the depth loads); at
// most 4, 8, 16, 32 and 64 levels between meetings: 3.50, 3.16 (before `seen`),
// 1.81, 1.68 and 1.60.  Bound by latency: two round trips a level (the row,
// then the claim) and three LDS syncs.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bfs_device.hpp"
#include "device_util.hpp"

namespace pbbs {

namespace {

constexpr int kPer = 8;   // row entries a lane reads together

template <typename T>
__device__ __forceinline__ T ld_agent(gptr<T> p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void st_agent(gptr<T> p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What the levels read and write, as global pointers.
template <typename OffT>
struct DeepView {
  gptr<const OffT> off;
  gptr<const int32_t> adj;
  gptr<int32_t> depth;
};

// A meeting word: superstep | overflow | levels advanced | entries.
constexpr unsigned kOverBit = 1u << 31;
constexpr int kAdvShift = 16;
constexpr unsigned kAdvMask = 0x7fff, kCountMask = 0xffff;
static_assert(kDeepCap <= (int)kCountMask, "a list's length fits its field");

struct DeepLds {
  unsigned long long q[2][kDeepCap];   // row start << 32 | row length
  unsigned pre[kDeepMaxGroups + 1];
  unsigned wsum[kDeepBlock / kWave];
  int cand[kDeepCand];                 // neighbours to claim
  int seen[1 << kDeepSeenBits];        // vertices met, by hash
  unsigned cnt[2], ncand;
  unsigned adv;
  int bad;                             // 1: a list overflowed, 2: the launch is to end
};

// One phase: the rows of q[from][0, n) claim their unreached neighbours at
// depth d; claimed vertices with edges go to q[from ^ 1].
//
// The rows are read first, kPer entries per lane together.  `seen` then drops
// a neighbour this workgroup has claimed before: at d or less, so its depth is
// no larger now (d never falls).  The table keeps one vertex per slot, and a
// vertex pushed out of it is only claimed once more.  The others are listed,
// and claimed one entry per lane, so that the atomics (a round trip each,
// which the compiler does not overlap within a lane) run on full wavefronts.
// The claimed rows' bounds load beside them.
//
// The table drops most of a row: the neighbours one level up and those a
// sister vertex leads to as well were claimed by this workgroup, whose list
// is a patch of the frontier.  Reading the depths to drop the rest cost more
// than claiming them (one more round trip a phase): 216^3 torus 2.22 ms
// against 1.98, relabelled at random 3.16 against 3.03.
template <typename OffT>
__device__ __forceinline__ void deep_expand(const DeepView<OffT>& A, DeepLds& s, int from,
                                            unsigned n, int d) {
  const unsigned long long* in = s.q[from];
  unsigned long long* out = s.q[from ^ 1];
  for (unsigned e = threadIdx.x; e < n; e += kDeepBlock) {
    const unsigned long long row = in[e];
    const unsigned lo = (unsigned)(row >> 32), deg = (unsigned)row;
    for (unsigned c = 0; c < deg; c += kPer) {
      int v[kPer];
#pragma unroll
      for (int i = 0; i < kPer; ++i) v[i] = A.adj[lo + min(c + i, deg - 1)];
      unsigned claims = 0;
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const unsigned slot = ((unsigned)v[i] * 0x9E3779B1u) >> (32 - kDeepSeenBits);
        if (c + i < deg) claims |= (unsigned)(atomicExch(&s.seen[slot], v[i]) != v[i]) << i;
      }
      unsigned at = atomicAdd(&s.ncand, (unsigned)__popc(claims));
#pragma unroll
      for (int i = 0; i < kPer; ++i)
        if ((claims >> i) & 1u) {
          if (at < (unsigned)kDeepCand) s.cand[at] = v[i];
          ++at;
        }
    }
  }
  __syncthreads();
  const unsigned nc = s.ncand;
  if (nc > (unsigned)kDeepCand && threadIdx.x == 0) s.bad = 1;
  const unsigned lim = nc < (unsigned)kDeepCand ? nc : (unsigned)kDeepCand;
  for (unsigned x = threadIdx.x; x < lim; x += kDeepBlock) {
    const int v = s.cand[x];
    const OffT o0 = A.off[v], o1 = A.off[v + 1];
    if (atomicMin(gen(A.depth + v), d) > d && o1 > o0) {   // the first to lower it to d
      const unsigned at = atomicAdd(&s.cnt[from ^ 1], 1u);
      if (at < (unsigned)kDeepCap)
        out[at] = (unsigned long long)(unsigned)o0 << 32 | (unsigned)(o1 - o0);
      else
        s.bad = 1;
    }
  }
}

// All levels.  Every wait is bounded by A->wait_ticks: a workgroup that runs
// out aborts the launch (host_status[2] = 1); a list that overflows, or a
// frontier large enough that bottom-up levels are due, ends it as well
// (host_status[2] = 2).  The host then runs the BFS again one level per
// launch, with the same outputs.
template <typename OffT>
__global__ __launch_bounds__(kDeepBlock) void bfs_deep_kernel(const BfsArgs<OffT>* __restrict__ Ap,
                                                              DeepWs ws) {
  __shared__ DeepLds s;
  const BfsArgs<OffT> A = *Ap;
  const DeepView<OffT> view{glob(A.off), glob(A.adj), glob(A.depth)};
  const gptr<int32_t> abort_flag = glob(&A.st->abort);
  const unsigned t = threadIdx.x, b = blockIdx.x, G = gridDim.x;
  for (unsigned i = t; i < (1u << kDeepSeenBits); i += kDeepBlock) s.seen[i] = -1;
  if (t == 0) {
    s.bad = 0;
    s.cnt[0] = 0;
    const int32_t src = A.q[0][0];
    const OffT lo = A.off[src], hi = A.off[src + 1];
    if (b == 0 && hi > lo) {
      s.q[0][0] = (unsigned long long)(unsigned)lo << 32 | (unsigned)(hi - lo);
      s.cnt[0] = 1;
    }
  }
  __syncthreads();
  unsigned T = 1;   // entries in all lists; a source without edges ends the first superstep
  float growth = 0;   // log2 of the frontier's growth per level over the last superstep
  int cur = 0, k = 0;
  for (unsigned step = 1;; ++step) {
    const bool solo = T <= (unsigned)kDeepSolo;
    // as many levels as a list may grow over without filling beyond a quarter
    const float room = log2f((float)(kDeepCap / 4)) - log2f(fmaxf((float)T / (float)G, 1.f));
    const int phases =
        solo ? kDeepPhases
             : max(1, (int)fminf((float)kDeepPhases, room / fmaxf(growth, 1e-3f)));
    unsigned n = s.cnt[cur];
    int adv = solo ? 0 : phases;
    if (!solo || b == 0) {
      for (int j = 0; j < phases; ++j) {
        if (n == 0 || (solo && n > (unsigned)kDeepSoloMax)) break;
        __syncthreads();   // everybody has read cnt
        if (t == 0) s.cnt[cur ^ 1] = s.ncand = 0;
        __syncthreads();
        deep_expand(view, s, cur, n, k + j + 1);
        __syncthreads();
        cur ^= 1;
        n = min(s.cnt[cur], (unsigned)kDeepCap);
        if (solo) ++adv;
      }
    }
    // publish this workgroup's list, then its word
    const gptr<unsigned long long> list =
        glob(ws.lists) + ((size_t)(step & 1) * G + b) * kDeepCap;
    for (unsigned e = t; e < n; e += kDeepBlock) st_agent(list + e, s.q[cur][e]);
    __builtin_amdgcn_s_waitcnt(0);   // this wavefront's stores are in
    __syncthreads();
    const gptr<unsigned long long> words = glob(ws.words) + (size_t)(step & 1) * kDeepMaxGroups;
    if (t == 0)
      st_agent(words + b, (unsigned long long)step << 32 | (s.bad == 1 ? kOverBit : 0u) |
                              (unsigned)adv << kAdvShift | n);
    // wait for everybody's; the counts' prefix
    constexpr int kWords = kDeepMaxGroups / kDeepBlock;
    unsigned c[kWords], mine = 0;
    const long long t0 = (long long)wall_clock64();
#pragma unroll
    for (int i = 0; i < kWords; ++i) {
      const unsigned g = t * kWords + i;
      unsigned long long w = 0;
      while (g < G) {
        w = ld_agent(words + g);
        if ((unsigned)(w >> 32) == step) break;
        if (ld_agent(abort_flag)) {
          s.bad = 2;
          break;
        }
        if ((long long)wall_clock64() - t0 > A.wait_ticks) {
          st_agent(abort_flag, (int32_t)1);
          __hip_atomic_store(&A.host_status[2], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
          s.bad = 2;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      c[i] = g < G ? (unsigned)w & kCountMask : 0u;
      if (g < G && ((unsigned)w & kOverBit)) s.bad = 1;
      if (g == 0) s.adv = (unsigned)w >> kAdvShift & kAdvMask;
      mine += c[i];
    }
    unsigned x = mine;
    for (int d = 1; d < kWave; d <<= 1) {
      const unsigned y = __shfl_up(x, d);
      if (__lane_id() >= (unsigned)d) x += y;
    }
    if (__lane_id() == kWave - 1) s.wsum[t / kWave] = x;
    __syncthreads();
    x -= mine;
    for (unsigned i = 0; i < t / kWave; ++i) x += s.wsum[i];
#pragma unroll
    for (int i = 0; i < kWords; ++i) {
      s.pre[t * kWords + i] = x;
      x += c[i];
    }
    if (t == kDeepBlock - 1) s.pre[kDeepMaxGroups] = x;
    __syncthreads();
    const unsigned before = T;
    T = s.pre[kDeepMaxGroups];
    growth = T > before ? log2f((float)T / (float)before) / (float)max(s.adv, 1u) : 0.f;
    k += (int)s.adv;
    const int bad = s.bad;
    // bottom-up levels are due, by an estimate: T is about |F|, more by vertices
    // claimed at too large a depth, and each has an edge at least
    const bool big = A.td_to_bu_div > 0 &&
                     (unsigned long long)T * 2 > (unsigned long long)A.m / (unsigned)A.td_to_bu_div &&
                     T > (unsigned)kDeepSolo;
    if (bad == 1 || (big && bad == 0)) {   // all workgroups see the same words
      if (b == 0 && t == 0) {
        st_agent(abort_flag, (int32_t)1);
        __hip_atomic_store(&A.host_status[2], 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
      return;
    }
    if (bad || T == 0) return;
    // this workgroup's part of the lists, end to end
    const bool one = T <= (unsigned)kDeepSolo;
    const unsigned e0 = one ? (b == 0 ? 0 : T) : (unsigned)((unsigned long long)T * b / G);
    const unsigned e1 = one ? T : (unsigned)((unsigned long long)T * (b + 1) / G);
    cur = 0;
    for (unsigned e = e0 + t; e < e1; e += kDeepBlock) {
      int lo = 0, hi = (int)G;   // pre[lo] <= e < pre[hi]
      while (hi - lo > 1) {
        const int mid = (lo + hi) / 2;
        if (s.pre[mid] <= e) lo = mid;
        else hi = mid;
      }
      const gptr<unsigned long long> from =
          glob(ws.lists) + ((size_t)(step & 1) * G + lo) * kDeepCap;
      s.q[0][e - e0] = ld_agent(from + (e - s.pre[lo]));
    }
    if (t == 0) s.cnt[0] = e1 > e0 ? e1 - e0 : 0;
    __syncthreads();
  }
}

// Parents from the final depths, and the run's totals.  A lane takes kV
// vertices at a time, so that the chain of round trips (depth and row bounds,
// row, the neighbours' depths) is paid once for all of them, and kPer entries
// of a row together from its top; sorted rows stop at the first hit.  Bound by
// the row stream and the depth gathers.
template <typename OffT>
__global__ __launch_bounds__(kBlock) void bfs_deep_parents_kernel(
    const BfsArgs<OffT>* __restrict__ Ap, DeepWs ws, int sorted) {
  constexpr int kV = 2, kP = 6;
  __shared__ unsigned long long red[kWavesPerBlock][4];
  const BfsArgs<OffT> A = *Ap;
  const DeepView<OffT> a{glob(A.off), glob(A.adj), glob(A.depth)};
  const gptr<int32_t> parent = glob(A.parent);
  BfsState* st = A.st;
  if (st->abort) return;
  const long long stride = (long long)gridDim.x * kBlock;
  unsigned long long reached = 0, edges = 0;
  int last = 0, levels = 0;   // largest depth; levels with a vertex to expand
  for (long long v0 = (long long)blockIdx.x * kBlock + threadIdx.x; v0 < A.n; v0 += kV * stride) {
    int dv[kV], best[kV];
    OffT lo[kV];
    unsigned deg[kV], most = 0;
#pragma unroll
    for (int j = 0; j < kV; ++j) {
      const long long v = v0 + j * stride < A.n ? v0 + j * stride : v0;
      dv[j] = a.depth[v];
      lo[j] = a.off[v];
      deg[j] = (unsigned)(a.off[v + 1] - lo[j]);
    }
#pragma unroll
    for (int j = 0; j < kV; ++j) {
      best[j] = -1;
      if ((j > 0 && v0 + j * stride >= A.n) || (long long)dv[j] >= A.n) {
        dv[j] = 0;
        deg[j] = 0;
        continue;
      }
      ++reached;
      edges += deg[j];
      last = max(last, dv[j]);
      if (deg[j]) levels = max(levels, dv[j] + 1);
      if (dv[j] == 0) deg[j] = 0;   // the source: its own parent already
      most = max(most, deg[j]);
    }
    for (unsigned c = 0; c < most; c += kP) {
      int u[kV][kP], du[kV][kP];
#pragma unroll
      for (int j = 0; j < kV; ++j)
#pragma unroll
        for (int i = 0; i < kP; ++i) {   // idle lanes read entry 0
          u[j][i] = a.adj[c + i < deg[j] ? lo[j] + (OffT)(deg[j] - 1 - c - i) : (OffT)0];
        }
#pragma unroll
      for (int j = 0; j < kV; ++j)
#pragma unroll
        for (int i = 0; i < kP; ++i) du[j][i] = a.depth[u[j][i]];
      most = 0;
#pragma unroll
      for (int j = 0; j < kV; ++j) {
#pragma unroll
        for (int i = 0; i < kP; ++i)
          if (c + i < deg[j] && du[j][i] == dv[j] - 1) best[j] = max(best[j], u[j][i]);
        if (sorted && best[j] >= 0) deg[j] = min(deg[j], c + kP);   // done
        most = max(most, deg[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < kV; ++j)
      if (best[j] >= 0) parent[v0 + j * stride] = best[j];
  }
  for (int d = 32; d >= 1; d >>= 1) {
    reached += __shfl_xor(reached, d);
    edges += __shfl_xor(edges, d);
    last = max(last, __shfl_xor(last, d));
    levels = max(levels, __shfl_xor(levels, d));
  }
  const unsigned w = threadIdx.x / kWave;
  if (__lane_id() == 0) {
    red[w][0] = reached;
    red[w][1] = edges;
    red[w][2] = (unsigned long long)last;
    red[w][3] = (unsigned long long)levels;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int i = 1; i < kWavesPerBlock; ++i) {
    reached += red[i][0];
    edges += red[i][1];
    last = max(last, (int)red[i][2]);
    levels = max(levels, (int)red[i][3]);
  }
  // not atomics on the totals: they share a line, and 4096 workgroups' adds
  // to it took 190 us of this kernel's 250
  unsigned long long* part = ws.part + (size_t)blockIdx.x * 4;
  part[0] = reached;
  part[1] = edges;
  part[2] = (unsigned long long)last;
  part[3] = (unsigned long long)levels;
}

// The totals of the parents pass's workgroups, to the host (one workgroup).
template <typename OffT>
__global__ __launch_bounds__(kBlock) void bfs_deep_totals_kernel(
    const BfsArgs<OffT>* __restrict__ Ap, DeepWs ws, int parts) {
  __shared__ unsigned long long red[kWavesPerBlock][4];
  if (Ap->st->abort) return;
  unsigned long long x[4] = {0, 0, 0, 0};
  for (int i = threadIdx.x; i < parts; i += kBlock) {
    const unsigned long long* p = ws.part + (size_t)i * 4;
    x[0] += p[0];
    x[1] += p[1];
    x[2] = p[2] > x[2] ? p[2] : x[2];
    x[3] = p[3] > x[3] ? p[3] : x[3];
  }
  for (int d = 32; d >= 1; d >>= 1)
    for (int j = 0; j < 4; ++j) {
      const unsigned long long y = __shfl_xor(x[j], d);
      x[j] = j < 2 ? x[j] + y : y > x[j] ? y : x[j];
    }
  if (__lane_id() == 0)
    for (int j = 0; j < 4; ++j) red[threadIdx.x / kWave][j] = x[j];
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int i = 1; i < kWavesPerBlock; ++i)
    for (int j = 0; j < 4; ++j)
      x[j] = j < 2 ? x[j] + red[i][j] : red[i][j] > x[j] ? red[i][j] : x[j];
  BfsState* h = Ap->host_state;
  h->reached = x[0];
  h->edges_reached = x[1];
  h->max_depth = (int32_t)x[2];
  h->td_levels = (int32_t)x[3];
  h->bu_levels = 0;
  __threadfence_system();
  __hip_atomic_store(&Ap->host_status[1], (int32_t)x[3], __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&Ap->host_status[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

template <typename OffT>
const void* deep_kernel_symbol() {
  return reinterpret_cast<const void*>(&bfs_deep_kernel<OffT>);
}

// After the init kernel (which clears ws.words): the levels (grid must be
// resident at once), the parents, the totals.
template <typename OffT>
hipError_t launch_bfs_deep(const BfsArgs<OffT>* dargs, const DeepWs& ws, bool sorted, int grid,
                           int parents_grid, hipStream_t stream) {
  if (grid < 1 || grid > kDeepMaxGroups || parents_grid < 1 || parents_grid > kDeepMaxParts)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(bfs_deep_kernel<OffT>, dim3(grid), dim3(kDeepBlock), 0, stream, dargs, ws);
  hipLaunchKernelGGL(bfs_deep_parents_kernel<OffT>, dim3(parents_grid), dim3(kBlock), 0, stream,
                     dargs, ws, sorted ? 1 : 0);
  hipLaunchKernelGGL(bfs_deep_totals_kernel<OffT>, dim3(1), dim3(kBlock), 0, stream, dargs, ws,
                     parents_grid);
  return hipGetLastError();
}

#define PBBS_DEEP_INSTANTIATE(OffT)                                                            \
  template const void* deep_kernel_symbol<OffT>();                                             \
  template hipError_t launch_bfs_deep<OffT>(const BfsArgs<OffT>*, const DeepWs&, bool, int,    \
                                            int, hipStream_t);
PBBS_DEEP_INSTANTIATE(uint32_t)
PBBS_DEEP_INSTANTIATE(int64_t)
#undef PBBS_DEEP_INSTANTIATE

}  // namespace pbbs
