// Maximal independent set on the BFS's CSR: the set PBBS's incrementalMIS
// computes (benchmarks/maximalIndependentSet/incrementalMIS/MIS.C:35-66), the
// lexicographically first one.  Vertex v joins unless a lower-numbered
// neighbour joins; it is decided once every lower neighbour is.
//
// Rounds, each over a block of vertices not looked at before and a worklist of
// vertices deferred by the rounds before.  The blocks go up in id, so when a
// vertex is first looked at, most of its lower neighbours are decided: with
// one block of all vertices 74% of an RMAT graph's first looks end at an
// undecided neighbour, with 16 blocks 11% (an RMAT graph of 2^20 vertices,
// decisions visible from the next round on).  Each vertex keeps a resume
// position in its row: entries before it are neighbours already known to be
// out of the set or not lower than v.  A round walks each vertex's row from
// there: a lower neighbour in the set makes v out; an undecided one stops the
// walk (v waits for the next round); reaching the end of the lower neighbours
// (the first entry >= v on sorted rows, the row end otherwise) with all of
// them out puts v in.  A vertex's state only goes from undecided to a final
// value, so a round may read one another workgroup has just written, or an
// older copy of it: either way v decides only on final values, and the result
// does not depend on timing.  A round past the last block that finds the list
// empty ends the run.
//
// States are two bits per vertex, {in, out} words of 32 vertices side by side:
// 4 MB at 2^24 vertices, about one XCD's L2, where a byte each (16 MB) cost a
// 128-byte line per neighbour read.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <climits>

#include "bfs_device.hpp"
#include "device_util.hpp"

namespace pbbs {

namespace {

__device__ __forceinline__ unsigned lanes_below_mask(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
// row entries read together: one load at any 4-byte alignment (adj is padded)
typedef int i32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef int i32x4u __attribute__((ext_vector_type(4), aligned(4)));
template <int kStep>
struct StepLoad;
template <>
struct StepLoad<2> {
  typedef i32x2u type;
};
template <>
struct StepLoad<4> {
  typedef i32x4u type;
};

enum { kOpen = 0, kIn = 1, kOut = 2, kLooking = 3 };

// The states of vertices u (of those lower than v; the others count as out):
// all loads, then all tests.
template <int kStep>
__device__ __forceinline__ void mis_states(gptr<const u32x2> st, const int32_t (&u)[kStep],
                                           int32_t v, u32x2 (&w)[kStep]) {
#pragma unroll
  for (int j = 0; j < kStep; ++j) w[j] = st[u[j] < v ? (uint32_t)u[j] >> 5 : 0u];
}

// The same in two steps, for looks at every lane's vertex: the first two
// entries, then the others unless one of the two is in (half of the vertices
// need no more).  A gather occupies a CU's address unit for as many cycles as
// it has lanes, which is what bounds these looks.
template <int kStep>
__device__ __forceinline__ void mis_states_first(gptr<const u32x2> st, const int32_t (&u)[kStep],
                                                 int32_t v, u32x2 (&w)[kStep]) {
#pragma unroll
  for (int j = 0; j < 2; ++j) w[j] = st[u[j] < v ? (uint32_t)u[j] >> 5 : 0u];
}
template <int kStep>
__device__ __forceinline__ void mis_states_rest(gptr<const u32x2> st, const int32_t (&u)[kStep],
                                                int32_t v, u32x2 (&w)[kStep]) {
  bool in = false;
#pragma unroll
  for (int j = 0; j < 2; ++j) in |= u[j] < v && (w[j].x >> (u[j] & 31)) & 1u;
#pragma unroll
  for (int j = 2; j < kStep; ++j) w[j] = st[u[j] < v && !in ? (uint32_t)u[j] >> 5 : 0u];
}

// What a look at entries u (INT32_MAX past the row's end) with state words w
// makes of v, whose row has `left` entries from u[0] on: kOut (a lower
// neighbour is in), kIn (every lower neighbour is out), kOpen (an undecided
// one; skip entries before it are settled) or kLooking (all settled, more of
// the row to read; skip = kStep).
template <int kStep, typename OffT>
__device__ __forceinline__ int mis_verdict(const int32_t (&u)[kStep], const u32x2 (&w)[kStep],
                                           int32_t v, OffT left, int sorted, int& skip) {
  bool any_in = false;
  int first_open = kStep;
#pragma unroll
  for (int j = kStep - 1; j >= 0; --j) {
    const bool low = u[j] < v;
    const unsigned in = (w[j].x >> (u[j] & 31)) & 1u, out = (w[j].y >> (u[j] & 31)) & 1u;
    any_in |= low && in;
    if (low && !(in | out)) first_open = j;
  }
  skip = first_open;
  if (any_in) return kOut;
  if (first_open < kStep) return kOpen;
  if (left <= (OffT)kStep) return kIn;
  if (sorted && u[kStep - 1] >= v) return kIn;   // the rest of the row is not lower
  return kLooking;
}

template <int kStep, typename OffT>
__device__ __forceinline__ void mis_entries(gptr<const int32_t> adj, OffT p, OffT left,
                                            int32_t (&u)[kStep]) {
  typedef typename StepLoad<kStep>::type vec;
  const vec x = *(gptr<const vec>)(adj + p);
#pragma unroll
  for (int j = 0; j < kStep; ++j) u[j] = (OffT)j < left ? x[j] : INT32_MAX;
}

// One look at vertex v from row position p: kStep entries read together (4 on
// rows averaging 16 entries or more, 2 on sparser graphs, where a wider look
// mostly reads states it does not need).  p moves past settled entries.
template <int kStep, typename OffT>
__device__ __forceinline__ int mis_look(const MisArgs<OffT>& a, int32_t v, OffT& p, OffT hi) {
  int32_t u[kStep];
  u32x2 w[kStep];
  mis_entries<kStep, OffT>(glob(a.adj), p, hi - p, u);
  mis_states<kStep>((gptr<const u32x2>)glob(a.state), u, v, w);
  int skip;
  const int r = mis_verdict<kStep, OffT>(u, w, v, hi - p, a.sorted, skip);
  if (r == kOpen || r == kLooking) p += (OffT)skip;
  return r;
}

// Marks v decided (rounds over the worklist: several wavefronts share words).
template <typename OffT>
__device__ __forceinline__ void mis_decide(const MisArgs<OffT>& a, int32_t v, int res) {
  atomicOr(gen(glob((unsigned*)a.state) + ((size_t)((uint32_t)v >> 5) * 2 + (res == kOut))),
           1u << (v & 31));
}

static_assert(kMisStripes == kWave, "one region count per lane of the scan");

// Region s of the round's list holds entries [pre[s], pre[s + 1]) of its
// index space; `s` is a hint no larger than the answer (indices a lane takes
// only grow within a chunk).
__device__ __forceinline__ int region_from(const unsigned long long* pre, unsigned long long i,
                                           int s) {
  while (pre[s + 1] <= i) ++s;
  return s;
}

__device__ __forceinline__ int region_of(const unsigned long long* pre, unsigned long long i) {
  int lo = 0, hi = kMisStripes;   // pre[lo] <= i < pre[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    if (pre[mid] <= i) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Fresh vertices [v0, v0 + kMisPer * 64) below v1, by one wavefront.  First
// one look at each, the loads of a lane's kMisPer vertices issued together
// (row bounds, then entries, then states); that decides most.  The others are
// compacted in LDS and looked at on full wavefronts, a lane taking the next
// one as soon as its own decides or is blocked, so that the few long walks do
// not hold up a whole wavefront each; one that was blocked at its first look
// has a second here, with the rest of the set decided and its row in cache.
// Still blocked, they go to the next list.  The wavefront owns the set's state
// words, so it collects them in LDS and stores them whole, after the first
// looks and at the end.
template <typename OffT>
struct FreshEntry {
  int32_t v;
  uint32_t p, hi;   // row position and end (m < 2^32)
};

template <typename OffT, int kStep>
__device__ __forceinline__ void mis_fresh(const MisArgs<OffT>& a, long long v0, long long v1,
                                          FreshEntry<OffT>* buf, unsigned* words, int32_t* out,
                                          gptr<unsigned long long> count) {
  const unsigned lane = __lane_id();
  const gptr<const OffT> off = glob(a.off);
  const gptr<const int32_t> adj = glob(a.adj);
  const gptr<const u32x2> st = (gptr<const u32x2>)glob(a.state);
  const gptr<u32x4> own = (gptr<u32x4>)(glob((unsigned*)a.state) + (size_t)(v0 >> 5) * 2);
  OffT lo[kMisPer], hi[kMisPer];
  int32_t u[kMisPer][kStep];
  u32x2 w[kMisPer][kStep];
#pragma unroll
  for (int j = 0; j < kMisPer; ++j) {
    const long long v = v0 + j * kWave + lane;
    const long long c = v < v1 ? v : v0;
    lo[j] = off[c];
    hi[j] = off[c + 1];
  }
#pragma unroll
  for (int j = 0; j < kMisPer; ++j) mis_entries<kStep, OffT>(adj, lo[j], hi[j] - lo[j], u[j]);
#pragma unroll
  for (int j = 0; j < kMisPer; ++j)
    mis_states_first<kStep>(st, u[j], (int32_t)(v0 + j * kWave + lane), w[j]);
#pragma unroll
  for (int j = 0; j < kMisPer; ++j)
    mis_states_rest<kStep>(st, u[j], (int32_t)(v0 + j * kWave + lane), w[j]);
  unsigned n = 0;
#pragma unroll
  for (int j = 0; j < kMisPer; ++j) {
    const int32_t v = (int32_t)(v0 + j * kWave + lane);
    int skip;
    int res = mis_verdict<kStep, OffT>(u[j], w[j], v, hi[j] - lo[j], a.sorted, skip);
    if (v0 + j * kWave + lane >= v1) res = -1;
    const unsigned long long in = __ballot(res == kIn), no = __ballot(res == kOut);
    const u32x4 x = {(unsigned)in, (unsigned)no, (unsigned)(in >> 32), (unsigned)(no >> 32)};
    if (lane == 0) {
      *(u32x4*)(words + 4 * j) = x;
      if (v0 + j * kWave < v1) own[j] = x;   // the state covers n rounded up to 64
    }
    const bool open = res == kOpen || res == kLooking;
    const unsigned long long m = __ballot(open);
    if (open)
      buf[n + lanes_below_mask(m)] = {v, (uint32_t)lo[j] + (uint32_t)skip, (uint32_t)hi[j]};
    n += (unsigned)__popcll(m);
  }
  if (!n) return;
  wave_lds_sync();
  FreshEntry<OffT> e = {0, 0, 0};
  bool have = lane < n;
  if (have) e = buf[lane];
  unsigned next = kWave, kept = 0;
  while (__ballot(have)) {
    int res = -1;
    if (have) {
      OffT p = (OffT)e.p;
      const int d = mis_look<kStep>(a, e.v, p, (OffT)e.hi);
      e.p = (uint32_t)p;
      if (d != kLooking) res = d;
      if (d == kIn || d == kOut) {
        const unsigned b = (unsigned)(e.v - (int32_t)v0);
        atomicOr(&words[(b >> 5) * 2 + (d == kOut)], 1u << (b & 31));
      }
    }
    wave_lds_sync();   // the entries taken so far have been read: their places are free
    const unsigned long long dm = __ballot(res == kOpen);
    if (res == kOpen) buf[kept + lanes_below_mask(dm)] = e;
    kept += (unsigned)__popcll(dm);
    const bool take = res >= 0 || !have;
    const unsigned long long fm = __ballot(take);
    if (take) {
      const unsigned i = next + lanes_below_mask(fm);
      have = i < n;
      if (have) e = buf[i];
    }
    next += (unsigned)__popcll(fm);
  }
  wave_lds_sync();
  if (lane < (unsigned)kMisPer && v0 + lane * kWave < v1) own[lane] = *(u32x4*)(words + 4 * lane);
  if (kept) {
    unsigned long long at = 0;
    if (lane == 0) at = atomicAdd(gen(count), (unsigned long long)kept);
    at = __shfl(at, 0);
    if (at + kept > (unsigned long long)a.region) {   // cannot happen; reported, never written
      if (lane == 0)
        __hip_atomic_store(&a.host_status[2], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    } else {
      for (unsigned i = lane; i < kept; i += kWave) {
        const FreshEntry<OffT> x = buf[i];
        glob(a.pos)[x.v] = x.p - (uint32_t)off[x.v];
        glob(out)[at + i] = x.v;
      }
    }
  }
  wave_lds_sync();   // buf and words are free again
}

// Round r takes the fresh vertices of block r (mis_block_start) and list[r & 1] with the count set r % 3 (round 0: no list); it appends to
// list[(r + 1) & 1] and count set (r + 1) % 3; workgroup 0 clears set
// (r + 2) % 3, which held round r - 1's counts.
//
// The wavefronts take the list first (its ids are lower), in chunks of
// consecutive entries, then the fresh vertices.  In a list chunk a lane holds
// one vertex and looks at it (mis_look) until it decides or meets an undecided
// lower neighbour; then it takes the chunk's next vertex, so a long row does
// not hold up the other 63 lanes.  Deferred vertices collect in LDS and go to
// the next list with one atomicAdd per chunk, on the count of the region that
// owns the chunk: chunk k of nchunks goes to region k * kMisStripes / nchunks,
// so the next list keeps the ids roughly ascending (lower ids first lets a
// round see more decisions made earlier in the same round), and a region
// receives at most ceil(nchunks / kMisStripes) chunks: at most
// count / kMisStripes + chunk entries; the same holds for the fresh vertices'
// sets of kMisPer x 64.  List and fresh vertices are at most n in all, so
// `region` holds both.
//
// 2^24 vertices, 381M entries (RMAT, relabelled), a call: 1.16 ms with every
// vertex in round 0 and byte states, 0.58 so; 256^3 torus, relabelled, 0.84 and
// 0.48.  A block of 2.6M vertices takes about 80 us, 70% of it with the CUs'
// address units busy on the state gathers (one lane's address a cycle), which
// hit the L2 at 75-78%.
template <typename OffT, int kStep>
__global__ __launch_bounds__(kBlock) void mis_round_kernel(MisArgs<OffT> a) {
  __shared__ int32_t defer[kWavesPerBlock][kMisMaxChunk];
  static_assert(sizeof(FreshEntry<OffT>) * kMisPer * kWave <= sizeof(defer[0]),
                "a set of fresh vertices fits the buffer");
  __shared__ alignas(16) unsigned words[kWavesPerBlock][4 * kMisPer];
  __shared__ unsigned long long pre[kMisStripes + 1];
  const int r = (int)a.wg_round[blockIdx.x];
  const unsigned lane = __lane_id();
  const long long f0 = mis_block_start(a.block, a.n, r), f1 = mis_block_start(a.block, a.n, r + 1);
  unsigned long long count = 0;
  if (r > 0) {
    if (threadIdx.x < kWave) {   // kMisStripes == kWave: one count per lane, scanned
      const unsigned long long* cin = a.ctr + (size_t)(r % 3) * kMisStripes * 16;
      unsigned long long c = cin[threadIdx.x * 16];
      // a count past the region (never expected; the host reports it) is cut
      // so that every read stays inside the list
      if (c > (unsigned long long)a.region) c = (unsigned long long)a.region;
      for (int d = 1; d < kWave; d <<= 1) {
        const unsigned long long t = __shfl_up(c, d);
        if (lane >= (unsigned)d) c += t;
      }
      pre[threadIdx.x + 1] = c;
      if (threadIdx.x == 0) pre[0] = 0;
    }
    __syncthreads();
    count = pre[kMisStripes];
  }
  if (count == 0 && f0 >= f1) {
    if (blockIdx.x == 0 && threadIdx.x == 0 && !*a.finished) {
      *a.finished = 1;
      __threadfence_system();
      __hip_atomic_store(&a.host_status[1], r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(&a.host_status[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    return;
  }
  if (blockIdx.x == 0 && threadIdx.x < kMisStripes) {
    a.ctr[((size_t)((r + 2) % 3) * kMisStripes + threadIdx.x) * 16] = 0;
    if (threadIdx.x == 0)
      __hip_atomic_store(&a.host_status[1], r + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  // selects, not an index into the argument block (which would copy it to scratch)
  const int32_t* in = (r & 1) ? a.list[1] : a.list[0];
  int32_t* out = (r & 1) ? a.list[0] : a.list[1];
  unsigned long long* cout = a.ctr + (size_t)((r + 1) % 3) * kMisStripes * 16;
  const unsigned wib = threadIdx.x / kWave;
  int32_t* dbuf = defer[wib];
  const unsigned long long nwaves = (unsigned long long)gridDim.x * kWavesPerBlock;
  const unsigned long long wave = (unsigned long long)blockIdx.x * kWavesPerBlock + wib;
  // chunk: the list spread over every wavefront, in multiples of 64, 64..kMisMaxChunk
  unsigned long long chunk = (count + nwaves - 1) / nwaves;
  chunk = ((chunk + kWave - 1) / kWave) * kWave;
  chunk = chunk < kWave ? kWave : (chunk > kMisMaxChunk ? kMisMaxChunk : chunk);
  const unsigned long long nchunks = (count + chunk - 1) / chunk;
  constexpr long long kSet = kMisPer * kWave;
  const unsigned long long nsets = (unsigned long long)((f1 - f0 + kSet - 1) / kSet);
  for (unsigned long long k = wave; k < nchunks + nsets; k += nwaves) {
    if (k >= nchunks) {
      const unsigned long long f = k - nchunks, t = f * kMisStripes / nsets;
      mis_fresh<OffT, kStep>(a, f0 + (long long)f * kSet, f1,
                             reinterpret_cast<FreshEntry<OffT>*>(dbuf), words[wib],
                             out + t * (size_t)a.region, glob(cout + t * 16));
      continue;
    }
    const unsigned long long c0 = k * chunk;
    const unsigned long long c1 = c0 + chunk < count ? c0 + chunk : count;
    unsigned long long next = c0 + kWave;   // the chunk's first entry no lane holds yet
    unsigned ndefer = 0;                    // wave-uniform
    int s = region_of(pre, c0);
    bool have = c0 + lane < c1;
    int32_t v = 0;
    OffT p = 0, lo = 0, hi = 0;
    if (have) {
      const unsigned long long i = c0 + lane;
      s = region_from(pre, i, s);
      v = in[(unsigned long long)s * a.region + (i - pre[s])];
      lo = a.off[v];
      hi = a.off[v + 1];
      p = lo + (OffT)a.pos[v];
    }
    while (__ballot(have)) {
      int res = -1;   // -1 looking on, 0 deferred, 1 / 2 decided
      if (have) {
        const int d = mis_look<kStep>(a, v, p, hi);
        if (d != kLooking) res = d;
      }
      if (res > 0) mis_decide(a, v, res);
      const unsigned long long dm = __ballot(res == 0);
      if (res == 0) {
        a.pos[v] = (uint32_t)(p - lo);
        dbuf[ndefer + lanes_below_mask(dm)] = v;
      }
      ndefer += (unsigned)__popcll(dm);
      // lanes that finished take the chunk's next entries
      const bool take = res >= 0 || !have;
      const unsigned long long free_m = __ballot(take);
      if (take) {
        const unsigned long long i = next + lanes_below_mask(free_m);
        have = i < c1;
        if (have) {
          s = region_from(pre, i, s);
          v = in[(unsigned long long)s * a.region + (i - pre[s])];
          lo = a.off[v];
          hi = a.off[v + 1];
          p = lo + (OffT)a.pos[v];
        }
      }
      next += (unsigned long long)__popcll(free_m);
    }
    // Look again at the chunk's deferred vertices, held in LDS: by now their
    // blockers have had a chunk's time to decide.  Vertices still blocked are
    // compacted to the front of the buffer (writes land below the read
    // cursor: a pass never writes more entries than it has taken).
    for (int pass = 0; pass < kMisRetry && ndefer; ++pass) {
      __builtin_amdgcn_wave_barrier();
      const unsigned total = ndefer;
      unsigned nd2 = 0, nxt = kWave;
      bool hv = lane < total;
      int32_t w = 0;
      OffT q = 0, wlo = 0, whi = 0;
      if (hv) {
        w = dbuf[lane];
        wlo = a.off[w];
        whi = a.off[w + 1];
        q = wlo + (OffT)a.pos[w];
      }
      while (__ballot(hv)) {
        int res = -1;
        if (hv) {
          const int d = mis_look<kStep>(a, w, q, whi);
          if (d != kLooking) res = d;
        }
        if (res > 0) mis_decide(a, w, res);
        const unsigned long long dm = __ballot(res == 0);
        if (res == 0) {
          a.pos[w] = (uint32_t)(q - wlo);
          dbuf[nd2 + lanes_below_mask(dm)] = w;
        }
        nd2 += (unsigned)__popcll(dm);
        __builtin_amdgcn_wave_barrier();
        const bool take = res >= 0 || !hv;
        const unsigned long long fm = __ballot(take);
        if (take) {
          const unsigned i = nxt + lanes_below_mask(fm);
          hv = i < total;
          if (hv) {
            w = dbuf[i];
            wlo = a.off[w];
            whi = a.off[w + 1];
            q = wlo + (OffT)a.pos[w];
          }
        }
        nxt += (unsigned)__popcll(fm);
      }
      ndefer = nd2;
    }
    __builtin_amdgcn_wave_barrier();
    if (ndefer) {
      const unsigned long long t = k * kMisStripes / nchunks;
      unsigned long long at = 0;
      if (lane == 0) at = atomicAdd(&cout[t * 16], (unsigned long long)ndefer);
      at = __shfl(at, 0);
      if (at + ndefer <= (unsigned long long)a.region) {
        int32_t* dst = out + t * (unsigned long long)a.region + at;
        for (unsigned i = lane; i < ndefer; i += kWave) dst[i] = dbuf[i];
      } else if (lane == 0) {   // cannot happen (see above); reported, never written
        __hip_atomic_store(&a.host_status[2], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
  if (threadIdx.x == 0) a.wg_round[blockIdx.x] = (uint32_t)(r + 1);
}

template <typename OffT>
__global__ __launch_bounds__(kBlock) void mis_init_kernel(MisArgs<OffT> a) {
  const long long tid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long nth = (long long)gridDim.x * blockDim.x;
  for (long long w = tid; w < mis_state_words(a.n); w += nth) a.state[w] = 0;
  for (long long i = tid; i < kMaxGrid; i += nth) a.wg_round[i] = 0;
  for (long long i = tid; i < 3 * kMisStripes; i += nth) a.ctr[i * 16] = 0;
  if (tid == 0) {
    *a.finished = 0;
    __threadfence_system();
    __hip_atomic_store(&a.host_status[2], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&a.host_status[1], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&a.host_status[0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Output in the reference's format (MISTime.C:38-43: one int per vertex, 1 in
// the set, 2 not), four vertices per thread, and each workgroup's count of
// set members in part[blockIdx.x].  Nothing before the run is over.
template <typename OffT>
__global__ __launch_bounds__(kBlock) void mis_output_kernel(MisArgs<OffT> a, int32_t* flags_out) {
  __shared__ unsigned wsum[kWavesPerBlock];
  if (!*a.finished) return;
  const long long tid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long nth = (long long)gridDim.x * blockDim.x;
  const long long n4 = a.n / 4;
  int4* o4 = reinterpret_cast<int4*>(flags_out);
  const bool vec = (reinterpret_cast<uintptr_t>(flags_out) & 15) == 0;
  unsigned c = 0;
  if (vec) {
    for (long long i = tid; i < n4; i += nth) {
      const unsigned in = (unsigned)a.state[i >> 3] >> (4 * (i & 7)) & 15u;   // low word: in
      o4[i] = make_int4(2 - (in & 1), 2 - (in >> 1 & 1), 2 - (in >> 2 & 1), 2 - (in >> 3));
      c += __popc(in);
    }
  }
  for (long long v = (vec ? 4 * n4 : 0) + tid; v < a.n; v += nth) {
    const unsigned in = (unsigned)a.state[v >> 5] >> (v & 31) & 1u;
    flags_out[v] = 2 - (int)in;
    c += in;
  }
  for (int d = 32; d >= 1; d >>= 1) c += __shfl_xor(c, d);
  if (__lane_id() == 0) wsum[threadIdx.x / kWave] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (int w = 0; w < kWavesPerBlock; ++w) t += wsum[w];
    a.part[blockIdx.x] = t;
  }
}

// The set's size, to the host: the sum of the output workgroups' counts (one
// workgroup).
template <typename OffT>
__global__ __launch_bounds__(kBlock) void mis_count_kernel(MisArgs<OffT> a, int parts) {
  __shared__ unsigned long long wsum[kWavesPerBlock];
  if (!*a.finished) return;
  unsigned long long c = 0;
  for (int i = threadIdx.x; i < parts; i += kBlock) c += a.part[i];
  for (int d = 32; d >= 1; d >>= 1) c += __shfl_xor(c, d);
  if (__lane_id() == 0) wsum[threadIdx.x / kWave] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (int w = 0; w < kWavesPerBlock; ++w) t += wsum[w];
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(a.host_status + 4), t,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Small graphs (at most kMisSmall vertices): the whole run in one workgroup and
// one launch, the states in LDS.  Vertices go 1024 at a time in id order, one per
// thread; all of them look until all are decided (every lower block is), then
// the next ones, whose row bounds and first entries were loaded meanwhile.
// Launches and round trips are all that counts here: 2^12 vertices of an RMAT
// graph 124 -> 52 us a call, a 20^3 torus 123 -> 51.
template <typename OffT>
__global__ __launch_bounds__(kMisSmallBlock) void mis_small_kernel(MisArgs<OffT> a,
                                                                   int32_t* flags_out) {
  constexpr int kStep = 4;
  __shared__ unsigned st[kMisSmall / 32][2];   // in, out
  __shared__ unsigned wsum[kMisSmallBlock / kWave];
  const int t = threadIdx.x, n = (int)a.n;
  const gptr<const OffT> off = glob(a.off);
  const gptr<const int32_t> adj = glob(a.adj);
  for (int i = t; i < kMisSmall / 32; i += kMisSmallBlock) st[i][0] = st[i][1] = 0;
  OffT lo = 0, hi = 0;
  int32_t u[kStep];
  auto load = [&](int v) {
    lo = v < n ? off[v] : (OffT)0;
    hi = v < n ? off[v + 1] : (OffT)0;
    mis_entries<kStep, OffT>(adj, lo, hi - lo, u);
  };
  load(t);
  __syncthreads();
  int rounds = 0;
  unsigned members = 0;
  for (int b = 0; b < n; b += kMisSmallBlock) {
    const int v = b + t;
    OffT p = lo;
    const OffT end = hi;
    int32_t e[kStep];
#pragma unroll
    for (int j = 0; j < kStep; ++j) e[j] = u[j];
    load(v + kMisSmallBlock);
    int res = v < n ? kLooking : kOut;
    do {
      if (res == kLooking || res == kOpen) {
        u32x2 w[kStep];
#pragma unroll
        for (int j = 0; j < kStep; ++j) {
          const int i = e[j] < v ? e[j] >> 5 : 0;
          w[j] = (u32x2){st[i][0], st[i][1]};
        }
        int skip;
        res = mis_verdict<kStep, OffT>(e, w, v, end - p, a.sorted, skip);
        if (res == kIn || res == kOut) {
          atomicOr(&st[v >> 5][res == kOut], 1u << (v & 31));
        } else if (res == kLooking) {
          p += (OffT)kStep;
          mis_entries<kStep, OffT>(adj, p, end - p, e);
        }
      }
      ++rounds;
    } while (__syncthreads_or(res == kLooking || res == kOpen));
    if (v < n) {
      flags_out[v] = res;
      members += res == kIn;
    }
  }
  for (int d = 32; d >= 1; d >>= 1) members += __shfl_xor(members, d);
  if (__lane_id() == 0) wsum[t / kWave] = members;
  __syncthreads();
  if (t == 0) {
    unsigned long long c = 0;
    for (int w = 0; w < kMisSmallBlock / kWave; ++w) c += wsum[w];
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(a.host_status + 4), c,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&a.host_status[2], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&a.host_status[1], rounds, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&a.host_status[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

}  // namespace

template <typename OffT>
hipError_t launch_mis_init(const MisArgs<OffT>& a, int grid, hipStream_t stream) {
  hipLaunchKernelGGL((mis_init_kernel<OffT>), dim3(grid), dim3(kBlock), 0, stream, a);
  return hipGetLastError();
}

// step: row entries per look, 2 or 4 (the caller picks it from the graph's
// average degree).
template <typename OffT>
hipError_t launch_mis_round(const MisArgs<OffT>& a, int step, int grid, hipStream_t stream) {
  if (grid < 1 || grid > kMaxGrid || (step != 2 && step != 4)) return hipErrorInvalidValue;
  if (step == 4)
    hipLaunchKernelGGL((mis_round_kernel<OffT, 4>), dim3(grid), dim3(kBlock), 0, stream, a);
  else
    hipLaunchKernelGGL((mis_round_kernel<OffT, 2>), dim3(grid), dim3(kBlock), 0, stream, a);
  return hipGetLastError();
}

template <typename OffT>
hipError_t launch_mis_small(const MisArgs<OffT>& a, int32_t* flags_out, hipStream_t stream) {
  if (a.n > kMisSmall) return hipErrorInvalidValue;
  hipLaunchKernelGGL((mis_small_kernel<OffT>), dim3(1), dim3(kMisSmallBlock), 0, stream, a,
                     flags_out);
  return hipGetLastError();
}

template <typename OffT>
const void* mis_round_symbol(int step) {
  return step == 4 ? reinterpret_cast<const void*>(&mis_round_kernel<OffT, 4>)
                   : reinterpret_cast<const void*>(&mis_round_kernel<OffT, 2>);
}

template <typename OffT>
hipError_t launch_mis_output(const MisArgs<OffT>& a, int32_t* flags_out, int grid,
                             hipStream_t stream) {
  if (grid < 1 || grid > kMaxGrid) return hipErrorInvalidValue;
  hipLaunchKernelGGL((mis_output_kernel<OffT>), dim3(grid), dim3(kBlock), 0, stream, a,
                     flags_out);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((mis_count_kernel<OffT>), dim3(1), dim3(kBlock), 0, stream, a, grid);
  return hipGetLastError();
}

#define PBBS_MIS_INSTANTIATE(OffT)                                                             \
  template hipError_t launch_mis_init<OffT>(const MisArgs<OffT>&, int, hipStream_t);           \
  template hipError_t launch_mis_round<OffT>(const MisArgs<OffT>&, int, int, hipStream_t);     \
  template hipError_t launch_mis_small<OffT>(const MisArgs<OffT>&, int32_t*, hipStream_t);     \
  template const void* mis_round_symbol<OffT>(int);                                            \
  template hipError_t launch_mis_output<OffT>(const MisArgs<OffT>&, int32_t*, int, hipStream_t);
PBBS_MIS_INSTANTIATE(uint32_t)
PBBS_MIS_INSTANTIATE(int64_t)
#undef PBBS_MIS_INSTANTIATE

}  // namespace pbbs
