// small.hip -- many levels of a traversal with small frontiers in one launch.
//
// A level of the general path is a compaction over the whole bitmap, an
// expansion over the whole chip and a host round trip: 45-65 us whatever the
// frontier holds.  Traversals of high diameter (paths, grids, the tails of
// any BFS) have hundreds or thousands of levels of a few vertices; there one
// block runs level after level with its queue in LDS and no launch, pass
// over n or host round trip between levels.
//
// One 1024-thread block (one CU: its barriers cost some 0.1 us, a barrier
// across the chip's eight XCDs several us).  A level is three dependent
// rounds of memory accesses:
//   1. degree, first-record address (and, for values, the current value) of
//      every queued vertex, then a block scan of the degrees;
//   2. the records, one edge per thread and step (four steps in flight),
//      each edge's entry found by a binary search of the scanned degrees;
//   3. the returning atomic on the destination (visited bit or value); the
//      winners append to the queue, one LDS atomic per wave.
// Bound: the latency of those rounds, about 0.8 us each: a 2,001-vertex path
// behind a 19,999-leaf star takes 5.4 ms (2.7 us a level) against 109 ms by
// the general path, SSSP on a 500 x 500 grid (2,260 rounds, and as many
// buckets again) 13.3 ms against 174.
//
// The block gives up (and the general path takes over) when a frontier has
// more than SPARSE_MAX vertices (its LDS holds 24 bytes of each) or SMALL_EDGES
// edges, or would find more than SMALL_NEW vertices: past that the chip
// finishes a level sooner than one CU does.
#include "internal.hpp"
#include "scan.hpp"

namespace thv {

namespace {

constexpr int SB = 1024;
constexpr uint32_t QCAP = SPARSE_MAX;
constexpr uint32_t UNR = 4;  // edges per thread in flight

__device__ __forceinline__ uint32_t ld_agent(const uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct SmallShared {
  unsigned long long ep[QCAP];  // address of the entry's record for edge 0 of the level
  uint32_t pre[QCAP];           // first edge of the entry
  uint32_t cval[QCAP];          // VAL: the entry's value
  uint32_t id[QCAP];            // queued vertices (this level's, then the next one's)
  uint32_t nval[QCAP];          // VAL: the values they were queued with
  unsigned long long part[SB / 64];
  unsigned long long sum[12];
  uint32_t cnt, over, fars, lo;
};

// One thread's vertices and edges of the frontier left in the bitmap (host,
// HBM): summed once at the end, since LDS adds to one address take turns.
struct Left {
  uint32_t nf[2] = {0, 0};
  unsigned long long mf[2] = {0, 0};
};

// Runs of lanes whose ids share a bitmap word.  One CU's atomics on one word
// take turns, 7-8 ns each (on different words 0.7-2): a sorted list of
// consecutive ids is best sent as one atomic a run (BFS from the hub of a star
// of 20,000 leaves: 298 us in this kernel with an atomic a leaf, 50 so; leaves
// spread over 4M ids 87 either way).
struct Runs {
  bool few;             // few enough runs to be worth the shuffles (wave-uniform)
  uint32_t start, end;  // this lane's run
};
__device__ __forceinline__ Runs runs_of(uint32_t word) {
  const uint32_t lane = lane_id(), before = __shfl_up(word, 1, 64);
  const unsigned long long heads = wave_ballot(lane == 0 || word != before);
  const unsigned long long upto = heads & (~0ull >> (63 - lane));
  const unsigned long long after = heads & ~(~0ull >> (63 - lane));
  Runs r;
  r.few = __popcll(heads) <= 16;
  r.start = 63 - __builtin_clzll(upto);
  r.end = after ? (uint32_t)__builtin_ctzll(after) - 1 : 63u;
  return r;
}
// OR of x over the lanes of the run up to this one.
__device__ __forceinline__ uint32_t run_or(uint32_t x, const Runs &r) {
  const uint32_t lane = lane_id();
#pragma unroll
  for (uint32_t d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d, 64);
    if (lane >= r.start + d) x |= y;
  }
  return x;
}

// The vertices of the lanes with `on` to the bitmap (BFS: counted).  Every
// lane of the wave takes part.
template <bool VAL>
__device__ __forceinline__ void leave(const SmallArgs &a, Left &left, bool on, uint32_t w) {
  const Runs r = runs_of(on ? w >> 5 : 0xFFFFFFFFu);
  uint32_t bits = on ? 1u << (w & 31) : 0u;
  bool send = on;
  if (r.few) {
    bits = run_or(bits, r);
    send = on && lane_id() == r.end;
  }
  if (send) atomicOr(&a.front[w >> 5], bits);
  if (VAL || !on) return;
  const uint32_t d = a.deg[w];
  const bool hbm = !a.split || ((a.rbit[w >> 5] >> (w & 31)) & 1u);
  left.nf[0] += d && !hbm;
  left.nf[1] += d && hbm;
  left.mf[0] += hbm ? 0u : d;
  left.mf[1] += hbm ? d : 0u;
}

// Appends (w, nv) for the lanes with `take`; past the queue's capacity the
// vertex goes to the bitmap and the block ends after this level.
template <bool VAL>
__device__ __forceinline__ void push(const SmallArgs &a, SmallShared &s, Left &left, bool take,
                                     uint32_t w, uint32_t nv) {
  const unsigned long long b = wave_ballot(take);
  if (!b) return;
  uint32_t at = 0;
  if (lane_id() == 0) at = atomicAdd(&s.cnt, (uint32_t)__popcll(b));
  at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) + lanes_below(b);
  if (take && at < QCAP) {
    s.id[at] = w;
    if (VAL) s.nval[at] = nv;
  }
  const bool out = take && at >= QCAP;
  if (!wave_ballot(out)) return;
  if (out) s.over = 1;
  leave<VAL>(a, left, out, w);
}

// Appends (w, nv) to the far list `to` (counted in s.fars).
__device__ __forceinline__ void push_far(const SmallArgs &a, SmallShared &s,
                                         unsigned long long *to, bool take, uint32_t w,
                                         uint32_t nv) {
  const unsigned long long b = wave_ballot(take);
  if (!b) return;
  uint32_t at = 0;
  if (lane_id() == 0) at = atomicAdd(&s.fars, (uint32_t)__popcll(b));
  at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) + lanes_below(b);
  if (!take) return;
  if (at < a.far_cap) {
    to[at] = (unsigned long long)nv << 32 | w;
  } else {
    s.over = 1;
    atomicOr(&a.front[w >> 5], 1u << (w & 31));
  }
}

// ALGO: A_BFS, A_CC or A_SSSP.  BFS: visited bits, values = level.  CC and
// SSSP (VAL): an improvement queues (vertex, value); an entry whose value
// was lowered again since is stale (its newer entry is queued too) and is
// skipped, so every improvement is relaxed at most once.  SSSP keeps the
// improvements at or above the bucket bound in a far list and opens the next
// bucket from it, as the general loop does from its pending bitmap.
template <int ALGO, int REC>
__global__ void __launch_bounds__(SB) k_small(SmallArgs a) {
  constexpr bool VAL = ALGO != A_BFS;
  constexpr bool FAR = ALGO == A_SSSP;
  __shared__ SmallShared s;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (tid < 12) s.sum[tid] = 0;
  if (tid == 0) {
    s.cnt = s.over = s.fars = 0;
    s.lo = 0xFFFFFFFFu;
  }
  __syncthreads();
  uint32_t thr = a.thr;
  unsigned long long *fin = a.far[0], *fout = a.far[1];
  uint32_t F = 0;
  unsigned long long state = 0;
  const uint32_t count = a.list ? *a.count : 1u;
  bool refused = false;
  Left rest;
  if (a.list && count > (FAR ? a.far_cap : QCAP)) {
    refused = true;
  } else if (!a.list) {
    F = 1;
    if (tid == 0) {
      s.id[0] = a.src;
      if (VAL) s.nval[0] = ld_agent(&a.val[a.src]);
      atomicAnd(&a.front[a.src >> 5], ~(1u << (a.src & 31)));
    }
  } else {
    // how many of the listed vertices are near (all of them without a far
    // list); more than the queue holds: nothing is touched
    if (FAR) {
      uint32_t c = 0;
      for (uint32_t i = tid; i < count; i += SB) c += a.val[a.list[i]] < thr;
      c = wave_sum(c);
      if (lane == 0) atomicAdd(&s.cnt, c);
      __syncthreads();
      refused = s.cnt > QCAP;
      __syncthreads();
      if (tid == 0) s.cnt = 0;
      __syncthreads();
    }
    if (!refused) {
      const uint32_t upto = (count + SB - 1) / SB * SB;
      for (uint32_t i = tid; i < upto; i += SB) {
        const bool in = i < count;
        const uint32_t v = in ? a.list[i] : 0u;
        const uint32_t x = VAL && in ? a.val[v] : 0u;
        if (in) atomicAnd(&a.front[v >> 5], ~(1u << (v & 31)));
        // the top-down loop leaves a frontier's level to its compaction
        if (!VAL && in) a.val[v] = a.level_value - 1;
        const bool near = in && (!FAR || x < thr);
        push<VAL>(a, s, rest, near, v, x);
        if (FAR) push_far(a, s, fin, in && !near, v, x);
      }
      __syncthreads();
      F = s.cnt;
    }
  }
  __syncthreads();
  uint32_t nfar = s.fars, levels = 0, lv = a.level_value, stamp = a.stamp;
  // without a near vertex the loop starts with the bucket step, which resets
  // s.fars: every wave has its copy first
  __syncthreads();
  uint64_t left = a.unvisited;
  // this thread's share of the totals over all levels
  unsigned long long tn = 0, te[2] = {0, 0}, tt = 0, last = 0;
  while (!refused) {
    if (F == 0 && FAR && nfar) {
      // the next bucket: the least value still current in the far list
      uint32_t lo = 0xFFFFFFFFu;
      for (uint32_t i = tid; i < nfar; i += SB) {
        const unsigned long long x = fin[i];
        if (ld_agent(&a.val[(uint32_t)x]) == (uint32_t)(x >> 32)) lo = min(lo, (uint32_t)(x >> 32));
      }
#pragma unroll
      for (int d = 32; d >= 1; d >>= 1) lo = min(lo, (uint32_t)__shfl_xor((int)lo, d, 64));
      if (tid == 0) s.cnt = s.fars = 0;
      if (lane == 0 && lo != 0xFFFFFFFFu) atomicMin(&s.lo, lo);
      __syncthreads();
      lo = s.lo;
      if (lo == 0xFFFFFFFFu) break;  // nothing pending
      const uint64_t t = (uint64_t)lo + a.delta;
      thr = t < 0xFFFFFFFFull ? (uint32_t)t : 0xFFFFFFFFu;
      const uint32_t upto = (nfar + SB - 1) / SB * SB;
      for (uint32_t i = tid; i < upto; i += SB) {
        const unsigned long long x = i < nfar ? fin[i] : 0ull;
        const uint32_t w = (uint32_t)x, nv = (uint32_t)(x >> 32);
        const bool cur = i < nfar && ld_agent(&a.val[w]) == nv;
        push<VAL>(a, s, rest, cur && nv < thr, w, nv);
        push_far(a, s, fout, cur && nv >= thr, w, nv);
      }
      __syncthreads();
      F = min(s.cnt, QCAP);
      nfar = min(s.fars, a.far_cap);
      if (tid == 0) s.lo = 0xFFFFFFFFu;
      unsigned long long *x = fin;
      fin = fout;
      fout = x;
      __syncthreads();
      if (s.over) {
        state = 1;
        break;
      }
    }
    if (F == 0) break;
    // round 1: the entries' lists, scanned
    unsigned long long E = 0, nz = 0;
    for (uint32_t r = 0; r < F; r += SB) {
      const uint32_t i = r + tid;
      uint32_t d = 0;
      unsigned long long p = 0;
      if (i < F) {
        const uint32_t id = s.id[i];
        d = a.deg[id];
        p = a.eptr[id];
        if (VAL) {
          const uint32_t x = s.nval[i];
          if (ld_agent(&a.val[id]) != x) d = 0;
          s.cval[i] = x;
        }
      }
      const unsigned long long inc = wave_incl_scan((unsigned long long)d);
      if (lane == 63) s.part[wv] = inc;
      __syncthreads();
      unsigned long long before = E;
      const uint32_t nw = min((F - r + 63) / 64, (uint32_t)(SB / 64));
      for (uint32_t k = 0; k < nw; k++) {
        const unsigned long long x = s.part[k];
        before += k < wv ? x : 0ull;
        E += x;
      }
      if (i < F) {
        const unsigned long long b = before + inc - d;
        s.pre[i] = (uint32_t)b;
        s.ep[i] = p - b * REC;
      }
      nz += __popcll(wave_ballot(d != 0));
      __syncthreads();
    }
    if (E == 0) {
      // nothing to expand; a far list may hold more
      F = 0;
      if (FAR && nfar) continue;
      break;
    }
    left -= min<uint64_t>(left, E);
    bool wide = E > a.edge_max ||
                (ALGO == A_BFS && (double)E * (double)left > (double)a.new_max * (double)a.edges);
    if (ALGO == A_BFS && a.split && !wide && 2 * E > a.edge_max) {  // host records count twice
      unsigned long long eh = 0;
      for (uint32_t i = tid; i < F; i += SB) {
        const uint32_t id = s.id[i], d = (i + 1 < F ? s.pre[i + 1] : (uint32_t)E) - s.pre[i];
        if (d && !((a.rbit[id >> 5] >> (id & 31)) & 1u)) eh += d;
      }
      eh = wave_sum(eh);
      if (lane == 0 && eh) atomicAdd(&s.sum[9], eh);
      __syncthreads();
      wide = E + s.sum[9] > a.edge_max;
      __syncthreads();
      if (tid == 0) s.sum[9] = 0;
    }
    if (wide || levels == a.max_levels ||
        (a.ratio > 0 && (double)E * a.ratio > (double)left)) {
      state = 1;
      break;
    }
    // this level's share of the totals (a host list's edges are summed per
    // entry: the scanned starts give the degrees)
    if (lane == 0) tn += nz;
    if (tid == 0) last = 0;
    if (a.split) {
      for (uint32_t i = tid; i < F; i += SB) {
        const uint32_t d = (i + 1 < F ? s.pre[i + 1] : (uint32_t)E) - s.pre[i];
        if (!d) continue;
        const uint32_t id = s.id[i];
        te[(a.rbit[id >> 5] >> (id & 31)) & 1u] += d;
        const uint32_t pt = a.vpart[id];
        if (!a.pres[pt] && atomicExch(&a.ptouch[pt], stamp) != stamp) tt++;
      }
    } else if (tid == 0) {
      te[1] += E;
    }
    if (lane == 0) atomicAdd(&s.sum[4], nz);
    __syncthreads();
    if (tid == 0) {
      last = s.sum[4];
      s.sum[4] = 0;
      s.cnt = 0;
      s.over = 0;
    }
    const uint32_t far0 = nfar;
    if (FAR && tid == 0) s.fars = far0;
    __syncthreads();
    // rounds 2 and 3: the edges
    const uint32_t Eu = (uint32_t)E;
    for (uint32_t e0 = 0; e0 < Eu; e0 += SB * UNR) {
      uint32_t w[UNR], x[UNR];
#pragma unroll
      for (uint32_t j = 0; j < UNR; j++) {
        const uint32_t e = e0 + j * SB + tid;
        w[j] = 0xFFFFFFFFu;
        x[j] = 0;
        if (e < Eu) {
          // the last entry that starts at or before e
          uint32_t lo = 0, n = F;
          while (n > 1) {
            const uint32_t h = n >> 1;
            if (s.pre[lo + h] <= e) lo += h;
            n -= h;
          }
          const unsigned long long at = s.ep[lo] + (unsigned long long)e * REC;
          typedef const __attribute__((address_space(1))) uint32_t *gp;
          w[j] = *reinterpret_cast<gp>(at);
          if (ALGO == A_SSSP) x[j] = *reinterpret_cast<gp>(at + 4);
          if (VAL) {
            const unsigned long long nv = (unsigned long long)s.cval[lo] + x[j];
            x[j] = nv < 0xFFFFFFFFull ? (uint32_t)nv : 0xFFFFFFFFu;
          }
        }
      }
      uint32_t old[UNR];
      if (ALGO == A_BFS) {
        // A narrow level is bound by the latency of its steps; a wide one tests
        // the word first and sends one atomic for a run of lanes on one word
        // (its last lane's, with the run's bits; a lane's bit that an earlier
        // lane of the run has too is that lane's).
        bool won[UNR];
        if (Eu > SB) {
          Runs r[UNR];
          uint32_t mine[UNR];  // few runs: the bits of the run's earlier lanes
#pragma unroll
          for (uint32_t j = 0; j < UNR; j++)
            old[j] = w[j] != 0xFFFFFFFFu ? a.vis[w[j] >> 5] : 0xFFFFFFFFu;
#pragma unroll
          for (uint32_t j = 0; j < UNR; j++) {
            const uint32_t bit = 1u << (w[j] & 31);
            won[j] = !(old[j] & bit);
            r[j] = runs_of(w[j] >> 5);
            uint32_t bits = won[j] ? bit : 0u;
            bool send = won[j];
            mine[j] = 0;
            if (r[j].few) {
              bits = run_or(bits, r[j]);
              mine[j] = __shfl_up(bits, 1, 64);
              if (lane == r[j].start) mine[j] = 0;
              send = lane == r[j].end && bits;
            }
            if (send) old[j] = atomicOr(&a.vis[w[j] >> 5], bits);
          }
#pragma unroll
          for (uint32_t j = 0; j < UNR; j++) {
            if (r[j].few) old[j] = __shfl(old[j], r[j].end, 64) | mine[j];
            won[j] = won[j] && !(old[j] & (1u << (w[j] & 31)));
          }
        } else {
#pragma unroll
          for (uint32_t j = 0; j < UNR; j++) {
            old[j] = 0xFFFFFFFFu;
            if (w[j] != 0xFFFFFFFFu) old[j] = atomicOr(&a.vis[w[j] >> 5], 1u << (w[j] & 31));
          }
#pragma unroll
          for (uint32_t j = 0; j < UNR; j++) won[j] = !(old[j] & (1u << (w[j] & 31)));
        }
#pragma unroll
        for (uint32_t j = 0; j < UNR; j++) {
          if (won[j]) a.val[w[j]] = lv;
          push<VAL>(a, s, rest, won[j], w[j], 0);
        }
      } else {
#pragma unroll
        for (uint32_t j = 0; j < UNR; j++)
          old[j] = w[j] != 0xFFFFFFFFu ? ld_agent(&a.val[w[j]]) : 0u;
#pragma unroll
        for (uint32_t j = 0; j < UNR; j++)
          if (x[j] < old[j]) old[j] = atomicMin(&a.val[w[j]], x[j]);
#pragma unroll
        for (uint32_t j = 0; j < UNR; j++) {
          const bool won = x[j] < old[j];
          const bool near = won && (!FAR || x[j] < thr);
          push<VAL>(a, s, rest, near, w[j], x[j]);
          if (FAR) push_far(a, s, fin, won && !near, w[j], x[j]);
        }
      }
    }
    __syncthreads();
    F = min(s.cnt, QCAP);
    if (FAR) nfar = min(s.fars, a.far_cap);
    const bool over = s.over != 0;
    levels++;
    lv++;
    stamp++;
    __syncthreads();
    if (over) {
      state = 1;
      break;
    }
  }
  // the frontier left goes to the bitmap, with its sums (a stale entry's
  // vertex is there through its newer entry)
  __syncthreads();
  if (state) {
    for (uint32_t i = tid; i < (F + SB - 1) / SB * SB; i += SB) {
      const uint32_t id = i < F ? s.id[i] : 0u;
      leave<VAL>(a, rest, i < F && (!VAL || ld_agent(&a.val[id]) == s.nval[i]), id);
    }
    if (FAR) {
      for (uint32_t i = tid; i < nfar; i += SB) {
        const unsigned long long x = fin[i];
        const uint32_t w = (uint32_t)x;
        if (ld_agent(&a.val[w]) == (uint32_t)(x >> 32)) atomicOr(&a.front[w >> 5], 1u << (w & 31));
      }
    }
  }
  tn = wave_sum(tn);
  te[0] = wave_sum(te[0]);
  te[1] = wave_sum(te[1]);
  tt = wave_sum(tt);
  if (state && !VAL) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const uint32_t nf = wave_sum(rest.nf[i]);
      const unsigned long long mf = wave_sum(rest.mf[i]);
      if (lane == 0 && nf) {
        atomicAdd(&s.sum[i], (unsigned long long)nf);
        atomicAdd(&s.sum[2 + i], mf);
      }
    }
  }
  if (lane == 0) {
    if (tn) atomicAdd(&s.sum[5], tn);
    if (te[0]) atomicAdd(&s.sum[6], te[0]);
    if (te[1]) atomicAdd(&s.sum[7], te[1]);
    if (tt) atomicAdd(&s.sum[8], tt);
  }
  __syncthreads();
  if (tid == 0) {
    SmallOut o;
    o.state = refused ? 2ull : state;
    o.levels = levels;
    o.thr = thr;
    o.last_nf = last;
    for (int i = 0; i < 2; i++) {
      o.nf[i] = s.sum[i];
      o.mf[i] = s.sum[2 + i];
      o.edges[i] = s.sum[6 + i];
    }
    o.vertices = s.sum[5];
    o.touched = s.sum[8];
    *a.out = o;
    if (a.list) *a.count = 0;  // for the next listing
    __threadfence_system();
  }
}

}  // namespace

void launch_small(Graph &g, Algo algo, const SmallArgs &a, hipStream_t s) {
  if (!a.val || !a.front || !a.out || (algo == A_BFS && !a.vis) || (a.list && !a.count) ||
      (algo == A_SSSP && (!a.far[0] || !a.far[1])))
    fail(THV_ESTATE, "small-frontier launch: missing array");
  if (!a.list && a.src >= g.n) fail(THV_EINVAL, "vertex out of range");
  const bool r8 = g.rec == 8;
  switch (algo) {
    case A_BFS:
      if (r8) hipLaunchKernelGGL((k_small<A_BFS, 8>), dim3(1), dim3(SB), 0, s, a);
      else hipLaunchKernelGGL((k_small<A_BFS, 4>), dim3(1), dim3(SB), 0, s, a);
      break;
    case A_CC:
      if (r8) hipLaunchKernelGGL((k_small<A_CC, 8>), dim3(1), dim3(SB), 0, s, a);
      else hipLaunchKernelGGL((k_small<A_CC, 4>), dim3(1), dim3(SB), 0, s, a);
      break;
    case A_SSSP:
      if (!r8) fail(THV_ENOTSUP, "SSSP needs 8-byte {dst, weight} records");
      hipLaunchKernelGGL((k_small<A_SSSP, 8>), dim3(1), dim3(SB), 0, s, a);
      break;
    default: fail(THV_EINVAL, "no small-frontier kernel for this algorithm");
  }
  HIPC(hipGetLastError());
}

}  // namespace thv
