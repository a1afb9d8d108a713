// batch.hip -- multi-source BFS / SSSP engine (multi.hpp) and thv_batch.
//
// No reference counterpart: the reference runs one source per process
// (src/main.cu:152-220).  The per-level pipeline reuses the split store and
// the partition compaction of the single-source path; only the expansion
// kernels and the per-vertex state differ.
#include <algorithm>

#include "chunk.hpp"
#include "multi.hpp"

namespace thv {

namespace {

constexpr int MBS = 256;
constexpr int ACC_HASH = 0, ACC_CNT = 64, ACC_LM = 128, RES_HASH = 129, RES_CNT = 193,
              RES_DEPTH = 257, ACC_LONG = 321, ACC_MU = 322, ACC_SCAN_HOST = 323,
              ACC_SCAN_HBM = 324, ACC_MF = 325, ACC_WORDS = 384;
// bottom-up levels: lists up to this length are scanned by one lane, longer
// ones by a group of BU_G lanes reading BU_R records each per step (measured
// on the 64-lane R-MAT 25 batch: 8 / 8 / 2 beat 32 / 16 / 2 by 5%; larger
// steps lose more to reads past the early exit than they save in steps; on
// R-MAT 22 both kernels' levels take 710 us with 8 / 8 / 2, 700 with 8 / 4 / 4,
// 725 with 4 or 16 / 8 / 2, 740 with 8 / 16 / 2)
constexpr uint32_t BU_SHORT = 8, BU_G = 8, BU_R = 2;
// per-wave LDS buffer of long-list vertices, flushed to the global queue with
// one atomic per flush (an atomic per wave step on one counter serialises)
constexpr uint32_t BU_LQ = 512;

struct MsArgs {
  const uint32_t *qv[2];
  const unsigned long long *qe[2];
  const uint32_t *qc[2];
  const LevelCtr *ctr;
  const uint64_t *eptr;
  const uint32_t *deg;  // BFS: to sum the next frontier's edges, or null
  const unsigned long long *F;
  unsigned long long *N, *seen;
  uint32_t *nb;
  uint32_t *dist;
  uint32_t *full;
  unsigned long long *acc;
  uint64_t n;
  uint32_t L;
  uint32_t level;
  uint32_t voff[64];
  unsigned long long fmask;  // BFS: lanes this expansion pushes (others run bottom-up)
};

// *p |= x where that sets a bit (blocks that bring nothing new do not queue
// for the address).
__device__ __forceinline__ void or_new(unsigned long long *p, unsigned long long x) {
  if (x & ~__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicOr(p, x);
}

// BFS: lane per edge, lane masks staged per queue entry.
template <int REC, int EPT>
__global__ void __launch_bounds__(MBS) k_ms_bfs(MsArgs a) {
  constexpr uint32_t C = MBS * EPT, NW = C / 32;
  __shared__ uint32_t s_mask[NW], s_pre[NW];
  __shared__ unsigned long long s_base[C + 1];
  __shared__ unsigned long long s_m[C + 1];
  __shared__ unsigned long long s_hash[64];
  __shared__ unsigned int s_cnt[64];
  __shared__ uint32_t s_val[64];
  __shared__ unsigned long long s_lm, s_mf;
  const uint32_t tid = threadIdx.x;
  if (tid < 64) {
    s_hash[tid] = 0;
    s_cnt[tid] = 0;
    s_val[tid] = a.level + 2 - a.voff[tid];
  }
  if (tid == 0) s_lm = s_mf = 0;
  unsigned long long mf = 0;  // edges of the vertices this lane put on the next frontier
  const ChunkSrc cs = chunk_src(a.ctr, C);
  for (uint32_t c = blockIdx.x; c < cs.total; c += gridDim.x) {
    int q;
    uint32_t cc;
    chunk_pick(cs, c, q, cc);
    const ChunkInfo ci = chunk_info<C>(cs, a.qc, q, cc);
    for (uint32_t t = tid; t < NW; t += MBS) s_mask[t] = 0;
    __syncthreads();
    for (uint32_t t = tid; t < ci.nent; t += MBS) {
      const uint32_t v = a.qv[q][ci.i0 + t];
      const unsigned long long b = a.qe[q][ci.i0 + t];
      const unsigned long long s = chunk_rel(b, ci.e0);
      if (s < C) {
        atomicOr(&s_mask[s >> 5], 1u << (s & 31));
        s_base[t] = a.eptr[v] - b * REC;
        s_m[t] = a.F[v] & a.fmask;
      }
    }
    __syncthreads();
    chunk_prefix<NW>(s_mask, s_pre);
    __syncthreads();
    uint32_t dst[EPT], ent[EPT];
#pragma unroll
    for (int j = 0; j < EPT; j++) {
      const uint32_t l = tid + j * MBS;
      dst[j] = 0xFFFFFFFFu;
      ent[j] = 0;
      if (l < ci.len) {
        const uint32_t k = chunk_rank(s_mask, s_pre, l);
        ent[j] = k;
        dst[j] = *reinterpret_cast<const uint32_t *>(s_base[k] + (ci.e0 + l) * REC);
      }
    }
    // phases over all EPT edges, each issuing its memory operations before
    // any result is used: the seen masks (an absent edge reads entry 0 and
    // is ignored), the seen atomics, the next-frontier atomics
    unsigned long long sw[EPT], add[EPT], gain[EPT], on[EPT];
#pragma unroll
    for (int j = 0; j < EPT; j++) sw[j] = a.seen[dst[j] != 0xFFFFFFFFu ? dst[j] : 0];
#pragma unroll
    for (int j = 0; j < EPT; j++) add[j] = dst[j] != 0xFFFFFFFFu ? s_m[ent[j]] & ~sw[j] : 0ull;
#pragma unroll
    for (int j = 0; j < EPT; j++) {
      sw[j] = ~0ull;
      if (add[j]) sw[j] = atomicOr(&a.seen[dst[j]], add[j]);
    }
#pragma unroll
    for (int j = 0; j < EPT; j++) gain[j] = add[j] & ~sw[j];
#pragma unroll
    for (int j = 0; j < EPT; j++) {
      on[j] = ~0ull;
      if (gain[j]) on[j] = atomicOr(&a.N[dst[j]], gain[j]);
    }
#pragma unroll
    for (int j = 0; j < EPT; j++) {
      const uint32_t w = dst[j];
      const unsigned long long gained = gain[j];
      if (!gained) continue;
      if (on[j] == 0ull) {
        atomicOr(&a.nb[w >> 5], 1u << (w & 31));
        if (a.deg) mf += a.deg[w];
      }
      atomicOr(&s_lm, gained);
      unsigned long long g = gained;
      while (g) {
        const int qq = __ffsll((long long)g) - 1;
        g &= g - 1;
        const uint32_t val = s_val[qq];
        atomicAdd(&s_hash[qq], mix64(((unsigned long long)w << 32) | val));
        atomicAdd(&s_cnt[qq], 1u);
        if (a.full) a.full[(uint64_t)qq * a.n + w] = val;
      }
    }
    __syncthreads();
  }
  if (mf) atomicAdd(&s_mf, mf);
  __syncthreads();
  if (tid < 64 && s_cnt[tid]) {
    atomicAdd(&a.acc[ACC_HASH + tid], s_hash[tid]);
    atomicAdd(&a.acc[ACC_CNT + tid], (unsigned long long)s_cnt[tid]);
  }
  if (tid == 0) {
    or_new(&a.acc[ACC_LM], s_lm);
    if (s_mf) atomicAdd(&a.acc[ACC_MF], s_mf);
  }
}

// ---- bottom-up BFS levels (symmetric graphs) ---------------------------------
//
// Every vertex w that some active lane has not reached looks for those lanes
// among its neighbours' frontier masks: N[w] = (OR of F[v] over the
// neighbours v) & ~seen[w], and the scan stops as soon as all of them are
// found.  On a symmetric graph w's out-list is its in-list, so the lanes
// found are exactly those a top-down level hands w.  Each w has one owner
// (a lane, or a group for a long list), so N, seen and the levels need no
// atomics; in the dense middle levels most vertices find all their missing
// lanes within a few records.
struct MsBuArgs {
  const uint64_t *eptr;
  const uint32_t *deg;
  const uint32_t *rbit;
  const unsigned long long *F;
  unsigned long long *N, *seen;
  uint32_t *nb;
  uint32_t *full;
  unsigned long long *acc;
  uint32_t *lq;                 // vertices with long lists, for k_ms_bu_long
  uint64_t n;
  unsigned long long act;       // active lanes
  uint32_t level;
  uint32_t uval;                // the level value when every active lane shares it, else 0
  uint32_t voff[64];
};

// Per-block digest state for bottom-up levels: lane q of every wave keeps
// query q's sum and count in registers.
struct BuDigest {
  unsigned long long h = 0, scan_host = 0, scan_hbm = 0, mu = 0, mf = 0, lm = 0;
  uint32_t cnt = 0;
};

__device__ __forceinline__ unsigned long long readlane64(unsigned long long x, int i) {
  return ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), i)
          << 32) |
         (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, i);
}

// The wave's gains, one vertex per set bit of `who` (a lane mask): lane q
// adds query q's pair (w, value) for each vertex whose gain holds q.  When
// all active lanes share one value (uval != 0), the vertex's owner lane has
// hashed the pair already (hw) and the other lanes only add it.
__device__ __forceinline__ void bu_digest_wave(unsigned long long who, unsigned long long gain,
                                               uint32_t w, unsigned long long hw, uint32_t uval,
                                               uint32_t myval, uint32_t lane, uint32_t *full,
                                               uint64_t n, BuDigest &d) {
  while (who) {
    const int i = __builtin_ctzll(who);
    who &= who - 1;
    const unsigned long long gi = readlane64(gain, i);
    d.lm |= gi;
    if (uval) {
      const unsigned long long hi = readlane64(hw, i);
      if ((gi >> lane) & 1ull) {
        d.h += hi;
        d.cnt++;
        if (full) full[(uint64_t)lane * n + (uint32_t)__builtin_amdgcn_readlane((int)w, i)] = uval;
      }
    } else {
      const uint32_t wi = (uint32_t)__builtin_amdgcn_readlane((int)w, i);
      if ((gi >> lane) & 1ull) {
        d.h += mix64(((unsigned long long)wi << 32) | myval);
        d.cnt++;
        if (full) full[(uint64_t)lane * n + wi] = myval;
      }
    }
  }
}

__device__ __forceinline__ void bu_digest_flush(BuDigest &d, unsigned long long *acc,
                                                unsigned long long *s_hash, unsigned int *s_cnt,
                                                unsigned long long *s_misc) {
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  if (d.cnt) {
    atomicAdd(&s_hash[lane], d.h);
    atomicAdd(&s_cnt[lane], d.cnt);
  }
  if (d.lm) atomicOr(&s_misc[0], d.lm);
  if (d.mu) atomicAdd(&s_misc[1], d.mu);
  if (d.scan_host) atomicAdd(&s_misc[2], d.scan_host);
  if (d.scan_hbm) atomicAdd(&s_misc[3], d.scan_hbm);
  if (d.mf) atomicAdd(&s_misc[4], d.mf);
  __syncthreads();
  if (tid < 64 && s_cnt[tid]) {
    atomicAdd(&acc[ACC_HASH + tid], s_hash[tid]);
    atomicAdd(&acc[ACC_CNT + tid], (unsigned long long)s_cnt[tid]);
  }
  if (tid == 0) {
    or_new(&acc[ACC_LM], s_misc[0]);
    if (s_misc[1]) atomicAdd(&acc[ACC_MU], s_misc[1]);
    if (s_misc[2]) atomicAdd(&acc[ACC_SCAN_HOST], s_misc[2]);
    if (s_misc[3]) atomicAdd(&acc[ACC_SCAN_HBM], s_misc[3]);
    if (s_misc[4]) atomicAdd(&acc[ACC_MF], s_misc[4]);
  }
}

// Frontier masks of R records (0 for absent ones), all loads in flight
// together.  Straight from F, which is zero off the frontier: asking the
// frontier bitmap first spared a fifth of the lines and cost a dependent
// read (64-source BFS, bitmap first / not: R-MAT 20 1.07 / 1.06 ms, 22 1.85 /
// 1.78, 25 10.4 / 9.9, whose F is larger than the last-level cache).
template <uint32_t R>
__device__ __forceinline__ void bu_masks(const MsBuArgs &a, const uint32_t (&v)[R],
                                         unsigned long long (&f)[R]) {
#pragma unroll
  for (uint32_t r = 0; r < R; r++) {
    f[r] = 0;
    if (v[r] != 0xFFFFFFFFu) f[r] = a.F[v[r]];
  }
}

// Copy a wave's LDS buffer of `nl` long-list vertices to the global queue.
__device__ __forceinline__ void bu_lq_flush(const uint32_t *buf, uint32_t nl,
                                            unsigned long long *acc, uint32_t *lq,
                                            uint32_t lane) {
  // the buffer was written by other lanes of this wave
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  uint32_t base = 0;
  if (lane == 0) base = (uint32_t)atomicAdd(&acc[ACC_LONG], (unsigned long long)nl);
  base = (uint32_t)__builtin_amdgcn_readlane((int)base, 0);
  for (uint32_t i = lane; i < nl; i += 64) lq[base + i] = buf[i];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sweep: one wave per 64 consecutive vertices.  Lists of up to BU_SHORT
// records are scanned by their own lane (4 records and 4 frontier masks in
// flight per step); longer ones are queued for k_ms_bu_long.  The next-
// frontier bitmap words come from a ballot, one plain store per half wave.
template <int REC>
__global__ void __launch_bounds__(MBS) k_ms_bu(MsBuArgs a) {
  __shared__ unsigned long long s_hash[64];
  __shared__ unsigned int s_cnt[64];
  __shared__ unsigned long long s_misc[5];
  __shared__ uint32_t s_lq[MBS / 64][BU_LQ];
  __shared__ uint32_t s_nl[MBS / 64], s_base;
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  uint32_t *my_lq = s_lq[tid >> 6];
  uint32_t nl = 0;  // entries in my_lq (wave-uniform)
  if (tid < 64) {
    s_hash[tid] = 0;
    s_cnt[tid] = 0;
  }
  if (tid < 5) s_misc[tid] = 0;
  __syncthreads();
  const uint32_t myval = a.level + 2 - a.voff[lane];
  BuDigest dg;
  const uint64_t nwaves = (uint64_t)gridDim.x * (MBS / 64);
  const uint64_t wstart = ((uint64_t)blockIdx.x * (MBS / 64) + (tid >> 6)) * 64;
  // the next step's degrees and seen masks load while this step's lists are
  // scanned
  uint32_t dn = 0;
  unsigned long long sn = 0;
  if (wstart + lane < a.n) {
    dn = a.deg[wstart + lane];
    sn = a.seen[wstart + lane];
  }
  for (uint64_t w0 = wstart; w0 < a.n; w0 += nwaves * 64) {
    const uint64_t w = w0 + lane, wn = w + nwaves * 64;
    const uint32_t d = dn;
    const unsigned long long sw = sn;
    unsigned long long U = 0;
    if (wn < a.n) {
      dn = a.deg[wn];
      sn = a.seen[wn];
    }
    if (w < a.n && d) U = a.act & ~sw;
    const bool lng = U && d > BU_SHORT;
    unsigned long long acc = 0;
    uint32_t scanned = 0;
    if (U && !lng) {
      const unsigned long long b = a.eptr[w];
      for (uint32_t k = 0; k < d; k += 4) {
        uint32_t v[4];
        unsigned long long f[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          v[j] = 0xFFFFFFFFu;
          if (k + j < d) v[j] = *reinterpret_cast<const uint32_t *>(b + (uint64_t)(k + j) * REC);
        }
        bu_masks<4>(a, v, f);
        acc |= f[0] | f[1] | f[2] | f[3];
        scanned = min(d, k + 4);
        if ((acc & U) == U) break;
      }
    }
    // queue the long lists through the wave's LDS buffer
    const unsigned long long lb = __ballot(lng);
    if (lb) {
      if (lng) my_lq[nl + __popcll(lb & ((1ull << lane) - 1))] = (uint32_t)w;
      nl += (uint32_t)__popcll(lb);
      if (nl > BU_LQ - 64) {
        bu_lq_flush(my_lq, nl, a.acc, a.lq, lane);
        nl = 0;
      }
    }
    const unsigned long long gain = acc & U;
    if (gain) {
      a.N[w] = gain;
      a.seen[w] = sw | gain;
      dg.mf += d;
    }
    if (!lng && (U & ~gain)) dg.mu += d;
    if (scanned) {
      const bool hbm = (a.rbit[w >> 5] >> (w & 31)) & 1u;
      if (hbm) dg.scan_hbm += scanned;
      else dg.scan_host += scanned;
    }
    const unsigned long long gb = __ballot(gain != 0);
    if (lane == 0 && (uint32_t)gb) a.nb[w0 >> 5] = (uint32_t)gb;
    if (lane == 32 && (gb >> 32)) a.nb[(w0 >> 5) + 1] = (uint32_t)(gb >> 32);
    unsigned long long hw = 0;
    if (a.uval && gain) hw = mix64((w << 32) | a.uval);
    bu_digest_wave(gb, gain, (uint32_t)w, hw, a.uval, myval, lane, a.full, a.n, dg);
  }
  // what is left in the waves' buffers: one atomic a block
  if (lane == 0) s_nl[tid >> 6] = nl;
  __syncthreads();
  uint32_t mine = 0, all = 0;
#pragma unroll
  for (uint32_t i = 0; i < MBS / 64; i++) {
    if (i < (tid >> 6)) mine += s_nl[i];
    all += s_nl[i];
  }
  if (tid == 0 && all) s_base = (uint32_t)atomicAdd(&a.acc[ACC_LONG], (unsigned long long)all);
  __syncthreads();
  for (uint32_t i = lane; i < nl; i += 64) a.lq[s_base + mine + i] = my_lq[i];
  bu_digest_flush(dg, a.acc, s_hash, s_cnt, s_misc);
}

// Long lists: a group of BU_G lanes per queued vertex reads BU_G * BU_R
// records per step, ORs their frontier masks across the group and stops
// when every missing lane is found.  Vertices need very different numbers of
// steps, so a group that is done takes the wave's next vertex at once
// instead of waiting for the wave's slowest group: a wave loads up to 64
// queued vertices with their degrees, masks and list addresses (lane i holds
// vertex i) and hands them out by shuffles.  Bound by the scattered reads of
// F.  The widest two levels of 64 sources on R-MAT 22: 305 and 145 us with
// groups that wait, 255 and 134 without waiting, 210 and 118 with the masks
// read directly (bu_masks).
template <int REC>
__global__ void __launch_bounds__(MBS) k_ms_bu_long(MsBuArgs a) {
  __shared__ unsigned long long s_hash[64];
  __shared__ unsigned int s_cnt[64];
  __shared__ unsigned long long s_misc[5];
  const uint32_t tid = threadIdx.x, lane = tid & 63, sub = tid & (BU_G - 1);
  if (tid < 64) {
    s_hash[tid] = 0;
    s_cnt[tid] = 0;
  }
  if (tid < 5) s_misc[tid] = 0;
  __syncthreads();
  const uint32_t myval = a.level + 2 - a.voff[lane];
  const uint64_t total = a.acc[ACC_LONG];
  constexpr uint32_t GPW = 64 / BU_G;  // groups per wave
  BuDigest dg;
  const uint64_t wave = (uint64_t)blockIdx.x * (MBS / 64) + (tid >> 6);
  const uint64_t nwaves = (uint64_t)gridDim.x * (MBS / 64);
  // vertices a wave loads together: its share of a short queue
  const uint32_t B = (uint32_t)min((uint64_t)64, max((uint64_t)GPW, (total + nwaves - 1) / nwaves));
  uint64_t i0 = wave * B;             // the next vertices to load
  uint32_t nxt = 0, have = 0;         // handed out, loaded (wave-uniform)
  uint32_t bw = 0, bd = 0;            // lane i: loaded vertex i
  unsigned long long bs = 0, bb = 0;
  uint32_t w = 0, d = 0, k = 0;       // the group's vertex
  unsigned long long U = 0, sw = 0, b = 0, acc = 0;
  bool live = false;
  for (;;) {
    const unsigned long long need = __ballot(!live && sub == 0);
    if (need) {
      if (nxt >= have && i0 < total) {
        have = (uint32_t)min((uint64_t)B, total - i0);
        nxt = 0;
        if (lane < have) {
          bw = a.lq[i0 + lane];
          bd = a.deg[bw];
          bs = a.seen[bw];
          bb = a.eptr[bw];
        }
        i0 += nwaves * B;
      }
      const uint32_t slot =
          nxt + (uint32_t)__popcll(need & ((1ull << (lane & ~(BU_G - 1))) - 1));
      const uint32_t from = slot & 63;
      const uint32_t nw = __shfl(bw, from), nd = __shfl(bd, from);
      const unsigned long long ns = __shfl(bs, from), nb = __shfl(bb, from);
      if (!live && slot < have) {
        live = true;
        w = nw;
        d = nd;
        sw = ns;
        b = nb;
        U = a.act & ~sw;
        acc = 0;
        k = 0;
      }
      nxt = min(nxt + (uint32_t)__popcll(need), have);
      if (!__ballot(live)) break;  // nothing in flight, so nothing was left to hand out
    }
    bool fin = false;
    if (live) {
      uint32_t v[BU_R];
      unsigned long long f[BU_R];
#pragma unroll
      for (uint32_t r = 0; r < BU_R; r++) {
        const uint32_t e = k + r * BU_G + sub;
        v[r] = 0xFFFFFFFFu;
        if (e < d) v[r] = *reinterpret_cast<const uint32_t *>(b + (uint64_t)e * REC);
      }
      bu_masks<BU_R>(a, v, f);
      unsigned long long x = f[0];
#pragma unroll
      for (uint32_t r = 1; r < BU_R; r++) x |= f[r];
#pragma unroll
      for (uint32_t o = BU_G / 2; o; o >>= 1) x |= __shfl_xor(x, o, BU_G);
      acc |= x;
      k = min(d, k + BU_G * BU_R);
      fin = k == d || (acc & U) == U;
    }
    const bool leader = fin && sub == 0;
    const unsigned long long gain = acc & U;
    if (leader) {
      if (gain) {
        a.N[w] = gain;
        a.seen[w] = sw | gain;
        atomicOr(&a.nb[w >> 5], 1u << (w & 31));
        dg.mf += d;
      }
      if (U & ~gain) dg.mu += d;
      const bool hbm = (a.rbit[w >> 5] >> (w & 31)) & 1u;
      if (hbm) dg.scan_hbm += k;
      else dg.scan_host += k;
    }
    if (fin) live = false;
    const unsigned long long who = __ballot(leader && gain != 0);
    if (who) {
      unsigned long long hw = 0;
      if (a.uval && leader) hw = mix64(((unsigned long long)w << 32) | a.uval);
      bu_digest_wave(who, gain, w, hw, a.uval, myval, lane, a.full, a.n, dg);
    }
  }
  bu_digest_flush(dg, a.acc, s_hash, s_cnt, s_misc);
}

// Bits of x at the even places of 64.
__device__ __forceinline__ unsigned long long spread_bits(uint32_t x) {
  unsigned long long v = x;
  v = (v | (v << 16)) & 0x0000FFFF0000FFFFull;
  v = (v | (v << 8)) & 0x00FF00FF00FF00FFull;
  v = (v | (v << 4)) & 0x0F0F0F0F0F0F0F0Full;
  v = (v | (v << 2)) & 0x3333333333333333ull;
  v = (v | (v << 1)) & 0x5555555555555555ull;
  return v;
}

// SSSP: a group of G lanes relaxes an edge, lane q of the group query q.  A
// wave owns 64 consecutive work-space edges at a time: each lane loads one
// record (coalesced) and ranks it once; the groups then take the 64 edges in
// turn, SSSP_U each in flight.  Bound by the distance rows (64 sources on R-MAT
// 20: 75M edges of two 256-byte rows, one of them mostly in L1).
// - Up to 32 queries: 8, 4 or 2 edges at once instead of idle lanes, ms a call
//   on R-MAT 20 with a whole wave an edge / the least group that holds them: 1
//   source 2.8 / 1.3, 8 4.4 / 1.8, 16 5.0 / 2.4, 32 5.3 / 3.4.
// - More, an even number (rows then start at 8-byte addresses): PAIR, two
//   queries a lane and two edges at once, half the load instructions.  64
//   sources on R-MAT 14 1.09 -> 1.05, 20 5.76 -> 4.81, 22 18.6 -> 15.5.
// - More, an odd number: a wave an edge.  Its edges are broadcast with
//   readlane, and a source's row is read once per run of its edges.
// SSSP_U: 8 need 103 registers and 2 hide too little (R-MAT 20, 64 sources, with
// 2 / 4 / 8: 5.1 / 4.8 / 5.3 ms).
// Chunks of 1,024 edges (4 waves x 4 x 64), or of 256 where a level has too
// few to fill the chip with those: a wave's edges are a serial chain (64 take
// 20 us, 256 80).  Batches of 64 sources, ms a call with 1,024 / 256 only
// (some of each since saved elsewhere): R-MAT 14 2.18 / 1.39, 20 8.24 / 7.96,
// 22 24.6 / 25.7; so 256 below 8 large chunks per CU.
constexpr uint32_t SSSP_U = 4;
constexpr uint32_t SSSP_C = 256, SSSP_LARGE = 1024;

template <uint32_t C, uint32_t G, bool PAIR = false>
__global__ void __launch_bounds__(MBS) k_ms_sssp(MsArgs a) {
  constexpr uint32_t NW = C / 32;
  constexpr uint32_t WAVES = MBS / 64, PER_WAVE = C / WAVES;
  __shared__ uint32_t s_mask[NW], s_pre[NW];
  __shared__ unsigned long long s_base[C + 1];
  __shared__ unsigned long long s_m[C + 1];
  __shared__ uint32_t s_v[C + 1];
  __shared__ unsigned long long s_lm;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const uint32_t L = a.L;
  const uint32_t sub = lane & (G - 1), eg = lane / G;
  const bool lane_ok = PAIR ? 2 * sub < L : sub < L;
  unsigned long long lm1 = 0;  // PAIR: the odd queries' (lm: the even ones')
  if (tid == 0) s_lm = 0;
  unsigned long long lm = 0;  // lanes (of all groups) improved somewhere
  const ChunkSrc cs = chunk_src(a.ctr, C);
  for (uint32_t c = blockIdx.x; c < cs.total; c += gridDim.x) {
    int q;
    uint32_t cc;
    chunk_pick(cs, c, q, cc);
    const ChunkInfo ci = chunk_info<C, C / SSSP_C>(cs, a.qc, q, cc);
    for (uint32_t t = tid; t < NW; t += MBS) s_mask[t] = 0;
    __syncthreads();
    for (uint32_t t = tid; t < ci.nent; t += MBS) {
      const uint32_t v = a.qv[q][ci.i0 + t];
      const unsigned long long b = a.qe[q][ci.i0 + t];
      const unsigned long long s = chunk_rel(b, ci.e0);
      if (s < C) {
        atomicOr(&s_mask[s >> 5], 1u << (s & 31));
        s_base[t] = a.eptr[v] - b * 8;
        s_m[t] = a.F[v];
        s_v[t] = v;
      }
    }
    __syncthreads();
    chunk_prefix<NW>(s_mask, s_pre);
    __syncthreads();
    for (uint32_t g0 = wv * PER_WAVE; g0 < (wv + 1) * PER_WAVE && g0 < ci.len; g0 += 64) {
      const uint32_t cnt = min(64u, ci.len - g0);
      // lane j holds edge g0 + j: destination, weight, entry
      uint32_t my_w = 0, my_wt = 0, my_k = 0;
      if (lane < cnt) {
        my_k = chunk_rank(s_mask, s_pre, g0 + lane);
        const uint2 r = *reinterpret_cast<const uint2 *>(s_base[my_k] + (ci.e0 + g0 + lane) * 8);
        my_w = r.x;
        my_wt = r.y;
      }
      uint32_t blo = 0, bhi = 0;  // lane j: the queries that edge g0 + j improved
      if (PAIR) {
        // lane q of 32 takes queries 2q and 2q + 1 of one of two edges
        uint32_t be = 0, bo = 0;  // lane j: edge g0 + j's even and odd queries
        for (uint32_t j0 = 0; j0 * 2 < cnt; j0 += SSSP_U) {
          uint32_t w[SSSP_U], wt[SSSP_U], m[SSSP_U];
          uint2 ds[SSSP_U], dw[SSSP_U];
#pragma unroll
          for (int j = 0; j < (int)SSSP_U; j++) {
            const uint32_t e = (j0 + j) * 2 + eg;
            w[j] = __shfl(my_w, e);
            wt[j] = __shfl(my_wt, e);
            const uint32_t k = __shfl(my_k, e);
            m[j] = e < cnt && lane_ok ? (uint32_t)(s_m[k] >> (2 * sub)) & 3u : 0u;
            ds[j] = dw[j] = make_uint2(0, 0);
            if (m[j]) {
              ds[j] = *reinterpret_cast<const uint2 *>(&a.dist[(uint64_t)s_v[k] * L + 2 * sub]);
              dw[j] = *reinterpret_cast<const uint2 *>(&a.dist[(uint64_t)w[j] * L + 2 * sub]);
            }
          }
#pragma unroll
          for (int j = 0; j < (int)SSSP_U; j++) {
            const unsigned long long n0 = (unsigned long long)ds[j].x + wt[j];
            const unsigned long long n1 = (unsigned long long)ds[j].y + wt[j];
            const bool i0 = (m[j] & 1u) && n0 < dw[j].x, i1 = (m[j] & 2u) && n1 < dw[j].y;
            uint32_t *p = &a.dist[(uint64_t)w[j] * L + 2 * sub];
            if (i0) atomicMin(p, (uint32_t)n0);
            if (i1) atomicMin(p + 1, (uint32_t)n1);
            const unsigned long long b0 = __ballot(i0), b1 = __ballot(i1);
            lm |= b0;
            lm1 |= b1;
            if (lane / 2 == j0 + j) {
              be = (uint32_t)(b0 >> ((lane & 1) * 32));
              bo = (uint32_t)(b1 >> ((lane & 1) * 32));
            }
          }
        }
        const unsigned long long b = spread_bits(be) | (spread_bits(bo) << 1);
        if (b && atomicOr(&a.N[my_w], b) == 0ull) atomicOr(&a.nb[my_w >> 5], 1u << (my_w & 31));
        continue;
      }
      if (G < 64) {
        constexpr uint32_t EPS = 64 / G;  // edges at once
        for (uint32_t j0 = 0; j0 * EPS < cnt; j0 += SSSP_U) {
          uint32_t w[SSSP_U], wt[SSSP_U], ds[SSSP_U], dw[SSSP_U];
          bool on[SSSP_U];
#pragma unroll
          for (int j = 0; j < (int)SSSP_U; j++) {
            const uint32_t e = (j0 + j) * EPS + eg;
            w[j] = __shfl(my_w, e);
            wt[j] = __shfl(my_wt, e);
            const uint32_t k = __shfl(my_k, e);
            on[j] = e < cnt && lane_ok && ((s_m[k] >> sub) & 1ull);
            ds[j] = on[j] ? a.dist[(uint64_t)s_v[k] * L + sub] : 0u;
            dw[j] = on[j] ? a.dist[(uint64_t)w[j] * L + sub] : 0u;
          }
#pragma unroll
          for (int j = 0; j < (int)SSSP_U; j++) {
            const unsigned long long nd = (unsigned long long)ds[j] + wt[j];
            const bool imp = on[j] && nd < dw[j];
            if (imp) atomicMin(&a.dist[(uint64_t)w[j] * L + sub], (uint32_t)nd);
            const unsigned long long b = __ballot(imp);
            lm |= b;
            if (lane / EPS == j0 + j)
              blo = (uint32_t)(b >> (lane % EPS * G)) & (uint32_t)((1ull << (G & 63)) - 1);
          }
        }
        if (blo && atomicOr(&a.N[my_w], (unsigned long long)blo) == 0ull)
          atomicOr(&a.nb[my_w >> 5], 1u << (my_w & 31));
        continue;
      }
      // consecutive edges mostly share their source: its lane mask and
      // distance row are read once per source, not once per edge (a stale
      // row is still a valid distance; an improved source is in N anyway)
      uint32_t kprev = 0xFFFFFFFFu, dprev = 0;
      bool mprev = false;
      for (uint32_t j0 = 0; j0 < cnt; j0 += 8) {
        uint32_t w[8], dw[8], wt[8], kk[8], ds[8];
        bool on[8], nw[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const uint32_t jj = min(j0 + j, cnt - 1);
          w[j] = __builtin_amdgcn_readlane(my_w, jj);
          wt[j] = __builtin_amdgcn_readlane(my_wt, jj);
          kk[j] = __builtin_amdgcn_readlane(my_k, jj);
          nw[j] = kk[j] != (j ? kk[j - 1] : kprev);  // a new source (uniform)
        }
        // the new sources' lane masks, then their rows and the destinations',
        // all in flight together
#pragma unroll
        for (int j = 0; j < 8; j++) {
          if (nw[j]) mprev = lane_ok && ((s_m[kk[j]] >> lane) & 1ull);
          on[j] = j0 + j < cnt && mprev;
        }
        kprev = kk[7];
#pragma unroll
        for (int j = 0; j < 8; j++) {
          ds[j] = 0u;
          if (nw[j] && on[j]) ds[j] = a.dist[(uint64_t)s_v[kk[j]] * L + lane];
        }
#pragma unroll
        for (int j = 0; j < 8; j++) dw[j] = on[j] ? a.dist[(uint64_t)w[j] * L + lane] : 0u;
        // An improvement is judged against the row just read, so the
        // atomicMin needs no result and the 8 edges' atomics stay in flight
        // together.  A lane whose atomicMin loses to a smaller concurrent
        // write is marked anyway: that write lowered dist[w] in this level
        // and marks the same (w, lane), so the next frontier is unchanged.
#pragma unroll
        for (int j = 0; j < 8; j++) {
          if (nw[j]) dprev = ds[j];
          bool imp = false;
          if (on[j]) {
            const unsigned long long nd = (unsigned long long)dprev + wt[j];
            if (nd < dw[j]) {
              imp = true;
              atomicMin(&a.dist[(uint64_t)w[j] * L + lane], (uint32_t)nd);
            }
          }
          const unsigned long long b = __ballot(imp);
          lm |= b;
          if (lane == j0 + j) {
            blo = (uint32_t)b;
            bhi = (uint32_t)(b >> 32);
          }
        }
      }
      // the marks of all 64 edges at once, a lane each
      const unsigned long long b = ((unsigned long long)bhi << 32) | blo;
      if (b && atomicOr(&a.N[my_w], b) == 0ull) atomicOr(&a.nb[my_w >> 5], 1u << (my_w & 31));
    }
    __syncthreads();
  }
  for (uint32_t o = 32; o >= G; o >>= 1) lm |= lm >> o;
  if (G < 64) lm &= (1ull << (G & 63)) - 1;
  if (PAIR) lm = spread_bits((uint32_t)lm) | (spread_bits((uint32_t)(lm1 | lm1 >> 32)) << 1);
  if (lane == 0 && lm) atomicOr(&s_lm, lm);
  __syncthreads();
  if (tid == 0) or_new(&a.acc[ACC_LM], s_lm);
}

template <uint32_t C>
void launch_sssp(const MsArgs &a, uint32_t grid, hipStream_t s) {
  if (a.L <= 8) hipLaunchKernelGGL((k_ms_sssp<C, 8>), dim3(grid), dim3(MBS), 0, s, a);
  else if (a.L <= 16) hipLaunchKernelGGL((k_ms_sssp<C, 16>), dim3(grid), dim3(MBS), 0, s, a);
  else if (a.L <= 32) hipLaunchKernelGGL((k_ms_sssp<C, 32>), dim3(grid), dim3(MBS), 0, s, a);
  else if (a.L % 2 == 0)
    hipLaunchKernelGGL((k_ms_sssp<C, 32, true>), dim3(grid), dim3(MBS), 0, s, a);
  else hipLaunchKernelGGL((k_ms_sssp<C, 64>), dim3(grid), dim3(MBS), 0, s, a);
}

struct AdmitArgs {
  uint32_t count;
  uint32_t lane[64];
  uint32_t src[64];
};

__global__ void k_ms_admit(AdmitArgs ad, int algo, unsigned long long *F, uint32_t *fb,
                           unsigned long long *seen, uint32_t *dist, uint32_t L,
                           uint32_t *full, uint64_t n, unsigned long long *acc) {
  const uint32_t i = threadIdx.x;
  if (i >= ad.count) return;
  const uint32_t q = ad.lane[i], s = ad.src[i];
  const unsigned long long bit = 1ull << q;
  if (algo == THV_ALGO_BFS) {
    atomicOr(&seen[s], bit);
    acc[ACC_HASH + q] = mix64(((unsigned long long)s << 32) | 1u);
    acc[ACC_CNT + q] = 1;
    if (full) full[(uint64_t)q * n + s] = 1;
  } else {
    dist[(uint64_t)s * L + q] = 1;
  }
  atomicOr(&F[s], bit);
  atomicOr(&fb[s >> 5], 1u << (s & 31));
}

// Frontier bitmap of some lanes: bit v is set when F[v] holds one of them.
// A wave takes 64 vertices, its ballot is their two bitmap words.
__global__ void __launch_bounds__(MBS) k_ms_lanebits(const unsigned long long *F, uint64_t n,
                                                     unsigned long long lanes, uint32_t *bits) {
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t nw = (uint64_t)gridDim.x * (MBS / 64);
  for (uint64_t w0 = ((uint64_t)blockIdx.x * (MBS / 64) + (threadIdx.x >> 6)) * 64; w0 < n;
       w0 += nw * 64) {
    const uint64_t v = w0 + lane;
    const unsigned long long b = __ballot(v < n && (F[v] & lanes) != 0);
    if (lane < 2) bits[(w0 >> 5) + lane] = (uint32_t)(b >> (32 * lane));
  }
}

// A level's start in one launch: the buffers it writes (last used two levels
// ago) and its counters cleared.  F holds a mask only where fb has a bit, so
// the pass reads n / 8 bytes and writes those masks, not all n.
__global__ void __launch_bounds__(MBS) k_ms_begin(unsigned long long *F, uint32_t *fb,
                                                  uint64_t words, unsigned long long *acc) {
  const uint32_t lane = threadIdx.x & 63;
  if (blockIdx.x == 0 && threadIdx.x < 6)
    acc[threadIdx.x < 1 ? ACC_LM : ACC_LONG + threadIdx.x - 1] = 0;
  const uint64_t nw = (uint64_t)gridDim.x * (MBS / 64);
  for (uint64_t w0 = ((uint64_t)blockIdx.x * (MBS / 64) + (threadIdx.x >> 6)) * 64; w0 < words;
       w0 += nw * 64) {
    const uint32_t x = w0 + lane < words ? fb[w0 + lane] : 0u;
    if (x) fb[w0 + lane] = 0;
    // two words (64 vertices) at a time, one vertex per lane
    for (unsigned long long any = wave_ballot(x != 0); any;) {
      const uint32_t i = (uint32_t)__builtin_ctzll(any) & ~1u;
      any &= ~(3ull << i);
      const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)x, (int)i);
      const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)x, (int)i + 1);
      if (((lane < 32 ? lo : hi) >> (lane & 31)) & 1u) F[(w0 + i) * 32 + lane] = 0;
    }
  }
}

// The level's results to the host: the lanes' counters and the compaction's.
__global__ void __launch_bounds__(MBS) k_ms_publish(const unsigned long long *acc,
                                                    unsigned long long *hacc,
                                                    const LevelCtr *c, LevelCtr *hc) {
  for (uint32_t i = threadIdx.x; i < ACC_WORDS; i += MBS) hacc[i] = acc[i];
  constexpr uint32_t W = (uint32_t)(sizeof(LevelCtr) / 8);
  if (c && threadIdx.x < W)
    reinterpret_cast<unsigned long long *>(hc)[threadIdx.x] =
        reinterpret_cast<const unsigned long long *>(c)[threadIdx.x];
  __threadfence_system();
}

__global__ void k_ms_clear(unsigned long long *seen, uint64_t n, unsigned long long keep) {
  for (uint64_t v = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; v < n;
       v += (uint64_t)gridDim.x * blockDim.x)
    seen[v] &= keep;
}

// Digest finished SSSP lanes: lane q of each wave reads column q of a row.
__global__ void __launch_bounds__(MBS)
k_ms_sssp_finish(uint32_t *dist, uint64_t n, uint32_t L, unsigned long long fm, uint32_t inf,
                 bool reset, unsigned long long *acc) {
  __shared__ unsigned long long s_h[MBS / 64][64], s_c[MBS / 64][64];
  __shared__ uint32_t s_d[MBS / 64][64];
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const bool mine = lane < L && ((fm >> lane) & 1ull);
  unsigned long long h = 0, cnt = 0;
  uint32_t dep = 0;
  const uint64_t nw = (uint64_t)gridDim.x * (MBS / 64);
  for (uint64_t v = blockIdx.x * (uint64_t)(MBS / 64) + wv; v < n; v += nw) {
    if (!mine) continue;
    uint32_t *p = &dist[v * L + lane];
    const uint32_t d = *p;
    if (d != inf) {
      h += mix64((v << 32) | d);
      cnt++;
      dep = max(dep, d);
      if (reset) *p = inf;
    }
  }
  s_h[wv][lane] = h;
  s_c[wv][lane] = cnt;
  s_d[wv][lane] = dep;
  __syncthreads();
  if (threadIdx.x < 64 && mine) {
    for (int i = 1; i < MBS / 64; i++) {
      h += s_h[i][lane];
      cnt += s_c[i][lane];
      dep = max(dep, s_d[i][lane]);
    }
    if (cnt) {
      atomicAdd(&acc[RES_HASH + lane], h);
      atomicAdd(&acc[RES_CNT + lane], cnt);
      atomicMax(&acc[RES_DEPTH + lane], (unsigned long long)dep);
    }
  }
}

__global__ void k_ms_gather(const uint32_t *dist, uint64_t n, uint32_t L, uint32_t q,
                            uint32_t *out) {
  for (uint64_t v = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; v < n;
       v += (uint64_t)gridDim.x * blockDim.x)
    out[v] = dist[v * L + q];
}

int grid_for(uint64_t n, int cap) {
  return (int)std::max<uint64_t>(1, std::min<uint64_t>((n + MBS - 1) / MBS, (uint64_t)cap));
}

}  // namespace

MultiEngine::MultiEngine(Graph &gr, int al, uint32_t lanes, bool kf)
    : g(gr), algo(al), L(lanes), keep_full(kf) {
  if (algo != THV_ALGO_BFS && algo != THV_ALGO_SSSP)
    fail(THV_EINVAL, "batched queries are BFS or SSSP");
  if (L == 0 || L > MAXL) fail(THV_EINVAL, "lanes must be in [1, 64]");
  if (algo == THV_ALGO_SSSP && g.rec != 8)
    fail(THV_ENOTSUP, "SSSP needs a weighted graph (8-byte records)");
  memset(&stats, 0, sizeof stats);
  mu_est = g.m;
  store_ensure(g);
  HIPC(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
  const uint64_t n = g.n, words = bitmap_words(n);
  qs.ensure(g, chunk());
  for (int i = 0; i < 2; i++) {
    fb[i].alloc(words * 4);
    F[i].alloc((n + 1) * 8);
    HIPC(hipMemsetAsync(fb[i].p, 0, words * 4, stream));
    HIPC(hipMemsetAsync(F[i].p, 0, (n + 1) * 8, stream));
  }
  if (algo == THV_ALGO_BFS) {
    seen.alloc((n + 1) * 8);
    HIPC(hipMemsetAsync(seen.p, 0, (n + 1) * 8, stream));
    tbits.alloc(words * 4);
    HIPC(hipMemsetAsync(tbits.p, 0, words * 4, stream));
    if (keep_full) full.alloc((uint64_t)L * n * 4 + 4);
  } else {
    dist.alloc((uint64_t)L * n * 4 + 4);
    if (n) launch_fill_u32(dist.as<uint32_t>(), (uint32_t)(n + 1), (uint64_t)L * n, stream);
    if (keep_full) full.alloc(n * 4 + 4);
  }
  acc.alloc(ACC_WORDS * 8);
  HIPC(hipMemsetAsync(acc.p, 0, ACC_WORDS * 8, stream));
  // fine-grained and mapped: kernels write the counters there (Workspace)
  constexpr unsigned HF = hipHostMallocMapped | hipHostMallocCoherent;
  HIPC(hipHostMalloc((void **)&h_acc, ACC_WORDS * 8, HF));
  HIPC(hipHostMalloc((void **)&h_ctr, 2 * sizeof(LevelCtr), HF));
  HIPC(hipHostGetDevicePointer((void **)&h_acc_dev, h_acc, 0));
  HIPC(hipHostGetDevicePointer((void **)&h_ctr_dev, h_ctr, 0));
  HIPC(hipStreamSynchronize(stream));
}

MultiEngine::~MultiEngine() {
  if (stream) {
    (void)hipStreamSynchronize(stream);
    (void)hipStreamDestroy(stream);
  }
  if (h_acc) (void)hipHostFree(h_acc);
  if (h_ctr) (void)hipHostFree(h_ctr);
}

uint64_t MultiEngine::bytes_needed(const Graph &g, int algo, uint32_t lanes, bool keep_full) {
  const uint64_t n = g.n, words = bitmap_words(n);
  uint64_t b = 2 * (words * 4 + (n + 1) * 8);                       // fb, F
  // queues (a table of one chunk start per 1,024 edges, as callers' budgets were
  // chosen for; the finer one in use takes 0.02 bytes an edge more)
  b += 2 * ((n + 1) * 12) + 2 * (g.m / 1024 + 2) * 4;
  b += (n / TILE + 1) * TILE * 4;                                     // long-list queue
  if (algo == THV_ALGO_BFS)
    b += (n + 1) * 8 + words * 4 + (keep_full ? (uint64_t)lanes * n * 4 : 0);
  else b += (uint64_t)lanes * n * 4 + (keep_full ? n * 4 : 0);
  return b;
}

uint64_t MultiEngine::bytes() const {
  uint64_t b = 0;
  for (const DevMem *m : {&fb[0], &fb[1], &F[0], &F[1], &tbits, &seen, &dist, &full, &acc})
    b += m->bytes;
  return b + qs.bytes();
}

uint32_t MultiEngine::chunk() const {
  return algo == THV_ALGO_SSSP ? SSSP_C : 256u * (uint32_t)g.shape.ept;
}

uint64_t MultiEngine::free_mask() const {
  const uint64_t all = L == 64 ? ~0ull : ((1ull << L) - 1);
  return all & ~active;
}

int MultiEngine::admit(uint32_t src, uint64_t tag) {
  if (src >= g.n) fail(THV_EINVAL, "source vertex out of range");
  const uint64_t fm = free_mask();
  if (!fm) return -1;
  const int q = __builtin_ctzll(fm);
  active |= 1ull << q;
  src_of[q] = src;
  tag_of[q] = tag;
  admit_q.emplace_back((uint32_t)q, src);
  return q;
}

void MultiEngine::launch_level() {
  const uint64_t n = g.n;
  const uint64_t words = bitmap_words(n);
  launched_expand = false;
  launched_finish = false;
  // finished BFS lanes keep their seen bits until a query is admitted (no
  // kernel reads the bits of an inactive lane); one pass clears them all
  if (pend_clear && !admit_q.empty()) {
    hipLaunchKernelGGL(k_ms_clear, dim3(grid_for(n, 8192)), dim3(MBS), 0, stream,
                       seen.as<unsigned long long>(), n, ~pend_clear);
    pend_clear = 0;
  }
  if (pend_finish && (!finish_last || !active)) {
    HIPC(hipMemsetAsync(acc.as<unsigned long long>() + RES_HASH, 0, 192 * 8, stream));
    hipLaunchKernelGGL(k_ms_sssp_finish, dim3(grid_for(n, 2048)), dim3(MBS), 0, stream,
                       dist.as<uint32_t>(), n, L, pend_finish, (uint32_t)(n + 1), true,
                       acc.as<unsigned long long>());
    finalizing = pend_finish;
    pend_finish = 0;
    launched_finish = true;
  }
  if (!admit_q.empty()) {
    AdmitArgs ad;
    memset(&ad, 0, sizeof ad);
    for (auto &x : admit_q) {
      const uint32_t q = x.first;
      if (algo == THV_ALGO_BFS && keep_full)
        launch_fill_u32(full.as<uint32_t>() + (uint64_t)q * n, (uint32_t)(n + 1), n, stream);
      ad.lane[ad.count] = q;
      ad.src[ad.count] = x.second;
      ad.count++;
      voff[q] = level;
      last_val[q] = 1;
      fsz[q] = 1;       // the source
      cnt_prev[q] = 1;
    }
    hipLaunchKernelGGL(k_ms_admit, dim3(1), dim3(64), 0, stream, ad, algo,
                       F[cur].as<unsigned long long>(), fb[cur].as<uint32_t>(),
                       seen.as<unsigned long long>(), dist.as<uint32_t>(), L,
                       full.as<uint32_t>(), n, acc.as<unsigned long long>());
    admit_q.clear();
    mu_est = g.m;  // new lanes miss every vertex
    mf_known = false;
  }
  level_bu = false;
  if (active) {
    hipLaunchKernelGGL(k_ms_begin, dim3(grid_for(words, 4 * g.cus)), dim3(MBS), 0, stream,
                       F[cur ^ 1].as<unsigned long long>(), fb[cur ^ 1].as<uint32_t>(), words,
                       acc.as<unsigned long long>());
    LevelCtr *c = qs.ctr.as<LevelCtr>() + (level & 1);
    if (algo == THV_ALGO_BFS && g.sym && g.dir_opt) {
      // direction: the frontier's edges against the edges of the vertices
      // some lane still misses (an upper bound kept since the last
      // bottom-up level; any admission resets it to m).  The last level has
      // summed the frontier's edges as it set the frontier's bits; only
      // admitted sources, which it did not see, make a counting pass and a
      // wait for its result necessary.
      uint64_t td = 0;  // lanes with small frontiers run top-down in any case
      const uint64_t thr = std::max<uint64_t>(1, n / LANE_TD_DIV);
      for (uint32_t q = 0; q < MAXL; q++)
        if (((active >> q) & 1ull) && fsz[q] < thr) td |= 1ull << q;
      const bool counted = td != active && !mf_known;
      uint64_t mf = mf_next;
      if (counted) {
        LevelSide cs;
        cs.pub_src = c;
        cs.pub = h_ctr_dev + (level & 1);
        cs.npub = 1;
        launch_compact(g, qs, fb[cur].as<uint32_t>(), c, stream, CMP_COUNT_ONLY, nullptr, 0, 1,
                       0xFFFFFFFFu, 0, nullptr, 0, nullptr, nullptr, &cs);
        HIPC(hipStreamSynchronize(stream));
        mf = h_ctr[level & 1].qw[0] + h_ctr[level & 1].qw[1];
      }
      level_bu = td != active && BU_ALPHA * mf > mu_est && mf > n / 8;
      if (!level_bu) td = 0;
      level_td_lanes = level_bu ? td : 0;
      if (level_bu) {
        launch_bottom_up(active & ~td);
        if (td) {
          hipLaunchKernelGGL(k_ms_lanebits, dim3(grid_for(n, g.shape.batch_bpc * g.cus)), dim3(MBS), 0, stream,
                             F[cur].as<unsigned long long>(), n, td, tbits.as<uint32_t>());
          launch_compact(g, qs, tbits.as<uint32_t>(), c, stream);
          launch_top_down(c, td);
        }
      } else {
        launch_compact(g, qs, fb[cur].as<uint32_t>(), c, stream, counted ? CMP_WRITE_ONLY : 0);
        launch_top_down(c);
      }
    } else {
      launch_compact(g, qs, fb[cur].as<uint32_t>(), c, stream);
      launch_top_down(c);
    }
    launched_expand = true;
  }
  const LevelCtr *c = qs.ctr.as<LevelCtr>() + (level & 1);
  hipLaunchKernelGGL(k_ms_publish, dim3(1), dim3(MBS), 0, stream, acc.as<unsigned long long>(),
                     h_acc_dev, launched_expand ? c : nullptr, h_ctr_dev + (level & 1));
  HIPC(hipGetLastError());
}

void MultiEngine::launch_bottom_up(uint64_t lanes) {
  const uint64_t n = g.n;
  MsBuArgs b;
  memset(&b, 0, sizeof b);
  b.eptr = g.store.d_eptr.as<uint64_t>();
  b.deg = g.d_deg.as<uint32_t>();
  b.rbit = g.store.d_rbit.as<uint32_t>();
  b.F = F[cur].as<unsigned long long>();
  b.N = F[cur ^ 1].as<unsigned long long>();
  b.seen = seen.as<unsigned long long>();
  b.nb = fb[cur ^ 1].as<uint32_t>();
  b.full = keep_full ? full.as<uint32_t>() : nullptr;
  b.acc = acc.as<unsigned long long>();
  b.lq = qs.slist.as<uint32_t>();
  b.n = n;
  b.act = lanes;
  b.level = level;
  for (uint32_t q = 0; q < MAXL; q++) b.voff[q] = voff[q];
  // one value for all active lanes (a cohort admitted together): hash each
  // gained vertex once
  b.uval = 0;
  for (uint32_t q = 0; q < MAXL; q++) {
    if (!((lanes >> q) & 1ull)) continue;
    const uint32_t v = level + 2 - voff[q];
    if (!b.uval) b.uval = v;
    else if (b.uval != v) {
      b.uval = 0;
      break;
    }
  }
  if (qs.slist.bytes < n * 4) fail(THV_ESTATE, "bottom-up queue too small");
  const int gs = grid_for(n, g.shape.batch_bpc * g.cus), gl = g.shape.batch_bpc * g.cus;
  if (g.rec == 8) {
    hipLaunchKernelGGL(k_ms_bu<8>, dim3(gs), dim3(MBS), 0, stream, b);
    hipLaunchKernelGGL(k_ms_bu_long<8>, dim3(gl), dim3(MBS), 0, stream, b);
  } else {
    hipLaunchKernelGGL(k_ms_bu<4>, dim3(gs), dim3(MBS), 0, stream, b);
    hipLaunchKernelGGL(k_ms_bu_long<4>, dim3(gl), dim3(MBS), 0, stream, b);
  }
  HIPC(hipGetLastError());
}

void MultiEngine::launch_top_down(LevelCtr *c, uint64_t lanes) {
  const uint64_t n = g.n;
  {
    MsArgs a;
    memset(&a, 0, sizeof a);
    for (int i = 0; i < 2; i++) {
      a.qv[i] = qs.qv[i].as<uint32_t>();
      a.qe[i] = qs.qe[i].as<unsigned long long>();
      a.qc[i] = qs.qc[i].as<uint32_t>();
    }
    a.ctr = c;
    a.eptr = g.store.d_eptr.as<uint64_t>();
    a.deg = algo == THV_ALGO_BFS && g.sym && g.dir_opt ? g.d_deg.as<uint32_t>() : nullptr;
    a.F = F[cur].as<unsigned long long>();
    a.N = F[cur ^ 1].as<unsigned long long>();
    a.seen = seen.as<unsigned long long>();
    a.nb = fb[cur ^ 1].as<uint32_t>();
    a.dist = dist.as<uint32_t>();
    a.full = algo == THV_ALGO_BFS && keep_full ? full.as<uint32_t>() : nullptr;
    a.acc = acc.as<unsigned long long>();
    a.n = n;
    a.L = L;
    a.level = level;
    a.fmask = lanes;
    for (uint32_t q = 0; q < MAXL; q++) a.voff[q] = voff[q];
    const int grid = g.shape.blocks_per_cu * g.cus;
    const bool r8 = g.rec == 8;
    if (qs.C != chunk()) fail(THV_ESTATE, "queue chunk size mismatch");
    if (algo == THV_ALGO_BFS) {
      if (g.shape.ept == 4) {
        if (r8) hipLaunchKernelGGL((k_ms_bfs<8, 4>), dim3(grid), dim3(MBS), 0, stream, a);
        else hipLaunchKernelGGL((k_ms_bfs<4, 4>), dim3(grid), dim3(MBS), 0, stream, a);
      } else {
        if (r8) hipLaunchKernelGGL((k_ms_bfs<8, 8>), dim3(grid), dim3(MBS), 0, stream, a);
        else hipLaunchKernelGGL((k_ms_bfs<4, 8>), dim3(grid), dim3(MBS), 0, stream, a);
      }
    } else {
      // One block per chunk, not a persistent grid, unless room is to be left:
      // an SSSP level runs for milliseconds, and short blocks let the
      // work-groups of other streams take CUs as they free up.  The chunk count
      // comes from the compaction just launched (one readback).
      LevelSide ps;
      ps.pub_src = c;
      ps.pub = h_ctr_dev + (level & 1);
      ps.npub = 1;
      launch_publish(ps, stream);
      HIPC(hipStreamSynchronize(stream));
      const LevelCtr &h = h_ctr[level & 1];
      const bool large = h.qw[0] + h.qw[1] >= 8ull * g.cus * SSSP_LARGE;
      const uint32_t C = large ? SSSP_LARGE : SSSP_C;
      const uint64_t chunks = div_up(h.qw[0], C) + div_up(h.qw[1], C);
      // (a level's time: its host records at the link's rate, some 50 ps a record)
      const double ms = (double)h.qw[0] * 8 / (g.do_link_gbps * 1e6) +
                        (double)(h.qw[0] + h.qw[1]) * 50e-9;
      const bool room = leave_room && ms >= ROOM_MS;
      const uint64_t most = room ? (uint64_t)ROOM_BPC * g.cus : 1u << 30;
      const uint64_t sg = std::max<uint64_t>(1, std::min<uint64_t>(chunks, most));
      if (large) launch_sssp<SSSP_LARGE>(a, (uint32_t)sg, stream);
      else launch_sssp<SSSP_C>(a, (uint32_t)sg, stream);
    }
    HIPC(hipGetLastError());
  }
}

void MultiEngine::finish_level(std::vector<LaneResult> &done) {
  HIPC(hipStreamSynchronize(stream));
  if (launched_finish) {
    for (uint32_t q = 0; q < L; q++) {
      if (!((finalizing >> q) & 1ull)) continue;
      // the lane may already hold a new query; its finished one was
      // recorded in fin_tag/fin_src when the digest was launched
      LaneResult r;
      r.tag = fin_tag[q];
      r.src = fin_src[q];
      r.reached = h_acc[RES_CNT + q];
      r.hash = h_acc[RES_HASH + q];
      r.depth = (uint32_t)h_acc[RES_DEPTH + q];
      done.push_back(r);
    }
    finalizing = 0;
  }
  just_finished = 0;
  if (!launched_expand) return;
  if (level_bu) {
    const uint64_t sh = h_acc[ACC_SCAN_HOST], sd = h_acc[ACC_SCAN_HBM];
    stats.edges_traversed += sh + sd;
    stats.host_bytes += sh * (uint64_t)g.rec;
    stats.hbm_bytes += sd * (uint64_t)g.rec;
    stats.bottom_up_levels++;
    mu_est = h_acc[ACC_MU];
    if (level_td_lanes) {  // the lanes that ran top-down in this level
      const LevelCtr &h = h_ctr[level & 1];
      stats.edges_traversed += h.qw[0] + h.qw[1];
      stats.host_bytes += h.qw[0] * (uint64_t)g.rec;
      stats.hbm_bytes += h.qw[1] * (uint64_t)g.rec;
      // their missing vertices' edges are not in the bottom-up measure
      mu_est = g.m;
    }
  } else {
    const LevelCtr &h = h_ctr[level & 1];
    stats.edges_traversed += h.qw[0] + h.qw[1];
    stats.host_bytes += h.qw[0] * (uint64_t)g.rec;
    stats.hbm_bytes += h.qw[1] * (uint64_t)g.rec;
  }
  mf_next = h_acc[ACC_MF];
  mf_known = true;
  stats.iterations++;
  stats.expand_launches++;
  const uint64_t lm = h_acc[ACC_LM];
  for (uint32_t q = 0; q < MAXL; q++) {  // each lane's next frontier: this level's gains
    if (!((active >> q) & 1ull)) continue;
    fsz[q] = h_acc[ACC_CNT + q] - cnt_prev[q];
    cnt_prev[q] = h_acc[ACC_CNT + q];
  }
  for (uint32_t q = 0; q < L; q++) {
    const uint64_t bit = 1ull << q;
    if (!(active & bit)) continue;
    if (lm & bit) {
      last_val[q] = level + 2 - voff[q];
      continue;
    }
    active &= ~bit;
    just_finished |= bit;
    if (algo == THV_ALGO_BFS) {
      LaneResult r;
      r.tag = tag_of[q];
      r.src = src_of[q];
      r.reached = h_acc[ACC_CNT + q];
      r.hash = h_acc[ACC_HASH + q];
      r.depth = last_val[q];
      done.push_back(r);
      pend_clear |= bit;
    } else {
      pend_finish |= bit;
      fin_tag[q] = tag_of[q];
      fin_src[q] = src_of[q];
    }
  }
  cur ^= 1;
  level++;
}

void MultiEngine::copy_full(uint32_t q, uint32_t *out) {
  if (!keep_full) fail(THV_ESTATE, "engine does not keep value arrays");
  const uint64_t n = g.n;
  if (algo == THV_ALGO_BFS) {
    HIPC(hipMemcpyAsync(out, full.as<uint32_t>() + (uint64_t)q * n, n * 4,
                        hipMemcpyDeviceToHost, stream));
  } else {
    hipLaunchKernelGGL(k_ms_gather, dim3(grid_for(n, 8192)), dim3(MBS), 0, stream,
                       dist.as<uint32_t>(), n, L, q, full.as<uint32_t>());
    HIPC(hipMemcpyAsync(out, full.p, n * 4, hipMemcpyDeviceToHost, stream));
  }
  HIPC(hipStreamSynchronize(stream));
}

// Engines of finished batches, kept for the next batch on their graph: making
// one (some 25 allocations, and as many frees) took 1.5-2.7 ms of a 64-source
// batch, as long as its levels at R-MAT 22.  An engine that is running is
// not here.  All of them together hold at most KEEP bytes; a graph's go when
// it is closed or its store changes, and all when an allocation fails or the
// free memory is asked for.
class IdleEngines {
 public:
  static constexpr uint64_t KEEP = 4ull << 30;
  static IdleEngines &get() {
    static IdleEngines *p = new IdleEngines();  // never destroyed: HIP may be gone by then
    return *p;
  }
  std::unique_ptr<MultiEngine> take(Graph &g, int algo, uint32_t k) {
    std::unique_ptr<MultiEngine> e;
    {
      std::lock_guard<std::mutex> lk(mu);
      for (size_t i = 0; i < idle.size(); i++) {
        MultiEngine &x = *idle[i];
        if (&x.g != &g || x.algo != algo || (algo == THV_ALGO_BFS ? x.L < k : x.L != k)) continue;
        e = std::move(idle[i]);
        idle.erase(idle.begin() + i);
        break;
      }
    }
    if (e) e->qs.ensure(g, e->chunk());  // the launch shape may have changed
    return e;
  }
  void put(std::unique_ptr<MultiEngine> e) {
    const uint64_t b = e->bytes();
    if (b > KEEP) return;
    std::vector<std::unique_ptr<MultiEngine>> out;  // freed without the lock
    std::lock_guard<std::mutex> lk(mu);
    for (size_t i = 0; i < idle.size();) {
      if (&idle[i]->g == &e->g && idle[i]->algo == e->algo) {
        out.push_back(std::move(idle[i]));
        idle.erase(idle.begin() + i);
      } else {
        i++;
      }
    }
    uint64_t sum = b;
    for (auto &x : idle) sum += x->bytes();
    while (sum > KEEP && !idle.empty()) {  // the longest unused first
      sum -= idle.front()->bytes();
      out.push_back(std::move(idle.front()));
      idle.erase(idle.begin());
    }
    idle.push_back(std::move(e));
  }
  // all engines, or those of one graph; how many there were
  size_t drop(const Graph *g) {
    std::vector<std::unique_ptr<MultiEngine>> out;
    std::lock_guard<std::mutex> lk(mu);
    for (size_t i = 0; i < idle.size();) {
      if (!g || &idle[i]->g == g) {
        out.push_back(std::move(idle[i]));
        idle.erase(idle.begin() + i);
      } else {
        i++;
      }
    }
    return out.size();
  }

 private:
  std::mutex mu;
  std::vector<std::unique_ptr<MultiEngine>> idle;
};

size_t drop_idle_engines(const Graph *g) { return IdleEngines::get().drop(g); }

void run_batch(Graph &g, int algo, const uint32_t *srcs, uint32_t k, uint64_t *hash,
               uint64_t *reached, uint32_t *depth, uint32_t *full, thv_stats *st) {
  if (k == 0) {
    if (st) memset(st, 0, sizeof *st);
    return;
  }
  for (uint32_t i = 0; i < k; i++)
    if (srcs[i] >= g.n) fail(THV_EINVAL, "source vertex out of range");
  // an engine kept from an earlier batch starts as a server's does between
  // queries: its finished lanes are cleared when the new ones are admitted
  std::unique_ptr<MultiEngine> own = full ? nullptr : IdleEngines::get().take(g, algo, k);
  if (!own) {
    // (a BFS engine's memory does not depend on its lanes: it serves any k)
    const uint32_t lanes = algo == THV_ALGO_BFS && !full ? MultiEngine::MAXL : k;
    own.reset(new MultiEngine(g, algo, lanes, full != nullptr));
  }
  MultiEngine &e = *own;
  e.finish_last = true;
  memset(&e.stats, 0, sizeof e.stats);
  for (uint32_t i = 0; i < k; i++) e.admit(srcs[i], i);
  std::vector<LaneResult> done;
  const uint64_t t0 = now_ns();
  while (e.busy()) {
    e.launch_level();
    e.finish_level(done);
    if (full && e.just_finished) {
      for (uint32_t q = 0; q < k; q++)
        if ((e.just_finished >> q) & 1ull) e.copy_full(q, full + (uint64_t)e.tag_of[q] * g.n);
    }
  }
  if (st) {
    *st = e.stats;
    st->ms = (now_ns() - t0) * 1e-6;
  }
  for (auto &r : done) {
    if (hash) hash[r.tag] = r.hash;
    if (reached) reached[r.tag] = r.reached;
    if (depth) depth[r.tag] = r.depth;
  }
  if (!full) IdleEngines::get().put(std::move(own));
}

}  // namespace thv
