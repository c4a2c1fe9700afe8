// Lane-per-pair join shared by the plain form (masks cut from the candidate bitset) and the
// batched form (masks from the survivor arena).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "device_common.hpp"
#include "kernels.hpp"

namespace sigmo_k {
namespace {

// Candidate masks of the survivor arena: k consecutive per pair, of 32 bits for molecules of <= 32
// nodes, 64 for 33..64 and 128 for wider ones.  `overflow` is the pair evaluation's arena-overflow
// flag: once set, offsets past the arena were handed out and no mask may be read, so the join does
// nothing and the host repeats the run with a larger arena.
struct ArenaMasks {
  const uint64_t* arena;
  const uint32_t* mask_off;
  const unsigned long long* overflow;
  __device__ __forceinline__ bool aborted() const { return uniform32(static_cast<uint32_t>(*overflow != 0ull)) != 0u; }
  __device__ __forceinline__ uint32_t base(uint64_t j) const { return mask_off[j]; }
  __device__ __forceinline__ uint64_t mask(uint32_t base, uint32_t, uint32_t depth, uint32_t, uint32_t n) const {
    const uint64_t* p = arena + base;
    return n <= 32 ? reinterpret_cast<const uint32_t*>(p)[depth] : p[depth];
  }
  // molecules of 65..128 nodes: two words per query node (positions 0-63, 64-127)
  __device__ __forceinline__ void mask2(uint32_t base, uint32_t, uint32_t depth, uint32_t, uint32_t, uint64_t& lo, uint64_t& hi) const {
    lo = arena[static_cast<uint64_t>(base) + 2 * depth];
    hi = arena[static_cast<uint64_t>(base) + 2 * depth + 1];
  }
  // The masks of query nodes 0..k-1 (entries from k on are not to be read), 16 bytes per load: a
  // pair's block starts on a 16-byte boundary and spans a multiple of four masks, so a load that
  // starts below k stays inside it.
  template <int N>
  __device__ __forceinline__ void masks(uint32_t base, uint32_t, uint32_t k, uint32_t, uint32_t n, uint64_t (&m)[N]) const {
    static_assert(N % 4 == 0, "masks come in fours");
    const uint4* p = reinterpret_cast<const uint4*>(arena + base);
    const uint32_t half = n <= 32;
    uint4 v[N / 2];  // one to two nodes each, or one to four
#pragma unroll
    for (uint32_t t = 0; t < static_cast<uint32_t>(N) / 2; ++t) {
      v[t] = make_uint4(0, 0, 0, 0);
      if (2 * t < (half ? (k + 1) / 2 : k)) v[t] = p[t];
    }
#pragma unroll
    for (uint32_t t = 0; t < static_cast<uint32_t>(N); t += 4) {
      const uint4 a = v[t / 4], b = v[t / 2], c = v[t / 2 + 1];
      m[t] = half ? a.x : b.x | (static_cast<uint64_t>(b.y) << 32);
      m[t + 1] = half ? a.y : b.z | (static_cast<uint64_t>(b.w) << 32);
      m[t + 2] = half ? a.z : c.x | (static_cast<uint64_t>(c.y) << 32);
      m[t + 3] = half ? a.w : c.z | (static_cast<uint64_t>(c.w) << 32);
    }
  }
  // The two-word masks of query nodes 0..k-1, one 16-byte load per node.
  template <int N>
  __device__ __forceinline__ void masks2(uint32_t base, uint32_t, uint32_t k, uint32_t, uint32_t, uint64_t (&lo)[N], uint64_t (&hi)[N]) const {
#pragma unroll
    for (uint32_t t = 0; t < static_cast<uint32_t>(N); ++t) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (t < k) v = *reinterpret_cast<const uint4*>(arena + static_cast<uint64_t>(base) + 2 * t);
      lo[t] = static_cast<uint64_t>(v.x) | (static_cast<uint64_t>(v.y) << 32);
      hi[t] = static_cast<uint64_t>(v.z) | (static_cast<uint64_t>(v.w) << 32);
    }
  }
};

// Candidate masks cut from the bitset row of the query node: positions s..s+n-1 (n <= 64 spans
// at most two 64-bit words), shifted to bit 0.
struct BitsetMasks {
  const uint64_t* bits;
  uint64_t W64;
  __device__ __forceinline__ bool aborted() const { return false; }
  __device__ __forceinline__ uint32_t base(uint64_t) const { return 0; }
  // Both words come from one 16-byte load.  The second may be the next row's first word, or the
  // word past the last row (the bitset allocation carries one spare word): it only fills bits
  // at positions >= 64 - sh, which n <= 64 - sh then masks off.
  __device__ __forceinline__ uint64_t mask(uint32_t, uint32_t qrow, uint32_t, uint32_t s, uint32_t n) const {
    typedef uint64_t u64x2 __attribute__((ext_vector_type(2))) __attribute__((aligned(8)));
    const uint64_t* row = bits + static_cast<uint64_t>(qrow) * W64;
    const uint32_t w0 = s >> 6, sh = s & 63;
    const u64x2 v = *reinterpret_cast<const u64x2*>(row + w0);
    const uint64_t lo = v.x, hi = v.y;
    uint64_t m = sh ? (lo >> sh) | (hi << (64 - sh)) : lo;
    if (n < 64) m &= (1ull << n) - 1;
    return m;
  }
  // positions s..s+n-1 with 64 < n <= 128: up to three words of the row, funnel-shifted
  __device__ __forceinline__ void mask2(uint32_t, uint32_t qrow, uint32_t, uint32_t s, uint32_t n, uint64_t& lo, uint64_t& hi) const {
    const uint64_t* row = bits + static_cast<uint64_t>(qrow) * W64;
    const uint32_t w0 = s >> 6, last = (s + n - 1) >> 6, sh = s & 63;
    const uint64_t x0 = row[w0];
    const uint64_t x1 = w0 + 1 <= last ? row[w0 + 1] : 0ull;
    const uint64_t x2 = w0 + 2 <= last ? row[w0 + 2] : 0ull;
    lo = sh ? (x0 >> sh) | (x1 << (64 - sh)) : x0;
    hi = sh ? (x1 >> sh) | (x2 << (64 - sh)) : x1;
    if (n < 128) hi &= (1ull << (n - 64)) - 1;
  }
  template <int N>
  __device__ __forceinline__ void masks(uint32_t base, uint32_t qoff, uint32_t k, uint32_t s, uint32_t n, uint64_t (&m)[N]) const {
#pragma unroll
    for (uint32_t t = 0; t < static_cast<uint32_t>(N); ++t) m[t] = t < k ? mask(base, qoff + t, t, s, n) : 0ull;
  }
  template <int N>
  __device__ __forceinline__ void masks2(uint32_t base, uint32_t qoff, uint32_t k, uint32_t s, uint32_t n, uint64_t (&lo)[N], uint64_t (&hi)[N]) const {
#pragma unroll
    for (uint32_t t = 0; t < static_cast<uint32_t>(N); ++t) {
      lo[t] = hi[t] = 0;
      if (t < k) mask2(base, qoff + t, t, s, n, lo[t], hi[t]);
    }
  }
};

// Query levels the lane join holds in LDS per lane.  Surviving pairs are mostly small queries (on
// LogNormal molecules and U[4,32]-node queries 92% have k <= 8, and they take 89% of the DFS
// steps), so a large join lists the pairs of deeper queries for a second pass; a small one runs
// them all in one pass that holds 12 levels and reaches deeper ones through global memory.
constexpr int kJoinShallow = 8;
constexpr int kJoinLevels = 12;
constexpr int kJoinWideLevels = 7;  // two words per position: LDS as for kJoinLevels of one
// Pair counts from which the lane join runs in two passes: the first gains a third of its time per pair,
// the second costs its longest searches' time again.  The join in one and two passes, find-first,
// 150,000 LogNormal molecules: 2.2 M pairs 0.51 and 0.80 ms, 3.6 M 0.90 and 1.11, 4.6 M 1.54 and 1.57, 6.4 M
// 1.70 and 1.67, 10.3 M 2.56 and 2.19; 100,000 Normal molecules: 3.4 M 0.72 and 0.83, 6.1 M 1.11 and 1.19,
// 7.5 M 1.57 and 1.38; with masks cut from the bitset the sides meet at 4 to 4.5 M.  Counting every
// embedding they meet between 6 and 8 M or lower (Normal 6.1 M: 2.80 and 2.28; LogNormal 6.4 M: 3.34 and
// 3.50, 8.4 M: 4.58 and 4.35).  Of a bound on the device 8 to 15% survive, and the better side varies with the
// searches: 20 M (2.2 M pairs) 0.45 and 0.34, 30 M (3.0 M) 0.73 and 0.89, 24 M that all survive 17.7 and 15.5.
constexpr uint64_t kJoinTwoPassPairs = 3ull << 21;
constexpr uint64_t kJoinTwoPassBound = 1ull << 24;
constexpr uint32_t kJoinDeepChunk = 128;            // pairs a wavefront claims at a time of the deep queries' list
constexpr uint32_t kJoinRefill = 24;                // idle lanes that make a wavefront hand out new pairs

// One wavefront's LDS: per level t and lane, the adjacency row of the position mapped at t and the
// candidates frame t started from (t < L = KC - 1), the candidate mask of query node t + 1, and
// the mapping (a byte per level); then the queue of the next pairs.
template <int KC, bool DEEP, bool WIDE>
struct JoinLds {
  static constexpr int L = KC - 1;
  static constexpr int H = WIDE ? 2 : 1;
  static constexpr int M = DEEP ? 40 : 8;  // mapping bytes per lane
  uint64_t row[H][L][kWave];
  uint64_t base[H][L][kWave];
  uint64_t mask[H][L][kWave];
  alignas(8) uint8_t map[kWave][M];
  uint64_t q_adj[kWave];
  uint32_t q_pair[kWave], q_start[kWave], q_qoff[kWave], q_base[kWave];
  uint16_t q_nk[kWave];
  uint32_t listed[DEEP ? 1 : 2 * kWave];  // pairs for the deep pass
};
constexpr uint32_t join_waves_per_cu(size_t lds) {  // wavefronts the 160 KB of LDS hold
  return static_cast<uint32_t>(160 * 1024 / ((lds + 511) / 512 * 512));
}
constexpr size_t kJoinAllLds = sizeof(JoinLds<kJoinLevels, true, false>) > sizeof(JoinLds<kJoinWideLevels, true, true>)
                                   ? sizeof(JoinLds<kJoinLevels, true, false>)
                                   : sizeof(JoinLds<kJoinWideLevels, true, true>);

// A lane's statistics.
struct JoinTotals {
  uint64_t sum = 0, matched = 0, steps = 0, overflow = 0, wave_iters = 0;
};

// Positions above c of a 64-position word.
__device__ __forceinline__ uint64_t bits_above(uint32_t c) { return (~0ull << c) << 1; }
__device__ __forceinline__ uint64_t bit_of(uint32_t c) { return 1ull << (c & 63u); }
// A candidate set after the row of one mapped node: x & row where `a` is all ones (a query
// neighbour), x & ~row where it is 0.  x & ~(row ^ a), table 0x90, one operation per 32 positions.
__device__ __forceinline__ uint64_t and_row(uint64_t x, uint64_t row, uint32_t a) {
  const uint32_t lo = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(x), static_cast<uint32_t>(row), a, 0x90);
  const uint32_t hi = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(x >> 32), static_cast<uint32_t>(row >> 32), a, 0x90);
  return lo | (static_cast<uint64_t>(hi) << 32);
}
// All ones when bit t (< 32) of q is set.
__device__ __forceinline__ uint32_t bit_spread(uint32_t q, uint32_t t) {
  return static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(q), t, 1u));
}

// Join with one lane per GMCR pair: the reference DFS of isomorphism.hpp:270-381 for the lane's
// pair with the reference's bookkeeping -- every mapping entry starts at local node 0, an
// exhausted frame unsets the visited bit of its (possibly stale) mapping entry, `visited` is
// cleared when depth 1 is exhausted, and a frame resumes at mapping[depth] + 1.  The validity
// test of isomorphism.hpp:150-168 -- for every j < depth, qAdj(j, depth) == dAdj(mapping[j], c)
// -- is set algebra on adjacency rows: adjacency is symmetric, so the candidates that pass are
// those in the row of every mapped query neighbour and in the row of no other mapped node.
//
// An iteration takes several DFS steps of a lane: it pops an exhausted frame, accepts the frame's
// next candidate, and forms the next frame's candidates at once; when those are none, the next
// frame's exhaustion is taken here too and the lane stays.  Most failing searches are accept /
// exhaust pairs two or three levels down (LogNormal molecules, U[4,32] queries: 16.8 steps per
// pair in 9.5 accepts).  A frame's candidates are kept in LDS for its return.  Rows at and above
// the current depth are kept zero, so the rows of all levels apply without a test per lane (a
// zero row at a non-adjacent level keeps every position), and their LDS reads go out together.
//
// Pairs come 64 at a time through three loading stages, a pair per lane, into a queue in LDS;
// idle lanes take queued pairs and load their masks.  Loads return in order, so a step's wait for
// its adjacency row also waits for every load issued before: the stages and the masks are
// therefore all issued together, when kJoinRefill lanes are idle, and a wavefront stalls on them
// once per that many pairs (16, 24 and 32 measure the same, 40 is 4% slower).  Results are stored then
// too, since a wait for a load also waits for every store before it: 1 M LogNormal molecules x
// 1,000 queries 10.7 -> 10.3 ms, 300,000 x 306 2.08 -> 2.01 ms.  Reading one word of each line of a
// pair's adjacency rows ahead, or all levels' rows in one group, gave nothing.
//
// Bound by VALU issue at 11 wavefronts per CU by LDS: on 68 M pairs 54% of the issue slots, 58% of the
// lanes active, wavefronts waiting 55% of their time, LDS a quarter busy.  One
// DFS step per iteration, all rows tested per lane and an atomic per listed batch took, for 1 M
// LogNormal molecules x 1,000 queries, 10.8 + 1.4 ms (molecules of <= 64 nodes) and 2.5 + 1.6 ms
// (wider ones); this takes 6.5 ms and, with k_join_all's second pass, 3.2, and 33,331 molecules x
// 257 queries find-all, whose last lanes run long searches, 2.7 ms less.
//
// Molecules of <= 64 nodes (!WIDE; pairs of larger ones are passed over) or, with WIDE, of 65..128
// nodes: positions then span two words, and `visited` stays one word addressed by position mod 64,
// the reference's Bitset aliasing (utils.hpp:71-73).  Queries of up to KC nodes; deeper ones are
// listed in `deep` (their count in stats[kStatDeep]), or, with DEEP, run here with the levels past LDS
// read through global memory.  With `list` the pairs are list[0..P).
template <bool FIND_FIRST, class Src, int KC, bool DEEP, bool WIDE>
__device__ __forceinline__ void join_pass(JoinLds<KC, DEEP, WIDE>& sh, const GraphDev& q, const GraphDev& d, const Src& src,
                                          const uint32_t* __restrict__ indices, const uint32_t* __restrict__ pair_graph, uint64_t P,
                                          uint32_t chunk, int32_t* __restrict__ counts, unsigned long long* __restrict__ stats,
                                          const uint32_t* __restrict__ list, uint32_t* __restrict__ deep, uint32_t cursor, JoinTotals& total) {
  static_assert(KC == 8 || KC == 12 || (WIDE && KC == 7), "levels in LDS");
  constexpr uint32_t L = KC - 1;
  const uint32_t lane = static_cast<uint32_t>(lane_id());
  const uint64_t below = (1ull << lane) - 1;
  const uint32_t* qfold = reinterpret_cast<const uint32_t*>(q.fold);  // query rows fit the low word (k <= 32)

  // pairs on their way to the queue, one per lane and stage: graphs and mask base (a), sizes and
  // offsets (b), query adjacency (c)
  // claimed pairs [next, end) (wave-uniform): a wavefront's first claim is its own, later ones come
  // from the cursor
  uint64_t next = static_cast<uint64_t>(blockIdx.x) * chunk, end = next + chunk < P ? next + chunk : P;
  const uint64_t claimed = static_cast<uint64_t>(gridDim.x) * chunk;
  bool exhausted = false, have_a = false, have_b = false, have_c = false;
  uint32_t qhead = 0, qcount = 0;
  bool av = false, bv = false, cv = false;
  uint32_t aj = 0, ag = 0, aq = 0, abase = 0;
  uint32_t bj = 0, bbase = 0, bs = 0, be = 0, bq = 0, bqe = 0;
  uint32_t cj = 0, cbase = 0, cs = 0, cn = 0, cq = 0, ck = 0;
  uint32_t ca[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) ca[t] = 0;

  // the lane's pair; `loading`: taken, its candidate masks on their way
  bool have = false, loading = false, finished = false;
  uint64_t mlo[KC], mhi[WIDE ? KC : 1];
#pragma unroll
  for (int t = 0; t < KC; ++t) mlo[t] = 0;
#pragma unroll
  for (int t = 0; t < (WIDE ? KC : 1); ++t) mhi[t] = 0;
  uint32_t j = 0, s = 0, n = 0, qoff = 0, k = 0, base = 0, depth = 0;
  uint64_t adj = 0, visited = 0, count = 0;      // adj: byte t = query row of node t < 8 over nodes < 8
  uint64_t cur = 0, cur_hi = 0, rem = 0, rem_hi = 0;  // the frame's candidates; positions past its last accept

  // Pairs for the deep pass gather in LDS and go out 64 at a time: an atomic per batch of 64 pairs on
  // one address (about 10 ns each across the XCDs) took 11 ms for 68 M pairs and bound the kernel.
  uint32_t ndeep = 0;
  auto list_flush = [&](uint32_t cnt) {
    unsigned long long b = 0;
    if (lane == 0) b = atomicAdd(&stats[kStatDeep], static_cast<unsigned long long>(cnt));
    const uint64_t ob = uniform64(__shfl(b, 0));
    if (lane < cnt) deep[ob + lane] = sh.listed[lane];
  };
  auto list_pairs = [&](bool mine, uint32_t pair) {
    const uint64_t m = __ballot(mine);
    if (!m) return;
    if (mine) sh.listed[ndeep + __popcll(m & below)] = pair;
    wave_sync();
    ndeep += static_cast<uint32_t>(__popcll(m));
    if (ndeep >= kWave) {
      list_flush(kWave);
      ndeep -= kWave;
      const uint32_t left = sh.listed[kWave + lane];
      wave_sync();
      sh.listed[lane] = left;
      wave_sync();
    }
  };
  // rows of the mapped positions at levels below `upto` (and, in LDS, the zero rows above)
  // applied to a candidate set; qm: the query row's bits below `upto`
  auto apply_rows = [&](uint32_t qm, uint32_t upto, uint64_t& lo, uint64_t& hi) {
    auto group = [&](uint32_t t0, uint32_t t1) {
      uint64_t r[4], rh[4];
#pragma unroll
      for (uint32_t t = t0; t < t1; ++t) {
        r[t - t0] = sh.row[0][t][lane];
        if constexpr (WIDE) rh[t - t0] = sh.row[1][t][lane];
      }
#pragma unroll
      for (uint32_t t = t0; t < t1; ++t) {
        const uint32_t a = bit_spread(qm, t);
        lo = and_row(lo, r[t - t0], a);
        if constexpr (WIDE) hi = and_row(hi, rh[t - t0], a);
      }
    };
    group(0, 4);
    if (__any(upto > 4)) {
      group(4, L < 8 ? L : 8);
      if constexpr (L > 8)
        if (__any(upto > 8)) group(8, L);
    }
    if constexpr (DEEP)
      for (uint32_t t = L; t < upto; ++t) {
        const uint64_t v = static_cast<uint64_t>(s) + sh.map[lane][t];
        const uint32_t a = bit_spread(qm, t);
        if constexpr (WIDE) {
          lo = and_row(lo, d.adj[2 * v], a);
          hi = and_row(hi, d.adj[2 * v + 1], a);
        } else {
          lo = and_row(lo, d.fold[v], a);
        }
      }
  };
  // the query adjacency row of node t < k (with bits of later rows above bit 7 when t < 8)
  auto query_row = [&](uint32_t t) -> uint32_t {
    uint32_t r = static_cast<uint32_t>(adj >> ((8 * t) & 63u));
    if constexpr (DEEP)
      if (t >= 8) r = qfold[2 * (static_cast<uint64_t>(qoff) + t)];
    return r;
  };
  // the candidate mask of query node t >= 1
  auto node_mask = [&](uint32_t t, uint64_t& lo, uint64_t& hi) {
    const uint32_t at = DEEP ? min(t - 1, L - 1) : t - 1;
    lo = sh.mask[0][at][lane];
    if constexpr (WIDE) hi = sh.mask[1][at][lane];
    if constexpr (DEEP)
      if (t > L) {
        if constexpr (WIDE) src.mask2(base, qoff + t, t, s, n, lo, hi);
        else lo = src.mask(base, qoff + t, t, s, n);
      }
  };

  while (true) {
    if (loading) {  // the taken pair's masks have arrived: start it
#pragma unroll
      for (int t = 0; t < (DEEP ? 32 : 8); t += 8) *reinterpret_cast<uint64_t*>(&sh.map[lane][t]) = 0;  // every entry: local node 0
#pragma unroll
      for (uint32_t t = 0; t < L; ++t) {
        sh.row[0][t][lane] = 0;
        sh.mask[0][t][lane] = mlo[t + 1];
        if constexpr (WIDE) {
          sh.row[1][t][lane] = 0;
          sh.mask[1][t][lane] = mhi[t + 1];
        }
      }
      cur = mlo[0];
      rem = ~0ull;
      if constexpr (WIDE) {
        cur_hi = mhi[0];
        rem_hi = ~0ull;
      }
      depth = 0;
      visited = 0;
      count = 0;
      have = true;
      loading = false;
    }
    const uint64_t idle = __ballot(!have);
    if (static_cast<uint32_t>(__popcll(idle)) >= kJoinRefill || idle == ~0ull) {  // wave-uniform
      if (finished) {  // stored here and not when the search ends: the next step's wait for its row would wait for it
        if (count > 0x7FFFFFFFull) total.overflow = 1;
        counts[j] = static_cast<int32_t>(count > 0x7FFFFFFFull ? 0x7FFFFFFFull : count);
        total.sum += count;
        total.matched += count > 0;
        finished = false;
      }
      if (qcount == 0 && have_c) {  // the third stage has arrived: queue its pairs
        const bool wide_pair = !WIDE && cn > 64;  // molecules of > 64 nodes belong to the two-word pass
        const bool deep_pair = !DEEP && cv && !wide_pair && ck > static_cast<uint32_t>(KC);
        if constexpr (!DEEP) list_pairs(deep_pair, cj);
        const bool mine = cv && !wide_pair && !deep_pair;
        const uint64_t mm = __ballot(mine);
        if (mine) {
          uint64_t a = 0;
#pragma unroll
          for (uint32_t t = 0; t < 8; ++t) a |= static_cast<uint64_t>(ca[t] & 0xFFu) << (8 * t);
          const uint32_t at = __popcll(mm & below);
          sh.q_adj[at] = a;
          sh.q_pair[at] = cj;
          sh.q_start[at] = cs;
          sh.q_qoff[at] = cq;
          sh.q_base[at] = cbase;
          sh.q_nk[at] = static_cast<uint16_t>(cn | (ck << 8));
        }
        wave_sync();
        qhead = 0;
        qcount = static_cast<uint32_t>(__popcll(mm));
        have_c = false;
      }
      if (!have_c && have_b) {
        cv = bv;
        cj = bj;
        cbase = bbase;
        cs = bs;
        cn = be - bs;
        cq = bq;
        ck = bqe - bq;
        if (cv) {
#pragma unroll
          for (uint32_t t = 0; t < 8; ++t) ca[t] = t < ck ? qfold[2 * (static_cast<uint64_t>(cq) + t)] : 0u;
        }
        have_c = true;
        have_b = false;
      }
      if (!have_b && have_a) {
        bv = av;
        bj = aj;
        bbase = abase;
        if (bv) {
          bs = d.go[ag];
          be = d.go[ag + 1];
          bq = q.go[aq];
          bqe = q.go[aq + 1];
        }
        have_b = true;
        have_a = false;
      }
      if (!have_a && !exhausted) {
        if (next >= end && claimed < P) {
          unsigned long long b = 0;
          if (lane == 0) b = atomicAdd(&stats[cursor], static_cast<unsigned long long>(chunk));
          next = claimed + uniform64(__shfl(b, 0));
          end = next + chunk < P ? next + chunk : P;
        }
        if (next >= end) {
          exhausted = true;
        } else {
          av = next + lane < end;
          if (av) {
            aj = list ? list[next + lane] : static_cast<uint32_t>(next + lane);
            ag = pair_graph[aj];
            aq = indices[aj];
            abase = src.base(aj);
          }
          next += kWave;
          have_a = true;
        }
      }
      if (qcount) {  // hand queued pairs to idle lanes
        const uint32_t cnt = min(qcount, static_cast<uint32_t>(__popcll(idle)));
        const uint32_t rn = __popcll(idle & below);
        if (!have && rn < cnt) {
          const uint32_t at = qhead + rn;
          adj = sh.q_adj[at];
          j = sh.q_pair[at];
          s = sh.q_start[at];
          qoff = sh.q_qoff[at];
          base = sh.q_base[at];
          n = sh.q_nk[at] & 0xFFu;
          k = sh.q_nk[at] >> 8;
          if constexpr (WIDE) src.masks2(base, qoff, k, s, n, mlo, mhi);
          else src.masks(base, qoff, k, s, n, mlo);
          loading = true;
        }
        qhead += cnt;
        qcount -= cnt;
      }
      if (__ballot(have || loading) == 0) {
        if (exhausted && !have_a && !have_b && !have_c && qcount == 0) break;
        continue;
      }
    }
    ++total.wave_iters;
    if (have) {
      bool done = false;
      uint32_t st = 0;
      uint64_t el = cur & ~visited & rem, eh = WIDE ? cur_hi & ~visited & rem_hi : 0ull;
      if ((el | eh) == 0) {  // exhausted frame (:346-354)
        st = 1;
        done = depth == 0;
        const uint32_t up = done ? 0u : depth - 1;
        const uint32_t m = sh.map[lane][depth], c = sh.map[lane][up];
        visited &= ~bit_of(m);
        if (depth == 1) visited = 0;
        if (!DEEP || up < L) {
          cur = sh.base[0][up][lane];
          sh.row[0][up][lane] = 0;
          if constexpr (WIDE) {
            cur_hi = sh.base[1][up][lane];
            sh.row[1][up][lane] = 0;
          }
        } else {
          node_mask(up, cur, cur_hi);
          const uint32_t qr = query_row(up);
          apply_rows(qr & ((1u << up) - 1u), up, cur, cur_hi);
        }
        depth = up;
        if constexpr (WIDE) {
          rem = c < 64 ? bits_above(c) : 0ull;
          rem_hi = c < 64 ? ~0ull : bits_above(c - 64);
          eh = done ? 0ull : cur_hi & ~visited & rem_hi;
        } else {
          rem = bits_above(c);
        }
        el = done ? 0ull : cur & ~visited & rem;
      }
      if (el | eh) {  // accept (:366-370)
        uint32_t c;
        if constexpr (WIDE) {
          c = el ? static_cast<uint32_t>(__builtin_ctzll(el)) : 64u + static_cast<uint32_t>(__builtin_ctzll(eh));
          rem = c < 64 ? bits_above(c) : 0ull;
          rem_hi = c < 64 ? ~0ull : bits_above(c - 64);
          visited |= bit_of(c);
        } else {
          c = static_cast<uint32_t>(__builtin_ctzll(el));
          const uint64_t bit = el & (0ull - el);
          rem = 0ull - (bit << 1);  // positions above c
          visited |= bit;
        }
        const uint64_t v = static_cast<uint64_t>(s) + c;
        uint64_t rlo, rhi = 0, nlo = 0, nhi = 0;
        if constexpr (WIDE) {
          rlo = d.adj[2 * v];
          rhi = d.adj[2 * v + 1];
        } else {
          rlo = d.fold[v];
        }
        const uint32_t nd = depth + 1;
        const bool leaf = nd == k;
        const uint32_t qr = query_row(leaf ? 0u : nd);
        node_mask(leaf ? 1u : nd, nlo, nhi);
        sh.map[lane][depth] = static_cast<uint8_t>(c);
        const uint32_t stale = sh.map[lane][leaf ? 0u : nd];
        apply_rows(qr & ((1u << depth) - 1u), depth, nlo, nhi);
        const uint32_t a = bit_spread(qr, depth);
        nlo = and_row(nlo, rlo, a);
        if constexpr (WIDE) nhi = and_row(nhi, rhi, a);
        const bool some = ((nlo & ~visited) | (WIDE ? nhi & ~visited : 0ull)) != 0;
        if (leaf) {  // (:336-344): the frame resumes past it
          ++count;
          done = FIND_FIRST;
        }
        if (!leaf && some) {  // the next frame
          st += 1;
          if (!DEEP || depth < L) {
            sh.base[0][depth][lane] = cur;
            sh.row[0][depth][lane] = rlo;
            if constexpr (WIDE) {
              sh.base[1][depth][lane] = cur_hi;
              sh.row[1][depth][lane] = rhi;
            }
          }
          depth = nd;
          cur = nlo;
          rem = ~0ull;
          if constexpr (WIDE) {
            cur_hi = nhi;
            rem_hi = ~0ull;
          }
        } else {  // the leaf, or the next frame's exhaustion
          st += 2;
          if (!leaf) visited = nd == 1 ? 0ull : visited & ~bit_of(stale);
        }
      }
      total.steps += st;
      if (done) {
        finished = true;
        have = false;
      }
    }
  }
  if constexpr (!DEEP)
    if (ndeep) list_flush(ndeep);
}

__device__ __forceinline__ void join_totals(const JoinTotals& total, unsigned long long* __restrict__ stats) {
  uint64_t sum = total.sum, matched = total.matched, steps = total.steps, overflow = total.overflow;
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    sum += __shfl_xor(sum, o);
    matched += __shfl_xor(matched, o);
    steps += __shfl_xor(steps, o);
    overflow |= __shfl_xor(overflow, o);
  }
  // one atomic for the four sums, which share a line (about 10 ns each on one line), and none of zero:
  // 100,000 pairs' wavefronts with nothing to join 40 -> 4 us
  const uint32_t lane = static_cast<uint32_t>(lane_id());
  const uint64_t mine = lane == 0 ? sum : (lane == 1 ? matched : (lane == 2 ? steps : total.wave_iters));
  const uint32_t at = lane == 0 ? kStatSum : (lane == 1 ? kStatMatched : (lane == 2 ? kStatSteps : kStatWaveIters));
  if (lane < 4 && mine) atomicAdd(&stats[at], static_cast<unsigned long long>(mine));
  if (lane == 0 && overflow) atomicOr(&stats[kStatOverflow], 1ull);
}

// One pass over the pairs, or those listed, of molecules of <= 64 nodes.  P_dev: their count left on
// the device; P, what the arrays were sized for, bounds it.
template <bool FIND_FIRST, class Src, int KC, bool DEEP>
__global__ __launch_bounds__(64) void k_join_lanes(GraphDev q, GraphDev d, Src src, const uint32_t* __restrict__ indices,
                                                   const uint32_t* __restrict__ pair_graph, uint64_t P, uint32_t chunk,
                                                   int32_t* __restrict__ counts, unsigned long long* __restrict__ stats,
                                                   const unsigned long long* __restrict__ P_dev, const uint32_t* __restrict__ list,
                                                   uint32_t* __restrict__ deep, uint32_t cursor) {
  __shared__ JoinLds<KC, DEEP, false> sh;
  if (src.aborted()) return;
  if (P_dev) P = min(P, static_cast<uint64_t>(*P_dev));
  JoinTotals total;
  join_pass<FIND_FIRST, Src, KC, DEEP, false>(sh, q, d, src, indices, pair_graph, P, chunk, counts, stats, list, deep, cursor, total);
  join_totals(total, stats);
}

// The pairs of molecules of > 64 nodes, listed in `wide`, then the other pairs (or those of `list`): a
// wavefront goes on to these as soon as no wide pair is left to claim.  The wide pairs are few but
// their longest searches take as long as the rest of a mid-size join; in a launch of their own,
// after the others and a round trip to the host for their count, they took 1.6 of 10.2 ms for 1 M
// LogNormal molecules x 1,000 query graphs, now 9.7 in all; 300,000 x 306 1.93 -> 1.59 ms, the plain
// form's 150,000 x 300 1.63 -> 1.19 ms.
template <bool FIND_FIRST, class Src>
__global__ __launch_bounds__(64) void k_join_all(GraphDev q, GraphDev d, Src src, const uint32_t* __restrict__ indices,
                                                 const uint32_t* __restrict__ pair_graph, uint64_t P, uint32_t chunk,
                                                 int32_t* __restrict__ counts, unsigned long long* __restrict__ stats,
                                                 const unsigned long long* __restrict__ P_dev, const uint32_t* __restrict__ wide, uint64_t wide_cap,
                                                 const uint32_t* __restrict__ list, uint32_t cursor) {
  __shared__ alignas(16) unsigned char lds[kJoinAllLds];
  if (src.aborted()) return;
  if (P_dev) P = min(P, static_cast<uint64_t>(*P_dev));
  JoinTotals total;
  join_pass<FIND_FIRST, Src, kJoinWideLevels, true, true>(*reinterpret_cast<JoinLds<kJoinWideLevels, true, true>*>(lds), q, d, src, indices, pair_graph,
                                                          min(wide_cap, static_cast<uint64_t>(stats[kStatWide])), kWave, counts, stats, wide, nullptr,
                                                          kStatWideCursor, total);
  wave_sync();
  join_pass<FIND_FIRST, Src, kJoinLevels, true, false>(*reinterpret_cast<JoinLds<kJoinLevels, true, false>*>(lds), q, d, src, indices, pair_graph, P,
                                                       chunk, counts, stats, list, nullptr, cursor, total);
  join_totals(total, stats);
}

// Lists the pairs of molecules of > 64 nodes (the ranges of their molecules in offsets, at most P):
// a thread per molecule and turn, one atomic per block, a wavefront writes a molecule's range.
constexpr uint32_t kListTurns = 8;
__global__ __launch_bounds__(256) void k_list_wide(GraphDev d, const uint32_t* __restrict__ offsets, uint64_t P, uint32_t* __restrict__ wide,
                                                   unsigned long long* __restrict__ stats) {
  __shared__ uint32_t waves[4];
  __shared__ unsigned long long base;
  const uint32_t lane = static_cast<uint32_t>(lane_id()), wave = threadIdx.x / kWave;
  const uint64_t m0 = blockIdx.x * static_cast<uint64_t>(256 * kListTurns) + wave * kWave * kListTurns;
  uint32_t start[kListTurns], cnt[kListTurns], mine = 0;
#pragma unroll
  for (uint32_t t = 0; t < kListTurns; ++t) {
    const uint64_t m = m0 + t * kWave + lane;
    start[t] = cnt[t] = 0;
    if (m < d.G && d.go[m + 1] - d.go[m] > 64) {
      start[t] = static_cast<uint32_t>(min(P, static_cast<uint64_t>(offsets[m])));
      cnt[t] = static_cast<uint32_t>(min(P, static_cast<uint64_t>(offsets[m + 1]))) - start[t];
    }
    mine += cnt[t];
  }
  uint32_t incl = mine;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t y = static_cast<uint32_t>(__shfl_up(static_cast<int>(incl), o));
    if (lane >= static_cast<uint32_t>(o)) incl += y;
  }
  if (lane == kWave - 1) waves[wave] = incl;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t all = waves[0] + waves[1] + waves[2] + waves[3];
    base = all ? atomicAdd(&stats[kStatWide], static_cast<unsigned long long>(all)) : 0ull;
  }
  __syncthreads();
  uint64_t at = base + incl - mine;
  for (uint32_t x = 0; x < wave; ++x) at += waves[x];
#pragma unroll
  for (uint32_t t = 0; t < kListTurns; ++t) {
    for (uint64_t left = __ballot(cnt[t] != 0); left; left &= left - 1) {  // wave-uniform
      const int i = static_cast<int>(__builtin_ctzll(left));
      const uint32_t s = rl32(start[t], i), n = rl32(cnt[t], i);
      const uint64_t to = uniform64(__shfl(at, i));
      for (uint32_t x = lane; x < n; x += kWave) wide[to + x] = s + x;
    }
    at += cnt[t];
  }
}

// Wavefronts (one-wavefront blocks) for `pairs` pairs: as many as stay resident by LDS, or the
// tuned share of them in quarters, and no more than have a pair each.
inline uint64_t join_blocks(size_t lds, uint64_t pairs, int num_cus, uint32_t quarters) {
  const uint64_t cus = static_cast<uint64_t>(num_cus > 0 ? num_cus : 256);
  const uint64_t per_cu = std::max<uint64_t>(1, uint64_t(join_waves_per_cu(lds)) * quarters / 4);
  return std::max<uint64_t>(1, std::min<uint64_t>((pairs + 63) / 64, cus * per_cu));
}

// The lane join over P pairs.  With `deep` and enough pairs, a kJoinShallow-level pass over all of them
// lists the deeper queries' pairs, whose count the next pass reads on the device; otherwise one pass
// takes them all.  With `wide` (capacity P) the pairs of molecules of > 64 nodes are listed first and
// run with the last pass; null when the data has none.  `quarters` (1..4: share of the resident
// wavefronts) and chunk (0: ~4 claims per wavefront, ~8 behind wide pairs, at most 1024 pairs: a claim
// is an atomic on one address) shape the pass over all pairs.
template <bool FIND_FIRST, class Src>
hipError_t launch_join_passes(hipStream_t s, const GraphDev& q, const GraphDev& d, const Src& src, const uint32_t* offsets, const uint32_t* indices,
                              const uint32_t* pair_graph, uint64_t P, int32_t* counts, unsigned long long* stats, uint32_t* wide, int num_cus,
                              const unsigned long long* P_dev, uint32_t* deep, uint32_t quarters, uint32_t chunk) {
  const auto claim = [&](uint64_t blocks, uint32_t claims) {
    return chunk ? chunk : static_cast<uint32_t>(std::min<uint64_t>(1024, std::max<uint64_t>(64, P / (blocks * claims) / 64 * 64)));
  };
  if (wide) k_list_wide<<<(d.G + 256 * kListTurns - 1) / (256 * kListTurns), 256, 0, s>>>(d, offsets, P, wide, stats);
  const bool two = deep && P >= (P_dev || !FIND_FIRST ? kJoinTwoPassBound : kJoinTwoPassPairs);
  if (two) {
    const uint64_t blocks = join_blocks(sizeof(JoinLds<kJoinShallow, false, false>), P, num_cus, quarters);
    k_join_lanes<FIND_FIRST, Src, kJoinShallow, false><<<static_cast<unsigned>(blocks), 64, 0, s>>>(
        q, d, src, indices, pair_graph, P, claim(blocks, 4), counts, stats, P_dev, nullptr, deep, kStatCursor);
    P_dev = stats + kStatDeep;
    quarters = 4;
  }
  const uint32_t* list = two ? deep : nullptr;
  const uint32_t cursor = two ? kStatDeepCursor : kStatCursor;
  const uint64_t blocks = join_blocks(wide ? kJoinAllLds : sizeof(JoinLds<kJoinLevels, true, false>), P, num_cus, quarters);
  const uint32_t claims = two ? kJoinDeepChunk : claim(blocks, wide ? 8 : 4);
  if (wide)
    k_join_all<FIND_FIRST, Src><<<static_cast<unsigned>(blocks), 64, 0, s>>>(q, d, src, indices, pair_graph, P, claims, counts, stats, P_dev, wide, P,
                                                                             list, cursor);
  else
    k_join_lanes<FIND_FIRST, Src, kJoinLevels, true><<<static_cast<unsigned>(blocks), 64, 0, s>>>(q, d, src, indices, pair_graph, P, claims, counts,
                                                                                                  stats, P_dev, list, nullptr, cursor);
  return hipGetLastError();
}
template <class Src>
hipError_t launch_join_lanes(hipStream_t s, const GraphDev& q, const GraphDev& d, const Src& src, const uint32_t* offsets, const uint32_t* indices,
                             const uint32_t* pair_graph, uint64_t P, int find_first, int32_t* counts, unsigned long long* stats, uint32_t* wide,
                             int num_cus, const unsigned long long* P_dev, uint32_t* deep, uint32_t quarters, uint32_t chunk) {
  if (!P) return hipSuccess;
  return find_first ? launch_join_passes<true>(s, q, d, src, offsets, indices, pair_graph, P, counts, stats, wide, num_cus, P_dev, deep, quarters, chunk)
                    : launch_join_passes<false>(s, q, d, src, offsets, indices, pair_graph, P, counts, stats, wide, num_cus, P_dev, deep, quarters, chunk);
}

}  // namespace
}  // namespace sigmo_k
