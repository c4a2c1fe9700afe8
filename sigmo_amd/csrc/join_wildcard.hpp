// The reference's wildcard/edge-label join, joinWildcardCandidates (isomorphism.hpp:428-556),
// one lane per search from a candidate of the first node.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_common.hpp"
#include "join_lanes.hpp"
#include "kernels.hpp"

namespace sigmo_k {
namespace {

constexpr int kWildcardLevels = 8;
constexpr uint32_t kWildcardRefill = 16;  // free pair slots that make a wavefront load new pairs

template <bool WIDE>
struct WildcardLds {
  static constexpr int L = kWildcardLevels - 1;
  static constexpr int H = WIDE ? 2 : 1;
  // per lane: the DFS it runs
  uint64_t row[H][L][kWave];   // adjacency row of the position mapped at order position t
  uint64_t base[H][L][kWave];  // candidates frame t started from
  alignas(8) uint8_t map[kWave][40];
  // per pair slot
  uint64_t mask[H][L][kWave];  // candidate mask of order position t + 1
  unsigned long long count[kWave];
  uint32_t start[kWave], qoff[kWave], shape[kWave];  // molecule's first node; query's; nodes | k << 8 | first << 16
  uint32_t running[kWave];                           // searches taken and not yet done
  uint8_t root[kWave], turn[kWave];                  // the next search's root; slots by turn
};

// Per pair, as the reference kernel does per sub-group:
//  * matching order (defineMatchingOrder, :383-408): the query node with most candidates in
//    the molecule first (ties: the larger index; every k <= 32 node is considered, as with a
//    sub-group of >= 32 lanes), then the other nodes ascending;
//  * one DFS per candidate of that node (:495-548), each from fresh state (every mapping
//    entry = local node 0), summed into the pair's count; find-first ends a DFS at its first
//    leaf;
//  * a candidate is valid when, for every earlier node of the order, query and data adjacency
//    agree and adjacent pairs carry equal edge labels (isValidMapping, :410-426);
//  * an exhausted frame unsets its node's (possibly stale) mapping, and a pop that leaves one
//    frame resets `visited` to the first node's candidate (:521-526); `visited` is one word
//    indexed by position mod 64 (utils.hpp:71-73).
// A frame resumes after its last accepted candidate, which is what advancing the reference's
// candidate index past it does.
//
// A wavefront holds up to 64 pairs in slots, loaded together, and its lanes take the searches of
// their roots as they become idle, a lane per search: a pair's searches are independent, and the
// longest pair takes 1,600 accepts where the longest search takes 73 (20,011 molecules x 64 query
// graphs; means 60 and 5).  The frames are k_join_lanes's: an accept forms the next frame's
// candidates at once, from rows and masks in LDS, less the neighbours of a mapped query neighbour
// whose edge label differs from the query's; frames past the seventh read masks and rows from
// memory.  That join took 4.35 ms with a lane per pair and every step rereading masks, rows and
// labels from memory, 2.6 ms with a lane per pair in these frames, and 1.02 ms with a lane per search:
// what bounds it is the chain of dependent steps, few waves in flight by LDS.  A step's loads are
// therefore two deep: the row offsets with the adjacency and query rows, then four CSR entries of either
// side, and all levels' rows come from LDS together; 0.72 ms, where entry after entry and row after row
// were a dozen waits.  Loading a new pair's masks four at a time gave nothing.
// Molecules of <= 64 nodes (!WIDE; pairs of larger ones are listed in `wide`) or, with WIDE, the
// listed pairs of larger ones.
template <bool FIND_FIRST, bool WIDE>
__global__ __launch_bounds__(64) void k_join_wildcard(GraphDev q, GraphDev d, const uint8_t* __restrict__ qel, const uint8_t* __restrict__ del,
                                                      BitsetMasks src, const uint32_t* __restrict__ indices,
                                                      const uint32_t* __restrict__ pair_graph, uint64_t P, uint32_t chunk,
                                                      int32_t* __restrict__ counts, unsigned long long* __restrict__ stats,
                                                      uint32_t* __restrict__ wide, const uint32_t* __restrict__ list,
                                                      const unsigned long long* __restrict__ P_dev, uint32_t cursor) {
  constexpr uint32_t L = kWildcardLevels - 1;
  __shared__ WildcardLds<WIDE> sh;
  if (P_dev) P = min(P, static_cast<uint64_t>(*P_dev));
  const uint32_t lane = static_cast<uint32_t>(lane_id());
  const uint64_t below = (1ull << lane) - 1;
  const uint32_t* qfold = reinterpret_cast<const uint32_t*>(q.fold);  // query rows fit the low word (k <= 32)
  uint64_t sum = 0, matched = 0, overflow = 0;
  // a wavefront's first claim is its own, later ones come from the cursor
  uint64_t next = static_cast<uint64_t>(blockIdx.x) * chunk, end = next + chunk < P ? next + chunk : P;
  const uint64_t claimed = static_cast<uint64_t>(gridDim.x) * chunk;
  bool exhausted = false;
  // the lane's slot: its pair and the roots not yet taken
  bool held = false;
  uint32_t pj = 0;
  uint64_t roots = 0, roots_hi = 0;
  // the lane's search
  bool have = false;
  uint32_t slot = 0, s = 0, n = 0, qoff = 0, k = 0, first = 0, depth = 0;
  uint64_t visited = 0, count = 0, cur = 0, cur_hi = 0, rem = 0, rem_hi = 0;

  auto node_of = [&](uint32_t t) -> uint32_t { return t == 0 ? first : (t <= first ? t - 1 : t); };  // query node at order position t
  // the query row of order position t, its bits by order position
  auto query_row = [&](uint32_t t) -> uint32_t {
    const uint32_t r = qfold[2 * (static_cast<uint64_t>(qoff) + node_of(t))], bit = 1u << first;
    return ((r & (bit - 1u)) << 1) | ((r >> first) & 1u) | (r & ~(bit | (bit - 1u)));
  };
  auto node_mask = [&](uint32_t t, uint64_t& lo, uint64_t& hi) {  // the candidate mask of order position t >= 1
    if (t <= L) {
      lo = sh.mask[0][t - 1][slot];
      if constexpr (WIDE) hi = sh.mask[1][t - 1][slot];
    } else if constexpr (WIDE) {
      src.mask2(0, qoff + node_of(t), 0, s, n, lo, hi);
    } else {
      lo = src.mask(0, qoff + node_of(t), 0, s, n);
    }
  };
  // order position t's candidate set after the mapped positions below it: rows and, for query
  // neighbours, edge labels.  qr: t's query row; [vi, ve): the CSR row of the position mapped at t - 1
  auto frame = [&](uint32_t t, uint32_t qr, uint32_t vi, uint32_t ve, uint64_t& lo, uint64_t& hi) {
    node_mask(t, lo, hi);
    const uint32_t mapped = qr & ((1u << t) - 1u);
    auto group = [&](uint32_t x0, uint32_t x1) {
      uint64_t r[4], rh[4];
#pragma unroll
      for (uint32_t x = x0; x < x1; ++x) {
        r[x - x0] = sh.row[0][x][lane];
        if constexpr (WIDE) rh[x - x0] = sh.row[1][x][lane];
      }
#pragma unroll
      for (uint32_t x = x0; x < x1; ++x) {  // an empty row of no neighbour keeps every position
        const uint32_t a = bit_spread(mapped, x);
        lo = and_row(lo, x < t ? r[x - x0] : 0ull, a);
        if constexpr (WIDE) hi = and_row(hi, x < t ? rh[x - x0] : 0ull, a);
      }
    };
    group(0, 4);
    if (__any(t > 4)) group(4, L);
    for (uint32_t x = L; x < t; ++x) {
      const uint64_t v = static_cast<uint64_t>(s) + sh.map[lane][x];
      const uint32_t a = bit_spread(mapped, x);
      lo = and_row(lo, d.adj[2 * v], a);
      if constexpr (WIDE) hi = and_row(hi, d.adj[2 * v + 1], a);
    }
    const uint32_t qn = qoff + node_of(t);
    for (uint32_t nb = mapped; nb && (lo | hi); nb &= nb - 1) {
      const uint32_t x = static_cast<uint32_t>(__builtin_ctz(nb));
      const uint32_t qx = qoff + node_of(x), v = s + sh.map[lane][x];
      uint32_t qi = q.ro[qx], di = vi, de = ve;
      const uint32_t qe = q.ro[qx + 1];
      if (x + 1 != t) {
        di = d.ro[v];
        de = d.ro[v + 1];
      }
      // the label of the first CSR entry of the query edge (graph.hpp:88-93), 255 if none, and the data
      // row's neighbours: four entries each at a time, past the end the last one again
      uint32_t want = 0xFFu, dc[4], dl[4];
      if (di < de) {
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
          dc[u] = d.ci[min(di + u, de - 1)];
          dl[u] = del[min(di + u, de - 1)];
        }
      }
      for (bool found = false; qi < qe && !found; qi += 4) {
        uint32_t qc[4], ql[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
          qc[u] = q.ci[min(qi + u, qe - 1)];
          ql[u] = qel[min(qi + u, qe - 1)];
        }
#pragma unroll
        for (int u = 3; u >= 0; --u)
          if (qc[u] == qn) {
            want = ql[u];
            found = true;
          }
      }
      uint64_t seen_lo = 0, seen_hi = 0;  // neighbours whose first CSR entry has passed
      while (di < de) {
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
          const uint32_t c = dc[u] - s;
          const uint64_t bit = bit_of(c);
          if (!WIDE || c < 64) {
            if (!(seen_lo & bit) && dl[u] != want) lo &= ~bit;
            seen_lo |= bit;
          } else {
            if (!(seen_hi & bit) && dl[u] != want) hi &= ~bit;
            seen_hi |= bit;
          }
        }
        di += 4;
        if (di < de) {
#pragma unroll
          for (uint32_t u = 0; u < 4; ++u) {
            dc[u] = d.ci[min(di + u, de - 1)];
            dl[u] = del[min(di + u, de - 1)];
          }
        }
      }
    }
  };
  // Accepts c at `depth` and forms the next frame (or counts the leaf); true when the search ends.
  auto accept = [&](uint32_t c) -> bool {
    sh.map[lane][depth] = static_cast<uint8_t>(c);
    const uint32_t nd = depth + 1;
    if (nd == k) {
      ++count;
      return FIND_FIRST;
    }
    // what the next frame reads from memory first, issued together
    const uint64_t v = static_cast<uint64_t>(s) + c;
    const uint64_t rlo = d.adj[2 * v], rhi = WIDE ? d.adj[2 * v + 1] : 0ull;
    const uint32_t vi = d.ro[v], ve = d.ro[v + 1], qr = query_row(nd);
    if (depth < L) {
      sh.row[0][depth][lane] = rlo;
      sh.base[0][depth][lane] = cur;
      if constexpr (WIDE) {
        sh.row[1][depth][lane] = rhi;
        sh.base[1][depth][lane] = cur_hi;
      }
    }
    uint64_t nlo = 0, nhi = 0;
    frame(nd, qr, vi, ve, nlo, nhi);
    if ((nlo & ~visited) | (WIDE ? nhi & ~visited : 0ull)) {
      depth = nd;
      cur = nlo;
      cur_hi = nhi;
      rem = rem_hi = ~0ull;
      return false;
    }
    // it would be exhausted at once
    visited &= ~bit_of(sh.map[lane][nd]);
    if (depth == 1) visited = bit_of(sh.map[lane][0]);
    return depth == 0;
  };

  while (true) {
    uint64_t idle = __ballot(!have);
    // finished pairs leave their slots; new ones are loaded when the slots' roots no longer feed the
    // idle lanes
    if (__popcll(idle) > __popcll(__ballot(held && (roots | roots_hi)))) {  // wave-uniform
      if (held && !(roots | roots_hi) && sh.running[lane] == 0) {
        const uint64_t total = sh.count[lane];
        if (total > 0x7FFFFFFFull) overflow = 1;
        counts[pj] = static_cast<int32_t>(total > 0x7FFFFFFFull ? 0x7FFFFFFFull : total);
        sum += total;
        matched += total > 0;
        held = false;
      }
      const uint64_t room = __ballot(!held);
      if (!exhausted && (static_cast<uint32_t>(__popcll(room)) >= kWildcardRefill || idle == ~0ull)) {
        if (next >= end && claimed < P) {
          unsigned long long b = 0;
          if (lane == 0) b = atomicAdd(&stats[cursor], static_cast<unsigned long long>(chunk));
          next = claimed + uniform64(__shfl(b, 0));
          end = next + chunk < P ? next + chunk : P;
        }
        if (next >= end) {
          exhausted = true;
        } else {
          const uint32_t cnt = min(static_cast<uint32_t>(end - next), static_cast<uint32_t>(__popcll(room)));
          const uint32_t rn = __popcll(room & below);
          const bool take = !held && rn < cnt;
          bool wide_pair = false;
          uint32_t ps = 0, pn = 0, pq = 0, pk = 0;
          if (take) {
            pj = list ? list[next + rn] : static_cast<uint32_t>(next + rn);
            const uint32_t dg = pair_graph[pj], qg = indices[pj];
            ps = d.go[dg];
            pn = d.go[dg + 1] - ps;
            pq = q.go[qg];
            pk = q.go[qg + 1] - pq;
            wide_pair = !WIDE && pn > 64;
          }
          next += cnt;
          if constexpr (!WIDE) {
            const uint64_t wm = __ballot(wide_pair);
            if (wm) {
              unsigned long long b = 0;
              if (lane == 0) b = atomicAdd(&stats[kStatWide], static_cast<unsigned long long>(__popcll(wm)));
              const uint64_t wb = uniform64(__shfl(b, 0));
              if (wide_pair) wide[wb + __popcll(wm & below)] = pj;
            }
          }
          if (take && !wide_pair) {
            // the first node of the matching order, then the masks by order position
            uint32_t maxc = 0, lead = 0;
            for (uint32_t t = 0; t < pk; ++t) {
              uint64_t lo = 0, hi = 0;
              if constexpr (WIDE) src.mask2(0, pq + t, 0, ps, pn, lo, hi);
              else lo = src.mask(0, pq + t, 0, ps, pn);
              const uint32_t c = static_cast<uint32_t>(__popcll(lo) + __popcll(hi));
              // until a later node takes its place as the first, node t's order position is t + 1
              if (t < L) {
                sh.mask[0][t][lane] = lo;
                if constexpr (WIDE) sh.mask[1][t][lane] = hi;
              }
              if (c >= maxc) {
                maxc = c;
                lead = t;
                roots = lo;
                roots_hi = hi;
              }
            }
            // nodes after the first keep their index as order position: masks move one place down
            for (uint32_t t = lead + 1; t < pk && t <= L; ++t) {
              uint64_t lo = 0, hi = 0;
              if (t < L) {
                lo = sh.mask[0][t][lane];
                if constexpr (WIDE) hi = sh.mask[1][t][lane];
              } else if constexpr (WIDE) {
                src.mask2(0, pq + t, 0, ps, pn, lo, hi);
              } else {
                lo = src.mask(0, pq + t, 0, ps, pn);
              }
              sh.mask[0][t - 1][lane] = lo;
              if constexpr (WIDE) sh.mask[1][t - 1][lane] = hi;
            }
            sh.start[lane] = ps;
            sh.qoff[lane] = pq;
            sh.shape[lane] = pn | (pk << 8) | (lead << 16);
            sh.count[lane] = 0;
            sh.running[lane] = 0;
            held = true;
          }
        }
      }
      if (exhausted && __ballot(held || have) == 0) break;
    }
    // each slot with roots left hands one to an idle lane
    const uint64_t ready = __ballot(held && (roots | roots_hi));
    if (ready && idle) {  // wave-uniform
      const uint32_t cnt = min(static_cast<uint32_t>(__popcll(ready)), static_cast<uint32_t>(__popcll(idle)));
      const uint32_t rank = __popcll(ready & below);
      if (((ready >> lane) & 1ull) && rank < cnt) {
        uint32_t c;
        if (roots) {
          c = static_cast<uint32_t>(__builtin_ctzll(roots));
          roots &= roots - 1;
        } else {
          c = 64u + static_cast<uint32_t>(__builtin_ctzll(roots_hi));
          roots_hi &= roots_hi - 1;
        }
        sh.root[lane] = static_cast<uint8_t>(c);
        sh.turn[rank] = static_cast<uint8_t>(lane);
        atomicAdd(&sh.running[lane], 1u);
      }
      wave_sync();
      const uint32_t rn = __popcll(idle & below);
      if (!have && rn < cnt) {  // a search from one root, from fresh state
        slot = sh.turn[rn];
        s = sh.start[slot];
        qoff = sh.qoff[slot];
        n = sh.shape[slot] & 0xFFu;
        k = (sh.shape[slot] >> 8) & 0xFFu;
        first = sh.shape[slot] >> 16;
        const uint32_t c = sh.root[slot];
#pragma unroll
        for (int t = 0; t < 32; t += 8) *reinterpret_cast<uint64_t*>(&sh.map[lane][t]) = 0;  // every entry: local node 0
        visited = bit_of(c);
        count = 0;
        depth = 0;
        have = !accept(c);  // queries have two nodes or more: no leaf yet
        if (!have) atomicSub(&sh.running[slot], 1u);
      }
      wave_sync();
    }
    if (have) {
      bool done = false;
      uint64_t el = cur & ~visited & rem, eh = WIDE ? cur_hi & ~visited & rem_hi : 0ull;
      if ((el | eh) == 0) {  // exhausted frame: pop
        visited &= ~bit_of(sh.map[lane][depth]);
        --depth;
        if (depth == 0) {
          done = true;
        } else {
          if (depth == 1) visited = bit_of(sh.map[lane][0]);
          const uint32_t c = sh.map[lane][depth];
          if (depth < L) {
            cur = sh.base[0][depth][lane];
            if constexpr (WIDE) cur_hi = sh.base[1][depth][lane];
          } else {
            const uint32_t v = s + sh.map[lane][depth - 1];
            frame(depth, query_row(depth), d.ro[v], d.ro[v + 1], cur, cur_hi);
          }
          rem = c < 64 ? bits_above(c) : 0ull;
          rem_hi = c < 64 ? ~0ull : bits_above(c - 64);
          el = cur & ~visited & rem;
          eh = WIDE ? cur_hi & ~visited & rem_hi : 0ull;
        }
      }
      if (!done && (el | eh)) {
        const uint32_t c = el ? static_cast<uint32_t>(__builtin_ctzll(el)) : 64u + static_cast<uint32_t>(__builtin_ctzll(eh));
        rem = c < 64 ? bits_above(c) : 0ull;
        rem_hi = c < 64 ? ~0ull : bits_above(c - 64);
        visited |= bit_of(c);
        done = accept(c);
      }
      if (done) {
        if (count) atomicAdd(&sh.count[slot], static_cast<unsigned long long>(count));
        atomicSub(&sh.running[slot], 1u);
        have = false;
      }
    }
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    sum += __shfl_xor(sum, o);
    matched += __shfl_xor(matched, o);
    overflow |= __shfl_xor(overflow, o);
  }
  if (lane == 0) {
    if (sum) atomicAdd(&stats[0], static_cast<unsigned long long>(sum));
    if (matched) atomicAdd(&stats[1], static_cast<unsigned long long>(matched));
    if (overflow) atomicOr(&stats[3], 1ull);
  }
}

}  // namespace
}  // namespace sigmo_k
