// Batched (non-materialising) form of SIGMo's filter -> refine -> GMCR -> join.
//
// The plain form writes a Q x D candidate bitset and passes over it 2R+2 times; after R = 6
// levels ~1% of its bits are set and ~8% of the (query graph, molecule) pairs survive GMCR.
// The batched form computes, for each (query graph, molecule) pair, the refined candidate
// mask of each query node directly inside the molecule, from level signatures prepared once
// per molecule, and stops at the first query node with no candidate -- the GMCR predicate of
// gmcr.hpp:56-61 (every query node has a candidate in the molecule).  Survivors keep their
// per-node masks, which are exactly the molecule-range slices of the plain form's rows, so
// GMCR and join results are identical.
//
// Semantics per query node q and molecule position p (paths relative to the SIGMo repository):
//   label(q) == label(p) or label(q) == 255                         isomorphism.hpp:49
//   for r = 1..R, for l < 16: sig_r(q)[l] <= sig_r(p)[l]             isomorphism.hpp:103-110
// with sig_r the PowerGraph level-r signature of signature.hpp:336-390 (sphere at BFS distance
// r over positions mod 64, labels read through the 64-position view).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <type_traits>
#include <chrono>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/iterator/counting_iterator.hpp>

#include "../../include/sigmo_hip.h"
#include "device_common.hpp"
#include "host_graphs.hpp"
#include "join_lanes.hpp"
#include "kernels.hpp"

namespace sigmo_k {
namespace {

constexpr uint32_t kMaxLevels = 8;        // token encoding keeps 3 bits of level
constexpr uint16_t kEndToken = 0xFFFF;    // closes a query node's token segment

// Tokens of one query node: [label] [requirement]* [end] .., with end tokens up to a whole quad of
// four.  A token is a plane of a label (6 bits) and a key, label | kind << 4 (6 bits): requirements of
// counts 1..4 (kind 0) and 5..8 (1) name plane 4 r + (c - 1) % 4 of level r < 8, larger counts (2) hold
// r and c - 8 there; the label token of a label < 16 is its plane 4 R; kind 3 has the end (key 63),
// the wildcard label (49) and the other labels (50, the label's upper bits above the key).
constexpr uint32_t kKeyWildcard = 49, kKeyOther = 50;
__device__ __forceinline__ uint32_t requirement_token(uint32_t r, uint32_t l, uint32_t c) {
  return (c <= 8 ? ((c - 1) & 3u) | (r << 2) | (((c - 1) >> 2) << 10) : r | ((c - 8) << 3) | (2u << 10)) | (l << 6);
}
__device__ __forceinline__ uint32_t token_level(uint32_t t) { return (t >> 10) == 2 ? t & 7u : (t >> 2) & 7u; }
__device__ __forceinline__ uint32_t token_count(uint32_t t) { return (t >> 10) == 2 ? 8 + ((t >> 3) & 7u) : 1 + (t & 3u) + 4 * (t >> 10); }
__device__ __forceinline__ uint32_t token_label(uint32_t t) { return (t >> 6) & 15u; }
__device__ __forceinline__ uint32_t label_token(uint32_t label, uint32_t R) {
  if (label < 16) return 4 * R | (label << 6);
  return label == 255 ? kKeyWildcard << 6 : (label & 63u) | (kKeyOther << 6) | ((label >> 6) << 12);
}
// The label of a label token, 255 for the wildcard.
__device__ __forceinline__ uint32_t labelled(uint32_t t) {
  const uint32_t key = (t >> 6) & 63u;
  return key < 16 ? key : (key == kKeyWildcard ? 255u : (t & 63u) | ((t >> 12) << 6));
}
__host__ __device__ constexpr uint32_t token_segment(uint32_t R) { return ((2 + 16 * R + 3) & ~3u) + 4; }

// Bit 0 of every nonzero nibble.
__device__ __forceinline__ uint64_t nibbles_set(uint64_t x) {
  x |= x >> 2;
  return (x | (x >> 1)) & 0x1111111111111111ull;
}

// 16 four-bit label counts of the nodes in r (labels >= 16 are not counted; counts saturate
// at 15), signature.hpp:44-51.
__device__ __forceinline__ uint64_t histogram16(uint64_t r, const uint64_t* __restrict__ lm) {
  uint64_t s = 0;
#pragma unroll
  for (int l = 0; l < 16; ++l) {
    uint32_t c = __popcll(r & lm[l]);
    c = c < 15 ? c : 15;
    s |= static_cast<uint64_t>(c) << (4 * l);
  }
  return s;
}

// Nibble-wise max.
__device__ __forceinline__ uint64_t nib_max(uint64_t a, uint64_t b) {
  constexpr uint64_t L = 0x0F0F0F0F0F0F0F0Full, H = 0x1010101010101010ull;
  const uint64_t ae = a & L, be = b & L, ao = (a >> 4) & L, bo = (b >> 4) & L;
  const uint64_t me = ((((ae | H) - be) & H) >> 4) * 0xFull;  // 0x0F in the fields where a >= b
  const uint64_t mo = ((((ao | H) - bo) & H) >> 4) * 0xFull;
  return ((ae & me) | (be & ~me)) | (((ao & mo) | (bo & ~mo)) << 4);
}

__device__ __forceinline__ uint64_t wave_nib_max(uint64_t x) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) x = nib_max(x, static_cast<uint64_t>(__shfl_xor(static_cast<unsigned long long>(x), o)));
  return x;
}


// Per-molecule facts the pair filter reads, stored in width-class order.
struct alignas(16) MolInfo {
  uint32_t m, s, n, mlab;  // molecule, first node, nodes, labels < 16 present
};

// Per-query-graph facts the pair pre-test reads.
struct QueryInfo {
  uint32_t qoff, k, qlab, qcls;  // first node, nodes, labels < 16 present, signature classes present (bit c)
};

// The database's signature classes: up to three labels (< 16), the database's most frequent, for
// which the pre-test keeps per-label maxima (l[c] = 0xFFFFFFFF: class c unused).
constexpr uint32_t kClasses = 3;
struct ClassLabels {
  uint32_t l[kClasses];
};

// Nibble-wise max over the 64 positions of a level signature, from its transposed planes (lane i
// holds plane i = bit i%4 of the count of label i/4): lane 4l reads the label's other three
// planes and takes the largest 4-bit value greedily from the top bit; four ballots then place
// bit b of label l's max at bit 4l + b.
__device__ __forceinline__ uint64_t planes_nib_max(uint64_t col) {
  const uint32_t lane = static_cast<uint32_t>(lane_id());
  const uint64_t p1 = static_cast<uint64_t>(__shfl_down(static_cast<unsigned long long>(col), 1));
  const uint64_t p2 = static_cast<uint64_t>(__shfl_down(static_cast<unsigned long long>(col), 2));
  const uint64_t p3 = static_cast<uint64_t>(__shfl_down(static_cast<unsigned long long>(col), 3));
  const uint64_t planes[4] = {col, p1, p2, p3};
  uint64_t cand = ~0ull;
  uint32_t v = 0;
#pragma unroll
  for (int b = 3; b >= 0; --b) {
    const uint64_t t = cand & planes[b];
    if (t) {
      v |= 1u << b;
      cand = t;
    }
  }
  const bool leader = (lane & 3u) == 0;
  uint64_t mx = 0;
#pragma unroll
  for (int b = 0; b < 4; ++b) mx |= __ballot(leader && ((v >> b) & 1u)) << b;
  return mx;
}

// One wavefront per molecule: lane p is position p (and p+64 for molecules of 65..128 nodes).
// The sort key of the width-class order: class (<= 32, 33..64, 65..128 nodes) << 23 | the
// molecule's label set (labels < 16) << 7 | (nodes - 1).  Sorted, molecules of one label set and
// similar size share wavefronts, so the pre-test's label test (and, mostly, its maxima tests)
// passes or fails for whole wavefronts and the tests after a failing one are skipped.
__global__ __launch_bounds__(256) void k_db_order_keys(uint32_t G, const uint32_t* __restrict__ go, const uint8_t* __restrict__ nl,
                                                       uint32_t* __restrict__ keys) {
  const uint64_t m = blockIdx.x * 256ull + threadIdx.x;
  if (m >= G) return;
  const uint32_t s = go[m], n = go[m + 1] - s;
  uint32_t labels = 0;
  for (uint32_t p = 0; p < n; ++p) {
    const uint32_t l = nl[s + p];
    if (l < 16) labels |= 1u << l;
  }
  const uint32_t cls = n <= 32 ? 0u : (n <= 64 ? 1u : 2u);
  keys[m] = (cls << 23) | (labels << 7) | ((n - 1) & 127u);
}

// The level planes are laid out for 64-lane groups of the width-class order.  A lane holds 32
// positions of a molecule: molecules of <= 32 nodes take one lane, of 33..64 two, wider ones four,
// so a group is 64, 32 or 16 neighbours of one class (the last group of a class may be short).
// planes[((group*R + r)*16 + l)*64 + lane] is the four plane words (bits 0..3 of the count of label
// l at level r+1) of the lane's positions, labs[(group*16 + l)*64 + lane] its positions labelled l:
// a group's words of one level and label are one coalesced kilobyte.
struct GroupOrder {
  uint32_t count[3];  // molecules of <= 32, 33..64 and 65..128 nodes, one class after another
  __host__ __device__ uint32_t groups(int cls) const { return (count[cls] + (64u >> cls) - 1) / (64u >> cls); }
  __host__ __device__ uint32_t total() const { return groups(0) + groups(1) + groups(2); }
};
// Group and first lane of the `at`-th molecule of a class.
__device__ __forceinline__ void group_place(const GroupOrder& o, int cls, uint32_t at, uint64_t& group, uint32_t& lane0) {
  const uint32_t per = 64u >> cls;
  group = at / per + (cls > 0 ? o.groups(0) : 0u) + (cls > 1 ? o.groups(1) : 0u);
  lane0 = (at % per) << cls;
}

// One wavefront per molecule of more than 32 nodes (width-class entries c0 and up), lane p =
// position p (and p+64 for molecules of 65..128 nodes): writes the molecule's planes and label
// masks, minfo[c], dmax[c*R + r], the nibble-wise max of the level-(r+1) signatures over the
// molecule's positions, and cmax[(k*R + r)*G + c], the same max over the positions labelled
// cl.l[k] (0 if none).
__global__ __launch_bounds__(256) void k_db_prepare(GraphDev g, uint32_t R, const uint32_t* __restrict__ cls_list, GroupOrder order,
                                                    uint32_t* __restrict__ planes, uint32_t* __restrict__ labs,
                                                    uint64_t* __restrict__ dmax, MolInfo* __restrict__ minfo, ClassLabels cl,
                                                    uint64_t* __restrict__ cmax, uint32_t c0) {
  __shared__ uint64_t fold_all[4][kWave];
  const uint32_t lane = static_cast<uint32_t>(lane_id());
  const uint64_t c = c0 + static_cast<uint64_t>(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (c >= g.G) return;  // wave-uniform
  const uint64_t m = cls_list[c];
  const uint32_t s = g.go[m], n = g.go[m + 1] - s;
  const int cls = c < static_cast<uint64_t>(order.count[0]) + order.count[1] ? 1 : 2;
  uint64_t group;
  uint32_t lane0;
  group_place(order, cls, static_cast<uint32_t>(c - order.count[0] - (cls > 1 ? order.count[1] : 0u)), group, lane0);
  const uint64_t* lm = g.lmask + m * 16;
  // the label masks of positions 0..63 and the labels that occur there (wave-uniform): the
  // histogram only visits those labels
  uint64_t lmv[16];
  uint32_t present = 0;
#pragma unroll
  for (int l = 0; l < 16; ++l) {
    lmv[l] = lm[l];
    if (lmv[l]) present |= 1u << l;
  }
  // Only positions 0..63 are ever expanded (frontier bit b expands node s + b), each by its
  // neighbours folded mod 64: stage those 64 words in LDS once.
  uint64_t* fold = fold_all[threadIdx.x / kWave];
  fold[lane] = lane < n ? g.fold[static_cast<uint64_t>(s) + lane] : 0ull;
  wave_sync();
  uint32_t labels = 0;
  for (uint32_t h = 0; h < static_cast<uint32_t>(cls); ++h) {
    const uint32_t pos = lane + 64 * h;
    const bool valid = pos < n;
    const uint32_t mylab = valid ? g.nl[s + pos] : 0x100u;
    if (mylab < 16) labels |= 1u << mylab;
    uint64_t cpos[kClasses];  // this half's positions of each class label
#pragma unroll
    for (uint32_t k = 0; k < kClasses; ++k) cpos[k] = __ballot(mylab == cl.l[k]);
    uint64_t self = 1ull << (pos & 63), ball = self, frontier = self;
    for (uint32_t r = 0; r < R; ++r) {
      uint64_t sig = 0;
      if (valid) {
        uint64_t next = 0;
        for (uint64_t f = frontier; f; f &= f - 1) next |= fold[__builtin_ctzll(f)];
        next &= ~ball;
        ball |= next;
        frontier = next;
#pragma unroll
        for (int l = 0; l < 16; ++l)
          if ((present >> l) & 1u) {  // counts saturate at 15 (signature.hpp:44-51)
            uint32_t cnt = __popcll(next & lmv[l]);
            cnt = cnt < 15 ? cnt : 15;
            sig |= static_cast<uint64_t>(cnt) << (4 * l);
          }
      }
      const uint64_t col = transpose64(sig);  // lane i: plane i = 4*label + bit over the 64 positions
      uint32_t* dst = planes + ((((group * R + r) * 16 + (lane >> 2)) * 64 + lane0 + 2 * h) * 4 + (lane & 3u));
      dst[0] = static_cast<uint32_t>(col);
      dst[4] = static_cast<uint32_t>(col >> 32);
      const uint64_t mx = planes_nib_max(col);
      if (lane == 0) dmax[c * R + r] = h == 0 ? mx : nib_max(dmax[c * R + r], mx);
#pragma unroll
      for (uint32_t k = 0; k < kClasses; ++k) {
        const uint64_t cm = planes_nib_max(col & cpos[k]);
        uint64_t* cd = cmax + (static_cast<uint64_t>(k) * R + r) * g.G + c;
        if (lane == 0) *cd = h == 0 ? cm : nib_max(*cd, cm);
      }
    }
    uint64_t mine = 0;
#pragma unroll
    for (int l = 0; l < 16; ++l) {
      const uint64_t b = __ballot(mylab == static_cast<uint32_t>(l));
      if (lane == static_cast<uint32_t>(l)) mine = b;
    }
    if (lane < 16) {
      uint32_t* dst = labs + (group * 16 + lane) * 64 + lane0 + 2 * h;
      dst[0] = static_cast<uint32_t>(mine);
      dst[1] = static_cast<uint32_t>(mine >> 32);
    }
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) labels |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(labels), o));
  if (lane == 0) {
    MolInfo info;
    info.m = static_cast<uint32_t>(m);
    info.s = s;
    info.n = n;
    info.mlab = labels;
    minfo[c] = info;
  }
}

// planes_nib_max of the two 32-position halves of a plane column at once (positions 0..31 and
// 32..63 of `col`): the nibble-wise maxima over each half's positions.
__device__ __forceinline__ void planes_nib_max2(uint64_t col, uint64_t& lo, uint64_t& hi) {
  const uint32_t lane = static_cast<uint32_t>(lane_id());
  const uint64_t p1 = static_cast<uint64_t>(__shfl_down(static_cast<unsigned long long>(col), 1));
  const uint64_t p2 = static_cast<uint64_t>(__shfl_down(static_cast<unsigned long long>(col), 2));
  const uint64_t p3 = static_cast<uint64_t>(__shfl_down(static_cast<unsigned long long>(col), 3));
  const uint64_t planes[4] = {col, p1, p2, p3};
  uint32_t ca = ~0u, cb = ~0u, va = 0, vb = 0;
#pragma unroll
  for (int b = 3; b >= 0; --b) {
    const uint32_t ta = ca & static_cast<uint32_t>(planes[b]), tb = cb & static_cast<uint32_t>(planes[b] >> 32);
    if (ta) {
      va |= 1u << b;
      ca = ta;
    }
    if (tb) {
      vb |= 1u << b;
      cb = tb;
    }
  }
  const bool leader = (lane & 3u) == 0;
  lo = hi = 0;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    lo |= __ballot(leader && ((va >> b) & 1u)) << b;
    hi |= __ballot(leader && ((vb >> b) & 1u)) << b;
  }
}

// k_db_prepare for molecules of <= 32 nodes, two per wavefront: lanes 0..31 hold the positions of
// width-class entry 2v, lanes 32..63 those of 2v+1 (none past `count`).  Each lane's BFS runs over
// its own molecule's positions; one 64 x 64 transpose gives both molecules' level planes (low and
// high 32 bits of each plane word), so the transposes, and the lanes, serve two molecules.
__global__ __launch_bounds__(256) void k_db_prepare_pairs(GraphDev g, uint32_t R, uint32_t count, const uint32_t* __restrict__ cls_list,
                                                          uint32_t* __restrict__ planes, uint32_t* __restrict__ labs,
                                                          uint64_t* __restrict__ dmax, MolInfo* __restrict__ minfo, ClassLabels cl,
                                                          uint64_t* __restrict__ cmax) {
  __shared__ uint64_t fold_all[4][kWave];
  const uint32_t lane = static_cast<uint32_t>(lane_id());
  const uint64_t v = static_cast<uint64_t>(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave;
  const uint64_t cA = 2 * v, cB = cA + 1;
  if (cA >= count) return;  // wave-uniform
  const bool hasB = cB < count;
  const uint32_t half = lane >> 5, p = lane & 31u;
  const uint64_t c = half ? cB : cA;
  const bool live = !half || hasB;
  const uint64_t m = live ? cls_list[c] : 0;
  const uint32_t s = live ? g.go[m] : 0, n = live ? g.go[m + 1] - s : 0;
  const uint64_t* lm = g.lmask + m * 16;
  uint64_t lmv[16];
  uint32_t present = 0;
#pragma unroll
  for (int l = 0; l < 16; ++l) {
    lmv[l] = live ? lm[l] : 0ull;
    if (lmv[l]) present |= 1u << l;
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) present |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(present), o));
  uint64_t* fold = fold_all[threadIdx.x / kWave];
  fold[lane] = p < n ? g.fold[static_cast<uint64_t>(s) + p] : 0ull;
  wave_sync();
  const uint64_t* myfold = fold + 32 * half;
  const bool valid = p < n;
  const uint32_t mylab = valid ? g.nl[s + p] : 0x100u;
  uint32_t labels = mylab < 16 ? 1u << mylab : 0u;
  uint64_t cpos[kClasses];
#pragma unroll
  for (uint32_t k = 0; k < kClasses; ++k) cpos[k] = __ballot(mylab == cl.l[k]);
  const uint64_t group = cA / 64;  // both molecules, on neighbouring lanes
  const uint32_t lane0 = static_cast<uint32_t>(cA % 64);
  uint64_t self = 1ull << p, ball = self, frontier = self;
  for (uint32_t r = 0; r < R; ++r) {
    uint64_t sig = 0;
    if (valid) {
      uint64_t next = 0;
      for (uint64_t f = frontier; f; f &= f - 1) next |= myfold[__builtin_ctzll(f)];
      next &= ~ball;
      ball |= next;
      frontier = next;
#pragma unroll
      for (int l = 0; l < 16; ++l)
        if ((present >> l) & 1u) {  // counts saturate at 15 (signature.hpp:44-51)
          uint32_t cnt = __popcll(next & lmv[l]);
          cnt = cnt < 15 ? cnt : 15;
          sig |= static_cast<uint64_t>(cnt) << (4 * l);
        }
    }
    const uint64_t col = transpose64(sig);
    uint32_t* dst = planes + ((((group * R + r) * 16 + (lane >> 2)) * 64 + lane0) * 4 + (lane & 3u));
    dst[0] = static_cast<uint32_t>(col);
    if (hasB) dst[4] = static_cast<uint32_t>(col >> 32);
    uint64_t ma, mb;
    planes_nib_max2(col, ma, mb);
    if (lane == 0) dmax[cA * R + r] = ma;
    if (lane == 1 && hasB) dmax[cB * R + r] = mb;
#pragma unroll
    for (uint32_t k = 0; k < kClasses; ++k) {
      planes_nib_max2(col & cpos[k], ma, mb);
      if (lane == 0) cmax[(static_cast<uint64_t>(k) * R + r) * g.G + cA] = ma;
      if (lane == 1 && hasB) cmax[(static_cast<uint64_t>(k) * R + r) * g.G + cB] = mb;
    }
  }
  uint64_t mine = 0;
#pragma unroll
  for (int l = 0; l < 16; ++l) {
    const uint64_t b = __ballot(mylab == static_cast<uint32_t>(l));
    if (lane == static_cast<uint32_t>(l)) mine = b;
  }
  if (lane < 16) {
    uint32_t* dst = labs + (group * 16 + lane) * 64 + lane0;
    dst[0] = static_cast<uint32_t>(mine);
    if (hasB) dst[1] = static_cast<uint32_t>(mine >> 32);
  }
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) labels |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(labels), o));  // within each half
  if (p == 0 && live) {
    MolInfo info;
    info.m = static_cast<uint32_t>(m);
    info.s = s;
    info.n = n;
    info.mlab = labels;
    minfo[c] = info;
  }
}

// One wavefront per query graph, lane i = node i (query graphs have <= 32 nodes, so
// positions never alias): writes each node's tokens, the graph's label set (labels < 16) and,
// per level, the nibble-wise max of its nodes' signatures.  The graph's nodes' token streams
// are packed one after another from the start of its region (token qoff * segment), each padded
// to a whole token word (4 tokens), so a pair walks one contiguous run of words: the next node
// starts at the word after the one holding the current node's end token.
__global__ __launch_bounds__(256) void k_query_prepare(GraphDev q, uint32_t R, uint16_t* __restrict__ tokens,
                                                       QueryInfo* __restrict__ qinfo, uint64_t* __restrict__ qmax) {
  __shared__ uint64_t fold_all[4][kWave];
  const uint32_t lane = static_cast<uint32_t>(lane_id());
  const uint64_t g = static_cast<uint64_t>(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (g >= q.G) return;  // wave-uniform; no block barrier follows
  const uint32_t prev = q.go[g], k = q.go[g + 1] - prev;
  const bool valid = lane < k;
  const uint32_t seg = token_segment(R);
  const uint32_t label = valid ? q.nl[prev + lane] : 0u;
  // the graph's adjacency in LDS: a level's expansion then waits on no memory
  uint64_t* fold = fold_all[threadIdx.x / kWave];
  fold[lane] = valid ? q.fold[static_cast<uint64_t>(prev) + lane] : 0ull;
  wave_sync();
  // the node's level signatures, and its token count: label + one per nonzero nibble + end
  uint64_t sig[kMaxLevels];
  uint64_t self = 1ull << (lane & 63), ball = self, frontier = valid ? self : 0ull;
  uint32_t ntok = 2;
#pragma unroll
  for (uint32_t r = 0; r < kMaxLevels; ++r) {
    sig[r] = 0;
    if (r < R) {
      uint64_t next = 0;
      for (; frontier; frontier &= frontier - 1) next |= fold[__builtin_ctzll(frontier)];
      next &= ~ball;
      ball |= next;
      frontier = next;
      if (next) sig[r] = histogram16(next, q.lmask + g * 16);
      ntok += static_cast<uint32_t>(__popcll(nibbles_set(sig[r])));
      const uint64_t mx = wave_nib_max(sig[r]);
      if (lane == 0) qmax[g * R + r] = mx;
    }
  }
  // exclusive scan of the padded lengths over the graph's nodes
  const uint32_t len = valid ? (ntok + 3) & ~3u : 0u;
  uint32_t incl = len;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t y = static_cast<uint32_t>(__shfl_up(static_cast<int>(incl), o));
    if (lane >= static_cast<uint32_t>(o)) incl += y;
  }
  uint16_t* t = tokens + static_cast<uint64_t>(prev) * seg + (incl - len);
  if (valid) {
    t[0] = static_cast<uint16_t>(label_token(label, R));
    for (uint32_t x = ntok - 1; x < len; ++x) t[x] = kEndToken;
    uint32_t at = 1;
#pragma unroll
    for (uint32_t r = 0; r < kMaxLevels; ++r)
      if (r < R)
        for (uint64_t nz = nibbles_set(sig[r]); nz; nz &= nz - 1) {
          const uint32_t sh = static_cast<uint32_t>(__builtin_ctzll(nz)), c = static_cast<uint32_t>(sig[r] >> sh) & 15u;
          t[at++] = static_cast<uint16_t>(requirement_token(r, sh / 4, c));
        }
  }
  uint32_t bits = valid && label < 16 ? 1u << label : 0u;
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) bits |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(bits), o));
  if (lane == 0) {
    QueryInfo info;
    info.qoff = prev;
    info.k = k;
    info.qlab = bits;
    info.qcls = 0;  // set by k_query_classes
    qinfo[g] = info;
  }
}

// The per-class signature maxima the pre-test reads, from the query graphs' token streams
// (k_query_prepare's output: each requirement token carries one nonzero count, of label l at
// level r, of its node's signature, and every (r, l) occurs at most once per node, so the max over
// a class's nodes is the max over their tokens).  qcmax[(g*3 + c)*R + r] is the nibble-wise max
// of the level-(r+1) signatures of graph g's nodes labelled cl.l[c], and bit c of qinfo[g].qcls is
// set when there is such a node.  One wavefront per graph reads the graph's token words 64 at a
// time, a word per lane: a node's stream starts on a word boundary with its label token and its
// last word holds the end token (which no label or requirement token equals), so the words that
// hold an end token delimit the nodes and give each word its node's label.  Counts go to per-class
// LDS maxima by atomic max; lanes then pack them into nibbles.
__global__ __launch_bounds__(256) void k_query_classes(uint32_t Gq, uint32_t R, const uint64_t* __restrict__ tok64, ClassLabels cl,
                                                       QueryInfo* __restrict__ qinfo, uint64_t* __restrict__ qcmax) {
  constexpr uint32_t kSlots = kClasses * kMaxLevels * 16;
  __shared__ uint32_t cnt_all[4][kSlots];
  const uint32_t lane = static_cast<uint32_t>(lane_id());
  const uint32_t wave = threadIdx.x / kWave;
  const uint64_t g = static_cast<uint64_t>(blockIdx.x) * 4 + wave;
  if (g >= Gq) return;  // wave-uniform; no block barrier follows
  uint32_t* cnt = cnt_all[wave];
  for (uint32_t t = lane; t < kSlots; t += kWave) cnt[t] = 0;
  wave_sync();
  const QueryInfo qi = qinfo[g];
  const uint64_t seg = token_segment(R);
  const uint64_t below = (1ull << lane) - 1;
  const uint64_t end = (static_cast<uint64_t>(qi.qoff) + qi.k) * seg / 4;
  uint32_t nodes = 0, carry_label = 0, qcls = 0;
  bool starts_new = true;  // the chunk's first word starts a node
  for (uint64_t base = static_cast<uint64_t>(qi.qoff) * seg / 4; base < end && nodes < qi.k; base += kWave) {  // wave-uniform
    const uint64_t idx = base + lane;
    const bool in = idx < end;
    const uint64_t w = in ? tok64[idx] : ~0ull;
    bool has_end = false;
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) has_end |= ((w >> (16 * j)) & 0xFFFFull) == kEndToken;
    const uint64_t ends = __ballot(in && has_end);
    const uint64_t prev = ends & below;  // end words before this lane's in the chunk
    const uint32_t start_lane = prev ? 64u - static_cast<uint32_t>(__builtin_clzll(prev)) : 0u;
    const uint32_t first = labelled(static_cast<uint32_t>(w & 0xFFFFull));
    const uint32_t lab_here = static_cast<uint32_t>(__shfl(static_cast<int>(first), static_cast<int>(start_lane)));
    const uint32_t label = prev || starts_new ? lab_here : carry_label;
    const bool is_start = prev ? lane == start_lane : (lane == 0 && starts_new);
    const bool valid = in && nodes + static_cast<uint32_t>(__popcll(prev)) < qi.k;
    uint32_t c = kClasses;
#pragma unroll
    for (uint32_t cc = 0; cc < kClasses; ++cc)
      if (c == kClasses && label == cl.l[cc]) c = cc;
    if (valid && c < kClasses) {
      if (is_start) qcls |= 1u << c;
      for (uint32_t j = is_start ? 1u : 0u; j < 4; ++j) {
        const uint32_t t = static_cast<uint32_t>(w >> (16 * j)) & 0xFFFFu;
        if (t == kEndToken) break;
        atomicMax(&cnt[(c * kMaxLevels + token_level(t)) * 16 + token_label(t)], token_count(t));
      }
    }
    nodes += static_cast<uint32_t>(__popcll(ends));
    starts_new = (ends >> 63) & 1ull;
    carry_label = static_cast<uint32_t>(__shfl(static_cast<int>(label), kWave - 1));
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) qcls |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(qcls), o));
  wave_sync();
  if (lane < kClasses * R) {
    const uint32_t c = lane / R, r = lane - c * R;
    uint64_t v = 0;
    for (uint32_t l = 0; l < 16; ++l) v |= static_cast<uint64_t>(cnt[(c * kMaxLevels + r) * 16 + l]) << (4 * l);
    qcmax[(g * kClasses + c) * R + r] = v;
  }
  if (lane == 0) qinfo[g].qcls = qcls;
}

// ---- pair pre-test ------------------------------------------------------------------------------
//
// Two exact necessary conditions for a (query graph, molecule) pair to survive GMCR, tested for
// every pair before any candidate mask is built: (1) the graph's label set (labels < 16) is
// contained in the molecule's, and at every level the graph's nibble-wise signature max is <=
// the molecule's (a node whose signature exceeds the max fits no position); (2) for each class
// label present in the graph, the same holds between the max over the graph's nodes of that label
// and the max over the molecule's positions of that label (a node's candidates carry its label,
// isomorphism.hpp:49).  Query nodes of label 255 only enter (1).

struct PretestArgs {
  uint32_t R, Gq, W, G;          // W: bitmask words per molecule; G: molecules
  const MolInfo* minfo;          // width-class order
  const uint64_t* dmax;          // [c * R + r]
  const uint64_t* cmax;          // [(k * R + r) * G + c]
  const QueryInfo* qinfo;
  const uint64_t* qmax;          // [g * R + r]
  const uint64_t* qcmax;         // [(g * 3 + k) * R + r]
  unsigned long long* surv;      // [m * W + w] out: bit g of word w = pair (g, m) passes
};

// Nibble-wise a <= b for the 16 four-bit fields of several words, bit-sliced: bit b of every
// nibble of a word is one plane (bits 4l), and four words share a set of planes, word j's
// fields at bits 4l + j.  Over the planes, b >= a is the lowest-bit-up chain of ge4_bits with the
// query's planes as per-position thresholds, one v_bitop3_b32 per plane and 32 positions: a
// group of four words costs 8 operations, where splitting each word into even and odd nibbles
// took two 64-bit subtractions and two ANDs per word.  Positions of an unused word hold 0 on both
// sides and pass.
constexpr uint64_t kNibBit = 0x1111111111111111ull;
__device__ __forceinline__ uint64_t nib_plane(uint64_t w, uint32_t b, uint32_t j) { return ((w >> b) & kNibBit) << j; }

// acc &= (x >= m) position-wise over four planes (lo and hi halves of 64 positions)
__device__ __forceinline__ void planes_ge(const uint64_t x[4], const uint64_t* m, uint32_t& acc_lo, uint32_t& acc_hi) {
  uint32_t lo = ge_first(static_cast<uint32_t>(x[0]), static_cast<uint32_t>(m[0]));
  uint32_t hi = ge_first(static_cast<uint32_t>(x[0] >> 32), static_cast<uint32_t>(m[0] >> 32));
#pragma unroll
  for (int b = 1; b < 4; ++b) {
    lo = ge_stage(static_cast<uint32_t>(x[b]), static_cast<uint32_t>(m[b]), lo);
    hi = ge_stage(static_cast<uint32_t>(x[b] >> 32), static_cast<uint32_t>(m[b] >> 32), hi);
  }
  acc_lo &= lo;
  acc_hi &= hi;
}

// One thread per molecule (width-class order) and the query graphs 64 at a time from an LDS tile
// (every lane reads the same graph: broadcast reads), for RR levels in GA groups of four.  Tile
// words of a graph: [0] label set | classes << 32, then the all-node maxima's planes (4 words per
// group), then each class's (4 words per group).  A graph whose label test, or whose all-node
// test, fails on all 64 molecules of a wavefront skips the rest.
template <uint32_t RR>
__global__ __launch_bounds__(256) void k_pair_pretest(PretestArgs a) {
  constexpr uint32_t GA = (RR + 3) / 4;
  constexpr uint32_t S = 1 + 4 * GA * (1 + kClasses);
  __shared__ uint64_t tile[kWave * S];
  const uint64_t c = blockIdx.x * 256ull + threadIdx.x;
  const bool valid = c < a.G;
  uint32_t mlab = 0, m = 0;
  uint64_t md[GA][4], mc[kClasses][GA][4];  // the molecule's maxima as planes
#pragma unroll
  for (uint32_t g = 0; g < GA; ++g)
#pragma unroll
    for (uint32_t b = 0; b < 4; ++b) {
      md[g][b] = 0;
#pragma unroll
      for (uint32_t k = 0; k < kClasses; ++k) mc[k][g][b] = 0;
    }
  if (valid) {
    const MolInfo mi = a.minfo[c];
    mlab = mi.mlab;
    m = mi.m;
  }
#pragma unroll
  for (uint32_t r = 0; r < RR; ++r) {
    const uint64_t d = valid ? a.dmax[c * RR + r] : 0ull;
#pragma unroll
    for (uint32_t b = 0; b < 4; ++b) md[r / 4][b] |= nib_plane(d, b, r % 4);
#pragma unroll
    for (uint32_t k = 0; k < kClasses; ++k) {
      const uint64_t x = valid ? a.cmax[(static_cast<uint64_t>(k) * RR + r) * a.G + c] : 0ull;
#pragma unroll
      for (uint32_t b = 0; b < 4; ++b) mc[k][r / 4][b] |= nib_plane(x, b, r % 4);
    }
  }
  for (uint32_t w = 0; w < a.W; ++w) {
    __syncthreads();  // the previous tile has been read
    for (uint32_t t = threadIdx.x; t < kWave * S; t += 256) {
      const uint32_t j = t / S, f = t - j * S;
      const uint32_t g = w * kWave + j;
      uint64_t v = 0;
      if (g < a.Gq) {
        if (f == 0) {
          const QueryInfo qi = a.qinfo[g];
          v = qi.qlab | (static_cast<uint64_t>(qi.qcls) << 32);
        } else {
          const uint32_t i = f - 1;                   // (class slot, group, plane)
          const uint32_t cs = i / (4 * GA), grp = (i / 4) % GA, b = i % 4;  // cs 0: all nodes, 1 + k: class k
          const uint64_t* src = cs == 0 ? a.qmax + static_cast<uint64_t>(g) * RR
                                        : a.qcmax + (static_cast<uint64_t>(g) * kClasses + (cs - 1)) * RR;
          for (uint32_t jj = 0; jj < 4 && 4 * grp + jj < RR; ++jj) v |= nib_plane(src[4 * grp + jj], b, jj);
        }
      }
      tile[j * S + f] = v;
    }
    __syncthreads();
    const uint32_t nj = min(static_cast<uint32_t>(kWave), a.Gq - w * kWave);
    uint64_t word = 0;
    for (uint32_t j = 0; j < nj; ++j) {
      const uint64_t* e = tile + j * S;
      const uint64_t h = e[0];
      const bool lab = valid && (static_cast<uint32_t>(h) & ~mlab) == 0u;
      if (!__ballot(lab)) continue;  // wave-uniform
      uint32_t acc_lo = ~0u, acc_hi = ~0u;
#pragma unroll
      for (uint32_t g = 0; g < GA; ++g) planes_ge(md[g], e + 1 + 4 * g, acc_lo, acc_hi);
      bool fits = lab && (acc_lo & acc_hi) == ~0u;
      const uint32_t qcls = static_cast<uint32_t>(h >> 32);
      if (qcls && __ballot(fits)) {  // wave-uniform
#pragma unroll
        for (uint32_t k = 0; k < kClasses; ++k)
          if ((qcls >> k) & 1u) {
#pragma unroll
            for (uint32_t g = 0; g < GA; ++g) planes_ge(mc[k][g], e + 1 + 4 * GA * (1 + k) + 4 * g, acc_lo, acc_hi);
          }
        fits = fits && (acc_lo & acc_hi) == ~0u;
      }
      word |= static_cast<uint64_t>(fits) << j;
    }
    if (valid) a.surv[static_cast<uint64_t>(m) * a.W + w] = word;
  }
}

// ---- pair evaluation ----------------------------------------------------------------------------

// Arena words of a pair's block: its k node masks (half a word each for molecules of <= 32 nodes,
// one for 33..64, two for wider ones), rounded up to four nodes, or to two of the wide ones.
__device__ __forceinline__ uint32_t pair_words(uint32_t k, int cls) {
  return cls == 0 ? ((k + 3) & ~3u) / 2 : (cls == 1 ? (k + 3) & ~3u : ((k + 1) & ~1u) * 2);
}

constexpr uint32_t kGroupWaves = 8;       // wavefronts per block of the pair evaluation
constexpr uint32_t kGroupStatSlots = 32;  // one address would take every wavefront's sums one after another (~10 ns each)

struct GroupArgs {
  GraphDev d;
  GroupOrder order;
  uint32_t R, Gq, W;
  uint32_t parts;          // blocks that share a group's query graphs (a power of two <= 8)
  uint32_t slots;          // labels whose planes LDS holds
  uint32_t rich;           // the database's most frequent label (>= 16: none)
  uint32_t chunk;          // arena words a wavefront claims at a time
  const MolInfo* minfo;    // width-class order
  const uint4* planes;     // [((group*R + r)*16 + l)*64 + lane]
  const uint32_t* labs;    // [(group*16 + l)*64 + lane]
  const uint64_t* tokens;  // quads
  const QueryInfo* qinfo;
  uint64_t* arena;
  uint64_t arena_cap;
  unsigned long long* surv;      // [Gd][W] in: the pre-test's pairs; out: bit qg of row m = the pair survives GMCR
  uint4* blocks;                 // [group * Gq + g] where the masks of group and query graph are: pair_block
  unsigned long long* counters;  // [1] arena words claimed past the wavefronts' first chunks, [2] item cursor, [3] overflow, [4] k_surv_words
  unsigned long long* stats;     // kGroupStatSlots x 16: [0] node evaluations, [1] their live lanes, [2] pre-tested pairs
};

// LDS: the planes (slot_planes), then the list of the group's live query graphs, of eight query words
// at a time, and GroupCounters.
struct GroupCounters {
  uint32_t next_item;
  uint32_t listed[2], taken[2];  // of this list and the next
};
constexpr uint32_t kGroupListBytes = kGroupWaves * kWave * sizeof(uint4) + sizeof(GroupCounters);
__host__ __device__ constexpr uint32_t group_lds_bytes(uint32_t slots, uint32_t R) {
  return (slots + 1) * slot_planes(R) * 256 + kGroupListBytes;
}

// The value of lane ^ 1 and lane ^ 2 (quad permutations).
__device__ __forceinline__ uint32_t quad_xor1(uint32_t x) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(x), 0xB1, 0xF, 0xF, false));
}
__device__ __forceinline__ uint32_t quad_xor2(uint32_t x) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(x), 0x4E, 0xF, 0xF, false));
}

// The record of a group and a query graph, {base, words, lanes lo, lanes hi}: the pre-tested pairs
// have consecutive blocks of `words` from `base` on, in the order of their molecules' first lanes.
__device__ __forceinline__ uint32_t pair_block(uint32_t base, uint32_t words, uint64_t lanes, uint32_t lane0) {
  return base + static_cast<uint32_t>(__popcll(lanes & ((1ull << lane0) - 1))) * words;
}

// The kernel's arguments, read where they are used: kept in registers, those of the rare paths would
// spill the loop's scalars.
__device__ __forceinline__ const __attribute__((address_space(4))) GroupArgs& group_args() {
  auto p = (const __attribute__((address_space(4))) GroupArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *p;
}

// A wavefront's arena chunk (wave-uniform) and statistics: lane 0 node evaluations, lane 1 their live
// lanes, lane 2 pre-tested pairs.
struct GroupState {
  uint64_t next;
  uint32_t left;
  uint32_t turn = 0;  // which of the list counters are this list's
  uint64_t sums = 0;
};

// One group of a class against the wavefront's share of the query graphs.  COMPACT: see k_pair_group.
template <int CLS, bool COMPACT>
__device__ __forceinline__ void group_item(const GroupArgs& a, uint32_t grp, uint32_t part, uint32_t wave, uint32_t* planes_lds, GroupState& st) {
  const uint32_t lane = static_cast<uint32_t>(lane_id()), lane4 = lane * 4;
  const uint32_t R = a.R, SP = slot_planes(R);
  const uint64_t seg = token_segment(R) / 4;
  const uint32_t first = (CLS > 0 ? a.order.count[0] : 0u) + (CLS > 1 ? a.order.count[1] : 0u);
  const uint64_t group = grp + (CLS > 0 ? a.order.groups(0) : 0u) + (CLS > 1 ? a.order.groups(1) : 0u);
  const uint32_t at = grp * (64u >> CLS) + (lane >> CLS);  // the lane's molecule within its class
  const uint32_t h = lane & ((1u << CLS) - 1u);            // its 32 positions within the molecule
  const bool valid = at < a.order.count[CLS];
  MolInfo mi = {};
  if (valid) mi = a.minfo[first + at];
  constexpr uint64_t leaders = CLS == 0 ? ~0ull : (CLS == 1 ? 0x5555555555555555ull : 0x1111111111111111ull);
  const uint64_t below = (1ull << (lane & ~((1u << CLS) - 1u))) - 1;
  uint32_t present = 0;  // labels that occur in the group
#pragma unroll
  for (uint32_t l = 0; l < 16; ++l) present |= static_cast<uint32_t>(__ballot((mi.mlab >> l) & 1u) != 0ull) << l;
  present = uniform32(present);
  const uint32_t occur = static_cast<uint32_t>(__popc(present)), staged = min(occur, a.slots);
  auto slot_of = [&](uint32_t l) -> uint32_t { return static_cast<uint32_t>(__popc(present & ((1u << l) - 1u))); };
  auto label_of = [&](uint32_t slot) -> uint32_t {  // the slot-th label that occurs
    uint32_t left = present;
    for (uint32_t x = 0; x < slot; ++x) left &= left - 1;
    return static_cast<uint32_t>(__builtin_ctz(left));
  };
  const uint32_t rich = a.rich < 16 && ((present >> a.rich) & 1u) && slot_of(a.rich) < staged ? a.rich : 16u;
  const uint32_t all_plane = a.slots * SP + 4 * R;  // the plane of every position
  auto plane = [&](uint32_t index) -> uint32_t& { return planes_lds[index * kWave + lane]; };
  // the wavefronts take every eighth (label, level), four loads in flight each
  for (uint32_t e0 = wave; e0 < staged * R; e0 += 4 * kGroupWaves) {
    uint4 v[4];
#pragma unroll
    for (uint32_t x = 0; x < 4; ++x) {
      const uint32_t e = e0 + x * kGroupWaves;
      v[x] = make_uint4(0, 0, 0, 0);
      if (e < staged * R && valid) v[x] = a.planes[((group * R + e % R) * 16 + label_of(e / R)) * 64 + lane];
    }
#pragma unroll
    for (uint32_t x = 0; x < 4; ++x) {
      const uint32_t e = e0 + x * kGroupWaves;
      if (e >= staged * R) break;
      stage_planes(planes_lds, R, e / R, e % R, v[x], a.slots, label_of(e / R) == rich);
    }
  }
  for (uint32_t slot = wave; slot < staged; slot += kGroupWaves)
    plane(slot * SP + 4 * R) = valid ? a.labs[(group * 16 + label_of(slot)) * 64 + lane] : 0u;
  const uint32_t positions = mi.n > 32 * h ? min(32u, mi.n - 32 * h) : 0u;
  if (wave == 0) plane(all_plane) = positions >= 32 ? ~0u : (1u << positions) - 1u;
  __syncthreads();

  // what each key's planes start at, << 8 the token bits that count from there; bit 31: LDS has none
  uint32_t keys;
  {
    const uint32_t l = lane & 15u, kind = lane >> 4, slot = kind == 1 ? a.slots : slot_of(l);
    const bool here = kind == 0 ? slot < staged : kind == 1 && l == rich;
    const bool any = kind == 3 && lane != kKeyOther;
    keys = here ? slot * SP | (63u << 8) : (all_plane | (any ? 0u : 1u << 31));
  }
  auto key_of = [&](uint32_t t) -> uint32_t {  // of the token in t's low half
    return static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(static_cast<int>((t >> 4) & 0xFCu), static_cast<int>(keys)));
  };

  uint4* list = reinterpret_cast<uint4*>(planes_lds + (a.slots + 1) * SP * kWave);
  GroupCounters* ctr = reinterpret_cast<GroupCounters*>(list + kGroupWaves * kWave);
  // 64 quads of a graph's tokens, one per lane (a graph's segment holds k * seg of them)
  auto quads = [&](uint32_t qoff, uint32_t k, uint32_t from) -> uint64_t {
    return a.tokens[qoff * seg + min(from + lane, static_cast<uint32_t>(k * seg) - 1)];
  };
  uint32_t nodes = 0, live = 0, scans = 0;
  for (uint32_t w0 = 0; w0 < a.W; w0 += kGroupWaves) {
    // eight query words, one per wavefront: transposed, a lane has a query graph and the lanes of its
    // pre-tested pairs; graphs that have some are listed with their first node and size
    {
      const auto& c = group_args();
      const uint32_t w = w0 + wave, g = w * kWave + lane;
      const uint64_t word = valid && w < c.W ? c.surv[static_cast<uint64_t>(mi.m) * c.W + w] : 0ull;
      if (__ballot(word != 0)) {  // wave-uniform
        const uint64_t act = transpose64(word);
        const bool mine = act != 0 && (lane & (c.parts - 1)) == part;
        const uint64_t mm = __ballot(mine);
        uint32_t b = 0;
        if (lane == 0) b = atomicAdd(&ctr->listed[st.turn], static_cast<uint32_t>(__popcll(mm)));
        b = uniform32(b);
        if (mine) {
          const QueryInfo* info = c.qinfo + g;
          list[b + static_cast<uint32_t>(__popcll(mm & ((1ull << lane) - 1)))] =
              make_uint4(static_cast<uint32_t>(act), static_cast<uint32_t>(act >> 32), info->qoff, (g << 5) | (info->k - 1));
        }
      }
    }
    __syncthreads();
    const uint32_t listed = uniform32(ctr->listed[st.turn]);
    if (threadIdx.x == 0) ctr->listed[st.turn ^ 1u] = ctr->taken[st.turn ^ 1u] = 0;
    uint32_t t = wave;
    uint4 entry = make_uint4(0, 0, 0, 0);
    uint64_t ahead = 0;
    auto fetch = [&]() {
      const uint4 e = list[t];
      entry = make_uint4(uniform32(e.x), uniform32(e.y), uniform32(e.z), uniform32(e.w));
      ahead = quads(entry.z, (entry.w & 31u) + 1, 0);
    };
    if (t < listed) fetch();
    while (t < listed) {  // wave-uniform
      const uint64_t act = entry.x | (static_cast<uint64_t>(entry.y) << 32), am = act & leaders;
      const uint32_t g = entry.w >> 5, qoff = entry.z, k = (entry.w & 31u) + 1;
      uint64_t raw = ahead;
      // the next graph, whose tokens are on their way meanwhile
      if (lane == 0) t = kGroupWaves + atomicAdd(&ctr->taken[st.turn], 1u);
      t = uniform32(t);
      if (t < listed) fetch();
      const uint32_t cnt = static_cast<uint32_t>(__popcll(am)), pw = pair_words(k, CLS);
      scans += cnt;
      if (cnt * pw > st.left) {
        const auto& c = group_args();
        unsigned long long b = 0;
        if (lane == 0) {
          b = static_cast<uint64_t>(gridDim.x) * kGroupWaves * c.chunk + atomicAdd(&c.counters[1], static_cast<unsigned long long>(c.chunk));
          if (b + c.chunk > c.arena_cap) atomicOr(&c.counters[3], 1ull);
        }
        st.next = uniform64(__shfl(b, 0));
        st.left = c.chunk;
      }
      const uint64_t base0 = st.next, base = base0 + static_cast<uint64_t>(__popcll(am & below)) * pw;
      const bool room = st.next + st.left <= a.arena_cap;

      // The quads are decoded once, each lane its own: four planes by their bytes.  A node's mask is the
      // AND of its quads' planes; `fars` marks quads with a token that LDS has no plane of.
      uint32_t from = 0, p = 0, dec = 0;
      uint64_t ends = 0, fars = 0;
      uint64_t alive = act;
      uint32_t m0 = 0, m1 = 0, m2 = 0, m3 = 0, i = 0;
      // nodes whose masks, with those before them, go out
      const uint32_t flush = (0x88888888u & ((2u << (k - 1)) - 1u)) | (1u << (k - 1));
      for (;; ++i) {  // wave-uniform
        if (ends == 0) {  // the node's quads (at most nine) cross the 64, or the first
          from += p;
          p = 0;
          if (from) raw = quads(qoff, k, from);
          ends = __ballot(static_cast<uint32_t>(raw >> 48) == kEndToken);  // every end quad ends in one
          const uint32_t t0 = static_cast<uint32_t>(raw), t1 = t0 >> 16, t2 = static_cast<uint32_t>(raw >> 32), t3 = t2 >> 16;
          const uint32_t k0 = key_of(t0), k1 = key_of(t1), k2 = key_of(t2), k3 = key_of(t3);
          const uint32_t d0 = k0 + (t0 & ((k0 >> 8) & 63u)), d1 = k1 + (t1 & ((k1 >> 8) & 63u));
          const uint32_t d2 = k2 + (t2 & ((k2 >> 8) & 63u)), d3 = k3 + (t3 & ((k3 >> 8) & 63u));
          dec = __builtin_amdgcn_perm(__builtin_amdgcn_perm(d3, d2, 0x0c0c0400u), __builtin_amdgcn_perm(d1, d0, 0x0c0c0400u), 0x05040100u);
          fars = __ballot(static_cast<int32_t>(k0 | k1 | k2 | k3) < 0);
        }
        const uint32_t count = static_cast<uint32_t>(__builtin_ctzll(ends)) + 1, p1 = p + count;
        ends >>= count;
        live += static_cast<uint32_t>(__popcll(alive));
        uint32_t mask = ~0u;
        if (fars) {
          const auto& c = group_args();
          for (uint32_t x = p; x < p1; ++x) {
            if (!((fars >> x) & 1ull)) continue;
            const uint64_t qw = rl32(static_cast<uint32_t>(raw), x) | (static_cast<uint64_t>(rl32(static_cast<uint32_t>(raw >> 32), x)) << 32);
            for (uint32_t y = 0; y < 4; ++y) {
              const uint32_t t = static_cast<uint32_t>(qw >> (16 * y)) & 0xFFFFu;
              if (t == kEndToken) break;
              const uint32_t key = (t >> 6) & 63u, label = token_label(t);
              if (x == p && y == 0) {  // the label: the filter's test (isomorphism.hpp:49)
                if (key < 16u) {
                  mask &= valid ? c.labs[(group * 16 + label) * 64 + lane] : 0u;
                } else if (key == kKeyOther) {
                  uint32_t at_label = 0;
                  if ((act >> lane) & 1ull)
                    for (uint32_t v = 0; v < positions; ++v)
                      if (c.d.nl[static_cast<uint64_t>(mi.s) + 32 * h + v] == labelled(t)) at_label |= 1u << v;
                  mask &= at_label;
                }
              } else {
                uint4 v = make_uint4(0, 0, 0, 0);
                if (valid) {
                  const uint4* src = c.planes;
                  v = src[((group * R + token_level(t)) * 16 + label) * 64 + lane];
                }
                mask &= ge4_bits<uint32_t>(v.x, v.y, v.z, v.w, token_count(t));
              }
            }
          }
        }
        mask = quad_tests(dec, p, p1, lane4, mask);
        p = p1;
        // a pair dies at its first node without candidates (gmcr.hpp:56-61)
        uint32_t some = mask;
        if (CLS >= 1) some |= quad_xor1(some);
        if (CLS == 2) some |= quad_xor2(some);
        alive &= __ballot(some != 0);
        if (!alive) break;
        m0 = m1;
        m1 = m2;
        m2 = m3;
        m3 = mask;
        if (((flush >> i) & 1u) == 0) continue;
        // masks go out four nodes at a time, in 16-byte stores (nodes past the last fall in the block's
        // padding)
        for (uint32_t x = i; (x & 3u) != 3u; ++x) {
          m0 = m1;
          m1 = m2;
          m2 = m3;
          m3 = 0;
        }
        const uint32_t i0 = i & ~3u;
        const bool store = room && __builtin_amdgcn_inverse_ballot_w64(alive);
        if (CLS == 0) {
          if (store) *reinterpret_cast<uint4*>(a.arena + base + i0 / 2) = make_uint4(m0, m1, m2, m3);
        } else if (CLS == 1) {  // the lanes of a molecule swap halves: each stores two nodes' words
          const uint32_t o0 = quad_xor1(h ? m0 : m2), o1 = quad_xor1(h ? m1 : m3);
          if (store) reinterpret_cast<uint4*>(a.arena + base + i0)[h] = h ? make_uint4(o0, m2, o1, m3) : make_uint4(m0, o0, m1, o1);
        } else if (store) {
          uint32_t* dst = reinterpret_cast<uint32_t*>(a.arena + base + 2 * i0) + h;
          dst[0] = m0;
          dst[4] = m1;
          if (i0 + 2 < k) {
            dst[8] = m2;
            dst[12] = m3;
          }
        }
        if (i + 1 < k) continue;
        uint64_t lanes = am;  // whose blocks these are
        uint32_t taken = cnt * pw;
        if constexpr (COMPACT) {
          lanes &= alive;
          taken = static_cast<uint32_t>(__popcll(lanes)) * pw;
          const uint64_t to = base0 + static_cast<uint64_t>(__popcll(lanes & below)) * pw;
          // a block moves to where an earlier molecule's is or was; a step loads 16 bytes of every block before
          // it stores them, each at the same place in its block, so none is lost
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
          if (store && to != base)
#pragma unroll 1
            for (uint32_t u = h; u < pw / 2; u += 1u << CLS) {
              const uint4 v = reinterpret_cast<const uint4*>(a.arena + base)[u];
              reinterpret_cast<uint4*>(a.arena + to)[u] = v;
            }
        }
        if (lane == 0)
          group_args().blocks[group * a.Gq + g] = make_uint4(static_cast<uint32_t>(base0), pw, static_cast<uint32_t>(lanes), static_cast<uint32_t>(lanes >> 32));
        st.next += taken;  // without survivors the next graph takes the same words
        st.left -= taken;
        break;
      }
      nodes += i + 1;
      if (__builtin_amdgcn_inverse_ballot_w64(am & ~alive)) {
        const auto& c = group_args();
        atomicAnd(&c.surv[static_cast<uint64_t>(mi.m) * c.W + g / kWave], ~(1ull << (g % kWave)));
      }
    }
    st.turn ^= 1u;
    __syncthreads();  // the list has been read
  }
  st.sums += lane == 0 ? nodes : (lane == 1 ? live : (lane == 2 ? scans : 0u));
}

// Pair evaluation: the exact candidates of every pre-tested pair's query nodes (isomorphism.hpp:49
// and :103-110), keeping the masks of the pairs that survive GMCR.
//
// A wavefront takes one query graph and one group, 64 lanes of neighbours in the width-class
// order, so a requirement is the same for 64 x 32 positions: a plane of LDS and an AND.  A lane that
// walked a pair of its own decoded every token for itself and gathered its token words and planes,
// about 40 operations a test, and a wavefront waited for its longest pair.  The order groups
// molecules of one label set and similar size, so a query graph passes the pre-test for none of a
// group's molecules three times out of four and for half of them otherwise (1 M LogNormal
// molecules, U[4,32]-node queries).
//
// A block of eight wavefronts stages the group's planes and label masks for the labels that occur
// in it (the first a.slots of them; the rest are read from the database), lists the query graphs
// that have pre-tested pairs, eight words of them at a time, and its wavefronts take them as they
// come: shared out by index, wavefronts waited a fifth of their time for the longest share.  Counts
// of 1 to 4 have planes for every label and 5 to 8 for the database's most frequent one, which leaves
// 0.3% of the requirements to be read from the database (7.5% with 1 to 4 alone).  The tokens of 64
// quads are decoded at once, a quad per lane, to the four planes' numbers in a word; a quad then
// takes one lane read, four byte permutations (the LDS addresses), four LDS reads and two ANDs, and
// its label, end and padding tokens are planes like the others.  With each token a scalar of its own
// a node took 75 scalar operations and 19 branches, now 45 and 12: one scalar unit serves the
// CU's 24 wavefronts and bounds the kernel, at 69% of its issue slots (VALU 58%; 1 M x 1,000).
//
// Node masks go straight to the pairs' arena blocks, which a wavefront takes from a chunk of its own;
// pairs that die clear their pre-test bits, and where none of a group survives the next query graph
// takes the blocks.  With COMPACT (a batch that size_arena moved to it) the survivors' blocks move
// together, so that the arena holds no others.  At most 80 registers: six wavefronts per SIMD (20 waves
// with 4-wavefront blocks: 8.1 instead of 6.8 ms).  With 64-bit masks for every molecule and an offset
// per pair, stored 4 KB apart, 174 M writes went to memory instead of 68 M of 64 bytes (4.4 GB).
//
// Measured: a lane per pair and a launch per size class, wavefronts by groups with scalar tokens, and
// this: 2,000 molecules x 20 query graphs 219, 13 and 10 us (three serial chains of ~100 us at
// first), 100,000 x 100 475, 118 and 73 us, 1 M x 25 1,242, 353 and 294 us, 1 M x 1,000 10.7, 5.6 and
// 3.2 to 3.5 ms.
template <bool COMPACT>
__global__ __launch_bounds__(kGroupWaves * 64, 6) void k_pair_group(GroupArgs a) {
  extern __shared__ uint32_t planes_lds[];
  GroupCounters* ctr = reinterpret_cast<GroupCounters*>(reinterpret_cast<uint4*>(planes_lds + (a.slots + 1) * slot_planes(a.R) * kWave) + kGroupWaves * kWave);
  if (threadIdx.x == 0) ctr->listed[0] = ctr->taken[0] = 0;  // before the barrier that ends the first staging
  const uint32_t wave = uniform32(threadIdx.x / kWave);
  const uint32_t items = a.order.total() * a.parts;
  // three quarters of the groups are shared out beforehand: claims meet on one address, where they take
  // about 10 ns each (1 M molecules x 25 query graphs: 16,000 claims for groups, as many for chunks)
  const uint32_t fixed = max(gridDim.x, items / 4 * 3 / gridDim.x * gridDim.x);
  GroupState st;
  st.next = (static_cast<uint64_t>(blockIdx.x) * kGroupWaves + wave) * a.chunk;
  st.left = a.chunk;
  if (blockIdx.x == 0 && threadIdx.x == 0 && static_cast<uint64_t>(gridDim.x) * kGroupWaves * a.chunk > a.arena_cap) atomicOr(&a.counters[3], 1ull);
  for (uint32_t item = blockIdx.x; item < items;) {
    const uint32_t part = item & (a.parts - 1), grp = item / a.parts;
    const uint32_t g0 = a.order.groups(0), g1 = a.order.groups(1);
    if (grp < g0) group_item<0, COMPACT>(a, grp, part, wave, planes_lds, st);
    else if (grp < g0 + g1) group_item<1, COMPACT>(a, grp - g0, part, wave, planes_lds, st);
    else group_item<2, COMPACT>(a, grp - g0 - g1, part, wave, planes_lds, st);
    item += gridDim.x;
    if (item < fixed) continue;
    if (gridDim.x >= items) break;
    if (threadIdx.x == 0) ctr->next_item = fixed + static_cast<uint32_t>(atomicAdd(&a.counters[2], 1ull));  // the staged planes have been read
    __syncthreads();
    item = uniform32(ctr->next_item);
  }
  if (lane_id() < 3 && st.sums) atomicAdd(&a.stats[(blockIdx.x % kGroupStatSlots) * 16 + lane_id()], static_cast<unsigned long long>(st.sums));
}

// The arena words of the pairs that survive (a thread per molecule of the width-class order).
__global__ __launch_bounds__(256) void k_surv_words(GroupOrder order, uint32_t G, uint32_t W, const MolInfo* __restrict__ minfo,
                                                    const QueryInfo* __restrict__ qinfo, const unsigned long long* __restrict__ surv,
                                                    unsigned long long* __restrict__ out) {
  const uint64_t c = blockIdx.x * 256ull + threadIdx.x;
  uint64_t words = 0;
  if (c < G) {
    const int cls = c < order.count[0] ? 0 : (c < static_cast<uint64_t>(order.count[0]) + order.count[1] ? 1 : 2);
    const uint64_t m = minfo[c].m;
    for (uint32_t w = 0; w < W; ++w)
      for (uint64_t x = surv[m * W + w]; x; x &= x - 1) words += pair_words(qinfo[w * kWave + static_cast<uint32_t>(__builtin_ctzll(x))].k, cls);
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) words += static_cast<uint64_t>(__shfl_xor(static_cast<unsigned long long>(words), o));
  if (lane_id() == 0 && words) atomicAdd(out, static_cast<unsigned long long>(words));
}

// Survivors per molecule: the popcount of its row of the survival bitmask.
__global__ __launch_bounds__(256) void k_surv_count(uint32_t Gd, uint32_t W, const unsigned long long* __restrict__ surv,
                                                    uint32_t* __restrict__ counts) {
  const uint64_t m = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x;
  if (m >= Gd) return;
  uint32_t c = 0;
  for (uint32_t w = 0; w < W; ++w) c += __popcll(surv[m * W + w]);
  counts[m] = c;
}

// Canonical GMCR arrays (gmcr.hpp:73-115 order: molecules ascending, query graphs ascending
// within a molecule) from the survival bitmask, with each pair's arena offset from its group's
// records.  A block takes one group of the width-class order and its wavefronts a quarter of the
// molecules each: for 64 query graphs at a time a lane holds one graph's record and the wavefront
// goes over its molecules, whose survivors go out in one coalesced store per array.  When the pair
// evaluation wrote every pair's offset to a [molecule][query graph] table and a wavefront per
// molecule read them back, 1 M x 1,000 took 1.6 ms here; this takes 1.1 ms.
__global__ __launch_bounds__(256) void k_surv_scatter(GroupOrder order, uint32_t Gq, uint32_t W, const MolInfo* __restrict__ minfo,
                                                      const unsigned long long* __restrict__ surv, const uint32_t* __restrict__ offsets,
                                                      const uint4* __restrict__ blocks, uint32_t* __restrict__ indices,
                                                      uint32_t* __restrict__ pair_graph, uint32_t* __restrict__ mask_off, uint64_t cap) {
  // `cap` bounds the writes: a replayed graph sized by an earlier run never writes past its
  // arrays (the replay then reports the changed pair count)
  const uint32_t group = blockIdx.x, lane = static_cast<uint32_t>(lane_id()), wave = uniform32(threadIdx.x / kWave);
  const uint32_t g0 = order.groups(0), g1 = order.groups(1);
  const uint32_t cls = group < g0 ? 0u : (group < g0 + g1 ? 1u : 2u);
  const uint32_t grp = group - (cls > 0 ? g0 : 0u) - (cls > 1 ? g1 : 0u), per = 64u >> cls;
  const uint32_t first = (cls > 0 ? order.count[0] : 0u) + (cls > 1 ? order.count[1] : 0u);
  // lane i < share: the wavefront's i-th molecule
  const uint32_t share = per / 4, slot = wave * share + lane, at = grp * per + slot;
  const bool valid = lane < share && at < (cls == 0 ? order.count[0] : (cls == 1 ? order.count[1] : order.count[2]));
  const uint32_t m = valid ? minfo[first + at].m : 0u;
  uint32_t o = valid ? offsets[m] : 0u;  // where its next survivor goes
  const uint64_t below = (1ull << lane) - 1;
  for (uint32_t w = 0; w < W; ++w) {
    const uint64_t xl = valid ? surv[static_cast<uint64_t>(m) * W + w] : 0ull;
    uint64_t left = __ballot(xl != 0ull);
    if (!left) continue;  // wave-uniform
    const uint32_t g = w * kWave + lane;
    uint4 rec = make_uint4(0, 0, 0, 0);
    if (g < Gq) rec = blocks[static_cast<uint64_t>(group) * Gq + g];  // unwritten, and not used, where no molecule of the group survives
    const uint64_t lanes = rec.z | (static_cast<uint64_t>(rec.w) << 32);
    for (; left; left &= left - 1) {
      const uint32_t i = static_cast<uint32_t>(__builtin_ctzll(left));
      const uint64_t x = rl32(static_cast<uint32_t>(xl), i) | (static_cast<uint64_t>(rl32(static_cast<uint32_t>(xl >> 32), i)) << 32);
      const uint32_t r = rl32(o, i) + static_cast<uint32_t>(__popcll(x & below)), mol = rl32(m, i);
      if (((x >> lane) & 1ull) && r < cap) {
        indices[r] = g;
        pair_graph[r] = mol;
        mask_off[r] = pair_block(rec.x, rec.y, lanes, (wave * share + i) << cls);
      }
    }
    o += static_cast<uint32_t>(__popcll(xl));
  }
}

// k_surv_scatter for at most 64 query graphs (one bitmask word per molecule): most molecules then
// have no or a few survivors, so a wavefront takes a group with a lane per molecule and goes over
// the query graphs that survive for any of them.
__global__ __launch_bounds__(256) void k_surv_scatter_lanes(GroupOrder order, uint32_t Gq, const MolInfo* __restrict__ minfo,
                                                            const unsigned long long* __restrict__ surv, const uint32_t* __restrict__ offsets,
                                                            const uint4* __restrict__ blocks, uint32_t* __restrict__ indices,
                                                            uint32_t* __restrict__ pair_graph, uint32_t* __restrict__ mask_off, uint64_t cap) {
  const uint32_t group = uniform32(blockIdx.x * 4 + threadIdx.x / kWave), lane = static_cast<uint32_t>(lane_id());
  if (group >= order.total()) return;  // wave-uniform; no block barrier follows
  const uint32_t g0 = order.groups(0), g1 = order.groups(1);
  const uint32_t cls = group < g0 ? 0u : (group < g0 + g1 ? 1u : 2u);
  const uint32_t grp = group - (cls > 0 ? g0 : 0u) - (cls > 1 ? g1 : 0u), per = 64u >> cls;
  const uint32_t first = (cls > 0 ? order.count[0] : 0u) + (cls > 1 ? order.count[1] : 0u);
  const uint32_t at = grp * per + lane;
  const bool valid = lane < per && at < (cls == 0 ? order.count[0] : (cls == 1 ? order.count[1] : order.count[2]));
  uint4 rec = make_uint4(0, 0, 0, 0);
  if (lane < Gq) rec = blocks[static_cast<uint64_t>(group) * Gq + lane];
  const uint32_t m = valid ? minfo[first + at].m : 0u;
  const uint64_t x = valid ? surv[m] : 0ull;
  uint32_t o = valid ? offsets[m] : 0u;
  uint32_t any_lo = static_cast<uint32_t>(x), any_hi = static_cast<uint32_t>(x >> 32);
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    any_lo |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(any_lo), d));
    any_hi |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(any_hi), d));
  }
  for (uint64_t bits = uniform64(any_lo | (static_cast<uint64_t>(any_hi) << 32)); bits; bits &= bits - 1) {  // wave-uniform
    const uint32_t g = static_cast<uint32_t>(__builtin_ctzll(bits));
    const uint32_t base = rl32(rec.x, g), words = rl32(rec.y, g);
    const uint64_t lanes = rl32(rec.z, g) | (static_cast<uint64_t>(rl32(rec.w, g)) << 32);
    if ((x >> g) & 1ull) {
      if (o < cap) {
        indices[o] = g;
        pair_graph[o] = m;
        mask_off[o] = pair_block(base, words, lanes, lane << cls);
      }
      ++o;
    }
  }
}

// Per-request statistics of a batch run.  Request r owns the batch's query graphs
// [rg[r], rg[r+1]); each GMCR pair (molecule m, query graph g, count c) adds its match flag,
// c, and mix64(mix64(((g - rg[r]) << 32) | m) + c) to its request (sums mod 2^64, mix64 being
// the splitmix64 finaliser).  Sums do not depend on the order pairs are visited, so a request's
// hash is the same whether it ran alone or batched with others.
__device__ __forceinline__ uint64_t mix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

constexpr uint32_t kMaxBatchRequests = 256;
constexpr uint32_t kStatsBlock = 1024;  // threads, and (request, copy) sums in LDS
constexpr uint32_t kStatsOutWords = 1024;

// Copies of the sums in device memory, each on lines of its own: blocks add to copy blockIdx % copies.
inline uint32_t stats_copies(uint32_t nreq) { return std::max(1u, std::min(16u, kMaxBatchRequests / nreq)); }
__host__ __device__ inline uint32_t stats_stride(uint32_t nreq) { return (3 * nreq + 15) & ~15u; }

// Bound by the reads of pairs (12 bytes each) and the 64-bit products of the hash.  A thread takes four
// pairs at a time and keeps the sums of its current request in registers; on a change they go to one
// of `shared` copies in LDS, since lanes that add to one address take turns.  Blocks are two per CU:
// each ends with three atomics per request, and with eight per CU on one copy these (about 10 ns each
// on one line) were most of a small batch's time.  1 M molecules x 25 query graphs in one request
// 81 -> 9 us, 300,000 x 306 in 12 164 -> 34 us, 1 M x 1,000 in 250 420 -> 297 us (3.0 TB/s).
__global__ __launch_bounds__(kStatsBlock) void k_request_stats(uint64_t P, const uint32_t* __restrict__ indices,
                                                               const uint32_t* __restrict__ pair_graph, const int32_t* __restrict__ counts,
                                                               const uint32_t* __restrict__ rg, uint32_t nreq, uint32_t shared, uint32_t copies,
                                                               unsigned long long* __restrict__ out) {
  __shared__ uint32_t srg[kMaxBatchRequests + 1];
  __shared__ unsigned long long acc_emb[kStatsBlock], acc_hash[kStatsBlock];
  __shared__ uint32_t acc_matched[kStatsBlock];  // a block has fewer than 2^32 pairs
  for (uint32_t t = threadIdx.x; t <= nreq; t += blockDim.x) srg[t] = rg[t];
  acc_emb[threadIdx.x] = acc_hash[threadIdx.x] = 0;
  acc_matched[threadIdx.x] = 0;
  __syncthreads();
  uint32_t r = 0, r0 = 0, r1 = srg[1], matched = 0;  // the current request and its query graphs [r0, r1)
  uint64_t emb = 0, hash = 0;
  const auto flush = [&]() {
    const uint32_t at = r * shared + (threadIdx.x & (shared - 1));
    if (matched) atomicAdd(&acc_matched[at], matched);
    if (emb) atomicAdd(&acc_emb[at], static_cast<unsigned long long>(emb));
    if (hash) atomicAdd(&acc_hash[at], static_cast<unsigned long long>(hash));
    matched = 0;
    emb = hash = 0;
  };
  const auto add = [&](uint32_t g, uint32_t m, int32_t c) {
    if (g < r0 || g >= r1) {
      flush();
      uint32_t lo = 0, hi = nreq;  // last r with srg[r] <= g
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (srg[mid] <= g) lo = mid;
        else hi = mid;
      }
      r = lo;
      r0 = srg[lo];
      r1 = srg[lo + 1];
    }
    matched += c > 0;
    emb += static_cast<uint64_t>(c);
    hash += mix64(mix64((static_cast<uint64_t>(g - r0) << 32) | m) + static_cast<uint32_t>(c));
  };
  for (uint64_t j = 4 * (blockIdx.x * static_cast<uint64_t>(kStatsBlock) + threadIdx.x); j < P; j += 4ull * kStatsBlock * gridDim.x) {
    if (j + 4 <= P) {
      const uint4 g = *reinterpret_cast<const uint4*>(indices + j), m = *reinterpret_cast<const uint4*>(pair_graph + j);
      const int4 c = *reinterpret_cast<const int4*>(counts + j);
      add(g.x, m.x, c.x);
      add(g.y, m.y, c.y);
      add(g.z, m.z, c.z);
      add(g.w, m.w, c.w);
    } else {
      for (uint64_t i = j; i < P; ++i) add(indices[i], pair_graph[i], counts[i]);
    }
  }
  flush();
  __syncthreads();
  unsigned long long* to = out + static_cast<uint64_t>(blockIdx.x % copies) * stats_stride(nreq);
  for (uint32_t t = threadIdx.x; t < nreq; t += blockDim.x) {
    unsigned long long sum[3] = {0, 0, 0};
    for (uint32_t i = 0; i < shared; ++i) {
      sum[0] += acc_matched[t * shared + i];
      sum[1] += acc_emb[t * shared + i];
      sum[2] += acc_hash[t * shared + i];
    }
    for (int f = 0; f < 3; ++f)
      if (sum[f]) atomicAdd(&to[3 * t + f], sum[f]);
  }
}

}  // namespace

// The first `small` width-class entries (molecules of <= 32 nodes) two per wavefront, the rest one
// per wavefront.
hipError_t db_prepare(hipStream_t s, const GraphDev& g, uint32_t R, const uint32_t* cls_list, const GroupOrder& order, uint32_t* planes,
                      uint32_t* labs, uint64_t* dmax, MolInfo* minfo, const ClassLabels& cl, uint64_t* cmax) {
  if (!g.G) return hipSuccess;
  const uint32_t small = order.count[0];
  if (small) {
    const uint32_t waves = (small + 1) / 2;
    k_db_prepare_pairs<<<(waves + 3) / 4, 256, 0, s>>>(g, R, small, cls_list, planes, labs, dmax, minfo, cl, cmax);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (g.G > small) k_db_prepare<<<(g.G - small + 3) / 4, 256, 0, s>>>(g, R, cls_list, order, planes, labs, dmax, minfo, cl, cmax, small);
  return hipGetLastError();
}

hipError_t query_prepare(hipStream_t s, const GraphDev& q, uint32_t R, uint16_t* tokens, QueryInfo* qinfo, uint64_t* qmax, const ClassLabels& cl,
                         uint64_t* qcmax) {
  if (!q.G) return hipSuccess;
  k_query_prepare<<<(q.G + 3) / 4, 256, 0, s>>>(q, R, tokens, qinfo, qmax);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  k_query_classes<<<(q.G + 3) / 4, 256, 0, s>>>(q.G, R, reinterpret_cast<const uint64_t*>(tokens), cl, qinfo, qcmax);
  return hipGetLastError();
}

// Node-label histogram (256 bins) of a graph batch.
__global__ __launch_bounds__(256) void k_label_hist(const uint8_t* __restrict__ nl, uint64_t N, unsigned long long* __restrict__ hist) {
  __shared__ unsigned int bins[256];
  bins[threadIdx.x] = 0;
  __syncthreads();
  for (uint64_t v = blockIdx.x * 256ull + threadIdx.x; v < N; v += static_cast<uint64_t>(gridDim.x) * 256) atomicAdd(&bins[nl[v]], 1u);
  __syncthreads();
  if (bins[threadIdx.x]) atomicAdd(&hist[threadIdx.x], static_cast<unsigned long long>(bins[threadIdx.x]));
}

hipError_t label_hist(hipStream_t s, const uint8_t* nl, uint64_t N, unsigned long long* hist) {
  hipError_t e = fill_u64(s, reinterpret_cast<uint64_t*>(hist), 256, 0);
  if (e != hipSuccess || !N) return e;
  const uint64_t blocks = std::min<uint64_t>(1024, (N + 255) / 256);
  k_label_hist<<<static_cast<unsigned>(blocks), 256, 0, s>>>(nl, N, hist);
  return hipGetLastError();
}

}  // namespace sigmo_k

// ---- host objects and C ABI -----------------------------------------------------------------------

namespace {

#define BATCH_HIP_TRY(expr)                                                                        \
  do {                                                                                             \
    hipError_t _e = (expr);                                                                        \
    if (_e != hipSuccess)                                                                          \
      return sigmo_err::set(_e == hipErrorOutOfMemory ? SIGMO_ERR_NOMEM : SIGMO_ERR_HIP,           \
                            std::string(#expr) + ": " + hipGetErrorString(_e));                    \
  } while (0)

#define BATCH_TRY(expr)            \
  do {                             \
    int _s = (expr);               \
    if (_s != SIGMO_OK) return _s; \
  } while (0)

template <typename T>
int balloc(T** p, uint64_t n) {
  *p = nullptr;
  hipError_t e = hipMalloc(reinterpret_cast<void**>(p), (n ? n : 1) * sizeof(T));
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
    return sigmo_err::set(SIGMO_ERR_NOMEM, "hipMalloc of " + std::to_string(n * sizeof(T)) + " bytes failed");
  }
  return SIGMO_OK;
}
template <typename T>
void bfree(T*& p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}
template <typename T>
int bgrow(T** p, uint64_t& cap, uint64_t need) {
  if (*p && cap >= need) return SIGMO_OK;
  bfree(*p);
  cap = 0;
  BATCH_TRY(balloc(p, need));
  cap = need;
  return SIGMO_OK;
}
// Growth with an eighth to spare, for buffers whose size follows the data of a streaming chunk:
// chunks of similar size then rarely reallocate (hipFree waits for the whole device).
template <typename T>
int bgrow_slack(T** p, uint64_t& cap, uint64_t need) {
  if (*p && cap >= need) return SIGMO_OK;
  return bgrow(p, cap, need + need / 8);
}

}  // namespace

// Internal views of the objects defined in capi.hip.
namespace sigmo_internal {
int ctx_info(sigmo_ctx* ctx, int* device, hipStream_t* stream, int* num_cus, unsigned long long** stats, unsigned long long** stats_host);
int ctx_timed(sigmo_ctx* ctx, int phase, int kernel, double bytes, bool begin, void** token);
int ctx_read_back(sigmo_ctx* ctx, const sigmo_k::HostCopy* copies, int n);
void ctx_add_bytes(sigmo_ctx* ctx, int kernel, double bytes);
const sigmo_k::GraphDev graph_dev(const sigmo_graph* g);
const std::vector<uint32_t>& graph_host_offsets(const sigmo_graph* g);
sigmo_ctx* graph_ctx(const sigmo_graph* g);
uint64_t graph_edges(const sigmo_graph* g);
}  // namespace sigmo_internal

using namespace sigmo_internal;

// Pair spaces up to this size run with one host synchronisation (sigmo_batch_run).
constexpr uint64_t kOneSyncPairs = 1ull << 25;
// Arena offsets are 32-bit.
constexpr uint64_t kMaxArenaWords = (1ull << 32) - 4;
// A run's device counters: 16 words, then the group evaluation's statistics.
constexpr uint64_t kCounterWords = 16 + 16 * sigmo_k::kGroupStatSlots;

struct sigmo_batch;
namespace sigmo_internal {
sigmo_ctx* batch_ctx(const sigmo_batch* b);
}

struct sigmo_db {
  sigmo_ctx* ctx = nullptr;
  const sigmo_graph* data = nullptr;
  uint32_t R = 0;
  uint32_t num_wide = 0;
  uint32_t num_labels = 0;            // node labels < 16 that occur in the data
  sigmo_k::GroupOrder order{{0, 0, 0}};  // molecules of <= 32, 33..64 and 65..128 nodes
  uint32_t* cls_list = nullptr;       // the three classes' molecules one after another, grouped by label set and size
  uint32_t *planes = nullptr, *labs = nullptr;  // level planes and label masks by group (GroupOrder)
  uint64_t* dmax = nullptr;                     // width-class order
  uint64_t* cmax = nullptr;                                                                // per-class maxima, [(k*R + r)*G + c]
  sigmo_k::MolInfo* minfo = nullptr;                                                       // width-class order
  sigmo_k::ClassLabels cls{{0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu}};                        // the pre-test's class labels
  uint64_t bytes = 0;
  uint64_t cap_G = 0, cap_planes = 0, cap_labs = 0, cap_dmax = 0, cap_cmax = 0;  // allocated elements
  uint64_t generation = 0;  // bumped whenever a rebind changes the data or any buffer address
  uint32_t* order_keys = nullptr;  // 2G: the sort keys and their sorted copy
  uint8_t* sort_tmp = nullptr;
  uint64_t cap_keys = 0, cap_sort = 0;
  ~sigmo_db() {
    bfree(order_keys);
    bfree(sort_tmp);
    bfree(cls_list);
    bfree(planes);
    bfree(labs);
    bfree(dmax);
    bfree(cmax);
    bfree(minfo);
  }
};

struct sigmo_batch {
  sigmo_ctx* ctx = nullptr;
  const sigmo_db* db = nullptr;
  // query side
  uint16_t* tokens = nullptr;
  sigmo_k::QueryInfo* qinfo = nullptr;
  uint64_t* qmax = nullptr;
  uint64_t* qcmax = nullptr;  // per-class maxima, [(g*3 + k)*R + r]
  uint64_t cap_tokens = 0, cap_qinfo = 0, cap_qmax = 0, cap_qcmax = 0;
  // pair evaluation
  uint64_t* arena = nullptr;
  uint64_t cap_arena = 0;
  bool compact = false;  // the arena keeps only the survivors' masks (size_arena)
  unsigned long long* surv = nullptr;
  uint64_t cap_surv = 0;
  uint4* blocks = nullptr;
  uint64_t cap_blocks = 0;
  uint32_t* mol_count = nullptr;
  uint64_t cap_mc = 0;
  unsigned long long* counters = nullptr;
  // canonical GMCR and join
  uint32_t *offsets = nullptr, *indices = nullptr, *pair_graph = nullptr, *mask_off = nullptr;
  uint64_t cap_off = 0, cap_idx = 0, cap_pg = 0, cap_mo = 0;
  uint64_t* scan_tmp = nullptr;
  uint64_t cap_scan = 0;
  uint64_t* total = nullptr;
  int32_t* counts = nullptr;
  uint64_t cap_counts = 0;
  uint32_t* wide_pairs = nullptr;  // pairs of molecules with > 64 nodes, for the two-word lane join
  uint64_t cap_wide = 0;
  uint32_t* deep_pairs = nullptr;  // pairs of queries deeper than the lane join's first pass holds
  uint64_t cap_deep = 0;
  unsigned long long* run_host = nullptr;  // pinned: a run's filter counters, then the GMCR total
  uint32_t* req_offsets = nullptr;        // per-request statistics
  unsigned long long* req_out = nullptr;
  sigmo_batch_tuning tune{};               // 0 fields: the built-in heuristics
  // a captured run (sigmo_batch_capture): the graph, its sizes and its pinned readback
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  unsigned long long* graph_host = nullptr;  // filter counters, GMCR total, 8 words of join stats
  uint64_t graph_P = 0, graph_nw = 0, graph_db_generation = 0;
  uint32_t graph_Gq = 0;
  int graph_find_first = 0;
  void drop_graph() {
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    if (graph) (void)hipGraphDestroy(graph);
    graph_exec = nullptr;
    graph = nullptr;
  }
  // bgrow, dropping a captured graph whose buffer addresses a reallocation would invalidate
  template <typename T>
  int grow(T** p, uint64_t& cap, uint64_t need, bool slack = false) {
    if (*p && cap >= need) return SIGMO_OK;
    drop_graph();
    return bgrow(p, cap, slack ? need + need / 4 : need);
  }
  uint64_t P = 0;
  uint32_t Gq = 0;
  bool ran = false;
  ~sigmo_batch() {
    bfree(tokens);
    bfree(qinfo);
    bfree(qmax);
    bfree(qcmax);
    bfree(arena);
    bfree(surv);
    bfree(blocks);
    bfree(mol_count);
    bfree(counters);
    bfree(offsets);
    bfree(indices);
    bfree(pair_graph);
    bfree(mask_off);
    bfree(scan_tmp);
    bfree(total);
    bfree(counts);
    bfree(wide_pairs);
    bfree(deep_pairs);
    bfree(req_offsets);
    bfree(req_out);
    drop_graph();
    if (graph_host) (void)hipHostFree(graph_host);
    if (run_host) (void)hipHostFree(run_host);
  }
};

sigmo_ctx* sigmo_internal::batch_ctx(const sigmo_batch* b) { return b->ctx; }

namespace {
// The pre-test's class labels: the three most frequent node labels < 16 of the data (ties to the
// smaller label), unused slots where fewer occur.  Any choice gives the same results; frequent
// labels prune most.
int choose_classes(sigmo_db* db, const sigmo_graph* data, hipStream_t s) {
  const sigmo_k::GraphDev g = graph_dev(data);
  unsigned long long* hist = nullptr;
  BATCH_TRY(balloc(&hist, 256));
  std::vector<unsigned long long> h(256, 0);
  hipError_t e = sigmo_k::label_hist(s, g.nl, g.N, hist);
  if (e == hipSuccess) e = hipMemcpyAsync(h.data(), hist, 256 * sizeof(unsigned long long), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  bfree(hist);
  if (e != hipSuccess) return sigmo_err::set(SIGMO_ERR_HIP, std::string("label histogram: ") + hipGetErrorString(e));
  db->num_labels = 0;
  for (uint32_t l = 0; l < 16; ++l) db->num_labels += h[l] != 0;
  for (uint32_t k = 0; k < sigmo_k::kClasses; ++k) {
    uint32_t best = 0xFFFFFFFFu;
    for (uint32_t l = 0; l < 16; ++l)
      if (h[l] && (best == 0xFFFFFFFFu || h[l] > h[best])) best = l;
    db->cls.l[k] = best;
    if (best != 0xFFFFFFFFu) h[best] = 0;
  }
  return SIGMO_OK;
}

// (Re)build the database's class lists and level planes for `data`; buffers are reused when
// the new graph fits them (a streaming chunk), grown otherwise.
int db_fill(sigmo_db* db, const sigmo_graph* data) {
  int device = 0, cus = 0;
  hipStream_t s;
  unsigned long long *st, *sh;
  BATCH_TRY(ctx_info(db->ctx, &device, &s, &cus, &st, &sh));
  const auto& go = graph_host_offsets(data);
  const uint32_t G = static_cast<uint32_t>(go.size() - 1);
  sigmo_k::GroupOrder order{{0, 0, 0}};
  for (uint32_t g = 0; g < G; ++g) {
    const uint32_t n = go[g + 1] - go[g];
    ++order.count[n <= 32 ? 0 : (n <= 64 ? 1 : 2)];
  }
  const uint64_t R = db->R, groups = order.total();
  uint64_t cap_g = db->cap_G;
  BATCH_TRY(bgrow(&db->cls_list, cap_g, G));
  cap_g = db->cap_G;
  BATCH_TRY(bgrow(&db->minfo, cap_g, G));
  db->cap_G = cap_g;
  BATCH_TRY(bgrow(&db->dmax, db->cap_dmax, uint64_t(G) * R));
  BATCH_TRY(bgrow(&db->cmax, db->cap_cmax, uint64_t(G) * R * sigmo_k::kClasses));
  BATCH_TRY(bgrow_slack(&db->planes, db->cap_planes, groups * R * 16 * 64 * 4));
  BATCH_TRY(bgrow_slack(&db->labs, db->cap_labs, groups * 16 * 64));
  db->data = data;
  db->generation++;
  db->num_wide = order.count[2];
  db->order = order;
  db->bytes = G * (4ull + sizeof(sigmo_k::MolInfo)) + groups * 16 * 64 * (16 * R + 4) + uint64_t(G) * R * 8 * (1 + sigmo_k::kClasses);
  BATCH_TRY(choose_classes(db, data, s));
  // the width-class order: molecules sorted by (class, label set, size), stably (by index within a key)
  BATCH_TRY(bgrow_slack(&db->order_keys, db->cap_keys, 2ull * G));
  const sigmo_k::GraphDev gd = graph_dev(data);
  hipLaunchKernelGGL(sigmo_k::k_db_order_keys, dim3((G + 255) / 256), dim3(256), 0, s, G, gd.go, gd.nl, db->order_keys);
  BATCH_HIP_TRY(hipGetLastError());
  size_t tmp_bytes = 0;
  const rocprim::counting_iterator<uint32_t> ids(0u);
  BATCH_HIP_TRY(rocprim::radix_sort_pairs(nullptr, tmp_bytes, db->order_keys, db->order_keys + G, ids, db->cls_list, G, 0u, 25u, s));
  BATCH_TRY(bgrow_slack(&db->sort_tmp, db->cap_sort, std::max<uint64_t>(tmp_bytes, 1)));
  BATCH_HIP_TRY(rocprim::radix_sort_pairs(db->sort_tmp, tmp_bytes, db->order_keys, db->order_keys + G, ids, db->cls_list, G, 0u, 25u, s));
  BATCH_TRY(sigmo_db_refresh(db));
  BATCH_HIP_TRY(hipStreamSynchronize(s));
  return SIGMO_OK;
}
}  // namespace

namespace sigmo_internal {
int db_rebind(sigmo_db* db, const sigmo_graph* data) {
  if (!db || !data) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  return db_fill(db, data);
}
}  // namespace sigmo_internal

extern "C" {

int sigmo_db_prepare(sigmo_ctx* ctx, const sigmo_graph* data, uint32_t refinement_steps, sigmo_db** out) {
  int device = 0, cus = 0;
  hipStream_t s;
  unsigned long long *st, *sh;
  BATCH_TRY(ctx_info(ctx, &device, &s, &cus, &st, &sh));
  if (!data || !out) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  if (refinement_steps == 0 || refinement_steps > sigmo_k::kMaxLevels)
    return sigmo_err::set(SIGMO_ERR_UNSUPPORTED, "the batched form supports 1..8 refinement levels");
  auto* db = new sigmo_db();
  db->ctx = ctx;
  db->R = refinement_steps;
  const int stt = db_fill(db, data);
  if (stt != SIGMO_OK) {
    delete db;
    return stt;
  }
  *out = db;
  return SIGMO_OK;
}

int sigmo_db_refresh(sigmo_db* db) {
  if (!db) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  int device = 0, cus = 0;
  hipStream_t s;
  unsigned long long *st, *sh;
  BATCH_TRY(ctx_info(db->ctx, &device, &s, &cus, &st, &sh));
  const sigmo_k::GraphDev g = graph_dev(db->data);
  // algorithmic bytes: the CSR and labels read once, R level signatures per data node written:
  // 4(D+1) + 4E + D + 8 R D
  const double bytes = 4.0 * (double(g.N) + 1.0) + 4.0 * double(graph_edges(db->data)) + double(g.N) + 8.0 * db->R * double(g.N);
  void* tok = nullptr;
  BATCH_TRY(ctx_timed(db->ctx, SIGMO_PHASE_SIG_DATA, SIGMO_KERNEL_DB_PREPARE, bytes, true, &tok));
  BATCH_HIP_TRY(sigmo_k::db_prepare(s, g, db->R, db->cls_list, db->order, db->planes, db->labs, db->dmax, db->minfo, db->cls, db->cmax));
  BATCH_TRY(ctx_timed(db->ctx, 0, 0, 0.0, false, &tok));
  return SIGMO_OK;
}

int sigmo_db_free(sigmo_db* db) {
  if (!db) return SIGMO_OK;
  int device = 0, cus = 0;
  hipStream_t s;
  unsigned long long *st, *sh;
  if (ctx_info(db->ctx, &device, &s, &cus, &st, &sh) == SIGMO_OK) (void)hipStreamSynchronize(s);
  delete db;
  return SIGMO_OK;
}

int sigmo_db_alloc_size(const sigmo_db* db, uint64_t* bytes) {
  if (!db || !bytes) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  *bytes = db->bytes;
  return SIGMO_OK;
}

int sigmo_batch_create(sigmo_ctx* ctx, const sigmo_db* db, sigmo_batch** out) {
  int device = 0, cus = 0;
  hipStream_t s;
  unsigned long long *st, *sh;
  BATCH_TRY(ctx_info(ctx, &device, &s, &cus, &st, &sh));
  if (!db || !out) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  auto* b = new sigmo_batch();
  b->ctx = ctx;
  b->db = db;
  int stt = balloc(&b->counters, kCounterWords);
  if (stt == SIGMO_OK) stt = balloc(&b->total, 1);
  if (stt != SIGMO_OK) {
    delete b;
    return stt;
  }
  *out = b;
  return SIGMO_OK;
}

int sigmo_batch_workspace_bytes(const sigmo_batch* b, uint32_t num_query_graphs, uint64_t query_nodes, uint64_t* bytes) {
  if (!b || !bytes) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  const sigmo_db* db = b->db;
  const uint64_t Gd = graph_dev(db->data).G, Gq = num_query_graphs, R = db->R;
  const uint64_t pairs = Gq * Gd, W = (Gq + 63) / 64;
  const double mean_k = Gq ? double(query_nodes) / double(Gq) : 0.0;
  // the arena's first sizing (see sigmo_batch_run) without the per-wavefront slack.  The GMCR
  // arrays (indices, molecule, arena offset, count: 16 B per pair) are sized for every pair on
  // the one-synchronisation path (pair space <= kOneSyncPairs, no molecule over 64 nodes), and
  // for the pairs that survive otherwise, priced at the arena's guess of 1/8 of the pairs (plus
  // 4 B per pair for the list of wide-molecule pairs).  A run whose survivors exceed the guess
  // grows the arena and those arrays to the measured demand; a batch keeps its buffers at their
  // largest size, so a caller admitting by this figure should leave room for that growth.  Not
  // priced: the wavefronts' chunks (twice L.first_chunks words in shape_run, 4 MB to 1.6 GB by the
  // pair space and the device) and the deep queries' list (4 B per GMCR pair).
  const uint64_t guess = std::min<uint64_t>(std::max<uint64_t>(pairs / 8, 1 << 16), 1ull << 26);
  const uint64_t arena_words = static_cast<uint64_t>(double(guess) * (mean_k + 1.0) * (db->num_wide ? 2.0 : 1.0));
  const bool one_sync = !db->num_wide && pairs && pairs <= kOneSyncPairs;
  const uint64_t gmcr_pairs = one_sync ? pairs : guess;
  *bytes = query_nodes * sigmo_k::token_segment(static_cast<uint32_t>(R)) * 2 + Gq * (sizeof(sigmo_k::QueryInfo) + 8 * R * (1 + sigmo_k::kClasses)) +
           Gd * W * 8 + uint64_t(db->order.total()) * Gq * 16 + arena_words * 8 + gmcr_pairs * 16 + (db->num_wide ? guess * 4 : 0) + (Gd + 1) * 8;
  return SIGMO_OK;
}

int sigmo_batch_request_stats(sigmo_batch* b, const uint32_t* request_graph_offsets, uint32_t num_requests, sigmo_request_stats* out) {
  if (!b || !b->ran) return sigmo_err::set(SIGMO_ERR_INVALID, "batch has not run");
  if (!request_graph_offsets || !out || num_requests == 0) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  if (num_requests > sigmo_k::kMaxBatchRequests) return sigmo_err::set(SIGMO_ERR_UNSUPPORTED, "at most 256 requests per batch");
  if (request_graph_offsets[0] != 0 || request_graph_offsets[num_requests] != b->Gq)
    return sigmo_err::set(SIGMO_ERR_INVALID, "request graph offsets must cover the batch's query graphs");
  for (uint32_t r = 0; r < num_requests; ++r)
    if (request_graph_offsets[r + 1] < request_graph_offsets[r]) return sigmo_err::set(SIGMO_ERR_INVALID, "request graph offsets must ascend");
  int device = 0, cus = 0;
  hipStream_t s;
  unsigned long long *st, *sh;
  BATCH_TRY(ctx_info(b->ctx, &device, &s, &cus, &st, &sh));
  if (!b->req_offsets) BATCH_TRY(balloc(&b->req_offsets, sigmo_k::kMaxBatchRequests + 1));
  if (!b->req_out) BATCH_TRY(balloc(&b->req_out, sigmo_k::kStatsOutWords));
  BATCH_HIP_TRY(hipMemcpyAsync(b->req_offsets, request_graph_offsets, (num_requests + 1) * 4ull, hipMemcpyHostToDevice, s));
  const uint32_t copies = sigmo_k::stats_copies(num_requests), stride = sigmo_k::stats_stride(num_requests);
  uint32_t shared = 64;  // copies of a request's sums in LDS
  while (shared * num_requests > sigmo_k::kStatsBlock) shared /= 2;
  BATCH_HIP_TRY(sigmo_k::fill_u64(s, reinterpret_cast<uint64_t*>(b->req_out), static_cast<uint64_t>(copies) * stride, 0));
  if (b->P) {
    const uint64_t per = 4ull * sigmo_k::kStatsBlock;
    const uint64_t blocks = std::min<uint64_t>((b->P + per - 1) / per, static_cast<uint64_t>(cus) * 2);
    hipLaunchKernelGGL(sigmo_k::k_request_stats, dim3(static_cast<unsigned>(blocks)), dim3(sigmo_k::kStatsBlock), 0, s, b->P, b->indices, b->pair_graph,
                       b->counts, b->req_offsets, num_requests, shared, copies, b->req_out);
    BATCH_HIP_TRY(hipGetLastError());
  }
  std::vector<unsigned long long> h(static_cast<uint64_t>(copies) * stride);
  const sigmo_k::HostCopy back = {h.data(), b->req_out, h.size() * 8};
  BATCH_TRY(ctx_read_back(b->ctx, &back, 1));
  for (uint32_t r = 0; r < num_requests; ++r) {
    out[r] = sigmo_request_stats{0, 0, 0};
    for (uint32_t i = 0; i < copies; ++i) {
      const unsigned long long* at = h.data() + static_cast<uint64_t>(i) * stride + 3 * r;
      out[r].matched_pairs += at[0];
      out[r].embeddings += at[1];
      out[r].hash += at[2];
    }
  }
  return SIGMO_OK;
}

int sigmo_batch_free(sigmo_batch* b) {
  if (!b) return SIGMO_OK;
  int device = 0, cus = 0;
  hipStream_t s;
  unsigned long long *st, *sh;
  if (ctx_info(b->ctx, &device, &s, &cus, &st, &sh) == SIGMO_OK) (void)hipStreamSynchronize(s);
  delete b;
  return SIGMO_OK;
}

}  // extern "C"

namespace {

// Launch shape and sizes of one batched run, fixed before any launch.
struct RunShape {
  sigmo_k::GraphDev qd, dd;
  uint32_t R = 0, Gq = 0, Gd = 0, W = 0;
  uint64_t pairs = 0, ksum = 0;
  int cus = 0;
  uint32_t group_blocks = 0, group_parts = 1, group_slots = 1, group_chunk = 0;  // the pair evaluation's launch
  uint64_t first_chunks = 0;  // arena words its wavefronts start with
};

int shape_run(const sigmo_batch* b, const sigmo_graph* query, int cus, RunShape& L) {
  const sigmo_db* db = b->db;
  L.qd = graph_dev(query);
  L.dd = graph_dev(db->data);
  const auto& qgo = graph_host_offsets(query);
  L.Gq = L.qd.G;
  L.Gd = L.dd.G;
  L.cus = cus;
  for (uint32_t g = 0; g < L.Gq; ++g) {
    const uint32_t k = qgo[g + 1] - qgo[g];
    if (k < 2) return sigmo_err::set(SIGMO_ERR_INVALID, "query graph " + std::to_string(g) + " has fewer than 2 nodes");
    if (k > SIGMO_MAX_QUERY_NODES) return sigmo_err::set(SIGMO_ERR_UNSUPPORTED, "query graph exceeds 32 nodes");
    L.ksum += k;
  }
  L.R = db->R;
  L.W = (L.Gq + 63) / 64;
  L.pairs = uint64_t(L.Gq) * L.Gd;
  const uint64_t groups = db->order.total(), ucus = static_cast<uint64_t>(cus);
  // a group's query graphs go to one block, or to more where the groups alone leave CUs idle
  while (L.group_parts < 8 && groups * L.group_parts < 2 * ucus && sigmo_k::kGroupWaves * L.group_parts < L.Gq)
    L.group_parts *= 2;
  const uint64_t items = groups * L.group_parts;
  // LDS for every label that occurs, within 64 KB (a byte names a plane); with blocks to
  // spare within 53 KB, so that three stay resident (a group of neighbours in the width-class order
  // holds 4 to 6 labels)
  const uint32_t lds = (items > 2 * ucus ? 53u : 64u) * 1024, block = sigmo_k::slot_planes(L.R) * 256;
  L.group_slots = std::max<uint32_t>(1, std::min<uint32_t>(db->num_labels, (lds - sigmo_k::kGroupListBytes) / block - 1));
  uint64_t per_cu = std::max<uint64_t>(1, std::min<uint64_t>(32 / sigmo_k::kGroupWaves, 160 * 1024 / sigmo_k::group_lds_bytes(L.group_slots, L.R)));
  if (b->tune.filter_blocks_per_cu) per_cu = std::min<uint64_t>(per_cu, b->tune.filter_blocks_per_cu);
  L.group_blocks = static_cast<uint32_t>(std::max<uint64_t>(1, std::min<uint64_t>(items, ucus * per_cu)));
  // a wavefront's arena chunk holds the largest query graph for a whole group (1,024 words) and, for
  // many pairs, more: claims meet on one address.  Every wavefront has one and may leave another's tail:
  // at most 1.6 GB for 6,144 wavefronts
  const uint64_t waves = uint64_t(L.group_blocks) * sigmo_k::kGroupWaves;
  uint64_t chunk = 2048;
  while (chunk < 16384 && chunk * waves * 4 < L.pairs) chunk *= 2;
  L.group_chunk = static_cast<uint32_t>(chunk);
  L.first_chunks = waves * chunk;
  return SIGMO_OK;
}

// Pair filter: the pre-test over every pair (its bits in surv), then the evaluation of the passing
// pairs.  Counters are cleared by a kernel.  Deaths clear their pre-test bit, so surv ends as the
// GMCR survival bitmask.
hipError_t launch_filter(sigmo_batch* b, const RunShape& L, hipStream_t s) {
  const sigmo_db* db = b->db;
  hipError_t e = sigmo_k::fill_u64(s, reinterpret_cast<uint64_t*>(b->counters), kCounterWords, 0);
  if (e != hipSuccess || !L.Gd || !L.Gq) return e;
  sigmo_k::PretestArgs p;
  p.R = L.R;
  p.Gq = L.Gq;
  p.W = L.W;
  p.G = L.Gd;
  p.minfo = db->minfo;
  p.dmax = db->dmax;
  p.cmax = db->cmax;
  p.qinfo = b->qinfo;
  p.qmax = b->qmax;
  p.qcmax = b->qcmax;
  p.surv = b->surv;
  const dim3 pgrid((L.Gd + 255) / 256);
  switch (L.R) {  // one instantiation per level count keeps the molecule's maxima in registers
    case 1: hipLaunchKernelGGL(sigmo_k::k_pair_pretest<1>, pgrid, dim3(256), 0, s, p); break;
    case 2: hipLaunchKernelGGL(sigmo_k::k_pair_pretest<2>, pgrid, dim3(256), 0, s, p); break;
    case 3: hipLaunchKernelGGL(sigmo_k::k_pair_pretest<3>, pgrid, dim3(256), 0, s, p); break;
    case 4: hipLaunchKernelGGL(sigmo_k::k_pair_pretest<4>, pgrid, dim3(256), 0, s, p); break;
    case 5: hipLaunchKernelGGL(sigmo_k::k_pair_pretest<5>, pgrid, dim3(256), 0, s, p); break;
    case 6: hipLaunchKernelGGL(sigmo_k::k_pair_pretest<6>, pgrid, dim3(256), 0, s, p); break;
    case 7: hipLaunchKernelGGL(sigmo_k::k_pair_pretest<7>, pgrid, dim3(256), 0, s, p); break;
    default: hipLaunchKernelGGL(sigmo_k::k_pair_pretest<8>, pgrid, dim3(256), 0, s, p); break;
  }
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  sigmo_k::GroupArgs a;
  a.d = L.dd;
  a.order = db->order;
  a.R = L.R;
  a.Gq = L.Gq;
  a.W = L.W;
  a.parts = L.group_parts;
  a.slots = L.group_slots;
  a.rich = db->cls.l[0];
  a.chunk = L.group_chunk;
  a.minfo = db->minfo;
  a.planes = reinterpret_cast<const uint4*>(db->planes);
  a.labs = db->labs;
  a.tokens = reinterpret_cast<const uint64_t*>(b->tokens);
  a.qinfo = b->qinfo;
  a.arena = b->arena;
  a.arena_cap = b->cap_arena;
  a.surv = b->surv;
  a.blocks = b->blocks;
  a.counters = b->counters;
  a.stats = b->counters + 16;
  hipLaunchKernelGGL(b->compact ? sigmo_k::k_pair_group<true> : sigmo_k::k_pair_group<false>, dim3(L.group_blocks), dim3(sigmo_k::kGroupWaves * 64),
                     sigmo_k::group_lds_bytes(L.group_slots, L.R), s, a);
  return hipGetLastError();
}

// The filter's statistics and arena demand from its counters on the host.
uint64_t read_counters(uint64_t first_chunks, const unsigned long long* cnt, sigmo_batch_result* res) {
  res->filter_wave_steps = res->filter_lane_steps = res->filter_scans = 0;
  for (uint32_t i = 0; i < sigmo_k::kGroupStatSlots; ++i) {
    res->filter_wave_steps += cnt[16 + 16 * i];
    res->filter_lane_steps += cnt[16 + 16 * i + 1];
    res->filter_scans += cnt[16 + 16 * i + 2];
  }
  return cnt[1] + first_chunks;
}

// What the arena is to hold after an overflow, given the run's demand.  Where the pre-tested pairs took
// more than twice what the survivors need (labels >= 16 and wildcards leave the pre-test little to go
// by), the batch goes over to the form that keeps only these, for this and later runs: in every run, it
// would take 4.36 instead of 3.49 ms for 1 M molecules x 1,000 query graphs.
int size_arena(sigmo_batch* b, const RunShape& L, hipStream_t s, uint64_t demand, uint64_t slack, uint64_t& want) {
  bool larger = true;
  if (!b->compact) {
    const sigmo_db* db = b->db;
    unsigned long long words = 0;
    hipLaunchKernelGGL(sigmo_k::k_surv_words, dim3((L.Gd + 255) / 256), dim3(256), 0, s, db->order, L.Gd, L.W, db->minfo, b->qinfo, b->surv,
                       b->counters + 4);
    BATCH_HIP_TRY(hipGetLastError());
    BATCH_HIP_TRY(hipMemcpyAsync(&words, b->counters + 4, sizeof(words), hipMemcpyDeviceToHost, s));
    BATCH_HIP_TRY(hipStreamSynchronize(s));
    if (demand > 2 * words + slack) {
      b->compact = true;
      demand = 2 * words;  // a wavefront may leave up to half of each chunk, of at least two groups' largest blocks
      larger = demand + slack > b->cap_arena;
    }
  }
  // the claim order (and so the space left unused at chunk ends) varies between runs, hence the 1/8 margin
  if (larger) {
    if (demand > kMaxArenaWords || want >= kMaxArenaWords) return sigmo_err::set(SIGMO_ERR_OVERFLOW, "candidate arena exceeds 2^32 words");
    want = std::min(kMaxArenaWords, std::max<uint64_t>(want + 1, demand + demand / 8 + slack));
  }
  return SIGMO_OK;
}

// GMCR: survivors per molecule and their exclusive scan (total in b->total).
hipError_t launch_count_scan(sigmo_batch* b, const RunShape& L, hipStream_t s) {
  if (L.Gd) {
    hipLaunchKernelGGL(sigmo_k::k_surv_count, dim3((L.Gd + 255) / 256), dim3(256), 0, s, L.Gd, L.W, b->surv, b->mol_count);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return sigmo_k::exclusive_scan(s, b->mol_count, L.Gd, b->offsets, b->scan_tmp, b->total);
}

hipError_t launch_scatter(sigmo_batch* b, const RunShape& L, hipStream_t s) {
  if (!L.Gd) return hipSuccess;
  const uint64_t cap = std::min(b->cap_idx, std::min(b->cap_pg, b->cap_mo));
  const sigmo_k::GroupOrder& order = b->db->order;
  if (L.W == 1) {  // at most 64 query graphs: a lane per molecule
    const dim3 grid((order.total() + 3) / 4);
    hipLaunchKernelGGL(sigmo_k::k_surv_scatter_lanes, grid, dim3(256), 0, s, order, L.Gq, b->db->minfo, b->surv, b->offsets, b->blocks, b->indices,
                       b->pair_graph, b->mask_off, cap);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(sigmo_k::k_surv_scatter, dim3(order.total()), dim3(256), 0, s, order, L.Gq, L.W, b->db->minfo, b->surv, b->offsets, b->blocks,
                     b->indices, b->pair_graph, b->mask_off, cap);
  return hipGetLastError();
}

// Lane join over P pairs: for many pairs a shallow first pass and a second over the pairs of deeper
// queries (deep_pairs); pairs of molecules of > 64 nodes are listed (wide_pairs) for the last pass.
hipError_t launch_join(sigmo_batch* b, const RunShape& L, hipStream_t s, unsigned long long* stats, uint64_t P, int find_first,
                       const unsigned long long* P_dev = nullptr) {
  if (!P) return hipSuccess;
  const uint32_t quarters = b->tune.join_blocks_per_cu ? std::min<uint32_t>(b->tune.join_blocks_per_cu, 4) : 4;
  return sigmo_k::launch_join_lanes(s, L.qd, L.dd, sigmo_k::ArenaMasks{b->arena, b->mask_off, b->counters + 3}, b->offsets, b->indices, b->pair_graph,
                                    P, find_first, b->counts, stats, b->db->num_wide ? b->wide_pairs : nullptr, L.cus, P_dev, b->deep_pairs, quarters,
                                    b->tune.join_chunk);
}

// Buffers of a run that do not depend on its results.
int size_fixed_buffers(sigmo_batch* b, const RunShape& L) {
  const uint64_t seg = sigmo_k::token_segment(L.R);
  if (L.qd.N * seg >= (1ull << 32)) return sigmo_err::set(SIGMO_ERR_UNSUPPORTED, "query batch too large for one batched run");
  BATCH_TRY(b->grow(&b->tokens, b->cap_tokens, L.qd.N * seg));
  BATCH_TRY(b->grow(&b->qinfo, b->cap_qinfo, L.Gq));
  BATCH_TRY(b->grow(&b->qmax, b->cap_qmax, uint64_t(L.Gq) * L.R));
  BATCH_TRY(b->grow(&b->qcmax, b->cap_qcmax, uint64_t(L.Gq) * L.R * sigmo_k::kClasses));
  BATCH_TRY(b->grow(&b->surv, b->cap_surv, uint64_t(L.Gd) * L.W));
  BATCH_TRY(b->grow(&b->blocks, b->cap_blocks, uint64_t(b->db->order.total()) * L.Gq));
  BATCH_TRY(b->grow(&b->mol_count, b->cap_mc, uint64_t(L.Gd) + 1));
  BATCH_TRY(b->grow(&b->offsets, b->cap_off, uint64_t(L.Gd) + 1));
  BATCH_TRY(b->grow(&b->scan_tmp, b->cap_scan, (uint64_t(L.Gd) + 1023) / 1024 + 1));
  return SIGMO_OK;
}

}  // namespace

extern "C" {

int sigmo_batch_run(sigmo_batch* b, const sigmo_graph* query, int find_first, sigmo_batch_result* res) {
  if (!b || !query || !res) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  int device = 0, cus = 0;
  hipStream_t s;
  unsigned long long *stats, *stats_host;
  BATCH_TRY(ctx_info(b->ctx, &device, &s, &cus, &stats, &stats_host));
  std::memset(res, 0, sizeof(*res));
  const sigmo_db* db = b->db;
  RunShape L;
  BATCH_TRY(shape_run(b, query, cus, L));
  const uint32_t R = L.R, Gq = L.Gq, Gd = L.Gd, W = L.W;
  // From here on the result arrays are overwritten: until this run succeeds, no earlier run's
  // results may be read (sigmo_batch_pairs, sigmo_batch_request_stats), so `ran` is cleared and
  // set again only on success.  `sized` remembers that an earlier run sized the arena.
  const bool sized = b->ran;
  b->ran = false;
  BATCH_TRY(size_fixed_buffers(b, L));
  {
    void* tok = nullptr;
    BATCH_TRY(ctx_timed(b->ctx, SIGMO_PHASE_SIG_QUERY, -1, 0.0, true, &tok));
    BATCH_HIP_TRY(sigmo_k::query_prepare(s, L.qd, R, b->tokens, b->qinfo, b->qmax, db->cls, b->qcmax));
    BATCH_TRY(ctx_timed(b->ctx, 0, 0, 0.0, false, &tok));
  }
  // arena capacity: start from 1/8 of the pairs (at most 2^26) plus every wavefront's open chunk.
  // On overflow the counter still holds the demand, so one replay with that size, or of the
  // survivors' masks alone, suffices; the capacity is kept for later runs.
  const double mean_k = Gq ? double(L.ksum) / Gq : 0.0;
  // every wavefront starts with a chunk and may leave its last one's tail unused
  const uint64_t slack_arena = 2 * L.first_chunks;
  const uint64_t guess = std::min<uint64_t>(std::max<uint64_t>(L.pairs / 8, 1 << 16), 1ull << 26);
  uint64_t want_arena = static_cast<uint64_t>(double(guess) * (mean_k + 1.0) * (db->num_wide ? 2.0 : 1.0)) + slack_arena;
  want_arena = std::max(std::min(want_arena, kMaxArenaWords), b->cap_arena);
  // One synchronisation per run once an earlier run has sized the arena: with no molecule of
  // more than 64 nodes and a pair space of at most kOneSyncPairs, the GMCR arrays are sized for
  // every pair, the join reads the pair count on the device, and the filter's counters and the
  // total are read after the join.  An arena overflow (data that changed) falls back to the
  // sized path below, which repeats the run.
  const uint64_t bound = uint64_t(Gq) * Gd;
  if (!b->run_host) BATCH_HIP_TRY(hipHostMalloc(reinterpret_cast<void**>(&b->run_host), (kCounterWords + 1) * sizeof(unsigned long long)));
  const unsigned long long* cnt = b->run_host;
  if (sized && !db->num_wide && bound && bound <= kOneSyncPairs && b->arena && b->cap_arena >= want_arena) {
    BATCH_TRY(b->grow(&b->indices, b->cap_idx, bound));
    BATCH_TRY(b->grow(&b->pair_graph, b->cap_pg, bound));
    BATCH_TRY(b->grow(&b->mask_off, b->cap_mo, bound));
    BATCH_TRY(b->grow(&b->counts, b->cap_counts, bound));
    BATCH_TRY(b->grow(&b->deep_pairs, b->cap_deep, bound));
    const double reads = (1.0 + 8.0 * R) * double(L.dd.N) + double(L.qd.N) * (1.0 + 2.0 * 16.0 * R) + double(Gq) * (4.0 + 8.0 * R);
    void* tok = nullptr;
    BATCH_TRY(ctx_timed(b->ctx, SIGMO_PHASE_FILTER, SIGMO_KERNEL_PAIR_FILTER, reads, true, &tok));
    BATCH_HIP_TRY(launch_filter(b, L, s));
    BATCH_TRY(ctx_timed(b->ctx, 0, 0, 0.0, false, &tok));
    res->one_sync = 1;
    BATCH_HIP_TRY(hipMemcpyAsync(b->run_host, b->counters, kCounterWords * sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
    BATCH_TRY(ctx_timed(b->ctx, SIGMO_PHASE_GMCR, -1, 0.0, true, &tok));
    BATCH_HIP_TRY(launch_count_scan(b, L, s));
    BATCH_HIP_TRY(launch_scatter(b, L, s));
    BATCH_TRY(ctx_timed(b->ctx, 0, 0, 0.0, false, &tok));
    BATCH_HIP_TRY(hipMemcpyAsync(b->run_host + kCounterWords, b->total, sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
    BATCH_TRY(ctx_timed(b->ctx, SIGMO_PHASE_JOIN, SIGMO_KERNEL_JOIN, 0.0, true, &tok));
    BATCH_HIP_TRY(sigmo_k::fill_u64(s, reinterpret_cast<uint64_t*>(stats), sigmo_k::kJoinStatWords, 0));
    BATCH_HIP_TRY(launch_join(b, L, s, stats, bound, find_first, reinterpret_cast<const unsigned long long*>(b->total)));
    BATCH_TRY(ctx_timed(b->ctx, 0, 0, 0.0, false, &tok));
    BATCH_HIP_TRY(hipMemcpyAsync(stats_host, stats, 8 * sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
    BATCH_HIP_TRY(hipStreamSynchronize(s));
    const uint64_t demand = read_counters(L.first_chunks, cnt, res);
    if (!cnt[3]) {
      const uint64_t P = b->run_host[kCounterWords];
      if (P >= (1ull << 32)) return sigmo_err::set(SIGMO_ERR_OVERFLOW, "GMCR pair count exceeds u32");
      if (stats_host[3]) return sigmo_err::set(SIGMO_ERR_OVERFLOW, "a per-pair match count exceeded int32");
      ctx_add_bytes(b->ctx, SIGMO_KERNEL_PAIR_FILTER, double(demand) * 8.0 + double(Gd) * W * 8.0);
      b->P = P;
      b->Gq = Gq;
      b->ran = true;
      res->num_matches = stats_host[0];
      res->matched_pairs = stats_host[1];
      res->gmcr_pairs = P;
      res->dfs_steps = stats_host[4];
      res->join_wave_steps = stats_host[7];
      return SIGMO_OK;
    }
    BATCH_TRY(size_arena(b, L, s, demand, slack_arena, want_arena));  // overflowed: size and repeat
    res->arena_repeats = 1;
  }
  for (int attempt = 0; attempt < 4; ++attempt) {
    BATCH_TRY(b->grow(&b->arena, b->cap_arena, want_arena));
    // algorithmic reads: the data side once per run -- a label byte and R level signatures per
    // data node, (1 + 8R) D -- plus the query side; writes are added once they are known.
    const double reads = (1.0 + 8.0 * R) * double(L.dd.N) + double(L.qd.N) * (1.0 + 2.0 * 16.0 * R) + double(Gq) * (4.0 + 8.0 * R);
    void* tok = nullptr;
    BATCH_TRY(ctx_timed(b->ctx, SIGMO_PHASE_FILTER, SIGMO_KERNEL_PAIR_FILTER, reads, true, &tok));
    BATCH_HIP_TRY(launch_filter(b, L, s));
    BATCH_TRY(ctx_timed(b->ctx, 0, 0, 0.0, false, &tok));
    BATCH_HIP_TRY(hipMemcpyAsync(b->run_host, b->counters, kCounterWords * sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
    BATCH_HIP_TRY(hipStreamSynchronize(s));
    const uint64_t demand = read_counters(L.first_chunks, cnt, res);
    if (res->filter_scans >= (1ull << 32)) return sigmo_err::set(SIGMO_ERR_OVERFLOW, "pre-tested pairs of one run exceed 2^32");
    // writes: candidate masks and the survival bits
    ctx_add_bytes(b->ctx, SIGMO_KERNEL_PAIR_FILTER, double(demand) * 8.0 + double(Gd) * W * 8.0);
    if (!cnt[3]) break;
    if (attempt == 3) return sigmo_err::set(SIGMO_ERR_NOMEM, "candidate arena overflowed repeatedly");
    res->arena_repeats++;
    BATCH_TRY(size_arena(b, L, s, demand, slack_arena, want_arena));
  }
  // canonical GMCR: count survivors per molecule, scan, scatter in (molecule, query graph) order
  void* tok = nullptr;
  BATCH_TRY(ctx_timed(b->ctx, SIGMO_PHASE_GMCR, -1, 0.0, true, &tok));
  BATCH_HIP_TRY(launch_count_scan(b, L, s));
  BATCH_HIP_TRY(hipMemcpyAsync(b->run_host + kCounterWords, b->total, sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
  BATCH_HIP_TRY(hipStreamSynchronize(s));
  const uint64_t P = b->run_host[kCounterWords];
  if (P >= (1ull << 32)) return sigmo_err::set(SIGMO_ERR_OVERFLOW, "GMCR pair count exceeds u32");
  // result-sized arrays regrow with a quarter to spare: each hipFree waits for the whole device
  BATCH_TRY(b->grow(&b->indices, b->cap_idx, P, true));
  BATCH_TRY(b->grow(&b->pair_graph, b->cap_pg, P, true));
  BATCH_TRY(b->grow(&b->mask_off, b->cap_mo, P, true));
  BATCH_TRY(b->grow(&b->counts, b->cap_counts, P, true));
  BATCH_TRY(b->grow(&b->wide_pairs, b->cap_wide, db->num_wide ? P : 1, true));
  BATCH_TRY(b->grow(&b->deep_pairs, b->cap_deep, P, true));
  BATCH_HIP_TRY(launch_scatter(b, L, s));
  BATCH_TRY(ctx_timed(b->ctx, 0, 0, 0.0, false, &tok));
  // join: lane per pair
  BATCH_TRY(ctx_timed(b->ctx, SIGMO_PHASE_JOIN, SIGMO_KERNEL_JOIN, 0.0, true, &tok));
  BATCH_HIP_TRY(sigmo_k::fill_u64(s, reinterpret_cast<uint64_t*>(stats), sigmo_k::kJoinStatWords, 0));
  BATCH_HIP_TRY(launch_join(b, L, s, stats, P, find_first));
  BATCH_TRY(ctx_timed(b->ctx, 0, 0, 0.0, false, &tok));
  BATCH_HIP_TRY(hipMemcpyAsync(stats_host, stats, 8 * sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
  BATCH_HIP_TRY(hipStreamSynchronize(s));
  if (stats_host[3]) return sigmo_err::set(SIGMO_ERR_OVERFLOW, "a per-pair match count exceeded int32");
  b->P = P;
  b->Gq = Gq;
  b->ran = true;
  res->num_matches = stats_host[0];
  res->matched_pairs = stats_host[1];
  res->gmcr_pairs = P;
  res->dfs_steps = stats_host[4];
  res->join_wave_steps = stats_host[7];
  return SIGMO_OK;
}

int sigmo_batch_set_tuning(sigmo_batch* b, const sigmo_batch_tuning* t) {
  if (!b || !t) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  if (t->join_blocks_per_cu > 4) return sigmo_err::set(SIGMO_ERR_INVALID, "join_blocks_per_cu must be 0..4");
  if (t->filter_claim > 64) return sigmo_err::set(SIGMO_ERR_INVALID, "filter_claim must be 0..64");
  if (t->filter_mode > 2) return sigmo_err::set(SIGMO_ERR_INVALID, "filter_mode must be 0..2");
  b->tune = *t;
  return SIGMO_OK;
}

int sigmo_batch_get_tuning(const sigmo_batch* b, sigmo_batch_tuning* t) {
  if (!b || !t) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  *t = b->tune;
  return SIGMO_OK;
}

int sigmo_batch_autotune(sigmo_batch* b, const sigmo_graph* query, int find_first, uint32_t repeats, sigmo_batch_tuning* chosen,
                         double* best_ms) {
  if (!b || !query) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  if (repeats == 0) repeats = 2;
  sigmo_batch_result r;
  BATCH_TRY(sigmo_batch_run(b, query, find_first, &r));  // sizes every buffer
  auto time_with = [&](const sigmo_batch_tuning& t, double* ms) -> int {
    b->tune = t;
    double best = 1e300;
    for (uint32_t i = 0; i < repeats; ++i) {
      const auto t0 = std::chrono::steady_clock::now();
      BATCH_TRY(sigmo_batch_run(b, query, find_first, &r));
      best = std::min(best, std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count());
    }
    *ms = best;
    return SIGMO_OK;
  };
  sigmo_batch_tuning best_t{};
  double best = 0;
  BATCH_TRY(time_with(best_t, &best));
  // coordinate search: the pair evaluation's blocks, then the join's shape
  const uint32_t filter_blocks[] = {1, 2, 4, 0};
  const uint32_t join_blocks[] = {2, 3, 4};
  const uint32_t join_chunks[] = {16, 64, 256, 0};
  auto sweep = [&](uint32_t sigmo_batch_tuning::*field, const uint32_t* vals, size_t n) -> int {
    for (size_t i = 0; i < n; ++i) {
      sigmo_batch_tuning t = best_t;
      t.*field = vals[i];
      if (t.*field == best_t.*field) continue;
      double ms = 0;
      BATCH_TRY(time_with(t, &ms));
      if (ms < best * 0.98) {  // a 2% margin against timing noise
        best = ms;
        best_t = t;
      }
    }
    return SIGMO_OK;
  };
  BATCH_TRY(sweep(&sigmo_batch_tuning::filter_blocks_per_cu, filter_blocks, 4));
  BATCH_TRY(sweep(&sigmo_batch_tuning::join_blocks_per_cu, join_blocks, 3));
  BATCH_TRY(sweep(&sigmo_batch_tuning::join_chunk, join_chunks, 4));
  b->tune = best_t;
  if (chosen) *chosen = best_t;
  if (best_ms) *best_ms = best;
  return SIGMO_OK;
}

int sigmo_batch_capture(sigmo_batch* b, const sigmo_graph* query, int find_first, int refresh_db) {
  if (!b || !query) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  int device = 0, cus = 0;
  hipStream_t s;
  unsigned long long *stats, *stats_host;
  BATCH_TRY(ctx_info(b->ctx, &device, &s, &cus, &stats, &stats_host));
  // a plain run first: it sizes the arena and the GMCR arrays and gives the pair counts
  sigmo_batch_result r;
  BATCH_TRY(sigmo_batch_run(b, query, find_first, &r));
  const uint64_t nw = stats_host[5];
  RunShape L;
  BATCH_TRY(shape_run(b, query, cus, L));
  if (!b->graph_host) BATCH_HIP_TRY(hipHostMalloc(reinterpret_cast<void**>(&b->graph_host), (kCounterWords + 16) * sizeof(unsigned long long)));
  b->drop_graph();
  const sigmo_db* db = b->db;
  BATCH_HIP_TRY(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  hipError_t e = hipSuccess;
  if (refresh_db)
    e = sigmo_k::db_prepare(s, L.dd, db->R, db->cls_list, db->order, db->planes, db->labs, db->dmax, db->minfo, db->cls, db->cmax);
  if (e == hipSuccess) e = sigmo_k::query_prepare(s, L.qd, L.R, b->tokens, b->qinfo, b->qmax, db->cls, b->qcmax);
  if (e == hipSuccess) e = launch_filter(b, L, s);
  if (e == hipSuccess) e = launch_count_scan(b, L, s);
  if (e == hipSuccess) e = launch_scatter(b, L, s);
  if (e == hipSuccess) e = sigmo_k::fill_u64(s, reinterpret_cast<uint64_t*>(stats), sigmo_k::kJoinStatWords, 0);
  // the joins read this replay's pair counts on the device (bounded by the captured sizes), so a
  // replay on changed data reads only entries the replay itself wrote
  if (e == hipSuccess) e = launch_join(b, L, s, stats, b->P, find_first, reinterpret_cast<const unsigned long long*>(b->total));
  if (e == hipSuccess) e = hipMemcpyAsync(b->graph_host, b->counters, kCounterWords * sizeof(unsigned long long), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipMemcpyAsync(b->graph_host + kCounterWords, b->total, sizeof(unsigned long long), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipMemcpyAsync(b->graph_host + kCounterWords + 1, stats, 8 * sizeof(unsigned long long), hipMemcpyDeviceToHost, s);
  hipGraph_t g = nullptr;
  const hipError_t end = hipStreamEndCapture(s, &g);
  if (e != hipSuccess || end != hipSuccess) {
    if (g) (void)hipGraphDestroy(g);
    return sigmo_err::set(SIGMO_ERR_HIP, std::string("graph capture: ") + hipGetErrorString(e != hipSuccess ? e : end));
  }
  b->graph = g;
  BATCH_HIP_TRY(hipGraphInstantiate(&b->graph_exec, g, nullptr, nullptr, 0));
  b->graph_P = b->P;
  b->graph_nw = nw;
  b->graph_Gq = L.Gq;
  b->graph_find_first = find_first;
  b->graph_db_generation = db->generation;
  return SIGMO_OK;
}

int sigmo_batch_replay(sigmo_batch* b, sigmo_batch_result* res) {
  if (!b || !res) return sigmo_err::set(SIGMO_ERR_INVALID, "null argument");
  if (!b->graph_exec)
    return sigmo_err::set(SIGMO_ERR_INVALID, "no captured graph (never captured, or a later run reallocated its buffers): capture again");
  if (b->db->generation != b->graph_db_generation)
    return sigmo_err::set(SIGMO_ERR_INVALID, "the database was rebound after the capture: capture again");
  int device = 0, cus = 0;
  hipStream_t s;
  unsigned long long *stats, *stats_host;
  BATCH_TRY(ctx_info(b->ctx, &device, &s, &cus, &stats, &stats_host));
  std::memset(res, 0, sizeof(*res));
  b->ran = false;  // the replay overwrites the result arrays
  void* tok = nullptr;
  BATCH_TRY(ctx_timed(b->ctx, SIGMO_PHASE_FILTER, -1, 0.0, true, &tok));  // the whole graph, as one timed region
  BATCH_HIP_TRY(hipGraphLaunch(b->graph_exec, s));
  BATCH_TRY(ctx_timed(b->ctx, 0, 0, 0.0, false, &tok));
  BATCH_HIP_TRY(hipStreamSynchronize(s));
  const unsigned long long* h = b->graph_host;
  const unsigned long long* js = h + kCounterWords + 1;  // join statistics
  if (h[3] || h[kCounterWords] != b->graph_P || (b->db->num_wide && js[5] != b->graph_nw)) {
    return sigmo_err::set(SIGMO_ERR_INVALID, "the captured graph no longer matches the data (arena or pair counts changed): capture again");
  }
  if (js[3]) return sigmo_err::set(SIGMO_ERR_OVERFLOW, "a per-pair match count exceeded int32");
  b->P = b->graph_P;
  b->Gq = b->graph_Gq;
  b->ran = true;
  res->num_matches = js[0];
  res->matched_pairs = js[1];
  res->gmcr_pairs = b->graph_P;
  res->dfs_steps = js[4];
  res->join_wave_steps = js[7];
  read_counters(0, h, res);
  return SIGMO_OK;
}

int sigmo_batch_pairs(sigmo_batch* b, uint32_t* data_graph_offsets, uint64_t n_offsets, uint32_t* query_graph_indices, int32_t* counts,
                      uint64_t n_pairs) {
  if (!b || !b->ran) return sigmo_err::set(SIGMO_ERR_INVALID, "batch has not run");
  int device = 0, cus = 0;
  hipStream_t s;
  unsigned long long *st, *sh;
  BATCH_TRY(ctx_info(b->ctx, &device, &s, &cus, &st, &sh));
  const uint64_t Gd = graph_dev(b->db->data).G;
  if (data_graph_offsets && n_offsets != Gd + 1) return sigmo_err::set(SIGMO_ERR_INVALID, "n_offsets must be Gd+1");
  if ((query_graph_indices || counts) && n_pairs != b->P) return sigmo_err::set(SIGMO_ERR_INVALID, "n_pairs must be the pair count");
  const sigmo_k::HostCopy out[3] = {{data_graph_offsets, b->offsets, data_graph_offsets ? n_offsets * 4 : 0},
                                    {query_graph_indices, b->indices, query_graph_indices ? n_pairs * 4 : 0},
                                    {counts, b->counts, counts ? n_pairs * 4 : 0}};
  BATCH_TRY(ctx_read_back(b->ctx, out, 3));
  return SIGMO_OK;
}

}  // extern "C"
