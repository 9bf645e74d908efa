// Closest-hit and any-hit traversal of one domain's 8-wide BVH.
//
// What bounds it: vector instructions (issued 70% of the time on a 64-domain
// 1024x1024 8 spp frame, two thirds of them in node visits), the address unit
// (60%: one lane a cycle and load) and, behind them, L2 misses.  So a visit
// reads 64 bytes in four loads, and what only leaves need lies elsewhere: one
// more dword load a visit costs 3%, and a node of 128 bytes in five loads took
// 16.07 ms where this takes 15.54 (256 uneven domains 10.5 -> 10.2, ambient
// occlusion 0.89 -> 0.86).
// Eight children against four: 20% fewer node visits, 32% fewer wave steps (a
// step keeps 68% of the lanes busy, 57% before, as a lane no longer stops at
// its second leaf).  Trace time of a pass, 4-wide -> 8-wide: 256x192 2 spp
// plain schedule 9.1 -> 7.8 ms, ambient occlusion 512x512 1.11 -> 1.03 ms, 256
// uneven domains 13.9 -> 13.5 ms, 64 even domains 17.4 -> 17.6 ms.  Tried on
// it and left out: choosing the nearest child by its entry distance (as many
// visits as in slot order, 3% slower); node lines fetched by four lanes each
// through LDS (5% slower); leaves of 3 or 4 triangles (3 and 5% slower); five
// waves a SIMD with half the LDS stack and triangles one at a time (a wash).
// Nodes of eight children on a grid of the node's own, slots by octant and
// groups of children on the stack are the method of Ylitie, Karras and Laine,
// "Efficient Incoherent Ray Traversal on GPUs Through Compressed Wide BVHs"
// (HPG 2017).
//
// Per-lane stack of node groups (a group: the children of one node that the
// ray has still to visit): the first kRing entries in LDS.  Each wave owns
// kRing x 64 entries of 8 bytes (entry e of lane l at (e * 64 + l) * 8 from
// the wave's base); entries past kRing go to a per-lane overflow stack in
// HBM.  A node leaves at most one group behind, so the tree's depth bounds
// the stack; the build rejects deeper trees.
#pragma once

#include "dmath.h"
#include "spray_internal.h"

namespace spray {

constexpr int kRing = 12;           // LDS entries, one of them the sentinel
constexpr int kOverflow = 40;       // HBM entries (2 words each)
constexpr int kOverflowWords = 2 * kOverflow;
constexpr int kStackMax = kRing - 1 + kOverflow;  // groups a traversal may hold
constexpr int kLeafList = 4;        // nodes with leaves to test that a lane may hold
constexpr uint32_t kStackEmpty = 0xffffffffu;
// Slack of the interval test (after Ize, "Robust BVH Ray Traversal", JCGT
// 2013): nodeBoxes' plane distances are within 2^-22 of exact, relatively
// (1/dir, base - org, their product and the fma round once each); the exit
// distance is inflated by 2^-20.
constexpr float kSlabInflate = 1.00000095367431640625f;
// A ray visits each node of a tree at most once, so it has as many visits as
// the tree has nodes (TravState::guard); that, and a bound on the steps of one
// node phase, stop a corrupt (cyclic) tree from spinning forever.
constexpr uint32_t kMaxPhaseSteps = 1u << 16;

// The ring pointer carries the LDS address space, so ring accesses stay
// ds_read/ds_write and are never merged with the overflow path into flat
// accesses.
typedef __attribute__((address_space(3))) uint32_t lds_u32;

// n counts the entries, the sentinel (an empty group) at the bottom included.
// A group is (the node's kids word, children left to visit by their visiting
// order in bits 0..7); only the sentinel has no children left.
struct LaneStack {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  typedef __attribute__((address_space(3))) u32x2 lds_u2;
  lds_u2* lane;        // this lane's entry 0 (entries 64 apart)
  lds_u32* list;       // this lane's leaf list (entries 64 words apart)
  uint32_t* ovf;       // overflow areas of the grid (`words` per thread)
  uint32_t words;
  uint32_t n;
  bool err;
  // area: the wave's LDS (kTravLdsWords)
  __device__ void init(uint32_t* area, uint32_t* ovf_base, uint32_t ovf_words = kOverflowWords) {
    lane = (lds_u2*)area + (threadIdx.x & 63);
    list = (lds_u32*)area + kRing * 128 + (threadIdx.x & 63);
    ovf = ovf_base;
    words = ovf_words;
    lane[0] = u32x2{0u, 0u};
    n = 1;
    err = false;
  }
  __device__ void reset() {
    lane[0] = u32x2{0u, 0u};
    n = 1;
  }
  __device__ bool overflowed() const { return err; }
  __device__ uint32_t* spilled(uint32_t e) const {  // only on the rare spill path
    return ovf + (blockIdx.x * (size_t)blockDim.x + threadIdx.x) * words + 2 * (e - kRing);
  }
  __device__ u32x2 get(uint32_t e) const {
    if (e < (uint32_t)kRing) return lane[e << 6];
    const uint32_t* p = spilled(e);
    return u32x2{p[0], p[1]};
  }
  __device__ bool put(uint32_t e, u32x2 g) {  // false: no room
    if (e < (uint32_t)kRing) {
      lane[e << 6] = g;
    } else if (e < (uint32_t)kRing + words / 2u) {
      uint32_t* p = spilled(e);
      p[0] = g.x;
      p[1] = g.y;
    } else {
      err = true;  // reported to the host; never silently dropped
      return false;
    }
    return true;
  }
};

// Work counters: node steps per wave (a sum of ballots, kept in scalar
// registers) and triangle tests per lane.
struct TravCount {
  unsigned long long nodes = 0;
  uint32_t tris = 0;
};

// Largest |1/dir| of the fused box test: a plane's 255 * scale * inv stays
// below 2^126 (quantizeNode keeps scale below 2^62), so where the other term
// overflows, it alone decides.
constexpr float kFusedInvMax = 1.4411518807585587e17f;  // 2^57
__device__ __forceinline__ bool needsSafeBoxes(const float inv[3]) {
  return !(fabsf(inv[0]) < kFusedInvMax && fabsf(inv[1]) < kFusedInvMax && fabsf(inv[2]) < kFusedInvMax);
}

// The bits of a where m is set, those of b elsewhere.
__device__ __forceinline__ uint32_t pickBits(uint32_t m, uint32_t a, uint32_t b) {
  return __builtin_amdgcn_bitop3_b32(m, a, b, 0xca);
}

// Tests the 8 child boxes of a node against [tnear, tfar]; returns the mask of
// the slots hit.  The distance of plane q is
//   (base + q * scale - org) * inv = fma(q, scale * inv, (base - org) * inv)
// where scale * inv is exact.  Its error is relative to t plus, where the two
// terms cancel, at most 2^-15 of a plane step: the boxes are at least 2^-9 of
// a step too large (quantizeNode), so no box the ray meets is missed, and no
// absolute pad is needed.  A ray's near planes are the lower ones where inv
// >= 0 and the upper ones elsewhere, one select per axis for four children.
// fma, add, mul and the three-operand bit operation issue in 2 cycles a wave,
// byte conversions, min, max, compares, selects and shifts in 4: so planes are
// picked by bits and a miss is a sign bit shifted in (1% of the trace time
// against selects, compares and carries).
// kSafe (travNodePhase chooses it by the wave): the difference first, then the
// product with a possibly infinite inv; 0 * inf = NaN (the origin on the
// plane) bounds nothing, as max and min drop NaN operands.  An axis that
// covers everything has a base that is not a number.  It is also the form for
// intervals that begin behind the origin: an exit distance below zero is
// inflated towards zero there, where kSlabInflate would move it away from it
// (3000 triangles of 0.002 that lie 1000 behind the origins: 271 of 20,000 rays
// answered wrongly; nearly all where the triangles lie in one plane).
template <bool kSafe>
__device__ __forceinline__ uint32_t nodeBoxes(const uint4& w0, const uint4 (&pl)[3], const float org[3],
                                              const float inv[3], float tnear, float tfar) {
  const float bo[3] = {__uint_as_float(w0.x) - org[0], __uint_as_float(w0.y) - org[1],
                       __uint_as_float(w0.z) - org[2]};
  const uint32_t wb[3] = {w0.x, w0.y, w0.z};
  uint32_t nq[3][2], fq[3][2];
  float m[3], c[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float scale = __uint_as_float((wb[k] << 23) & 0x7f800000u);
    const uint32_t neg = (uint32_t)((int32_t)__float_as_uint(inv[k]) >> 31);
    nq[k][0] = pickBits(neg, pl[k].z, pl[k].x);
    nq[k][1] = pickBits(neg, pl[k].w, pl[k].y);
    fq[k][0] = pickBits(neg, pl[k].x, pl[k].z);
    fq[k][1] = pickBits(neg, pl[k].y, pl[k].w);
    m[k] = kSafe ? scale : scale * inv[k];
    c[k] = kSafe ? bo[k] : bo[k] * inv[k];
  }
  uint32_t miss = 0;
#pragma unroll
  for (int i = 7; i >= 0; --i) {
    float tn[3], tf[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float qn = (float)((nq[k][i >> 2] >> (8 * (i & 3))) & 255u);
      const float qf = (float)((fq[k][i >> 2] >> (8 * (i & 3))) & 255u);
      tn[k] = __builtin_fmaf(qn, m[k], c[k]);
      tf[k] = __builtin_fmaf(qf, m[k], c[k]);
      if (kSafe) {
        tn[k] *= inv[k];
        tf[k] *= inv[k];
      }
    }
    const float t0 = fmaxf(fmaxf(fmaxf(tn[0], tn[1]), tn[2]), tnear);
    const float t1 = fminf(fminf(fminf(tf[0], tf[1]), tf[2]), tfar);
    // a miss is the sign of the inflated t1 - t0, shifted in
    const float d = kSafe ? __builtin_fmaf(fabsf(t1), kSlabInflate - 1.0f, t1) - t0
                          : __builtin_fmaf(t1, kSlabInflate, -t0);
    miss = __builtin_amdgcn_alignbit(miss, __float_as_uint(d), 31u);
  }
  return ~miss & 255u;
}

// Resumable traversal of one ray (closest or any hit) in two wave-wide
// phases (after Aila & Laine 2009, "while-while" with speculative traversal):
// in the node phase every lane visits nodes; leaves met on the way are noted
// in the lane's leaf list, and the lane goes on.  In the leaf phase the wave
// tests all noted leaves together.
//
// Closest hit: `tlim` is the best t so far (initially the ray's tfar, which
// is therefore also the reported t of a miss); an exact tie in t goes to the
// lower primitive id.  Any hit: `tlim` stays tfar and prim becomes 1.
struct TravState {
  float org[3], inv[3];
  float Sx, Sy, Sz;
  uint32_t kk;          // kx | ky << 2 | kz << 4 | any << 8 | negative directions << 16
  float tnear, tlim, u, v;
  int prim;
  uint32_t cur;         // node to visit (kStackEmpty: none)
  int guard;            // visits left: a lane's own, not the steps it waits through
  uint32_t listed;      // leaf list: entries | leaves << 8
  uint32_t share;       // lane that owns the ray | lowest stack entry not given away << 8
  uint32_t node_base, tri_base;  // the domain's first node / leaf-ordered triangle
};

__device__ __forceinline__ void travInit(TravState& s, uint32_t node_base, uint32_t tri_base, int num_nodes,
                                         const float org[3], const float dir[3], float tnear,
                                         float tfar, bool any, LaneStack& st) {
  s.org[0] = org[0];
  s.org[1] = org[1];
  s.org[2] = org[2];
  s.inv[0] = 1.0f / dir[0];
  s.inv[1] = 1.0f / dir[1];
  s.inv[2] = 1.0f / dir[2];
  RayPre rp = rayPre(dir);
  s.Sx = rp.Sx;
  s.Sy = rp.Sy;
  s.Sz = rp.Sz;
  s.kk = (uint32_t)rp.kx | ((uint32_t)rp.ky << 2) | ((uint32_t)rp.kz << 4) | (any ? 256u : 0u) |
         (s.inv[0] < 0.f ? 1u << 16 : 0u) | (s.inv[1] < 0.f ? 2u << 16 : 0u) | (s.inv[2] < 0.f ? 4u << 16 : 0u);
  s.tnear = tnear;
  s.tlim = tfar;
  s.u = s.v = 0.f;
  s.prim = -1;
  s.cur = 0;
  s.listed = 0;
  s.share = (threadIdx.x & 63u) | (1u << 8);
  s.guard = num_nodes;
  s.node_base = node_base;
  s.tri_base = tri_base;
  st.reset();
}

__device__ __forceinline__ bool travDone(const TravState& s) {
  return s.cur == kStackEmpty && s.listed == 0u;
}

// Bit i of the result is bit i ^ o of m (8 bits).
__device__ __forceinline__ uint32_t permuteSlots(uint32_t m, uint32_t o) {
  m = (o & 1u) ? ((m >> 1) & 0x55u) | ((m & 0x55u) << 1) : m;
  m = (o & 2u) ? ((m >> 2) & 0x33u) | ((m & 0x33u) << 2) : m;
  return (o & 4u) ? (m >> 4) | ((m & 0x0fu) << 4) : m;
}

// The child in `slot` of a node with this kids word.
__device__ __forceinline__ uint32_t groupChild(uint32_t kids, uint32_t slot) {
  return (kids & 0xffffffu) + (uint32_t)__popc(__builtin_amdgcn_ubfe(kids, 24u, slot));
}

// One node: leaves that the ray hits are listed, the inner children become a
// group, and `cur` the first child of that group, or of the group on top of
// the stack when there is none.  The top group is read beside the node, so
// the common path has no branch and no pop that waits for LDS.
template <bool kSafe>
__device__ __forceinline__ void travNode(TravState& s, LaneStack& st,
                                         const BNode8* __restrict__ nodes) {
  typedef LaneStack::u32x2 u32x2;
  const BNode8* nd = &nodes[s.node_base + s.cur];
  const uint4 w0 = ((const uint4*)nd)[0];
  const uint4 pl[3] = {((const uint4*)nd)[1], ((const uint4*)nd)[2], ((const uint4*)nd)[3]};
  const bool fast = st.n < (uint32_t)kRing;
  u32x2 top = st.lane[(min(st.n, (uint32_t)kRing) - 1u) << 6];
  if (!fast) top = st.get(st.n - 1u);
  const uint32_t mask = nodeBoxes<kSafe>(w0, pl, s.org, s.inv, s.tnear, s.tlim);
  const uint32_t im = w0.w >> 24, leaves = mask & ~im;
  st.list[(s.listed & 255u) << 6] = (s.cur << 8) | leaves;  // kept when it has leaves
  s.listed += leaves ? 1u + ((uint32_t)__popc(leaves) << 8) : 0u;
  const uint32_t oct = (s.kk >> 16) & 7u;
  const uint32_t pm = permuteSlots(mask & im, oct);
  const bool down = pm != 0u;
  const uint32_t gb = down ? w0.w : top.x, gm = down ? pm : top.y;
  const uint32_t slot = ((uint32_t)__ffs((int)gm) - 1u) ^ oct;
  // the inner children below `slot` come before it
  const uint32_t child = groupChild(gb, slot);
  uint32_t rest = gm & (gm - 1u);
  const uint32_t at = down ? st.n : st.n - 1u;
  if (at < (uint32_t)kRing)
    st.lane[at << 6] = u32x2{gb, rest};
  else if (!st.put(at, u32x2{gb, rest}))
    rest = 0u;
  st.n = at + (rest ? 1u : 0u);
  s.cur = gm ? child : kStackEmpty;
}

// Node phase over the wave: lanes visit nodes until three quarters of the
// wave's rays have leaves to test, or fewer than half have a node to visit.
// (1024x1024, 8 spp, 64 domains, trace time of a frame: 16.3 ms; leaving at
// half or all of the rays with leaves 16.5 and 16.7; at a third or three
// quarters of the rays still stepping 17.3 and 16.7.)
template <bool kSafe>
__device__ __forceinline__ void travNodeLoop(TravState& s, LaneStack& st, TravCount& cnt,
                                             bool active, const BNode8* __restrict__ nodes) {
  auto steps_on = [&] {
    return active && s.cur != kStackEmpty && (s.listed & 255u) < (uint32_t)kLeafList;
  };
  const int nlive = __popcll(__ballot(active));
  unsigned long long sm = __ballot(steps_on());
  uint32_t steps = 0;
  while (sm != 0ull) {
    cnt.nodes += (unsigned long long)__popcll(sm);
    if (steps_on()) {
      travNode<kSafe>(s, st, nodes);
      --s.guard;
    }
    sm = __ballot(steps_on());
    const int nleaf = __popcll(__ballot(active && s.listed != 0u));
    ++steps;
    if (__popcll(sm) * 2 < nlive || nleaf * 4 >= nlive * 3 || steps >= kMaxPhaseSteps) break;
  }
  if (active && s.guard < 0) {
    st.err = true;
    s.cur = kStackEmpty;
    s.listed = 0;
  }
}

// The safe box tests only in waves with an axis-parallel (or nearly so) ray, or
// one that looks behind its origin: two copies of the loop, so that the common
// one carries no handling of them.
__device__ __forceinline__ void travNodePhase(TravState& s, LaneStack& st, TravCount& cnt,
                                              bool active, const BNode8* __restrict__ nodes) {
  if (__ballot(active && (needsSafeBoxes(s.inv) || s.tnear < 0.f)) != 0ull)
    travNodeLoop<true>(s, st, cnt, active, nodes);
  else
    travNodeLoop<false>(s, st, cnt, active, nodes);
}

// Leaf phase over the wave.  Lanes hold different numbers of leaves, so the
// wave's leaves are pooled: every lane lists its leaves in LDS, and the wave
// tests 64 of the list at a time, each lane one leaf of whichever ray owns it
// (the owner's ray comes by lane permutes; travShare: a ray's owner is not
// always the lane that met the leaf).  A hit goes to its owner by a
// minimum over (t, primitive id), the order that testing one triangle after
// another keeps.
constexpr int kLeafItems = 192;  // leaves listed at once
// per wave: stack, leaf lists, pooled leaves, hit keys, hit records
constexpr int kTravLdsWords = kRing * 128 + kLeafList * 64 + kLeafItems + 64 * 2 + 64 * 4;
static_assert(kLeafMax <= 2, "a leaf's triangles are loaded together");
static_assert(kLeafItems >= 8 * kLeafList, "a lane's leaves fit the list");
static_assert(kLeafItems >= 64 * 3, "travShare's slots");

// Sum of n (below 64) over the lanes before this one, and over the wave.
__device__ __forceinline__ uint32_t rankSmall(uint32_t n, uint32_t* total) {
  const unsigned long long lt = (1ull << __lane_id()) - 1ull;
  uint32_t r = 0, sum = 0;
#pragma unroll
  for (int b = 0; b < 6; ++b) {
    const unsigned long long m = __ballot((n >> b) & 1u);
    r += (uint32_t)__popcll(m & lt) << b;
    sum += (uint32_t)__popcll(m) << b;
  }
  *total = sum;
  return r;
}
__device__ __forceinline__ void ldsWaveSync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ uint32_t laneGet(uint32_t v, int src) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)v);
}
__device__ __forceinline__ float laneGetF(float v, int src) {
  return __uint_as_float(laneGet(__float_as_uint(v), src));
}
__device__ __forceinline__ uint32_t orderedT(float t) {  // monotone bits; -0 as +0
  const uint32_t u = __float_as_uint(t + 0.f);
  return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}

// Every lane of the wave calls it, converged (area: the wave's LDS).
__device__ __forceinline__ void travLeafPhase(TravState& s, LaneStack& st, TravCount& cnt,
                                              bool active, const NodeLeaves* __restrict__ leaves,
                                              const LTri* __restrict__ tris, uint32_t* area) {
  typedef __attribute__((address_space(3))) unsigned long long lds_u64;
  typedef __attribute__((address_space(3))) float lds_f;
  lds_u32* items = (lds_u32*)area + kRing * 128 + kLeafList * 64;
  lds_u64* keys = (lds_u64*)(items + kLeafItems);
  lds_f* recs = (lds_f*)(items + kLeafItems + 128);
  const int lane = __lane_id();
  const uint32_t entries = active ? s.listed & 255u : 0u, n = active ? s.listed >> 8 : 0u;
  uint32_t total;
  const uint32_t rank = rankSmall(n, &total);
  if (total == 0u) return;
  // lanes past the list's end keep their leaves for the next turn
  const bool take = n > 0u && rank + n <= (uint32_t)kLeafItems;
  if (take) {
    uint32_t at = rank;
    for (uint32_t e = 0; e < entries; ++e) {
      const uint32_t w = st.list[e << 6];
      const uint32_t item = ((s.share & 63u) << 26) | ((w >> 8) << 3);
      for (uint32_t m = w & 255u; m != 0u; m &= m - 1u) items[at++] = item | ((uint32_t)__ffs((int)m) - 1u);
    }
    s.listed = 0;
  }
  const unsigned long long tm = __ballot(take);
  const uint32_t count = __builtin_amdgcn_readlane(rank + n, 63 - __builtin_clzll(tm));
  keys[lane] = ~0ull;
  const bool any = (s.kk >> 8) & 1u;
  // closest: t <= tlim counts once a hit exists (ties go to the lower id), so
  // the bound is the next float above tlim
  const uint32_t lim_u = __float_as_uint(s.tlim + 0.f);
  const float ub = (any || s.prim < 0) ? s.tlim : __uint_as_float(lim_u + (uint32_t)((int32_t)lim_u >> 31 | 1));
  ldsWaveSync();
  for (uint32_t base = 0; base < count; base += 64u) {
    const bool in = base + (uint32_t)lane < count;
    const uint32_t it = in ? items[base + lane] : (uint32_t)lane << 26;
    const int own = (int)(it >> 26);
    const uint32_t nb = laneGet(s.node_base, own), tb = laneGet(s.tri_base, own);
    const uint32_t word = in ? leaves[nb + ((it >> 3) & 0x7fffffu)].leaf[it & 7u] : 0u;
    const uint32_t kk = laneGet(s.kk, own);
    const RayPre rp{(int)(kk & 3u), (int)((kk >> 2) & 3u), (int)((kk >> 4) & 3u),
                    laneGetF(s.Sx, own), laneGetF(s.Sy, own), laneGetF(s.Sz, own)};
    const float org[3] = {laneGetF(s.org[0], own), laneGetF(s.org[1], own), laneGetF(s.org[2], own)};
    const float tn = laneGetF(s.tnear, own);
    float lim = laneGetF(ub, own);
    const uint32_t ntri = (word >> 24) & 0x7fu;
    cnt.tris += ntri;
    const float4* tq = (const float4*)&tris[tb + (word & 0x00ffffffu)];
    float4 a[2], b[2], c[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if ((uint32_t)j < ntri) {
        a[j] = tq[3 * j];
        b[j] = tq[3 * j + 1];
        c[j] = tq[3 * j + 2];
      }
    float t = 0.f, u = 0.f, v = 0.f;
    int p = 0;
    bool hit = false;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if ((uint32_t)j < ntri) {
        const float v0[3] = {a[j].x, a[j].y, a[j].z}, v1[3] = {b[j].x, b[j].y, b[j].z},
                    v2[3] = {c[j].x, c[j].y, c[j].z};
        const int q = __float_as_int(a[j].w);
        float t1, u1, w1;
        if (triHit(rp, org, v0, v1, v2, tn, lim, &t1, &u1, &w1) && (!hit || t1 < t || (t1 == t && q < p))) {
          t = t1;
          u = u1;
          v = w1;
          p = q;
          hit = true;
        }
      }
    if (__ballot(hit) == 0ull) continue;
    const unsigned long long key = ((unsigned long long)orderedT(t) << 32) | (uint32_t)p;
    if (hit) (void)__hip_atomic_fetch_min(&keys[own], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    ldsWaveSync();
    if (hit && keys[own] == key) {
      recs[own] = t;
      recs[64 + own] = u;
      recs[128 + own] = v;
      recs[192 + own] = __int_as_float(p);
    }
  }
  ldsWaveSync();
  if (keys[lane] != ~0ull) {
    const float t = recs[lane];
    const int p = __float_as_int(recs[192 + lane]);
    if (any) {
      s.prim = 1;
      s.cur = kStackEmpty;
      s.listed = 0;
    } else if (s.prim < 0 || t < s.tlim || p < s.prim) {
      s.tlim = t;
      s.u = recs[64 + lane];
      s.v = recs[128 + lane];
      s.prim = p;
    }
  }
  ldsWaveSync();
}

// Idle lanes take over part of a busy lane's ray: the lowest (largest and
// farthest) group of its stack, which becomes the busy lane's new sentinel.
// A helper traverses with a copy of the ray; its leaves are listed for the
// ray's owner, which receives the hits, so the result is the owner's minimum
// over (t, primitive id) whoever meets the triangle.  Where a launch has few
// rays, or at its end, this shortens the longest ray's chain of dependent
// node visits, which the launch otherwise waits for.  Trace time of a pass:
// 96x72 preview 200 -> 173 us, plain schedule 7.3 -> 5.4 ms, in-situ frame 3.4
// -> 2.0 ms, 48 domains with 12 cached 6.4 -> 4.3 ms, 256 uneven domains
// 1279x719 8 spp 12.6 -> 10.4 ms (20 launches, each with such an end), 64 even
// domains 1024x1024 8 spp 16.9 -> 16.1 ms.  Every lane of the wave
// calls it, converged; idle: has no ray; live: traverses one.  Returns
// whether this lane became a helper.
__device__ __forceinline__ bool travShare(TravState& s, LaneStack& st, bool idle, bool live,
                                          uint32_t* area) {
  typedef LaneStack::u32x2 u32x2;
  lds_u32* slots = (lds_u32*)area + kRing * 128 + kLeafList * 64;  // the pooled leaves' place
  const uint32_t bot = s.share >> 8;
  const bool donor = live && st.n > bot && bot < (uint32_t)kRing;
  const unsigned long long dm = __ballot(donor), im = __ballot(idle);
  const int k = min(__popcll(dm), __popcll(im));
  if (k == 0) return false;
  const unsigned long long lt = (1ull << __lane_id()) - 1ull;
  const int dr = __popcll(dm & lt), ir = __popcll(im & lt);
  ldsWaveSync();
  if (donor && dr < k) {
    const u32x2 g = st.lane[bot << 6];
    st.lane[bot << 6] = u32x2{0u, 0u};
    s.share += 1u << 8;
    slots[dr] = s.share & 63u;
    slots[64 + dr] = g.x;
    slots[128 + dr] = g.y;
  }
  ldsWaveSync();
  const bool take = idle && ir < k;
  const int own = take ? (int)slots[ir] : __lane_id();
  const uint32_t gb = take ? slots[64 + ir] : 0u, gm = take ? slots[128 + ir] : 0u;
  const float o0 = laneGetF(s.org[0], own), o1 = laneGetF(s.org[1], own), o2 = laneGetF(s.org[2], own);
  const float i0 = laneGetF(s.inv[0], own), i1 = laneGetF(s.inv[1], own), i2 = laneGetF(s.inv[2], own);
  const float tn = laneGetF(s.tnear, own), tl = laneGetF(s.tlim, own);
  const uint32_t kk = laneGet(s.kk, own), nb = laneGet(s.node_base, own);
  const int left = (int)laneGet((uint32_t)s.guard, own);  // (owner and helper visit different nodes)
  if (take) {
    s.org[0] = o0;
    s.org[1] = o1;
    s.org[2] = o2;
    s.inv[0] = i0;
    s.inv[1] = i1;
    s.inv[2] = i2;
    s.tnear = tn;
    s.tlim = tl;
    s.kk = kk;
    s.node_base = nb;
    s.listed = 0;
    s.guard = left;
    s.share = (uint32_t)own | (1u << 8);
    const uint32_t slot = ((uint32_t)__ffs((int)gm) - 1u) ^ ((kk >> 16) & 7u);
    s.cur = groupChild(gb, slot);
    const uint32_t rest = gm & (gm - 1u);
    st.lane[0] = u32x2{0u, 0u};
    st.lane[64] = u32x2{gb, rest};
    st.n = rest ? 2u : 1u;
  }
  ldsWaveSync();
  return take;
}

// Helpers take their ray's current limit from its owner, and stop when an
// any-hit query is answered.  Every lane of the wave calls it, converged.
__device__ __forceinline__ void travFollow(TravState& s, bool helping) {
  const int own = (int)(s.share & 63u);
  const float tl = laneGetF(s.tlim, own);
  const uint32_t pr = laneGet((uint32_t)s.prim, own);
  if (helping) {
    s.tlim = tl;
    if (((s.kk >> 8) & 1u) && (int)pr > 0) {
      s.cur = kStackEmpty;
      s.listed = 0;
    }
  }
}

// Whether some live helper works on this lane's ray.  Every lane of the wave
// calls it, converged.
__device__ __forceinline__ bool travHelped(const TravState& s, bool helping, uint32_t* area) {
  lds_u32* flags = (lds_u32*)area + kRing * 128 + kLeafList * 64;
  ldsWaveSync();
  flags[__lane_id()] = 0u;
  ldsWaveSync();
  if (helping) flags[s.share & 63u] = 1u;
  ldsWaveSync();
  const bool r = flags[__lane_id()] != 0u;
  ldsWaveSync();
  return r;
}

}  // namespace spray
