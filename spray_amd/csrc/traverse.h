// Closest-hit and any-hit traversal of one domain's 4-wide BVH.
//
// Per-lane short stack: a 16-entry ring in LDS.  Each wave owns kRing x 64
// words (slot s of lane l of wave w at lds[(w * kRing + s) * 64 + l], so a
// wave's pushes hit 64 consecutive banks and the address needs no block
// size);
// when the ring is full its bottom entry spills to a per-lane overflow
// stack in HBM, which is popped only once the ring is empty.  The overflow
// depth bounds the BVH depth; the build rejects deeper trees.
#pragma once

#include "dmath.h"
#include "spray_internal.h"

namespace spray {

constexpr int kRing = 16;
constexpr int kOverflow = 112;
constexpr uint32_t kStackEmpty = 0xffffffffu;
// Slack of the interval test (after Ize, "Robust BVH Ray Traversal", JCGT
// 2013): nodeBoxes' plane distances are within 2^-22 of exact, relatively
// (1/dir, base - org, their product and the fma round once each); the exit
// distance is inflated by 2^-20.
constexpr float kSlabInflate = 1.00000095367431640625f;
// a ray visits each node of a tree at most once; the bound only stops a
// corrupt (cyclic) tree from spinning forever
constexpr uint32_t kMaxNodeVisits = 1u << 22;

// The stack state is one packed word per lane: ring head (bits 0-3), ring
// fill (4-8), overflow fill (9-15), overflow error (16).  The ring pointer
// carries the LDS address space, so ring accesses stay ds_read/ds_write and
// are never merged with the overflow path into flat accesses.
typedef __attribute__((address_space(3))) uint32_t lds_u32;

struct LaneStack {
  lds_u32* lds;        // this block's ring base
  uint32_t* ovf;       // overflow areas of the grid (kOverflow words per thread)
  uint32_t w;
  __device__ void init(uint32_t* lds_base, uint32_t* ovf_base) {
    lds = (lds_u32*)lds_base;
    ovf = ovf_base;
    w = 0;
  }
  __device__ void reset() { w &= 1u << 16; }
  __device__ bool overflowed() const { return (w >> 16) & 1u; }
  __device__ uint32_t count() const { return (w >> 4) & 31u; }
  __device__ uint32_t* lane_ovf() const {  // only on the rare spill path
    return ovf + (blockIdx.x * (size_t)blockDim.x + threadIdx.x) * kOverflow;
  }
  __device__ lds_u32& slot(uint32_t s) const {
    return lds[(((threadIdx.x >> 6) * kRing + (s & (kRing - 1))) << 6) + (threadIdx.x & 63)];
  }
  __device__ void push(uint32_t x) {
    uint32_t head = w & 15u, count = (w >> 4) & 31u, spilled = (w >> 9) & 127u, err = w >> 16;
    if (count == kRing) {
      uint32_t bottom = slot(head);
      if (spilled < kOverflow)
        lane_ovf()[spilled++] = bottom;
      else
        err = 1;  // reported to the host; never silently dropped
      head = (head + 1) & (kRing - 1);
      --count;
    }
    slot(head + count) = x;
    ++count;
    w = head | (count << 4) | (spilled << 9) | (err << 16);
  }
  // Pushes the first n (<= 3) of x0, x1, x2 (x0 deepest).  With room for
  // three entries all three slots above the top are written (the unused
  // ones hold nothing live), so the common case has no branch; a nearly
  // full ring takes the spilling path.
  __device__ void push3(uint32_t x0, uint32_t x1, uint32_t x2, uint32_t n) {
    uint32_t head = w & 15u, count = (w >> 4) & 31u;
    if (count + 3u <= (uint32_t)kRing) {
      slot(head + count) = x0;
      slot(head + count + 1u) = x1;
      slot(head + count + 2u) = x2;
      w += n << 4;
    } else {
      if (n >= 1u) push(x0);
      if (n >= 2u) push(x1);
      if (n >= 3u) push(x2);
    }
  }
  __device__ uint32_t pop() {
    uint32_t head = w & 15u, count = (w >> 4) & 31u, spilled = (w >> 9) & 127u;
    if (count > 0) {
      w -= 1u << 4;
      return slot(head + count - 1u);
    }
    if (spilled > 0) {
      --spilled;
      w = (w & ~(127u << 9)) | (spilled << 9);
      return lane_ovf()[spilled];
    }
    return kStackEmpty;
  }
};

// Work counters: node steps per wave (a sum of ballots, kept in scalar
// registers) and triangle tests per lane.
struct TravCount {
  unsigned long long nodes = 0;
  uint32_t tris = 0;
};

// Largest |1/dir| of the fused box test: beyond it scale * inv could
// overflow (quantizeNode keeps scale below 2^62).
constexpr float kFusedInvMax = 1.8446744073709552e19f;  // 2^64
__device__ __forceinline__ bool needsSafeBoxes(const float inv[3]) {
  return !(fabsf(inv[0]) < kFusedInvMax && fabsf(inv[1]) < kFusedInvMax && fabsf(inv[2]) < kFusedInvMax);
}

// Tests the 4 child boxes of a node against [tnear, tfar]; returns a 4-bit
// hit mask and the entry distances.  The distance of plane q is
//   (base + q * scale - org) * inv = fma(q, scale * inv, (base - org) * inv)
// where scale * inv is exact.  Its error is relative to t plus, where the two
// terms cancel, at most 2^-15 of a plane step: the boxes are at least 2^-9 of
// a step too large (quantizeNode), so no box the ray meets is missed, and no
// absolute pad is needed.  A ray's near planes are the lower ones where inv
// >= 0 and the upper ones elsewhere, one select per axis for all four
// children.  kSafe (waves with an axis-parallel ray): the difference first,
// then the product with a possibly infinite inv; 0 * inf = NaN (the origin on
// the plane) bounds nothing, as max and min drop NaN operands.
template <bool kSafe>
__device__ __forceinline__ int nodeBoxes(const BNode4* __restrict__ nd, const float org[3],
                                         const float inv[3], float tnear, float tfar,
                                         float tmin_o[4], int child_o[4]) {
  const float4* q = (const float4*)nd;
  const float4 w0 = q[0];
  const uint4 w1 = ((const uint4*)nd)[1], w2 = ((const uint4*)nd)[2];
  const int4 ch = ((const int4*)nd)[3];
  child_o[0] = ch.x;
  child_o[1] = ch.y;
  child_o[2] = ch.z;
  child_o[3] = ch.w;
  const float bo[3] = {w0.x - org[0], w0.y - org[1], w0.z - org[2]};
  const float sc[3] = {w0.w, __uint_as_float(w1.x), __uint_as_float(w1.y)};
  const uint32_t lo[3] = {w1.z, w2.x, w2.z}, hi[3] = {w1.w, w2.y, w2.w};
  uint32_t nq[3], fq[3];
  float m[3], c[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const bool neg = inv[k] < 0.f;
    nq[k] = neg ? hi[k] : lo[k];
    fq[k] = neg ? lo[k] : hi[k];
    m[k] = kSafe ? sc[k] : sc[k] * inv[k];
    c[k] = kSafe ? bo[k] : bo[k] * inv[k];
  }
  int mask = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float tn[3], tf[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float qn = (float)((nq[k] >> (8 * i)) & 255u), qf = (float)((fq[k] >> (8 * i)) & 255u);
      tn[k] = __builtin_fmaf(qn, m[k], c[k]);
      tf[k] = __builtin_fmaf(qf, m[k], c[k]);
      if (kSafe) {
        tn[k] *= inv[k];
        tf[k] *= inv[k];
      }
    }
    const float t0 = fmaxf(fmaxf(fmaxf(tn[0], tn[1]), tn[2]), tnear);
    const float t1 = fminf(fminf(fminf(tf[0], tf[1]), tf[2]), tfar) * kSlabInflate;
    tmin_o[i] = t0;
    if (t0 <= t1) mask |= 1 << i;
  }
  return mask;
}

// Resumable traversal of one ray (closest or any hit) in two wave-wide
// phases (Aila & Laine 2009, "while-while" with speculative traversal):
// in the node phase every lane descends inner nodes; a lane that reaches a
// leaf postpones it (one slot, `pend`) and keeps descending while other
// lanes of its wave have not found a leaf yet.  In the leaf phase every lane
// tests its postponed leaf and then the leaves at the top of its stack.
// Node refs and leaf refs share the stack: a leaf ref is the child word of
// its parent (bit 31, count << 24, first triangle).
//
// Closest hit: `tlim` is the best t so far (initially the ray's tfar, which
// is therefore also the reported t of a miss); an exact tie in t goes to the
// lower primitive id.  Any hit: `tlim` stays tfar and prim becomes 1.
struct TravState {
  float org[3], inv[3];
  float Sx, Sy, Sz;
  uint32_t kk;          // kx | ky << 2 | kz << 4 | any << 8
  float tnear, tlim, u, v;
  int prim;
  uint32_t cur, pend, guard;
  uint32_t node_base, tri_base;  // the domain's first node / leaf-ordered triangle
};

__device__ __forceinline__ bool isInnerRef(uint32_t r) { return (int32_t)r >= 0; }
__device__ __forceinline__ bool isLeafRef(uint32_t r) { return (int32_t)r < 0 && r != kStackEmpty; }

__device__ __forceinline__ void travInit(TravState& s, uint32_t node_base, uint32_t tri_base,
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
  s.kk = (uint32_t)rp.kx | ((uint32_t)rp.ky << 2) | ((uint32_t)rp.kz << 4) | (any ? 256u : 0u);
  s.tnear = tnear;
  s.tlim = tfar;
  s.u = s.v = 0.f;
  s.prim = -1;
  s.cur = 0;
  s.pend = kStackEmpty;
  s.guard = 0;
  s.node_base = node_base;
  s.tri_base = tri_base;
  st.reset();
}

__device__ __forceinline__ bool travDone(const TravState& s) {
  return s.cur == kStackEmpty && s.pend == kStackEmpty;
}

__device__ __forceinline__ void cswap(float& ka, int& ia, float& kb, int& ib) {
  bool sw = kb < ka;
  float tk = sw ? kb : ka;
  int ti = sw ? ib : ia;
  kb = sw ? ka : kb;
  ib = sw ? ia : ib;
  ka = tk;
  ia = ti;
}

// One inner node: the hit children (inner nodes and leaves) in order of
// entry distance; the nearest becomes `cur`, the others are pushed.
template <bool kSafe>
__device__ __forceinline__ void travNode(TravState& s, LaneStack& st,
                                         const BNode4* __restrict__ nodes) {
  if (++s.guard > kMaxNodeVisits) {
    st.w |= 1u << 16;
    s.cur = s.pend = kStackEmpty;
    return;
  }
  float tmin[4];
  int child[4];
  const BNode4* nd = &nodes[s.node_base + s.cur];
  int mask = nodeBoxes<kSafe>(nd, s.org, s.inv, s.tnear, s.tlim, tmin, child);
  float ks[4];
  int m = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    bool ok = (mask >> i) & 1;
    ks[i] = ok ? fminf(tmin[i], 3.0e38f) : kInfF;
    m += ok ? 1 : 0;
  }
  float k0 = ks[0], k1 = ks[1], k2 = ks[2], k3 = ks[3];
  int i0 = child[0], i1 = child[1], i2 = child[2], i3 = child[3];
  cswap(k0, i0, k1, i1);
  cswap(k2, i2, k3, i3);
  cswap(k0, i0, k2, i2);
  cswap(k1, i1, k3, i3);
  cswap(k1, i1, k2, i2);
  if (m == 0) {
    s.cur = st.pop();
    return;
  }
  // farther children below nearer ones: i3 (if hit) deepest, i1 on top
  uint32_t x0 = (uint32_t)(m > 3 ? i3 : (m > 2 ? i2 : i1));
  uint32_t x1 = (uint32_t)(m > 3 ? i2 : i1);
  st.push3(x0, x1, (uint32_t)i1, (uint32_t)(m - 1));
  s.cur = (uint32_t)i0;
}

// Node phase over the wave: lanes with an inner `cur` descend until every
// busy lane holds a postponed leaf, none can descend further, or fewer than
// half of the wave's rays would take a step.
template <bool kSafe>
__device__ __forceinline__ void travNodeLoop(TravState& s, LaneStack& st, TravCount& cnt,
                                             bool active, const BNode4* __restrict__ nodes) {
  while (true) {
    const bool step = active && isInnerRef(s.cur);
    cnt.nodes += (unsigned long long)__popcll(__ballot(step));
    if (step) {
      travNode<kSafe>(s, st, nodes);
      if (isLeafRef(s.cur) && s.pend == kStackEmpty) {
        s.pend = s.cur;
        s.cur = st.pop();
      }
    }
    bool more = active && isInnerRef(s.cur);
    bool hungry = active && s.pend == kStackEmpty && s.cur != kStackEmpty;
    // leave when no lane lacks a leaf, or when fewer than half of the
    // wave's rays would step: the rest go to the leaf phase instead of
    // idling behind a few deep lanes (they resume in the next round).  On
    // C2, C3 and C5 half was 1% faster than a third and than two thirds.
    const int nmore = __popcll(__ballot(more));
    if (nmore == 0 || __ballot(hungry) == 0ull || nmore * 2 < __popcll(__ballot(active))) break;
  }
}

// The safe box tests only in waves with an axis-parallel (or nearly so) ray:
// two copies of the loop, so that the common one carries no handling of them.
__device__ __forceinline__ void travNodePhase(TravState& s, LaneStack& st, TravCount& cnt,
                                              bool active, const BNode4* __restrict__ nodes) {
  if (__ballot(active && needsSafeBoxes(s.inv)) != 0ull)
    travNodeLoop<true>(s, st, cnt, active, nodes);
  else
    travNodeLoop<false>(s, st, cnt, active, nodes);
}

// Leaf phase over the wave.  Most lanes hold one or two triangles at this
// point and a few hold more, so the wave's triangles are pooled: every lane
// lists its triangles (its postponed leaf, and `cur` when that is a leaf too)
// in LDS, and the wave tests 64 of the list at a time, each lane one triangle
// of whichever ray owns it (the owner's ray comes by lane permutes).  A hit
// goes to its owner by a minimum over (t, primitive id), the order that
// testing one triangle after another keeps.  One triangle per lane and step
// of the lane's own ray kept 13-23% of the lanes busy, in five steps a round;
// pooled, a round takes one or two steps.  Measured: 256 uneven domains,
// 1279x719, 8 spp 22.2 -> 20.7 ms a frame; plain schedule, 256x192 11.7 ->
// 10.1 ms; 3 M closest-hit queries on one domain 3.16 -> 2.68 ms.
constexpr int kLeafItems = 128;                                 // triangles listed at once
constexpr int kLeafLdsWords = kLeafItems + 64 * 2 + 64 * 4;     // per wave: list, keys, hit records
static_assert(kLeafMax <= 2, "a lane lists at most 4 triangles (two leaves)");

// Rank of this lane's first item and the wave's total, for 0..4 items a lane.
__device__ __forceinline__ uint32_t rankSmall(uint32_t n, uint32_t* total) {
  const unsigned long long b0 = __ballot(n & 1u), b1 = __ballot(n & 2u), b2 = __ballot(n & 4u);
  *total = (uint32_t)(__popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2));
  const unsigned long long lt = (1ull << __lane_id()) - 1ull;
  return (uint32_t)(__popcll(b0 & lt) + 2 * __popcll(b1 & lt) + 4 * __popcll(b2 & lt));
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

// Every lane of the wave calls it, converged (lds: the wave's leaf area).
__device__ __forceinline__ void travLeafPhase(TravState& s, LaneStack& st, TravCount& cnt,
                                              bool active, const LTri* __restrict__ tris,
                                              uint32_t* lds) {
  typedef __attribute__((address_space(3))) unsigned long long lds_u64;
  typedef __attribute__((address_space(3))) float lds_f;
  lds_u32* items = (lds_u32*)lds;
  lds_u64* keys = (lds_u64*)(items + kLeafItems);
  lds_f* recs = (lds_f*)(items + kLeafItems + 128);
  const int lane = __lane_id();
  while (true) {
    const bool has = active && s.pend != kStackEmpty;
    const bool has2 = active && isLeafRef(s.cur);
    const uint32_t n1 = has ? (s.pend >> 24) & 0x7fu : 0u, n2 = has2 ? (s.cur >> 24) & 0x7fu : 0u;
    if (__ballot(has || has2) == 0ull) break;
    const uint32_t n = n1 + n2;
    uint32_t total;
    const uint32_t rank = rankSmall(n, &total);
    // lanes past the list's end keep their leaves for the next turn
    const bool take = (has || has2) && rank + n <= (uint32_t)kLeafItems;
    const uint32_t listed = min(total, (uint32_t)kLeafItems);
    if (take) {
      const uint32_t own = (uint32_t)lane << 24;
      const uint32_t p0 = own | (s.pend & 0x00ffffffu), c0 = own | (s.cur & 0x00ffffffu);
      for (uint32_t i = 0; i < n1; ++i) items[rank + i] = p0 + i;
      for (uint32_t i = 0; i < n2; ++i) items[rank + n1 + i] = c0 + i;
      s.pend = kStackEmpty;
      if (has2) s.cur = st.pop();
    }
    // the last lane taken may end below `listed`: unlisted slots are skipped
    const unsigned long long tm = __ballot(take && n > 0u);
    const uint32_t count = tm == 0ull ? 0u : min(listed, __builtin_amdgcn_readlane(rank + n, 63 - __builtin_clzll(tm)));
    cnt.tris += take ? n : 0u;
    if (count == 0u) continue;
    keys[lane] = ~0ull;
    const bool any = (s.kk >> 8) & 1u;
    // closest: t <= tlim counts once a hit exists (ties go to the lower id)
    const float ub = (any || s.prim < 0) ? s.tlim : __uint_as_float(__float_as_uint(s.tlim) + 1u);
    ldsWaveSync();
    for (uint32_t base = 0; base < count; base += 64u) {
      const bool in = base + (uint32_t)lane < count;
      const uint32_t it = in ? items[base + lane] : (uint32_t)lane << 24;
      const int own = (int)(it >> 24);
      const uint32_t kk = laneGet(s.kk, own);
      const RayPre rp{(int)(kk & 3u), (int)((kk >> 2) & 3u), (int)((kk >> 4) & 3u),
                      laneGetF(s.Sx, own), laneGetF(s.Sy, own), laneGetF(s.Sz, own)};
      const float org[3] = {laneGetF(s.org[0], own), laneGetF(s.org[1], own), laneGetF(s.org[2], own)};
      const float tn = laneGetF(s.tnear, own), lim = laneGetF(ub, own);
      const uint32_t tb = laneGet(s.tri_base, own);
      float t = 0.f, u = 0.f, v = 0.f;
      int p = 0;
      bool hit = false;
      if (in) {
        const float4* tq = (const float4*)&tris[tb + (it & 0x00ffffffu)];
        const float4 a = tq[0], b = tq[1], c = tq[2];
        const float v0[3] = {a.x, a.y, a.z}, v1[3] = {b.x, b.y, b.z}, v2[3] = {c.x, c.y, c.z};
        p = __float_as_int(a.w);
        hit = triHit(rp, org, v0, v1, v2, tn, lim, &t, &u, &v);
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
        s.cur = s.pend = kStackEmpty;
      } else if (s.prim < 0 || t < s.tlim || p < s.prim) {
        s.tlim = t;
        s.u = recs[64 + lane];
        s.v = recs[128 + lane];
        s.prim = p;
      }
    }
    ldsWaveSync();
    break;
  }
  // a leaf left in `cur` is the next postponed leaf
  if (active && s.pend == kStackEmpty && isLeafRef(s.cur)) {
    s.pend = s.cur;
    s.cur = st.pop();
  }
}

}  // namespace spray
