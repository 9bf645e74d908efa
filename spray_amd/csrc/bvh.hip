// HBM domain pool: vertex normals, BVH build (Morton codes, LDS radix sort,
// PLOC clustering or a Karras hierarchy whose inner boxes are leaf-range
// unions, collapse to a 8-wide BVH)
// and the batch ray queries behind spray_trace_rays / spray_domain_list.
//
// Replaces the reference's per-domain Embree scene (rtcCommit in
// render/trimesh_buffer.cc:213-224) and TriMeshBuffer::computeNormals
// (render/trimesh_buffer.cc:267-326).
#include <hip/hip_runtime.h>

#include <mutex>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>

#include "ctx.h"
#include "kernels_common.h"
#include "traverse.h"

namespace spray {

// ---------------------------------------------------------------------------
// Vertex normals: the reference adds each face's unnormalised normal to its
// three vertices in face order.  A vertex-parallel gather over the faces of
// each vertex, visited in ascending face order, reproduces that float
// summation order exactly.
// Face corners are numbered in 32 bits: a domain has fewer than 2^24 faces.
//
// The build kernels take many domains per launch, domain blockIdx.y of the
// array G each (blockIdx.x and gridDim.x count that domain's blocks): a
// domain alone is a launch of a few microseconds that fills a fraction of the
// GPU, and 47 of them per domain were bound by issuing them.
struct BuildDom {
  const float* vtx;
  const uint32_t *face, *rgb;
  float* nrm;
  float4* fshade;
  LTri* tris;
  BNode8* nodes;
  NodeLeaves* leaves;
  // scratch: vertex adjacency, centroid bounds, sort buffers, leaf-range unions
  uint32_t *cnt, *off, *adj, *rank, *bmm, *keys[2], *vals[2], *hist;
  float *rpre, *rsuf, *rbox8, *rtab;
  // binary tree: leaf and inner boxes; per inner node its children (left,
  // right: c >= 0 inner, c < 0 leaf ~c) and leaf range (first, last)
  float *leafbox, *innerbox;
  int4* tree;
  int* front[2];           // collapse frontiers: binary inner nodes
  int* cc;                 // level counters (kLevelWords)
  int nf, nv, node_cap;
};

__global__ void kVertClear(const BuildDom* __restrict__ G) {
  const BuildDom& B = G[blockIdx.y];
  const uint32_t n = (uint32_t)B.nv + 1u;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) B.cnt[i] = 0u;
}
// The count hands each corner its place in its vertex's list, so that filling
// the lists takes no second round of atomics (0.74 + 0.90 -> 0.85 + 0.28 ms).
__global__ void kVertCount(const BuildDom* __restrict__ G) {
  const BuildDom& B = G[blockIdx.y];
  const uint32_t nc = (uint32_t)B.nf * 3u;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nc; i += gridDim.x * blockDim.x)
    B.rank[i] = atomicAdd(&B.cnt[B.face[i]], 1u);
}
__global__ void kVertFill(const BuildDom* __restrict__ G) {
  const BuildDom& B = G[blockIdx.y];
  const uint32_t nc = (uint32_t)B.nf * 3u;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nc; i += gridDim.x * blockDim.x) {
    B.adj[B.off[B.face[i]] + B.rank[i]] = i / 3u;
  }
}
// Most vertices have at most kVertFaces faces: their list is sorted in
// registers, which leaves every load of it and of its faces independent of the
// others (128 domains of 114k triangles: 0.99 -> 0.74 ms; sorted in HBM).
constexpr int kVertFaces = 8;
__global__ void kVertNormal(const BuildDom* __restrict__ G) {
  const BuildDom& B = G[blockIdx.y];
  const float* __restrict__ vtx = B.vtx;
  const uint32_t* __restrict__ face = B.face;
  for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < B.nv; v += gridDim.x * blockDim.x) {
    uint32_t b = B.off[v], n = B.cnt[v];
    uint32_t* L = B.adj + b;
    float ax = 0.0f, ay = 0.0f, az = 0.0f;
    auto add = [&](uint32_t f) {
      const uint32_t* fc = face + (size_t)f * 3;
      const float* p0 = vtx + (size_t)fc[0] * 3;
      const float* p1 = vtx + (size_t)fc[1] * 3;
      const float* p2 = vtx + (size_t)fc[2] * 3;
      float ux = p1[0] - p0[0], uy = p1[1] - p0[1], uz = p1[2] - p0[2];
      float wx = p2[0] - p0[0], wy = p2[1] - p0[1], wz = p2[2] - p0[2];
      ax += uy * wz - uz * wy;
      ay += uz * wx - ux * wz;
      az += ux * wy - uy * wx;
    };
    if (n <= (uint32_t)kVertFaces) {
      uint32_t x[kVertFaces];
#pragma unroll
      for (int i = 0; i < kVertFaces; ++i) x[i] = (uint32_t)i < n ? L[i] : 0xffffffffu;
#pragma unroll
      for (int r = 0; r < kVertFaces; ++r)  // odd-even transposition
#pragma unroll
        for (int i = r & 1; i + 1 < kVertFaces; i += 2) {
          const uint32_t lo = min(x[i], x[i + 1]), hi = max(x[i], x[i + 1]);
          x[i] = lo;
          x[i + 1] = hi;
        }
#pragma unroll
      for (int i = 0; i < kVertFaces; ++i)
        if ((uint32_t)i < n) add(x[i]);
    } else {
      for (uint32_t i = 1; i < n; ++i) {
        uint32_t x = L[i];
        int j = (int)i - 1;
        while (j >= 0 && L[j] > x) {
          L[j + 1] = L[j];
          --j;
        }
        L[j + 1] = x;
      }
      for (uint32_t i = 0; i < n; ++i) add(L[i]);
    }
    B.nrm[(size_t)v * 3] = ax;
    B.nrm[(size_t)v * 3 + 1] = ay;
    B.nrm[(size_t)v * 3 + 2] = az;
  }
}

// Shading record per face: the three vertex normals and colours of the
// face in one 48-byte record, so shading reads one record per hit instead
// of the face and then six vertex attributes.
// It also sets the centroid bounds (ordered bits, see kCentroidBounds) to
// their starting values for the Morton pass that follows it on the stream.
__global__ void kFaceShade(const BuildDom* __restrict__ G) {
  const BuildDom& B = G[blockIdx.y];
  if (blockIdx.x == 0 && threadIdx.x < 6) B.bmm[threadIdx.x] = threadIdx.x < 3 ? 0xffffffffu : 0u;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < B.nf; i += gridDim.x * blockDim.x) {
    for (int k = 0; k < 3; ++k) {
      uint32_t v = B.face[(size_t)i * 3 + k];
      B.fshade[(size_t)i * 3 + k] = make_float4(B.nrm[(size_t)v * 3], B.nrm[(size_t)v * 3 + 1],
                                                B.nrm[(size_t)v * 3 + 2], __uint_as_float(B.rgb[v]));
    }
  }
}

// ---------------------------------------------------------------------------
// Centroid bounds and Morton codes
__device__ __forceinline__ uint32_t orderedBits(float f) {
  uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float fromOrdered(uint32_t u) {
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// Launched on a small grid (kBoundsGrid blocks): per-block reduction in LDS,
// then one atomic per block and bound, so the six bound words see few
// same-address atomics.
constexpr int kBoundsGrid = 256;
__global__ void __launch_bounds__(256) kCentroidBounds(const BuildDom* __restrict__ G) {
  __shared__ float red[6][4];
  const BuildDom& B = G[blockIdx.y];
  const float* __restrict__ vtx = B.vtx;
  const uint32_t* __restrict__ face = B.face;
  const int nf = B.nf;
  uint32_t *bmin = B.bmm, *bmax = B.bmm + 3;
  float lo[3] = {kInfF, kInfF, kInfF}, hi[3] = {-kInfF, -kInfF, -kInfF};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nf; i += gridDim.x * blockDim.x) {
    for (int k = 0; k < 3; ++k) {
      float a = vtx[(size_t)face[i * 3] * 3 + k], b = vtx[(size_t)face[i * 3 + 1] * 3 + k],
            c = vtx[(size_t)face[i * 3 + 2] * 3 + k];
      float cen = 0.5f * (fminf(a, fminf(b, c)) + fmaxf(a, fmaxf(b, c)));
      lo[k] = fminf(lo[k], cen);
      hi[k] = fmaxf(hi[k], cen);
    }
  }
  const int w = threadIdx.x >> 6;
  for (int k = 0; k < 3; ++k) {
    float l = waveMin(lo[k]), h = waveMax(hi[k]);
    if ((threadIdx.x & 63) == 0) {
      red[k][w] = l;
      red[3 + k][w] = h;
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int k = threadIdx.x;
    float v = red[k][0];
    for (int i = 1; i < (int)(blockDim.x >> 6); ++i) v = k < 3 ? fminf(v, red[k][i]) : fmaxf(v, red[k][i]);
    if (k < 3)
      atomicMin(&bmin[k], orderedBits(v));
    else
      atomicMax(&bmax[k - 3], orderedBits(v));
  }
}

__device__ __forceinline__ uint32_t expandBits10(uint32_t v) {
  v = (v * 0x00010001u) & 0xFF0000FFu;
  v = (v * 0x00000101u) & 0x0F00F00Fu;
  v = (v * 0x00000011u) & 0xC30C30C3u;
  v = (v * 0x00000005u) & 0x49249249u;
  return v;
}

__global__ void kMorton(const BuildDom* __restrict__ G) {
  const BuildDom& B = G[blockIdx.y];
  const float* __restrict__ vtx = B.vtx;
  const uint32_t* __restrict__ face = B.face;
  const int nf = B.nf;
  const uint32_t *bmin = B.bmm, *bmax = B.bmm + 3;
  uint32_t *keys = B.keys[0], *vals = B.vals[0];
  float lo[3], ext[3];
  for (int k = 0; k < 3; ++k) {
    lo[k] = fromOrdered(bmin[k]);
    float e = fromOrdered(bmax[k]) - lo[k];
    ext[k] = e > 0.f ? e : 1.f;
  }
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nf; i += gridDim.x * blockDim.x) {
    uint32_t q[3];
    for (int k = 0; k < 3; ++k) {
      float a = vtx[(size_t)face[i * 3] * 3 + k], b = vtx[(size_t)face[i * 3 + 1] * 3 + k],
            c = vtx[(size_t)face[i * 3 + 2] * 3 + k];
      float cen = 0.5f * (fminf(a, fminf(b, c)) + fmaxf(a, fmaxf(b, c)));
      float x = (cen - lo[k]) / ext[k] * 1024.0f;
      x = fminf(fmaxf(x, 0.0f), 1023.0f);
      q[k] = (uint32_t)x;
    }
    keys[i] = (expandBits10(q[0]) << 2) | (expandBits10(q[1]) << 1) | expandBits10(q[2]);
    vals[i] = (uint32_t)i;
  }
}

// ---------------------------------------------------------------------------
// LSD radix sort of (key, value) pairs, 8-bit digits, 2048-key tiles.
// Ranking inside a tile is stable: each 256-key round is split per wave with
// a ballot-based digit match, waves are ordered through LDS counters and a
// running per-digit count carries across rounds.
constexpr int kRsBlock = 256;
constexpr int kRsItems = 8;
constexpr int kRsTile = kRsBlock * kRsItems;

__host__ __device__ inline int rsTiles(int n) { return (n + kRsTile - 1) / kRsTile; }

// hist[digit][tile] of pass `pass` (8 bits each, buffers alternating)
__global__ void kRsHist(const BuildDom* __restrict__ G, int pass) {
  __shared__ uint32_t h[256];
  const BuildDom& B = G[blockIdx.y];
  const int n = B.nf, tiles = rsTiles(n), shift = 8 * pass;
  if ((int)blockIdx.x >= tiles) return;
  const uint32_t* __restrict__ keys = B.keys[pass & 1];
  h[threadIdx.x] = 0;
  __syncthreads();
  int base = blockIdx.x * kRsTile;
  for (int j = 0; j < kRsItems; ++j) {
    int idx = base + j * kRsBlock + threadIdx.x;
    if (idx < n) atomicAdd(&h[(keys[idx] >> shift) & 255u], 1u);
  }
  __syncthreads();
  B.hist[threadIdx.x * tiles + blockIdx.x] = h[threadIdx.x];
}

__global__ void kRsScatter(const BuildDom* __restrict__ G, int pass) {
  __shared__ uint32_t base[256];
  __shared__ uint32_t run[256];
  __shared__ uint32_t wc[4][256];
  const BuildDom& B = G[blockIdx.y];
  const int n = B.nf, tiles = rsTiles(n), shift = 8 * pass;
  if ((int)blockIdx.x >= tiles) return;
  const uint32_t* __restrict__ kin = B.keys[pass & 1];
  const uint32_t* __restrict__ vin = B.vals[pass & 1];
  uint32_t* __restrict__ kout = B.keys[(pass & 1) ^ 1];
  uint32_t* __restrict__ vout = B.vals[(pass & 1) ^ 1];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  base[tid] = B.hist[tid * tiles + blockIdx.x];
  run[tid] = 0;
  const int tile = blockIdx.x * kRsTile;
  for (int j = 0; j < kRsItems; ++j) {
    wc[0][tid] = 0;
    wc[1][tid] = 0;
    wc[2][tid] = 0;
    wc[3][tid] = 0;
    __syncthreads();
    int idx = tile + j * kRsBlock + tid;
    bool valid = idx < n;
    uint32_t key = valid ? kin[idx] : 0u;
    uint32_t d = (key >> shift) & 255u;
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      bool bit = (d >> b) & 1u;
      uint64_t m = __ballot(bit);
      peers &= bit ? m : ~m;
    }
    uint32_t rank = __popcll(peers & ((1ull << lane) - 1ull));
    if (valid && rank == 0) wc[w][d] = (uint32_t)__popcll(peers);
    __syncthreads();
    {
      uint32_t c0 = wc[0][tid], c1 = wc[1][tid], c2 = wc[2][tid], c3 = wc[3][tid];
      uint32_t r = run[tid];
      wc[0][tid] = r;
      wc[1][tid] = r + c0;
      wc[2][tid] = r + c0 + c1;
      wc[3][tid] = r + c0 + c1 + c2;
      run[tid] = r + c0 + c1 + c2 + c3;
    }
    __syncthreads();
    if (valid) {
      uint32_t dst = base[d] + wc[w][d] + rank;
      kout[dst] = key;
      vout[dst] = vin[idx];
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Karras 2012 hierarchy over sorted keys; duplicate keys are ordered by index.
__device__ __forceinline__ int deltaK(const uint32_t* keys, int n, int i, int j) {
  if (j < 0 || j >= n) return -1;
  uint32_t a = keys[i], b = keys[j];
  if (a == b) return 32 + __clz((uint32_t)(i ^ j));
  return __clz(a ^ b);
}

// inner node i: children encoded c >= 0 inner, c < 0 leaf ~c (sorted position)
__global__ void kKarras(const BuildDom* __restrict__ G) {
  const BuildDom& B = G[blockIdx.y];
  const uint32_t* __restrict__ keys = B.keys[0];
  const int n = B.nf;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n - 1; i += gridDim.x * blockDim.x) {
    int d = (deltaK(keys, n, i, i + 1) - deltaK(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = deltaK(keys, n, i, i - d);
    int lmax = 2;
    while (deltaK(keys, n, i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for (int t = lmax / 2; t >= 1; t /= 2)
      if (deltaK(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int j = i + l * d;
    int dnode = deltaK(keys, n, i, j);
    int s = 0;
    int t = l;
    do {
      t = (t + 1) >> 1;
      if (deltaK(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    int gamma = i + s * d + (d < 0 ? d : 0);
    int lo = i < j ? i : j, hi = i < j ? j : i;
    int lc = (lo == gamma) ? ~gamma : gamma;
    int rc = (hi == gamma + 1) ? ~(gamma + 1) : gamma + 1;
    B.tree[i] = make_int4(lc, rc, lo, hi);
  }
}

// Leaf boxes in sorted order + the leaf-ordered triangle array of the pool
// (order: null for the Morton order).
__global__ void kLeaves(const BuildDom* __restrict__ G, const uint32_t* order_or_null) {
  const BuildDom& B = G[blockIdx.y];
  const float* __restrict__ vtx = B.vtx;
  const uint32_t* __restrict__ face = B.face;
  const uint32_t* __restrict__ order = order_or_null ? order_or_null : B.vals[0];
  float* leafbox = B.leafbox;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < B.nf; i += gridDim.x * blockDim.x) {
    uint32_t p = order[i];
    const float* a = vtx + (size_t)face[p * 3] * 3;
    const float* b = vtx + (size_t)face[p * 3 + 1] * 3;
    const float* c = vtx + (size_t)face[p * 3 + 2] * 3;
    LTri t;
    for (int k = 0; k < 3; ++k) {
      t.v0[k] = a[k];
      t.v1[k] = b[k];
      t.v2[k] = c[k];
      leafbox[(size_t)i * 6 + k] = fminf(a[k], fminf(b[k], c[k]));
      leafbox[(size_t)i * 6 + 3 + k] = fmaxf(a[k], fmaxf(b[k], c[k]));
    }
    t.v0[3] = __int_as_float((int)p);
    t.v1[3] = 0.f;
    t.v2[3] = 0.f;
    B.tris[i] = t;
  }
}

// Inner-node boxes without a bottom-up climb: in a Karras hierarchy inner
// node p covers the sorted leaves [first[p], last[p]], so its box is the
// union of those leaf boxes, a range min/max.  Leaves are grouped in eights
// and in blocks of 64; kLeafScan writes, per leaf, the union from its eight's
// start (prefix) and to its eight's end (suffix), and the boxes of eights and
// blocks; a sparse table over block boxes (level j: unions of 2^j consecutive
// blocks) answers the whole blocks of a range with two lookups, so a range
// takes at most 2 + 14 + 2 boxes.  (With prefixes and suffixes over blocks of
// 64, ranges within a block were walked leaf by leaf, up to 64 of them, the
// whole wave behind the longest: 0.80 -> 0.43 ms for 128 domains of 114k triangles.)  min/max are exact and order-free,
// so the boxes equal a bottom-up refit's, with no device-scope fences or atomics.
constexpr int kRangeBlock = 64;

// Floats before table level j (level 0: block boxes; level j: nblk - 2^j + 1
// entries of 6).
__host__ __device__ inline long long rangeOff(long long nblk, int j) {
  return 6 * ((long long)j * (nblk + 1) - ((1ll << j) - 1));
}
__host__ __device__ inline long long rangeBlocks(int n) { return (n + kRangeBlock - 1) / kRangeBlock; }
inline int rangeLevels(int n) {
  int j = 0;
  for (long long w = 1; w <= rangeBlocks(n) && j < 32; w <<= 1) ++j;
  return j;
}

__device__ __forceinline__ void boxMerge(float lo[3], float hi[3], const float* b) {
  for (int k = 0; k < 3; ++k) {
    lo[k] = fminf(lo[k], b[k]);
    hi[k] = fmaxf(hi[k], b[3 + k]);
  }
}

__global__ void __launch_bounds__(256) kLeafScan(const BuildDom* __restrict__ G) {
  const BuildDom& B = G[blockIdx.y];
  const float* __restrict__ leafbox = B.leafbox;
  float *__restrict__ pre = B.rpre, *__restrict__ suf = B.rsuf, *__restrict__ box8 = B.rbox8,
        *__restrict__ blockbox = B.rtab;
  const int n = B.nf;
  const int lane = threadIdx.x & 63;
  const long long nblk = (n + kRangeBlock - 1) / kRangeBlock;
  const long long nw = ((long long)gridDim.x * blockDim.x) >> 6;
  for (long long b = (blockIdx.x * (long long)blockDim.x + threadIdx.x) >> 6; b < nblk; b += nw) {
    const long long i = b * kRangeBlock + lane;
    const bool in = i < n;
    float plo[3], phi[3], slo[3], shi[3];
    for (int k = 0; k < 3; ++k) {
      plo[k] = slo[k] = in ? leafbox[i * 6 + k] : kInfF;
      phi[k] = shi[k] = in ? leafbox[i * 6 + 3 + k] : -kInfF;
    }
    // (a lane whose partner lies outside its eight meets itself)
    for (int o = 1; o < 8; o <<= 1)
      for (int k = 0; k < 3; ++k) {
        plo[k] = fminf(plo[k], __shfl_up(plo[k], o, 8));
        phi[k] = fmaxf(phi[k], __shfl_up(phi[k], o, 8));
        slo[k] = fminf(slo[k], __shfl_down(slo[k], o, 8));
        shi[k] = fmaxf(shi[k], __shfl_down(shi[k], o, 8));
      }
    if (in)
      for (int k = 0; k < 3; ++k) {
        pre[i * 6 + k] = plo[k];
        pre[i * 6 + 3 + k] = phi[k];
        suf[i * 6 + k] = slo[k];
        suf[i * 6 + 3 + k] = shi[k];
        if ((lane & 7) == 0) {
          box8[(i >> 3) * 6 + k] = slo[k];
          box8[(i >> 3) * 6 + 3 + k] = shi[k];
        }
      }
    for (int o = 8; o < 64; o <<= 1)
      for (int k = 0; k < 3; ++k) {
        slo[k] = fminf(slo[k], __shfl_xor(slo[k], o, 64));
        shi[k] = fmaxf(shi[k], __shfl_xor(shi[k], o, 64));
      }
    if (lane == 0)
      for (int k = 0; k < 3; ++k) {
        blockbox[b * 6 + k] = slo[k];
        blockbox[b * 6 + 3 + k] = shi[k];
      }
  }
}

// Levels j and j + 1 of the sparse table in one launch, from level j - 1
// (h = 2^(j-1) blocks per entry): level j entry i = union(src[i], src[i + h])
// for i < mj, and level j + 1 entry i = union(level j [i], level j [i + 2h])
// for i < mj2 (mj2 <= 0: no such level), each level-j box formed alike.
__global__ void kRangeLevel2(const BuildDom* __restrict__ G, int j) {
  const BuildDom& B = G[blockIdx.y];
  const long long nblk = rangeBlocks(B.nf), h = 1ll << (j - 1);
  const long long mj = nblk - (1ll << j) + 1, mj2 = nblk - (1ll << (j + 1)) + 1;
  const float* __restrict__ src = B.rtab + rangeOff(nblk, j - 1);
  float *__restrict__ dst = B.rtab + rangeOff(nblk, j), *__restrict__ dst2 = B.rtab + rangeOff(nblk, j + 1);
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < mj;
       i += (long long)gridDim.x * blockDim.x) {
    float lo[3], hi[3];
    for (int k = 0; k < 3; ++k) {
      lo[k] = fminf(src[i * 6 + k], src[(i + h) * 6 + k]);
      hi[k] = fmaxf(src[i * 6 + 3 + k], src[(i + h) * 6 + 3 + k]);
      dst[i * 6 + k] = lo[k];
      dst[i * 6 + 3 + k] = hi[k];
    }
    if (i < mj2) {
      const long long a = i + 2 * h, b = i + 3 * h;
      for (int k = 0; k < 3; ++k) {
        dst2[i * 6 + k] = fminf(lo[k], fminf(src[a * 6 + k], src[b * 6 + k]));
        dst2[i * 6 + 3 + k] = fmaxf(hi[k], fmaxf(src[a * 6 + 3 + k], src[b * 6 + 3 + k]));
      }
    }
  }
}

__global__ void kRangeBoxes(const BuildDom* __restrict__ G) {
  const BuildDom& B = G[blockIdx.y];
  const int ninner = B.nf - 1;
  const int4* __restrict__ tree = B.tree;
  const float *__restrict__ leafbox = B.leafbox, *__restrict__ pre = B.rpre, *__restrict__ suf = B.rsuf,
              *__restrict__ box8 = B.rbox8, *__restrict__ table = B.rtab;
  float* __restrict__ innerbox = B.innerbox;
  const long long nblk = rangeBlocks(B.nf);
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < ninner; p += gridDim.x * blockDim.x) {
    const int a = tree[p].z, b = tree[p].w;
    const int ea = a >> 3, eb = b >> 3;
    float lo[3] = {kInfF, kInfF, kInfF}, hi[3] = {-kInfF, -kInfF, -kInfF};
    if (ea == eb) {
      for (int i = a; i <= b; ++i) boxMerge(lo, hi, leafbox + (size_t)i * 6);
    } else {
      boxMerge(lo, hi, suf + (size_t)a * 6);
      boxMerge(lo, hi, pre + (size_t)b * 6);
      // whole eights [x, y), of which the whole blocks [bx, by) through the table
      constexpr int kPer = kRangeBlock / 8;
      int x = ea + 1, y = eb;
      const int bx = (x + kPer - 1) / kPer, by = y / kPer;
      if (bx < by) {
        const int j = 31 - __clz(by - bx);
        const float* lv = table + rangeOff(nblk, j);
        boxMerge(lo, hi, lv + (size_t)bx * 6);
        boxMerge(lo, hi, lv + (size_t)(by - (1 << j)) * 6);
        for (int i = by * kPer; i < y; ++i) boxMerge(lo, hi, box8 + (size_t)i * 6);
        y = bx * kPer;
      }
      for (; x < y; ++x) boxMerge(lo, hi, box8 + (size_t)x * 6);
    }
    for (int k = 0; k < 3; ++k) {
      innerbox[(size_t)p * 6 + k] = lo[k];
      innerbox[(size_t)p * 6 + 3 + k] = hi[k];
    }
  }
}

// 8-wide nodes of a domain of nf triangles, at most.  In the collapsed tree
// a node with fewer than eight children has only leaf children, so it covers
// more than kLeafMax triangles, and those nodes are disjoint.  With N8 nodes
// of eight children and Ns of fewer (two or more): 7 N8 + Ns <= nf - 1 and
// Ns <= nf / (kLeafMax + 1), so N8 + Ns <= (nf - 1) / 7 + 6 nf / (7 (kLeafMax
// + 1)).
__host__ __device__ inline long long nodeCap(long long nf) {
  return nf / 7 + (6 * nf) / (7 * (kLeafMax + 1)) + 16;
}
// leaf lists number a domain's nodes in 23 bits (a domain has fewer than 2^24 faces)
static_assert((1 << 24) / 7 + (6ll * (1 << 24)) / (7 * (kLeafMax + 1)) + 16 < (1 << 23), "node numbers");

// 8-wide collapse levels launched per host wait, and at most (deeper trees
// do not fit the traversal stack anyway); a level counter block is an unused
// word, the overflow flag and the item count of every level
constexpr int kLevelBatch = 16;
constexpr int kMaxLevels = 48;
constexpr int kLevelWords = 2 + kMaxLevels + 1;

__device__ __forceinline__ float boxArea(const float* b) {
  float dx = fmaxf(b[3] - b[0], 0.f), dy = fmaxf(b[4] - b[1], 0.f), dz = fmaxf(b[5] - b[2], 0.f);
  return dx * dy + dy * dz + dz * dx;
}

// Reductions over the 8 lanes of a group (lanes 8i .. 8i + 7), the result in
// every lane: exchanges within pairs, pairs of pairs, and both quads.
template <int kCtl>
__device__ __forceinline__ uint32_t dpp8u(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtl, 0xf, 0xf, true);
}
template <int kCtl>
__device__ __forceinline__ float dpp8(float v) {
  return __uint_as_float(dpp8u<kCtl>(__float_as_uint(v)));
}
__device__ __forceinline__ float groupMin(float v) {
  v = fminf(v, dpp8<0xB1>(v));
  v = fminf(v, dpp8<0x4E>(v));
  return fminf(v, dpp8<0x141>(v));
}
__device__ __forceinline__ float groupMax(float v) {
  v = fmaxf(v, dpp8<0xB1>(v));
  v = fmaxf(v, dpp8<0x4E>(v));
  return fmaxf(v, dpp8<0x141>(v));
}
// the lanes of the group with p set, bit i for its lane i
__device__ __forceinline__ uint32_t groupBallot(bool p) {
  return (uint32_t)(__ballot(p) >> (threadIdx.x & 56)) & 255u;
}

// The largest float at least 1/64 of a step (2^e) below lo whose last byte is
// e + 127.
__device__ __forceinline__ float gridBase(float lo, int e, double step) {
  const double bd = (double)lo - step * 0.015625;
  float f = (float)bd;
  if ((double)f > bd) f = nextafterf(f, -kInfF);
  const uint32_t u = __float_as_uint(f), byte = (uint32_t)(e + 127);
  uint32_t w = (u & ~255u) | byte;
  if (u >> 31) {
    if (w < u) w += 256u;
  } else if (w > u) {
    w = u >= 256u ? w - 256u : 0x80000000u | byte;
  }
  return __uint_as_float(w);
}

// Writes a node's grid and child planes; called by the 8 lanes of a group,
// each with the box (lo xyz, hi xyz) and slot of one child (used), the other
// lanes with a slot of their own among those left.  Per
// axis the step is the power of two that covers the children's extent in at
// most 253 steps (at least 2^-20 of the largest coordinate), or the next one:
// base, whose last byte is the step's exponent, lies 1/64 of a step to 33
// steps below the lowest plane, and the highest has to be within 255 steps of
// it.  Planes are rounded outwards with 2^-9 of a step to spare: the distance
// test's cancellation error (nodeBoxes) is below 2^-15 of a step.  An axis
// whose extent is not finite, or would need a step of 2^62 or more, covers
// everything.  Lane k of the group works out axis k's grid.
__device__ __forceinline__ void quantizeNode(const float (&b)[6], bool used, uint32_t slot, BNode8* nd) {
  const int me = threadIdx.x & 7;
  float lo = 0.f, hi = 0.f;
  bool finite = false;
  const bool any = groupBallot(used) != 0u;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float l = groupMin(used ? b[k] : kInfF), h = groupMax(used ? b[3 + k] : -kInfF);
    const bool f = groupBallot(used && !(fabsf(b[k]) < kInfF && fabsf(b[3 + k]) < kInfF)) == 0u;
    if (me == k) {
      lo = l;
      hi = h;
      finite = any && f;
    }
  }
  auto exponent = [](double x) { return (int)((__double2hiint(x) >> 20) & 2047) - 1023; };
  auto power = [](int x) { return __hiloint2double((x + 1023) << 20, 0); };
  const double ext = (double)hi - (double)lo;  // (of floats: no subnormal double)
  const double big = fmax(fabs((double)lo), fabs((double)hi));
  int e = -126;
  if (finite) {
    // smallest e with 253 * 2^e >= ext and 2^e >= big * 2^-20
    if (ext > 0.0) {
      e = max(e, exponent(ext) - 7);
      if (253.0 * power(e) < ext) ++e;
    }
    if (big > 0.0) e = max(e, exponent(big) - 19);
  }
  const bool all = !finite || e >= 61;
  // all: not a number, so every plane distance is not a number and bounds
  // nothing (a finite base as low as that would overflow against 1/dir)
  float base = __uint_as_float(0x7fc000f8u);
  if (all) {
    e = 121;
  } else {
    base = gridBase(lo, e, power(e));
    // at twice the step the extent is below 127 steps, and base's distance halves
    if (((double)hi - (double)base) * power(-e) + 0.001953125 > 255.0) {
      ++e;
      base = gridBase(lo, e, power(e));
    }
  }
  if (me < 3) nd->base[me] = base;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int ek = __shfl(e, k, 8);
    const float bk = __shfl(base, k, 8), inv = __uint_as_float((uint32_t)(127 - ek) << 23);
    const bool allk = ek == 121;
    uint32_t l = 255u, h = 0u;  // unused slots: inverted
    if (used) {
      // (rounding b - base is below 2^-16 of a step, far less than is to spare)
      l = allk ? 0u : (uint32_t)fminf(fmaxf(floorf((b[k] - bk) * inv - 0.001953125f), 0.f), 255.f);
      h = allk ? 255u : (uint32_t)fminf(fmaxf(ceilf((b[3 + k] - bk) * inv + 0.001953125f), 0.f), 255.f);
    }
    nd->plane[k][slot] = (uint8_t)l;
    nd->plane[k][8 + slot] = (uint8_t)h;
  }
}

// Slot of each lane's child (one child per used lane of the group; the other
// lanes get the slots left): greedily the (child, slot) pair whose child
// centre lies farthest to the slot's side of the node (bit k of the slot: the
// upper side of axis k).  Distances are compared as ordered integers with the
// pair in their last six bits, so that one maximum over a lane's slots and
// the group's lanes names the pair; a distance that is not a number comes
// last.
__device__ __forceinline__ uint32_t assignSlot(const float (&b)[6], bool used) {
  const uint32_t me = threadIdx.x & 7;
  float d[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float lo = groupMin(used ? b[k] : kInfF), hi = groupMax(used ? b[3 + k] : -kInfF);
    d[k] = (b[k] + b[3 + k]) - (lo + hi);
  }
  uint32_t key[8];  // > 0 while the slot is free
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const float t = ((s & 1) ? d[0] : -d[0]) + ((s & 2) ? d[1] : -d[1]) + ((s & 4) ? d[2] : -d[2]);
    const uint32_t u = __float_as_uint(t == t ? t : -kInfF);
    key[s] = ((u ^ ((u >> 31) ? 0xffffffffu : 0x80000000u)) & ~63u) | ((7u - me) << 3) | (7u - s);
  }
  uint32_t slot = 0, frees = 255u;
  bool open = used;
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    uint32_t top = 0;
#pragma unroll
    for (int s = 0; s < 8; ++s) top = max(top, key[s]);
    top = open ? top : 0u;
    top = max(top, dpp8u<0xB1>(top));
    top = max(top, dpp8u<0x4E>(top));
    top = max(top, dpp8u<0x141>(top));
    if (top != 0u) {  // (0: no child left)
      const uint32_t bs = 7u - (top & 7u);
      if (me == 7u - ((top >> 3) & 7u)) {
        slot = bs;
        open = false;
      }
      frees &= ~(1u << bs);
#pragma unroll
      for (int s = 0; s < 8; ++s) key[s] &= (uint32_t)__builtin_amdgcn_sbfe((int)frees, s, 1);
    }
  }
  const uint32_t taken = groupBallot(used);  // (of all the group's lanes)
  if (!used) {  // the r-th unused lane takes the r-th free slot
    int r = __popc(~taken & ((1u << me) - 1u));
    for (; r > 0; --r) frees &= frees - 1u;
    slot = (uint32_t)__ffs((int)frees) - 1u;
  }
  return slot;
}

// One frontier level l of every domain of the launch: cc[2 + l] items (0:
// nothing to do), the next level's counted in cc[3 + l]; cc[1] is the
// overflow flag.  A level's items are its nodes, numbered after those of the
// levels above.  Launched level after level without host round trips; the
// loop bound is uniform per block.
//
// Eight lanes take an item, one per child: a lane holds its child's box and
// record, so that opening the largest inner child is one round of loads by
// the two lanes that get its children, and the node leaves through LDS as one
// line.  Bound by vector issue (about 1570 instructions per wave of 8 items,
// 55% of the time) and the chain of six rounds of loads.  One lane per item,
// all eight boxes in its registers, spilled at 128 registers, took an eighth
// of the waves and read left, right, first and last of each child from four
// arrays: the collapse launches of a remesh of 128 domains (8 x 4 x 4, field
// resolution 72) took 5.8 ms, now 3.4 ms.
__global__ void __launch_bounds__(256) kCollapseLevel(const BuildDom* __restrict__ G, int l) {
  __shared__ BNode8 img[32];
  __shared__ NodeLeaves limg[32];
  __shared__ int alloc[32];
  const BuildDom& B = G[blockIdx.y];
  const int nin = B.cc[2 + l];
  const int over = B.cc[1];  // 1 + the level that overflowed (its blocks all finish)
  if (nin <= (int)(blockIdx.x * 32) || (over != 0 && over <= l)) return;
  int start = 0;  // nodes of the levels above
  for (int j = 0; j < l; ++j) start += B.cc[2 + j];
  const int* __restrict__ fin = B.front[l & 1];
  int* fout = B.front[(l & 1) ^ 1];
  const int4* __restrict__ tree = B.tree;
  const float *__restrict__ leafbox = B.leafbox, *__restrict__ innerbox = B.innerbox;
  const int me = threadIdx.x & 7, grp = threadIdx.x >> 3;
  for (int base = blockIdx.x * 32; base < nin; base += gridDim.x * 32) {
    const int it = base + grp;
    const bool act = it < nin;
    int c = 0;               // this lane's child, its record, box and area when it can be opened
    int4 rec{0, 0, 0, 0};
    float b[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float area = -1.f;
    auto load = [&] {
      const float2* src = (const float2*)(c < 0 ? leafbox + (size_t)(~c) * 6 : innerbox + (size_t)c * 6);
      rec = c < 0 ? make_int4(0, 0, ~c, ~c) : tree[c];
      const float2 x = src[0], y = src[1], z = src[2];
      b[0] = x.x, b[1] = x.y, b[2] = y.x, b[3] = y.y, b[4] = z.x, b[5] = z.y;
      area = rec.w - rec.z + 1 > kLeafMax ? boxArea(b) : -1.f;
    };
    int nc = 0;
    if (act) {
      const int4 root = tree[fin[it]];
      nc = 2;
      if (me < 2) {
        c = me == 0 ? root.x : root.y;
        load();
      }
    }
    // open the inner child of the largest area, the first such; its lane
    // takes the left child and the next free lane the right one
    for (int n = 0; n < 6; ++n) {
      const float top = groupMax(area);
      const bool go = top > -1.f;
      if (__ballot(go) == 0ull) break;
      const int best = __ffs((int)groupBallot(area == top)) - 1;
      const int lc = __shfl(rec.x, best, 8), rc = __shfl(rec.y, best, 8);
      if (go && (me == best || me == nc)) {
        c = me == best ? lc : rc;
        load();
      }
      nc += go ? 1 : 0;
    }
    const bool used = me < nc;
    const int cnt = rec.w - rec.z + 1;
    const bool inner = used && cnt > kLeafMax;
    const uint32_t slot = assignSlot(b, used);
    // children of a node that are inner nodes take consecutive numbers in slot order
    uint32_t im = inner ? 1u << slot : 0u;
    for (int o = 1; o < 8; o <<= 1) im |= (uint32_t)__shfl_xor((int)im, o, 8);
    if (me == 0) alloc[grp] = __popc(im);
    __syncthreads();
    if (threadIdx.x < 64) {
      const int lane = threadIdx.x;
      const int own = lane < 32 ? alloc[lane] : 0;
      int incl = own;
      for (int o = 1; o < 32; o <<= 1) {
        const int v = __shfl_up(incl, o, 64);
        if (lane >= o) incl += v;
      }
      const int total = __shfl(incl, 31, 64);
      int first = 0;
      if (lane == 0 && total > 0) first = atomicAdd(&B.cc[3 + l], total);
      first = __shfl(first, 0, 64);
      if (lane < 32) alloc[lane] = first + incl - own;
    }
    __syncthreads();
    const int q = alloc[grp], cbase = start + nin + q;
    const bool fits = cbase + __popc(im) <= B.node_cap;
    if (!fits && me == 0) atomicExch(&B.cc[1], l + 1);  // the levels below return at once
    quantizeNode(b, used, slot, &img[grp]);
    if (me == 0) img[grp].kids = ((uint32_t)cbase & 0xffffffu) | (im << 24);
    limg[grp].leaf[slot] = used && !inner ? ((uint32_t)cnt << 24) | (uint32_t)rec.z : 0u;
    if (inner && fits) fout[q + __popc(im & ((1u << slot) - 1u))] = c;
    __syncthreads();
    if (act && me < 4)
      ((float4*)(B.nodes + start + it))[me] = ((const float4*)&img[grp])[me];
    else if (act && me < 6)
      ((float4*)(B.leaves + start + it))[me - 4] = ((const float4*)&limg[grp])[me - 4];
    __syncthreads();
  }
}

// Collapse state of each domain: no overflow, one frontier item (binary node
// `root`) at level 0 (none for a domain of one leaf, whose root kTinyRoot
// writes), empty later levels.
__global__ void kCollapseInit(const BuildDom* __restrict__ G, int root) {
  const BuildDom& B = G[blockIdx.y];
  for (int i = threadIdx.x; i < kLevelWords; i += blockDim.x)
    B.cc[i] = i == 2 && B.nf > kLeafMax ? 1 : 0;
  if (threadIdx.x == 0) B.front[0][0] = root;
}

// Primitive ids in leaf order.
__global__ void kPrimIds(const LTri* __restrict__ tris, int nf, uint32_t* order) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nf; i += gridDim.x * blockDim.x)
    order[i] = __float_as_uint(tris[i].v0[3]);
}

// Root for tiny domains (<= kLeafMax triangles): one leaf child.  One group.
__global__ void kTinyRoot(const BuildDom* __restrict__ G) {
  const int nf = G->nf, me = threadIdx.x;
  const float* leafbox = G->leafbox;
  BNode8* nd = G->nodes;
  float b[6] = {kInfF, kInfF, kInfF, -kInfF, -kInfF, -kInfF};
  for (int i = 0; i < nf; ++i)
    for (int k = 0; k < 3; ++k) {
      b[k] = fminf(b[k], leafbox[i * 6 + k]);
      b[3 + k] = fmaxf(b[3 + k], leafbox[i * 6 + 3 + k]);
    }
  quantizeNode(b, me == 0 && nf > 0, (uint32_t)me, nd);
  if (me == 0) nd->kids = 0;
  G->leaves->leaf[me] = me == 0 ? (uint32_t)nf << 24 : 0u;
}

// ---------------------------------------------------------------------------
// PLOC hierarchy (Meister & Bittner, "Parallel Locally-Ordered Clustering
// for Bounding Volume Hierarchy Construction", IEEE TVCG 2018).  Clusters
// start as the leaves in Morton order.  Each pass pairs every cluster with
// the neighbour within +-kPlocRadius array positions whose union box has the
// least surface area, merges mutual pairs into a new inner node that takes
// the lower position, and compacts the array in order.  Distance ties go to
// the lexicographically smallest (lower, upper) position pair, a strict
// order on pairs, so the globally closest pair is always mutual and every
// pass merges at least one pair.  Inner node ids follow creation order; the
// root is the last one (nf - 2).
constexpr int kPlocRadius = 16;
constexpr int kPlocBlock = 256;

__global__ void kPlocInit(const float* __restrict__ vtx, const uint32_t* __restrict__ face, int nf,
                          const uint32_t* __restrict__ order, int* cid, float* cbox) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nf; i += gridDim.x * blockDim.x) {
    uint32_t p = order[i];
    const float* a = vtx + (size_t)face[p * 3] * 3;
    const float* b = vtx + (size_t)face[p * 3 + 1] * 3;
    const float* c = vtx + (size_t)face[p * 3 + 2] * 3;
    for (int k = 0; k < 3; ++k) {
      cbox[(size_t)i * 6 + k] = fminf(a[k], fminf(b[k], c[k]));
      cbox[(size_t)i * 6 + 3 + k] = fmaxf(a[k], fmaxf(b[k], c[k]));
    }
    cid[i] = ~i;
  }
}

__device__ __forceinline__ float unionArea(const float* a, const float* b) {
  float dx = fmaxf(a[3], b[3]) - fminf(a[0], b[0]);
  float dy = fmaxf(a[4], b[4]) - fminf(a[1], b[1]);
  float dz = fmaxf(a[5], b[5]) - fminf(a[2], b[2]);
  return dx * dy + dy * dz + dz * dx;
}

// nn[i] = nearest neighbour of cluster i; the block's boxes plus a halo of
// kPlocRadius on each side are staged in LDS.
__global__ void __launch_bounds__(kPlocBlock) kPlocNearest(const float* __restrict__ cbox, int n,
                                                            int* __restrict__ nn) {
  constexpr int kSpan = kPlocBlock + 2 * kPlocRadius;
  __shared__ float sb[kSpan * 6];
  const int lo = blockIdx.x * kPlocBlock - kPlocRadius;
  for (int t = threadIdx.x; t < kSpan * 6; t += kPlocBlock) {
    int g = lo * 6 + t;
    sb[t] = (g >= 0 && g < n * 6) ? cbox[g] : 0.f;
  }
  __syncthreads();
  const int i = blockIdx.x * kPlocBlock + threadIdx.x;
  if (i >= n) return;
  float me[6];
  for (int k = 0; k < 6; ++k) me[k] = sb[(i - lo) * 6 + k];
  const int jlo = max(i - kPlocRadius, 0), jhi = min(i + kPlocRadius, n - 1);
  float best = kInfF;
  int bj = -1;
  // ascending j visits the candidate pairs in ascending (lower, upper) order,
  // so a strict comparison keeps the smallest pair among equal areas
  for (int j = jlo; j <= jhi; ++j) {
    if (j == i) continue;
    float a = unionArea(me, sb + (j - lo) * 6);
    if (a < best || bj < 0) {
      best = a;
      bj = j;
    }
  }
  nn[i] = bj;
}

// mflag[i]: cluster i starts a merge (mutual pair, lower position);
// kflag[i]: cluster i keeps a position after the pass.
__global__ void kPlocFlags(const int* __restrict__ nn, int n, uint32_t* mflag, uint32_t* kflag) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i <= n; i += gridDim.x * blockDim.x) {
    if (i == n) {
      mflag[n] = 0u;
      kflag[n] = 0u;
      continue;
    }
    int j = nn[i];
    bool mutual = nn[j] == i;
    mflag[i] = (mutual && i < j) ? 1u : 0u;
    kflag[i] = (mutual && j < i) ? 0u : 1u;
  }
}

__global__ void kPlocMerge(const int* __restrict__ nn, int n, const int* __restrict__ cid,
                           const float* __restrict__ cbox, const uint32_t* __restrict__ mpos,
                           const uint32_t* __restrict__ kpos, int node_base, int* cid2,
                           float* cbox2, int4* tree, float* innerbox, int* icount) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    int j = nn[i];
    bool mutual = nn[j] == i;
    if (mutual && j < i) continue;
    uint32_t o = kpos[i];
    if (mutual) {
      int id = node_base + (int)mpos[i];
      int a = cid[i], b = cid[j];
      tree[id].x = a;
      tree[id].y = b;
      icount[id] = (a < 0 ? 1 : icount[a]) + (b < 0 ? 1 : icount[b]);
      for (int k = 0; k < 3; ++k) {
        float l = fminf(cbox[(size_t)i * 6 + k], cbox[(size_t)j * 6 + k]);
        float h = fmaxf(cbox[(size_t)i * 6 + 3 + k], cbox[(size_t)j * 6 + 3 + k]);
        innerbox[(size_t)id * 6 + k] = l;
        innerbox[(size_t)id * 6 + 3 + k] = h;
        cbox2[(size_t)o * 6 + k] = l;
        cbox2[(size_t)o * 6 + 3 + k] = h;
      }
      cid2[o] = id;
    } else {
      for (int k = 0; k < 6; ++k) cbox2[(size_t)o * 6 + k] = cbox[(size_t)i * 6 + k];
      cid2[o] = cid[i];
    }
  }
}

// Depth-first leaf ranges, top-down over the nodes one pass created (their
// parents come from later passes and are already placed).  Leaf children are
// renumbered to their depth-first position q, and perm[q] keeps the Morton
// position they came from.
__global__ void kPlocRanges(int id_lo, int id_hi, int4* tree, const int* __restrict__ icount,
                            uint32_t* perm) {
  for (int id = id_lo + blockIdx.x * blockDim.x + threadIdx.x; id < id_hi;
       id += gridDim.x * blockDim.x) {
    int f = tree[id].z;
    int a = tree[id].x, b = tree[id].y;
    int fb = f + (a < 0 ? 1 : icount[a]);
    if (a < 0) {
      perm[f] = (uint32_t)(~a);
      tree[id].x = ~f;
    } else {
      tree[a].z = f;
    }
    if (b < 0) {
      perm[fb] = (uint32_t)(~b);
      tree[id].y = ~fb;
    } else {
      tree[b].z = fb;
    }
    tree[id].w = f + icount[id] - 1;
  }
}

__global__ void kComposeOrder(const uint32_t* __restrict__ perm, const uint32_t* __restrict__ morton,
                              int n, uint32_t* order) {
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x)
    order[q] = morton[perm[q]];
}

// ---------------------------------------------------------------------------
static int gridFor(long long n, int block) {
  long long g = (n + block - 1) / block;
  if (g < 1) g = 1;
  if (g > 65535) g = 65535;
  return (int)g;
}

// One domain's build scratch within a pipeline's memory (a slot): byte
// offsets, sized for the largest domain.
struct SlotLayout {
  size_t keys[2], vals[2], hist, cnt, bmm, vsums, hsums, adj, rank, rpre, rsuf, rbox8, rtab, lb, ib, tree,
      front[2], bytes = 0;
  SlotLayout(int maxf, long long maxv) {
    auto take = [&](size_t b) {
      const size_t at = bytes;
      bytes += (b + 255) & ~(size_t)255;
      return at;
    };
    const size_t f = (size_t)maxf + 1, f4 = f * 4, hist_n = (size_t)256 * rsTiles(maxf);
    for (size_t* x : {&keys[0], &keys[1], &vals[0], &vals[1]}) *x = take(f4);
    hist = take(hist_n * 4);
    cnt = take((size_t)(maxv + 1) * 8);
    bmm = take(64);
    vsums = take((size_t)scanSumsWords(maxv + 1) * 4);
    hsums = take((size_t)scanSumsWords((long long)hist_n) * 4);
    adj = take(f * 12);
    rank = take(f * 12);
    tree = take(f * sizeof(int4));
    for (size_t* x : {&rpre, &rsuf, &lb, &ib}) *x = take(f * 24);
    rbox8 = take((f / 8 + 1) * 24);
    rtab = take((size_t)rangeOff(rangeBlocks(maxf), rangeLevels(maxf)) * 4 + 64);
    // a frontier level holds disjoint subtrees of more than kLeafMax triangles
    for (size_t* x : {&front[0], &front[1]}) *x = take(((size_t)maxf / (kLeafMax + 1) + 64) * 4);
  }
};
constexpr int kBuildStreams = 4;  // pipelines of a whole-scene LBVH build
constexpr int kBuildGroup = 16;   // domains per launch, at most
// Slots of all pipelines together: this, or a sixteenth of the free HBM if that
// is less.  Domains alone in their launches (a small budget) leave the narrow
// levels of their trees waiting for memory: remeshes of 128 domains of 563k
// triangles take 61.4 / 54.3 / 49.2 / 47.6 / 47.6 ms with 0.5 / 1 / 2 / 4 / 8 GB,
// of 32 of 1.06 M 28.2 / 28.2 / 25.4 / 25.1 / 24.4 ms.
// Domains too large for that still go one to a launch in as many pipelines as
// half of the free HBM holds, and in one where it holds none.
constexpr size_t kSlotBudget = (size_t)8 << 30;

struct PlocScratch {
  DevBuf pc, pc2, pb, pb2, pnn, pcnt, pmf, pkf, pmp, pkp, pperm, pord;
  void reserve(int maxf) {
    const size_t f4 = (size_t)maxf * 4 + 64;
    for (DevBuf* b : {&pc, &pc2, &pnn, &pcnt, &pmf, &pkf, &pmp, &pkp, &pperm, &pord}) b->reserve(f4);
    pb.reserve((size_t)maxf * 24 + 64);
    pb2.reserve((size_t)maxf * 24 + 64);
  }
  ~PlocScratch() {
    for (DevBuf* b : {&pc, &pc2, &pb, &pb2, &pnn, &pcnt, &pmf, &pkf, &pmp, &pkp, &pperm, &pord}) b->release();
  }
};

// Build memory: slots of each pipeline, domain descriptors and scan jobs,
// level counters of every domain.
struct BuildCache {
  DevBuf slots;
  DevBuf descs, levels;
  ~BuildCache() {
    slots.release();
    descs.release();
    levels.release();
  }
};

void buildCacheRelease(Ctx* c) {
  delete c->build_cache;
  c->build_cache = nullptr;
}

void HostMeshSource::fill(Ctx* c, int d, float* v, uint32_t* f, uint32_t* rgb, hipStream_t s) {
  (void)c;
  SPRAY_HIP(hipMemcpyAsync(v, m[d].v.data(), m[d].v.size() * 4, hipMemcpyHostToDevice, s));
  SPRAY_HIP(hipMemcpyAsync(f, m[d].f.data(), m[d].f.size() * 4, hipMemcpyHostToDevice, s));
  SPRAY_HIP(hipMemcpyAsync(rgb, m[d].rgb.data(), m[d].rgb.size() * 4, hipMemcpyHostToDevice, s));
}

void buildPool(Ctx* c, MeshSource& src, bool keep_buffers) {
  auto t_start = std::chrono::steady_clock::now();
  DomainPool& P = c->pool;
  hipStream_t s = c->stream;
  int nd = (int)c->scene.domains.size();
  // a cache smaller than the scene pages domains (raw meshes are staged one
  // domain at a time, images kept in pinned host memory)
  const bool paged = c->cache_size > 0 && c->cache_size < nd;
  if (keep_buffers && !paged && !P.paged) {
    P.desc.clear();  // device buffers stay; they grow when too small
  } else {
    P.release(!paged);
  }
  if (paged && !c->tracer) c->frame_mem.release();
  P.ndomains = nd;
  P.desc.resize(nd);
  P.nverts.resize(nd);
  long long tv = 0, tf = 0, tn = 0;
  int maxf = 0;
  long long maxv = 0, max_nodes = 0;
  for (int d = 0; d < nd; ++d) {
    const HostDomain& hd = c->scene.domains[d];
    DomainDesc& D = P.desc[d];
    long long nv = src.numVerts(d), nf = src.numFaces(d);
    P.nverts[d] = nv;
    if (nf >= (1 << 24)) throw StatusError(SPRAY_ERR_CAPACITY, "domain has more than 2^24 faces");
    D.vtx_off = paged ? 0 : tv;
    D.face_off = paged ? 0 : tf;
    D.tri_off = tf;
    D.node_off = tn;
    D.shade_off = D.face_off;
    D.num_tris = (int)nf;
    D.num_nodes = 0;
    for (int k = 0; k < 3; ++k) {
      D.lo[k] = hd.lo[k];
      D.hi[k] = hd.hi[k];
    }
    D.mtl = hd.mtl;
    D.eta_a = hd.eta_a;
    D.eta_b = hd.eta_b;
    tv += nv;
    tf += nf;
    tn += nodeCap(nf);
    maxf = std::max(maxf, (int)nf);
    maxv = std::max(maxv, nv);
    max_nodes = std::max(max_nodes, nodeCap(nf));
  }
  P.total_verts = tv;
  P.total_tris = tf;
  if (paged) {
    P.paged = true;
    P.capacity = c->cache_size;
    P.block_nodes = max_nodes;
    P.block_tris = maxf;
    P.vtx.reserve(maxv * 12 + 64);
    P.face.reserve((size_t)maxf * 12 + 64);
    P.rgb.reserve(maxv * 4 + 64);
    P.nrm.reserve(maxv * 12 + 64);
    P.tris.reserve((size_t)P.capacity * maxf * sizeof(LTri) + 64);
    P.fshade.reserve((size_t)P.capacity * maxf * 48 + 64);
    P.nodes.reserve((size_t)P.capacity * max_nodes * sizeof(BNode8) + 64);
    P.leaves.reserve((size_t)P.capacity * max_nodes * sizeof(NodeLeaves) + 64);
    size_t bytes = 0;
    P.h_image_off.resize(nd);
    for (int d = 0; d < nd; ++d) {
      P.h_image_off[d] = (long long)bytes;
      const size_t nf = (size_t)P.desc[d].num_tris;
      bytes += (ImageLayout(nodeCap((long long)nf), (long long)nf, P.nverts[d]).bytes + 255) & ~(size_t)255;
    }
    SPRAY_HIP(hipHostMalloc(&P.h_image, bytes, hipHostMallocDefault));
    P.h_nrm.resize(nd);
  } else {
    BufPlan plan;
    plan.want(P.vtx, tv * 12);
    plan.want(P.face, tf * 12);
    plan.want(P.rgb, tv * 4);
    plan.want(P.nrm, tv * 12);
    plan.want(P.tris, tf * sizeof(LTri));
    plan.want(P.fshade, tf * 48 + 64);
    plan.want(P.nodes, tn * sizeof(BNode8));
    plan.want(P.leaves, tn * sizeof(NodeLeaves));
    if (!plan.fits()) plan.place(P.mem);
  }
  // A whole-scene LBVH build takes the domains in groups, one launch per
  // build step for a group, up to kBuildStreams groups side by side (one per
  // free hardware queue, each with its own slots); the collapse launches a
  // fixed number of levels with no host wait, and the level counts of every
  // domain are checked once after the last.  PLOC and paged builds take one
  // domain at a time in one stream with a host check per domain.
  const bool multi = !paged && c->bvh_builder == 0 && nd > 1;
  if (!paged) {
    if (!src.fillAll(c, P.desc, P.vtx.as<float>(), P.face.as<uint32_t>(), P.rgb.as<uint32_t>(), s))
      for (int d = 0; d < nd; ++d) {
        const DomainDesc& D = P.desc[d];
        src.fill(c, d, P.vtx.as<float>() + D.vtx_off * 3, P.face.as<uint32_t>() + D.face_off * 3,
                 P.rgb.as<uint32_t>() + D.vtx_off, s);
      }
    src.check(c);
  }
  // a remesh of the same domain structure launches the previous depth + 4
  // levels (a domain that needs more is rebuilt with host-checked levels)
  std::vector<int> prev_depth;
  if (keep_buffers && (int)P.bvh_depth.size() == nd) prev_depth = P.bvh_depth;
  P.bvh_depth.assign(nd, 0);
  // a remesh keeps the build memory for the next remesh (it only grows), so
  // repeated remeshes allocate nothing here; other builds hold none afterwards
  BuildCache local;
  BuildCache* M = &local;
  if (multi && src.rebuilds() && keep_buffers) {
    if (!c->build_cache) c->build_cache = new BuildCache;
    M = c->build_cache;
  } else {
    buildCacheRelease(c);
  }
  const SlotLayout SL(std::max(maxf, 1), maxv);
  int K = 1, GN = 1;
  if (multi) {
    size_t free_b = 0, total_b = 0;
    SPRAY_HIP(hipMemGetInfo(&free_b, &total_b));
    const size_t avail = free_b + M->slots.bytes, budget = std::min(kSlotBudget, avail / 16);
    K = (int)std::max<size_t>(1, std::min<size_t>({(size_t)pipelineCount(kBuildStreams), (size_t)nd,
                                                   avail / 2 / SL.bytes}));
    GN = (int)std::max<size_t>(1, std::min<size_t>({(size_t)kBuildGroup, (size_t)((nd + K - 1) / K),
                                                    budget / ((size_t)K * SL.bytes)}));
  }
  const int ngroups = (nd + GN - 1) / GN;
  M->slots.reserve((size_t)K * GN * SL.bytes);
  M->levels.reserve((size_t)nd * kLevelWords * 4 + 64);
  M->descs.reserve((size_t)nd * (sizeof(BuildDom) + 2 * sizeof(ScanJob)) + 64);
  const BuildDom* dev = M->descs.as<BuildDom>();
  const ScanJob* vscan = (const ScanJob*)(dev + nd);
  const ScanJob* hscan = vscan + nd;
  {
    std::vector<char> host((size_t)nd * (sizeof(BuildDom) + 2 * sizeof(ScanJob)));
    BuildDom* hb = (BuildDom*)host.data();
    ScanJob* hv = (ScanJob*)(hb + nd);
    ScanJob* hh = hv + nd;
    for (int d = 0; d < nd; ++d) {
      DomainDesc& D = P.desc[d];
      if (paged) {  // built into block d % capacity from the staged mesh
        const int b = d % P.capacity;
        D.node_off = (long long)b * P.block_nodes;
        D.tri_off = D.shade_off = (long long)b * P.block_tris;
      }
      char* slot = M->slots.as<char>() + ((size_t)((d / GN) % K) * GN + d % GN) * SL.bytes;
      BuildDom& B = hb[d];
      B.vtx = P.vtx.as<float>() + D.vtx_off * 3;
      B.face = P.face.as<uint32_t>() + D.face_off * 3;
      B.rgb = P.rgb.as<uint32_t>() + D.vtx_off;
      B.nrm = P.nrm.as<float>() + D.vtx_off * 3;
      B.fshade = P.fshade.as<float4>() + D.shade_off * 3;
      B.tris = P.tris.as<LTri>() + D.tri_off;
      B.nodes = P.nodes.as<BNode8>() + D.node_off;
      B.leaves = P.leaves.as<NodeLeaves>() + D.node_off;
      B.nf = D.num_tris;
      B.nv = (int)src.numVerts(d);
      B.node_cap = (int)nodeCap(D.num_tris);
      B.cnt = (uint32_t*)(slot + SL.cnt);
      B.off = B.cnt + (B.nv + 1);
      B.adj = (uint32_t*)(slot + SL.adj);
      B.rank = (uint32_t*)(slot + SL.rank);
      B.bmm = (uint32_t*)(slot + SL.bmm);
      for (int k = 0; k < 2; ++k) {
        B.keys[k] = (uint32_t*)(slot + SL.keys[k]);
        B.vals[k] = (uint32_t*)(slot + SL.vals[k]);
        B.front[k] = (int*)(slot + SL.front[k]);
      }
      B.hist = (uint32_t*)(slot + SL.hist);
      B.rpre = (float*)(slot + SL.rpre);
      B.rsuf = (float*)(slot + SL.rsuf);
      B.rbox8 = (float*)(slot + SL.rbox8);
      B.rtab = (float*)(slot + SL.rtab);
      B.leafbox = (float*)(slot + SL.lb);
      B.innerbox = (float*)(slot + SL.ib);
      B.tree = (int4*)(slot + SL.tree);
      B.cc = M->levels.as<int>() + (size_t)d * kLevelWords;
      hv[d] = ScanJob{B.cnt, B.off, (uint32_t*)(slot + SL.vsums), (long long)B.nv + 1};
      hh[d] = ScanJob{B.hist, B.hist, (uint32_t*)(slot + SL.hsums), 256ll * rsTiles(B.nf)};
    }
    SPRAY_HIP(hipMemcpy(M->descs.p, host.data(), host.size(), hipMemcpyHostToDevice));
  }
  // domains [a, a + m) on stream st: normals, shading records, Morton order
  auto sortStage = [&](int a, int m, hipStream_t st) {
    int f = 0, v = 0;
    for (int d = a; d < a + m; ++d) {
      f = std::max(f, P.desc[d].num_tris);
      v = std::max(v, (int)src.numVerts(d));
    }
    const BuildDom* G = dev + a;
    auto grid = [&](long long n) { return dim3((unsigned)gridFor(n, 256), (unsigned)m); };
    kVertClear<<<grid(v + 1ll), 256, 0, st>>>(G);
    kVertCount<<<grid(3ll * f), 256, 0, st>>>(G);
    exclusiveScanMany(vscan + a, m, (long long)v + 1, st);
    kVertFill<<<grid(3ll * f), 256, 0, st>>>(G);
    kVertNormal<<<grid(v), 256, 0, st>>>(G);
    // Morton codes (kFaceShade sets the centroid bounds' starting values)
    kFaceShade<<<grid(f), 256, 0, st>>>(G);
    kCentroidBounds<<<dim3((unsigned)std::min(gridFor(f, 256), kBoundsGrid), (unsigned)m), 256, 0, st>>>(G);
    kMorton<<<grid(f), 256, 0, st>>>(G);
    const dim3 tiles((unsigned)std::max(1, rsTiles(f)), (unsigned)m);
    for (int pass = 0; pass < 4; ++pass) {
      kRsHist<<<tiles, kRsBlock, 0, st>>>(G, pass);
      exclusiveScanMany(hscan + a, m, 256ll * rsTiles(f), st);
      kRsScatter<<<tiles, kRsBlock, 0, st>>>(G, pass);
    }
    return f;
  };
  // the same domains' leaves and Karras hierarchies (f: the most triangles),
  // inner boxes as unions over leaf ranges; one-leaf roots are written
  auto treeStage = [&](int a, int m, int f, hipStream_t st) {
    const BuildDom* G = dev + a;
    auto grid = [&](long long n) { return dim3((unsigned)gridFor(n, 256), (unsigned)m); };
    kLeaves<<<grid(f), 256, 0, st>>>(G, nullptr);
    kKarras<<<grid(f), 256, 0, st>>>(G);
    const long long nblk = rangeBlocks(f);
    kLeafScan<<<grid(nblk * 64), 256, 0, st>>>(G);
    for (int j = 1; j < rangeLevels(f); j += 2)  // two levels per launch
      kRangeLevel2<<<grid(nblk - (1ll << j) + 1), 256, 0, st>>>(G, j);
    kRangeBoxes<<<grid(f - 1), 256, 0, st>>>(G);
    for (int d = a; d < a + m; ++d)
      if (P.desc[d].num_tris <= kLeafMax) {
        kTinyRoot<<<1, 8, 0, st>>>(dev + d);
        P.desc[d].num_nodes = 1;
        P.bvh_depth[d] = 1;
      }
  };
  // level l holds at most 8^l items (one root, at most eight children per item)
  auto collapseBlocks = [](int f, int l, int m) {
    const int most = std::min(gridFor(std::max(1, f / (kLeafMax + 1)), 32), 4096 / m);
    return (unsigned)(l < 8 ? std::min<long long>(most, ((1ll << (3 * l)) + 31) / 32) : most);
  };
  // Collapse of domain d's binary tree under `root`, kLevelBatch levels per
  // host wait (a level past the last finds 0 items); returns the number of
  // levels with items (kMaxLevels + 1 when deeper than kMaxLevels).
  auto collapseChecked = [&](int d, int root, hipStream_t st) {
    const BuildDom* G = dev + d;
    kCollapseInit<<<1, 64, 0, st>>>(G, root);
    for (int done = 0;;) {
      const int upto = std::min(done + kLevelBatch, kMaxLevels);
      for (int l = done; l < upto; ++l) kCollapseLevel<<<collapseBlocks(P.desc[d].num_tris, l, 1), 256, 0, st>>>(G, l);
      done = upto;
      int h[kLevelWords];
      SPRAY_HIP(hipMemcpyAsync(h, M->levels.as<int>() + (size_t)d * kLevelWords, sizeof(h), hipMemcpyDeviceToHost, st));
      SPRAY_HIP(hipStreamSynchronize(st));
      if (h[1]) throw StatusError(SPRAY_ERR_CAPACITY, "BVH node capacity exceeded");
      if (h[2 + done] == 0 || done == kMaxLevels) {
        int depth = 0;
        P.desc[d].num_nodes = 0;
        while (depth < done && h[2 + depth] > 0) P.desc[d].num_nodes += h[2 + depth++];
        return h[2 + done] > 0 ? kMaxLevels + 1 : depth;
      }
    }
  };
  auto fitsStack = [](int depth) { return depth <= kStackMax; };
  PlocScratch PS;
  if (!multi && c->bvh_builder == 1) PS.reserve(maxf);
  // one domain with host-checked levels (PLOC, paged pools, single domains,
  // domains deeper than the levels their group launched)
  auto buildOne = [&](int d, bool ploc) {
    DomainDesc& D = P.desc[d];
    const int nf = D.num_tris;
    const long long nv = src.numVerts(d);
    if (paged) {
      src.fill(c, d, P.vtx.as<float>(), P.face.as<uint32_t>(), P.rgb.as<uint32_t>(), s);
      src.check(c);
    }
    const BuildDom* G = dev + d;
    sortStage(d, 1, s);
    int depth = nf <= kLeafMax ? 1 : -1;
    if (ploc && depth < 0) {
      // PLOC passes until one cluster is left
      const char* slot = M->slots.as<char>();  // one-domain builds use slot 0
      int4* T = (int4*)(slot + SL.tree);
      float* inner = (float*)(slot + SL.ib);
      const uint32_t* va = (const uint32_t*)(slot + SL.vals[0]);
      const float* vtx = P.vtx.as<float>() + D.vtx_off * 3;
      const uint32_t* face = P.face.as<uint32_t>() + D.face_off * 3;
      int* cid = PS.pc.as<int>();
      int* cid2 = PS.pc2.as<int>();
      float* cbox = PS.pb.as<float>();
      float* cbox2 = PS.pb2.as<float>();
      int* nn = PS.pnn.as<int>();
      int* icount = PS.pcnt.as<int>();
      uint32_t* mflag = PS.pmf.as<uint32_t>();
      uint32_t* kflag = PS.pkf.as<uint32_t>();
      uint32_t* mpos = PS.pmp.as<uint32_t>();
      uint32_t* kpos = PS.pkp.as<uint32_t>();
      kPlocInit<<<gridFor(nf, 256), 256, 0, s>>>(vtx, face, nf, va, cid, cbox);
      std::vector<int> pass_base{0};
      int n = nf, made = 0;
      bool ok = true;
      while (n > 1) {
        kPlocNearest<<<(n + kPlocBlock - 1) / kPlocBlock, kPlocBlock, 0, s>>>(cbox, n, nn);
        kPlocFlags<<<gridFor(n + 1, 256), 256, 0, s>>>(nn, n, mflag, kflag);
        exclusiveScan(mflag, mpos, n + 1, s);
        exclusiveScan(kflag, kpos, n + 1, s);
        kPlocMerge<<<gridFor(n, 256), 256, 0, s>>>(nn, n, cid, cbox, mpos, kpos, made, cid2, cbox2,
                                                    T, inner, icount);
        uint32_t h[2];
        SPRAY_HIP(hipMemcpyAsync(&h[0], mpos + n, 4, hipMemcpyDeviceToHost, s));
        SPRAY_HIP(hipMemcpyAsync(&h[1], kpos + n, 4, hipMemcpyDeviceToHost, s));
        SPRAY_HIP(hipStreamSynchronize(s));
        if (h[0] == 0 || (int)h[1] != n - (int)h[0]) {  // no progress: non-finite boxes
          ok = false;
          break;
        }
        made += (int)h[0];
        pass_base.push_back(made);
        n = (int)h[1];
        std::swap(cid, cid2);
        std::swap(cbox, cbox2);
      }
      if (ok) {
        // depth-first leaf order: roots of later passes first
        const int root = made - 1;
        uint32_t* perm = PS.pperm.as<uint32_t>();
        SPRAY_HIP(hipMemsetAsync(&T[root].z, 0, 4, s));
        for (int p = (int)pass_base.size() - 1; p > 0; --p) {
          int lo = pass_base[p - 1], hi = pass_base[p];
          kPlocRanges<<<gridFor(hi - lo, 256), 256, 0, s>>>(lo, hi, T, icount, perm);
        }
        uint32_t* order = PS.pord.as<uint32_t>();
        kComposeOrder<<<gridFor(nf, 256), 256, 0, s>>>(perm, va, nf, order);
        kLeaves<<<gridFor(nf, 256), 256, 0, s>>>(G, order);
        depth = collapseChecked(d, root, s);
        if (!fitsStack(depth)) depth = -1;
      }
    }
    if (depth < 0 || nf <= kLeafMax) {
      treeStage(d, 1, nf, s);
      if (nf > kLeafMax) {
        depth = collapseChecked(d, 0, s);
        if (!fitsStack(depth))
          throw StatusError(SPRAY_ERR_CAPACITY, "BVH too deep for the traversal stack");
      }
    }
    P.bvh_depth[d] = depth;
    if (paged) {  // the finished image goes to pinned host memory, the normals to the host
      char* dst = (char*)P.h_image + P.h_image_off[d];
      const ImageLayout L(D.num_nodes, nf, nv);
      auto put = [&](size_t off, const void* src, size_t n) {
        SPRAY_HIP(hipMemcpyAsync(dst + off, src, n, hipMemcpyDeviceToHost, s));
      };
      put(0, P.nodes.as<BNode8>() + D.node_off, (size_t)D.num_nodes * sizeof(BNode8));
      put(L.leaves, P.leaves.as<NodeLeaves>() + D.node_off, (size_t)D.num_nodes * sizeof(NodeLeaves));
      if (L.indexed) {
        uint32_t* order = (uint32_t*)(M->slots.as<char>() + SL.keys[1]);  // (the sort is done with it)
        kPrimIds<<<gridFor(nf, 256), 256, 0, s>>>(P.tris.as<LTri>() + D.tri_off, nf, order);
        put(L.order, order, (size_t)nf * 4);
        put(L.face, P.face.p, (size_t)nf * 12);
        put(L.vtx, P.vtx.p, (size_t)nv * 12);
        put(L.nrm, P.nrm.p, (size_t)nv * 12);
        put(L.rgb, P.rgb.p, (size_t)nv * 4);
      } else {
        put(L.tris, P.tris.as<LTri>() + D.tri_off, (size_t)nf * sizeof(LTri));
        put(L.shade, P.fshade.as<float4>() + D.shade_off * 3, (size_t)nf * 48);
      }
      P.h_nrm[d].resize((size_t)nv * 3);
      SPRAY_HIP(hipMemcpyAsync(P.h_nrm[d].data(), P.nrm.p, (size_t)nv * 12, hipMemcpyDeviceToHost, s));
      SPRAY_HIP(hipStreamSynchronize(s));
    }
  };
  if (!multi) {
    for (int d = 0; d < nd; ++d) buildOne(d, c->bvh_builder == 1);
  } else {
    std::vector<int> launched(nd, 0);  // collapse levels launched per domain
    {
      // pipeline 0 on s, the others on their own streams
      StreamSet side(std::min(K, ngroups) - 1, s);
      for (int g = 0; g < ngroups; ++g) {
        const int a = g * GN, m = std::min(GN, nd - a), k = g % K;
        hipStream_t st = k == 0 ? s : side[k - 1];
        const int f = sortStage(a, m, st);
        treeStage(a, m, f, st);
        int levels = prev_depth.empty() ? kMaxLevels : 1;
        if (!prev_depth.empty())
          for (int d = a; d < a + m; ++d) levels = std::max(levels, std::min(kMaxLevels, prev_depth[d] + 4));
        kCollapseInit<<<dim3(1, (unsigned)m), 64, 0, st>>>(dev + a, 0);
        for (int l = 0; l < levels; ++l)
          kCollapseLevel<<<dim3(collapseBlocks(f, l, m), (unsigned)m), 256, 0, st>>>(dev + a, l);
        for (int d = a; d < a + m; ++d) launched[d] = levels;
        SPRAY_HIP(hipGetLastError());
      }
    }  // waits for the side streams
    SPRAY_HIP(hipStreamSynchronize(s));  // pipeline 0
    std::vector<int> h((size_t)nd * kLevelWords);
    SPRAY_HIP(hipMemcpy(h.data(), M->levels.p, h.size() * 4, hipMemcpyDeviceToHost));
    std::vector<int> redo;
    for (int d = 0; d < nd; ++d) {
      if (P.desc[d].num_tris <= kLeafMax) continue;  // one-leaf root, written directly
      const int* cc = &h[(size_t)d * kLevelWords];
      if (cc[1]) throw StatusError(SPRAY_ERR_CAPACITY, "BVH node capacity exceeded");
      if (cc[2 + launched[d]] > 0) {  // items left after the last launched level
        if (launched[d] >= kMaxLevels)
          throw StatusError(SPRAY_ERR_CAPACITY, "BVH too deep for the traversal stack");
        redo.push_back(d);
        continue;
      }
      int depth = 0, nodes = 0;
      while (depth < launched[d] && cc[2 + depth] > 0) nodes += cc[2 + depth++];
      if (!fitsStack(depth))
        throw StatusError(SPRAY_ERR_CAPACITY, "BVH too deep for the traversal stack");
      P.desc[d].num_nodes = nodes;
      P.bvh_depth[d] = depth;
    }
    for (int d : redo) buildOne(d, false);  // deeper than last time: host-checked
  }
  SPRAY_HIP(hipStreamSynchronize(s));
  long long used = 0;
  for (auto& D : P.desc) used += D.num_nodes;
  P.total_nodes = used;
  if (paged) {
    // the last `capacity` domains built stay in their blocks (least recently
    // built first); the raw-mesh staging arrays are no longer needed
    std::vector<std::pair<int, int>> resident;
    for (int d = std::max(0, nd - P.capacity); d < nd; ++d) resident.push_back({d, d % P.capacity});
    for (DevBuf* b : {&P.vtx, &P.face, &P.rgb, &P.nrm}) b->release();
    P.d_desc.reserve(sizeof(DomainDesc) * nd);
    SPRAY_HIP(hipMemcpy(P.d_desc.p, P.desc.data(), sizeof(DomainDesc) * nd, hipMemcpyHostToDevice));
    poolInitPaging(c, resident);
  } else {
    P.d_desc.reserve(sizeof(DomainDesc) * nd);
    SPRAY_HIP(hipMemcpy(P.d_desc.p, P.desc.data(), sizeof(DomainDesc) * nd, hipMemcpyHostToDevice));
  }
  P.build_ms =
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start).count();
}

// ---------------------------------------------------------------------------
// Batch queries (parity entry points)
constexpr int kQBlock = 256;

// A persistent grid: wave w takes rays [w * range, (w + 1) * range) and then
// ranges from the counter; finished lanes take the wave's next rays once
// kQRefill are idle.  With fewer rays than lanes the rays are spread over all
// the waves, kQMinRange or more each, and idle lanes help (travShare).
// Bound, as the frame's trace kernel is, by vector instructions and by the
// longest rays at the end.  Against one block of 256 rays a compute unit, each
// wave in step with its longest ray (as many blocks as overflow stacks of the
// greatest depth fitted the static scratch): 3 M closest hits among 524 k
// triangles 2275 -> 625 us (4.8 G rays/s), 1 M any hits among 180 k 695 -> 241
// us, 1500 closest hits 50 -> 25 us (8 rays a wave 36, 2 and 1 rays 28).
constexpr int kQRefill = 16;
constexpr uint32_t kQMinRange = 4;
__global__ void __launch_bounds__(kQBlock, 4) kTraceRays(
    const BNode8* __restrict__ nodes, const NodeLeaves* __restrict__ leaves, int num_nodes,
    const LTri* __restrict__ tris, const float* __restrict__ org, const float* __restrict__ dir, const float* __restrict__ tnear, const float* __restrict__ tfar,
    uint32_t n, uint32_t range, int mode, float* t_o, float* u_o, float* v_o, int* prim_o,
    uint32_t* ovf, uint32_t ovf_words, uint32_t* ctr, int* err) {
  __shared__ __align__(16) uint32_t lds[(kQBlock / 64) * kTravLdsWords];
  const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t* area = lds + w * kTravLdsWords;
  LaneStack st;
  st.init(area, ovf, ovf_words);
  TravCount tc;
  TravState s;
  const unsigned long long dyn0 = (unsigned long long)gridDim.x * (kQBlock / 64) * range;
  unsigned long long cur = (unsigned long long)(blockIdx.x * (kQBlock / 64) + w) * range;
  unsigned long long end = min(cur + range, (unsigned long long)n);
  bool active = false, helping = false, shared = false, exhausted = cur >= n;
  uint32_t ray = 0;
  while (true) {
    bool done = active && travDone(s);
    if (shared) done = !travHelped(s, helping, area) && done;
    const unsigned long long dm = __ballot(done);
    unsigned long long idle = __ballot(!active || done);
    const int nidle = __popcll(idle), nready = exhausted ? __popcll(dm) : nidle;
    if (dm != 0ull && (nready >= kQRefill || nidle == 64)) {
      if (done) {
        active = false;
        if (mode == 0) {
          t_o[ray] = s.tlim;
          u_o[ray] = s.u;
          v_o[ray] = s.v;
          prim_o[ray] = s.prim;
        } else {
          prim_o[ray] = s.prim > 0 ? 1 : 0;
        }
      }
    }
    if (!exhausted && (nidle >= kQRefill || nidle == 64)) {
      if (cur >= end) {  // the next range
        cur = n;
        if (dyn0 < n) {
          uint32_t a = 0;
          if (__lane_id() == 0) a = atomicAdd(ctr, 1u);
          cur = dyn0 + (unsigned long long)__builtin_amdgcn_readfirstlane(a) * range;
        }
        end = min(cur + range, (unsigned long long)n);
        if (cur >= n) exhausted = true;
      }
      idle = __ballot(!active);
      if (!exhausted) {
        const unsigned long long i = cur + (unsigned long long)__popcll(idle & ((1ull << __lane_id()) - 1ull));
        if (!active && i < end) {
          ray = (uint32_t)i;
          const size_t q = (size_t)ray * 3;
          float o[3] = {org[q], org[q + 1], org[q + 2]};
          float d[3] = {dir[q], dir[q + 1], dir[q + 2]};
          travInit(s, 0u, 0u, num_nodes, o, d, tnear[ray], tfar[ray], mode != 0, st);
          active = true;
        }
        cur = min(cur + (unsigned long long)__popcll(idle), end);
      }
    }
    if (__ballot(active) == 0ull) {
      if (exhausted) break;
      continue;
    }
    const bool live = (active || helping) && !travDone(s);
    travNodePhase(s, st, tc, live, nodes);
    travLeafPhase(s, st, tc, live, leaves, tris, area);
    if (shared) travFollow(s, helping);
    if (exhausted) {
      helping = helping && !travDone(s);
      if (travShare(s, st, !active && !helping, (active || helping) && !travDone(s), area)) helping = true;
      shared = __ballot(helping) != 0ull;
    }
  }
  if (st.overflowed()) __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void kClearWord(uint32_t* w) { *w = 0u; }

// A query's launch: blocks, rays a wave takes at once, and overflow words per
// lane.  A tree of `depth` levels leaves at most one group per level on the
// stack, so most trees need no overflow; with a bound on the overflow memory
// (max_words) a deep tree runs with fewer lanes.
struct QueryLaunch {
  int grid;
  uint32_t range, words;
};
static QueryLaunch queryLaunch(Ctx* c, size_t n, int domain, size_t max_words) {
  QueryLaunch q;
  const int depth = c->pool.bvh_depth[domain];
  q.words = 2u * (uint32_t)std::max(0, std::min(depth + 2 - kRing, kOverflow));
  if (c->q_resident == 0) {
    int per_cu = 0;
    SPRAY_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kTraceRays, kQBlock, 0));
    int cus = 0;
    SPRAY_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
    c->q_resident = std::max(1, per_cu) * std::max(1, cus);
  }
  long long grid = c->q_resident;
  if (q.words) grid = std::min<long long>(grid, (long long)(max_words / ((size_t)q.words * kQBlock)));
  const long long waves = kQBlock / 64;
  grid = std::max(1ll, std::min(grid, ((long long)n + waves * kQMinRange - 1) / (waves * (long long)kQMinRange)));
  q.grid = (int)grid;
  // at most 64 rays a wave while those cover every ray, else 64 or 256 at a time
  const long long per_wave = ((long long)n + grid * waves - 1) / (grid * waves);
  q.range = (uint32_t)(per_wave <= 64 ? std::max<long long>(per_wave, kQMinRange) : per_wave >= 1024 ? 256 : 64);
  return q;
}

// One launch, waited for.  The work counter is cleared only where the grid does
// not take every ray at once, and the error flag, which the kernel sets in host
// memory, needs no copy: a call with 1500 rays 57.5 -> 41.4 us.
static void runQuery(Ctx* c, const QueryLaunch& q, const DomainDesc& D, const float* d_org, const float* d_dir,
                     const float* d_tnear, const float* d_tfar, uint32_t n, int mode, float* d_t, float* d_u,
                     float* d_v, int* d_prim, uint32_t* ovf) {
  uint32_t* ctr = c->q_ctr.as<uint32_t>();
  if ((unsigned long long)q.grid * (kQBlock / 64) * q.range < n) kClearWord<<<1, 1, 0, c->stream>>>(ctr);
  *c->q_err = 0;
  kTraceRays<<<q.grid, kQBlock, 0, c->stream>>>(
      c->pool.nodes.as<BNode8>() + D.node_off, c->pool.leaves.as<NodeLeaves>() + D.node_off,
      D.num_nodes, c->pool.tris.as<LTri>() + D.tri_off, d_org, d_dir, d_tnear, d_tfar, n, q.range, mode, d_t, d_u, d_v, d_prim,
      ovf, q.words, ctr, c->q_err);
  SPRAY_HIP(hipGetLastError());
  SPRAY_HIP(hipStreamSynchronize(c->stream));
  if (*(volatile int*)c->q_err) throw StatusError(SPRAY_ERR_CAPACITY, "traversal stack overflow or corrupt BVH");
}

void traceRaysDevice(Ctx* c, const float* d_org, const float* d_dir, const float* d_tnear,
                     const float* d_tfar, size_t n, int mode, int domain, float* d_t, float* d_u,
                     float* d_v, int* d_prim) {
  const DomainDesc& D = c->pool.desc[domain];
  // ray numbers are 32 bits in the kernel: longer batches go in parts
  constexpr size_t kPart = (size_t)1 << 30;
  for (size_t at = 0; at < n; at += kPart) {
    const size_t m = std::min(kPart, n - at);
    const QueryLaunch q = queryLaunch(c, m, domain, ~(size_t)0);
    const size_t ovf_bytes = (size_t)q.grid * kQBlock * q.words * 4;
    c->q_out.reserve(ovf_bytes + 64);
    runQuery(c, q, D, d_org + at * 3, d_dir + at * 3, d_tnear + at, d_tfar + at, (uint32_t)m, mode, d_t + at,
             d_u + at, d_v + at, d_prim + at, c->q_out.as<uint32_t>());
  }
}

// ---------------------------------------------------------------------------
// spray_trace_rays_device: the same query on caller-owned device arrays with
// no allocation.  Its scratch (the traversal overflow stacks) is this
// file-scope array, which every GPU the library runs on holds until the process ends.  Host
// code never uses the array's name as an address: scratchInit looks up each
// device's copy once (hipGetSymbolAddress) and keeps the pointer per device.
constexpr size_t kScratchStackBytes = (size_t)28 << 20;
static __device__ __align__(256) unsigned char scratch[kScratchStackBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch[kMaxDevices] = {};
}  // namespace

void scratchInit(int device) {
  if (device < 0 || device >= kMaxDevices)
    throw StatusError(SPRAY_ERR_DEVICE, "device ordinal beyond the scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch[device]) return;
  int cur = 0;
  SPRAY_HIP(hipGetDevice(&cur));
  SPRAY_HIP(hipSetDevice(device));
  void* ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  (void)hipSetDevice(cur);
  if (e != hipSuccess || ptr == nullptr)
    throw DeviceError(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
  g_scratch[device] = ptr;
}

size_t scratchBytes() { return kScratchStackBytes; }

void traceRaysNoAlloc(Ctx* c, const float* d_org, const float* d_dir, const float* d_tnear,
                      const float* d_tfar, size_t n, int mode, int domain, float* d_t, float* d_u,
                      float* d_v, int* d_prim) {
  void* base = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    base = (c->device >= 0 && c->device < kMaxDevices) ? g_scratch[c->device] : nullptr;
  }
  if (!base) throw StatusError(SPRAY_ERR_STATE, "scratch not set up on this device");
  const DomainDesc& D = c->pool.desc[domain];
  const QueryLaunch q = queryLaunch(c, n, domain, kScratchStackBytes / 4);
  runQuery(c, q, D, d_org, d_dir, d_tnear, d_tfar, (uint32_t)n, mode, d_t, d_u, d_v, d_prim, (uint32_t*)base);
}

// Domain list per ray: brute force over the domain AABBs staged in LDS,
// insertion into a (t, id)-sorted list of at most maxk entries.
constexpr int kMaxList = 64;
__global__ void __launch_bounds__(256) kDomainList(const DomainDesc* __restrict__ desc, int nd,
                                                   const float* __restrict__ org,
                                                   const float* __restrict__ dir, long long n,
                                                   int maxk, int* counts, int* ids, float* ts) {
  extern __shared__ float boxes[];  // 6 floats per domain
  for (int i = threadIdx.x; i < nd; i += blockDim.x)
    for (int k = 0; k < 3; ++k) {
      boxes[i * 6 + k] = desc[i].lo[k];
      boxes[i * 6 + 3 + k] = desc[i].hi[k];
    }
  __syncthreads();
  for (long long r = blockIdx.x * (long long)blockDim.x + threadIdx.x; r < n;
       r += (long long)gridDim.x * blockDim.x) {
    float o[3] = {org[r * 3], org[r * 3 + 1], org[r * 3 + 2]};
    float d[3] = {dir[r * 3], dir[r * 3 + 1], dir[r * 3 + 2]};
    int cnt = 0, kept = 0;
    int* my_ids = ids + r * maxk;
    float* my_ts = ts + r * maxk;
    for (int i = 0; i < nd; ++i) {
      float tmin;
      if (!slabDomain(&boxes[i * 6], &boxes[i * 6 + 3], o, d, &tmin)) continue;
      ++cnt;
      // insert (tmin, i) keeping the maxk smallest, ordered by (t, id)
      int j = kept;
      if (kept == maxk) {
        float lt = my_ts[maxk - 1];
        if (!(tmin < lt)) continue;  // ids ascend, so equal t keeps the earlier id
        j = maxk - 1;
      } else {
        ++kept;
      }
      while (j > 0 && my_ts[j - 1] > tmin) {
        my_ts[j] = my_ts[j - 1];
        my_ids[j] = my_ids[j - 1];
        --j;
      }
      my_ts[j] = tmin;
      my_ids[j] = i;
    }
    counts[r] = cnt;
  }
}

void domainListDevice(Ctx* c, const float* d_org, const float* d_dir, size_t n, int maxk,
                      int* d_counts, int* d_ids, float* d_ts) {
  int nd = c->pool.ndomains;
  int grid = std::min<long long>(4096, std::max<long long>(1, ((long long)n + 255) / 256));
  kDomainList<<<grid, 256, nd * 6 * sizeof(float), c->stream>>>(
      c->pool.d_desc.as<DomainDesc>(), nd, d_org, d_dir, (long long)n, maxk, d_counts, d_ids, d_ts);
  SPRAY_HIP(hipGetLastError());
  SPRAY_HIP(hipStreamSynchronize(c->stream));
}

}  // namespace spray
