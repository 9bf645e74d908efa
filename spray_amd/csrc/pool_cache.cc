// Paged domain pool: an LRU cache of domain blocks in HBM over per-domain
// images in pinned host memory.
//
// Replaces the reference's LruCache (render/lru_cache.cc:41-171) and
// TriMeshBuffer::load (render/trimesh_buffer.cc:117-169): the reference
// reads a missing domain's PLY file and builds its Embree scene; here every
// domain is built once at load time and its image (BVH nodes, mesh, leaf
// order) is kept in pinned host memory, so a miss is one host-to-HBM copy into
// a stage and one launch that unpacks it into the evicted block.  There are two
// stages, taken in turn, each with a stream on which its copy, its unpacking
// and the domain's descriptor follow one another.  The unpacking also waits for
// the last kernels that used the block (block_free) and for the block's last
// filling (block_ready), the descriptor for the load before; the trace stream
// waits for the block's own load.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ctx.h"

namespace spray {

void DomainPool::releasePaging() {
  for (hipEvent_t e : block_free) (void)hipEventDestroy(e);
  for (hipEvent_t e : block_ready) (void)hipEventDestroy(e);
  block_free.clear();
  block_ready.clear();
  if (h_image) (void)hipHostFree(h_image);
  if (h_desc_pinned) (void)hipHostFree(h_desc_pinned);
  for (int k = 0; k < 2; ++k) {
    if (load_stream[k]) (void)hipStreamDestroy(load_stream[k]);
    load_stream[k] = nullptr;
    stage[k].release();
  }
  next_stage = 0;
  last_load = -1;
  h_image = nullptr;
  h_desc_pinned = nullptr;
  h_image_off.clear();
  h_nrm.clear();
  block_domain.clear();
  domain_block.clear();
  block_tick.clear();
  pending.clear();
  pinned.clear();
  paged = false;
  capacity = 0;
  tick = hits = misses = bytes_in = 0;
}

// A staged image into a block's arrays: the same records that the build's
// kLeaves and kFaceShade write.  The host link bounds a miss (50 GB/s), so
// what crosses it is the mesh: 53 bytes a triangle of a mesh with two
// triangles a vertex where the finished arrays have 120.  A 400x300 4 spp frame
// of 48 domains with 12 cached (168 misses) 28.1 -> 13.1 ms, of which the
// unpacking, beside the copies, takes 1.5 ms.  A mesh of 3 vertices a triangle
// would take 100 bytes of 96: its image holds the finished arrays.
__global__ void __launch_bounds__(256) kUnpack(const char* __restrict__ img, ImageLayout L, int nn, int nf,
                                               BNode8* nodes, NodeLeaves* leaves, LTri* tris, float4* fshade) {
  const long long i0 = blockIdx.x * (long long)blockDim.x + threadIdx.x, n = (long long)gridDim.x * blockDim.x;
  auto copy = [&](void* dst, size_t off, long long words) {
    for (long long i = i0; i < words; i += n) ((float4*)dst)[i] = ((const float4*)(img + off))[i];
  };
  copy(nodes, 0, nn * 4ll);
  copy(leaves, L.leaves, nn * 2ll);
  if (!L.indexed) {
    copy(tris, L.tris, nf * 3ll);
    copy(fshade, L.shade, nf * 3ll);
    return;
  }
  const uint32_t *order = (const uint32_t*)(img + L.order), *face = (const uint32_t*)(img + L.face),
                 *rgb = (const uint32_t*)(img + L.rgb);
  const float *vtx = (const float*)(img + L.vtx), *nrm = (const float*)(img + L.nrm);
  for (long long i = i0; i < nf; i += n) {
    const uint32_t p = order[i];
    const float* a = vtx + (size_t)face[p * 3] * 3;
    const float* b = vtx + (size_t)face[p * 3 + 1] * 3;
    const float* c = vtx + (size_t)face[p * 3 + 2] * 3;
    float4* t = (float4*)(tris + i);
    t[0] = make_float4(a[0], a[1], a[2], __int_as_float((int)p));
    t[1] = make_float4(b[0], b[1], b[2], 0.f);
    t[2] = make_float4(c[0], c[1], c[2], 0.f);
    for (int k = 0; k < 3; ++k) {
      const uint32_t v = face[i * 3 + k];
      fshade[i * 3 + k] = make_float4(nrm[(size_t)v * 3], nrm[(size_t)v * 3 + 1], nrm[(size_t)v * 3 + 2],
                                      __uint_as_float(rgb[v]));
    }
  }
}

// Points domain d's descriptor at block b (host copy and device copy, the
// latter ordered on stream s).
static void bindBlock(DomainPool& P, int d, int b, hipStream_t s) {
  DomainDesc& D = P.desc[d];
  D.node_off = (long long)b * P.block_nodes;
  D.tri_off = (long long)b * P.block_tris;
  D.shade_off = (long long)b * P.block_tris;
  P.h_desc_pinned[d] = D;
  SPRAY_HIP(hipMemcpyAsync(P.d_desc.as<DomainDesc>() + d, P.h_desc_pinned + d, sizeof(DomainDesc),
                           hipMemcpyHostToDevice, s));
}

// LruCache::load (lru_cache.cc:65-171): a hit promotes the domain's block to
// most recently used; a miss takes the next free block or evicts the least
// recently used one (never `keep`'s block) and copies the image in.
// Returns the block.  A domain loaded ahead of its access (pending) is not
// counted again when the access comes.
static int lruLoad(Ctx* c, int d, int keep) {
  DomainPool& P = c->pool;
  if (P.pending[d]) {
    P.pending[d] = 0;
    return P.domain_block[d];
  }
  int b = P.domain_block[d];
  if (b >= 0) {
    ++P.hits;
    P.block_tick[b] = ++P.tick;
    return b;
  }
  ++P.misses;
  int victim = -1;
  for (int i = 0; i < P.capacity; ++i) {
    if (P.block_domain[i] < 0) {  // not full: blocks fill in order
      victim = i;
      break;
    }
    if ((keep >= 0 && P.block_domain[i] == keep) || P.pinned[P.block_domain[i]]) continue;
    if (victim < 0 || P.block_tick[i] < P.block_tick[victim]) victim = i;
  }
  if (victim < 0) throw StatusError(SPRAY_ERR_STATE, "no evictable cache block");
  if (P.block_domain[victim] >= 0) P.domain_block[P.block_domain[victim]] = -1;
  P.block_domain[victim] = d;
  P.domain_block[d] = victim;
  P.block_tick[victim] = ++P.tick;
  // Copy, unpacking and descriptor follow one another on the stage's stream;
  // the unpacking waits for the block's last users and its last filling, the
  // descriptor for the descriptor before it, so descriptors change in the
  // order of the loads.  (The domain's own last users are done by then: its
  // old block was unpacked into, or is this one.)  A stream per stage, not one
  // for the copies and one for the unpacking: the next image's copy starts
  // when its own stage is free and no unpacking waits for an event of the
  // copies (400x300 path trace of 4 samples, 48 domains, 12 blocks: 13.3 ->
  // 11.0 ms, and 17.0 -> 14.3 to 15.9 in a process whose other streams leave
  // the trace stream to share a hardware queue with a stage's; 1920x1080, 256
  // domains, 128 blocks: 877 -> 785 ms).
  const DomainDesc& D = P.desc[d];
  const char* src = (const char*)P.h_image + P.h_image_off[d];
  const ImageLayout L(D.num_nodes, D.num_tris, P.nverts[d]);
  const int k = P.next_stage;
  P.next_stage ^= 1;
  hipStream_t us = P.load_stream[k];
  SPRAY_HIP(hipMemcpyAsync(P.stage[k].p, src, L.bytes, hipMemcpyHostToDevice, us));
  SPRAY_HIP(hipStreamWaitEvent(us, P.block_free[victim], 0));
  SPRAY_HIP(hipStreamWaitEvent(us, P.block_ready[victim], 0));
  kUnpack<<<std::max(1, std::min((D.num_tris + 255) / 256, 2048)), 256, 0, us>>>(
      P.stage[k].as<char>(), L, D.num_nodes, D.num_tris, P.nodes.as<BNode8>() + (size_t)victim * P.block_nodes,
      P.leaves.as<NodeLeaves>() + (size_t)victim * P.block_nodes, P.tris.as<LTri>() + (size_t)victim * P.block_tris,
      P.fshade.as<float4>() + (size_t)victim * P.block_tris * 3);
  SPRAY_HIP(hipGetLastError());
  if (P.last_load >= 0) SPRAY_HIP(hipStreamWaitEvent(us, P.block_ready[P.last_load], 0));
  bindBlock(P, d, victim, us);
  SPRAY_HIP(hipEventRecord(P.block_ready[victim], us));
  P.last_load = victim;
  P.bytes_in += L.bytes;
  return victim;
}

void poolAcquire(Ctx* c, int d, hipStream_t s) {
  DomainPool& P = c->pool;
  if (!P.paged) return;
  const int b = lruLoad(c, d, -1);
  SPRAY_HIP(hipStreamWaitEvent(s, P.block_ready[b], 0));
}

void poolPrefetch(Ctx* c, int d, int keep) {
  DomainPool& P = c->pool;
  if (!P.paged || P.capacity < 2 || P.pending[d]) return;
  if (P.domain_block[d] >= 0) return;  // resident: its access is counted when it comes
  lruLoad(c, d, keep);
  P.pending[d] = 1;
}

void poolRelease(Ctx* c, int d, hipStream_t s) {
  DomainPool& P = c->pool;
  if (!P.paged) return;
  SPRAY_HIP(hipEventRecord(P.block_free[P.domain_block[d]], s));
}

// Sets up the cache after the build: `resident` lists the (domain, block)
// pairs the build left in HBM, least recently used first.
void poolInitPaging(Ctx* c, const std::vector<std::pair<int, int>>& resident) {
  DomainPool& P = c->pool;
  const int nd = P.ndomains;
  P.block_domain.assign(P.capacity, -1);
  P.domain_block.assign(nd, -1);
  P.block_tick.assign(P.capacity, 0);
  P.pending.assign(nd, 0);
  P.pinned.assign(nd, 0);
  size_t most = 0;
  for (int d = 0; d < nd; ++d)
    most = std::max(most, ImageLayout(P.desc[d].num_nodes, P.desc[d].num_tris, P.nverts[d]).bytes);
  for (int k = 0; k < 2; ++k) {
    P.stage[k].reserve(most + 64);
    SPRAY_HIP(hipStreamCreate(&P.load_stream[k]));
  }
  P.block_free.resize(P.capacity);
  P.block_ready.resize(P.capacity);
  for (int b = 0; b < P.capacity; ++b) {
    SPRAY_HIP(hipEventCreateWithFlags(&P.block_free[b], hipEventDisableTiming));
    SPRAY_HIP(hipEventCreateWithFlags(&P.block_ready[b], hipEventDisableTiming));
  }
  for (size_t i = 0; i < resident.size(); ++i) {
    const int d = resident[i].first, b = resident[i].second;
    P.block_domain[b] = d;
    P.domain_block[d] = b;
    P.block_tick[b] = ++P.tick;
  }
  if (!P.h_desc_pinned)
    SPRAY_HIP(hipHostMalloc((void**)&P.h_desc_pinned, sizeof(DomainDesc) * nd, hipHostMallocDefault));
  std::copy(P.desc.begin(), P.desc.end(), P.h_desc_pinned);
  P.hits = P.misses = P.bytes_in = 0;
}

}  // namespace spray
