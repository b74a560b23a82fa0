// pm_gather_lane.hip -- render with one lane per pixel and a per-lane kNN.
//
// Same inputs, outputs and neighbour sets as pm_gather.hip (the reference
// counterpart is photon_mapping_kernel, photonMappingKernel.cu:1409-1462, with
// computePixelColor :926-1017 and the gathers :314-389, :831-870), organised
// for throughput instead of per-query latency:
//  * a wave renders an 8x8 pixel tile, one pixel per lane, so the 64 queries
//    in flight are spatially coherent (neighbouring pixels, same march step);
//  * each lane keeps its k best (FP32 bits of d^2, photon index) keys in a
//    bounded max-heap in LDS (k <= 64 slots x 8 B per lane, slot-major so the
//    lanes of a wave touch consecutive banks);
//  * traversal is stackless: near-first depth-first search over the
//    heap-ordered tree using the implicit parent (h-1)/2 and each internal
//    node's point range, so no per-lane stack memory is needed;
//  * the volume query along the march is seeded with the bound
//    (r_prev + |q - q_prev|)^2 from the same lane's previous query; when fewer
//    than k keys fall under it the query is repeated with the full radius cap,
//    so the result is always the exact kNN set.
#include "pm_lane_knn.h"
#include "pm_lane_knn2.h"
#include "pm_lane_knn3.h"
#include "pm_tiles.h"

namespace pm {

// Radiance of pixel (px, py): the mean of its spp samples, compensated sum.
// heap: this wave's LDS heap, `slots` keys per lane (k <= slots).
template <bool FP64T, bool CONE>
__device__ __forceinline__ V3f lane_pixel(const Scene& sc, const RenderParams& rp, const GatherMap& gs,
                                          const GatherMap& gv, uint32_t* heap, int slots, int lane, uint32_t px,
                                          uint32_t py, uint32_t& nsurf, uint32_t& nvol) {
  LaneGather<CONE> g;
  g.gs = gs;
  g.gv = gv;
  g.hp.H = heap;
  g.hp.Lo = heap + slots * 64;
  g.hp.lane = lane;
  g.hp.k = 0;
  g.hp.size = 0;
  g.hg_g = sc.med.g;
  g.nsurf = 0u;
  g.nvol = 0u;
  g.prev_r = -1.0f;
  NSum3<float> acc;
  nsum3_init(acc);
  for (int s = 0; s < rp.spp; ++s) {
    V3f v = FP64T ? render_sample_t<float, double>(sc, rp, px, py, (uint32_t)s, g)
                  : render_sample_t<float, float>(sc, rp, px, py, (uint32_t)s, g);
    nsum3_add(acc, v);
  }
  nsurf = g.nsurf;
  nvol = g.nvol;
  return nsum3_get(acc) * (1.0f / (float)rp.spp);
}

// The same with the 4-byte-heap gather (pm_lane_knn2.h); heap: `64` slots of
// 4 bytes per lane.
template <bool FP64T, bool CONE>
__device__ __forceinline__ V3f lane_pixel2(const Scene& sc, const RenderParams& rp, const GatherMap& gs,
                                           const GatherMap& gv, uint32_t* heap, int lane, uint32_t px, uint32_t py,
                                           uint32_t& nsurf, uint32_t& nvol) {
  LaneGather2<CONE> g;
  g.gs = gs;
  g.gv = gv;
  g.hp.H = heap;
  g.hp.lane = lane;
  g.hp.k = 0;
  g.hp.size = 0;
  g.hg_g = sc.med.g;
  g.nsurf = 0u;
  g.nvol = 0u;
  g.prev_r = -1.0f;
  NSum3<float> acc;
  nsum3_init(acc);
  for (int s = 0; s < rp.spp; ++s) {
    V3f v = FP64T ? render_sample_t<float, double>(sc, rp, px, py, (uint32_t)s, g)
                  : render_sample_t<float, float>(sc, rp, px, py, (uint32_t)s, g);
    nsum3_add(acc, v);
  }
  nsurf = g.nsurf;
  nvol = g.nvol;
  return nsum3_get(acc) * (1.0f / (float)rp.spp);
}

// The same with the 2-byte-heap gather (pm_lane_knn3.h).
template <bool FP64T, bool CONE, int NB = 8>
__device__ __forceinline__ V3f lane_pixel3(const Scene& sc, const RenderParams& rp, const GatherMap& gs,
                                           const GatherMap& gv, uint16_t* heap, int lane, uint32_t px, uint32_t py,
                                           uint32_t& nsurf, uint32_t& nvol) {
  LaneGather3<CONE, NB> g;
  g.gs = gs;
  g.gv = gv;
  g.hp.H = heap;
  g.hp.lane = lane;
  g.hp.k = 0;
  g.hp.size = 0;
  g.hg_g = sc.med.g;
  g.nsurf = 0u;
  g.nvol = 0u;
  g.prev_r = -1.0f;
  NSum3<float> acc;
  nsum3_init(acc);
  for (int s = 0; s < rp.spp; ++s) {
    V3f v = FP64T ? render_sample_t<float, double>(sc, rp, px, py, (uint32_t)s, g)
                  : render_sample_t<float, float>(sc, rp, px, py, (uint32_t)s, g);
    nsum3_add(acc, v);
  }
  nsurf = g.nsurf;
  nvol = g.nvol;
  return nsum3_get(acc) * (1.0f / (float)rp.spp);
}

// One wave (one workgroup) per 8x8 tile of the crop; lane = pixel.
template <bool FP64T, bool CONE>
__global__ void __launch_bounds__(64) k_render_lane(RenderLaunch r) {
  extern __shared__ uint32_t heap_lds[];  // [2][64 slots][64 lanes]
  const int lane = lane_id();
  int lx, ly;
  if (!lane_tile(r, lane, lx, ly)) return;
  const uint32_t px = (uint32_t)(r.x0 + lx), py = (uint32_t)(r.y0 + ly);
  uint32_t ns, nv;
  V3f v = lane_pixel<FP64T, CONE>(r.sc, r.rp, r.gs, r.gv, heap_lds, 64, lane, px, py, ns, nv);
  store_pixel(r.rgb, r.u8, (size_t)ly * (size_t)r.w + (size_t)lx, v, r.exposure);
  if (r.counters) {
    atomicAdd(&r.counters[0], (unsigned long long)ns);
    atomicAdd(&r.counters[1], (unsigned long long)nv);
  }
}

// Gather mode 2: k_render_lane with the 4-byte heap (16 KB of LDS per wave).
template <bool FP64T, bool CONE>
__global__ void __launch_bounds__(64) k_render_lane2(RenderLaunch r) {
  extern __shared__ uint32_t heap_lds[];  // [64 slots][64 lanes]
  const int lane = lane_id();
  int lx, ly;
  if (!lane_tile(r, lane, lx, ly)) return;
  const uint32_t px = (uint32_t)(r.x0 + lx), py = (uint32_t)(r.y0 + ly);
  uint32_t ns, nv;
  V3f v = lane_pixel2<FP64T, CONE>(r.sc, r.rp, r.gs, r.gv, heap_lds, lane, px, py, ns, nv);
  store_pixel(r.rgb, r.u8, (size_t)ly * (size_t)r.w + (size_t)lx, v, r.exposure);
  if (r.counters) {
    atomicAdd(&r.counters[0], (unsigned long long)ns);
    atomicAdd(&r.counters[1], (unsigned long long)nv);
  }
}

// Gather mode 4: the 2-byte heap (8 KB of LDS per wave), leaf points loaded 4
// at a time, with the register budget of 5 waves per SIMD.
template <bool FP64T, bool CONE>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(5))) k_render_lane4(RenderLaunch r) {
  extern __shared__ uint16_t heap16_lds[];  // [64 slots][64 lanes]
  const int lane = lane_id();
  int lx, ly;
  if (!lane_tile(r, lane, lx, ly)) return;
  const uint32_t px = (uint32_t)(r.x0 + lx), py = (uint32_t)(r.y0 + ly);
  uint32_t ns, nv;
  V3f v = lane_pixel3<FP64T, CONE, 4>(r.sc, r.rp, r.gs, r.gv, heap16_lds, lane, px, py, ns, nv);
  store_pixel(r.rgb, r.u8, (size_t)ly * (size_t)r.w + (size_t)lx, v, r.exposure);
  if (r.counters) {
    atomicAdd(&r.counters[0], (unsigned long long)ns);
    atomicAdd(&r.counters[1], (unsigned long long)nv);
  }
}

hipError_t launch_render_lane4(const RenderLaunch& r, hipStream_t st) {
  if (r.w <= 0 || r.h <= 0) return hipSuccess;
  const unsigned tiles = lane_grid(r);
  size_t lds = 64 * 64 * sizeof(uint16_t);
  const bool fp64 = r.rp.fp64_transmittance != 0, cone = r.estimator == 1;
  if (fp64 && cone) hipLaunchKernelGGL((k_render_lane4<true, true>), dim3(tiles), dim3(64), lds, st, r);
  else if (fp64) hipLaunchKernelGGL((k_render_lane4<true, false>), dim3(tiles), dim3(64), lds, st, r);
  else if (cone) hipLaunchKernelGGL((k_render_lane4<false, true>), dim3(tiles), dim3(64), lds, st, r);
  else hipLaunchKernelGGL((k_render_lane4<false, false>), dim3(tiles), dim3(64), lds, st, r);
  return hipGetLastError();
}

hipError_t launch_render_lane2(const RenderLaunch& r, hipStream_t st) {
  if (r.w <= 0 || r.h <= 0) return hipSuccess;
  const unsigned tiles = lane_grid(r);
  size_t lds = 64 * 64 * sizeof(uint32_t);
  const bool fp64 = r.rp.fp64_transmittance != 0, cone = r.estimator == 1;
  if (fp64 && cone) hipLaunchKernelGGL((k_render_lane2<true, true>), dim3(tiles), dim3(64), lds, st, r);
  else if (fp64) hipLaunchKernelGGL((k_render_lane2<true, false>), dim3(tiles), dim3(64), lds, st, r);
  else if (cone) hipLaunchKernelGGL((k_render_lane2<false, true>), dim3(tiles), dim3(64), lds, st, r);
  else hipLaunchKernelGGL((k_render_lane2<false, false>), dim3(tiles), dim3(64), lds, st, r);
  return hipGetLastError();
}

hipError_t launch_render_lane(const RenderLaunch& r, hipStream_t st) {
  if (r.w <= 0 || r.h <= 0) return hipSuccess;
  const unsigned tiles = lane_grid(r);
  size_t lds = 2 * 64 * 64 * sizeof(uint32_t);
  const bool fp64 = r.rp.fp64_transmittance != 0, cone = r.estimator == 1;
  if (fp64 && cone) hipLaunchKernelGGL((k_render_lane<true, true>), dim3(tiles), dim3(64), lds, st, r);
  else if (fp64) hipLaunchKernelGGL((k_render_lane<true, false>), dim3(tiles), dim3(64), lds, st, r);
  else if (cone) hipLaunchKernelGGL((k_render_lane<false, true>), dim3(tiles), dim3(64), lds, st, r);
  else hipLaunchKernelGGL((k_render_lane<false, false>), dim3(tiles), dim3(64), lds, st, r);
  return hipGetLastError();
}

// Batched render: one persistent grid over the 8x8 tiles of every scene of a
// batch.  Each wave takes the next (scene, tile) item from a device work
// queue (an atomic counter over an item list ordered by decreasing expected
// cost) until the list is exhausted, so scenes of very different sizes keep
// all waves busy.  Per pixel the arithmetic is that of the one-scene lane
// render with the same gather (KB = 8: mode 1, 4: mode 2, 2: mode 4; mode 7 is
// k_render_batch_packet), so every scene's image is bit-identical to its own
// render in that mode.  heap_slots (32 or 64 keys per lane) and the key width
// size each wave's LDS heap.
template <bool FP64T, bool CONE, int KB>
__global__ void __launch_bounds__(256) k_render_batch(BatchRenderLaunch r) {
  extern __shared__ uint32_t lds[];
  const int lane = lane_id();
  const int wave = (int)uniform(threadIdx.x >> 6);  // wave-uniform: the LDS regions' addresses stay scalar
  const size_t heap_words = (size_t)r.heap_slots * 64u * KB / 4u;
  uint32_t* heap = lds + (size_t)wave * heap_words;
  unsigned long long ns_tot = 0, nv_tot = 0;
  for (;;) {
    uint32_t it = 0;
    if (lane == 0) it = atomicAdd(r.head, 1u);
    it = read_lane(it, 0);
    if (it >= r.nitems) break;
    const uint2 item = r.items[it];
    // wave-uniform scene and tile: scalar loads of the scene descriptor
    const BatchRenderScene& S = r.scenes[uniform(item.x)];
    const uint32_t tile = uniform(item.y);
    const int tiles_x = (S.w + 7) / 8;
    const int tx = (int)tile % tiles_x, ty = (int)tile / tiles_x;
    const int lx = tx * 8 + (lane & 7), ly = ty * 8 + (lane >> 3);
    if (lx < S.w && ly < S.h) {
      uint32_t ns, nv;
      V3f v;
      if (KB == 8)
        v = lane_pixel<FP64T, CONE>(S.sc, S.rp, S.gs, S.gv, heap, r.heap_slots, lane, (uint32_t)lx, (uint32_t)ly, ns,
                                    nv);
      else if (KB == 4)
        v = lane_pixel2<FP64T, CONE>(S.sc, S.rp, S.gs, S.gv, heap, lane, (uint32_t)lx, (uint32_t)ly, ns, nv);
      else
        v = lane_pixel3<FP64T, CONE, 4>(S.sc, S.rp, S.gs, S.gv, (uint16_t*)heap, lane, (uint32_t)lx, (uint32_t)ly, ns,
                                        nv);
      store_pixel(r.rgb + 3 * S.img_off, nullptr, (size_t)ly * (size_t)S.w + (size_t)lx, v, S.exposure);
      ns_tot += ns;
      nv_tot += nv;
    }
  }
  if (r.counters) {
    atomicAdd(&r.counters[0], ns_tot);
    atomicAdd(&r.counters[1], nv_tot);
  }
}

static size_t render_batch_lds_bytes(int block_threads, int heap_slots, int key_bytes) {
  return (size_t)(block_threads / 64) * ((size_t)heap_slots * 64u * (size_t)key_bytes);
}

template <int KB>
static const void* batch_kernel(int fp64, int cone) {
  if (fp64) return cone ? (const void*)k_render_batch<true, true, KB> : (const void*)k_render_batch<true, false, KB>;
  return cone ? (const void*)k_render_batch<false, true, KB> : (const void*)k_render_batch<false, false, KB>;
}

static const void* batch_kernel(int key_bytes, int fp64, int cone) {
  if (key_bytes == 8) return batch_kernel<8>(fp64, cone);
  if (key_bytes == 4) return batch_kernel<4>(fp64, cone);
  return batch_kernel<2>(fp64, cone);
}

hipError_t launch_render_batch(const BatchRenderLaunch& r, int fp64, int cone, int block_threads, int grid,
                               hipStream_t st) {
  if (r.nitems == 0) return hipSuccess;
  if (r.counting) return launch_render_batch_packet(r, fp64, cone, block_threads, grid, st);
  const size_t lds = render_batch_lds_bytes(block_threads, r.heap_slots, r.key_bytes);
  BatchRenderLaunch arg = r;
  void* args[] = {&arg};
  return hipLaunchKernel(batch_kernel(r.key_bytes, fp64, cone), dim3(grid), dim3(block_threads), args, lds, st);
}

int render_batch_occupancy(int fp64, int cone, int block_threads, int heap_slots, int key_bytes, int counting) {
  if (counting) return render_batch_packet_occupancy(fp64, cone, block_threads);
  int nb = 0;
  const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &nb, batch_kernel(key_bytes, fp64, cone), block_threads,
      render_batch_lds_bytes(block_threads, heap_slots, key_bytes));
  return e == hipSuccess ? nb : 0;
}

__global__ void k_tonemap(const float* __restrict__ rgb, size_t npix, float exposure, uchar4* __restrict__ out) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npix) return;
  uchar4 q;
  q.x = tonemap_u8(rgb[3 * i], exposure);
  q.y = tonemap_u8(rgb[3 * i + 1], exposure);
  q.z = tonemap_u8(rgb[3 * i + 2], exposure);
  q.w = 0;
  out[i] = q;
}

hipError_t launch_tonemap(const float* rgb, size_t npix, float exposure, uchar4* out, hipStream_t st) {
  if (npix == 0) return hipSuccess;
  hipLaunchKernelGGL(k_tonemap, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0, st, rgb, npix, exposure, out);
  return hipGetLastError();
}

}  // namespace pm
