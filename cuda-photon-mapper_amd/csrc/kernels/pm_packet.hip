// pm_packet.hip -- render with the packet gather (gather mode 7): one lane per
// eye sample, the 64 radiance queries of a wave answered together
// (pm_packet.h).  The eye path is that of render_sample_t
// (core/pm_transport.h) with the wave kept together: every lane takes each
// march step and each surface gather, with or without a query of its own, so
// that all lanes share in the search.  Reference counterpart:
// photon_mapping_kernel, photonMappingKernel.cu:1409-1462, with
// computePixelColor :926-1017 and the gathers :314-389, :831-870.
#include <math.h>

#include <algorithm>

#include "pm_mlp.h"
#include "pm_packet.h"
#include "pm_tiles.h"

namespace pm {

// In-scattered power at a march point toward wo.
template <class P>
struct PkVolAdd {
  typename P::Phase hg;
  V3f wo;
  PowerSum s;
  __device__ void reset() { psum_init(s); }
  __device__ void operator()(V3f pw, V3f dir, float) { P::add(s, pw, dir, wo, hg); }
  __device__ PkVolAdd of_lane(int b) const {
    PkVolAdd o = *this;
    o.wo = v3(u2f(read_lane(f2u(wo.x), b)), u2f(read_lane(f2u(wo.y), b)), u2f(read_lane(f2u(wo.z), b)));
    return o;
  }
  __device__ void reduce() { psum_reduce(s); }
  __device__ void take(const PkVolAdd& o) { s = o.s; }
};

// Power of the photons that arrived from the side of n; with the cone filter
// also power x distance, for the weight 1 - d / (1.1 r) once r is known.
template <bool CONE>
struct PkSurfAdd {
  V3f n;
  PowerSum s0, s1;
  __device__ void reset() {
    psum_init(s0);
    if (CONE) psum_init(s1);
  }
  __device__ void operator()(V3f pw, V3f dir, float d2) {
    if (dot(dir, n) < 0.0f) {
      psum_add(s0, pw);
      if (CONE) psum_add(s1, pw, sqrt_(d2));
    }
  }
  __device__ PkSurfAdd of_lane(int b) const {
    PkSurfAdd o = *this;
    o.n = v3(u2f(read_lane(f2u(n.x), b)), u2f(read_lane(f2u(n.y), b)), u2f(read_lane(f2u(n.z), b)));
    return o;
  }
  __device__ void reduce() {
    psum_reduce(s0);
    if (CONE) psum_reduce(s1);
  }
  __device__ void take(const PkSurfAdd& o) {
    s0 = o.s0;
    if (CONE) s1 = o.s1;
  }
};

// Terms of a cache row's sum: training rows (KIND 0) and fallback rows.
template <int KIND>
struct RowSum {
  using type = SumFp64;
};
template <>
struct RowSum<0> {
  using type = SumTarget;
};

__device__ __forceinline__ V3f pk_scale(const GatherMap& g) { return v3(g.scale[0], g.scale[1], g.scale[2]); }

// Eye sample s of pixel (px, py) for each lane with act set; every lane of
// the wave calls it.  A sample has 2^lu adjacent lanes, all with its path; at
// each turn of the march lane u of them takes step j0 + u, and the steps'
// terms are then added in step order by all of them, as by one lane marching
// alone.
template <bool FP64T, bool CONE>
__device__ __forceinline__ V3f packet_sample(const Scene& sc, const RenderParams& rp, const GatherMap& gs,
                                             const GatherMap& gv, PacketLds& S, int lane, int lu, bool act,
                                             uint32_t px, uint32_t py, uint32_t s, uint32_t& nsurf, uint32_t& nvol) {
  V3f o, d;
  float xi;
  camera_ray(rp, px, py, s, &o, &d, &xi);
  V3f thr = v3(1.0f, 1.0f, 1.0f);
  NSum3<float> L;
  nsum3_init(L);
  bool in_glass = false, alive = act;
  const Medium& m = sc.med;
  const bool media = rp.media_on && m.type != MED_NONE;
  const uint32_t pixel = py * (uint32_t)rp.width + px;
  const float ds = rp.march_step;
  const float st = m.sigma_s + m.sigma_a;
  PkVolAdd<SumFp64> va;
  va.hg = SumFp64::phase(m.g);
  const int U = 1 << lu, u = lane & (U - 1), ray = lane - u;  // ray: the sample's first lane
  for (int depth = 0; depth < rp.max_depth; ++depth) {
    if (ballot(alive) == 0ull) break;
    Hit<float> h;
    h.kind = HIT_NONE;
    h.id = 0;
    h.t = 0.0f;
    float t0 = 0.0f, t1 = 0.0f;
    bool seg = false;
    if (alive) {
      h = intersect(sc, o, d);
      if (media && !in_glass) {
        if (o.z < 0.0f) t0 = d.z > 0.0f ? -o.z / d.z : 3.0e38f;
        t1 = h.kind != HIT_NONE ? h.t : (o.z < 0.0f ? 0.0f : t_exit_front(o, d));
        seg = t1 > t0;
      }
    }
    if (ballot(seg)) {
      // FP64 transmittance on long segments through the density field
      const bool wide = FP64T && m.type == MED_NOISE && t1 - t0 >= (float)kLongSegmentSteps * ds;
      float tau = 0.0f, s_last = 0.0f, t_last = t0;
      double tau64 = 0.0, s_last64 = 0.0;
      bool sampled = false;
      uint32_t seed = kPkNoSeed;
      const V3f wo = -d;
      va.wo = wo;
      for (int j0 = 0; j0 < rp.max_steps; j0 += U) {
        const int j = j0 + u;
        const float t = t0 + ((float)j + xi) * ds;
        const bool on = seg && t < t1 && j < rp.max_steps;
        if (ballot(on) == 0ull) break;
        const V3f x = o + d * t;
        float Tj = 0.0f;
        if (m.type == MED_HOMOGENEOUS) {
          Tj = exp_(-st * (t - t0));
        } else {
          // the optical depth to each of the U steps, in step order
          const float mine = on ? sigma_t_at(m, x) : 0.0f;
          for (int v = 0; v < U; ++v) {
            const float sg = U == 1 ? mine : lane_read_f(mine, ray + v);
            const float tv = t0 + ((float)(j0 + v) + xi) * ds;
            if (seg && tv < t1 && j0 + v < rp.max_steps) {
              if (FP64T && wide) {
                tau64 = tau64 + (sampled ? (s_last64 + (double)sg) * 0.5 : (double)sg) * (double)(tv - t_last);
                s_last64 = (double)sg;
              } else {
                tau = tau + (sampled ? (s_last + sg) * 0.5f : sg) * (tv - t_last);
                s_last = sg;
              }
              t_last = tv;
              sampled = true;
              if (v == u) Tj = FP64T && wide ? (float)exp_(-tau64) : exp_(-tau);
            }
          }
        }
        const V3f w = thr * (Tj * ds);
        if (on) ++nvol;
        if (U > 1) seed = lane_read(seed, ray + U - 1);  // the turn's last step is the nearest earlier one
        uint32_t cnt;
        float r2;
        packet_gather<false>(gv, S, lane, on, x, seed, va, cnt, r2);
        V3f v = v3(0.0f, 0.0f, 0.0f);
        if (on && cnt) v = mul(psum_get(va.s), pk_scale(gv)) * volume_norm(r2);
        v = mul(w, v);
        if (U == 1) {
          if (on) nsum3_add(L, v);
        } else {
          for (int e = 0; e < U; ++e) {
            const V3f ve = v3(lane_read_f(v.x, ray + e), lane_read_f(v.y, ray + e), lane_read_f(v.z, ray + e));
            if (seg && t0 + ((float)(j0 + e) + xi) * ds < t1 && j0 + e < rp.max_steps) nsum3_add(L, ve);
          }
        }
      }
      if (seg) {
        float Tseg;
        if (m.type == MED_HOMOGENEOUS) {
          Tseg = exp_(-st * (t1 - t0));
        } else if (FP64T && wide) {
          if (!sampled) s_last64 = (double)sigma_t_at(m, o + d * ((t0 + t1) * 0.5f));
          Tseg = (float)exp_(-(tau64 + s_last64 * (double)(t1 - t_last)));
        } else {
          if (!sampled) s_last = sigma_t_at(m, o + d * ((t0 + t1) * 0.5f));
          Tseg = exp_(-(tau + s_last * (t1 - t_last)));
        }
        thr = thr * Tseg;
      }
    }
    alive = alive && h.kind != HIT_NONE;
    V3f x = v3(0.0f, 0.0f, 0.0f), nf = x;
    bool front = false;
    int mat = MAT_DIFFUSE;
    if (alive) {
      x = o + d * h.t;
      const V3f n = hit_normal(sc, h, x);
      front = dot(n, d) < 0.0f;
      nf = front ? n : -n;
      mat = hit_material(sc, h.kind, h.id);
    }
    const bool surf = alive && mat == MAT_DIFFUSE;
    if (ballot(surf)) {
      PkSurfAdd<CONE> sa;
      sa.n = nf;
      uint32_t seed = kPkNoSeed, cnt;
      float r2;
      packet_gather<false>(gs, S, lane, surf && u == 0, x, seed, sa, cnt, r2);
      V3f v = v3(0.0f, 0.0f, 0.0f);
      if (surf && u == 0) {
        ++nsurf;
        if (cnt) {
          v = psum_get(sa.s0);
          if (CONE) v = v - psum_get(sa.s1) * (1.0f / (1.1f * sqrt_(r2)));
          v = mul(mul(v, hit_albedo<float>(sc, h.kind, h.id)), pk_scale(gs)) * surface_norm(r2, CONE);
        }
      }
      if (U > 1) v = v3(lane_read_f(v.x, ray), lane_read_f(v.y, ray), lane_read_f(v.z, ray));
      if (surf) {
        nsum3_add(L, mul(thr, v));
        alive = false;
      }
    }
    if (alive) {
      if (mat == MAT_MIRROR) {
        thr = mul(thr, hit_albedo<float>(sc, h.kind, h.id));
        d = normalize(reflect(d, nf));
        o = x + nf * rp.eps;
      } else {
        const U4 re = rng(rp.seed, pixel, s, (uint32_t)depth, TAG_EYE);
        const float eta = front ? 1.0f / sc.spheres[h.id].ior : sc.spheres[h.id].ior;
        const float ci = -dot(d, nf);
        float ct;
        const float R = fresnel(ci, eta, &ct);
        if (u01(re.x) < R) {
          d = normalize(reflect(d, nf));
          o = x + nf * rp.eps;
        } else {
          d = normalize(refract(d, nf, eta, ci, ct));
          o = x - nf * rp.eps;
          in_glass = front;
        }
      }
    }
  }
  return nsum3_get(L);
}

__device__ __forceinline__ void count_queries(unsigned long long* counters, uint32_t ns, uint32_t nv) {
  if (!counters) return;
  atomicAdd(&counters[0], (unsigned long long)ns);
  atomicAdd(&counters[1], (unsigned long long)nv);
}

// Pixel (lx, ly) of this lane in item `sub` of tile (tx, ty): the tiles of a
// launch hold 2^lp pixels, an item of more march lanes (lv) the quarter `sub`
// of its tile.
__device__ __forceinline__ void item_pixel(int lane, int lu, int ls, int lv, int sub, int tx, int ty, int& lx, int& ly) {
  const int lp = 6 - lu - ls, lq = 6 - lv - ls, p = lane >> (lv + ls);
  lx = (tx << ((lp + 1) / 2)) + (p & (pk_tile_w(lq) - 1));
  ly = (ty << (lp / 2)) + (p >> ((lq + 1) / 2));
  if (lv != lu) {
    lx += (sub & 1) << ((lq + 1) / 2);
    ly += (sub >> 1) << (lq / 2);
  }
}

// The classes of a launch's tiles (RenderItems): a wave takes a tile, and its
// lanes look where the tile's eye rays go.  Rays that meet a mirror or a
// dielectric spread afterwards, and close to the light the neighbour balls
// are small, so such a tile's queries fall into many groups and its wave takes
// several times the others' time: it is listed first, in quarters of four
// times the march lanes (the same queries, the steps' terms in the same order).
constexpr float kNearLight = 0.1f;
__device__ __forceinline__ bool heavy_ray(const Scene& sc, const RenderParams& rp, uint32_t px, uint32_t py, uint32_t s) {
  V3f o, d;
  float xi;
  camera_ray(rp, px, py, s, &o, &d, &xi);
  const Hit<float> h = intersect(sc, o, d);
  if (h.kind == HIT_NONE) return false;
  if (hit_material(sc, h.kind, h.id) != MAT_DIFFUSE) return true;
  if (!rp.media_on) return false;
  const V3f l = v3(sc.light[0], sc.light[1], sc.light[2]) - o;
  const float t = fmin_(fmax_(dot(l, d), 0.0f), h.t);
  const V3f c = l - d * t;
  return dot(c, c) < kNearLight * kNearLight;
}

__global__ void __launch_bounds__(64) k_packet_tiles(RenderLaunch r, int lu, int ls, uint32_t ntiles) {
  const int lane = lane_id(), lp = 6 - lu - ls;
  const int tiles_x = (r.w + pk_tile_w(lp) - 1) >> ((lp + 1) / 2);
  for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    int lx, ly;
    item_pixel(lane, lu, ls, lu, 0, (int)tile % tiles_x, (int)tile / tiles_x, lx, ly);
    const bool act = lx < r.w && ly < r.h;
    const uint32_t s0 = (uint32_t)(lane >> lu) & ((1u << ls) - 1u);
    const bool heavy =
        ballot(act && heavy_ray(r.sc, r.rp, (uint32_t)(r.x0 + lx), (uint32_t)(r.y0 + ly), s0)) != 0ull;
    if (lane == 0) {
      if (heavy) {
        const uint32_t n = lp >= 2 ? 4u : 1u, at = atomicAdd(&r.items.head[1], n);
        for (uint32_t i = 0; i < n; ++i) r.items.heavy[at + i] = tile * 4u + i;
      } else {
        r.items.light[atomicAdd(&r.items.head[2], 1u)] = tile;
      }
    }
  }
}

// Renders the crop's tiles: a wave per tile in the order of tile_of_block, or,
// with r.items, a persistent grid whose waves take the next item, heavy ones
// first, until none is left.  lu: log2 of the march lanes; ls: log2 of the
// samples in lanes (0: each lane loops over the pixel's samples).
template <bool FP64T, bool CONE>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) k_render_packet(RenderLaunch r, int lu,
                                                                                               int ls) {
  __shared__ PacketLds S;
  const int lane = lane_id();
  const int lp = 6 - lu - ls;
  const bool queue = r.items.head != nullptr;
  uint32_t ns = 0u, nv = 0u;
  for (;;) {
    int tx, ty, lv = lu, sub = 0;
    bool in = true;
    if (queue) {
      uint32_t it = 0;
      if (lane == 0) it = atomicAdd(&r.items.head[0], 1u);
      it = read_lane(it, 0);
      const uint32_t nh = uniform(r.items.head[1]), nl = uniform(r.items.head[2]);
      if (it >= nh + nl) break;
      uint32_t tile;
      if (it < nh) {
        const uint32_t h = uniform(r.items.heavy[it]);
        tile = h >> 2;
        if (lp >= 2) {
          sub = (int)(h & 3u);
          lv = lu + 2;
        }
      } else {
        tile = uniform(r.items.light[it - nh]);
      }
      const int tiles_x = (r.w + pk_tile_w(lp) - 1) >> ((lp + 1) / 2);
      tx = (int)tile % tiles_x;
      ty = (int)tile / tiles_x;
    } else {
      in = tile_of_block(r, pk_tile_w(lp), pk_tile_h(lp), ls > 0, tx, ty);
    }
    int lx, ly;
    item_pixel(lane, lu, ls, lv, sub, tx, ty, lx, ly);
    const bool act = in && lx < r.w && ly < r.h;
    const uint32_t px = (uint32_t)(r.x0 + lx), py = (uint32_t)(r.y0 + ly);
    NSum3<float> acc;
    nsum3_init(acc);
    const int s0 = (lane >> lv) & ((1 << ls) - 1);
    for (int s = 0; s < r.rp.spp; s += 1 << ls) {
      const V3f v = packet_sample<FP64T, CONE>(r.sc, r.rp, r.gs, r.gv, S, lane, lv, act, px, py, (uint32_t)(s + s0),
                                               ns, nv);
      if (ls == 0) {
        nsum3_add(acc, v);
      } else {  // the pixel's samples in order, as in the sample loop
        const int base = lane & ~((1 << (lv + ls)) - 1);
        for (int t = 0; t < 1 << ls; ++t)
          nsum3_add(acc, v3(lane_read_f(v.x, base + (t << lv)), lane_read_f(v.y, base + (t << lv)),
                            lane_read_f(v.z, base + (t << lv))));
      }
    }
    if (act && (lane & ((1 << (lv + ls)) - 1)) == 0)
      store_pixel(r.rgb, r.u8, (size_t)ly * (size_t)r.w + (size_t)lx, nsum3_get(acc) * (1.0f / (float)r.rp.spp),
                  r.exposure);
    if (!queue) break;
  }
  if (ns | nv) count_queries(r.counters, ns, nv);
}

// The volume estimate's neighbour radius at the map's mean density, or the cap.
static double mean_radius(const GatherMap& gv) {
  return std::min(sqrt((double)gv.rcap2), cbrt((double)gv.k / (4.2 * (double)std::max(gv.n, 1u))));
}

// A frame's march lanes: as few as fill the chip with waves, while the steps of
// a turn stay within a neighbour ball; of very few waves up to 16, since each
// wave's chain of march turns is then all there is.  Room scene (r = 0.05) at
// lu = 0, 1, 2, 3, 4: 64x48 pixels 12.4, 4.2, 1.7, 1.1, 0.7 ms; 256x256 7.4, 1.8,
// 1.75, 1.5, 2.2 (rule: 3); 480x270 7.6, 1.9, 2.0, 2.3, 2.7 (2); 960x540 6.2, 3.7,
// 3.3, 3.7, 6.4 (0: 28 waves a CU are too few there).  Fog (r = 0.02) at lu = 0,
// 1, 2: 1920x1080 with 4 samples in lanes 146, 206, 349 from the list, with one
// 48, 60, 96; 480x270 around the light with one 12.0, 10.4, 21.6 (1).
int packet_march_lanes(const RenderParams& rp, const GatherMap& gv, int ls, uint64_t pixels, int cus) {
  if (!rp.media_on) return 0;
  int lu = 0;
  for (; lu < 4; ++lu) {
    const uint64_t waves = (pixels << (lu + ls)) >> 6;
    const double span = (double)(2 << lu) * rp.march_step;
    if (!(waves < 28ull * (uint64_t)cus && span <= 1.7 * mean_radius(gv)) &&
        !(waves < 4ull * (uint64_t)cus && span <= 0.32))
      break;
  }
  return lu < 6 - ls ? lu : 6 - ls;
}

// The same of a scene among many in one launch.  More march lanes make a
// wave's queries longer along the rays and narrower across them, so the box
// they span is smallest where the two balance: with pixel pitch p (at distance
// 1) 8 p / sqrt(2^lu) against 2^lu march steps.  The constant was fitted to
// render times; 8 scenes at lu = 0, 1, 2, 3, k = 32, r <= 0.05, 250,000 photons
// each (ms): 128^2: 21.9, 9.8, 5.7, 6.0   256^2: 24.1, 11.1, 9.1, 10.8   512^2:
// 26.5, 17.9, 19.5, 27.6   1024^2: 46.4, 48.1, 58.1, 94.5; the rule takes 2, 2, 1, 1.
int packet_march_lanes_batch(const RenderParams& rp, const GatherMap& gv, uint64_t pixels, int cus) {
  if (!rp.media_on) return 0;
  const double pitch = 1.0 / ((double)rp.focal * (double)rp.height);
  int lu = (int)floor(1.9 + log2(8.0 * pitch / (double)rp.march_step) / 1.5);
  lu = lu < 0 ? 0 : (lu > 4 ? 4 : lu);
  return std::max(lu, packet_march_lanes(rp, gv, 0, pixels, cus));
}

size_t packet_item_words(uint32_t tiles) { return 4 + 5ull * tiles; }

// Launches of at least this many tiles take no work list (launch_render_packet).
uint32_t packet_list_tiles(int cus) { return 64u * (uint32_t)cus; }

// log2 of the samples of a pixel that go to adjacent lanes.
static int packet_sample_lanes(const RenderLaunch& r) {
  const int spp = r.rp.spp;
  const int ls = r.sample_lanes && (spp == 2 || spp == 4 || spp == 8 || spp == 16) ? __builtin_ctz((unsigned)spp) : 0;
  // a launch holds fewer than 2^32 lanes
  return (((uint64_t)r.w + 7) * ((uint64_t)r.h + 7)) << ls >= 1ull << 31 ? 0 : ls;
}

// Whether the packet gather renders a scene faster than the 8-byte heap of mode
// 1 (its 2-byte form in a batch): ls and lu are the log2 of its sample and march
// lanes, pixels those of the launch.  Searches are shared, so the packet gather
// loses where a wave's balls do not overlap: each of its 64 queries is then a
// search of its own, 64 in a row.
//
// With a march, a wave's points are spread over a march step along their rays
// (the samples' offsets), so balls of about a step or less in which hardly any
// photon lies go to the heap, unless the launch is so small that eight march
// lanes split its chains; fewer photons are enough where four samples or more
// lie together in lanes, and one neighbour's ball counts in place of the cap.
// 256x256 room, 2,452 to 718,541 records, r <= 0.005, k = 1 to 64: heap 1.2 to
// 4.3 ms, packet 16 to 22; r <= 0.02: 1.4 to 9.5 and 1.1 to 3.9 (k = 1: 9.7);
// 640x360 with 4 samples, r <= 0.05: 10 to 180 and 2 to 14.
//
// Without one, a wave makes one search, without a seed.  Four or more samples
// in lanes pay for it (640x360x4, k = 32, r <= 0.05: heap 1.1 to 5.2 ms, packet
// 0.5 to 1.8) unless the cap is so much wider than the ball that the first
// bound is loose (k = 8, r <= 0.47, a ball of a quarter tile: 1.5 and 4.5).
// Otherwise full balls, of 13 neighbours or more, pay where the cap is not far
// beyond them (718,541 records, 640x360, k = 32: 1.3 and 0.7 at r <= 0.02, 1.3
// and 3.7 at r <= 0.15) and the launch is of less than a wave per CU, or of
// many, or its balls are as wide as four tiles (48,578 records, r <= 0.05,
// 3,600 waves, 1.5 tiles: 0.8 and 1.6); and emptier ones if wider than five.
//
// Over 4,800 random frames (scene, photons, k, cap, size, samples) the choice
// takes 1.017 times the faster one's time with a march (the packet gather
// always: 1.05, and up to 11 times the heap's) and 1.07 without (1.33, up to 31).
bool packet_pays(const RenderParams& rp, bool march, const GatherMap& gs, const GatherMap& gv, int ls, int lu,
                 uint64_t pixels, int cus) {
  const uint64_t waves = (pixels << ls) >> 6, cu = (uint64_t)cus;  // without march lanes
  const GatherMap& g = march ? gv : gs;
  const double cap2 = (double)g.rcap2, cap = sqrt(cap2), n = (double)g.n, k = (double)g.k;
  if (march) {
    if (lu >= 3) return true;
    const double step = (double)rp.march_step, in_cap = 4.2 * n * cap2 * cap;
    const double ball = in_cap > 1.0 ? cap / cbrt(in_cap) : cap;  // one neighbour's
    if (g.k == 1 && ls < 2 && ball < 1.7 * step) return false;
    return cap >= 1.2 * step || in_cap >= (ls < 2 ? 0.3 : 0.002);
  }
  constexpr double kWalls = 5.0;                   // area of the room's five walls
  const double in_cap = 3.14 * n * cap2 / kWalls;  // photons within the cap of a hit
  const double tile = (double)pk_tile_w(6 - ls) / ((double)rp.focal * (double)rp.height);  // at distance 1
  const double tiles = cap * (in_cap > k ? sqrt(k / in_cap) : 1.0) / tile;                 // a ball's radius
  if (ls >= 2) return in_cap <= 5000.0 || tiles >= 0.4;
  if (std::min(in_cap, k) >= 13.0)
    return in_cap <= 1500.0 && (waves <= cu || (in_cap >= 45.0 && (waves >= 16u * cu || tiles >= 4.0)));
  return tiles >= 5.4 && waves < 32u * cu;
}

// The same for the exact values of a cache frame's records, in the volume map:
// listed rows are further apart than a tile's march points, so it is only
// whether a photon or none is near.  64x48 to 640x360 frames with all records
// gathered, packet over heap (2-byte keys) time of the frame, medians: fewer
// than 0.001 photons within the cap 1.8 to 2.6, 0.01 to 0.1 1.1 to 1.8, 0.1 to 1
// 0.7 to 1.1 (at caps of a step and more), more 0.4 to 0.7.
bool packet_pays_rows(const GatherMap& gv) {
  return 4.2 * (double)gv.n * (double)gv.rcap2 * sqrt((double)gv.rcap2) >= 0.1;
}

// The launch's lane layout and tile count.
static uint32_t packet_layout(const RenderLaunch& r, int& lu, int& ls) {
  ls = packet_sample_lanes(r);
  lu = packet_march_lanes(r.rp, r.gv, ls, (uint64_t)r.w * (uint64_t)r.h, r.cus);
  const int lp = 6 - lu - ls;
  return (uint32_t)((r.w + pk_tile_w(lp) - 1) / pk_tile_w(lp)) * (uint32_t)((r.h + pk_tile_h(lp) - 1) / pk_tile_h(lp));
}

bool packet_pays(const RenderLaunch& r) {
  int lu, ls;
  packet_layout(r, lu, ls);
  return packet_pays(r.rp, r.rp.media_on != 0, r.gs, r.gv, ls, lu, (uint64_t)r.w * (uint64_t)r.h, r.cus);
}

hipError_t launch_packet_tiles(RenderLaunch& r, int lu, int ls, uint32_t tiles, hipStream_t st) {
  r.items.heavy = r.items.head + 4;
  r.items.light = r.items.heavy + 4ull * tiles;
  hipError_t e = launch_fill_u32(r.items.head, 0u, 4, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_packet_tiles, dim3(std::min(tiles, 32u * (unsigned)r.cus)), dim3(64), 0, st, r, lu, ls, tiles);
  return hipGetLastError();
}

hipError_t launch_render_packet(const RenderLaunch& r, hipStream_t st) {
  if (r.w <= 0 || r.h <= 0) return hipSuccess;
  const bool fp64 = r.rp.fp64_transmittance != 0, cone = r.estimator == 1;
  int lu, ls;
  const uint32_t tiles = packet_layout(r, lu, ls);
  const int lp = 6 - lu - ls;
  RenderLaunch q = r;
  dim3 grid(tile_grid(r, pk_tile_w(lp), pk_tile_h(lp), ls > 0));
  // The heavy tiles first and split where the launch ends on them: frames of
  // few waves, or, in a map so dense that a wave's march takes milliseconds, of
  // few rounds of waves.  Windows of the fog at the frame's centre, list
  // against grid: 480x270 10.3 and 21.9 ms at 1 sample, 30 and 69 at 3, 21 and 35
  // at 4; 1200x675 at 1: 30 and 74; the whole 1920x1080 frame (129,600 tiles) at
  // 4: 146 and 129, so not there (at 1 sample, 32,400 tiles, 48 and 59 still).
  // Room (march lanes): 64x48 0.71 and 0.93, 256x256 1.55 and 1.98, 640x360 2.07
  // and 3.34.  With less than a tile a CU all waves start at once and the
  // list only costs (120x68 at 1: 2.5 and 2.25).
  const double rm = mean_radius(r.gv);
  const bool dense = rm * rm < 0.999 * r.gv.rcap2;
  const bool few = dense ? tiles > (unsigned)r.cus && tiles < packet_list_tiles(r.cus)
                         : lu > 0 && tiles < 34u * (unsigned)r.cus;
  if (r.tile_regions == 0 && r.rp.media_on && few && r.items.head && r.items.words >= packet_item_words(tiles)) {
    hipError_t e = launch_packet_tiles(q, lu, ls, tiles, st);
    if (e != hipSuccess) return e;
    grid = dim3(std::min(4u * tiles, (unsigned)(16 * r.cus)));
  } else {
    q.items.head = nullptr;
  }
  if (fp64 && cone) hipLaunchKernelGGL((k_render_packet<true, true>), grid, dim3(64), 0, st, q, lu, ls);
  else if (fp64) hipLaunchKernelGGL((k_render_packet<true, false>), grid, dim3(64), 0, st, q, lu, ls);
  else if (cone) hipLaunchKernelGGL((k_render_packet<false, true>), grid, dim3(64), 0, st, q, lu, ls);
  else hipLaunchKernelGGL((k_render_packet<false, false>), grid, dim3(64), 0, st, q, lu, ls);
  return hipGetLastError();
}

// Batched render: the work queue of k_render_batch (pm_gather_lane.hip) with
// the packet gather.  Each wave has its own PacketLds.
template <bool FP64T, bool CONE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_render_batch_packet(BatchRenderLaunch r) {
  extern __shared__ __align__(16) unsigned char lds[];
  const int lane = lane_id();
  const int wave = (int)uniform(threadIdx.x >> 6);
  PacketLds& P = ((PacketLds*)lds)[wave];
  unsigned long long ns_tot = 0, nv_tot = 0;
  for (;;) {
    uint32_t it = 0;
    if (lane == 0) it = atomicAdd(r.head, 1u);
    it = read_lane(it, 0);
    if (it >= r.nitems) break;
    const uint2 item = r.items[it];
    const BatchRenderScene& S = r.scenes[uniform(item.x)];
    const int lu = S.lu, lp = 6 - lu;
    const uint32_t tile = uniform(item.y);
    const int tiles_x = (S.w + pk_tile_w(lp) - 1) >> ((lp + 1) / 2);
    int lx, ly;
    item_pixel(lane, lu, 0, lu, 0, (int)tile % tiles_x, (int)tile / tiles_x, lx, ly);
    const bool act = lx < S.w && ly < S.h;
    uint32_t ns = 0u, nv = 0u;
    NSum3<float> acc;
    nsum3_init(acc);
    for (int s = 0; s < S.rp.spp; ++s)
      nsum3_add(acc, packet_sample<FP64T, CONE>(S.sc, S.rp, S.gs, S.gv, P, lane, lu, act, (uint32_t)lx, (uint32_t)ly,
                                                (uint32_t)s, ns, nv));
    if (act) {
      if ((lane & ((1 << lu) - 1)) == 0)
        store_pixel(r.rgb + 3 * S.img_off, nullptr, (size_t)ly * (size_t)S.w + (size_t)lx,
                    nsum3_get(acc) * (1.0f / (float)S.rp.spp), S.exposure);
      ns_tot += ns;
      nv_tot += nv;
    }
  }
  if (r.counters) {
    atomicAdd(&r.counters[0], ns_tot);
    atomicAdd(&r.counters[1], nv_tot);
  }
}

static const void* batch_packet_kernel(int fp64, int cone) {
  if (fp64) return cone ? (const void*)k_render_batch_packet<true, true> : (const void*)k_render_batch_packet<true, false>;
  return cone ? (const void*)k_render_batch_packet<false, true> : (const void*)k_render_batch_packet<false, false>;
}

hipError_t launch_render_batch_packet(const BatchRenderLaunch& r, int fp64, int cone, int block_threads, int grid,
                                      hipStream_t st) {
  BatchRenderLaunch arg = r;
  void* args[] = {&arg};
  return hipLaunchKernel(batch_packet_kernel(fp64, cone), dim3(grid), dim3(block_threads), args,
                         sizeof(PacketLds) * (size_t)(block_threads / 64), st);
}

int render_batch_packet_occupancy(int fp64, int cone, int block_threads) {
  int nb = 0;
  const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &nb, batch_packet_kernel(fp64, cone), block_threads, sizeof(PacketLds) * (size_t)(block_threads / 64));
  return e == hipSuccess ? nb : 0;
}

// Exact values of cache rows, 64 or 16 rows a wave.  KIND 1 and 2: the fallback's
// surface and volume rows, listed so that a wave's rows lie together (surface
// rows in record order, a compact patch of the image; volume rows ordered by
// k_order_rows), each started from its record's seed of the previous frame.
// KIND 0: the training rows, of either kind, in the order of launch_sort_rows.
// One lane per row with its own heap and traversal took 2.4 ms for 2^18
// training rows of the 1M + 2M photon maps.
constexpr uint32_t kRowNoSeed = 0xffffu, kRowFew = 0xfffeu;  // the 16-bit forms of kPkNoSeed and kPkFew

// Rows per wave: 16 of the training rows and of volume lists of fewer than
// 2^21, where the launch would hold few waves, since the waves whose rows are
// far apart, or near the light, take several times the others' time and end the
// launch; 64, whose lanes share more, in a longer list.  256,000 volume rows:
// 14.6 ms at 64, 4.6 at 16; 129M: 117 ms at 64, 204 at 16; the seeded fallback
// of the 1920x1080 cache frame with the line at 2^18, 2^21, 2^24: 3.4, 3.5, 4.8.
constexpr uint32_t kFewRows = 1u << 21;

template <int KIND>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) k_values_packet(CacheValueLaunch v,
                                                                                               uint32_t rows) {
  using P = typename RowSum<KIND>::type;
  __shared__ PacketLds S;
  const int lane = lane_id();
  const uint32_t i = blockIdx.x * rows + (uint32_t)lane;
  const bool act = (uint32_t)lane < rows && i < v.n;
  const uint32_t rec = act ? v.list[i] : 0u;
  V3f x = v3(0.0f, 0.0f, 0.0f), d = x, nrm = x;
  uint32_t seed = kPkNoSeed;
  if (act) {
    const float* p = v.in + (size_t)rec * MLP_IN;
    x = v3(p[0], p[1], p[2]);
    if (KIND != 1) d = v3(p[3], p[4], p[5]);
    if (KIND != 2) nrm = v3(p[6], p[7], p[8]);
    if (KIND != 0 && v.seed_q) {
      const uint32_t q = v.seed_q[rec];
      seed = q == kRowNoSeed ? kPkNoSeed : (q == kRowFew ? kPkFew : q);
    }
  }
  const bool surf = KIND == 1 || (KIND == 0 && !(nrm.x == 0.0f && nrm.y == 0.0f && nrm.z == 0.0f));
  uint32_t cnt;
  float r2;
  V3f val = v3(0.0f, 0.0f, 0.0f);
  if (KIND != 2 && (KIND == 1 || ballot(act && surf))) {
    PkSurfAdd<false> add;
    add.n = nrm;
    packet_gather<KIND != 0>(v.gs, S, lane, act && surf, x, seed, add, cnt, r2);
    if (cnt) val = mul(psum_get(add.s0), pk_scale(v.gs)) * surface_norm(r2, false);
  }
  if (KIND != 1 && (KIND == 2 || ballot(act && !surf))) {
    PkVolAdd<P> add;
    add.hg = P::phase(v.hg_g);
    add.wo = d;
    packet_gather<KIND != 0>(v.gv, S, lane, act && !surf, x, seed, add, cnt, r2);
    if (cnt) val = mul(psum_get(add.s), pk_scale(v.gv)) * volume_norm(r2);
  }
  if (!act) return;
  if (KIND != 0 && v.seed_q)
    v.seed_q[rec] = (uint16_t)(seed == kPkFew ? kRowFew : (seed == kPkNoSeed ? kRowNoSeed : seed));
  v.out[3 * (size_t)rec] = val.x;
  v.out[3 * (size_t)rec + 1] = val.y;
  v.out[3 * (size_t)rec + 2] = val.z;
}

hipError_t launch_cache_values_packet(const CacheValueLaunch& v, hipStream_t st) {
  if (v.n == 0) return hipSuccess;
  const uint32_t rows = v.kind == 0 || (v.kind == 2 && v.n < kFewRows) ? 16u : 64u;
  const dim3 grid((v.n + rows - 1) / rows);
  if (v.kind == 1) hipLaunchKernelGGL(k_values_packet<1>, grid, dim3(64), 0, st, v, rows);
  else if (v.kind == 2) hipLaunchKernelGGL(k_values_packet<2>, grid, dim3(64), 0, st, v, rows);
  else hipLaunchKernelGGL(k_values_packet<0>, grid, dim3(64), 0, st, v, rows);
  return hipGetLastError();
}

__device__ __forceinline__ uint32_t cell10(float v) {
  const float c = v * 1024.0f;
  return c > 0.0f ? (c < 1023.0f ? (uint32_t)c : 1023u) : 0u;
}
__device__ __forceinline__ uint32_t spread10(uint32_t v) {
  v = (v | (v << 16)) & 0x030000ffu;
  v = (v | (v << 8)) & 0x0300f00fu;
  v = (v | (v << 4)) & 0x030c30c3u;
  return (v | (v << 2)) & 0x09249249u;
}
__device__ __forceinline__ uint32_t row_morton(const float* p) {
  return spread10(cell10(p[0])) | (spread10(cell10(p[1])) << 1) | (spread10(cell10(p[2])) << 2);
}

// Orders each run of 1,024 listed rows by the Morton code of its position, in
// place.  Volume records follow one another along their ray, so 64 in record
// order lie on a few lines through the whole room; 1,024 of them (the rays of a
// 4x4 pixel block) ordered by position put 64 into a short stretch of those
// rays.  Bitonic sort of 64-bit (code, row) keys in LDS.
constexpr uint32_t kOrderRun = 1024;
__global__ void __launch_bounds__(256) k_order_rows(const float* __restrict__ in, uint32_t* __restrict__ list, uint32_t n) {
  __shared__ uint64_t K[kOrderRun];
  const uint32_t b0 = blockIdx.x * kOrderRun, tid = threadIdx.x;
  for (uint32_t j = tid; j < kOrderRun; j += 256u) {
    uint64_t k = ~0ull;
    if (b0 + j < n) {
      const uint32_t r = list[b0 + j];
      k = ((uint64_t)row_morton(in + (size_t)r * MLP_IN) << 32) | r;
    }
    K[j] = k;
  }
  for (uint32_t size = 2; size <= kOrderRun; size <<= 1) {
    for (uint32_t stride = size >> 1; stride; stride >>= 1) {
      __syncthreads();
#pragma unroll
      for (uint32_t t = 0; t < kOrderRun / 512; ++t) {
        const uint32_t e = tid + t * 256u;
        const uint32_t a = ((e & ~(stride - 1u)) << 1) | (e & (stride - 1u)), b = a | stride;
        const uint64_t x = K[a], y = K[b];
        if ((x > y) == ((a & size) == 0u)) {
          K[a] = y;
          K[b] = x;
        }
      }
    }
  }
  __syncthreads();
  for (uint32_t j = tid; j < kOrderRun; j += 256u)
    if (b0 + j < n) list[b0 + j] = (uint32_t)K[j];
}

hipError_t launch_order_rows(const float* in, uint32_t* list, uint32_t n, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_order_rows, dim3((n + kOrderRun - 1) / kOrderRun), dim3(256), 0, st, in, list, n);
  return hipGetLastError();
}

// 16-bit keys of the training rows: kind, then the top 15 bits of the Morton code.
__global__ void k_row_keys(const float* __restrict__ in, uint32_t n, uint32_t* __restrict__ keys,
                           uint32_t* __restrict__ vals) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const float* p = in + (size_t)i * MLP_IN;
  const bool surf = !(p[6] == 0.0f && p[7] == 0.0f && p[8] == 0.0f);
  keys[i] = (row_morton(p) >> 15) | (surf ? 0x8000u : 0u);
  vals[i] = i;
}

size_t sort_rows_words(uint32_t n) { return 3ull * n + radix_temp_words(n); }

hipError_t launch_sort_rows(const float* in, uint32_t n, uint32_t* order, uint32_t* temp, hipStream_t st) {
  if (n == 0) return hipSuccess;
  uint32_t *k0 = temp, *k1 = k0 + n, *v1 = k1 + n, *rt = v1 + n;
  hipLaunchKernelGGL(k_row_keys, dim3((n + 255) / 256), dim3(256), 0, st, in, n, k0, order);
  hipError_t e = radix_pass(k0, order, n, 0, rt, k1, v1, st);
  return e != hipSuccess ? e : radix_pass(k1, v1, n, 8, rt, k0, order, st);
}

}  // namespace pm
