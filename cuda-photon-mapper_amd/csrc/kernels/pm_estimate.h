// pm_estimate.h -- the sums of a density estimate on the GPU: photon power
// weighted by the phase function, accumulated in FP64.  Device-only.
#pragma once

#include "../core/pm_transport.h"
#include "pm_wave.h"

namespace pm {

// Sum of power x weight over a query's neighbours.  The FP32 factors are
// exact in FP64 and FP64 fused multiply-adds run at the FP32 rate on gfx950,
// so a term takes one conversion and three instructions where the FP32
// compensated sum took three products and 21.  64 terms of one sign differ from
// the exact sum by less than 2^-46 of it, so traversals that meet the same
// neighbours in another order give the same FP32 sum, except where the exact
// one lies that close to the middle of two FP32 values (one sum in about four
// million): there it may be either.  Summing such cases again in one order would
// make the orders equal always, at 3 % of the 1920x1080 fog frame and more where
// the powers have few bits (30 % of the cache frame with BF16 powers).
struct PowerSum {
  double x, y, z;
};
__device__ __forceinline__ void psum_init(PowerSum& s) { s.x = s.y = s.z = 0.0; }
__device__ __forceinline__ void psum_add(PowerSum& s, V3f pw, float w) {
  const double d = (double)w;
  s.x = __builtin_fma((double)pw.x, d, s.x);
  s.y = __builtin_fma((double)pw.y, d, s.y);
  s.z = __builtin_fma((double)pw.z, d, s.z);
}
__device__ __forceinline__ void psum_add(PowerSum& s, V3f pw) {
  s.x += (double)pw.x;
  s.y += (double)pw.y;
  s.z += (double)pw.z;
}
// The sum over the wave, in every lane: row shifts by 1, 2, 4, 8, then rows
// 15 -> 16 and 31 -> 32 broadcast, and the total from lane 63.
template <int CTRL>
__device__ __forceinline__ double dpp_or_zero(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xf, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double wave_total(double v) {
  v += dpp_or_zero<0x111>(v);
  v += dpp_or_zero<0x112>(v);
  v += dpp_or_zero<0x114>(v);
  v += dpp_or_zero<0x118>(v);
  // the broadcasts only into the rows that take them: rows 1 and 3, then 2 and 3
  const int lane = lane_id();
  const double b = dpp_or_zero<0x142>(v);
  v += (lane & 16) ? b : 0.0;
  const double c = dpp_or_zero<0x143>(v);
  v += (lane & 32) ? c : 0.0;
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  return __builtin_bit_cast(double, ((uint64_t)read_lane((uint32_t)(u >> 32), 63) << 32) | read_lane((uint32_t)u, 63));
}
__device__ __forceinline__ void psum_reduce(PowerSum& s) {
  s.x = wave_total(s.x);
  s.y = wave_total(s.y);
  s.z = wave_total(s.z);
}
__device__ __forceinline__ V3f psum_get(const PowerSum& s) { return v3((float)s.x, (float)s.y, (float)s.z); }

// Henyey-Greenstein phase function of the gathers, with the constants of one
// g.  den^(-3/2) from the hardware reciprocal square root (1 ulp) and two
// products: within 4e-7 of the closed form on the FP32 den, against 6e-7 for
// the Newton steps of phase_hg (core/pm_scene.h), and 10 instructions fewer.
// |g| < 1 gives den >= 2^-48 for directions of unit length.  A longer one (BF16
// storage rounds each component to 2^-9, and callers give their own) can take
// den below 0: such a photon has no weight, as in phase_hg, whose Newton steps
// underflow there (down to -0.2; below that, and for infinite directions, they
// give NaN, which a branch to them would keep at 3.7 % of the fog frame against
// 1.2 for the select).
struct HgPhase {
  float a, b, c;  // 1 + g^2, -2 g, (1 - g^2) / (4 pi)
};
__device__ __forceinline__ HgPhase hg_phase(float g) {
  return HgPhase{1.0f + g * g, -2.0f * g, 0.0795774715459476678844418816863f * (1.0f - g * g)};
}
__device__ __forceinline__ float hg_eval(const HgPhase& h, V3f dir, V3f wo) {
  const float cs = __builtin_fmaf(dir.z, wo.z, __builtin_fmaf(dir.y, wo.y, dir.x * wo.x));
  const float den = __builtin_fmaf(h.b, cs, h.a);
  const float y = __builtin_amdgcn_rsqf(den);
  return den < 0.0f ? 0.0f : h.c * ((y * y) * y);
}

// The two kinds of terms a gather sums.  SumFp64: the renders and the cache's
// exact fallback.  SumTarget: the cache's training targets, whose terms keep
// FP32 products and the Newton phase function: a last-bit change of many
// targets moves the trained weights by BF16 rounding steps here and there, and
// the cached frames with them (6e-4 of the frame).
struct SumFp64 {
  using Phase = HgPhase;
  static __device__ __forceinline__ Phase phase(float g) { return hg_phase(g); }
  static __device__ __forceinline__ void add(PowerSum& s, V3f pw, V3f dir, V3f wo, const Phase& h) {
    psum_add(s, pw, hg_eval(h, dir, wo));
  }
};
struct SumTarget {
  using Phase = float;
  static __device__ __forceinline__ Phase phase(float g) { return g; }
  static __device__ __forceinline__ void add(PowerSum& s, V3f pw, V3f dir, V3f wo, Phase g) {
    psum_add(s, pw * phase_hg(dot(dir, wo), g));
  }
};

}  // namespace pm
