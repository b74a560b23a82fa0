// pm_packet.h -- the packet gather (gather mode 7): exact k-NN density
// estimates for the 64 queries of a wave at once.  Device-only.
//
// The queries of a wave lie close together (the march points of a small tile
// of pixels at one step, or their surface hits), so their neighbour balls
// overlap almost entirely.  Instead of 64 tree searches the wave makes one:
//   stage   the lanes test node boxes in parallel (8 nodes x 8 descendants
//           three levels down at a time) against the box of the queries grown
//           by the search bound, then the points of the leaves that pass; the
//           points within the bound of the query box are packed into LDS;
//   count   every lane runs over the staged points (the same point for all
//           lanes, one LDS broadcast) and counts them in a window of 128
//           buckets of d^2 (FP32 bits >> 16, 2^-7 wide) around its previous
//           query's k-th-neighbour bucket, in 4-bit LDS counters; the bucket
//           Q of its k-th neighbour is where the running count reaches k.  A
//           lane whose k-th neighbour lies outside its window moves the
//           window; one whose counter wrapped bisects its window instead;
//   sum     every lane runs over the staged points again: those in buckets
//           below Q contribute, with the payload of the point read once for
//           all lanes; of the bucket-Q points the (d^2, index) smallest that
//           complete k are picked at the end.
// Queries that are not near each other are gathered in groups, each with its
// own stage, so any set of queries gives the same neighbour sets.  The order
// of their FP64 sums depends on the grouping, their FP32 results therefore in
// the last bit now and then (pm_estimate.h): so do a crop and its frame, a batch
// and a single scene, and seeded and unseeded rows.
//
// Bounds are exact: with the operation order of dist2 and monotonic FP32
// rounding, no point has a smaller computed d^2 to a query than the computed
// d^2 between the query box and the point (or a box that holds the point).
#pragma once

#include "pm_estimate.h"
#include "pm_kernels.h"
#include "pm_lane_knn.h"
#include "pm_wave.h"

namespace pm {

// Sizes measured one at a time (render ms; "fog" the 1920x1080 frame with 4
// samples, "window" its 480x270 crop around the light at 1 sample, "surfaces"
// the frame without the march, "room" the 480x270 room, "batch" 8 scenes).
constexpr uint32_t kPkCand = 320;     // staged points: what leaves 16 waves' LDS
constexpr uint32_t kPkBuckets = 128;  // counting window (8 counters per LDS word)
// Window top above the previous query's bucket: lower ones stage fewer points
// and move more windows.  16, 32, 48, 64: fog 156, 133.8, 129.4, 133.2.
constexpr uint32_t kPkUp = 48;
constexpr uint32_t kPkStack = 192;    // node stack (see pk_stage)
constexpr uint32_t kPkTie = 8;        // bucket-Q points kept per lane
// Groups of at most this many queries go one query at a time.  4, 8, 16: window
// 11.3, 10.4, 10.2, surfaces 5.8, 5.6, 5.6, room 1.8, 2.0, 1.9, batch 19.0, 18.8,
// 19.3.
constexpr uint32_t kPkSolo = 8;
constexpr uint32_t kPkSoloFew = 12;   // the same where at most 32 queries start (8 to 20: the same)
constexpr uint32_t kPkNoSeed = 0xffffffffu, kPkFew = 0xfffffffeu;

// LDS of one wave: 10 KB, 16 waves per CU.
struct PacketLds {
  float4 cand[kPkCand];  // x, y, z, bits(tree position)
  union {
    uint32_t cnt[kPkBuckets / 8 * 64];  // counters: word w of lane l at [w * 64 + l]
    struct {
      float4 a[64];  // power, direction x
      float2 b[64];  // direction y, z
    } pay;
    uint32_t tie[kPkTie * 64];
  };
  uint32_t stack[kPkStack];
  uint32_t leaf[64];
};

__device__ __forceinline__ void pk_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ uint32_t pk_rank(uint64_t m) {  // set bits of m below this lane
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
template <int CTRL>
__device__ __forceinline__ uint32_t pk_dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, false);
}
// Reductions over the 64 lanes (row shifts by 1, 2, 4, 8, then rows 15 -> 16
// and 31 -> 32 broadcast); the result, uniform, from lane 63.
__device__ __forceinline__ float pk_min(float v) {
  uint32_t x = f2u(v);
#define PK_STEP(C) x = f2u(__builtin_fminf(u2f(x), u2f(pk_dpp<C>(x))));
  PK_STEP(0x111) PK_STEP(0x112) PK_STEP(0x114) PK_STEP(0x118) PK_STEP(0x142) PK_STEP(0x143)
#undef PK_STEP
  return u2f(read_lane(x, 63));
}
__device__ __forceinline__ float pk_max(float v) { return -pk_min(-v); }
__device__ __forceinline__ uint32_t pk_umax(uint32_t x) {
#define PK_STEP(C) { const uint32_t o = pk_dpp<C>(x); x = x > o ? x : o; }
  PK_STEP(0x111) PK_STEP(0x112) PK_STEP(0x114) PK_STEP(0x118) PK_STEP(0x142) PK_STEP(0x143)
#undef PK_STEP
  return read_lane(x, 63);
}

// Box of a group of queries (wave-uniform).
struct PkBox {
  V3f lo, hi;
};
// d^2 between the query box and the box [mn, mx].
__device__ __forceinline__ float pk_box_d2(const PkBox& b, V3f mn, V3f mx) {
  const float dx = __builtin_fmaxf(__builtin_fmaxf(mn.x - b.hi.x, b.lo.x - mx.x), 0.0f);
  const float dy = __builtin_fmaxf(__builtin_fmaxf(mn.y - b.hi.y, b.lo.y - mx.y), 0.0f);
  const float dz = __builtin_fmaxf(__builtin_fmaxf(mn.z - b.hi.z, b.lo.z - mx.z), 0.0f);
  return (dx * dx + dy * dy) + dz * dz;
}

// Packs the points within bound2 of the query box into S.cand; full(M) is
// called each time the stage is full (false stops the search).  Returns the
// points left in the stage.  All 64 lanes call it.
template <class F>
__device__ __forceinline__ uint32_t pk_stage(const GatherMap& g, PacketLds& S, int lane, const PkBox& box,
                                             float bound2, F&& full) {
  const uint32_t n = g.n, nl = g.nl, L = g.L, last = 2u * nl - 2u;
  const uint32_t deep = 31u - (uint32_t)__builtin_clz(2u * nl - 1u);  // level of the last node
  const uint32_t first_deep = (1u << deep) - 1u, ndeep = last - first_deep + 1u;
  const uint32_t lg = L <= 1u ? 0u : 32u - (uint32_t)__builtin_clz(L - 1u);  // a leaf's lanes: 2^lg >= L
  uint32_t M = 0, sp = 0;
  uint32_t span = 6u;  // first step: the root's 64 descendants six levels down
  for (;;) {
    // this lane's node: descendant i of `h`, up to `span` levels below
    uint32_t h = 0u, i = (uint32_t)lane;
    bool ok = true;
    if (span == 3u) {
      if (sp == 0u) break;
      // Take p nodes: each leaves at most 8 on the stack for itself.  Taking
      // one at a time grows the stack by at most 7 per 3 levels, 63 for the 27
      // levels below the first step, so p is what keeps room for that.
      const uint32_t room = kPkStack - 63u > sp ? (kPkStack - 63u - sp) / 7u : 0u;
      uint32_t n8 = sp < 8u ? sp : 8u;
      n8 = n8 < room ? n8 : (room > 0u ? room : 1u);
      const uint32_t slot = (uint32_t)lane >> 3;
      ok = slot < n8;
      sp -= n8;
      h = ok ? S.stack[sp + slot] : 0u;
      i = (uint32_t)lane & 7u;
    }
    const uint32_t below = deep - (31u - (uint32_t)__builtin_clz(h + 1u));  // levels below h
    const uint32_t lv = below < span ? below : span, up = span - lv;
    uint64_t t64 = ((uint64_t)(h + 1u) << lv) - 1ull + (uint64_t)(i >> up);
    ok = ok && (i & ((1u << up) - 1u)) == 0u;
    if (t64 > (uint64_t)last) {  // the last level is not full: the node above, once
      t64 = (t64 - 1ull) >> 1;
      ok = ok && ((i >> up) & 1u) == 0u;
    }
    span = 3u;
    const uint32_t t = (uint32_t)t64;
    if (ok) {
      const float4 mn = g.bmin[t], mx = g.bmax[t];
      ok = pk_box_d2(box, v3(mn.x, mn.y, mn.z), v3(mx.x, mx.y, mx.z)) <= bound2;
    }
    const bool leaf = t + 1u >= nl;
    const uint64_t mi = ballot(ok && !leaf), ml = ballot(ok && leaf);
    pk_sync();  // the stack entries above have been read
    if (ok && !leaf) S.stack[sp + pk_rank(mi)] = t;
    sp += (uint32_t)__builtin_popcountll(mi);
    if (ok && leaf) S.leaf[pk_rank(ml)] = t;
    const uint32_t nleaf = (uint32_t)__builtin_popcountll(ml);
    pk_sync();
    for (uint32_t b0 = 0; b0 < nleaf; b0 += 64u >> lg) {
      const uint32_t slot = b0 + ((uint32_t)lane >> lg), idx = (uint32_t)lane & ((1u << lg) - 1u);
      bool in = slot < nleaf && idx < L;
      float4 p = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      uint32_t pos = 0u;
      if (in) {
        const uint32_t lf = S.leaf[slot];
        const uint32_t rank = lf >= first_deep ? lf - first_deep : ndeep + (lf - (nl - 1u));
        pos = rank * L + idx;
        in = pos < n;
        if (in) {
          p = g.tpts[pos];
          const V3f x = v3(p.x, p.y, p.z);
          in = pk_box_d2(box, x, x) <= bound2;
        }
      }
      const uint64_t m = ballot(in);
      const uint32_t c = (uint32_t)__builtin_popcountll(m);
      if (M + c > kPkCand) {
        pk_sync();
        if (!full(M)) return M;
        pk_sync();
        M = 0u;
      }
      if (in) S.cand[M + pk_rank(m)] = make_float4(p.x, p.y, p.z, u2f(pos));
      M += c;
    }
  }
  pk_sync();
  return M;
}

// Keeps the staged points within bound2 of the box (the count stage holds
// points up to the window tops).
__device__ __forceinline__ uint32_t pk_restage(PacketLds& S, int lane, const PkBox& box, float bound2, uint32_t M) {
  uint32_t out = 0;
  for (uint32_t c0 = 0; c0 < M; c0 += 64u) {
    const uint32_t c = c0 + (uint32_t)lane;
    bool in = c < M;
    float4 p = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (in) {
      p = S.cand[c];
      const V3f x = v3(p.x, p.y, p.z);
      in = pk_box_d2(box, x, x) <= bound2;
    }
    const uint64_t m = ballot(in);
    pk_sync();
    if (in) S.cand[out + pk_rank(m)] = p;
    out += (uint32_t)__builtin_popcountll(m);
  }
  pk_sync();
  return out;
}

// An upper bound, as a bucket top, of the k-th smallest d^2 from c: that of
// the first 128 points of the smallest node around c that holds k points.
// 0xffffffff when the map holds fewer than k points.  c is wave-uniform.
__device__ __forceinline__ uint32_t pk_upper_bound(const GatherMap& g, int lane, V3f c, uint32_t k) {
  if (g.n < k) return 0xffffffffu;
  uint32_t h = 0, lo = 0, hi = g.n;
  while (h + 1u < g.nl) {
    const KdNode nd = g.nodes[h];
    const int a = kd_axis(nd.meta);
    const float ca = a == 0 ? c.x : (a == 1 ? c.y : c.z);
    const uint32_t mid = lo + kd_left_count(nd.meta);
    const bool left = uniform(ca - nd.split < 0.0f ? 1u : 0u) != 0u;
    const uint32_t cn = left ? mid - lo : hi - mid;
    if (cn < k) break;
    h = left ? 2u * h + 1u : 2u * h + 2u;
    if (left) hi = mid;
    else lo = mid;
    h = uniform(h);
    lo = uniform(lo);
    hi = uniform(hi);
  }
  uint32_t d0 = 0x7fffffffu, d1 = 0x7fffffffu;
  if (lo + (uint32_t)lane < hi) {
    const float4 p = g.tpts[lo + (uint32_t)lane];
    d0 = f2u(dist2(c.x, c.y, c.z, p.x, p.y, p.z));
  }
  if (lo + 64u + (uint32_t)lane < hi) {
    const float4 p = g.tpts[lo + 64u + (uint32_t)lane];
    d1 = f2u(dist2(c.x, c.y, c.z, p.x, p.y, p.z));
  }
  uint32_t T = 0u;  // the smallest bucket that at least k of the points do not exceed
  for (uint32_t bit = 0x4000u; bit; bit >>= 1) {
    const uint32_t t = ((T | bit) << 16) - 1u;  // points in buckets below T | bit
    const uint32_t c2 = (uint32_t)(__builtin_popcountll(ballot(d0 <= t)) + __builtin_popcountll(ballot(d1 <= t)));
    if (c2 < k) T |= bit;
  }
  return (T << 16) | 0xffffu;
}

// Per-lane first-pass state of a query.
struct PkQuery {
  uint32_t state;  // 0: to be counted, 1: Q found, 2: fewer than k points within the cap (or guessed so)
  uint32_t K0;     // counting window [K0, K0 + 128)
  uint32_t top;    // search bound: the window's top or the cap (FP32 bits of d^2, inclusive)
  uint32_t blo, bhi;  // bisection: fewer than k points below blo << 16, at least k below bhi << 16
  bool bisect;
  uint32_t Q;
  __device__ void window(uint32_t hiq, uint32_t caph) {
    const uint32_t capq = caph >> 16;
    hiq = hiq < capq ? hiq : capq;
    K0 = hiq >= kPkBuckets - 1u ? hiq - (kPkBuckets - 1u) : 0u;
    const uint32_t t = ((K0 + kPkBuckets) << 16) - 1u;
    top = t < caph ? t : caph;
  }
};

// Gathers the queries of the wave's lanes with act set: q, the seed bucket of
// the lane's previous query (kPkNoSeed, or kPkFew: it had fewer than k
// neighbours within the cap) and the contributions `add`:
//   add.reset(), add(power, direction, d2);
//   add.of_lane(b): lane b's functor, in every lane; reduce(): the sums of all
//   lanes, in every lane; take(o): o's sums.
// SAME: the seed is of the same query in an earlier gather, most likely its
// bucket still; it is then summed from without a first pass, and the counts
// that the sum gathers say whether it was right (any seed gives the same
// result).  On return seed is this query's; m its number of neighbours (at
// most k) and r2 the k-th d^2 (the cap's when m < k).  Every lane of the wave
// calls it.
template <bool SAME, class Add>
__device__ __forceinline__ void packet_gather(const GatherMap& g, PacketLds& S, int lane, bool act, V3f q,
                                              uint32_t& seed, Add& add, uint32_t& m_out, float& r2_out) {
  const uint32_t k = (uint32_t)g.k, caph = f2u(g.rcap2);
  m_out = 0u;
  r2_out = g.rcap2;
  add.reset();
  uint64_t todo = ballot(act);
  if (g.n == 0u || todo == 0ull) return;
  PkQuery s;
  s.state = 0u;
  s.bisect = false;
  bool unseeded = act && seed == kPkNoSeed;
  bool guess = act && seed == kPkFew;  // count and sum in one pass, over the cap
  if (guess) s.state = 2u;
  else if (!unseeded) s.window(seed + kPkUp, caph);
  if (SAME && act && seed <= caph >> 16) {
    guess = true;
    s.state = 1u;
    s.Q = seed;
  }
  // Few queries at once (lists of rows far apart) use few lanes of the passes
  // below, so more of them go one at a time, and without seeds only the very
  // near ones share a stage (1.2M such rows of the fog map 4.5 -> 2.3 ms).
  // A group's half width in radii of its leader: without seeds 0.08, 0.15, 0.3:
  // batch 17.7, 18.8, 22.0, the rest the same; else 0.5, 0.75, 1.0: surfaces 5.2,
  // 5.6, 5.6, window 11.5, 10.4, 10.0, room 2.3, 2.0, 1.6, batch 20.7, 18.8, 18.2,
  // 5M unseeded rows 107, 110, 113.  Halved where the stage is too small, down
  // to the leader alone (from 0.01 or 0.1 of it: the same).
  const bool sparse = __builtin_popcountll(todo) <= 32;
  const uint32_t solo = sparse ? kPkSoloFew : kPkSolo;
  float shrink = 1.0f;
  uint32_t last_top = 0xffffffffu;  // search bound that held the last group's neighbours
  while (todo) {
    // ---- the group: the lanes near the first one left
    const int lead = (int)__builtin_ctzll(todo);
    const V3f c = v3(u2f(read_lane(f2u(q.x), lead)), u2f(read_lane(f2u(q.y), lead)), u2f(read_lane(f2u(q.z), lead)));
    const bool lead_un = ((ballot(unseeded) >> lead) & 1ull) != 0ull;
    const bool mine = ((todo >> lane) & 1ull) != 0ull;
    uint32_t lead_top;  // search bound of the leader
    bool rough = false;  // it is the last group's, not one of this place
    if (lead_un) {
      // the first group's from the tree; later ones start where the last one
      // ended (a window that is wrong moves)
      rough = last_top != 0xffffffffu;
      lead_top = rough ? last_top : pk_upper_bound(g, lane, c, k);
      lead_top = lead_top < caph ? lead_top : caph;
    } else {
      const uint32_t t = s.state == 2u ? caph : (s.state == 1u ? (s.Q << 16) | 0xffffu : s.top);
      lead_top = read_lane(t, lead);
      lead_top = lead_top < caph ? lead_top : caph;
    }
    const float rad = sqrt_(u2f(lead_top));
    const float dx = q.x - c.x, dy = q.y - c.y, dz = q.z - c.z;
    const float D = (sparse && lead_un ? 0.15f : 0.75f) * shrink * rad;
    bool grp = mine && (lane == lead || (shrink > 0.01f && __builtin_fabsf(dx) <= D && __builtin_fabsf(dy) <= D &&
                                         __builtin_fabsf(dz) <= D));
    // a lane without a seed: the leader's bound, moved to its query
    const bool fresh = grp && unseeded;
    auto fresh_window = [&](float r) {
      const float b = (r + sqrt_((dx * dx + dy * dy) + dz * dz)) * 1.0001f;
      const float b2 = b * b;
      s.window(b2 < g.rcap2 ? f2u(b2) >> 16 : caph >> 16, caph);
    };
    if (fresh) {
      fresh_window(rad);
      unseeded = false;
    }
    PkBox box;
    const float inf = u2f(0x7f800000u);
    box.lo = v3(pk_min(grp ? q.x : inf), pk_min(grp ? q.y : inf), pk_min(grp ? q.z : inf));
    box.hi = v3(pk_max(grp ? q.x : -inf), pk_max(grp ? q.y : -inf), pk_max(grp ? q.z : -inf));
    uint32_t M = 0, staged = 0;  // points in the stage; bound they are complete to (0: none)
    // ---- a small group: one query at a time, the lanes over the points
    if ((uint32_t)__builtin_popcountll(ballot(grp)) <= solo) {
      uint32_t bound = pk_umax(grp ? (s.state == 2u ? caph : (s.state == 1u ? (s.Q << 16) | 0xffffu : s.top)) : 0u);
      bound = bound < caph ? bound : caph;
      uint32_t lo = 0u, hi = LKEY_INF;  // bounds with too few points, with more than the stage holds
      bool whole = true;
      for (;;) {
        whole = true;
        M = pk_stage(g, S, lane, box, u2f(bound), [&](uint32_t) {
          whole = false;
          return false;
        });
        if (!whole) {
          pk_sync();
          if ((uint32_t)__builtin_popcountll(ballot(grp)) > 1u) break;  // the passes below, in pieces
          // one query: within its own bound, then by bisection
          if (rough && lo == 0u) {
            rough = false;
            const uint32_t ub = pk_upper_bound(g, lane, c, k);
            bound = ub < bound ? ub : bound;
          } else {
            hi = bound;
            if (hi - lo < 2u) break;
            bound = lo == 0u && hi > (2u << 23) ? hi - (1u << 23) : lo + (hi - lo) / 2u;
          }
          continue;
        }
        uint32_t d[kPkCand / 64];
        uint64_t left = ballot(grp) & todo;
        uint32_t most = k;  // the fewest points that one of these has
        bool more = false;  // a query has fewer than k points under a bound below the cap
        while (left) {
          const int b = (int)__builtin_ctzll(left);
          left &= left - 1ull;
          const V3f x = v3(u2f(read_lane(f2u(q.x), b)), u2f(read_lane(f2u(q.y), b)), u2f(read_lane(f2u(q.z), b)));
          uint32_t n_in = 0u;
#pragma unroll
          for (uint32_t j = 0; j < kPkCand / 64; ++j) {
            d[j] = LKEY_INF;
            if (j * 64u < M) {
              const uint32_t c0 = j * 64u + (uint32_t)lane;
              const float4 p = S.cand[c0];
              const uint32_t e = f2u(dist2(x.x, x.y, x.z, p.x, p.y, p.z));
              if (c0 < M && e <= bound) d[j] = e;
              n_in += (uint32_t)__builtin_popcountll(ballot(d[j] != LKEY_INF));
            }
          }
          if (n_in < k && bound != caph) {
            more = true;
            most = most < n_in ? most : n_in;
            continue;
          }
          uint32_t dk = caph;  // points up to dk contribute, but of those at dk itself only the first `at_dk`
          uint32_t at_dk = LKEY_INF;
          if (n_in >= k) {
            // dk: the largest value that fewer than k points lie below, by
            // bisection over the five octaves under the bound, or all when it
            // is not there; a value with exactly k points below it ends it
            auto below_of = [&](uint32_t t) {
              uint32_t n = 0u;
#pragma unroll
              for (uint32_t j = 0; j < kPkCand / 64; ++j)
                if (j * 64u < M) n += (uint32_t)__builtin_popcountll(ballot(d[j] < t));
              return n;
            };
            const uint32_t oct = bound & 0x7f800000u;
            dk = oct > (4u << 23) ? oct - (4u << 23) : 0u;
            uint32_t bit = 1u << 25;
            if (below_of(dk) >= k) {
              dk = 0u;
              bit = 0x40000000u;
            }
            uint32_t cut = 0u;
            for (; bit; bit >>= 1) {
              const uint32_t n = below_of(dk + bit);
              if (n == k) {
                cut = dk + bit;
                break;
              }
              if (n < k) dk += bit;
            }
            uint32_t below = 0u, upto = k;
            if (cut) {
              uint32_t m = 0u;
#pragma unroll
              for (uint32_t j = 0; j < kPkCand / 64; ++j)
                if (j * 64u < M && d[j] < cut) m = m > d[j] ? m : d[j];
              dk = pk_umax(m);
            } else {
              below = below_of(dk);
              upto = below_of(dk + 1u);
            }
            if (upto > k) {
              // equal distances at the k-th: by photon index
              uint32_t idx[kPkCand / 64];
#pragma unroll
              for (uint32_t j = 0; j < kPkCand / 64; ++j)
                idx[j] = d[j] == dk ? f2u(g.tpts[f2u(S.cand[j * 64u + (uint32_t)lane].w)].w) : LKEY_INF;
              at_dk = 0u;  // the largest index that fewer than k - below of them lie below
              for (uint32_t bit = 0x80000000u; bit; bit >>= 1) {
                uint32_t n = 0u;
#pragma unroll
                for (uint32_t j = 0; j < kPkCand / 64; ++j)
                  n += (uint32_t)__builtin_popcountll(ballot(idx[j] < (at_dk | bit)));
                if (n < k - below) at_dk |= bit;
              }
#pragma unroll
              for (uint32_t j = 0; j < kPkCand / 64; ++j)
                if (d[j] == dk && idx[j] > at_dk) d[j] = LKEY_INF;
            }
          }
          Add part = add.of_lane(b);
          part.reset();
#pragma unroll
          for (uint32_t j = 0; j < kPkCand / 64; ++j) {
            if (j * 64u < M && d[j] <= dk) {
              V3f pw, dir;
              load_payload_tree(g, f2u(S.cand[j * 64u + (uint32_t)lane].w), pw, dir);
              part(pw, dir, u2f(d[j]));
            }
          }
          part.reduce();
          if (lane == b) {
            add.take(part);
            m_out = n_in < k ? n_in : k;
            r2_out = u2f(dk);
            seed = n_in < k ? kPkFew : dk >> 16;
          }
          last_top = n_in < k ? caph : dk | 0xffffu;
          todo &= ~(1ull << b);
        }
        if (!more) break;
        pk_sync();
        lo = bound;
        const float b2 = (2u * most >= k ? 1.5f : (4u * most >= k ? 2.0f : 4.0f)) * u2f(bound);
        bound = hi != LKEY_INF ? (lo + (hi - lo) / 2u) : (b2 < g.rcap2 ? f2u(b2) : caph);
        if (hi - lo < 2u) {
          whole = false;
          break;
        }
      }
      pk_sync();
      if (whole) continue;
      M = 0u;  // more points at one distance than the stage holds: the passes below, in pieces
      grp = grp && ((todo >> lane) & 1ull) != 0ull;
    }
    // ---- first pass: count until every lane of the group has its bucket
    for (;;) {
      const bool need = grp && s.state == 0u;
      if (ballot(need) == 0ull) break;
      uint32_t base = 0u, width = 0u, below = 0u, inwin = 0u;
      if (need) {
        base = s.K0 << 16;
        width = s.top - base + 1u;
        if (s.bisect) {
          base = ((s.blo + s.bhi) >> 1) << 16;
          base = base < caph + 1u ? base : caph + 1u;
          width = 0u;
        }
      }
#pragma unroll
      for (uint32_t w = 0; w < kPkBuckets / 8; ++w) S.cnt[w * 64 + lane] = 0u;
      auto count = [&](uint32_t m) {
        for (uint32_t c0 = 0; c0 < m; c0 += 4u) {
          float4 p[4];
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j) p[j] = S.cand[c0 + j];
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j) {
            if (c0 + j >= m) break;
            const uint32_t d = f2u(dist2(q.x, q.y, q.z, p[j].x, p[j].y, p[j].z));
            const uint32_t t = d - base;
            below += d < base ? 1u : 0u;
            const bool in = t < width;
            inwin += in ? 1u : 0u;
            if (in)
              __hip_atomic_fetch_add(&S.cnt[(t >> 19) * 64u + (uint32_t)lane], 1u << ((t >> 14) & 28u),
                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
          }
        }
        return true;
      };
      const uint32_t bound = pk_umax(need ? s.top : 0u);
      if (staged < bound) {
        bool whole = true;
        uint32_t pieces = 0u;
        M = pk_stage(g, S, lane, box, u2f(bound), [&](uint32_t m) {
          whole = false;
          return rough && ++pieces > 4u ? false : count(m);  // 1, 4, 16: those rows 112.9, 110.1, 110.0
        });
        staged = whole ? bound : 0u;
        if (pieces > 4u) {
          // far too many points under a bound of another place: this place's
          rough = false;
          pk_sync();
          uint32_t ub = pk_upper_bound(g, lane, c, k);
          ub = ub < caph ? ub : caph;
          if (fresh) fresh_window(sqrt_(u2f(ub)));
          continue;
        }
      }
      count(M);
      if (!need) continue;
      if (s.bisect) {
        const uint32_t mid = (s.blo + s.bhi) >> 1;
        if (below >= k) s.bhi = mid;
        else s.blo = mid;
      } else if (below + inwin < k) {
        if (s.top == caph) {
          s.state = 2u;
        } else {
          s.window(s.K0 + 2u * kPkBuckets - 1u, caph);
        }
        continue;
      } else if (below >= k) {
        s.window(s.K0 - 1u, caph);
        continue;
      } else {
        // the first word, then the first counter in it, at which the running
        // count reaches what is left of k
        const uint32_t left = k - below;
        uint32_t cum = 0u, wq = 0u, vq = 0u, before = 0u;
        bool found = false;
#pragma unroll
        for (uint32_t w = 0; w < kPkBuckets / 8; ++w) {
          const uint32_t v = S.cnt[w * 64 + lane];
          const uint32_t b = (v & 0x0F0F0F0Fu) + ((v >> 4) & 0x0F0F0F0Fu);
          const uint32_t cn = cum + ((b * 0x01010101u) >> 24);
          if (!found && cn >= left) {
            found = true;
            wq = w;
            vq = v;
            before = cum;
          }
          cum = cn;
        }
        if (cum == inwin) {
          uint32_t run = before, at = 0u;
#pragma unroll
          for (int j = 0; j < 7; ++j) {
            run += (vq >> (4 * j)) & 15u;
            at += run < left ? 1u : 0u;
          }
          s.Q = s.K0 + 8u * wq + at;
          s.state = 1u;
          continue;
        }
        // a counter passed 15 and carried, which lowers the sum of the
        // counters and never raises it: bisect the window by plain counts
        s.bisect = true;
        s.blo = s.K0;
        s.bhi = s.K0 + kPkBuckets;
      }
      if (s.bhi - s.blo == 1u) {
        s.Q = s.blo;
        s.bisect = false;
        s.state = 1u;
      }
    }
    // ---- second pass: sums
    uint32_t Qb = 0u, eqw = 0u;
    if (grp) {
      if (s.state == 1u) {
        Qb = s.Q << 16;
        eqw = caph - Qb < 0xffffu ? caph - Qb + 1u : 0x10000u;
      } else {
        Qb = caph + 1u;
      }
    }
    const uint32_t bound = pk_umax(grp ? Qb + eqw - 1u : 0u);
    uint32_t nin = 0u, ntie = 0u, tie_lo = 0u, tie_hi = 0u;
    auto sum = [&](uint32_t m) {
      for (uint32_t c0 = 0; c0 < m; c0 += 64u) {
        const uint32_t cl = c0 + (uint32_t)lane;
        pk_sync();
        if (cl < m) {
          V3f pw, dir;
          load_payload_tree(g, f2u(S.cand[cl].w), pw, dir);
          S.pay.a[lane] = make_float4(pw.x, pw.y, pw.z, dir.x);
          S.pay.b[lane] = make_float2(dir.y, dir.z);
        }
        pk_sync();
        const uint32_t ce = m - c0 < 64u ? m - c0 : 64u;
        for (uint32_t c1 = 0; c1 < ce; c1 += 4u) {
          float4 p[4];
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j) p[j] = S.cand[c0 + c1 + j];
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j) {
            if (c1 + j >= ce) break;
            const uint32_t d = f2u(dist2(q.x, q.y, q.z, p[j].x, p[j].y, p[j].z));
            const uint32_t t = d - Qb;
            if ((int)t < 0) {
              const float4 a = S.pay.a[c1 + j];
              const float2 b = S.pay.b[c1 + j];
              add(v3(a.x, a.y, a.z), v3(a.w, b.x, b.y), u2f(d));
              ++nin;
            }
            if (t < eqw) {
              tie_hi = (tie_hi << 8) | (tie_lo >> 24);
              tie_lo = (tie_lo << 8) | (c0 + c1 + j);
              ++ntie;
            }
          }
        }
      }
      return true;
    };
    bool whole = true;  // the stage holds every point of the second pass
    if (staged >= bound && staged != 0u) {
      M = pk_restage(S, lane, box, u2f(bound), M);
      whole = M <= 256u;
    } else {
      M = pk_stage(g, S, lane, box, u2f(bound), [&](uint32_t) {
        whole = false;
        return false;
      });
      whole = whole && M <= 256u;
    }
    if (!whole && __builtin_popcountll(ballot(grp)) > 1) {
      // too many points for one stage: a smaller group (what was counted stays)
      shrink *= 0.5f;
      continue;
    }
    if (whole) {
      sum(M);
    } else {
      M = pk_stage(g, S, lane, box, u2f(bound), sum);
      sum(M);
    }
    // ---- the (d^2, index) smallest of the bucket-Q points that complete k
    bool done = grp;
    if (done && guess && (nin >= k || (s.state == 1u && nin + ntie < k))) {
      // a wrong guess: k points within the cap after all (count from the cap
      // down), or the seed's bucket does not hold the k-th neighbour
      s.window(s.state == 1u ? s.Q + kPkUp : caph >> 16, caph);
      guess = false;
      s.state = 0u;
      add.reset();
      done = false;
    }
    const bool full = done && s.state == 1u;
    const uint32_t want = full ? k - nin : 0u;  // nin: points in buckets below Q
    const bool small = whole && ntie <= kPkTie;
    const uint32_t tmax = pk_umax(full && small ? ntie : 0u);
    if (tmax) {
      pk_sync();
      for (uint32_t e = 0; e < tmax; ++e) {
        if (full && small && e < ntie) {
          const float4 p = S.cand[((e < 4u ? tie_lo : tie_hi) >> (8u * (e & 3u))) & 255u];
          S.tie[e * 64 + lane] = f2u(dist2(q.x, q.y, q.z, p.x, p.y, p.z));
        }
      }
      uint32_t kth = 0u;
      for (uint32_t e = 0; e < tmax; ++e) {
        if (!(full && small && e < ntie)) continue;
        const uint32_t de = S.tie[e * 64 + lane];
        const uint32_t ce = ((e < 4u ? tie_lo : tie_hi) >> (8u * (e & 3u))) & 255u;
        uint32_t rank = 0u;
        for (uint32_t f = 0; f < ntie; ++f) {
          const uint32_t df = S.tie[f * 64 + lane];
          bool less = df < de;
          if (df == de && f != e) {  // equal distances: by photon index
            const uint32_t cf = ((f < 4u ? tie_lo : tie_hi) >> (8u * (f & 3u))) & 255u;
            less = f2u(g.tpts[f2u(S.cand[cf].w)].w) < f2u(g.tpts[f2u(S.cand[ce].w)].w);
          }
          rank += less ? 1u : 0u;
        }
        if (rank < want) {
          V3f pw, dir;
          load_payload_tree(g, f2u(S.cand[ce].w), pw, dir);
          add(pw, dir, u2f(de));
          kth = kth > de ? kth : de;
        }
      }
      if (full && small) r2_out = u2f(kth);
    }
    // more bucket points than a lane keeps: one exact pass per neighbour
    const bool slow = full && !small;
    if (ballot(slow)) {
      uint32_t kd = 0u, ki = 0u;
      bool any = false;
      const uint32_t rounds = pk_umax(slow ? want : 0u);
      for (uint32_t r = 0; r < rounds; ++r) {
        uint32_t bd = LKEY_INF, bi = LKEY_INF, bpos = 0u;
        const bool on = slow && r < want;
        auto next = [&](uint32_t m) {
          for (uint32_t c0 = 0; c0 < m; ++c0) {
            const float4 p = S.cand[c0];
            const uint32_t d = f2u(dist2(q.x, q.y, q.z, p.x, p.y, p.z));
            if (on && d - Qb < eqw) {
              const uint32_t idx = f2u(g.tpts[f2u(p.w)].w);
              if ((!any || key_less(kd, ki, d, idx)) && key_less(d, idx, bd, bi)) {
                bd = d;
                bi = idx;
                bpos = f2u(p.w);
              }
            }
          }
          return true;
        };
        if (!whole) M = pk_stage(g, S, lane, box, u2f(bound), next);
        next(M);
        if (on && bi != LKEY_INF) {
          V3f pw, dir;
          load_payload_tree(g, bpos, pw, dir);
          add(pw, dir, u2f(bd));
          kd = bd;
          ki = bi;
          any = true;
        }
      }
      if (slow) r2_out = u2f(kd);
    }
    if (done) {
      m_out = full ? k : nin;
      seed = full ? s.Q : kPkFew;
    }
    if (ballot(done)) last_top = pk_umax(done ? (full ? ((s.Q + kPkUp) << 16) | 0xffffu : caph) : 0u);
    todo &= ~ballot(done);
    shrink = shrink < 1.0f ? 2.0f * shrink : 1.0f;
    pk_sync();  // the stage is rewritten
  }
}

}  // namespace pm
