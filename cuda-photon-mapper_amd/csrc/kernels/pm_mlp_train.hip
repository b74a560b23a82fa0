// pm_mlp_train.hip -- the learned cache's training pass (forward, loss,
// backward, weight and bias gradients) on gfx950, three launches a step with
// Adam: k_fwd_bwd takes 64 rows through all layers and back with the
// activations in LDS, k_wgrad computes the five layers' weight gradients.
//
// No reference counterpart (the reference has no learned component).
//
// Every product of a training step has the form C[m][n] = sum_k A[m][k] B[n][k]
// once each operand is kept in the layout that makes K its contiguous axis:
//   forward      H_l [rows x out] = X_{l} [rows x in] . W_l [out x in]^T
//   delta        D_{l-1} [rows x in] = D_l [rows x out] . (W_l^T) [in x out]^T
//   weight grad  dW_l [out x in] = (D_l^T) [out x rows] . (X_l^T) [in x rows]^T
// so k_fwd_bwd writes the encoded inputs, the activations and the deltas
// transposed (the weight gradients' operands), and the BF16 weights are kept
// in both orders (W and W^T, refreshed by Adam).  Every element of a product
// accumulates its K in ascending steps of 32 from zero on
// v_mfma_f32_16x16x32_bf16, then bias, ReLU or mask, then BF16: which wave
// computes it, and in which tile, does not change its bits.  The weight
// gradients split the batch (K) over slices that write FP32 partial tiles, and
// the bias gradients (row sums of D^T) likewise; the slices of every layer are
// added in slice order (deterministic), by one kernel or by Adam itself.
#include "pm_kernels.h"
#include "pm_mlp.h"
#include "pm_wave.h"

namespace pm {

namespace {

// Barrier for data exchanged through LDS only: it does not wait for the
// wave's global loads and stores, which no other wave of the workgroup reads.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- forward and backward
// A training batch from the inputs to the deltas in one launch.  A workgroup
// of 16 waves takes 64 rows: it encodes them, runs the five layers, forms the
// loss gradient (with t = log(1 + max(target, 0)), d = y - t per channel,
// dy = 2 d / (3 rows), row_err = sum of d^2) and takes it back through the
// hidden layers, D_{l-1} = (D_l . W_l) x [H_{l-1} > 0].  When esum is set,
// each row's row_err (capped at 1e6) is added in 2^-24 fixed point to the
// error tracker's cell of its input, and the cell's count incremented (integer
// atomics: the bins do not depend on the order).
//
// A batch is 128 to 256 workgroups of one per CU, so the time is the chain of
// nine dependent products of one tile, and what bounds it is latency: the
// next product's weights are loaded into registers before a product's K loop
// and written to the other LDS buffer after it (one barrier a product), the
// ReLU masks stay in registers as one bit per element (the deltas have the
// activations' shape and lane mapping), and an element's four consecutive
// rows are stored to the transposed arrays from registers, 8 bytes at a time.
// Wave w computes n-tile w % 8 of m-tiles 2 (w / 8) and 2 (w / 8) + 1.
// Two kernels of 4 waves (forward; backward with H, y and dy through memory)
// took 38 + 32 us for 8,192 rows and 138 + 115 us for 65,536; this one 39 us
// for 16,384.
constexpr int FF_XS = MLP_KPAD + 8;  // LDS row length (bf16) of X and W1
constexpr int FF_HS = MLP_HID + 8;   // of the hidden activations, deltas and W2..W5
constexpr int FB_THREADS = 1024;
constexpr int FB_YS = 4;             // LDS row length (floats) of y and of the targets
constexpr size_t FB_LDS = 2u * (64u * FF_XS + 2u * 64u * FF_HS + 128u * FF_XS + 128u * FF_HS) + 4u * 2u * 64u * FB_YS;
static_assert(FB_LDS <= 160u * 1024u, "one workgroup's LDS");

// Two FP32 values to BF16, round to nearest even (one instruction; the bits of
// f32_to_bf16 for finite values).
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  const bf16x2_t v = __builtin_convertvector((f32x2_t{a, b}), bf16x2_t);
  return __builtin_bit_cast(uint32_t, v);
}

struct FwdBwdArgs {
  uint32_t rows;
  uint32_t ld;
  const float* in;                       // [rows x IN] query rows
  const float* target;                   // [rows x OUT]
  const uint16_t* w[MLP_LAYERS];
  const uint16_t* wbt[MLP_LAYERS];       // W_l^T [kin x nout]
  const float* b[MLP_LAYERS];
  uint16_t* XT;                          // [KPAD x ld] encoded inputs, transposed
  uint16_t* HT[MLP_HIDDEN_LAYERS];       // [HID x ld]
  uint16_t* dT[MLP_HIDDEN_LAYERS];       // [HID x ld]
  uint16_t* dyT;                         // [OUTPAD x ld]
  float* row_err;                        // [rows]
  unsigned long long* esum;              // error tracker (null: none)
  unsigned int* ecnt;
};

// Weights of one product, on their way from memory to LDS through registers:
// `nrow` rows of `ncol` (a multiple of 8) at src, row length `ls` in LDS.
struct WStage {
  uint4 v[2];
  __device__ __forceinline__ void load(const uint16_t* src, int nrow, int ncol) {
    const int per = ncol / 8;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = (int)threadIdx.x + j * FB_THREADS;
      if (i < nrow * per) v[j] = *(const uint4*)&src[(size_t)i * 8];
    }
  }
  __device__ __forceinline__ void store(uint16_t* dst, int nrow, int ncol) const {
    const int per = ncol / 8;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = (int)threadIdx.x + j * FB_THREADS;
      if (i < nrow * per) *(uint4*)&dst[(i / per) * FF_HS + (i % per) * 8] = v[j];
    }
  }
};

// This wave's two 16x16 tiles of act . Ws^T over K = kin.
__device__ __forceinline__ void fb_product(const uint16_t* act, int as, const uint16_t* Ws, int ws, int kin, int wave,
                                           int r16, int q, f32x4_t acc[2]) {
  acc[0] = acc[1] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  const uint16_t* a0 = &act[(32 * (wave >> 3) + r16) * as + 8 * q];
  const uint16_t* b0 = &Ws[(16 * (wave & 7) + r16) * ws + 8 * q];
  for (int ks = 0; ks < kin; ks += 32) {
    const uint4 va0 = *(const uint4*)&a0[ks], va1 = *(const uint4*)&a0[16 * as + ks], vb = *(const uint4*)&b0[ks];
    acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t*)&va0, *(const bf16x8_t*)&vb, acc[0], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t*)&va1, *(const bf16x8_t*)&vb, acc[1], 0, 0, 0);
  }
}

// Stores the wave's elements h (rows 16 t + 4 q + 0..3 of column n, in pairs)
// to the LDS tile and, as 8-byte groups, to the transposed array.
__device__ __forceinline__ void fb_store(const uint32_t h[2][2], uint16_t* out, uint16_t* T, uint32_t ld, uint32_t m0,
                                         int wave, int r16, int q) {
  const int n = 16 * (wave & 7) + r16;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int m = 32 * (wave >> 3) + 16 * t + 4 * q;
    if (out) {
#pragma unroll
      for (int e = 0; e < 4; ++e) out[(m + e) * FF_HS + n] = (uint16_t)(h[t][e >> 1] >> (16 * (e & 1)));
    }
    *(uint2*)&T[(size_t)n * ld + m0 + (uint32_t)m] = make_uint2(h[t][0], h[t][1]);
  }
}

__global__ void __launch_bounds__(FB_THREADS) k_fwd_bwd(FwdBwdArgs A) {
  extern __shared__ __align__(16) unsigned char fl[];
  uint16_t* const Xs = (uint16_t*)fl;               // [64][FF_XS]
  uint16_t* const Hs0 = Xs + 64 * FF_XS;            // [64][FF_HS] each, ping-pong
  uint16_t* const Hs1 = Hs0 + 64 * FF_HS;
  uint16_t* const WA = Hs1 + 64 * FF_HS;            // [128][FF_XS]
  uint16_t* const WB = WA + 128 * FF_XS;            // [128][FF_HS]
  float* const ys = (float*)(WB + 128 * FF_HS);     // [64][FB_YS] the outputs
  float* const ts = ys + 64 * FB_YS;                // [64][FB_YS] log(1 + max(target, 0))
  const int tid = (int)threadIdx.x, lane = lane_id(), wave = tid >> 6, r16 = lane & 15, q = lane >> 4;
  const uint32_t m0 = blockIdx.x * 64u, rows = A.rows;
  const bool ok = m0 + (uint32_t)lane < rows;       // this lane's row, where a wave's lanes are the rows
  const float* const in = A.in + (size_t)(m0 + (uint32_t)lane) * MLP_IN;
  uint4 w0[4];  // W1 on its way to LDS
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int v = tid + j * FB_THREADS;
    if (v < MLP_HID * (MLP_KPAD / 8)) w0[j] = *(const uint4*)&A.w[0][(size_t)v * 8];
  }
  // the tile's encoded inputs: {sin, cos}(2 pi 2^(b-1) v) of each input v at
  // column 24 i + 2b (+1), padding columns and rows past the batch zero; a
  // wave takes four bands of an input of the 64 rows at a time
  for (int i = wave; i < MLP_IN * 3; i += FB_THREADS / 64) {
    const int v = i / 3, b0 = 4 * (i % 3);
    uint16_t* xt = A.XT + (size_t)(v * 2 * MLP_BANDS) * A.ld + m0 + (uint32_t)lane;
    const float x = ok ? in[v] : 0.0f;
    float scale = 0.5f * (float)(1 << b0);
#pragma unroll
    for (int b = b0; b < b0 + 4; ++b) {
      float sn, cs;
      sincos_turns(x * scale, &sn, &cs);
      const uint32_t p = ok ? bf16_pair(sn, cs) : 0u;
      *(uint32_t*)&Xs[lane * FF_XS + v * 2 * MLP_BANDS + 2 * b] = p;
      xt[(size_t)(2 * b) * A.ld] = (uint16_t)p;
      xt[(size_t)(2 * b + 1) * A.ld] = (uint16_t)(p >> 16);
      scale *= 2.0f;
    }
  }
  // the waves with one encoding task fewer: the targets, the zero rows of X^T
  // and dy^T, and the rows' error cells
  uint32_t cell = 0u;
  if (wave >= 11 && wave < 11 + MLP_OUT) {
    const int c = wave - 11;
    ts[lane * FB_YS + c] = ok ? log_(1.0f + fmax_(A.target[(size_t)(m0 + (uint32_t)lane) * MLP_OUT + c], 0.0f)) : 0.0f;
  } else if (wave == 14) {
    uint16_t* xt = A.XT + (size_t)MLP_FEAT * A.ld + m0 + (uint32_t)lane;
#pragma unroll
    for (int k = 0; k < MLP_KPAD - MLP_FEAT; ++k) xt[(size_t)k * A.ld] = 0;
    *(uint4*)&Xs[lane * FF_XS + MLP_FEAT] = make_uint4(0u, 0u, 0u, 0u);
  } else if (wave == 15) {
    for (int c = MLP_OUT; c < MLP_OUTPAD; ++c)
      if (ok) A.dyT[(size_t)c * A.ld + m0 + (uint32_t)lane] = 0;
    if (ok && A.esum) cell = err_cell(in);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int v = tid + j * FB_THREADS;
    if (v < MLP_HID * (MLP_KPAD / 8)) *(uint4*)&WA[(v / (MLP_KPAD / 8)) * FF_XS + (v % (MLP_KPAD / 8)) * 8] = w0[j];
  }
  lds_barrier();
  // ---- forward: hidden layers, the weights alternately in WA and WB
  WStage ww;
  uint32_t mask = 0u;  // bit 8 l + 4 t + e: element (t, e) of H_l is positive
  f32x4_t acc[2];
  uint32_t h[2][2];
  const int n = 16 * (wave & 7) + r16;
#pragma unroll
  for (int l = 0; l < MLP_HIDDEN_LAYERS; ++l) {
    const int nnext = l + 1 < MLP_HIDDEN_LAYERS ? MLP_HID : MLP_OUTPAD;
    ww.load(A.w[l + 1], nnext, MLP_HID);
    const float bias = A.b[l][n];
    const uint16_t* act = l == 0 ? Xs : ((l & 1) ? Hs0 : Hs1);
    fb_product(act, l == 0 ? FF_XS : FF_HS, (l & 1) ? WB : WA, l == 0 ? FF_XS : FF_HS, l == 0 ? MLP_KPAD : MLP_HID,
               wave, r16, q, acc);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        float v0 = acc[t][e] + bias, v1 = acc[t][e + 1] + bias;
        v0 = v0 > 0.0f ? v0 : 0.0f;
        v1 = v1 > 0.0f ? v1 : 0.0f;
        const uint32_t p = bf16_pair(v0, v1);
        h[t][e >> 1] = p;
        mask |= (p & 0xffffu) != 0u ? 1u << (8 * l + 4 * t + e) : 0u;
        mask |= p >= 0x10000u ? 2u << (8 * l + 4 * t + e) : 0u;
      }
    fb_store(h, (l & 1) ? Hs1 : Hs0, A.HT[l], A.ld, m0, wave, r16, q);
    ww.store((l & 1) ? WA : WB, nnext, MLP_HID);
    lds_barrier();
  }
  // ---- output layer: 16 columns (3 used), no ReLU, FP32 y; waves 0..3 take
  // an m-tile each.  H_4 is in Hs1, W_5 in WA; W_5^T goes to WB, its K of 16
  // zero-padded to 32
  ww.load(A.wbt[MLP_HIDDEN_LAYERS], MLP_HID, MLP_OUTPAD);
  if (wave < 4) {
    f32x4_t o = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    for (int ks = 0; ks < MLP_HID; ks += 32) {
      const uint4 va = *(const uint4*)&Hs1[(16 * wave + r16) * FF_HS + ks + 8 * q];
      const uint4 vb = *(const uint4*)&WA[r16 * FF_HS + ks + 8 * q];
      o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t*)&va, *(const bf16x8_t*)&vb, o, 0, 0, 0);
    }
    const float bias = A.b[MLP_HIDDEN_LAYERS][r16];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (r16 < MLP_OUT) ys[(16 * wave + 4 * q + e) * FB_YS + r16] = o[e] + bias;
  }
  ww.store(WB, MLP_HID, MLP_OUTPAD);
  if (tid < MLP_HID * 2) *(uint4*)&WB[(tid >> 1) * FF_HS + MLP_OUTPAD + (tid & 1) * 8] = make_uint4(0u, 0u, 0u, 0u);
  lds_barrier();
  // ---- loss gradient and error bins, the last wave's lanes the rows; dy (zero
  // past the batch and in the padding columns) into Hs0
  WStage wn;
  wn.load(A.wbt[MLP_HIDDEN_LAYERS - 1], MLP_HID, MLP_HID);
  float e2 = 0.0f;
  if (wave == 15) {
    const float inv = 2.0f / (float)((int)rows * MLP_OUT);
    uint16_t g[MLP_OUT] = {0, 0, 0};
    if (ok) {
#pragma unroll
      for (int c = 0; c < MLP_OUT; ++c) {
        const float d = ys[lane * FB_YS + c] - ts[lane * FB_YS + c];
        e2 += d * d;
        g[c] = f32_to_bf16(d * inv);
      }
    }
    *(uint4*)&Hs0[lane * FF_HS] = make_uint4((uint32_t)g[0] | ((uint32_t)g[1] << 16), (uint32_t)g[2], 0u, 0u);
#pragma unroll
    for (int j = 8; j < 32; j += 8) *(uint4*)&Hs0[lane * FF_HS + j] = make_uint4(0u, 0u, 0u, 0u);
    if (ok) {
#pragma unroll
      for (int c = 0; c < MLP_OUT; ++c) A.dyT[(size_t)c * A.ld + m0 + (uint32_t)lane] = g[c];
      A.row_err[m0 + (uint32_t)lane] = e2;
    }
  }
  lds_barrier();
  if (wave == 15 && ok && A.esum) {
    const float e = e2 < 1e6f ? e2 : 1e6f;
    atomicAdd(&A.esum[cell], (unsigned long long)(e * 16777216.0f));
    atomicAdd(&A.ecnt[cell], 1u);
  }
  // ---- backward: W_l^T alternately in WB (l = 4, 2) and WA (l = 3, 1), the
  // deltas in Hs0 (D_4 = dy, D_2) and Hs1 (D_3, D_1)
#pragma unroll
  for (int l = MLP_HIDDEN_LAYERS; l >= 1; --l) {
    const bool even = (l & 1) == 0;
    fb_product(even ? Hs0 : Hs1, FF_HS, even ? WB : WA, FF_HS, l == MLP_HIDDEN_LAYERS ? 32 : MLP_HID, wave, r16, q, acc);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        const uint32_t b = mask >> (8 * (l - 1) + 4 * t + e);
        h[t][e >> 1] = bf16_pair(b & 1u ? acc[t][e] : 0.0f, b & 2u ? acc[t][e + 1] : 0.0f);
      }
    fb_store(h, l > 1 ? (even ? Hs1 : Hs0) : nullptr, A.dT[l - 1], A.ld, m0, wave, r16, q);
    if (l > 1) {
      wn.store(even ? WA : WB, MLP_HID, MLP_HID);
      if (l > 2) wn.load(A.wbt[l - 2], MLP_HID, MLP_HID);
      lds_barrier();
    }
  }
}

// ---------------------------------------------------------------- weight gradients
// The five layers' dW_l [nout x kin] = A [nout x rows] . B [kin x rows]^T in
// one launch, the rows split into slices: a workgroup of 8 waves takes one
// slice of a layer's whole output (two halves of kin for layer 0), so an
// operand is read once per slice, and writes the FP32 partial; the first half
// also the row sums of A (the bias gradients), summed in ascending k.  K is
// staged through LDS 128 at a time; the next stage's loads are in registers
// while the current one is multiplied.  64x64 tiles of 4 waves without the
// prefetch took 17 us for 8,192 rows and 96 us for 65,536.
constexpr int WG_THREADS = 512;
constexpr int WG_KC = 128;
constexpr int WG_LS = WG_KC + 8;  // LDS row length (bf16), padded
constexpr int WG_VEC = 2 * 128 * (WG_KC / 8) / WG_THREADS;  // 16-byte vectors per thread and stage

struct WgradArgs {
  const uint16_t* A[MLP_LAYERS];  // D_l^T [nout x ld]
  const uint16_t* B[MLP_LAYERS];  // X^T or H_{l-1}^T [kin x ld]
  float* part[MLP_LAYERS];        // [slices][nout][kin]
  float* bpart[MLP_LAYERS];       // [slices][nout]
  uint32_t rows, ld, kps;         // kps: rows per slice
  int slices;
};

// Stage vector j of this thread: rows [0, M) of A, then N rows of B, k0 .. k0 + 127.
__device__ __forceinline__ uint4 wg_load(const uint16_t* A, int M, const uint16_t* B, int N, uint32_t ld, int j,
                                         uint32_t k0, uint32_t k_end) {
  const int i = (int)threadIdx.x + j * WG_THREADS, r = i / (WG_KC / 8), kk = (i % (WG_KC / 8)) * 8;
  uint4 q = make_uint4(0u, 0u, 0u, 0u);
  const uint16_t* row = r < 128 ? (r < M ? A + (size_t)r * ld : nullptr) : (r - 128 < N ? B + (size_t)(r - 128) * ld : nullptr);
  const uint32_t k = k0 + (uint32_t)kk;
  if (row && k + 8u <= k_end) {
    q = *(const uint4*)&row[k];
  } else if (row && k < k_end) {
    uint32_t e[8];
#pragma unroll
    for (uint32_t t = 0; t < 8; ++t) e[t] = k + t < k_end ? row[k + t] : 0u;
    q = make_uint4(e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16));
  }
  return q;
}

__global__ void __launch_bounds__(WG_THREADS) k_wgrad(WgradArgs g) {
  __shared__ __align__(16) uint16_t S[256 * WG_LS];  // rows 0..127: A, 128..255: B
  const int lane = lane_id(), wave = (int)(threadIdx.x >> 6), r16 = lane & 15, q = lane >> 4;
  // products: layer 0's two halves, then layers 1..4; slices fastest
  const int z = (int)blockIdx.x % g.slices, prod = (int)blockIdx.x / g.slices;
  const int l = prod < 2 ? 0 : prod - 1, n0 = prod == 1 ? MLP_KPAD / 2 : 0;
  const int M = l == MLP_HIDDEN_LAYERS ? MLP_OUTPAD : MLP_HID, kin = l == 0 ? MLP_KPAD : MLP_HID;
  const int N = l == 0 ? MLP_KPAD / 2 : MLP_HID;
  const uint16_t* A = g.A[l];
  const uint16_t* B = g.B[l] + (size_t)n0 * g.ld;
  const uint32_t k_begin = (uint32_t)z * g.kps, k_end = min(g.rows, k_begin + g.kps);
  // wave: m-tiles 4 (wave / 4) + 0..3, n-tiles 2 (wave % 4) + 0..1 (with one
  // m-tile, the output layer: m-tile 0, n-tile wave)
  const bool thin = M == MLP_OUTPAD;
  const int mt = thin ? 0 : 4 * (wave >> 2), nt = thin ? wave : 2 * (wave & 3);
  f32x4_t acc[4][2];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  float rowsum = 0.0f;
  const bool want_rowsum = n0 == 0 && (int)threadIdx.x < M;
  uint4 v[WG_VEC];
  if (k_begin < k_end) {
#pragma unroll
    for (int j = 0; j < WG_VEC; ++j) v[j] = wg_load(A, M, B, N, g.ld, j, k_begin, k_end);
  }
  for (uint32_t k0 = k_begin; k0 < k_end; k0 += WG_KC) {
    lds_barrier();  // the previous stage has been read
#pragma unroll
    for (int j = 0; j < WG_VEC; ++j) {
      const int i = (int)threadIdx.x + j * WG_THREADS;
      *(uint4*)&S[(i / (WG_KC / 8)) * WG_LS + (i % (WG_KC / 8)) * 8] = v[j];
    }
    lds_barrier();
    if (k0 + WG_KC < k_end) {
#pragma unroll
      for (int j = 0; j < WG_VEC; ++j) v[j] = wg_load(A, M, B, N, g.ld, j, k0 + WG_KC, k_end);
    }
    const int kc = (int)min((uint32_t)WG_KC, (k_end - k0 + 31u) / 32u * 32u);
    for (int ks = 0; ks < kc; ks += 32) {
      uint4 af[4], bf[2];
#pragma unroll
      for (int b = 0; b < 2; ++b)
        if (b == 0 || !thin) bf[b] = *(const uint4*)&S[(128 + 16 * (nt + b) + r16) * WG_LS + ks + 8 * q];
#pragma unroll
      for (int a = 0; a < 4; ++a)
        if (a == 0 || !thin) af[a] = *(const uint4*)&S[(16 * (mt + a) + r16) * WG_LS + ks + 8 * q];
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          if ((a == 0 && b == 0) || !thin)
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t*)&af[a], *(const bf16x8_t*)&bf[b],
                                                                acc[a][b], 0, 0, 0);
    }
    if (want_rowsum) {
      for (int k = 0; k < kc; k += 8) {
        const uint4 p = *(const uint4*)&S[(int)threadIdx.x * WG_LS + k];
        const uint32_t w[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          rowsum += u2f(w[t] << 16);
          rowsum += u2f(w[t] & 0xffff0000u);
        }
      }
    }
  }
  // lane holds C[16 (mt + a) + 4q + e][16 (nt + b) + r16]
  float* P = g.part[l] + (size_t)z * M * kin;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      if (thin && (a > 0 || b > 0)) continue;
      const int n = 16 * (nt + b) + r16;
      if (n >= N) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) P[(size_t)(16 * (mt + a) + 4 * q + e) * kin + n0 + n] = acc[a][b][e];
    }
  if (want_rowsum) g.bpart[l][(size_t)z * M + threadIdx.x] = rowsum;
}

// The gradients of every layer from the split partials: gw[l][i] = sum over
// slices z (in order) of part_l[z][i], gb[l][m] = sum over z of bpart_l[z][m].
struct GradSum {
  const float* part[MLP_LAYERS];
  const float* bpart[MLP_LAYERS];
  float* gw[MLP_LAYERS];
  float* gb[MLP_LAYERS];
  uint32_t nw[MLP_LAYERS], nb[MLP_LAYERS];
  uint32_t first[MLP_LAYERS + 1];  // first thread of layer l (weights then biases)
  int slices;
};

__global__ void k_grad_sum(GradSum S) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= S.first[MLP_LAYERS]) return;
  int l = 0;
  while (l + 1 < MLP_LAYERS && t >= S.first[l + 1]) ++l;
  const uint32_t i = t - S.first[l];
  if (i < S.nw[l]) {
    S.gw[l][i] = slice_sum(S.part[l] + i, S.nw[l], S.slices);
  } else {
    const uint32_t m = i - S.nw[l];
    S.gb[l][m] = slice_sum(S.bpart[l] + m, S.nb[l], S.slices);
  }
}

}  // namespace

size_t mlp_train_partial_floats(uint32_t rows) {
  const int slices = mlp_train_slices(rows);
  size_t n = 0;
  for (int l = 0; l < MLP_LAYERS; ++l) n += (mlp_w_count(l) + mlp_b_count(l)) * (size_t)slices;
  return n;
}

int mlp_train_slices(uint32_t rows) { return (int)std::max<uint32_t>(1u, std::min<uint32_t>(32u, (rows + 255u) / 256u)); }

uint32_t mlp_train_ld(uint32_t rows) { return (rows + 63u) / 64u * 64u; }

hipError_t mlp_train_grads(const MlpDev& w, const float* in, uint32_t rows, const float* target, MlpTrainBufs& tb,
                           MlpTrainT& tt, bool reduce, hipStream_t st, unsigned long long* esum, unsigned int* ecnt) {
  if (rows == 0) return hipSuccess;
  const uint32_t ld = tt.ld;
  if (ld < mlp_train_ld(rows)) return hipErrorInvalidValue;
  hipError_t e;
  {
    FwdBwdArgs f;
    memset(&f, 0, sizeof(f));
    f.rows = rows;
    f.ld = ld;
    f.in = in;
    f.target = target;
    for (int l = 0; l < MLP_LAYERS; ++l) {
      f.w[l] = w.wb[l];
      f.wbt[l] = w.wbt[l];
      f.b[l] = w.b[l];
    }
    f.XT = tt.XT;
    for (int l = 0; l < MLP_HIDDEN_LAYERS; ++l) {
      f.HT[l] = tt.HT[l];
      f.dT[l] = tt.dT[l];
    }
    f.dyT = tt.dyT;
    f.row_err = tb.row_err;
    f.esum = esum;
    f.ecnt = ecnt;
    hipLaunchKernelGGL(k_fwd_bwd, dim3((rows + 63) / 64), dim3(FB_THREADS), FB_LDS, st, f);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  const int slices = mlp_train_slices(rows);
  const int kps = (int)(((rows + (uint32_t)slices - 1u) / (uint32_t)slices + 31u) / 32u * 32u);
  GradSum S;
  memset(&S, 0, sizeof(S));
  S.slices = slices;
  WgradArgs wg;
  memset(&wg, 0, sizeof(wg));
  wg.rows = rows;
  wg.ld = ld;
  wg.kps = (uint32_t)kps;
  wg.slices = slices;
  float* part = tt.part;  // partials of layer 4 first, then 3, ..., 0
  for (int l = MLP_HIDDEN_LAYERS; l >= 0; --l) {
    const int nout = mlp_nout(l), kl = mlp_kin(l);
    wg.A[l] = l == MLP_HIDDEN_LAYERS ? tt.dyT : tt.dT[l];
    wg.B[l] = l == 0 ? tt.XT : tt.HT[l - 1];
    wg.part[l] = part;
    wg.bpart[l] = part + (size_t)slices * nout * kl;
    S.part[l] = wg.part[l];
    S.bpart[l] = wg.bpart[l];
    tt.part_w[l] = wg.part[l];
    tt.part_b[l] = wg.bpart[l];
    S.gw[l] = tb.gw[l];
    S.gb[l] = tb.gb[l];
    S.nw[l] = (uint32_t)(nout * kl);
    S.nb[l] = (uint32_t)nout;
    part += (size_t)slices * (nout * kl + nout);
  }
  hipLaunchKernelGGL(k_wgrad, dim3((unsigned)(slices * (MLP_LAYERS + 1))), dim3(WG_THREADS), 0, st, wg);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  tt.slices = slices;
  if (!reduce) return hipSuccess;
  uint32_t tot = 0;
  for (int l = 0; l < MLP_LAYERS; ++l) {
    S.first[l] = tot;
    tot += S.nw[l] + S.nb[l];
  }
  S.first[MLP_LAYERS] = tot;
  hipLaunchKernelGGL(k_grad_sum, dim3((tot + 255) / 256), dim3(256), 0, st, S);
  return hipGetLastError();
}

}  // namespace pm
