// shp_mlp.hip - the learned warm start: a 14-128-128-128-2 SiLU MLP that
// predicts the initial (normal, friction) impulses of contacts that were not
// in last frame's cache, where the reference starts at zero
// (shapes/src/Physics/Solvers/Contact.hs:91-99).  Weights are BF16 on the
// device, every product accumulates in FP32 on the matrix cores
// (v_mfma_f32_16x16x16_bf16), biases and activations are FP32 and are
// rounded to BF16 only where they feed the next product.
//
// Kernels:
//   k_mlp_eval      forward of feature rows, 16 at a time (4 waves)
//   k_mlp_infer     the same on a step's cache misses, features and output
//                   head included
//   k_mlp_rows      training: forward and backward of 16 rows at a time; the
//                   activations and their gradients in fragments
//   k_mlp_weights   training: the weight gradients from those, summed in a
//                   fixed order (deterministic), then Adam on the FP32
//                   master weights and their BF16 fragments
//
// The inference kernels keep the weights in registers: wave w computes output
// columns [32 w, 32 w + 32) of every layer, so it needs 2 x (1 + 8 + 8 + 8)
// fragments (shp_mlp.h), loaded once per workgroup, and a layer reads only
// activations from LDS.  They compute the transposed products W^T h^T: a lane
// then holds four consecutive columns of one row and stores them with one
// 8-byte LDS write, where the next layer's operand is one 8-byte read.  The
// sums over k are those of h W, in the same order.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <string>
#include <vector>

#include "../../include/shapes_gpu.h"
#include "shp_engine.h"
#include "shp_mlp.h"
#include "shp_records.h"

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f) {  // round to nearest even
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  uint32_t r = u + 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(r >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }
__device__ __forceinline__ float dsilu(float z) {
  float s = 1.0f / (1.0f + __expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Operand fragments of v_mfma_f32_16x16x16_bf16: lane l holds
//   A[row = l%16][k = 4*(l/16) + 0..3]   B[k = 4*(l/16) + 0..3][col = l%16]
// and receives D[row = 4*(l/16) + i][col = l%16], i = 0..3.
#define TILE 64  // rows of a training tile: weight gradients are summed over a tile, then over tiles
#define MLP_PARTS 64  // ... in this many sums, tile t in sum t % MLP_PARTS, which are added in order

// Master weight i (padded layout) into its BF16 fragments.
__device__ __forceinline__ void store_weight(int i, float x, uint16_t* wfr) {
  const uint16_t v = f2bf(x);
  int f = -1, g = -1, k = 0, o = 0, nkb = 1, gkb = 1;  // fragments of its layer, row, column
  if (i < MLP_OFF_B1) {
    f = MLP_F1;
    k = i >> 7;
    o = i & 127;
  } else if (i >= MLP_OFF_W2 && i < MLP_OFF_B2) {
    f = MLP_F2;
    g = MLP_G2;
    gkb = 8;
    k = (i - MLP_OFF_W2) >> 7;
    o = (i - MLP_OFF_W2) & 127;
    nkb = 8;
  } else if (i >= MLP_OFF_W3 && i < MLP_OFF_B3) {
    f = MLP_F3;
    g = MLP_G3;
    gkb = 8;
    k = (i - MLP_OFF_W3) >> 7;
    o = (i - MLP_OFF_W3) & 127;
    nkb = 8;
  } else if (i >= MLP_OFF_W4 && i < MLP_OFF_B4) {
    f = MLP_F4;
    g = MLP_G4;
    k = (i - MLP_OFF_W4) >> 4;
    o = (i - MLP_OFF_W4) & 15;
    nkb = 8;
  }
  if (f < 0) return;  // a bias
  const int lane = (o & 15) + 16 * ((k & 15) >> 2);
  wfr[f + ((o >> 4) * nkb + (k >> 4)) * MLP_FRAG + 4 * lane + (k & 3)] = v;
  if (g < 0) return;  // the first layer has no backward product
  const int glane = (k & 15) + 16 * ((o & 15) >> 2);
  wfr[g + ((k >> 4) * gkb + (o >> 4)) * MLP_FRAG + 4 * glane + (o & 3)] = v;
}

// What a training call does with gradient entry i (padded layout): writes it
// (grad), or takes an Adam step on the FP32 master weights (padding entries
// stay zero).
struct MlpStep {
  float* grad;  // null: Adam
  float *w, *mom, *vel;
  uint16_t* wfr;
  float lr, b1c, b2c;
};

__device__ __forceinline__ void apply_gradient(const MlpStep& s, int i, float g, bool real) {
  if (s.grad) {
    s.grad[i] = g;
    return;
  }
  if (!real) return;
  float m = 0.9f * s.mom[i] + 0.1f * g;
  float v = 0.999f * s.vel[i] + 0.001f * g * g;
  s.mom[i] = m;
  s.vel[i] = v;
  float x = s.w[i] - s.lr * (m / s.b1c) / (sqrtf(v / s.b2c) + 1e-8f);
  s.w[i] = x;
  store_weight(i, x, s.wfr);
}

// The BF16 copies of every master weight.
__global__ void k_mlp_pack(const float* w, uint16_t* wfr) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < MLP_NPARAM_PAD) store_weight(i, w[i], wfr);
}

// features (n x 14 FP32) -> padded BF16 rows (rows x 16), zero rows beyond n
__global__ void k_pack_features(const float* f, long n, long rows, uint16_t* X) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * 16) return;
  long r = i >> 4;
  int cc = (int)(i & 15);
  X[i] = (r < n && cc < MLP_IN) ? f2bf(f[r * MLP_IN + cc]) : (uint16_t)0;
}

// ---- inference ----------------------------------------------------------------

// Row strides in LDS (BF16 entries): a fragment read takes 8 bytes of each of
// 16 rows, which then start 8 bytes further round the banks each.
constexpr int HS = 132, XS = 20;

// Wave w's fragments of every layer.
struct WaveWeights {
  bf16x4 w1[2], w2[2][8], w3[2][8], w4[8];
};

__device__ __forceinline__ void load_weights(const uint16_t* wfr, WaveWeights& W) {
  const bf16x4* f = (const bf16x4*)wfr + (threadIdx.x & 63);
  const int c0 = 2 * (threadIdx.x >> 6);
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    W.w1[c] = f[(MLP_F1 / MLP_FRAG + c0 + c) * 64];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      W.w2[c][k] = f[(MLP_F2 / MLP_FRAG + (c0 + c) * 8 + k) * 64];
      W.w3[c][k] = f[(MLP_F3 / MLP_FRAG + (c0 + c) * 8 + k) * 64];
    }
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) W.w4[k] = f[(MLP_F4 / MLP_FRAG + k) * 64];
}

__device__ __forceinline__ bf16x4 act_frag(const uint16_t* h, int stride, int kb) {
  const int l = threadIdx.x & 63;
  return *(const bf16x4*)(h + (l & 15) * stride + 16 * kb + 4 * (l >> 4));
}

// silu(acc + bias) of this lane's four columns from `col`, to row `row`
__device__ __forceinline__ void put_acts(uint16_t* h, int row, int col, f32x4 acc, const float* bias) {
  const float4 b = *(const float4*)(bias + col);
  uint32_t lo = f2bf(silu(acc[0] + b.x)) | (uint32_t)f2bf(silu(acc[1] + b.y)) << 16;
  uint32_t hi = f2bf(silu(acc[2] + b.z)) | (uint32_t)f2bf(silu(acc[3] + b.w)) << 16;
  *(uint2*)(h + row * HS + col) = make_uint2(lo, hi);
}

// The layers of 16 rows (BF16 features x in LDS, stride XS) by 4 waves; ha
// and hb hold 16 rows of HS.  sb: b1, b2, b3, b4.  Calls out(row, y0, y1) from
// one lane per row.  Begins and ends with a barrier.
template <class Out>
__device__ __forceinline__ void mlp_layers(const WaveWeights& W, const float* sb, const uint16_t* x,
                                           uint16_t* ha, uint16_t* hb, Out out) {
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int c0 = 32 * wv + 4 * (l >> 4), r = l & 15;
  __syncthreads();
  {
    const bf16x4 v = act_frag(x, XS, 0);
#pragma unroll
    for (int c = 0; c < 2; ++c)
      put_acts(ha, r, c0 + 16 * c, mfma16(W.w1[c], v, f32x4{0.f, 0.f, 0.f, 0.f}), sb);
  }
  __syncthreads();
#pragma unroll
  for (int layer = 0; layer < 2; ++layer) {
    const uint16_t* in = layer ? hb : ha;
    f32x4 acc[2];
    acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const bf16x4 v = act_frag(in, HS, k);
#pragma unroll
      for (int c = 0; c < 2; ++c) acc[c] = mfma16(layer ? W.w3[c][k] : W.w2[c][k], v, acc[c]);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
      put_acts(layer ? ha : hb, r, c0 + 16 * c, acc[c], sb + 128 * (layer + 1));
    __syncthreads();
  }
  if (wv == 0) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 8; ++k) acc = mfma16(W.w4[k], act_frag(ha, HS, k), acc);
    if (l < 16) out(l, acc[0] + sb[384], acc[1] + sb[385]);
  }
  __syncthreads();
}

__device__ __forceinline__ void load_biases(const float* w, float* sb) {
  for (int i = threadIdx.x; i < 3 * 128 + 16; i += blockDim.x)
    sb[i] = i < 128   ? w[MLP_OFF_B1 + i]
            : i < 256 ? w[MLP_OFF_B2 + i - 128]
            : i < 384 ? w[MLP_OFF_B3 + i - 256]
                      : w[MLP_OFF_B4 + i - 384];
}

// out[2 r + k] = output k of row r (n x 14 FP32 features), tiles of 16 rows
// (tiles of 32 and 64 took as long or longer from 4 k to 65 k rows).  Bound by
// the chain of layers while every workgroup has one tile, by the
// activations' exponentials and divisions beyond.  One launch and 2 floats
// written a row (before: features packed, 16 floats a row, outputs taken):
// 4099 rows 27 -> 6.8 us, 65536 rows 26.6 us.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_mlp_eval(const uint16_t* __restrict__ wfr,
                                                  const float* __restrict__ w,
                                                  const float* __restrict__ feats, int n,
                                                  float* __restrict__ out) {
  __shared__ __align__(16) uint16_t x[16 * XS], ha[16 * HS], hb[16 * HS];
  __shared__ __align__(16) float sb[3 * 128 + 16];
  WaveWeights W;
  load_weights(wfr, W);
  load_biases(w, sb);
  for (int t = blockIdx.x; t * 16 < n; t += gridDim.x) {
    const int row0 = t * 16, r = threadIdx.x >> 4, q = threadIdx.x & 15;
    const float f = row0 + r < n && q < MLP_IN ? feats[(size_t)(row0 + r) * MLP_IN + q] : 0.0f;
    x[r * XS + q] = f2bf(f);
    mlp_layers(W, sb, x, ha, hb, [&](int i, float y0, float y1) {
      if (row0 + i >= n) return;
      out[2 * (size_t)(row0 + i)] = y0;
      out[2 * (size_t)(row0 + i) + 1] = y1;
    });
  }
}

// ---- training -----------------------------------------------------------------

// Where a training call's rows come from: row r is row idx[r] of the BF16 set
// dX / dT, or (idx null) row r of FP32 features and targets.
struct TrainRows {
  const uint16_t* dX;
  const float* dT;
  const int32_t* idx;
  const float* feats;
  const float* targets;
};

__device__ __forceinline__ bf16x4 wfrag(const uint16_t* wfr, int f) {
  return ((const bf16x4*)wfr)[f / MLP_FRAG * 64 + (threadIdx.x & 63)];
}

// What the backward pass leaves for the weight gradients, per 16 rows: the
// rows' features, h1, h2, h3, the gradients of the three pre-activations and
// of the outputs as fragments (lane l: column 16 ct + l % 16, rows 4 (l / 16) +
// 0..3), 1.6 KB a row, and the columns' FP32 gradient sums over each lane's
// four rows.
#define MLP_RX 0
#define MLP_RH (MLP_RX + MLP_FRAG)          // 3 x 8
#define MLP_RD (MLP_RH + 24 * MLP_FRAG)     // 3 x 8
#define MLP_RY (MLP_RD + 24 * MLP_FRAG)
#define MLP_RSUB (MLP_RY + MLP_FRAG)        // entries per 16 rows
#define MLP_BSUB 400                        // of 4 rows: b1, b2, b3, b4

// A barrier for LDS alone: global loads and stores stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Forward and backward of the mean loss over n rows: squared error (huber =
// 0), dY = 2 (Y - T) / n, or twice the Huber loss with threshold `huber`, dY =
// 2 clamp(Y - T, +-huber) / n (the same gradient where |Y - T| <= huber), for
// the rows of whole tiles (those beyond n with dY = 0).  frags and bsum: see
// above; y and t (rows x 2, may be null) receive outputs and targets.
//
// 4 waves take 16 rows: wave w owns columns [32 w, 32 w + 32) of every layer,
// whose pre-activations stay in its registers from the forward to the
// backward pass; the rows move between layers through LDS.  A lane holds four
// rows of one column, which is a fragment of the weight gradients' products
// as it is.  A batch of 4096 rows is one workgroup to a CU, bound by the chain
// of 7 layers: 16.4 us; separate forward and backward kernels on 64-row
// tiles, which stored the FP32 pre-activations, took 94, one kernel on such
// tiles with the weight gradients in it 35 (64 CUs, bound by the
// activations' exponentials and divisions).
__global__ __launch_bounds__(256) void k_mlp_rows(const uint16_t* __restrict__ wfr,
                                                  const float* __restrict__ w, TrainRows rows, int n,
                                                  uint16_t* __restrict__ frags,
                                                  float* __restrict__ bsum, float huber, float* y,
                                                  float* t) {
  __shared__ __align__(16) uint16_t x[16 * XS], dy[16 * XS], hbuf[2][16 * HS];
  __shared__ __align__(16) float sb[3 * 128 + 16];
  __shared__ f32x4 z[3 * 2][256];  // each lane's own pre-activations
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, c = l & 15, r4 = 4 * (l >> 4);
  load_biases(w, sb);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  const float inv_n = 2.0f / (float)n;
  const int subs = (n + TILE - 1) / TILE * (TILE / 16);
  bf16x4 a[2][8];  // a layer's fragments, fetched a layer ahead
  auto fetch = [&](int f) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int k = 0; k < 8; ++k) a[q][k] = wfrag(wfr, f + (8 * (2 * wv + q) + k) * MLP_FRAG);
  };
  auto product = [&](const uint16_t* in, f32x4* acc) {
    acc[0] = acc[1] = zero;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const bf16x4 v = act_frag(in, HS, k);
#pragma unroll
      for (int q = 0; q < 2; ++q) acc[q] = mfma16(v, a[q][k], acc[q]);
    }
  };
  // this lane's four rows of column 32 wv + 16 q + c: to LDS and to fragment f
  auto put = [&](uint16_t* rowbuf, uint16_t* f, int q, const uint16_t* h) {
#pragma unroll
    for (int i = 0; i < 4; ++i) rowbuf[(r4 + i) * HS + 32 * wv + 16 * q + c] = h[i];
    *(uint2*)(f + (2 * wv + q) * MLP_FRAG + 4 * l) =
        make_uint2(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16);
  };
#pragma unroll 1
  for (int sub = blockIdx.x; sub < subs; sub += gridDim.x) {
    const int row0 = 16 * sub;
    uint16_t* out = frags + (size_t)sub * MLP_RSUB;
    float* bout = bsum + (size_t)(4 * sub + (l >> 4)) * MLP_BSUB;
    // the targets of the lanes that hold outputs (columns 0 and 1 in wave 0)
    const bool has_out = wv == 0 && c < 2;
    float target[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = row0 + r4 + i;
      target[i] = 0.f;
      if (has_out && row < n)
        target[i] = rows.idx ? rows.dT[2L * rows.idx[row] + c] : rows.targets[2L * row + c];
    }
    {
      const int r = threadIdx.x >> 4, q = threadIdx.x & 15, row = row0 + r;
      uint16_t v = 0;
      if (row < n) {
        if (rows.idx)
          v = rows.dX[(long)rows.idx[row] * 16 + q];
        else if (q < MLP_IN)
          v = f2bf(rows.feats[(size_t)row * MLP_IN + q]);
      }
      x[r * XS + q] = v;
    }
    bf16x4 a1[2], a4[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      a1[q] = wfrag(wfr, MLP_F1 + (2 * wv + q) * MLP_FRAG);
      a4[q] = wfrag(wfr, MLP_G4 + (2 * wv + q) * MLP_FRAG);
    }
    fetch(MLP_F2);
    lds_barrier();
    if (wv == 0) {
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (short)x[(r4 + i) * XS + c];
      *(bf16x4*)(out + MLP_RX + 4 * l) = v;
    }
    f32x4 acc[2];
#pragma unroll 1
    for (int L = 0; L < 3; ++L) {
      if (L == 0) {
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[q] = mfma16(act_frag(x, XS, 0), a1[q], zero);
      } else {
        product(hbuf[(L - 1) & 1], acc);
        fetch(L == 1 ? MLP_F3 : MLP_G3);
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float b = sb[128 * L + 32 * wv + 16 * q + c];
        uint16_t h[4];
        f32x4 zz;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          zz[i] = acc[q][i] + b;
          h[i] = f2bf(silu(zz[i]));
        }
        z[2 * L + q][threadIdx.x] = zz;
        put(hbuf[L & 1], out + MLP_RH + L * 8 * MLP_FRAG, q, h);
      }
      lds_barrier();
    }
    if (wv == 0) {  // outputs and their gradient
      f32x4 o = zero;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        o = mfma16(act_frag(hbuf[0], HS, k), wfrag(wfr, MLP_F4 + k * MLP_FRAG), o);
      const float b = sb[384 + c];
      float sum = 0.f;
      uint16_t h[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + r4 + i;
        float d = 0.f;
        if (has_out && row < n) {
          const float yy = o[i] + b;
          float e = yy - target[i];
          if (y) y[2L * row + c] = yy;
          if (t) t[2L * row + c] = target[i];
          if (huber > 0.f) e = fminf(fmaxf(e, -huber), huber);
          d = e * inv_n;
        }
        h[i] = f2bf(d);
        sum += d;
        dy[(r4 + i) * XS + c] = h[i];
      }
      *(uint2*)(out + MLP_RY + 4 * l) =
          make_uint2(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16);
      bout[384 + c] = sum;
    }
    lds_barrier();
#pragma unroll 1
    for (int L = 2; L >= 0; --L) {
      if (L == 2) {
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[q] = mfma16(act_frag(dy, XS, 0), a4[q], zero);
      } else {
        product(hbuf[L & 1], acc);
        if (L == 1) fetch(MLP_G2);
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const f32x4 zz = z[2 * L + q][threadIdx.x];
        uint16_t h[4];
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float d = acc[q][i] * dsilu(zz[i]);
          h[i] = f2bf(d);
          sum += d;
        }
        put(hbuf[(L + 1) & 1], out + MLP_RD + L * 8 * MLP_FRAG, q, h);
        bout[128 * L + 32 * wv + 16 * q + c] = sum;
      }
      lds_barrier();
    }
  }
}

// Weight gradients and what follows from them (apply_gradient).  Workgroups
// [0, 144): one 16x16 block of a weight matrix each: the products of every
// tile are summed in MFMA accumulators, tile t into sum t % MLP_PARTS (each
// wave has an eighth of the sums), and the sums are added in order; the rest:
// 64 bias entries each, likewise.  What the row kernel wrote is read from L2
// (12 MB a 4096-row batch over the blocks): 10.6 us, Adam included (one partial of
// 149 KB a tile, then summing those, took 20).
constexpr int W_BLOCKS = 8 + 64 + 64 + 8, B_BLOCKS = (386 + 63) / 64;

__global__ __launch_bounds__(512) void k_mlp_weights(const uint16_t* __restrict__ frags,
                                                     const float* __restrict__ bsum, int tiles,
                                                     MlpStep step) {
  __shared__ float s_sum[MLP_PARTS][256];
  constexpr int PER = MLP_PARTS / 8, SUBS = TILE / 16;
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, blk = blockIdx.x;
  const int parts = tiles < MLP_PARTS ? tiles : MLP_PARTS;
  if (blk < W_BLOCKS) {
    // matrix W(L + 1), block (it, jt): fragments of its inputs and of the
    // gradients of its outputs
    int in, dz, off, ld, it, jt;
    if (blk < 8) {
      it = 0;
      jt = blk;
      in = MLP_RX;
      dz = MLP_RD + jt * MLP_FRAG;
      off = MLP_OFF_W1;
      ld = 128;
    } else if (blk < 136) {
      const int L = (blk - 8) >> 6;
      it = ((blk - 8) >> 3) & 7;
      jt = blk & 7;
      in = MLP_RH + (8 * L + it) * MLP_FRAG;
      dz = MLP_RD + (8 * (L + 1) + jt) * MLP_FRAG;
      off = L ? MLP_OFF_W3 : MLP_OFF_W2;
      ld = 128;
    } else {
      it = blk - 136;
      jt = 0;
      in = MLP_RH + (16 + it) * MLP_FRAG;
      dz = MLP_RY;
      off = MLP_OFF_W4;
      ld = 16;
    }
    f32x4 acc[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) acc[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int t0 = wv * PER; t0 < tiles; t0 += MLP_PARTS) {
      bf16x4 u[PER][SUBS], v[PER][SUBS];  // in flight together
#pragma unroll
      for (int q = 0; q < PER; ++q) {
        const int tile = t0 + q < tiles ? t0 + q : t0;
        const uint16_t* f = frags + (size_t)tile * SUBS * MLP_RSUB + 4 * l;
#pragma unroll
        for (int k = 0; k < SUBS; ++k) {
          u[q][k] = *(const bf16x4*)(f + k * MLP_RSUB + in);
          v[q][k] = *(const bf16x4*)(f + k * MLP_RSUB + dz);
        }
      }
#pragma unroll
      for (int q = 0; q < PER; ++q)
        if (t0 + q < tiles)
#pragma unroll
          for (int k = 0; k < SUBS; ++k) acc[q] = mfma16(u[q][k], v[q][k], acc[q]);
    }
#pragma unroll
    for (int q = 0; q < PER; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) s_sum[wv * PER + q][(4 * (l >> 4) + i) * 16 + (l & 15)] = acc[q][i];
    __syncthreads();
    if (threadIdx.x >= 256) return;
    const int r = threadIdx.x >> 4, c = threadIdx.x & 15;
    float g = 0.f;
#pragma unroll 16
    for (int p = 0; p < parts; ++p) g += s_sum[p][threadIdx.x];
    const bool real = off == MLP_OFF_W1 ? r < MLP_IN : off == MLP_OFF_W4 ? c < 2 : true;
    apply_gradient(step, off + (16 * it + r) * ld + 16 * jt + c, g, real);
    return;
  }
  const int e = 64 * (blk - W_BLOCKS) + l;  // bias entry
  for (int q = 0; q < PER; ++q) {
    float sum = 0.f;
    for (int tile = wv * PER + q; tile < tiles; tile += MLP_PARTS) {
      const float* b = bsum + (size_t)tile * TILE / 4 * MLP_BSUB + (e < 386 ? e : 0);
      float part[TILE / 4];
#pragma unroll
      for (int k = 0; k < TILE / 4; ++k) part[k] = b[k * MLP_BSUB];
#pragma unroll
      for (int k = 0; k < TILE / 4; ++k) sum += part[k];
    }
    s_sum[wv * PER + q][l] = sum;
  }
  __syncthreads();
  if (wv != 0) return;
  float g = 0.f;
  for (int p = 0; p < parts; ++p) g += s_sum[p][l];
  const int i = e < 128   ? MLP_OFF_B1 + e
                : e < 256 ? MLP_OFF_B2 + e - 128
                : e < 384 ? MLP_OFF_B3 + e - 256
                          : MLP_OFF_B4 + e - 384;
  if (e < 386) apply_gradient(step, i, g, true);
}

// outputs of a call on overlapping buffers, to where they belong
__global__ void k_mlp_place(const float2* y, int n, float* out) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  out[2 * (size_t)r] = y[r].x;
  out[2 * (size_t)r + 1] = y[r].y;
}

// 4 workgroups on each of 256 CUs
void launch_eval(const MlpParams& p, const float* feats, int n, float* out, hipStream_t s) {
  const int tiles = (n + 15) / 16;
  k_mlp_eval<<<tiles < 1024 ? tiles : 1024, 256, 0, s>>>(p.wfr, p.w, feats, n, out);
}

}  // namespace

// ------------------------------------------------------------------ host

// The published blob and the padded layout: W1 has 14 of 16 rows, W4 2 of 16
// columns, b4 2 of 16 entries; b1 to b3 are the same range of both.
constexpr int BLOB_B1 = MLP_IN * 128, BLOB_W4 = BLOB_B1 + (MLP_OFF_W4 - MLP_OFF_B1);

template <class T>
static void mlp_pad(const T* blob, T* pad) {
  memcpy(pad + MLP_OFF_W1, blob, BLOB_B1 * sizeof(T));
  memcpy(pad + MLP_OFF_B1, blob + BLOB_B1, (BLOB_W4 - BLOB_B1) * sizeof(T));
  for (int k = 0; k < 128; ++k)
    for (int q = 0; q < 2; ++q) pad[MLP_OFF_W4 + 16 * k + q] = blob[BLOB_W4 + 2 * k + q];
  for (int q = 0; q < 2; ++q) pad[MLP_OFF_B4 + q] = blob[BLOB_W4 + 256 + q];
}

static void mlp_unpad(const float* pad, float* blob) {
  memcpy(blob, pad + MLP_OFF_W1, BLOB_B1 * sizeof(float));
  memcpy(blob + BLOB_B1, pad + MLP_OFF_B1, (BLOB_W4 - BLOB_B1) * sizeof(float));
  for (int k = 0; k < 128; ++k)
    for (int q = 0; q < 2; ++q) blob[BLOB_W4 + 2 * k + q] = pad[MLP_OFF_W4 + 16 * k + q];
  for (int q = 0; q < 2; ++q) blob[BLOB_W4 + 256 + q] = pad[MLP_OFF_B4 + q];
}

shp_status mlp_params_alloc(MlpParams* p) {
  if (hipMalloc(&p->w, MLP_NPARAM_PAD * sizeof(float)) != hipSuccess) return SHP_E_OOM;
  if (hipMalloc(&p->wfr, MLP_NFRAG * sizeof(uint16_t)) != hipSuccess) return SHP_E_OOM;
  return SHP_OK;
}

void mlp_params_free(MlpParams* p) {
  if (p->w) (void)hipFree(p->w);
  if (p->wfr) (void)hipFree(p->wfr);
  p->w = nullptr;
  p->wfr = nullptr;
}

shp_status mlp_params_upload(MlpParams* p, const float* params, hipStream_t s) {
  std::vector<float> pad(MLP_NPARAM_PAD, 0.0f);
  mlp_pad(params, pad.data());
  if (hipMemcpyAsync(p->w, pad.data(), pad.size() * 4, hipMemcpyHostToDevice, s) != hipSuccess) return SHP_E_HIP;
  k_mlp_pack<<<(MLP_NPARAM_PAD + 255) / 256, 256, 0, s>>>(p->w, p->wfr);
  if (hipStreamSynchronize(s) != hipSuccess) return SHP_E_HIP;
  return SHP_OK;
}

// ---- engine hooks ------------------------------------------------------------

// Learned warm start of the step's cache misses: the features rounded to
// BF16, the forward pass on the matrix cores, then the output head lambda_n =
// max(y0, 0) / mn, lambda_t = y1 / mt projected onto |lambda_t| <= mu *
// lambda_n.  The contact is marked warm (2) so the solver applies the
// predicted impulses like a cached solution (the coloured solver's manifold
// record, already written, gets them too); a non-finite prediction keeps the
// zero start.  A miss's contact and bodies lie on about 27 cache lines of
// their own, whose gathers bound the kernel, so a workgroup gathers for 64
// misses at once (256 piles, 43 k misses: 75 us; with 32 misses a
// workgroup of 8 waves 95 us; with the weights in LDS, which left one
// workgroup to a CU, 160 us).
constexpr int INFER_ROWS = MLP_INFER_ROWS, INFER_THREADS = MLP_INFER_THREADS;

__global__ __launch_bounds__(INFER_THREADS) __attribute__((amdgpu_waves_per_eu(3))) void k_mlp_infer(Ctx c) {
  __shared__ __align__(16) uint16_t sx[INFER_ROWS * XS], ha[16 * HS], hb[16 * HS];
  __shared__ __align__(16) float sb[3 * 128 + 16];
  __shared__ float2 sy[INFER_ROWS];
  int n = c.counters[CNT_MISS];
  if (n > c.miss_cap) n = c.miss_cap;
  if ((int)blockIdx.x * INFER_ROWS >= n) return;  // nothing to do (no barrier follows)
  WaveWeights W;
  load_weights(c.mlp_wfr, W);
  load_biases(c.mlp_w, sb);
  static_assert(INFER_ROWS == 64 && INFER_THREADS == 256, "a row per lane of the first wavefront");
  const int r = threadIdx.x;
  const bool row_lane = r < INFER_ROWS;
  for (int t = blockIdx.x; t * INFER_ROWS < n; t += gridDim.x) {
    const int row0 = t * INFER_ROWS;
    // the output head's inputs of this lane's row, loaded with the features so
    // that the head waits on no load after the layers
    const bool row_ok = row_lane && row0 + r < n;
    int hk = 0, hmr = -1;
    double hmcn = 1.0, hmct = 1.0, hmu = 0.0;
    if (row_ok) {
      hk = c.miss_idx[row0 + r];
      hmr = c.solver == SHP_SOLVER_COLORED_F32 ? c.miss_rec[row0 + r] : -1;
      hmcn = c.mcn[hk];
      hmct = c.mct[hk];
      hmu = (c.mu[c.ga[hk]] + c.mu[c.gb[hk]]) / 2.0;
    }
    if (c.features_in_contacts) {
      for (int i = threadIdx.x; i < INFER_ROWS * 16; i += INFER_THREADS) {
        const int i_r = i >> 4, q = i & 15;
        float f = (row0 + i_r < n && q < MLP_IN) ? c.miss_feat[(size_t)(row0 + i_r) * MLP_IN + q] : 0.0f;
        sx[i_r * XS + q] = f2bf(f);
      }
    } else if (row_lane) {
      // the features of the stored contact, as the contact kernel would
      // compute them (the velocities are those it saw: nothing has changed
      // them since)
      float f[MLP_IN];
      for (int q = 0; q < MLP_IN; ++q) f[q] = 0.0f;
      if (row_ok) {
        const int k = hk;
        const int ga = c.ga[k], gb = c.gb[k];
        const double v[6] = {c.vx[ga], c.vy[ga], c.w[ga], c.vx[gb], c.vy[gb], c.w[gb]};
        const double sgn = c.flip[k] ? -1.0 : 1.0;
        mlp_features(sgn * c.cnx[k], sgn * c.cny[k], c.depth[k], v, c.rax[k], c.ray[k], c.rbx[k],
                     c.rby[k], c.iml[ga], c.iml[gb], c.imr[ga], c.imr[gb],
                     (c.mu[ga] + c.mu[gb]) / 2.0, f);
      }
      for (int q = 0; q < 16; ++q) sx[r * XS + q] = f2bf(q < MLP_IN ? f[q] : 0.0f);
    }
    for (int o = 0; o < INFER_ROWS; o += 16)
      mlp_layers(W, sb, sx + o * XS, ha, hb,
                 [&](int i, float y0, float y1) { sy[o + i] = make_float2(y0, y1); });
    bool set = false;
    if (row_ok) {
      const int k = hk;
      double ln = (double)sy[r].x;
      ln = ln > 0.0 ? ln / hmcn : 0.0;
      double lt = (double)sy[r].y / hmct;
      const double thr = ln * hmu;
      lt = lt > thr ? thr : (lt < -thr ? -thr : lt);
      if (ln - ln == 0.0 && lt - lt == 0.0) {
        c.ln[k] = ln;
        c.lt[k] = lt;
        c.warm[k] = 2;
        set = true;
        if (hmr >= 0) shp::patch_record_warm(shp::packf(c), hmr >> 1, hmr & 1, ln, lt);
      }
    }
    const unsigned long long setm = __ballot(set);  // one atomic per tile
    if (threadIdx.x == 0 && setm) atomicAdd(&c.counters[CNT_LEARNED], (int)__popcll(setm));
    // (the next rows' features and outputs are written behind barriers)
  }
}

// After the solve: append (features, lambda_n * mn, lambda_t * mt) of the
// step's cache misses to the training log.
__global__ void k_mlp_log(Ctx c) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  int n = c.counters[CNT_MISS];
  if (n > c.miss_cap) n = c.miss_cap;
  if (s >= n) return;
  unsigned long long pos = atomicAdd(c.log_count, 1ull);
  if ((long)pos >= c.log_cap) return;
  int k = c.miss_idx[s];
  for (int q = 0; q < MLP_IN; ++q) c.log_feat[pos * MLP_IN + q] = c.miss_feat[(size_t)s * MLP_IN + q];
  c.log_tgt[pos * 2] = (float)(c.ln[k] * c.mcn[k]);
  c.log_tgt[pos * 2 + 1] = (float)(c.lt[k] * c.mct[k]);
}

void mlp_launch_infer(shp_batch* b) {
  k_mlp_infer<<<b->plan.g_infer, INFER_THREADS, 0, b->stream>>>(b->ctx);
}

// sx, ha, hb (BF16), sb and sy (FP32) of k_mlp_infer
size_t mlp_infer_static_lds() {
  return lds16(INFER_ROWS * XS * 2) + 2 * lds16(16 * HS * 2) + lds16((3 * 128 + 16) * 4) +
         lds16(INFER_ROWS * 8);
}

void mlp_launch_log(shp_batch* b) {
  k_mlp_log<<<b->plan.g_log, 256, 0, b->stream>>>(b->ctx);
}

// ---- training handle -------------------------------------------------------

// rows of one shp_mlp_forward_noalloc call
#define MLP_NOALLOC_MAX_ROWS 65536

struct shp_mlp {
  int device = 0;  // the GPU the handle's weights live on
  hipStream_t stream = nullptr;
  MlpParams p{};
  float *mom = nullptr, *vel = nullptr, *grad = nullptr;
  float2* staged = nullptr;  // MLP_NOALLOC_MAX_ROWS outputs
  // of cap_tiles training tiles: fragments and bias sums (k_mlp_rows)
  int cap_tiles = 0;
  uint16_t* frags = nullptr;
  float* bsum = nullptr;
  int cap_fwd = 0;
  float* Fin = nullptr;    // cap_fwd x 14 staging
  float* out = nullptr;    // cap_fwd x 2 outputs
  float* T = nullptr;      // cap_fwd x 2 targets
  int32_t* didx = nullptr;  // cap_idx row indices of a training call
  long cap_idx = 0;
  long adam_t = 0;
  // training set on device
  uint16_t* dX = nullptr;
  float* dT = nullptr;
  long n_data = 0;
  float huber = 0.f;  // 0: squared error
};

static shp_status mlp_fail(shp_status s, const char* m) {
  shp_set_error(m);
  return s;
}

#define MCHK(x) \
  do { if ((x) != hipSuccess) return mlp_fail(SHP_E_HIP, #x); } while (0)

// feature rows, outputs and targets of calls on host memory
static shp_status mlp_reserve(shp_mlp* h, int rows) {
  if (rows <= h->cap_fwd) return SHP_OK;
  for (void* q : {(void*)h->Fin, (void*)h->out, (void*)h->T})
    if (q) (void)hipFree(q);
  h->Fin = h->out = h->T = nullptr;
  h->cap_fwd = 0;
  rows = ((rows + 63) / 64) * 64;
  MCHK(hipMalloc(&h->Fin, (size_t)rows * MLP_IN * 4));
  MCHK(hipMalloc(&h->out, (size_t)rows * 2 * 4));
  MCHK(hipMalloc(&h->T, (size_t)rows * 2 * 4));
  h->cap_fwd = rows;
  return SHP_OK;
}

static shp_status mlp_reserve_tiles(shp_mlp* h, int n) {
  const int tiles = (n + TILE - 1) / TILE;
  if (tiles <= h->cap_tiles) return SHP_OK;
  for (void* q : {(void*)h->frags, (void*)h->bsum})
    if (q) (void)hipFree(q);
  h->frags = nullptr;
  h->bsum = nullptr;
  h->cap_tiles = 0;
  const size_t subs = (size_t)tiles * (TILE / 16);
  MCHK(hipMalloc(&h->frags, subs * MLP_RSUB * sizeof(uint16_t)));
  MCHK(hipMalloc(&h->bsum, 4 * subs * MLP_BSUB * sizeof(float)));
  h->cap_tiles = tiles;
  return SHP_OK;
}

// The gradient over n rows (at most the reserved tiles), then `step`.
static void launch_train(shp_mlp* h, const TrainRows& rows, int n, float* y, float* t,
                         const MlpStep& step) {
  const int tiles = (n + TILE - 1) / TILE, subs = tiles * (TILE / 16);
  k_mlp_rows<<<subs < 1024 ? subs : 1024, 256, 0, h->stream>>>(h->p.wfr, h->p.w, rows, n, h->frags,
                                                              h->bsum, h->huber, y, t);
  k_mlp_weights<<<W_BLOCKS + B_BLOCKS, 512, 0, h->stream>>>(h->frags, h->bsum, tiles, step);
}

extern "C" {

int32_t shp_mlp_param_count(void) { return MLP_NPARAM; }

shp_status shp_mlp_create(const float* params, shp_mlp** out) {
  if (!params || !out) return mlp_fail(SHP_E_INVAL, "null argument");
  shp_mlp* h = new shp_mlp();
  if (hipGetDevice(&h->device) != hipSuccess) {
    delete h;
    return mlp_fail(SHP_E_HIP, "no HIP device");
  }
  if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess) {
    delete h;
    return mlp_fail(SHP_E_HIP, "stream");
  }
  shp_status st = mlp_params_alloc(&h->p);
  if (st == SHP_OK) st = mlp_params_upload(&h->p, params, h->stream);
  if (st == SHP_OK) {
    if (hipMalloc(&h->mom, MLP_NPARAM_PAD * 4) != hipSuccess || hipMalloc(&h->vel, MLP_NPARAM_PAD * 4) != hipSuccess ||
        hipMalloc(&h->grad, MLP_NPARAM_PAD * 4) != hipSuccess ||
        hipMalloc(&h->staged, MLP_NOALLOC_MAX_ROWS * sizeof(float2)) != hipSuccess)
      st = SHP_E_OOM;
  }
  if (st == SHP_OK) {
    std::vector<float> zero(MLP_NPARAM_PAD, 0.f);
    if (hipMemcpy(h->mom, zero.data(), MLP_NPARAM_PAD * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(h->grad, zero.data(), MLP_NPARAM_PAD * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(h->vel, zero.data(), MLP_NPARAM_PAD * 4, hipMemcpyHostToDevice) != hipSuccess)
      st = SHP_E_HIP;
  }
  if (st != SHP_OK) {
    shp_mlp_destroy(h);
    return mlp_fail(st, "mlp allocation failed");
  }
  *out = h;
  return SHP_OK;
}

shp_status shp_mlp_destroy(shp_mlp* h) {
  if (!h) return SHP_OK;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  mlp_params_free(&h->p);
  void* ptrs[] = {h->mom, h->vel, h->grad, h->staged, h->frags, h->bsum, h->T, h->Fin,
                  h->out, h->didx, h->dX, h->dT};
  for (void* q : ptrs)
    if (q) (void)hipFree(q);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
  return SHP_OK;
}

shp_status shp_mlp_get_params(shp_mlp* h, float* params) {
  if (!h || !params) return mlp_fail(SHP_E_INVAL, "null argument");
  std::vector<float> pad(MLP_NPARAM_PAD);
  MCHK(hipStreamSynchronize(h->stream));
  MCHK(hipMemcpy(pad.data(), h->p.w, MLP_NPARAM_PAD * 4, hipMemcpyDeviceToHost));
  mlp_unpad(pad.data(), params);
  return SHP_OK;
}

shp_status shp_mlp_forward(shp_mlp* h, const float* feats, int32_t n, float* out) {
  if (!h || n < 0 || (n > 0 && (!feats || !out))) return mlp_fail(SHP_E_INVAL, "bad argument");
  if (n == 0) return SHP_OK;
  shp_status st = mlp_reserve(h, n);
  if (st != SHP_OK) return st;
  MCHK(hipMemcpyAsync(h->Fin, feats, (size_t)n * MLP_IN * 4, hipMemcpyHostToDevice, h->stream));
  launch_eval(h->p, h->Fin, n, h->out, h->stream);
  MCHK(hipGetLastError());
  MCHK(hipMemcpyAsync(out, h->out, (size_t)n * 2 * 4, hipMemcpyDeviceToHost, h->stream));
  MCHK(hipStreamSynchronize(h->stream));
  return SHP_OK;
}

shp_status shp_mlp_forward_noalloc(shp_mlp* h, const float* d_feats, int32_t n, float* d_out,
                                   void* stream) {
  if (!h || n < 0 || (n > 0 && (!d_feats || !d_out))) return mlp_fail(SHP_E_INVAL, "bad argument");
  if (n > MLP_NOALLOC_MAX_ROWS)
    return mlp_fail(SHP_E_INVAL, "n exceeds 65536 rows");
  if (n == 0) return SHP_OK;
  int dev = -1;
  MCHK(hipGetDevice(&dev));
  if (dev != h->device) return mlp_fail(SHP_E_INVAL, "the current device is not the handle's");
  const hipStream_t s = stream ? (hipStream_t)stream : h->stream;
  // a workgroup's outputs must not reach rows that another one has yet to read
  const uintptr_t in = (uintptr_t)d_feats, out = (uintptr_t)d_out;
  const bool overlap = in < out + (size_t)n * 2 * 4 && out < in + (size_t)n * MLP_IN * 4;
  launch_eval(h->p, d_feats, n, overlap ? (float*)h->staged : d_out, s);
  if (overlap) k_mlp_place<<<(n + 255) / 256, 256, 0, s>>>(h->staged, n, d_out);
  MCHK(hipGetLastError());
  return SHP_OK;
}

shp_status shp_mlp_gradient(shp_mlp* h, const float* feats, const float* targets, int32_t n,
                            float* grad_out, float* loss_out) {
  if (!h || n <= 0 || !feats || !targets || !grad_out) return mlp_fail(SHP_E_INVAL, "bad argument");
  shp_status st = mlp_reserve(h, n);
  if (st == SHP_OK) st = mlp_reserve_tiles(h, n);
  if (st != SHP_OK) return st;
  MCHK(hipMemcpyAsync(h->Fin, feats, (size_t)n * MLP_IN * 4, hipMemcpyHostToDevice, h->stream));
  MCHK(hipMemcpyAsync(h->T, targets, (size_t)n * 2 * 4, hipMemcpyHostToDevice, h->stream));
  MlpStep step{};
  step.grad = h->grad;
  launch_train(h, TrainRows{nullptr, nullptr, nullptr, h->Fin, h->T}, n, h->out, nullptr, step);
  MCHK(hipGetLastError());
  std::vector<float> g(MLP_NPARAM_PAD), y((size_t)n * 2);
  MCHK(hipMemcpyAsync(g.data(), h->grad, g.size() * 4, hipMemcpyDeviceToHost, h->stream));
  if (loss_out) MCHK(hipMemcpyAsync(y.data(), h->out, y.size() * 4, hipMemcpyDeviceToHost, h->stream));
  MCHK(hipStreamSynchronize(h->stream));
  mlp_unpad(g.data(), grad_out);
  if (loss_out) {
    double l = 0.0;
    for (size_t i = 0; i < y.size(); ++i) {
      const double d = (double)y[i] - targets[i];
      l += d * d;
    }
    *loss_out = (float)(l / n);
  }
  return SHP_OK;
}

shp_status shp_mlp_set_loss(shp_mlp* h, float huber_delta) {
  if (!h || !(huber_delta >= 0.f))
    return mlp_fail(SHP_E_INVAL, "huber_delta must be >= 0");
  h->huber = huber_delta;
  return SHP_OK;
}

shp_status shp_mlp_set_data(shp_mlp* h, const float* feats, const float* targets, int64_t n) {
  if (!h || n <= 0 || !feats || !targets) return mlp_fail(SHP_E_INVAL, "bad argument");
  if (h->dX) (void)hipFree(h->dX);
  if (h->dT) (void)hipFree(h->dT);
  h->dX = nullptr;
  h->dT = nullptr;
  MCHK(hipMalloc(&h->dX, (size_t)n * 16 * 2));
  MCHK(hipMalloc(&h->dT, (size_t)n * 2 * 4));
  float* stage = nullptr;
  const long chunk = 1 << 20;
  MCHK(hipMalloc(&stage, (size_t)chunk * MLP_IN * 4));
  for (long o = 0; o < n; o += chunk) {
    long m = n - o < chunk ? n - o : chunk;
    MCHK(hipMemcpy(stage, feats + o * MLP_IN, (size_t)m * MLP_IN * 4, hipMemcpyHostToDevice));
    k_pack_features<<<(int)((m * 16 + 255) / 256), 256, 0, h->stream>>>(stage, m, m, h->dX + o * 16);
    MCHK(hipStreamSynchronize(h->stream));
  }
  (void)hipFree(stage);
  MCHK(hipMemcpy(h->dT, targets, (size_t)n * 2 * 4, hipMemcpyHostToDevice));
  h->n_data = n;
  return SHP_OK;
}

// `steps` Adam steps on mini-batches whose row indices (steps x batch,
// into the training set) are given by the caller; loss_out[s] receives the
// mean squared error of step s's batch before its update.
shp_status shp_mlp_train(shp_mlp* h, const int32_t* indices, int32_t steps, int32_t batch, float lr,
                         float* loss_out) {
  if (!h || !indices || steps <= 0 || batch <= 0 || batch % TILE) return mlp_fail(SHP_E_INVAL, "bad argument");
  if (!h->dX) return mlp_fail(SHP_E_INVAL, "no training data");
  const long total = (long)steps * batch;
  int32_t lo = 0, hi = 0;
  for (long i = 0; i < total; ++i) {
    lo = indices[i] < lo ? indices[i] : lo;
    hi = indices[i] > hi ? indices[i] : hi;
  }
  if (lo < 0 || hi >= h->n_data) return mlp_fail(SHP_E_INVAL, "training index out of range");
  shp_status st = mlp_reserve_tiles(h, batch);
  if (st == SHP_OK && loss_out) st = mlp_reserve(h, batch);
  if (st != SHP_OK) return st;
  if (total > h->cap_idx) {
    if (h->didx) (void)hipFree(h->didx);
    h->didx = nullptr;
    h->cap_idx = 0;
    MCHK(hipMalloc(&h->didx, (size_t)total * 4));
    h->cap_idx = total;
  }
  MCHK(hipMemcpy(h->didx, indices, (size_t)total * 4, hipMemcpyHostToDevice));
  std::vector<float> y((size_t)batch * 2), t((size_t)batch * 2);
  for (int s = 0; s < steps; ++s) {
    const TrainRows rows{h->dX, h->dT, h->didx + (size_t)s * batch, nullptr, nullptr};
    ++h->adam_t;
    float b1c = 1.0f - powf(0.9f, (float)h->adam_t);
    float b2c = 1.0f - powf(0.999f, (float)h->adam_t);
    launch_train(h, rows, batch, loss_out ? h->out : nullptr, loss_out ? h->T : nullptr,
                 MlpStep{nullptr, h->p.w, h->mom, h->vel, h->p.wfr, lr, b1c, b2c});
    MCHK(hipGetLastError());
    if (loss_out) {
      MCHK(hipMemcpyAsync(y.data(), h->out, y.size() * 4, hipMemcpyDeviceToHost, h->stream));
      MCHK(hipMemcpyAsync(t.data(), h->T, t.size() * 4, hipMemcpyDeviceToHost, h->stream));
      MCHK(hipStreamSynchronize(h->stream));
      double l = 0.0;
      for (size_t i = 0; i < y.size(); ++i) {
        const double d = (double)y[i] - t[i];
        l += d * d;
      }
      loss_out[s] = (float)(l / batch);
    }
  }
  (void)hipStreamSynchronize(h->stream);
  return SHP_OK;
}

}  // extern "C"
