// MLP surrogate of the SMA return map on gfx950 BF16 MFMA.
//
// Network 16 -> 128 -> 128 -> 128 -> 128 -> 12, SiLU on the hidden layers,
// BF16 weights and activations, FP32 accumulation (v_mfma_f32_16x16x32_bf16).
// Device layouts pad the input to 32 features and the output to 32 so every
// GEMM is made of 16x16x32 tiles:
//   layer 0: W [128][32]   layers 1-3: W [128][128]   layer 4: W [32][128]
// (row n holds the weights into output n; rows/cols beyond the real sizes
// are zero).  The reference has no surrogate; its closest analogue is
// ann_framework%eval(nvec, input, output) (alya-ann/mod_ann_framework.f90:
// 489-556), which scales inputs, runs the network and unscales outputs per
// Gauss point, as sma_surrogate_eval does here.
//
// MFMA 16x16x32 lane layout (wave64), lane l:
//   A fragment: A[row = l%16][k = 8*(l/16) + j], j = 0..7
//   B fragment: B[k = 8*(l/16) + j][col = l%16]
//   D fragment: D[row = 4*(l/16) + i][col = l%16], i = 0..3
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "sma_law.hpp"
#include "surrogate_features.hpp"

namespace mlp {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int KP0 = 32, NP4 = 32;      // padded input / output widths
constexpr int NLAYER = 5;
__host__ __device__ constexpr int layer_k(int l) { return l == 0 ? KP0 : NH; }
__host__ __device__ constexpr int layer_n(int l) { return l == 4 ? NP4 : NH; }
__host__ __device__ constexpr int layer_kreal(int l) { return l == 0 ? NIN : NH; }
__host__ __device__ constexpr int layer_nreal(int l) { return l == 4 ? NOUT : NH; }
// offsets (elements) of each padded layer in the packed weight / bias arrays
__host__ __device__ constexpr int woff(int l) {
  return l == 0 ? 0 : l == 1 ? NH * KP0 : l == 2 ? NH * KP0 + NH * NH
       : l == 3 ? NH * KP0 + 2 * NH * NH : NH * KP0 + 3 * NH * NH;
}
constexpr int WPAD_TOTAL = NH * KP0 + 3 * NH * NH + NP4 * NH;   // 57344
__host__ __device__ constexpr int boff(int l) { return l * NH; }
constexpr int BPAD_TOTAL = 4 * NH + NP4;                         // 544
// canonical (unpadded) master layout: W_l [nreal][kreal] then all biases
__host__ __device__ constexpr int woff_c(int l) {
  return l == 0 ? 0 : l == 1 ? NH * NIN : l == 2 ? NH * NIN + NH * NH
       : l == 3 ? NH * NIN + 2 * NH * NH : NH * NIN + 3 * NH * NH;
}
constexpr int W_TOTAL = NH * NIN + 3 * NH * NH + NOUT * NH;      // 52736
constexpr int B_TOTAL = 4 * NH + NOUT;                           // 524

// output rows of a layer held in LDS (the output layer needs its first 16)
__host__ __device__ constexpr int inf_n(int l) { return l == NLAYER - 1 ? 16 : NH; }
static_assert(NOUT <= 16, "the output layer is one 16-feature block");
// Inference layout of the weights (a device copy, kept by pack_params and
// reduce_adam, that the inference kernel copies into LDS as it is).  Rows of
// K + 8 BF16 (16 more bytes) per row.  An A fragment is
// 16 rows x 16 bytes read at once; with rows of K = 128 (or 32) BF16 every
// row starts in the same LDS bank group, and the 16 reads would queue on it.
__host__ __device__ constexpr int wld(int l) { return layer_k(l) + 8; }
__host__ __device__ constexpr int woff_lds(int l) {
  return l == 0 ? 0 : woff_lds(l - 1) + inf_n(l - 1) * wld(l - 1);
}
constexpr int WLDS_TOTAL = woff_lds(NLAYER);
constexpr int BLDS_TOTAL = (NLAYER - 1) * NH + 16;
// input position, in a hidden layer's stored weight row, of the previous
// layer's feature f = 16 b + 4 q + i: 32 (b >> 1) + 8 q + 4 (b & 1) + i
__host__ __device__ constexpr int kperm(int f) {
  return 32 * (f >> 5) + 8 * ((f >> 2) & 3) + 4 * ((f >> 4) & 1) + (f & 3);
}

constexpr bool kperm_is_bijection() {
  bool seen[NH] = {};
  for (int f = 0; f < NH; ++f) {
    const int p = kperm(f);
    if (p < 0 || p >= NH || seen[p]) return false;
    seen[p] = true;
  }
  return true;
}
static_assert(kperm_is_bijection(), "kperm permutes the hidden inputs");

// index of padded weight (l, n, k) in the inference layout; -1: not kept
__host__ __device__ constexpr int inf_index(int l, int n, int k) {
  return n < inf_n(l) ? woff_lds(l) + n * wld(l) + (l == 0 ? k : kperm(k)) : -1;
}


// z sigmoid(z) with the hardware reciprocal (1 ulp): the result is rounded to
// BF16 (8 significant bits) before it is used
__device__ __forceinline__ float silu(float z) {
  return z * __builtin_amdgcn_rcpf(1.0f + __expf(-z));
}
// s = sigmoid(z) to half an ulp or so (one Newton step on the hardware
// reciprocal), silu(z) = z s and silu'(z) = s (1 + z (1 - s)).
__device__ __forceinline__ void silu_both(float z, float& y, float& g) {
  const float t = 1.0f + __expf(-z);
  float s = __builtin_amdgcn_rcpf(t);
  y = z * s;
  // t is infinite below z = -88: s and both results are then 0, however large -z
  s = fmaf(fmaf(-fminf(t, 0x1.fffffep127f), s, 1.0f), s, s);
  g = s * (1.0f + z * (1.0f - s));
}

// ----------------------------------------------------------------------------
// Training: forward, loss, backward and weight gradients of TR_ROWS rows in one
// workgroup, one launch per mini-batch.  What bounds it at 16384 rows (256
// workgroups, one per CU): the chain of ~14 phases between barriers, each a
// load or LDS read, 8 MFMA deep, an activation and an LDS write (a 1000-row
// batch, 16 workgroups, takes 27 us; the activations are 4 us of it, the bias
// sums 1; counters: a wave waits 58% of its time, the VALU is busy 0.27 and the
// matrix cores 0.07), then writing the partial gradients (213 KB a workgroup, 54
// MB, 7 us; reduce_adam reads them once).  Neither the 5.2 GFLOP (4 us at the rate
// of a large BF16 product) nor the 1.8 MB of samples count.  Separate launches
// per layer, product and activation with FP32 intermediates in memory took 930
// us for those rows (45 launches, 0.5 GB); this takes 35, reduce_adam 13.
// Half as many workgroups (and partials) take 1.5 times as long; loading the
// biases, targets and output weights ahead spills and gains nothing.
//   Products are formed as in the inference kernel (weights or their transposes
// as the A operand), so a lane (r, q) = (lane & 15, lane >> 4) holds features
// 4 q + i of row r of each 16x16 block: 8 waves share a layer's 128 features x
// 64 rows as 4 x 2 blocks of 32 x 32.  silu' stays in registers (FP32) from the
// forward to the backward pass.  LDS holds, in BF16, the layer input by rows
// (operand of the next layer) and every layer's output and dZ by features
// (operands of the weight gradient, whose sum runs over rows), 146 KB in all.
//   Precision as before: BF16 weights, activations and dZ in the products, FP32
// accumulation, FP32 Z, silu', dZ and bias gradients.
// ----------------------------------------------------------------------------
constexpr int TR_ROWS = 64, TR_WAVES = 8, TR_THREADS = TR_WAVES * 64;
constexpr int TR_MAX_GRID = 256;                  // workgroups (= partial gradients)
constexpr int GRAD_TOTAL = W_TOTAL + B_TOTAL;     // a partial gradient: canonical weights, then biases
static_assert(GRAD_TOTAL % 4 == 0 && W_TOTAL % 4 == 0, "partials are read four at a time");
constexpr int TR_NS = NH + 8;                     // row stride by rows (16 bytes more than 128 features)
constexpr int TR_TS = TR_ROWS + 8;                // row stride by features
constexpr int TR_XS = KP0 + 8;                    // row stride of the 32-wide input and output rows
// transposed weights [k][n] of layers 1..4 (padded as the forward copy)
__host__ __device__ constexpr int wtoff(int l) { return (l - 1) * NH * NH; }
constexpr int WT_TOTAL = 3 * NH * NH + NH * NP4;

struct TrainLds {
  __bf16 rows[2][TR_ROWS * TR_NS];                // layer inputs, then dZ, by rows
  __bf16 x0[TR_ROWS * TR_XS], d4[TR_ROWS * TR_XS];
  __bf16 yt[4][NH * TR_TS];                       // Y_0..Y_3 by features
  __bf16 t0[NH * TR_TS];                          // dZ by features
  __bf16 x0t[NIN * TR_TS], d4t[16 * TR_TS];
  float db[2][B_TOTAL];                           // bias gradients of the two row halves (hidden layers)
  float db4[4][16];                               // and of the output layer's four row blocks
  float loss[4];
};

struct TrainArgs {
  const __bf16* Wp;      // padded weights [n][k]
  const __bf16* Wt;      // transposed weights of layers 1..4
  const float* bp;
  const float* X;        // [n][16]
  const float* T;        // [n][12]
  const float* w;        // loss weights
  int64_t n;
  int chunks;            // ceil(n / TR_ROWS); workgroup b takes chunks b, b + grid, ...
  float* part;           // [grid][GRAD_TOTAL]
  float* loss_part;      // [grid]
};

__device__ __forceinline__ void zero_blocks(f32x4 (&acc)[2][2]) {
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int k = 0; k < 2; ++k) acc[f][k] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// A operand of a wave's 32 features of a layer (rows of K weights, 8
// consecutive ones per lane), loaded ahead of the product that uses it
template <int K>
struct Weights {
  bf16x8 a[K / 32][2];
  __device__ __forceinline__ void load(const __bf16* A, int f0, int r, int q) {
#pragma unroll
    for (int c = 0; c < K / 32; ++c)
#pragma unroll
      for (int k = 0; k < 2; ++k)
        a[c][k] = *reinterpret_cast<const bf16x8*>(A + (f0 + 16 * k + r) * K + 32 * c + 8 * q);
  }
};

// acc[fb][rb] = A (32 features x K) B (K x 32 rows), B rows of stride ls in LDS
template <int K>
__device__ __forceinline__ void block_product(f32x4 (&acc)[2][2], const Weights<K>& w, const __bf16* B, int ls,
                                              int r0, int r, int q) {
  zero_blocks(acc);
#pragma unroll
  for (int c = 0; c < K / 32; ++c) {
    bf16x8 b[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
      b[k] = *reinterpret_cast<const bf16x8*>(B + (r0 + 16 * k + r) * ls + 32 * c + 8 * q);
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int k = 0; k < 2; ++k)
        acc[f][k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.a[c][f], b[k], acc[f][k], 0, 0, 0);
  }
}

// Workgroup barrier for LDS alone: loads of weights for the next layer and
// stores of gradients stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// sum over the 16 lanes r of a quarter wave (DPP exchanges with l ^ 1, l ^ 2,
// l ^ 7 and l ^ 15: after each the sums of a growing group agree)
__device__ __forceinline__ float sum16(float v) {
  auto add = [&](auto ctrl) {
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  add(std::integral_constant<int, 0xB1>{});
  add(std::integral_constant<int, 0x4E>{});
  add(std::integral_constant<int, 0x141>{});
  add(std::integral_constant<int, 0x140>{});
  return v;
}

// 4 consecutive features of one row to the layout by rows (one 8-byte write)
// and by features
__device__ __forceinline__ void put4(bf16x4 h, __bf16* rows, int ls, __bf16* feat, int f, int row) {
  if (rows) *reinterpret_cast<bf16x4*>(rows + row * ls + f) = h;
#pragma unroll
  for (int i = 0; i < 4; ++i) feat[(f + i) * TR_TS + row] = h[i];
}

// weight gradient blocks: out[n][k] (+)= sum over the rows of dZ[n] Y[k], K-blocks
// of 16 (kt by features) and one block of 16 n (dt)
template <int NKB>
__device__ __forceinline__ void grad_blocks(const __bf16* kt, const __bf16* dt, int k0, int n0, float* out,
                                            int ldo, int nreal, bool first, int r, int q) {
  const int n = n0 + r;
  f32x4 acc[NKB];
#pragma unroll
  for (int k = 0; k < NKB; ++k) {
    acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (!first && n < nreal) acc[k] = *reinterpret_cast<const f32x4*>(out + n * ldo + k0 + 16 * k + 4 * q);
  }
#pragma unroll
  for (int s = 0; s < TR_ROWS / 32; ++s) {
    const bf16x8 d = *reinterpret_cast<const bf16x8*>(dt + n * TR_TS + 32 * s + 8 * q);
#pragma unroll
    for (int k = 0; k < NKB; ++k) {
      const bf16x8 y = *reinterpret_cast<const bf16x8*>(kt + (k0 + 16 * k + r) * TR_TS + 32 * s + 8 * q);
      acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y, d, acc[k], 0, 0, 0);
    }
  }
  if (n < nreal) {
#pragma unroll
    for (int k = 0; k < NKB; ++k)
      *reinterpret_cast<f32x4*>(out + n * ldo + k0 + 16 * k + 4 * q) = acc[k];
  }
}

__device__ __forceinline__ int opaque_index(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

__global__ void __launch_bounds__(TR_THREADS, 2) mlp_train(TrainArgs A) {
  extern __shared__ __align__(16) unsigned char smem[];
  TrainLds& S = *reinterpret_cast<TrainLds*>(smem);
  const int tid = threadIdx.x;
  float* part = A.part + (int64_t)blockIdx.x * GRAD_TOTAL;
  for (int i = tid; i < 2 * B_TOTAL; i += TR_THREADS) (&S.db[0][0])[i] = 0.f;
  if (tid < 64) (&S.db4[0][0])[tid] = 0.f;
  for (int i = tid; i < TR_ROWS * TR_XS; i += TR_THREADS) S.d4[i] = (__bf16)0.f;
  float loss = 0.f;
  bool first = true;
  for (int ch = blockIdx.x; ch < A.chunks; ch += gridDim.x, first = false) {
    const int64_t m0 = (int64_t)ch * TR_ROWS;
    // the thread index passes through an empty asm in every phase, so that
    // addresses are formed where they are used and not held through the loop
    int lane, wave, r, q, f0, rg, r0;
    auto phase = [&]() {
      const int t = opaque_index(tid);
      lane = t & 63;
      wave = __builtin_amdgcn_readfirstlane(t >> 6);
      r = lane & 15;
      q = lane >> 4;
      f0 = 32 * (wave & 3);
      rg = wave >> 2;
      r0 = 32 * rg;
    };
    // inputs: 16 features a row (zero beyond the batch), 16 more of padding
    for (int i = tid; i < TR_ROWS * KP0; i += TR_THREADS) {
      const int row = i / KP0, k = i % KP0;
      const __bf16 x = (__bf16)((m0 + row < A.n && k < NIN) ? A.X[(m0 + row) * NIN + k] : 0.f);
      S.x0[row * TR_XS + k] = x;
      if (k < NIN) S.x0t[k * TR_TS + row] = x;
    }
    lds_barrier();
    f32x4 g[4][2][2];   // silu'(Z_l) of the wave's block
    f32x4 acc[2][2];
    // Z_l in acc -> Y_l by rows and by features, silu'(Z_l)
    auto activate = [&](int l) {
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        const int feat = f0 + 16 * f + 4 * q;
        const f32x4 b = *reinterpret_cast<const f32x4*>(A.bp + boff(l) + feat);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          bf16x4 h;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float y, gi;
            silu_both(acc[f][k][i] + b[i], y, gi);
            h[i] = (__bf16)y;
            g[l][f][k][i] = gi;
          }
          put4(h, S.rows[l & 1], TR_NS, S.yt[l], feat, r0 + 16 * k + r);
        }
      }
    };
    Weights<NH> w;
    {
      Weights<KP0> w0;
      phase();
      w0.load(A.Wp + woff(0), f0, r, q);
      w.load(A.Wp + woff(1), f0, r, q);
      block_product<KP0>(acc, w0, S.x0, TR_XS, r0, r, q);
      activate(0);
      lds_barrier();
    }
#pragma unroll
    for (int l = 1; l < 4; ++l) {
      phase();
      block_product<NH>(acc, w, S.rows[(l - 1) & 1], TR_NS, r0, r, q);
      w.load(l < 3 ? A.Wp + woff(l + 1) : A.Wt + wtoff(3), f0, r, q);
      activate(l);
      lds_barrier();
    }
    // output layer, loss and its gradient: waves 0..3, 16 rows each
    phase();
    if (wave < 4) {
      const int row = 16 * wave + r;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NH / 32; ++c) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(A.Wp + woff(4) + r * NH + 32 * c + 8 * q);
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(S.rows[1] + row * TR_NS + 32 * c + 8 * q);
        o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, o, 0, 0, 0);
      }
      bf16x4 h;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = 4 * q + i;
        float gj = 0.f;
        if (m0 + row < A.n && j < NOUT) {
          const float d = o[i] + A.bp[boff(4) + j] - A.T[(m0 + row) * NOUT + j];
          loss += A.w[j] * d * d;
          gj = 2.f * A.w[j] * d / (float)A.n;
        }
        h[i] = (__bf16)gj;
        const float sj = sum16(gj);
        if (r == 0 && j < NOUT) S.db4[wave][j] += sj;
      }
      put4(h, S.d4, TR_XS, S.d4t, 4 * q, row);
    }
    Weights<NP4> w4;
    w4.load(A.Wt + wtoff(4), f0, r, q);
    lds_barrier();
    // backward: the weight gradient of layer l and dZ of layer l - 1
    auto back = [&](int l, __bf16* rows, __bf16* feat) {
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        const int fe = f0 + 16 * f + 4 * q;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          bf16x4 h;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float d = acc[f][k][i] * g[l][f][k][i];
            h[i] = (__bf16)d;
            s[i] += d;
          }
          put4(h, rows, TR_NS, feat, fe, r0 + 16 * k + r);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float t = sum16(s[i]);
          if (r == 0) S.db[rg][boff(l) + fe + i] += t;
        }
      }
    };
    phase();
    block_product<NP4>(acc, w4, S.d4, TR_XS, r0, r, q);
    back(3, S.rows[0], S.t0);
    grad_blocks<1>(S.yt[3], S.d4t, 16 * wave, 0, part + woff_c(4), NH, NOUT, first, r, q);
    lds_barrier();
#pragma unroll
    for (int l = 3; l >= 1; --l) {
      // dZ_3 and dZ_1 by features lie in t0, dZ_2 and dZ_0 over Y_3 (whose last
      // reader was the output layer's gradient)
      const __bf16* dt = (l & 1) ? S.t0 : S.yt[3];
      phase();
      block_product<NH>(acc, w, S.rows[(l & 1) ^ 1], TR_NS, r0, r, q);
      if (l > 1) w.load(A.Wt + wtoff(l - 1), f0, r, q);
      back(l - 1, l > 1 ? S.rows[l & 1] : nullptr, (l & 1) ? S.yt[3] : S.t0);
      phase();
#pragma unroll
      for (int b = 0; b < 2; ++b)   // the gradient: 32 n x 64 k a wave
        grad_blocks<4>(S.yt[l - 1], dt, 64 * rg, f0 + 16 * b, part + woff_c(l), NH, NH, first, r, q);
      lds_barrier();
    }
    phase();
    grad_blocks<1>(S.x0t, S.yt[3], 0, 16 * wave, part + woff_c(0), NIN, NH, first, r, q);
    lds_barrier();   // the next chunk writes x0t and Y_3
  }
  for (int i = tid; i < B_TOTAL; i += TR_THREADS) {
    const int j = i - boff(4);
    part[W_TOTAL + i] = j < 0 ? S.db[0][i] + S.db[1][i]
                              : (S.db4[0][j] + S.db4[1][j]) + (S.db4[2][j] + S.db4[3][j]);
  }
  for (int d = 32; d > 0; d >>= 1) loss += __shfl_xor(loss, d);
  if ((tid & 63) == 0 && tid < 256) S.loss[tid >> 6] = loss;
  __syncthreads();
  if (tid == 0) A.loss_part[blockIdx.x] = (S.loss[0] + S.loss[1]) + (S.loss[2] + S.loss[3]);
}

// Sum of the partial gradients in a fixed order (deterministic), then Adam on
// the canonical FP32 master parameters; refreshes the padded BF16 weights and
// FP32 biases the kernels read.  W null: the gradient alone, to gW and gb.
// Bound by reading the partials (54 MB at 256 workgroups): 16 threads share an
// element's partials (a quarter of a wave reads 64 consecutive floats of one),
// so that enough loads are in flight.
struct AdamArgs {
  const float* part; int parts;
  float* W; float* b;            // master, canonical
  float* mW; float* vW; float* mb; float* vb;
  float* gW; float* gb;          // gradient out (W null)
  __bf16* Wp; float* bp;         // padded device copies
  __bf16* Wi;                    // inference layout
  __bf16* Wt;                    // transposed weights
  float lr, beta1, beta2, eps, bc1, bc2;
};

__device__ __forceinline__ void adam1(float& p, float& m, float& v, float g, const AdamArgs& A) {
  m = A.beta1 * m + (1.f - A.beta1) * g;
  v = A.beta2 * v + (1.f - A.beta2) * g * g;
  const float mh = m / A.bc1, vh = v / A.bc2;
  p -= A.lr * mh / (sqrtf(vh) + A.eps);
}

constexpr int RED_ELEMS = 64;    // gradient elements per workgroup of 256
__global__ void __launch_bounds__(256) reduce_adam(AdamArgs A) {
  __shared__ float red[16][RED_ELEMS];
  const int c = threadIdx.x & 15, z = threadIdx.x >> 4;
  const int i4 = blockIdx.x * RED_ELEMS + 4 * c;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  if (i4 < GRAD_TOTAL) {
#pragma unroll 8
    for (int p = z; p < A.parts; p += 16)
      s += *reinterpret_cast<const f32x4*>(A.part + (int64_t)p * GRAD_TOTAL + i4);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) red[z][4 * c + k] = s[k];
  __syncthreads();
  if (threadIdx.x >= RED_ELEMS) return;
  const int i = blockIdx.x * RED_ELEMS + threadIdx.x;
  if (i >= GRAD_TOTAL) return;
  float g = 0.f;
#pragma unroll
  for (int k = 0; k < 16; ++k) g += red[k][threadIdx.x];
  if (!A.W) {
    if (i < W_TOTAL) A.gW[i] = g;
    else A.gb[i - W_TOTAL] = g;
    return;
  }
  if (i < W_TOTAL) {
    float w = A.W[i];
    adam1(w, A.mW[i], A.vW[i], g, A);
    A.W[i] = w;
    int l = 0;
    while (l < 4 && i >= woff_c(l + 1)) ++l;
    const int kr = layer_kreal(l), K = layer_k(l);
    const int j = i - woff_c(l), n = j / kr, k = j % kr;
    const __bf16 h = (__bf16)w;
    A.Wp[woff(l) + n * K + k] = h;
    const int ii = inf_index(l, n, k);
    if (ii >= 0) A.Wi[ii] = h;
    if (l > 0) A.Wt[wtoff(l) + k * layer_n(l) + n] = h;
  } else {
    const int k = i - W_TOTAL;
    float w = A.b[k];
    adam1(w, A.mb[k], A.vb[k], g, A);
    A.b[k] = w;
    A.bp[k] = w;
  }
}

// Canonical FP32 params -> padded device copies (pads zero).
__global__ void pack_params(const float* __restrict__ W, const float* __restrict__ b,
                            __bf16* __restrict__ Wp, __bf16* __restrict__ Wi,
                            __bf16* __restrict__ Wt, float* __restrict__ bp) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < WPAD_TOTAL) {
    int l = 0;
    while (l < 4 && i >= woff(l + 1)) ++l;
    const int K = layer_k(l), j = i - woff(l), n = j / K, k = j % K;
    float v = 0.f;
    if (n < layer_nreal(l) && k < layer_kreal(l)) v = W[woff_c(l) + n * layer_kreal(l) + k];
    Wp[i] = (__bf16)v;
    const int ii = inf_index(l, n, k);
    if (ii >= 0) Wi[ii] = (__bf16)v;
    if (l > 0) Wt[wtoff(l) + k * layer_n(l) + n] = (__bf16)v;
  }
  if (i < BPAD_TOTAL) bp[i] = (i < B_TOTAL) ? b[i] : 0.f;
}

// ----------------------------------------------------------------------------
// Fused inference: all 5 layers of a block of 32 rows in one wave, weights
// staged in LDS once per workgroup.  Y [n][12] fp32.
//
// The product is formed transposed (weights as the A operand, activations
// as the B operand of v_mfma_f32_16x16x32_bf16), so a layer leaves lane
// (r, q) = (lane & 15, lane >> 4) holding features 16 b + 4 q + i (b = 0..7,
// i = 0..3) of row r of each 16-row block.  The next layer's B fragment for
// inputs 32 c .. 32 c + 31 wants, in lane (r, q), 8 inputs of row r: the
// hidden layers' weight columns are stored permuted (kperm) so that these 8
// are the lane's own features of blocks b = 2 c and 2 c + 1.  Activations
// therefore stay in registers from layer to layer (no LDS round trip, no
// barrier), and LDS holds only the weights: 121 KB, one workgroup per CU.
// A wave carries two 16-row blocks (each A fragment read from LDS feeds two
// MFMA) in 228 VGPRs, so the workgroup has 8 waves, two per SIMD: one
// wave's SiLU epilogue (the kernel's largest cost) overlaps the other's MFMA.
// What bounds it: the VALU is busy 0.60 of the time (counters; 35 cycles an
// activation, two transcendentals of 8 cycles among them: 23 us for 200 000
// rows), the matrix cores 0.23 (9 us), and two waves a SIMD leave a part of either
// and of the LDS reads of the weights uncovered.  Waves take 32-row blocks round
// robin over the grid (block k on workgroup k mod grid), so a short list spreads
// over every CU; the rows left after the full rounds go by 16 to a wave when that
// takes them all, since a wave with a lone 32-row block at the end runs half a
// round longer.
// Rows, before -> with 16-row ends: 500 10.4 -> 7.8 us, 16384 11.1 -> 8.7,
// 200000 44.9 -> 41.5, 400000 80 -> 78; the same where the rest is more than half
// a round (40000: 15.8).
// ----------------------------------------------------------------------------
constexpr int INF_WAVES = 8;
constexpr int INF_THREADS = INF_WAVES * 64;
constexpr int INF_RB = 2;                        // 16-row MFMA blocks per wave block
constexpr int INF_ROWS = 16 * INF_RB;            // rows per wave block
__device__ __forceinline__ bf16x8 cat4(bf16x4 a, bf16x4 b) {
  return bf16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

// A layer's accumulators start at its bias (lane (r, q) holds features
// 16 b + 4 q + i), so the MFMA chain leaves Z = W x + b and the epilogue
// adds nothing
template <int RB>
__device__ __forceinline__ void bias_init(f32x4 (&acc)[RB][8], const float* bias, int q) {
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const f32x4 bc = *reinterpret_cast<const f32x4*>(bias + 16 * b + 4 * q);
#pragma unroll
    for (int a = 0; a < RB; ++a) acc[a][b] = bc;
  }
}

// SiLU of one layer's Z into the next layer's inputs
template <int RB>
__device__ __forceinline__ void hidden_epilogue(const f32x4 (&acc)[RB][8], bf16x4 (&h)[RB][8]) {
#pragma unroll
  for (int b = 0; b < 8; ++b)
#pragma unroll
    for (int a = 0; a < RB; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i) h[a][b][i] = (__bf16)silu(acc[a][b][i]);
}

__global__ void __launch_bounds__(INF_THREADS) mlp_infer(const __bf16* __restrict__ Wi,
                                                         const float* __restrict__ bp,
                                                         const float* __restrict__ X, int64_t n_host,
                                                         const unsigned* __restrict__ seg_count,
                                                         int64_t seg_cap, float* __restrict__ Y) {
  // rows 0 .. n_host - 1 of X and Y, or the step's list: its segment
  // counters are read on the device (graph-captured steps), the i-th listed
  // point's row is its slot
  __shared__ unsigned off[LIST_SEGS + 1];
  const int64_t n = seg_count ? (int64_t)list_scan(seg_count, off) : n_host;
  // full rounds of INF_ROWS rows for every wave, then the rest: 16 rows a wave
  // if that takes them all, so that a last round costs half a block's time
  const int64_t nwaves = (int64_t)gridDim.x * INF_WAVES;
  const int64_t full = n / (nwaves * INF_ROWS), rest0 = full * nwaves * INF_ROWS, rest = n - rest0;
  const int rest_rows = rest > 16 * nwaves ? INF_ROWS : 16;
  // a workgroup without a row block leaves before copying the weights
  if (full == 0 && (int64_t)blockIdx.x * rest_rows >= rest) return;
  extern __shared__ __align__(16) unsigned char smem[];
  __bf16* sW = reinterpret_cast<__bf16*>(smem);
  float* sb = reinterpret_cast<float*>(smem + WLDS_TOTAL * sizeof(__bf16));
  const int tid = threadIdx.x;
  // the inference layout as it is, 16 bytes per copy
  static_assert(WLDS_TOTAL % 8 == 0, "whole 16-byte chunks");
  for (int t = tid; t < WLDS_TOTAL / 8; t += blockDim.x)
    reinterpret_cast<bf16x8*>(sW)[t] = reinterpret_cast<const bf16x8*>(Wi)[t];
  for (int i = tid; i < BLDS_TOTAL; i += blockDim.x) sb[i] = bp[i];
  __syncthreads();
  const int lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  static_assert(INF_ROWS <= 64, "one lane holds the slot of each row of a block");
  // RB 16-row blocks from row0 on
  auto block = [&](auto rb, int64_t row0) {
    constexpr int RB = decltype(rb)::value;
    // lane l < 16 RB: the slot of row row0 + l
    int slot_l = 0;
    if (lane < 16 * RB && row0 + lane < n)
      slot_l = seg_count ? (int)list_slot(off, (unsigned)(row0 + lane), seg_cap) : (int)(row0 + lane);
    // layer 0's B fragments: inputs 8 q .. 8 q + 7 of row 16 a + r (NIN = 16
    // real inputs; lanes q >= 2 hold the zero padding)
    bf16x8 x0[RB];
#pragma unroll
    for (int a = 0; a < RB; ++a) {
      const int64_t sl = __shfl(slot_l, 16 * a + r);
      float4 lo = make_float4(0.f, 0.f, 0.f, 0.f), hi = lo;
      if (q < 2 && row0 + 16 * a + r < n) {
        const float4* src = reinterpret_cast<const float4*>(X + sl * NIN + 8 * q);
        lo = src[0];
        hi = src[1];
      }
      x0[a] = bf16x8{(__bf16)lo.x, (__bf16)lo.y, (__bf16)lo.z, (__bf16)lo.w,
                     (__bf16)hi.x, (__bf16)hi.y, (__bf16)hi.z, (__bf16)hi.w};
    }
    bf16x4 h[RB][8];
    f32x4 acc[RB][8];
    // layer 0 (K = 32)
    bias_init(acc, sb + boff(0), q);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bf16x8 wf = *reinterpret_cast<const bf16x8*>(sW + (16 * b + r) * wld(0) + 8 * q);
#pragma unroll
      for (int a = 0; a < RB; ++a)
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, x0[a], acc[a][b], 0, 0, 0);
    }
    hidden_epilogue(acc, h);
    // hidden layers 1 .. NLAYER - 2 (K = 128)
#pragma unroll 1
    for (int l = 1; l < NLAYER - 1; ++l) {
      const __bf16* W = sW + woff_lds(1) + (l - 1) * NH * wld(1);
      bias_init(acc, sb + boff(l), q);
#pragma unroll
      for (int c = 0; c < NH / 32; ++c) {
        bf16x8 xf[RB];
#pragma unroll
        for (int a = 0; a < RB; ++a) xf[a] = cat4(h[a][2 * c], h[a][2 * c + 1]);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          const bf16x8 wf =
              *reinterpret_cast<const bf16x8*>(W + (16 * b + r) * wld(1) + 32 * c + 8 * q);
#pragma unroll
          for (int a = 0; a < RB; ++a)
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf[a], acc[a][b], 0, 0, 0);
        }
      }
      hidden_epilogue(acc, h);
    }
    // output layer: one 16-feature block, Y = Z (fp32)
    {
      constexpr int l = NLAYER - 1;
      const __bf16* W = sW + woff_lds(l);
      // features 4 q .. 4 q + 3 of the output block, from its bias (zero
      // beyond NOUT)
      const f32x4 bo = *reinterpret_cast<const f32x4*>(sb + boff(l) + 4 * q);
      f32x4 o[RB];
#pragma unroll
      for (int a = 0; a < RB; ++a) o[a] = bo;
#pragma unroll
      for (int c = 0; c < NH / 32; ++c) {
        const bf16x8 wf = *reinterpret_cast<const bf16x8*>(W + r * wld(l) + 32 * c + 8 * q);
#pragma unroll
        for (int a = 0; a < RB; ++a)
          o[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, cat4(h[a][2 * c], h[a][2 * c + 1]),
                                                         o[a], 0, 0, 0);
      }
#pragma unroll
      for (int a = 0; a < RB; ++a) {
        const int64_t m = row0 + 16 * a + r;
        const int64_t sl = __shfl(slot_l, 16 * a + r);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int col = 4 * q + i;
          if (m < n && col < NOUT) Y[sl * NOUT + col] = o[a][i];
        }
      }
    }
  };
  const int64_t wid = (int64_t)wave * gridDim.x + blockIdx.x;
  for (int64_t k = 0; k < full; ++k) block(std::integral_constant<int, INF_RB>{}, (k * nwaves + wid) * INF_ROWS);
  if (wid * rest_rows < rest) {
    if (rest_rows == INF_ROWS) block(std::integral_constant<int, INF_RB>{}, rest0 + wid * INF_ROWS);
    else block(std::integral_constant<int, 1>{}, rest0 + wid * 16);
  }
}

constexpr size_t INF_SMEM = WLDS_TOTAL * sizeof(__bf16) + BLDS_TOTAL * sizeof(float);

// splitmix64 counter-based generator
__device__ __forceinline__ uint64_t smix(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}
struct Rng {
  uint64_t s;
  __device__ double uni() {  // (0, 1)
    s = smix(s);
    return ((double)(s >> 11) + 0.5) * (1.0 / 9007199254740992.0);
  }
  __device__ double normal() {
    const double u1 = uni(), u2 = uni();
    return sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
  }
};

// Principal values (descending) of a symmetric 3x3 log-strain tensor.
__device__ __forceinline__ void principal(const double (&s)[6], double& l0, double& l1, double& l2) {
  double q[9];
  sma::eig3<double>(s[0], s[3], s[4], s[1], s[5], s[2], l0, l1, l2, q);
}

struct GenArgs {
  int64_t n;
  uint64_t seed;
  const double* props;     // base material [18]
  double strain_sd, step_sd, jitter;
  float* X;                // [n][16]
  float* T;                // [n][12]
  uint32_t* flags;         // [n]
};

// Training samples drawn like the material-point workload: log-strain components ~ N(0, sd^2),
// the previous state one increment (~ N(0, step_sd^2)) away, xS_0 in [0, 1]
// (the transformation strain eL xS_0 inside the 0.05 ball), T ~ U[290, 340],
// material parameters jittered +-jitter.  Labels from the exact FP64 map.
__global__ void __launch_bounds__(256) gen_samples(GenArgs G) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= G.n) return;
  Rng rng{smix(G.seed * 0x2545F4914F6CDD1Dull + (uint64_t)i)};
  double p[18];
#pragma unroll
  for (int k = 0; k < 18; ++k) p[k] = G.props[k];
  const int jit[7] = {0, 1, 2, 3, 4, 9, 10};  // E, nu, eL, sigma_s/f AS, sigma_s/f SA
#pragma unroll
  for (int k = 0; k < 7; ++k) p[jit[k]] *= 1.0 + G.jitter * (2.0 * rng.uni() - 1.0);
  const double E = p[0];
  const double T = 290.0 + 50.0 * rng.uni();
  double eps[6], prev[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    eps[k] = G.strain_sd * rng.normal();
    prev[k] = eps[k] - G.step_sd * rng.normal();
  }
  const double u = rng.uni();
  double xS0 = (u < 0.15) ? 0.0 : (u < 0.25) ? 1.0 : rng.uni();
  double l0, l1, l2, q0, q1, q2;
  principal(eps, l0, l1, l2);
  principal(prev, q0, q1, q2);
  const double th = l0 + l1 + l2, thp = q0 + q1 + q2;
  const double e0 = l0 - th / 3.0, e1 = l1 - th / 3.0, e2 = l2 - th / 3.0;
  const double ep0 = q0 - thp / 3.0, ep1 = q1 - thp / 3.0, ep2 = q2 - thp / 3.0;
  const double en = sqrt(e0 * e0 + e1 * e1 + e2 * e2);
  const double enp = sqrt(ep0 * ep0 + ep1 * ep1 + ep2 * ep2);
  const sma::Mat m = sma::make_mat(p, E);
  const double FAS0 = sma::loading(m, m.C_AS, thp, enp, xS0);
  const double FSA0 = sma::loading(m, m.C_SA, thp, enp, xS0);
  const double Ftr = sma::loading(m, m.C_AS, th, en, xS0);
  const sma::ReturnMap rm = sma::return_map(m, th, en, xS0, FAS0, FSA0);
  float* f = G.X + i * NIN;
  make_features(p, E, T, e0, e1, e2, th, xS0, FAS0, FSA0, Ftr, f);
  const double d0 = en > 0 ? e0 / en : 0.0, d1 = en > 0 ? e1 / en : 0.0, d2 = en > 0 ? e2 / en : 0.0;
  const double vol = m.K * (th - 3.0 * m.alfa * m.eL * rm.xS);
  float* t = G.T + i * NOUT;
  t[0] = (float)((vol + 2.0 * m.G * (e0 - m.eL * rm.xS * d0)) * Scale::tau);
  t[1] = (float)((vol + 2.0 * m.G * (e1 - m.eL * rm.xS * d1)) * Scale::tau);
  t[2] = (float)((vol + 2.0 * m.G * (e2 - m.eL * rm.xS * d2)) * Scale::tau);
  t[3] = (float)(m.eL * rm.xS * d0 * Scale::etr);
  t[4] = (float)(m.eL * rm.xS * d1 * Scale::etr);
  t[5] = (float)(m.eL * rm.xS * d2 * Scale::etr);
  t[6] = (float)rm.xS;
  t[7] = (float)(rm.F_AS * Scale::F);
  t[8] = (float)(rm.F_SA * Scale::F);
  t[9] = (rm.flags & sma::FLAG_KF_AS) ? 1.f : 0.f;
  t[10] = (rm.flags & sma::FLAG_KF_SA) ? 1.f : 0.f;
  t[11] = (float)((rm.xS - xS0) * Scale::dx);
  G.flags[i] = rm.flags;
}

}  // namespace mlp
