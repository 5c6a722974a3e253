// C ABI of the MLP surrogate: parameters, fused BF16-MFMA inference,
// training (forward, backward, Adam) and the data generator.  Kernels are in
// surrogate.hpp; declarations in include/alya_sma.h.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <algorithm>
#include <random>
#include <string>
#include <vector>

#include "alya_sma.h"
#include "common.hpp"
#include "once_per_device.hpp"
#include "surrogate.hpp"

namespace {
#define SCHK(x) SMA_HIPCHK(x)
unsigned nb(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// The dynamic LDS limit of `kernel` on the current device (a limit holds for
// one device), whose CU count is returned.
int lds_limit(sma_abi::OncePerDevice& once, const void* kernel, int bytes, int* ncu = nullptr) {
  int dev = 0;
  SCHK(hipGetDevice(&dev));
  if (ncu) (void)hipDeviceGetAttribute(ncu, hipDeviceAttributeMultiprocessorCount, dev);
  return once(dev, [&]() -> int {
    SCHK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
    return SMA_OK;
  });
}
sma_abi::OncePerDevice g_infer_lds, g_train_lds;

int infer_lds(int* ncu) { return lds_limit(g_infer_lds, (const void*)mlp::mlp_infer, (int)mlp::INF_SMEM, ncu); }
}  // namespace

struct sma_mlp {
  // canonical FP32 master parameters and Adam state
  float *W = nullptr, *b = nullptr, *mW = nullptr, *vW = nullptr, *mb = nullptr, *vb = nullptr;
  // padded copies read by the kernels
  __bf16* Wp = nullptr;
  __bf16* Wi = nullptr;        // inference layout (mlp::inf_index)
  __bf16* Wt = nullptr;        // transposed weights of layers 1..4 (backward products)
  float* bp = nullptr;
  int64_t step = 0;
  // training workspace: partial gradients and losses (grown on demand)
  int cap = 0;
  float* part = nullptr;
  float* loss_part = nullptr;
  float* wloss = nullptr;
};

namespace {

int grow(sma_mlp* m, int parts) {
  if (parts <= m->cap) return 0;
  if (m->part) (void)hipFree(m->part);
  if (m->loss_part) (void)hipFree(m->loss_part);
  m->part = m->loss_part = nullptr;
  m->cap = 0;
  SCHK(hipMalloc((void**)&m->part, (size_t)parts * mlp::GRAD_TOTAL * sizeof(float)));
  SCHK(hipMalloc((void**)&m->loss_part, (size_t)parts * sizeof(float)));
  m->cap = parts;
  return 0;
}

mlp::AdamArgs adam_args(sma_mlp* m, int parts) {
  mlp::AdamArgs A{};
  A.part = m->part;
  A.parts = parts;
  return A;
}

// Forward, loss and backward of a mini-batch into `parts` partial gradients
// (returned through parts_out).
int train_pass(sma_mlp* m, int64_t n, const float* X, const float* T, int* parts_out, hipStream_t s) {
  if (n > (int64_t)INT32_MAX * mlp::TR_ROWS)
    return sma_abi::fail(SMA_ERR_ARG, "sma_mlp: mini-batch too large");
  if (int rc = lds_limit(g_train_lds, (const void*)mlp::mlp_train, (int)sizeof(mlp::TrainLds))) return rc;
  const int64_t chunks = (n + mlp::TR_ROWS - 1) / mlp::TR_ROWS;
  const int parts = (int)std::min<int64_t>(chunks, mlp::TR_MAX_GRID);
  if (int rc = grow(m, parts)) return rc;
  mlp::TrainArgs A{m->Wp, m->Wt, m->bp, X, T, m->wloss, n, (int)chunks, m->part, m->loss_part};
  hipLaunchKernelGGL(mlp::mlp_train, dim3(parts), dim3(mlp::TR_THREADS), sizeof(mlp::TrainLds), s, A);
  SCHK(hipGetLastError());
  *parts_out = parts;
  return 0;
}

int reduce(const mlp::AdamArgs& A, hipStream_t s) {
  hipLaunchKernelGGL(mlp::reduce_adam, dim3(nb(mlp::GRAD_TOTAL, mlp::RED_ELEMS)), dim3(256), 0, s, A);
  SCHK(hipGetLastError());
  return 0;
}

// Mean loss of the last train_pass (waits for the stream).
int mean_loss(sma_mlp* m, int64_t n, int parts, float* loss_out, hipStream_t s) {
  std::vector<float> lp(parts);
  SCHK(hipMemcpyAsync(lp.data(), m->loss_part, parts * sizeof(float), hipMemcpyDeviceToHost, s));
  SCHK(hipStreamSynchronize(s));
  double t = 0.0;
  for (float v : lp) t += v;
  *loss_out = (float)(t / (double)n);
  return 0;
}

}  // namespace

extern "C" {

int sma_mlp_create(uint64_t seed, sma_mlp** out) {
  if (!out) return sma_abi::fail(SMA_ERR_ARG, "sma_mlp_create: null out");
  sma_mlp* m = new sma_mlp();
  auto A = [&](auto** p, size_t bytes) -> int {
    SCHK(hipMalloc((void**)p, bytes));
    SCHK(hipMemset(*p, 0, bytes));
    return 0;
  };
  int rc = 0;
  if ((rc = A(&m->W, mlp::W_TOTAL * 4)) || (rc = A(&m->b, mlp::B_TOTAL * 4)) ||
      (rc = A(&m->mW, mlp::W_TOTAL * 4)) || (rc = A(&m->vW, mlp::W_TOTAL * 4)) ||
      (rc = A(&m->mb, mlp::B_TOTAL * 4)) || (rc = A(&m->vb, mlp::B_TOTAL * 4)) ||
      (rc = A(&m->Wp, mlp::WPAD_TOTAL * 2)) || (rc = A(&m->Wi, mlp::WLDS_TOTAL * 2)) ||
      (rc = A(&m->Wt, mlp::WT_TOTAL * 2)) || (rc = A(&m->bp, mlp::BPAD_TOTAL * 4)) ||
      (rc = A(&m->wloss, 16 * 4))) {
    sma_mlp_destroy(m);
    return rc;
  }
  // He-uniform initialisation, seeded
  std::mt19937_64 g(seed);
  std::vector<float> W(mlp::W_TOTAL), b(mlp::B_TOTAL, 0.f);
  for (int l = 0; l < 5; ++l) {
    const int kr = mlp::layer_kreal(l), nr = mlp::layer_nreal(l);
    const float lim = std::sqrt(6.0f / kr) * (l == 4 ? 0.5f : 1.0f);
    std::uniform_real_distribution<float> U(-lim, lim);
    for (int i = 0; i < nr * kr; ++i) W[mlp::woff_c(l) + i] = U(g);
  }
  rc = sma_mlp_set_params(m, W.data(), b.data());
  if (rc) { sma_mlp_destroy(m); return rc; }
  std::vector<float> w(16, 1.0f);
  if (hipMemcpy(m->wloss, w.data(), 16 * 4, hipMemcpyHostToDevice) != hipSuccess) {
    sma_mlp_destroy(m);
    return sma_abi::fail(SMA_ERR_HIP, "upload loss weights");
  }
  *out = m;
  return SMA_OK;
}

int sma_mlp_destroy(sma_mlp* m) {
  if (!m) return SMA_OK;
  void* ps[] = {m->W, m->b, m->mW, m->vW, m->mb, m->vb, m->Wp, m->Wi, m->Wt, m->bp, m->part,
                m->loss_part, m->wloss};
  for (void* p : ps) if (p) (void)hipFree(p);
  delete m;
  return SMA_OK;
}

int sma_mlp_set_params(sma_mlp* m, const float* W, const float* b) {
  if (!m || !W || !b) return sma_abi::fail(SMA_ERR_ARG, "sma_mlp_set_params: null argument");
  SCHK(hipMemcpy(m->W, W, mlp::W_TOTAL * 4, hipMemcpyHostToDevice));
  SCHK(hipMemcpy(m->b, b, mlp::B_TOTAL * 4, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(mlp::pack_params, dim3(nb(mlp::WPAD_TOTAL, 256)), dim3(256), 0, nullptr, m->W,
                     m->b, m->Wp, m->Wi, m->Wt, m->bp);
  SCHK(hipGetLastError());
  SCHK(hipDeviceSynchronize());
  return SMA_OK;
}

int sma_mlp_get_params(sma_mlp* m, float* W, float* b) {
  if (!m || !W || !b) return sma_abi::fail(SMA_ERR_ARG, "sma_mlp_get_params: null argument");
  SCHK(hipDeviceSynchronize());
  SCHK(hipMemcpy(W, m->W, mlp::W_TOTAL * 4, hipMemcpyDeviceToHost));
  SCHK(hipMemcpy(b, m->b, mlp::B_TOTAL * 4, hipMemcpyDeviceToHost));
  return SMA_OK;
}

int sma_mlp_set_loss_weights(sma_mlp* m, const float* w12) {
  if (!m || !w12) return sma_abi::fail(SMA_ERR_ARG, "null argument");
  std::vector<float> w(16, 0.f);
  std::memcpy(w.data(), w12, 12 * sizeof(float));
  SCHK(hipMemcpy(m->wloss, w.data(), 16 * 4, hipMemcpyHostToDevice));
  return SMA_OK;
}

int sma_mlp_forward_device(sma_mlp* m, int64_t n, const float* X, float* Y, void* stream) {
  if (!m || n < 0 || (n > 0 && (!X || !Y))) return sma_abi::fail(SMA_ERR_ARG, "sma_mlp_forward_device: bad arguments");
  if (n > INT32_MAX) return sma_abi::fail(SMA_ERR_ARG, "sma_mlp_forward_device: n must be below 2^31");
  if (n == 0) return SMA_OK;
  int ncu = 256;
  if (int rc = infer_lds(&ncu)) return rc;
  const int64_t nblk = (n + 15) / 16;   // the smallest row blocks
  const unsigned grid = (unsigned)std::min<int64_t>(nblk, ncu);
  hipLaunchKernelGGL(mlp::mlp_infer, dim3(grid), dim3(mlp::INF_THREADS), mlp::INF_SMEM, (hipStream_t)stream, m->Wi,
                     m->bp, X, n, (const unsigned*)nullptr, (int64_t)0, Y);
  SCHK(hipGetLastError());
  return SMA_OK;
}

int sma_mlp_grad_device(sma_mlp* m, int64_t n, const float* X, const float* T, float* gW, float* gb,
                        float* loss_out, void* stream) {
  if (!m || n <= 0 || !X || !T || !gW || !gb) return sma_abi::fail(SMA_ERR_ARG, "sma_mlp_grad_device: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  int parts = 0;
  if (int rc = train_pass(m, n, X, T, &parts, s)) return rc;
  mlp::AdamArgs A = adam_args(m, parts);
  A.gW = gW;
  A.gb = gb;
  if (int rc = reduce(A, s)) return rc;
  return loss_out ? mean_loss(m, n, parts, loss_out, s) : SMA_OK;
}

int sma_mlp_train_step_device(sma_mlp* m, int64_t n, const float* X, const float* T, double lr,
                              float* loss_out, void* stream) {
  if (!m || n <= 0 || !X || !T) return sma_abi::fail(SMA_ERR_ARG, "sma_mlp_train_step_device: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  int parts = 0;
  if (int rc = train_pass(m, n, X, T, &parts, s)) return rc;
  m->step += 1;
  mlp::AdamArgs A = adam_args(m, parts);
  A.W = m->W;
  A.b = m->b;
  A.mW = m->mW;
  A.vW = m->vW;
  A.mb = m->mb;
  A.vb = m->vb;
  A.Wp = m->Wp;
  A.bp = m->bp;
  A.Wi = m->Wi;
  A.Wt = m->Wt;
  A.lr = (float)lr;
  A.beta1 = 0.9f;
  A.beta2 = 0.999f;
  A.eps = 1e-8f;
  A.bc1 = (float)(1.0 - std::pow(0.9, (double)m->step));
  A.bc2 = (float)(1.0 - std::pow(0.999, (double)m->step));
  if (int rc = reduce(A, s)) return rc;
  return loss_out ? mean_loss(m, n, parts, loss_out, s) : SMA_OK;
}

int sma_mlp_gen_samples_device(int64_t n, uint64_t seed, const double* props_dev, double strain_sd,
                               double step_sd, double jitter, float* X, float* T, uint32_t* flags,
                               void* stream) {
  if (n < 0 || (n > 0 && (!props_dev || !X || !T || !flags)))
    return sma_abi::fail(SMA_ERR_ARG, "sma_mlp_gen_samples_device: bad arguments");
  if (n == 0) return SMA_OK;
  mlp::GenArgs G{n, seed, props_dev, strain_sd, step_sd, jitter, X, T, flags};
  hipLaunchKernelGGL(mlp::gen_samples, dim3(nb(n, 256)), dim3(256), 0, (hipStream_t)stream, G);
  SCHK(hipGetLastError());
  return SMA_OK;
}

}  // extern "C"

// Internal: inference over the step's list of points (its segment counters
// are read on the device; seg_cap slots per segment).
int sma_mlp_infer_listed(sma_mlp* m, const float* X, const unsigned* seg_count, int64_t seg_cap,
                         float* Y, hipStream_t s) {
  int ncu = 256;
  if (int rc = infer_lds(&ncu)) return rc;
  const int64_t cap = seg_cap * mlp::LIST_SEGS;
  const unsigned grid =
      (unsigned)std::max<int64_t>(1, std::min<int64_t>((cap + 15) / 16, ncu));
  hipLaunchKernelGGL(mlp::mlp_infer, dim3(grid), dim3(mlp::INF_THREADS), mlp::INF_SMEM, s, m->Wi, m->bp, X,
                     (int64_t)0, seg_count, seg_cap, Y);
  SCHK(hipGetLastError());
  return 0;
}
