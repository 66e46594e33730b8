// C ABI of the closure network: creation (seeded Glorot-uniform weights),
// parameter I/O, batched inference, loss + gradient, and Adam training over
// device-resident samples.  Kernels are in sg_mlp.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "sg_context.hpp"
#include "sg_mlp.hpp"

using namespace sg;

struct sg_mlp {
  MlpWork w;
  hipStream_t stream = nullptr;
  std::string err;
  std::vector<void*> allocs;
  int step = 0;                 // Adam step counter (bias correction)
  float* Y = nullptr;           // forward output staging [cap]
  float* Xd = nullptr;          // staged inputs [cap][5] / targets [cap]
  float* Td = nullptr;
  float* set = nullptr;         // sg_mlp_train: samples, losses, permutation
  size_t set_words = 0;
};

namespace {

int mlp_fail(sg_mlp* n, int code, const std::string& msg) {
  if (n) n->err = msg;
  return code;
}

#define MLP_TRY(expr, what)                                                            \
  do {                                                                                 \
    hipError_t e_ = (expr);                                                            \
    if (e_ != hipSuccess) return mlp_fail(net, SG_ERR_HIP, std::string(what) + ": " + \
                                                                  hipGetErrorString(e_)); \
  } while (0)

template <class T>
hipError_t dalloc(sg_mlp* net, T*& p, size_t count) {
  void* v = nullptr;
  hipError_t e = hipMalloc(&v, std::max<size_t>(count, 1) * sizeof(T));
  if (e == hipSuccess) {
    net->allocs.push_back(v);
    p = static_cast<T*>(v);
  }
  return e;
}

// splitmix64 (Steele, Lea & Flood 2014): seeded, platform-independent stream.
struct SplitMix {
  unsigned long long s;
  unsigned long long next() {
    unsigned long long z = (s += 0x9E3779B97F4A7C15ULL);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
  }
  double uniform() { return (double)(next() >> 11) * (1.0 / 9007199254740992.0); }
};

void glorot(std::vector<float>& p, unsigned long long seed) {
  SplitMix r{seed};
  std::fill(p.begin(), p.end(), 0.0f);
  auto fill = [&](int off, int fan_out, int fan_in) {
    const double lim = std::sqrt(6.0 / (fan_in + fan_out));
    for (int k = 0; k < fan_out * fan_in; ++k) p[off + k] = (float)((2.0 * r.uniform() - 1.0) * lim);
  };
  fill(MLP_W1, MLP_H, MLP_IN);
  fill(MLP_W2, MLP_H, MLP_H);
  fill(MLP_W3, 1, MLP_H);
}

}  // namespace

int sg_mlp_create(sg_mlp** out, int max_rows, unsigned long long seed) {
  if (!out || max_rows <= 0) return SG_ERR_ARG;
  *out = nullptr;
  sg_mlp* net = new sg_mlp();
  auto fail = [&](int code) {
    sg_mlp_destroy(net);
    return code;
  };
  if (hipStreamCreate(&net->stream) != hipSuccess) return fail(SG_ERR_HIP);
  MlpWork& w = net->w;
  const size_t cap = (size_t)max_rows;
  w.cap = max_rows;
  if (dalloc(net, w.P, MLP_NPARAM) || dalloc(net, w.m, MLP_NPARAM) || dalloc(net, w.v, MLP_NPARAM) ||
      dalloc(net, w.grad, MLP_NPARAM) || dalloc(net, w.W2b, MLP_H * MLP_H) || dalloc(net, w.W2t, MLP_H * MLP_H) ||
      dalloc(net, w.part, (size_t)MLP_MAX_BLOCKS * MLP_NPART) || dalloc(net, w.loss, 1) || dalloc(net, net->Y, cap) ||
      dalloc(net, net->Xd, cap * MLP_IN) || dalloc(net, net->Td, cap))
    return fail(SG_ERR_HIP);
  std::vector<float> p(MLP_NPARAM);
  glorot(p, seed);
  int rc = sg_mlp_set_params(net, p.data());
  if (rc) return fail(rc);
  *out = net;
  return SG_OK;
}

void sg_mlp_destroy(sg_mlp* net) {
  if (!net) return;
  if (net->stream) (void)hipStreamSynchronize(net->stream);
  for (void* p : net->allocs) (void)hipFree(p);
  if (net->set) (void)hipFree(net->set);
  if (net->stream) (void)hipStreamDestroy(net->stream);
  delete net;
}

const char* sg_mlp_last_error(const sg_mlp* net) { return net ? net->err.c_str() : "null network"; }

// New parameters also reset the Adam state.
int sg_mlp_set_params(sg_mlp* net, const float* params) {
  if (!net || !params) return SG_ERR_ARG;
  MlpWork& w = net->w;
  MLP_TRY(hipMemcpyAsync(w.P, params, MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice, net->stream), "H2D");
  MLP_TRY(hipMemsetAsync(w.m, 0, MLP_NPARAM * sizeof(float), net->stream), "memset");
  MLP_TRY(hipMemsetAsync(w.v, 0, MLP_NPARAM * sizeof(float), net->stream), "memset");
  MLP_TRY(mlp_w2_to_bf16(w.P, w.W2b, w.W2t, net->stream), "w2 bf16");
  MLP_TRY(hipStreamSynchronize(net->stream), "set params");
  net->step = 0;
  return SG_OK;
}

int sg_mlp_get_params(sg_mlp* net, float* params) {
  if (!net || !params) return SG_ERR_ARG;
  MLP_TRY(hipMemcpyAsync(params, net->w.P, MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost, net->stream), "D2H");
  MLP_TRY(hipStreamSynchronize(net->stream), "get params");
  return SG_OK;
}

int sg_mlp_forward(sg_mlp* net, int n, const float* x, float* y) {
  if (!net || n < 0 || (n > 0 && (!x || !y))) return SG_ERR_ARG;
  const int cap = net->w.cap;
  for (int r0 = 0; r0 < n; r0 += cap) {
    const int m = std::min(cap, n - r0);
    MLP_TRY(hipMemcpyAsync(net->Xd, x + (size_t)r0 * MLP_IN, (size_t)m * MLP_IN * sizeof(float),
                           hipMemcpyHostToDevice, net->stream), "H2D");
    MLP_TRY(mlp_forward(net->w, m, net->Xd, net->Y, net->stream), "forward");
    MLP_TRY(hipMemcpyAsync(y + r0, net->Y, (size_t)m * sizeof(float), hipMemcpyDeviceToHost, net->stream), "D2H");
  }
  MLP_TRY(hipStreamSynchronize(net->stream), "forward");
  return SG_OK;
}

int sg_mlp_loss_grad(sg_mlp* net, int n, const float* x, const float* t, float* loss, float* grad) {
  if (!net || n <= 0 || !x || !t) return SG_ERR_ARG;
  if (n > net->w.cap) return mlp_fail(net, SG_ERR_ARG, "more rows than the network was created for");
  MLP_TRY(hipMemcpyAsync(net->Xd, x, (size_t)n * MLP_IN * sizeof(float), hipMemcpyHostToDevice, net->stream), "H2D");
  MLP_TRY(hipMemcpyAsync(net->Td, t, (size_t)n * sizeof(float), hipMemcpyHostToDevice, net->stream), "H2D");
  MLP_TRY(mlp_train_step(net->w, n, net->Xd, nullptr, net->Td, net->w.grad, net->w.loss, 0, 0.f, net->stream),
          "loss/grad");
  float l = 0.f;
  MLP_TRY(hipMemcpyAsync(&l, net->w.loss, sizeof(float), hipMemcpyDeviceToHost, net->stream), "D2H");
  if (grad)
    MLP_TRY(hipMemcpyAsync(grad, net->w.grad, MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost, net->stream), "D2H");
  MLP_TRY(hipStreamSynchronize(net->stream), "loss/grad");
  if (loss) *loss = l;
  return SG_OK;
}

int sg_mlp_train(sg_mlp* net, int n, const float* x, const float* t, int epochs, int batch, float lr,
                 unsigned long long seed, float* loss_hist) {
  if (!net || n <= 0 || !x || !t || epochs < 0 || batch <= 0 || !(lr > 0.f)) return SG_ERR_ARG;
  const int bs = std::min(batch, n);
  if (bs > net->w.cap) return mlp_fail(net, SG_ERR_ARG, "minibatch larger than the network was created for");
  const int nb = n / bs;
  // the training set stays allocated with the network, at its largest so far
  const size_t rows = (size_t)n, need = rows * (MLP_IN + 1 + 1 + 5) + (size_t)std::max(1, epochs) * nb;
  if (need > net->set_words) {
    if (net->set) {
      MLP_TRY(hipStreamSynchronize(net->stream), "training set");
      (void)hipFree(net->set);
      net->set = nullptr;
      net->set_words = 0;
    }
    if (hipMalloc((void**)&net->set, need * sizeof(float)) != hipSuccess) {
      net->set = nullptr;
      return mlp_fail(net, SG_ERR_HIP, "hipMalloc of the training set failed");
    }
    net->set_words = need;
  }
  float *X = net->set, *T = X + rows * MLP_IN, *L = T + rows;
  int *perm = reinterpret_cast<int*>(L + (size_t)std::max(1, epochs) * nb), *work = perm + rows;
  MLP_TRY(hipMemcpyAsync(X, x, rows * MLP_IN * sizeof(float), hipMemcpyHostToDevice, net->stream), "H2D");
  MLP_TRY(hipMemcpyAsync(T, t, rows * sizeof(float), hipMemcpyHostToDevice, net->stream), "H2D");
  MLP_TRY(mlp_shuffle_init(n, work, net->stream), "shuffle");
  for (int e = 0; e < epochs; ++e) {
    MLP_TRY(mlp_shuffle(n, seed, e, work, perm, net->stream), "shuffle");
    for (int b = 0; b < nb; ++b) {
      ++net->step;
      MLP_TRY(mlp_train_step(net->w, bs, X, perm + (size_t)b * bs, T, net->w.grad, L + (size_t)e * nb + b, net->step,
                             lr, net->stream), "training step");
    }
  }
  std::vector<float> lh((size_t)std::max(1, epochs) * nb);
  if (epochs > 0)
    MLP_TRY(hipMemcpyAsync(lh.data(), L, lh.size() * sizeof(float), hipMemcpyDeviceToHost, net->stream), "D2H");
  MLP_TRY(hipStreamSynchronize(net->stream), "train");
  if (loss_hist)
    for (int e = 0; e < epochs; ++e) {
      double s = 0.0;
      for (int b = 0; b < nb; ++b) s += lh[(size_t)e * nb + b];
      loss_hist[e] = (float)(s / nb);
    }
  return SG_OK;
}

int sg_set_closure_mlp(sg_ctx* ctx, const sg_mlp* cnet) {
  if (!ctx || !cnet) return SG_ERR_ARG;
  sg_mlp* net = const_cast<sg_mlp*>(cnet);
  MLP_TRY(hipStreamSynchronize(net->stream), "network");
  std::vector<float> p(MLP_NPARAM);
  MLP_TRY(hipMemcpy(p.data(), net->w.P, MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost), "D2H");
  return sg_set_closure(ctx, SG_CLOSURE_MLP, nullptr, p.data());
}
