// Learned SA closure: a 5 -> 64 -> 64 -> 1 tanh MLP (see sg_mlp.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace sg {

constexpr int MLP_IN = 5;
constexpr int MLP_H = 64;
// parameter offsets in the packed FP32 vector
constexpr int MLP_W1 = 0;
constexpr int MLP_B1 = MLP_W1 + MLP_H * MLP_IN;  // 320
constexpr int MLP_W2 = MLP_B1 + MLP_H;           // 384
constexpr int MLP_B2 = MLP_W2 + MLP_H * MLP_H;   // 4480
constexpr int MLP_W3 = MLP_B2 + MLP_H;           // 4544
constexpr int MLP_B3 = MLP_W3 + MLP_H;           // 4608
constexpr int MLP_NPARAM = MLP_B3 + 1;           // 4609

// a block's gradient sums: the parameters, then the sum of squared errors
constexpr int MLP_NPART = MLP_NPARAM + 1;
constexpr int MLP_MAX_BLOCKS = 256;              // of one pass

// Device work space of one network (all pointers device memory).
struct MlpWork {
  float* P = nullptr;      // FP32 master parameters
  float* m = nullptr;      // Adam first moment
  float* v = nullptr;      // Adam second moment
  float* grad = nullptr;   // last gradient
  __bf16* W2b = nullptr;   // BF16 copy of W2 used by the matrix cores
  __bf16* W2t = nullptr;   // and of its transpose
  int cap = 0;             // rows of one forward/backward pass
  float *part = nullptr, *loss = nullptr;  // MLP_MAX_BLOCKS x MLP_NPART gradient sums; the last loss
};

hipError_t mlp_w2_to_bf16(const float* P, __bf16* W2b, __bf16* W2t, hipStream_t s);
hipError_t mlp_forward(const MlpWork& w, int n, const float* X, float* Y, hipStream_t s);
hipError_t mlp_shuffle_init(int n, int* work, hipStream_t s);
hipError_t mlp_shuffle(int n, unsigned long long seed, int epoch, int* work, int* perm, hipStream_t s);
hipError_t mlp_train_step(const MlpWork& w, int n, const float* X, const int* idx, const float* T, float* grad,
                          float* loss, int step, float lr, hipStream_t s);

}  // namespace sg
