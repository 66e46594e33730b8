// Learned closure: a 5 -> 64 -> 64 -> 1 tanh MLP mapping local flow features
// to the SA production multiplier beta = 1 + MLP(features).
//
// One kernel runs the forward pass and, for training, the backward pass and
// the parameter gradients; everything between the features and the per-block
// gradient sums stays in registers and LDS.  The three 64 x 64 products run on
// the matrix cores: BF16 operands, FP32 accumulation
// (v_mfma_f32_16x16x32_bf16; fragment layout, lane l of the wave:
// A[l%16][8(l/16)+t], B[8(l/16)+t][l%16], C[4(l/16)+i][l%16]).  The 5 -> 64 and
// 64 -> 1 layers, activations, loss, Adam and every reduction are FP32;
// reductions use fixed orders, so training is bitwise reproducible.
// Parameters (FP32 master copy, 4609 floats):
//   W1[64][5] | b1[64] | W2[64][64] | b2[64] | W3[64] | b3
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sg_closure.hpp"
#include "sg_mlp.hpp"

namespace sg {

// ---- the network on 32 rows per wave ----------------------------------------
//
// A wave takes 32 rows as two sub-tiles of 16, row r of a sub-tile on the four
// lanes l with l % 16 = r.  Those hold the hidden units u = 16 a + 4 q + i
// (q = l / 16; a, i = 0..3), 16 each: the layout in which the matrix cores
// return a product whose columns are rows of the batch (C[unit][row]).  With
// the summation index of the next product enumerated as
//   slot (s, q, t) -> unit 32 s + 16 (t / 4) + 4 q + t % 4
// the same registers are its B operand, so layer 1 is computed in place, layer
// 2 follows from it, and the backward product dH2 W2 from layer 2, without any
// exchange between lanes; only W2 is read in that order (rows of W2b forward,
// of its transpose backward).  The weight gradient dH2^T H1 sums over rows:
// its operands go through LDS once, the two sub-tiles of a lane's row
// together (4 bytes), which enumerates the rows as 2 (l % 16) + sub-tile for
// both operands alike.  (Four sub-tiles at a time spilled 105 registers: a lane
// keeps 192 gradient sums.)
//
// What bounds it: a launch of 65,536 rows gives every SIMD one wave with two
// tiles of 32 rows, 5 us each (its tanh, 4 k cycles, and the latencies of one
// wave alone), after 14 us for the weights, the gathers and the block's
// gradient sums.  Against eleven kernels that passed every activation through
// memory, a training step of 65,536 rows (forward, backward, Adam) takes 24 +
// 5 us instead of 565.
constexpr int SUB = 2, MLP_ROWS = 16 * SUB, MLP_WAVES = 4;  // sub-tiles and rows per wave, waves per block
constexpr int kTld = 40;                     // LDS row stride (BF16) of the row-summed operands
constexpr int kRld = 68;                     // LDS row stride (float) of the lane-summed values

struct MlpLds {
  float w1[MLP_H][8];  // W1 row, b1
  float b2[MLP_H], w3[MLP_H];
  union {
    __bf16 t[MLP_WAVES][2][MLP_H][kTld];  // dH2 and H1, [unit][row]
    float red[MLP_WAVES][MLP_H][kRld];    // gradient sums
  };
  float tail[MLP_WAVES][2];  // sums of e^2 and dy
};

template <bool BWD>
__global__ __launch_bounds__(64 * MLP_WAVES) __attribute__((amdgpu_waves_per_eu(1, 1))) void mlp_kernel(
    int n, const float* __restrict__ X, const int* __restrict__ idx, const float* __restrict__ T,
    const float* __restrict__ P, const __bf16* __restrict__ W2b, const __bf16* __restrict__ W2t, float inv_ntot,
    float* __restrict__ Y, float* __restrict__ part) {
  __shared__ MlpLds sh;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, q = lane >> 4, r16 = lane & 15;
  for (int e = tid; e < MLP_H * 8; e += 64 * MLP_WAVES) {
    const int u = e >> 3, c = e & 7;
    sh.w1[u][c] = c < MLP_IN ? P[MLP_W1 + u * MLP_IN + c] : c == MLP_IN ? P[MLP_B1 + u] : 0.f;
  }
  if (tid < MLP_H) {
    sh.b2[tid] = P[MLP_B2 + tid];
    sh.w3[tid] = P[MLP_W3 + tid];
  }
  __syncthreads();
  const float b3 = P[MLP_B3];
  // fragment of a 64 x 64 matrix M (row-major): rows 16 a + l % 16, slots of s
  auto frag = [&](const __bf16* M, int a, int s) {
    const __bf16* p = M + (16 * a + r16) * MLP_H + 32 * s + 4 * q;
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    const bf16x4 lo = *reinterpret_cast<const bf16x4*>(p), hi = *reinterpret_cast<const bf16x4*>(p + 16);
    bf16x8 f;
#pragma unroll
    for (int t = 0; t < 4; ++t) { f[t] = lo[t]; f[t + 4] = hi[t]; }
    return f;
  };
  // gradient sums of this lane's units over its rows, and of the wave's dW2
  float gw1[16][MLP_IN], gb1[16], gb2[16], gw3[16], se = 0.f, sdy = 0.f;
  f32x4 gw2[4][4];
  if (BWD) {
#pragma unroll
    for (int u = 0; u < 16; ++u) {
#pragma unroll
      for (int c = 0; c < MLP_IN; ++c) gw1[u][c] = 0.f;
      gb1[u] = gb2[u] = gw3[u] = 0.f;
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) gw2[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int tiles = (n + MLP_ROWS - 1) / MLP_ROWS, stride = gridDim.x * MLP_WAVES;
  for (int tile = blockIdx.x * MLP_WAVES + w; tile < tiles; tile += stride) {
    float x[SUB][MLP_IN], tt[SUB], h1[SUB][16];
    bool live[SUB];
    int src[SUB];
#pragma unroll
    for (int m = 0; m < SUB; ++m) {
      const int r = tile * MLP_ROWS + 16 * m + r16;
      live[m] = r < n;
      src[m] = live[m] ? (idx ? idx[r] : r) : 0;
    }
#pragma unroll
    for (int m = 0; m < SUB; ++m) {
#pragma unroll
      for (int c = 0; c < MLP_IN; ++c) x[m][c] = live[m] ? X[(long)src[m] * MLP_IN + c] : 0.f;
      if (BWD) tt[m] = live[m] ? T[src[m]] : 0.f;
    }
    // layer 1
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const float* w1 = sh.w1[16 * (u >> 2) + 4 * q + (u & 3)];
      float a[SUB];
#pragma unroll
      for (int m = 0; m < SUB; ++m) a[m] = w1[MLP_IN];
#pragma unroll
      for (int c = 0; c < MLP_IN; ++c)
#pragma unroll
        for (int m = 0; m < SUB; ++m) a[m] = fmaf(w1[c], x[m][c], a[m]);
#pragma unroll
      for (int m = 0; m < SUB; ++m) h1[m][u] = tanh_fast(a[m]);
    }
    // layer 2, output, loss and dH2, a sub-tile at a time
    bf16x8 hb[SUB][2], db[SUB][2];
#pragma unroll
    for (int m = 0; m < SUB; ++m) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < 8; ++t) hb[m][s][t] = (__bf16)h1[m][8 * s + t];
      float h2[16], y = 0.f;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 2; ++s) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(W2b, a, s), hb[m][s], c, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int u = 16 * a + 4 * q + i;
          h2[4 * a + i] = tanh_fast(c[i] + sh.b2[u]);
          y = fmaf(sh.w3[u], h2[4 * a + i], y);
        }
      }
      y += __shfl_xor(y, 16);
      y += __shfl_xor(y, 32);
      y += b3;
      if (Y && live[m] && q == 0) Y[tile * MLP_ROWS + 16 * m + r16] = y;
      if (BWD) {
        const float e = live[m] ? y - tt[m] : 0.f, dy = 2.f * e * inv_ntot;
        if (q == 0) {
          se = fmaf(e, e, se);
          sdy += dy;
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const float d = dy * sh.w3[16 * (u >> 2) + 4 * q + (u & 3)] * (1.f - h2[u] * h2[u]);
          gb2[u] += d;
          gw3[u] = fmaf(dy, h2[u], gw3[u]);
          db[m][u >> 3][u & 7] = (__bf16)d;
        }
      }
    }
    if constexpr (BWD) {
      // dH1 = (dH2 W2) (1 - h1^2) and the sums it enters
#pragma unroll
      for (int m = 0; m < SUB; ++m)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int s = 0; s < 2; ++s)
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(W2t, a, s), db[m][s], c, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int u = 4 * a + i;
            const float d = c[i] * (1.f - h1[m][u] * h1[m][u]);
            gb1[u] += d;
#pragma unroll
            for (int k = 0; k < MLP_IN; ++k) gw1[u][k] = fmaf(d, x[m][k], gw1[u][k]);
          }
        }
      // dW2[j][k] += sum over rows of dH2[row][j] H1[row][k]
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        bf16x2 d, h;
#pragma unroll
        for (int m = 0; m < SUB; ++m) { d[m] = db[m][u >> 3][u & 7]; h[m] = hb[m][u >> 3][u & 7]; }
        const int row = 16 * (u >> 2) + 4 * q + (u & 3);
        *reinterpret_cast<bf16x2*>(&sh.t[w][0][row][SUB * r16]) = d;
        *reinterpret_cast<bf16x2*>(&sh.t[w][1][row][SUB * r16]) = h;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
      {
        bf16x8 fd[4], fh[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          fd[a] = *reinterpret_cast<const bf16x8*>(&sh.t[w][0][16 * a + r16][8 * q]);
          fh[a] = *reinterpret_cast<const bf16x8*>(&sh.t[w][1][16 * a + r16][8 * q]);
        }
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int b = 0; b < 4; ++b)
            gw2[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fd[a], fh[b], gw2[a][b], 0, 0, 0);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
    }
  }
  if constexpr (BWD) {
    float* out = part + (size_t)blockIdx.x * MLP_NPART;
    // the lanes' sums over rows: 128 values per lane, 64 at a time, each summed
    // over the 16 lanes of its units and the waves by one thread
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      __syncthreads();
#pragma unroll
      for (int v = 0; v < 64; ++v) {
        const int e = 64 * half + v;  // gw1 (80), gb1, gb2, gw3 (16 each)
        const float g = e < 80 ? gw1[e / 5][e % 5] : e < 96 ? gb1[e - 80] : e < 112 ? gb2[e - 96] : gw3[e - 112];
        sh.red[w][v][lane] = g;
      }
      __syncthreads();
      const int v = tid & 63, g4 = tid >> 6;  // thread: value v of the units of lane group g4
      float s = 0.f;
#pragma unroll
      for (int ww = 0; ww < MLP_WAVES; ++ww)
#pragma unroll
        for (int l = 0; l < 16; ++l) s += sh.red[ww][v][16 * g4 + l];
      const int e = 64 * half + v;
      auto unit = [&](int u) { return 16 * (u >> 2) + 4 * g4 + (u & 3); };
      if (e < 80) out[MLP_W1 + unit(e / 5) * MLP_IN + e % 5] = s;
      else if (e < 96) out[MLP_B1 + unit(e - 80)] = s;
      else if (e < 112) out[MLP_B2 + unit(e - 96)] = s;
      else out[MLP_W3 + unit(e - 112)] = s;
    }
    // the waves' dW2
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) sh.red[w][16 * a + 4 * q + i][16 * b + r16] = gw2[a][b][i];
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      se += __shfl_xor(se, o);
      sdy += __shfl_xor(sdy, o);
    }
    if (lane == 0) {
      sh.tail[w][0] = sdy;
      sh.tail[w][1] = se;
    }
    __syncthreads();
    for (int e = tid; e < MLP_H * MLP_H; e += 64 * MLP_WAVES) {
      float s = 0.f;
#pragma unroll
      for (int ww = 0; ww < MLP_WAVES; ++ww) s += sh.red[ww][e >> 6][e & 63];
      out[MLP_W2 + e] = s;
    }
    if (tid < 2) {
      float s = 0.f;
#pragma unroll
      for (int ww = 0; ww < MLP_WAVES; ++ww) s += sh.tail[ww][tid];
      out[MLP_B3 + tid] = s;  // db3, then the sum of e^2
    }
  }
}

// grad[p] = sum over the blocks' partials (fixed order: slices of blocks, then
// the slices), the loss from the entry after the parameters; with ADAM the
// step (Kingma & Ba 2015) on the FP32 master parameters and the BF16 copies of
// W2 that the matrix cores read.
constexpr int RED_P = 32, RED_S = 16;  // parameters per block, slices
template <bool ADAM>
__global__ __launch_bounds__(RED_P* RED_S) void mlp_reduce_kernel(int nblk, const float* __restrict__ part,
                                                                  float* __restrict__ grad, float loss_scale,
                                                                  float* __restrict__ loss, float* P, float* m,
                                                                  float* v, float lr, float b1, float b2, float eps,
                                                                  float c1, float c2, __bf16* W2b, __bf16* W2t) {
  __shared__ float red[RED_S][RED_P];
  const int p = blockIdx.x * RED_P + threadIdx.x % RED_P, s = threadIdx.x / RED_P;
  float a = 0.f;
  if (p < MLP_NPART) {
    const int per = (nblk + RED_S - 1) / RED_S, e = min(nblk, (s + 1) * per);
    int b = s * per;
    for (; b + 4 <= e; b += 4) {
      float u[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) u[k] = part[(size_t)(b + k) * MLP_NPART + p];
#pragma unroll
      for (int k = 0; k < 4; ++k) a += u[k];
    }
    for (; b < e; ++b) a += part[(size_t)b * MLP_NPART + p];
  }
  red[s][threadIdx.x % RED_P] = a;
  __syncthreads();
  if (s != 0 || p >= MLP_NPART) return;
  float g = 0.f;
#pragma unroll
  for (int k = 0; k < RED_S; ++k) g += red[k][threadIdx.x];
  if (p == MLP_NPARAM) {
    *loss = g * loss_scale;
    return;
  }
  if (grad) grad[p] = g;
  if (ADAM) {
    const float mp = b1 * m[p] + (1.f - b1) * g;
    const float vp = b2 * v[p] + (1.f - b2) * g * g;
    m[p] = mp;
    v[p] = vp;
    const float w = P[p] - lr * (mp / c1) / (sqrtf(vp / c2) + eps);
    P[p] = w;
    if (p >= MLP_W2 && p < MLP_B2) {
      const int e = p - MLP_W2;
      W2b[e] = (__bf16)w;
      W2t[(e & 63) * MLP_H + (e >> 6)] = (__bf16)w;
    }
  }
}

// BF16 copy of W2, and (if W2t) of its transpose
__global__ void mlp_w2_to_bf16_kernel(const float* P, __bf16* W2b, __bf16* W2t) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= MLP_H * MLP_H) return;
  const __bf16 w = (__bf16)P[MLP_W2 + e];
  W2b[e] = w;
  if (W2t) W2t[(e & 63) * MLP_H + (e >> 6)] = w;
}

// ---- the epoch's shuffle ------------------------------------------------------
// Fisher-Yates from k = n - 1 down to 1, swapping places k and j_k = draw % (k +
// 1), with all steps at once.  Write c(k) for what place k holds just before
// step k: if steps k' > k drew k, the last of them (the smallest) left what
// place k' held then, c(k'), else place k still holds k.  Step k leaves in
// place k what place j_k held: c(k) if j_k = k, else c of the smallest k' > k
// that drew j_k too, else j_k.  The draws are the counter-based splitmix64
// stream (Steele, Lea & Flood 2014), so step k of epoch e is one evaluation.
// The steps that drew a place form a linked list in any order; only its
// smallest member past k is used, so the result does not depend on the order.
// On the host a shuffle of 147,456 took 430 us, twenty times the kernels of a
// minibatch.
__device__ __forceinline__ unsigned long long splitmix(unsigned long long z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ int next_step(const int* head, const int* link, int place, int k) {
  int best = -1;
  for (int s = head[place]; s >= 0; s = link[s])
    if (s > k && (best < 0 || s < best)) best = s;
  return best;
}
__global__ __launch_bounds__(256) void mlp_fill_kernel(size_t n, int* a, int v) {
  const size_t k = blockIdx.x * (size_t)256 + threadIdx.x;
  if (k < n) a[k] = v;
}
__global__ __launch_bounds__(256) void mlp_draw_kernel(int n, unsigned long long seed, unsigned long long first,
                                                       int* draw, int* head, int* link) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k < 1 || k >= n) return;
  const unsigned long long t = first + (unsigned long long)(n - k);  // draws so far, this one included
  const int j = (int)(splitmix(seed + t * 0x9E3779B97F4A7C15ull) % (unsigned long long)(k + 1));
  draw[k] = j;
  link[k] = atomicExch(&head[j], k);
}
__global__ __launch_bounds__(256) void mlp_held_kernel(int n, const int* head, const int* link, int* up, int* clear) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  up[k] = next_step(head, link, k, k);
  clear[k] = -1;  // the next epoch's lists
}
__global__ __launch_bounds__(256) void mlp_shuffle_kernel(int n, const int* draw, const int* head, const int* link,
                                                          const int* up, int* perm) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  int s = k;
  if (k > 0 && draw[k] != k) {
    s = next_step(head, link, draw[k], k);
    if (s < 0) {
      perm[k] = draw[k];
      return;
    }
  }
  for (int u = up[s]; u >= 0; u = up[s]) s = u;
  perm[k] = s;
}

// ---- host-side drivers ------------------------------------------------------
hipError_t mlp_w2_to_bf16(const float* P, __bf16* W2b, __bf16* W2t, hipStream_t s) {
  hipLaunchKernelGGL(mlp_w2_to_bf16_kernel, dim3((MLP_H * MLP_H + 255) / 256), dim3(256), 0, s, P, W2b, W2t);
  return hipGetLastError();
}

// blocks of a pass over n rows: one tile per wave while that does not exceed
// one block per CU, then the waves take several (each block's sums cost 18 KB
// of partials, which the reduction reads back)
static int mlp_blocks(int n) {
  return std::min((n + MLP_ROWS * MLP_WAVES - 1) / (MLP_ROWS * MLP_WAVES), MLP_MAX_BLOCKS);
}

// perm = the epoch's permutation of n rows.  work: 5 n ints; the first 2 n hold
// the lists' heads of alternating epochs, -1 before epoch 0 (mlp_shuffle_init).
hipError_t mlp_shuffle_init(int n, int* work, hipStream_t s) {
  const size_t heads = 2 * (size_t)n;
  hipLaunchKernelGGL(mlp_fill_kernel, dim3((unsigned)((heads + 255) / 256)), dim3(256), 0, s, heads, work, -1);
  return hipGetLastError();
}
hipError_t mlp_shuffle(int n, unsigned long long seed, int epoch, int* work, int* perm, hipStream_t s) {
  int *head = work + (size_t)(epoch & 1) * n, *other = work + (size_t)(~epoch & 1) * n;
  int *draw = work + 2 * (size_t)n, *link = draw + n, *up = link + n;
  const dim3 grid((n + 255) / 256), block(256);
  hipLaunchKernelGGL(mlp_draw_kernel, grid, block, 0, s, n, seed,
                     (unsigned long long)epoch * (unsigned long long)(n - 1), draw, head, link);
  hipLaunchKernelGGL(mlp_held_kernel, grid, block, 0, s, n, head, link, up, other);
  hipLaunchKernelGGL(mlp_shuffle_kernel, grid, block, 0, s, n, draw, head, link, up, perm);
  return hipGetLastError();
}

hipError_t mlp_forward(const MlpWork& w, int n, const float* X, float* Y, hipStream_t s) {
  hipLaunchKernelGGL(mlp_kernel<false>, dim3(mlp_blocks(n)), dim3(64 * MLP_WAVES), 0, s, n, X, nullptr, nullptr, w.P,
                     w.W2b, w.W2t, 0.f, Y, nullptr);
  return hipGetLastError();
}

// Mean squared error over n rows (gathered by idx if given) and its gradient;
// with step > 0 the Adam step of that number as well.
hipError_t mlp_train_step(const MlpWork& w, int n, const float* X, const int* idx, const float* T, float* grad,
                          float* loss, int step, float lr, hipStream_t s) {
  const int nb = mlp_blocks(n);
  hipLaunchKernelGGL(mlp_kernel<true>, dim3(nb), dim3(64 * MLP_WAVES), 0, s, n, X, idx, T, w.P, w.W2b, w.W2t,
                     1.0f / (float)n, nullptr, w.part);
  const dim3 grid((MLP_NPART + RED_P - 1) / RED_P), block(RED_P * RED_S);
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  if (step > 0) {
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(mlp_reduce_kernel<true>, grid, block, 0, s, nb, w.part, grad, 1.0f / (float)n, loss, w.P, w.m,
                       w.v, lr, b1, b2, eps, c1, c2, w.W2b, w.W2t);
  } else {
    hipLaunchKernelGGL(mlp_reduce_kernel<false>, grid, block, 0, s, nb, w.part, grad, 1.0f / (float)n, loss, w.P, w.m,
                       w.v, lr, b1, b2, eps, 1.f, 1.f, w.W2b, w.W2t);
  }
  return hipGetLastError();
}

}  // namespace sg
