// Device linear algebra used by the Newton-Krylov driver (sg_linalg.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

#include "sg_device.hpp"

namespace sg {

constexpr int NSLOT = 13;  // Jacobian stencil blocks kept per cell

// 64-bit words of the slots of the reductions below, which every call finds and
// leaves empty; reduce_slots_init writes their head and empties them first.
size_t reduce_slots(int kmax);
struct Slots {
  double* p;
  int polls;  // bound of a wait on them
};
hipError_t reduce_slots_init(double* slots, size_t n, hipStream_t s, int polls = kWaitPolls);
// out[i] = V_i . w for i < k (V_i = V + i*ldv); out is device memory.  With
// ga and gb (device doubles) the kernel runs only if *ga < gf * *gb and
// otherwise writes nothing: a conditional pass decided on the device.
hipError_t multi_dot(const double* V, size_t ldv, int k, const double* w, size_t n, Slots slots, double* out,
                     hipStream_t s, const double* ga = nullptr, const double* gb = nullptr, double gf = 0.5);
// w -= sum_i c[i] V_i, c device memory, and *norm2 = |w|^2 after it; gated as
// multi_dot
hipError_t multi_axpy(const double* V, size_t ldv, int k, const double* c, double* w, size_t n, Slots slots,
                      double* norm2, hipStream_t s, const double* ga = nullptr, const double* gb = nullptr,
                      double gf = 0.5);
// The end of an Arnoldi step j: h[0..j+1] = V^T w and |w|^2, y[j+1] = |w'|^2
// after the projection; if y[j+1] < gf h[j+1] a second one ran, with y[0..j]
// its projections and *norm2b the norm after it.  Scales w to unit norm (a
// zero w stays) and leaves in res (host memory the device can write, preset to
// kNoValue) the column's entries 0..j, then the norm and whether the second
// pass ran (1 or 0; NaN if |w|^2 is), each as one 64-bit store.
hipError_t arnoldi_finish(double* w, size_t n, int j, const double* h, const double* y, const double* norm2b, double gf,
                          double* res, hipStream_t s);
// y (+)= sum_i c[i] X_i, c device memory
hipError_t lincomb(const double* X, size_t ldx, int k, const double* c_dev, double* y, size_t n, bool accumulate,
                   hipStream_t s);
hipError_t axpby(double a, const double* x, double b, double* y, size_t n, hipStream_t s);
hipError_t zero_fill(double* x, size_t n, hipStream_t s);
hipError_t line_factor(int nic, int njc, int ldi, int nv, const double* idt, const double* blocks, double* fac,
                       bool jacobi, hipStream_t s);
hipError_t line_solve(int nic, int njc, int ldi, int nv, const double* fac, const double* b, double* x, hipStream_t s);
// symmetric multicolour line Gauss-Seidel colour step (see sg_linalg.hip)
hipError_t line_gs(int nic, int njc, int ldi, int nv, int colour, const double* blocks, const double* fac,
                   const double* bvec, double* t, double* x, hipStream_t s);
// multicolour (5 colours) block ILU(0) of I/dt - J on the 13-point stencil
hipError_t ilu_factor(int nic, int njc, int ldi, int nv, const double* idt, const double* blocks, double* ilu,
                      hipStream_t s);
hipError_t ilu_apply(int nic, int njc, int ldi, int nv, const double* ilu, const double* b, double* z, hipStream_t s);
// level-scheduled block ILU(0) of I/dt - J in natural j-major order (one
// persistent work-group); apply with transpose = true solves with (LU)^T
hipError_t lilu_factor(int nic, int njc, int ldi, int nv, const double* idt, const double* blocks, double* ilu,
                       hipStream_t s);
hipError_t lilu_apply(int nic, int njc, int ldi, int nv, const double* ilu, const double* b, double* z, bool transpose,
                      hipStream_t s);
// chunked line block ILU(0) (sg_cilu.hip): chunks of w in {8, 16, 24, 32}
// columns, on the 13-point stencil or (nine) the 3x3-box pattern; cilu_size
// is the storage in doubles that cilu_factor writes and cilu_apply reads: the
// links between column groups with their SlotHead (empty between applies), the
// FP32 factors in the order of M^-1 and of M^-T, and the factorisation's operands
// gathered in level order.  apart (the same in all three): the apply takes a
// launch per pass, for a device on which not every CU takes part; polls bounds
// the apply's waits on the links
bool cilu_width_ok(int w);
size_t cilu_size(int nic, int njc, int nv, int w, bool nine, bool apart);
hipError_t cilu_factor(int nic, int njc, int ldi, int nv, int w, bool nine, bool apart, const double* idt,
                       const double* blocks, double* rec, hipStream_t s);
hipError_t cilu_apply(int nic, int njc, int ldi, int nv, int w, bool nine, double* store, const double* b, double* z,
                      bool transpose, bool apart, int polls, hipStream_t s);
// adjoint helpers: J^T psi from the blocks, or with idt psi idt - J^T psi
hipError_t jt_gather(int nic, int njc, int ldi, int nv, const double* blocks, const double* psi, double* out,
                     hipStream_t s, const double* idt = nullptr);
hipError_t dbeta_apply(int nic, int njc, int ldi, const double* psi, const double* diag, double* out, hipStream_t s);
hipError_t ilu_apply_t(int nic, int njc, int ldi, int nv, const double* ilu, const double* b, double* z, hipStream_t s);
// per-block minima of the admissible update fraction (see sg_linalg.hip)
hipError_t update_limit(int nic, int njc, int ldi, const double* q, const double* dq, double f, double* block_min,
                        int nblocks, hipStream_t s);
hipError_t invert_dt(const double* dt, double* idt, int nic, int njc, int ldi, hipStream_t s);

}  // namespace sg
