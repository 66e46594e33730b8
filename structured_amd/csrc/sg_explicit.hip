// Explicit pseudo-time stepping on the device: the build of Solver::step
// without ADOL-C (src/solver/solver.cpp:103-121) and the loop of
// Solver::solve (:197-236).
//
// A Runge-Kutta stage is one launch: the residual kernel writes the stage's
// state instead of R, with the cell's local time step recomputed from the
// step's base state (the reference computes dt once per step from q, calc_dt,
// before the stages).  Only the last stage's norms are formed, the others are
// never seen.  Forward Euler updates the residual's own input, so its update
// is a kernel of its own, which moves q (nv) + R (nv) + the shorter face length
// in and nv values out.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>

#include "sg_context.hpp"
#include "sg_kernels.hpp"

using namespace sg;

#define SG_TRY(expr, what)                         \
  do {                                             \
    int rc_ = sg_hip(ctx, (expr), what);           \
    if (rc_ != SG_OK) return rc_;                  \
  } while (0)

namespace {

// q += R dt with dt = calc_dt(q) of the cell: update_forward_euler,
// src/solver/solver.cpp:12-18.
__global__ __launch_bounds__(256) void forward_euler_kernel(DevGeom g, int nv, double* q, const double* R,
                                                            const double* dsmin, double mu_inf, double cfl) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (i >= g.nic) return;
  const size_t c = (size_t)j * g.ldi + i;
  double qv[5], rv[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    if (k < nv) { qv[k] = q[k * g.plane + c]; rv[k] = R[k * g.plane + c]; }
  }
  const double dt = cell_dt(qv[0], qv[1], qv[2], qv[3], dsmin[c], mu_inf, cfl);
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    if (k < nv) {
#pragma clang fp contract(off)
      q[k * g.plane + c] = qv[k] + rv[k] * dt;
    }
  }
}

// The residual of forward Euler, or the two stage states of RK4.
int ensure_buffers(sg_ctx* ctx, int scheme) {
  const size_t n = ctx->nsoa();
  const bool euler = scheme == SG_SCHEME_FORWARD_EULER;
  for (DevBuf* b : {euler ? &ctx->ex_r : &ctx->ex_a, euler ? &ctx->ex_r : &ctx->ex_b})
    if (b->n != n) SG_TRY(b->alloc(n), "explicit work buffers");
  return SG_OK;
}

// Enqueues one step; the norms of the last stage's residual land in ctx->l2.
int enqueue_step(sg_ctx* ctx, double* q, int scheme, double cfl) {
  const DevGeom& g = ctx->g;
  if (scheme == SG_SCHEME_FORWARD_EULER) {
    double* R = ctx->ex_r.p;
    SG_TRY(launch_residual(g, ctx->ph, ctx->bc, ctx->sa, q, R, ctx->partial.p, ctx->l2.p, ctx->stream, ctx->clo,
                           ctx->nvar),
           "residual");
    hipLaunchKernelGGL(forward_euler_kernel, dim3((g.nic + 255) / 256, g.njc), dim3(256), 0, ctx->stream, g, ctx->nvar, q,
                       R, ctx->dsmin.p, ctx->ph.mu_inf, cfl);
    SG_TRY(hipGetLastError(), "update");
    return SG_OK;
  }
  // RK4-Jameson (update_rk4, src/solver/solver.cpp:20-26): the stage input
  // starts at q (q_tmp = q at the start of every step of the reference),
  // stages ping-pong between two buffers and the last one writes q itself.
  const double* in = q;
  double* stage_buf[2] = {ctx->ex_a.p, ctx->ex_b.p};
  for (int s = 0; s < 4; ++s) {
    const bool last = s == 3;
    const ExplicitStage st{q, ctx->dsmin.p, ctx->ph.mu_inf, cfl, 4.0 - s, last ? q : stage_buf[s & 1]};
    SG_TRY(launch_stage(g, ctx->ph, ctx->bc, ctx->sa, in, st, last ? ctx->partial.p : nullptr, last ? ctx->l2.p : nullptr,
                        ctx->stream, ctx->clo),
           "stage");
    in = st.out;
  }
  return SG_OK;
}

int check_args(sg_ctx* ctx, int scheme, double cfl) {
  if (scheme != SG_SCHEME_FORWARD_EULER && scheme != SG_SCHEME_RK4_JAMESON)
    return sg_fail(ctx, SG_ERR_ARG, "scheme must be SG_SCHEME_FORWARD_EULER or SG_SCHEME_RK4_JAMESON");
  if (!(cfl > 0.0) || !std::isfinite(cfl)) return sg_fail(ctx, SG_ERR_ARG, "cfl must be positive and finite");
  return SG_OK;
}

double seconds_since(std::chrono::steady_clock::time_point t0) {
  return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
}

}  // namespace

extern "C" {

int sg_step_explicit_dev(sg_ctx* ctx, double* q_dev, int scheme, double cfl, double* l2) {
  if (!ctx || !q_dev) return SG_ERR_ARG;
  int rc;
  if ((rc = check_args(ctx, scheme, cfl))) return rc;
  if ((rc = ensure_buffers(ctx, scheme))) return rc;
  if ((rc = enqueue_step(ctx, q_dev, scheme, cfl))) return rc;
  double h[10];
  SG_TRY(hipMemcpyAsync(h, ctx->l2.p, ctx->nvar * sizeof(double), hipMemcpyDeviceToHost, ctx->stream), "D2H");
  SG_TRY(hipStreamSynchronize(ctx->stream), "explicit step");
  sg_norms_returned(ctx, h, ctx->nvar);
  if (l2) std::copy(h, h + ctx->nvar, l2);
  for (int k = 0; k < ctx->nvar; ++k)
    if (!std::isfinite(h[k])) return sg_fail(ctx, SG_ERR_NAN, "non-finite residual norm in an explicit step");
  return SG_OK;
}

int sg_solve_explicit(sg_ctx* ctx, double* q_aos, const sg_explicit_opts* o, sg_solve_report* rep, double* l2_hist) {
  if (!ctx || !q_aos || !o) return SG_ERR_ARG;
  int rc;
  if ((rc = check_args(ctx, o->scheme, o->cfl))) return rc;
  if (o->iteration_max < 0) return sg_fail(ctx, SG_ERR_ARG, "iteration_max must be >= 0");
  if ((rc = ensure_buffers(ctx, o->scheme))) return rc;
  const auto t0 = std::chrono::steady_clock::now();
  const int nv = ctx->nvar;
  const size_t ncell = ctx->ncell();
  double* q = ctx->q.p;
  SG_TRY(hipMemcpyAsync(ctx->aos_a.p, q_aos, ncell * nv * sizeof(double), hipMemcpyHostToDevice, ctx->stream), "H2D");
  SG_TRY(launch_aos_to_soa(ctx->geo.nic, ctx->geo.njc, ctx->g.ldi, nv, ctx->aos_a.p, q, ctx->stream), "aos->soa");
  sg_solve_report R{};
  double cfl = o->cfl, l2[10];
  int counter = 0;
  rc = SG_OK;
  for (;; ++counter) {
    if ((rc = enqueue_step(ctx, q, o->scheme, cfl))) return rc;
    SG_TRY(hipMemcpyAsync(l2, ctx->l2.p, nv * sizeof(double), hipMemcpyDeviceToHost, ctx->stream), "D2H");
    SG_TRY(hipStreamSynchronize(ctx->stream), "explicit step");
    sg_norms_returned(ctx, l2, nv);
    if (counter == 0) std::copy(l2, l2 + nv, R.l2_initial);
    if (l2_hist) std::copy(l2, l2 + nv, l2_hist + (size_t)counter * nv);
    if (o->verbose && counter % o->verbose == 0)
      std::fprintf(stderr, "explicit %6d  cfl %.3e  |R| %.3e %.3e %.3e %.3e\n", counter, cfl, l2[0], l2[1], l2[2], l2[3]);
    bool finite = true, below = o->tolerance > 0.0;
    for (int k = 0; k < nv; ++k) {
      finite = finite && std::isfinite(l2[k]);
      below = below && l2[k] < o->tolerance;
    }
    if (!finite) { rc = sg_fail(ctx, SG_ERR_NAN, "non-finite residual norm in the explicit loop"); break; }
    if (below) { R.converged = 1; break; }
    if (counter > o->iteration_max) break;  // solver.cpp:136 (after the update)
    if (o->cfl_ramp && counter + 1 > o->cfl_ramp_iteration) cfl = std::min(std::pow(cfl, o->cfl_ramp_exponent), 1e12);
  }
  std::copy(l2, l2 + nv, R.l2_final);
  R.iterations = counter + 1;
  R.cfl_final = cfl;
  SG_TRY(launch_soa_to_aos(ctx->geo.nic, ctx->geo.njc, ctx->g.ldi, nv, q, ctx->aos_b.p, ctx->stream), "soa->aos");
  SG_TRY(hipMemcpyAsync(q_aos, ctx->aos_b.p, ncell * nv * sizeof(double), hipMemcpyDeviceToHost, ctx->stream), "D2H");
  SG_TRY(hipStreamSynchronize(ctx->stream), "download");
  R.wall_s = R.residual_s = seconds_since(t0);
  if (rep) *rep = R;
  return rc;
}

}  // extern "C"
