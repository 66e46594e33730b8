// Internal C++ interface between the host context and the kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "sg_device.hpp"

namespace sg {

size_t norm_slots(const DevGeom& g, int norms);
// Norms (optional: both of slots and l2, or neither): slots holds nv or 2 nv
// partial sums per tile (norm_slots words with the head), all empty before
// the first launch and after every launch.  The launch's last block adds them
// and writes the L2 norms of R, then of V R, to l2 (device): l2_count entries
// (0: all 2 nv; nv: the norms of R only).
hipError_t launch_residual(const DevGeom& g, const DevPhys& ph, const DevBc& bc, bool sa, const double* q, double* r,
                           double* slots, double* l2, hipStream_t s, const DevClosure& clo = DevClosure(),
                           int l2_count = 0);
// out = q0 + (R(q) dt(q0)) / denom, the stages of an explicit step; with slots
// the norms of R (nv entries of l2).  out may be q0, but not q.
struct ExplicitStage {
  const double *q0, *dsmin;
  double mu_inf, cfl, denom;
  double* out;
};
hipError_t launch_stage(const DevGeom& g, const DevPhys& ph, const DevBc& bc, bool sa, const double* q,
                        const ExplicitStage& st, double* slots, double* l2, hipStream_t s, const DevClosure& clo);
// J.v (+ (dR/dbeta).beta_dot when beta_dot is not null; v may be all zero);
// with idt (per cell) jv receives v idt - J.v instead
hipError_t launch_jv(const DevGeom& g, const DevPhys& ph, const DevBc& bc, bool sa, const double* q, const double* v,
                     double* r, double* jv, hipStream_t s, const double* beta_dot = nullptr,
                     const DevClosure& clo = DevClosure(), const double* idt = nullptr);
// Jacobian blocks at q by coloured directions (per 5: the 13-point stencil; 3:
// the 3x3 box, the +-2 slots are not written)
hipError_t launch_blocks(const DevGeom& g, const DevPhys& ph, const DevBc& bc, bool sa, const double* q, int per,
                         double* blocks, hipStream_t s, const DevClosure& clo);
hipError_t launch_dt(const DevGeom& g, double mu_inf, int nv, const double* q, const double* dsmin, double cfl,
                     double* dt, hipStream_t s);
hipError_t launch_aos_to_soa(int nic, int njc, int ldi, int nv, const double* aos, double* soa, hipStream_t s);
hipError_t launch_soa_to_aos(int nic, int njc, int ldi, int nv, const double* soa, double* aos, hipStream_t s);
hipError_t launch_wall(const DevGeom& g, const DevPhys& ph, const DevBc& bc, bool sa, const double* q, int first,
                       int nb, const double* xv0, const double* yv0, double qinf, double* cp, double* cf, double* fsum,
                       hipStream_t s);

// tangent of the wall Cf along v (dcf has nb entries)
hipError_t launch_wall_tangent(const DevGeom& g, const DevPhys& ph, const DevBc& bc, bool sa, const double* q,
                               const double* v, int first, int nb, const double* xv0, const double* yv0, double qinf,
                               double* dcf, hipStream_t s);

}  // namespace sg
