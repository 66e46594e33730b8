// Plain-data descriptors shared by the host context and the kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace sg {
// An empty slot of a reduction across work-groups: a signalling NaN, which no
// arithmetic produces.
constexpr unsigned long long kNoValue = 0x7FF4534C4F545321ull;

// Polls before a wait for another work-group's value gives up (each takes about
// a microsecond, so several seconds).  Such waits are for work-groups started
// earlier, so they end.
constexpr int kWaitPolls = 1 << 22;

// Slots of a reduction across work-groups (device memory): a head, then the
// values, which are empty between launches.  A wait that gave up makes its result
// NaN and fills the head's state: values that came late may then lie in the
// slots, where the next reduction would take them for its own.  So later results
// are not used until reduce_slots_init: the residual's norms are NaN then, and
// the Krylov solver, which looks at every result, ends.
struct SlotHead {
  unsigned long long state;  // empty, or a wait gave up
  unsigned long long polls;  // bound of the norms' waits
};
constexpr int kSlotHead = 16;  // words: a line of its own
}  // namespace sg

namespace sg {

// Device geometry, struct-of-arrays.  Cell arrays: a[j*ldi + i] (i < nic,
// j < njc).  Chi-face arrays (faces i = 0..ni-1 between cells i-1 and i):
// a[j*ldf + i].  Eta-face arrays (faces j = 0..nj-1): a[j*ldi + i].
struct DevGeom {
  int ni, nj, nic, njc;
  int ldi, ldf;
  size_t plane;              // njc * ldi, stride between state components
  const double* ncx;         // normal_chi x, [njc][ldf]
  const double* ncy;
  const double* nex;         // normal_eta x, [nj][ldi]
  const double* ney;
  const double* vol;         // [njc][ldi]
  const double* wd;          // wall distance (SA)
  const double* beta;        // SA production multiplier
};

// Tiles of the residual kernel: TX x TY faces, (TX - 1) x (TY - 1) cells.
constexpr int TX = 32, OX = TX - 1;
constexpr int kTileSmall = 8, kTileLarge = 16;  // TY
inline __host__ __device__ int residual_tiles(const DevGeom& g, int ty) {
  return ((g.nic + OX - 1) / OX) * ((g.njc + ty - 2) / (ty - 1));
}

struct DevPhys {
  double rho_inf, u_inf, v_inf, p_inf, T_inf, mu_inf, pr, nut_inf;
  double R, cp;              // gas constant p/(rho T) and cp = gamma R/(gamma-1)
  double iR, ipr, iTinf;     // 1/R, 1/Pr, 1/T_inf
  double eps_chi, eps_eta;   // limiter epsilons (10/nic)^3, (10/njc)^3
  double dpdx, dpdy;
  int order;                 // 1 or 2
  int viscous;               // mu_inf > 1e-15
  int flux;                  // FluxKind
  int pad_;
};

// Convective flux scheme (solver.flux).
enum FluxKind { FLUX_ROE = 0, FLUX_AUSM = 1 };

// One boundary-condition evaluation.  Operand refs: >= 0 is an interior
// cell (cj*nic + ci), < 0 is another node -(ref+1).
enum BcOp { OP_FREESTREAM = 0, OP_SLIP = 1, OP_WALL = 2, OP_ISO = 3, OP_OUTFLOW = 4, OP_COPY = 5 };
struct BcNode {
  int op, ra, rb, pad;
  double c0, c1, c2;         // (u_bc, v_bc, T_bc) or (nx, ny) of the wall face
};

// Ghost ring: perimeter index of ghosted cell (gi, gj):
//   bottom row gj=0          : gi                      (gi = 0..nic+1)
//   top row    gj=njc+1      : (nic+2) + gi
//   left col   gi=0,  gj=1..njc : 2(nic+2) + gj-1
//   right col  gi=nic+1       : 2(nic+2) + njc + gj-1
// ghost_map[perimeter] = final node id, or -1 if no boundary writes it.
struct DevBc {
  const BcNode* nodes;
  const int* ghost_map;
};

// Closure for the SA production multiplier beta:
//   CLOSURE_FIELD    beta from the per-cell field DevGeom::beta (default)
//   CLOSURE_ANALYTIC beta = 1 + amp tanh(a . f + a0), FP64, f the local features
//   CLOSURE_MLP      beta = 1 + MLP(f) on the matrix cores (BF16 operands,
//                    FP32 accumulation), W1/b1/b2/W3/b3 FP32, W2 BF16
enum ClosureKind { CLOSURE_FIELD = 0, CLOSURE_ANALYTIC = 1, CLOSURE_MLP = 2 };
struct DevClosure {
  int kind = CLOSURE_FIELD;
  double coef[7] = {0, 0, 0, 0, 0, 0, 0};  // analytic: a[5], a0, amp
  const float* params = nullptr;           // MLP packed FP32 parameters
  const void* w2 = nullptr;                // MLP W2 as BF16 [64 out][64 in]
  double* aux = nullptr;                   // optional output: features (5 planes) and beta (1 plane)
};

constexpr double kGamma = 1.4;

// SA-noft2 constants (Spalart & Allmaras 1994 as catalogued by NASA TMR),
// SA-neg branch for nu~ < 0 (c_t3 = 1.2, c_n1 = 16).
constexpr double kCb1 = 0.1355, kSigma = 2.0 / 3.0, kCb2 = 0.622, kKappa = 0.41;
constexpr double kCw2 = 0.3, kCw3 = 2.0, kCv1 = 7.1, kCv2 = 0.7, kCv3 = 0.9, kPrt = 0.9;
constexpr double kCt3 = 1.2, kCn1 = 16.0;

// Local time step of one cell, EulerEquation::calc_dt
// (src/model/eulerequation.cpp:237-259): CFL / (lambda/l + 2 mu_inf/l^2) with
// lambda = c + |u| + |v| and l the shorter face length; IEEE divisions and
// square root in the reference's order, so the value is the reference's.
__device__ __forceinline__ double cell_dt(double r, double ru, double rv, double rE, double len, double mu_inf,
                                          double cfl) {
  const double u = ru / r, v = rv / r;
  const double p = (rE - 0.5 * r * (u * u + v * v)) * (kGamma - 1.0);
  const double lam = sqrt(kGamma * p / r) + fabs(u) + fabs(v);
  return cfl / (lam / len + 2.0 * mu_inf / len / len);
}

// Wavefront sum in a fixed order with DPP lane moves (no LDS round trips):
// xor 1 and xor 2 inside quads, the mirrors inside 8 and 16 lanes, then the
// row broadcasts of lanes 15 and 31 carry the row sums up; lane 63 ends with
// the total.  Lanes a move does not write receive 0.
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ double dpp_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROW_MASK, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROW_MASK, 0xF, false);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ unsigned long long slot_load(const unsigned long long* slot) {
  return __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void slot_store(unsigned long long* slot, unsigned long long v) {
  __hip_atomic_store(slot, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The head as it was when the launch began; slots: the first value.
__device__ __forceinline__ SlotHead slot_head(const unsigned long long* slots) {
  return *reinterpret_cast<const SlotHead*>(slots - kSlotHead);
}
__device__ __forceinline__ void slots_lost(unsigned long long* slots) { slot_store(slots - kSlotHead, 0); }

// Sum over each row of 16 lanes, in all of them.
__device__ __forceinline__ double row_sum(double v) {
  v += dpp_move<0xB1>(v);        // quad_perm [1,0,3,2]
  v += dpp_move<0x4E>(v);        // quad_perm [2,3,0,1]
  v += dpp_move<0x141>(v);       // row_half_mirror
  v += dpp_move<0x140>(v);       // row_mirror
  return v;
}
__device__ __forceinline__ double wave_sum_lane63(double v) {
  v = row_sum(v);
  v += dpp_move<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
  v += dpp_move<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}

}  // namespace sg
