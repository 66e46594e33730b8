// Kernel launchers of the residual / tangent path (the residual kernel
// finalises its own norms) and the small helper kernels (local time step,
// layout conversion, wall quantities).  Everything is FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "sg_kernels.hpp"
#include "sg_residual.hpp"

namespace sg {

// Rows so long (some 27 million columns) that the rows a tile reads span more
// than 32-bit byte offsets can.
static bool wide_rows(const DevGeom& g) {
  return (size_t)(kTileLarge + 4) * (size_t)std::max(g.ldi, g.ldf) * sizeof(double) > 0xFFFFFFFFull;
}

// Tile height by the size of the grid.  Tiles of 16 rows of faces (512
// threads) recompute 10% of the faces and stage 43% more cells than they own;
// tiles of 8 rows 18% and 77%.  But the launch takes as long as the CU with
// the most work-groups, and a work-group of 16 rows takes twice as long as one
// of 8 (dual numbers 2.2 times: one of 16 rows or two of 8 fill the CU's
// registers, and the one has nothing to run at its barriers).  Measured, 16
// against 8 rows, states from memory, SA residual: 67.5 / 74.6 us at 1409x641,
// 23.1 / 25.9 at 705x321, and where the rule takes 8: 58.1 / 61.4 at 1201x601,
// 44.5 / 45.3 at 1001x501, 37.4 / 35.5 at 865x449, 22.6 / 23.0 at 545x385, 20.2 /
// 18.1 at 481x257, 14.8 / 12.1 at 281x151; laminar 18.8 / 21.3 at 705x321, 18.4 /
// 18.4 at 545x385.  J.v: 33.6 / 38.3 at 705x321, and 8: 123 / 118 at 1409x641,
// 75.8 / 71.3 at 1001x501, 32.6 / 32.4 at 545x385.
// Jacobian blocks (a coloured direction per z-layer) take 8 rows: 1,367 / 1,352 us
// at 385x193, 403 / 347 at 193x97, 1,168 / 1,157 at 545x385 (45 directions), 9,207 /
// 9,257 at 1001x501.
template <class S>
static int tile_rows(const DevGeom& g) {
  constexpr int kCUs = 256, kRatio = sizeof(S) == sizeof(double) ? 20 : 22;  // tenths
  const int small = (residual_tiles(g, kTileSmall) + kCUs - 1) / kCUs;
  const int large = (residual_tiles(g, kTileLarge) + kCUs - 1) / kCUs;
  return !wide_rows(g) && kRatio * large < 10 * small ? kTileLarge : kTileSmall;
}

size_t norm_slots(const DevGeom& g, int norms) { return kSlotHead + (size_t)residual_tiles(g, tile_rows<double>(g)) * norms; }
static unsigned long long* norm_words(double* slots) {
  return slots ? reinterpret_cast<unsigned long long*>(slots) + kSlotHead : nullptr;
}

template <int TY, class I, class S, bool SA, class F, class O>
static void launch_tiles(unsigned extra, unsigned nz, hipStream_t s, const DevGeom& g, const DevPhys& ph, const DevBc& bc, F fq, O fo,
                         const double* beta_dot, const DevClosure& clo, NormOut no) {
  const dim3 grid((unsigned)residual_tiles(g, TY) + extra, 1, nz), block(TX * TY);
  if constexpr (SA) {
    if (clo.kind == CLOSURE_ANALYTIC) {
      hipLaunchKernelGGL((residual_kernel<TY, I, S, SA, CLOSURE_ANALYTIC, F, O>), grid, block, 0, s, g, ph, bc, fq, fo,
                         beta_dot, clo, no);
      return;
    }
    if (clo.kind == CLOSURE_MLP) {
      hipLaunchKernelGGL((residual_kernel<TY, I, S, SA, CLOSURE_MLP, F, O>), grid, block, 0, s, g, ph, bc, fq, fo, beta_dot,
                         clo, no);
      return;
    }
  }
  hipLaunchKernelGGL((residual_kernel<TY, I, S, SA, CLOSURE_FIELD, F, O>), grid, block, 0, s, g, ph, bc, fq, fo, beta_dot,
                     clo, no);
}
template <class S, bool SA, class F, class O>
static void launch_cl(hipStream_t s, const DevGeom& g, const DevPhys& ph, const DevBc& bc, F fq, O fo,
                      const double* beta_dot, const DevClosure& clo, NormOut no = NormOut(),
                      unsigned nz = 1) {
  const unsigned extra = no.slots ? 1 : 0;  // the work-group that sums the norms
  if (wide_rows(g)) launch_tiles<kTileSmall, size_t, S, SA>(extra, nz, s, g, ph, bc, fq, fo, beta_dot, clo, no);
  else if constexpr (std::is_same_v<F, SeedField>)
    launch_tiles<kTileSmall, unsigned, S, SA>(extra, nz, s, g, ph, bc, fq, fo, beta_dot, clo, no);
  else if (tile_rows<S>(g) == kTileLarge)
    launch_tiles<kTileLarge, unsigned, S, SA>(extra, nz, s, g, ph, bc, fq, fo, beta_dot, clo, no);
  else launch_tiles<kTileSmall, unsigned, S, SA>(extra, nz, s, g, ph, bc, fq, fo, beta_dot, clo, no);
}

hipError_t launch_residual(const DevGeom& g, const DevPhys& ph, const DevBc& bc, bool sa, const double* q, double* r,
                           double* slots, double* l2, hipStream_t s, const DevClosure& clo, int l2_count) {
  if ((l2 != nullptr) != (slots != nullptr)) return hipErrorInvalidValue;
  const int nv2 = 2 * (sa ? 5 : 4);
  if (l2_count <= 0 || l2_count > nv2) l2_count = nv2;
  Field<double> fq{q};
  OutField<double> fo{r};
  const NormOut no{norm_words(slots), l2, l2_count};
  if (sa) launch_cl<double, true>(s, g, ph, bc, fq, fo, nullptr, clo, no);
  else launch_cl<double, false>(s, g, ph, bc, fq, fo, nullptr, DevClosure(), no);
  return hipGetLastError();
}

// A Runge-Kutta stage as the residual's output: q0 + (R dt) / denom with the
// cell's local time step at q0, which is read here, so neither R nor dt goes
// through memory (a stage kernel after the residual was 3.9 us and a launch of
// 15 at 281x151).  out may be q0's own array, but not the residual's input.
struct StageField {
  ExplicitStage st;
  __device__ __forceinline__ void begin(int) {}
  template <int NV>
  __device__ __forceinline__ void put(size_t plane, size_t idx, int, int, const double* x) const {
    double q[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) q[k] = st.q0[k * plane + idx];
    const double dt = cell_dt(q[0], q[1], q[2], q[3], st.dsmin[idx], st.mu_inf, st.cfl);
#pragma unroll
    for (int k = 0; k < NV; ++k) {
#pragma clang fp contract(off)
      st.out[k * plane + idx] = q[k] + (x[k] * dt) / st.denom;
    }
  }
};
hipError_t launch_stage(const DevGeom& g, const DevPhys& ph, const DevBc& bc, bool sa, const double* q,
                        const ExplicitStage& st, double* slots, double* l2, hipStream_t s, const DevClosure& clo) {
  if ((l2 != nullptr) != (slots != nullptr)) return hipErrorInvalidValue;
  const NormOut no{norm_words(slots), l2, sa ? 5 : 4};
  if (sa) launch_cl<double, true>(s, g, ph, bc, Field<double>{q}, StageField{st}, nullptr, clo, no);
  else launch_cl<double, false>(s, g, ph, bc, Field<double>{q}, StageField{st}, nullptr, DevClosure(), no);
  return hipGetLastError();
}

hipError_t launch_jv(const DevGeom& g, const DevPhys& ph, const DevBc& bc, bool sa, const double* q, const double* v,
                     double* r, double* jv, hipStream_t s, const double* beta_dot, const DevClosure& clo,
                     const double* idt) {
  Field<Dual> fq{q, v};
  OutField<Dual> fo{r, jv, idt, v};
  if (sa) launch_cl<Dual, true>(s, g, ph, bc, fq, fo, beta_dot, clo);
  else launch_cl<Dual, false>(s, g, ph, bc, fq, fo, nullptr, DevClosure());
  return hipGetLastError();
}

// Jacobian blocks of the residual at q: one launch takes every coloured
// direction (per^2 nv of them, 45 or 125 with SA) as the third dimension of
// its grid, seeds it where the state is loaded and stores its columns where the
// tangent is formed.  A launch per direction with a seed and an extraction
// kernel around it took 29 us each at 385x193 (20 of them the sweep, whose 406
// tiles do not fill the chip), 27 at 97x65, where the sweep is 40 tiles; now
// 6.2 and 4.1.
hipError_t launch_blocks(const DevGeom& g, const DevPhys& ph, const DevBc& bc, bool sa, const double* q, int per,
                         double* blocks, hipStream_t s, const DevClosure& clo) {
  if (per != 3 && per != 5) return hipErrorInvalidValue;
  const Direction d{per, sa ? 5 : 4};
  const SeedField fq{q, d};
  const OutBlocks fo{blocks, d};
  const unsigned nz = (unsigned)d.count();
  const NormOut no;
  if (sa) launch_cl<Dual, true>(s, g, ph, bc, fq, fo, nullptr, clo, no, nz);
  else launch_cl<Dual, false>(s, g, ph, bc, fq, fo, nullptr, DevClosure(), no, nz);
  return hipGetLastError();
}

// EulerEquation::calc_dt, src/model/eulerequation.cpp:237-259.
__global__ void dt_kernel(DevGeom g, double mu_inf, int nv, const double* q, const double* dsmin, double cfl, double* dt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (i >= g.nic) return;
  const size_t c = (size_t)j * g.ldi + i;
  const double val = cell_dt(q[c], q[g.plane + c], q[2 * g.plane + c], q[3 * g.plane + c], dsmin[c], mu_inf, cfl);
  for (int k = 0; k < nv; ++k) dt[k * g.plane + c] = val;
}

hipError_t launch_dt(const DevGeom& g, double mu_inf, int nv, const double* q, const double* dsmin, double cfl,
                     double* dt, hipStream_t s) {
  hipLaunchKernelGGL(dt_kernel, dim3((g.nic + 255) / 256, g.njc), dim3(256), 0, s, g, mu_inf, nv, q, dsmin, cfl, dt);
  return hipGetLastError();
}

// AoS q[i][j][k] <-> SoA a[k][j][i]; one thread per cell.
__global__ void aos_to_soa_kernel(int nic, int njc, int ldi, int nv, const double* aos, double* soa) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (i >= nic) return;
  const size_t plane = (size_t)njc * ldi;
  const double* src = aos + ((size_t)i * njc + j) * nv;
  for (int k = 0; k < nv; ++k) soa[k * plane + (size_t)j * ldi + i] = src[k];
}
__global__ void soa_to_aos_kernel(int nic, int njc, int ldi, int nv, const double* soa, double* aos) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (i >= nic) return;
  const size_t plane = (size_t)njc * ldi;
  double* dst = aos + ((size_t)i * njc + j) * nv;
  for (int k = 0; k < nv; ++k) dst[k] = soa[k * plane + (size_t)j * ldi + i];
}

hipError_t launch_aos_to_soa(int nic, int njc, int ldi, int nv, const double* aos, double* soa, hipStream_t s) {
  hipLaunchKernelGGL(aos_to_soa_kernel, dim3((nic + 127) / 128, njc), dim3(128), 0, s, nic, njc, ldi, nv, aos, soa);
  return hipGetLastError();
}
hipError_t launch_soa_to_aos(int nic, int njc, int ldi, int nv, const double* soa, double* aos, hipStream_t s) {
  hipLaunchKernelGGL(soa_to_aos_kernel, dim3((nic + 127) / 128, njc), dim3(128), 0, s, nic, njc, ldi, nv, soa, aos);
  return hipGetLastError();
}

// Wall quantities, IOManager::write_surface (src/utils/io.cpp:181-255): one
// block; each thread takes wall cells, recomputes the eta-face (j = 0)
// Green-Gauss gradients of u, v (the reference reads them from the last
// residual evaluation), Cp from the first two interior cells and Cf from
// mu_inf (u_y - v_x); the four force sums are reduced in a fixed order.
template <class S, bool SA>
__global__ void wall_kernel(DevGeom g, DevPhys ph, DevBc bc, Field<S> fq, int first, int nb, const double* xv0,
                            const double* yv0, double qinf, double* cp_out, double* cf_out, double* dcf_out,
                            double* fsum) {
  __shared__ double red[4][256];
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  const int nic = g.nic;
  for (int n = threadIdx.x; n < nb; n += blockDim.x) {
    const int ci = first + n;
    auto prim = [&](int a, int b) -> Prim<S> {
      if (a >= 0 && a < nic && b >= 0 && b < g.njc) return prim_interior<S, SA>(fq, g, ph, a, b);
      return eval_node<S, SA>(bc.ghost_map[ghost_index(a, b, nic, g.njc)], bc, fq, g, ph);
    };
    Prim<S> c0 = prim(ci, 0), c1 = prim(ci, 1);
    S cp = (0.5 * (c0.p + c1.p) - ph.p_inf) / qinf;
    // eta face j = 0 of column ci (src/utils/mesh.cpp:99-104,124-125)
    Prim<S> s0 = prim(ci, -1), w0 = prim(ci - 1, 0), ws = prim(ci - 1, -1), e0 = prim(ci + 1, 0), es = prim(ci + 1, -1);
    auto NX = [&](int a, int b) { return g.nex[(size_t)b * g.ldi + a]; };
    auto NY = [&](int a, int b) { return g.ney[(size_t)b * g.ldi + a]; };
    auto CX = [&](int a, int b) { return g.ncx[(size_t)b * g.ldf + a]; };
    auto CY = [&](int a, int b) { return g.ncy[(size_t)b * g.ldf + a]; };
    const double tx = 0.5 * (NX(ci, 0) + NX(ci, 1)), ty = 0.5 * (NY(ci, 0) + NY(ci, 1));
    const double bx = NX(ci, 0), by = NY(ci, 0), lx = CX(ci, 0), ly = CY(ci, 0), rx = CX(ci + 1, 0), ry = CY(ci + 1, 0);
    const double V = g.vol[ci];
    auto grad = [&](S t, S b, S w, S wsv, S e, S esv, S* o) {
      S l = 0.25 * (t + b + w + wsv), r = 0.25 * (t + b + e + esv);
      o[0] = (tx * t - bx * b + rx * r - lx * l) / V;
      o[1] = (ty * t - by * b + ry * r - ly * l) / V;
    };
    S gu[2], gv[2];
    grad(c0.u, s0.u, w0.u, ws.u, e0.u, es.u, gu);
    grad(c0.v, s0.v, w0.v, ws.v, e0.v, es.v, gv);
    S tau = ph.mu_inf * (gu[1] - gv[0]) / qinf;
    if (cp_out) cp_out[n] = val(cp);
    if (cf_out) cf_out[n] = val(tau);
    if (dcf_out) dcf_out[n] = tan_(tau);
    const double dx = xv0[ci + 1] - xv0[ci], dy = yv0[ci + 1] - yv0[ci];
    double sfdiv = 2.0 / 3.0 * (val(gu[0]) + val(gv[1]));
    double sxx = ph.mu_inf * (2.0 * val(gu[0]) - sfdiv) / qinf;
    double syy = ph.mu_inf * (2.0 * val(gv[1]) - sfdiv) / qinf;
    acc[0] += -val(cp) * dx;
    acc[1] += val(cp) * dy;
    acc[2] += -val(tau) * dy + syy * dx;
    acc[3] += val(tau) * dx - sxx * dy;
  }
  for (int k = 0; k < 4; ++k) red[k][threadIdx.x] = acc[k];
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int k = 0; k < 4; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + w];
    __syncthreads();
  }
  if (fsum && threadIdx.x < 4) fsum[threadIdx.x] = red[threadIdx.x][0];
}

hipError_t launch_wall(const DevGeom& g, const DevPhys& ph, const DevBc& bc, bool sa, const double* q, int first,
                       int nb, const double* xv0, const double* yv0, double qinf, double* cp, double* cf, double* fsum,
                       hipStream_t s) {
  Field<double> fq{q};
  if (sa) hipLaunchKernelGGL((wall_kernel<double, true>), dim3(1), dim3(256), 0, s, g, ph, bc, fq, first, nb, xv0, yv0,
                             qinf, cp, cf, nullptr, fsum);
  else hipLaunchKernelGGL((wall_kernel<double, false>), dim3(1), dim3(256), 0, s, g, ph, bc, fq, first, nb, xv0, yv0,
                          qinf, cp, cf, nullptr, fsum);
  return hipGetLastError();
}

hipError_t launch_wall_tangent(const DevGeom& g, const DevPhys& ph, const DevBc& bc, bool sa, const double* q,
                               const double* v, int first, int nb, const double* xv0, const double* yv0, double qinf,
                               double* dcf, hipStream_t s) {
  Field<Dual> fq{q, v};
  if (sa) hipLaunchKernelGGL((wall_kernel<Dual, true>), dim3(1), dim3(256), 0, s, g, ph, bc, fq, first, nb, xv0, yv0,
                             qinf, nullptr, nullptr, dcf, nullptr);
  else hipLaunchKernelGGL((wall_kernel<Dual, false>), dim3(1), dim3(256), 0, s, g, ph, bc, fq, first, nb, xv0, yv0,
                          qinf, nullptr, nullptr, dcf, nullptr);
  return hipGetLastError();
}

}  // namespace sg
