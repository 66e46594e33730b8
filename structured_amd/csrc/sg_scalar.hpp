// Scalar types for the device kernels: plain double, and a forward dual
// number (value + one tangent) so that the same templated residual code
// yields the exact matrix-free tangent J.v in one sweep.
#pragma once
#include <hip/hip_runtime.h>

namespace sg {

struct Dual {
  double v, d;
  __host__ __device__ Dual() : v(0.0), d(0.0) {}
  __host__ __device__ Dual(double x) : v(x), d(0.0) {}
  __host__ __device__ Dual(double x, double t) : v(x), d(t) {}
};

__device__ __forceinline__ Dual operator+(Dual a, Dual b) { return Dual(a.v + b.v, a.d + b.d); }
__device__ __forceinline__ Dual operator-(Dual a, Dual b) { return Dual(a.v - b.v, a.d - b.d); }
__device__ __forceinline__ Dual operator-(Dual a) { return Dual(-a.v, -a.d); }
__device__ __forceinline__ Dual operator*(Dual a, Dual b) { return Dual(a.v * b.v, a.d * b.v + a.v * b.d); }
__device__ __forceinline__ Dual operator/(Dual a, Dual b) {
  double r = a.v / b.v;
  return Dual(r, (a.d - r * b.d) / b.v);
}
__device__ __forceinline__ Dual operator+(Dual a, double b) { return Dual(a.v + b, a.d); }
__device__ __forceinline__ Dual operator+(double a, Dual b) { return Dual(a + b.v, b.d); }
__device__ __forceinline__ Dual operator-(Dual a, double b) { return Dual(a.v - b, a.d); }
__device__ __forceinline__ Dual operator-(double a, Dual b) { return Dual(a - b.v, -b.d); }
__device__ __forceinline__ Dual operator*(Dual a, double b) { return Dual(a.v * b, a.d * b); }
__device__ __forceinline__ Dual operator*(double a, Dual b) { return Dual(a * b.v, a * b.d); }
__device__ __forceinline__ Dual operator/(Dual a, double b) { return Dual(a.v / b, a.d / b); }
__device__ __forceinline__ Dual operator/(double a, Dual b) {
  double r = a / b.v;
  return Dual(r, -r * b.d / b.v);
}
__device__ __forceinline__ Dual& operator+=(Dual& a, Dual b) { a = a + b; return a; }
__device__ __forceinline__ Dual& operator-=(Dual& a, Dual b) { a = a - b; return a; }

// Reciprocal from the hardware estimate refined by two Newton steps
// (r <- r + r (1 - x r)); within ~1 ulp for the normal, finite operands of
// this solver.  Used in place of IEEE division on the hot path.
__device__ __forceinline__ double frcp(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = __builtin_fma(-x, r, 1.0);
  r = __builtin_fma(r, e, r);
  e = __builtin_fma(-x, r, 1.0);
  return __builtin_fma(r, e, r);
}
__device__ __forceinline__ double srcp(double x) { return frcp(x); }
__device__ __forceinline__ Dual srcp(Dual x) {
  double r = frcp(x.v);
  return Dual(r, -r * r * x.d);
}
__device__ __forceinline__ double sdiv(double a, double b) { return a * frcp(b); }
__device__ __forceinline__ Dual sdiv(Dual a, Dual b) {
  double ib = frcp(b.v), r = a.v * ib;
  return Dual(r, (a.d - r * b.d) * ib);
}
__device__ __forceinline__ Dual sdiv(Dual a, double b) {
  double ib = frcp(b);
  return Dual(a.v * ib, a.d * ib);
}
__device__ __forceinline__ Dual sdiv(double a, Dual b) {
  double ib = frcp(b.v), r = a * ib;
  return Dual(r, -r * b.d * ib);
}

// x^(2/3) for x > 0 without pow: z = x^(-2/3) solves z^-3 = x^2; seed from
// the single-precision log2/exp2 units, then two Newton steps
// z <- z (4 - x^2 z^3) / 3 (relative error 2e^2 per step), and
// x^(2/3) = x^2 z^2.
__device__ __forceinline__ double pow23(double x) {
  const float xf = (float)x;
  const float zf = __builtin_amdgcn_exp2f(-(2.0f / 3.0f) * __builtin_amdgcn_logf(xf));
  const double a = x * x;
  double z = (double)zf;
  z = z * (4.0 - a * (z * z * z)) * (1.0 / 3.0);
  z = z * (4.0 - a * (z * z * z)) * (1.0 / 3.0);
  return a * z * z;
}

__device__ __forceinline__ double val(double x) { return x; }
__device__ __forceinline__ double val(Dual x) { return x.v; }
__device__ __forceinline__ double tan_(double) { return 0.0; }
__device__ __forceinline__ double tan_(Dual x) { return x.d; }

// Square root of a positive normal x from the hardware reciprocal square
// root estimate: y = x r, h = r / 2, one coupled Newton (Goldschmidt) step,
// then two residual corrections y + (x - y^2) h (Markstein).  No scaling of
// tiny or huge inputs and no special cases: 0, infinities and negatives are
// not handled (the callers pass squared magnitudes bounded away from zero).
__device__ __forceinline__ double fsqrt(double x) {
  const double r = __builtin_amdgcn_rsq(x);
  double y = x * r, h = 0.5 * r;
  const double e = __builtin_fma(-y, h, 0.5);
  y = __builtin_fma(y, e, y);
  h = __builtin_fma(h, e, h);
  double d = __builtin_fma(-y, y, x);
  y = __builtin_fma(d, h, y);
  d = __builtin_fma(-y, y, x);
  return __builtin_fma(d, h, y);
}

// z^(1/6) for z > 0 without pow: seed from the single-precision log2 / exp2
// units, then two Newton steps on y^6 = z: y <- y (5 + z / y^6) / 6.
__device__ __forceinline__ double pow16(double z) {
  double y = (double)__builtin_amdgcn_exp2f((1.0f / 6.0f) * __builtin_amdgcn_logf((float)z));
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const double y2 = y * y;
    y = y * (5.0 + z * frcp(y2 * y2 * y2)) * (1.0 / 6.0);
  }
  return y;
}

__device__ __forceinline__ double ssqrt(double x) { return fsqrt(x); }
__device__ __forceinline__ Dual ssqrt(Dual x) {
  double r = fsqrt(x.v);
  return Dual(r, x.d * frcp(2.0 * r));
}
__device__ __forceinline__ double sabs(double x) { return fabs(x); }
__device__ __forceinline__ Dual sabs(Dual x) { return x.v < 0.0 ? -x : x; }
// x^(2/3) for the power-law viscosity (src/model/fluid.cpp:38-40).
__device__ __forceinline__ double spow23(double x) { return pow23(x); }
__device__ __forceinline__ Dual spow23(Dual x) {
  double r = pow23(x.v);
  return Dual(r, (2.0 / 3.0) * r * frcp(x.v) * x.d);
}
__device__ __forceinline__ double spow(double x, double e) { return pow(x, e); }
__device__ __forceinline__ Dual spow(Dual x, double e) {
  double r = pow(x.v, e);
  return Dual(r, e * pow(x.v, e - 1.0) * x.d);
}
// z^(1/6) (SA destruction f_w)
__device__ __forceinline__ double spow16(double z) { return pow16(z); }
__device__ __forceinline__ Dual spow16(Dual z) {
  const double y = pow16(z.v);
  return Dual(y, (1.0 / 6.0) * y * frcp(z.v) * z.d);
}
__device__ __forceinline__ double ssel(bool c, double a, double b) { return c ? a : b; }
__device__ __forceinline__ Dual ssel(bool c, Dual a, Dual b) { return Dual(c ? a.v : b.v, c ? a.d : b.d); }
__device__ __forceinline__ double smin(double a, double b) { return a < b ? a : b; }
__device__ __forceinline__ Dual smin(Dual a, double b) { return a.v < b ? a : Dual(b); }

// Element (r, c) of a row-major array, for the cells of one tile: the tile's
// origin (jo, io) goes into the scalar base, so that a lane needs one byte
// offset for all arrays of the same row length.  I: 32 bits, or 64 where a
// tile's rows span more than 4 GiB.
template <class I>
__device__ __forceinline__ double tile_at(const double* a, int ld, int jo, int io, int c, int r) {
  const char* base = reinterpret_cast<const char*>(a + (size_t)jo * ld + io);
  return *reinterpret_cast<const double*>(base + ((I)(r - jo) * (I)ld + (I)(c - io)) * 8u);
}

// Loads of a state component for scalar type S: component k of the cell with
// index idx (column ci, row cj).  The dual reads the tangent from a second
// array of the same layout.
template <class S>
struct Field;
template <>
struct Field<double> {
  const double* v;
  __device__ __forceinline__ void begin(int) {}
  __device__ __forceinline__ double at(int k, size_t plane, size_t idx, int, int) const { return v[k * plane + idx]; }
  template <int NQ, class I>
  __device__ __forceinline__ void load(double* o, size_t plane, int ld, int jo, int io, int c, int r) const {
#pragma unroll
    for (int k = 0; k < NQ; ++k) o[k] = tile_at<I>(v + k * plane, ld, jo, io, c, r);
  }
};
template <>
struct Field<Dual> {
  const double* v;
  const double* d;
  __device__ __forceinline__ void begin(int) {}
  __device__ __forceinline__ Dual at(int k, size_t plane, size_t idx, int, int) const {
    return Dual(v[k * plane + idx], d[k * plane + idx]);
  }
  template <int NQ, class I>
  __device__ __forceinline__ void load(Dual* o, size_t plane, int ld, int jo, int io, int c, int r) const {
#pragma unroll
    for (int k = 0; k < NQ; ++k)
      o[k] = Dual(tile_at<I>(v + k * plane, ld, jo, io, c, r), tile_at<I>(d + k * plane, ld, jo, io, c, r));
  }
};

// One coloured direction: tangent 1 in component m of the cells of colour
// (a, b) = (column, row) mod per, 0 elsewhere.  A launch takes every
// direction in its grid's third dimension.  per = 5 separates the 13-point
// stencil (reach 2), per = 3 the 3x3 box (reach 1).
struct Direction {
  int per, nv;
  int a = 0, b = 0, m = 0;
  __host__ __device__ int count() const { return per * per * nv; }
  __device__ __forceinline__ void begin(int z) {
    m = z % nv;
    b = z / nv % per;
    a = z / nv / per;
  }
};
struct SeedField {
  const double* v;
  Direction dir;
  __device__ __forceinline__ void begin(int z) { dir.begin(z); }
  __device__ __forceinline__ Dual at(int k, size_t plane, size_t idx, int ci, int cj) const {
    const bool on = k == dir.m && ci % dir.per == dir.a && cj % dir.per == dir.b;
    return Dual(v[k * plane + idx], on ? 1.0 : 0.0);
  }
  template <int NQ, class I>
  __device__ __forceinline__ void load(Dual* o, size_t plane, int ld, int jo, int io, int c, int r) const {
    const bool colour = c % dir.per == dir.a && r % dir.per == dir.b;
#pragma unroll
    for (int k = 0; k < NQ; ++k) o[k] = Dual(tile_at<I>(v + k * plane, ld, jo, io, c, r), colour && k == dir.m ? 1.0 : 0.0);
  }
};

template <class S>
struct OutField;
template <>
struct OutField<double> {
  double* v;
  __device__ __forceinline__ void begin(int) {}
  template <int NV>
  __device__ __forceinline__ void put(size_t plane, size_t idx, int, int, const double* x) const {
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k * plane + idx] = x[k];
  }
};
template <>
struct OutField<Dual> {
  double* v;  // may be null: value not stored
  double* d;
  // with idt (per cell), d receives z idt - tangent: the operator z/dt - J z
  const double* idt = nullptr;
  const double* z = nullptr;
  __device__ __forceinline__ void begin(int) {}
  template <int NV>
  __device__ __forceinline__ void put(size_t plane, size_t idx, int, int, const Dual* x) const {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      if (v) v[k * plane + idx] = x[k].v;
      d[k * plane + idx] = idt ? z[k * plane + idx] * idt[idx] - x[k].d : x[k].d;
    }
  }
};

// Jacobian blocks from coloured directions: the tangent at row cell r is
// column m of the block J[r, c] for the one cell c of the direction's colour
// in r's per x per window.  blocks[((slot nv + row) nv + col) plane + cell];
// slots are the 3x3 box, then (0,-+2) and (-+2,0).
struct OutBlocks {
  double* blocks;
  Direction dir;
  __device__ __forceinline__ void begin(int z) { dir.begin(z); }
  template <int NV>
  __device__ __forceinline__ void put(size_t plane, size_t idx, int ci, int cj, const Dual* x) const {
    const int h = dir.per / 2;
    int di = (dir.a - ci) % dir.per, dj = (dir.b - cj) % dir.per;
    di += di < -h ? dir.per : 0;
    di -= di > h ? dir.per : 0;
    dj += dj < -h ? dir.per : 0;
    dj -= dj > h ? dir.per : 0;
    const bool box = di >= -1 && di <= 1 && dj >= -1 && dj <= 1;
    // (dj, di) of the box in rows -1, 0, 1, four bits each
    constexpr unsigned long long kBox = 0x827403615ull;  // (1,1)8 (0,1)2 (-1,1)7 (1,0)4 (0,0)0 (-1,0)3 (1,-1)6 (0,-1)1 (-1,-1)5
    int slot = box ? (int)(kBox >> (4 * (3 * (dj + 1) + di + 1))) & 15 : -1;
    if (!box && di == 0) slot = dj < 0 ? 9 : 10;
    if (!box && dj == 0) slot = di < 0 ? 11 : 12;
    if (slot < 0) return;
#pragma unroll
    for (int k = 0; k < NV; ++k) blocks[(size_t)((slot * NV + k) * NV + dir.m) * plane + idx] = x[k].d;
  }
};

}  // namespace sg
