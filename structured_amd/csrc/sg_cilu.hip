// Chunked line block ILU(0) of A = I/dt - J on the 13-point stencil.
//
// The i-range is cut into chunks of W columns.  Inside a chunk the cells are
// ordered column by column with j fastest (o = (i - i0) njc + j), so every
// wall-normal line is contiguous and its banded part is factored exactly;
// couplings between chunks are dropped (block Jacobi over chunks).  In that
// order the lower neighbours of (i, j) are (-2,0), (-1,-1), (-1,0), (-1,+1),
// (0,-2), (0,-1).  A cell can be solved two rows behind the column before it.
//
// The factorisation walks a chunk's levels L = j + 2 (i - i0) with one
// work-group per chunk.  The apply cuts the chunk once more, into groups of
// up to 6 (nv 5) or 8 (nv 4) columns, twice that on very wide grids and where not
// every CU of the device takes part, with one solving wave each: a column depends
// on earlier columns only, so the groups run as a pipeline, each on its own CU,
// and hand the solved values of their edge columns on through memory.
//
// Factors are stored in FP32 (the preconditioner only has to approximate
// A^-1; FGMRES runs in FP64) in the order the solving waves read them, see
// Lay below.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "sg_linalg.hpp"
#include "sg_pass_order.hpp"

namespace sg {

// Work-group barrier that orders LDS only: the level loop keeps the next
// level's global loads in flight across it (the usual barrier also waits for
// every outstanding global load).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Compile-time stencil tables (fully unrolled loops fold them away):
// offsets and the neighbour slots of the factorisation.
namespace ct {
constexpr int Di[NSLOT] = {0, 0, 0, -1, 1, -1, 1, -1, 1, 0, 0, -2, 2};
constexpr int Dj[NSLOT] = {0, -1, 1, 0, 0, -1, -1, 1, 1, -2, 2, 0, 0};
constexpr int Low[6] = {11, 5, 3, 7, 9, 1};
constexpr int Up[6] = {2, 10, 6, 4, 8, 12};
// The 3x3-box pattern (slots 0-8; the +-2 slots dropped): four lower and
// four upper neighbours, in the same order as above.
constexpr int Low9[4] = {5, 3, 7, 1};
constexpr int Up9[4] = {2, 6, 4, 8};
template <bool NINE>
constexpr int nn() { return NINE ? 4 : 6; }
template <bool NINE>
constexpr int low(int n) { return NINE ? Low9[n] : Low[n]; }
template <bool NINE>
constexpr int up(int n) { return NINE ? Up9[n] : Up[n]; }
constexpr bool in_box(int s) { return s >= 0 && s < 9; }
// offsets of a slot known at run time, four bits each, plus 2
constexpr unsigned long long pack(const int* d) {
  unsigned long long v = 0;
  for (int s = 0; s < NSLOT; ++s) v |= (unsigned long long)(d[s] + 2) << (4 * s);
  return v;
}
constexpr unsigned long long kDi = pack(Di), kDj = pack(Dj);
__device__ __forceinline__ int di(int s) { return (int)(kDi >> (4 * s) & 15) - 2; }
__device__ __forceinline__ int dj(int s) { return (int)(kDj >> (4 * s) & 15) - 2; }
// The apply's neighbours, in the order of their records: lower ones for the
// ascending pass, upper ones for the descending pass, entry n of one being
// the opposite offset of entry n of the other.  0-2 are the column before
// (its oldest, middle and newest solved cell in reach), 3 the cell's own
// column, 4 and 5 the +-2 couplings of the 13-point stencil.
constexpr int Asc[6] = {5, 3, 7, 1, 9, 11};
constexpr int Desc[6] = {8, 4, 6, 2, 10, 12};
__device__ __forceinline__ int asc(int n) { return (int)(0xB91735ull >> (4 * n)) & 15; }
__device__ __forceinline__ int desc(int n) { return (int)(0xCA2648ull >> (4 * n)) & 15; }
static_assert(Asc[0] == 5 && Asc[1] == 3 && Asc[2] == 7 && Asc[3] == 1 && Asc[4] == 9 && Asc[5] == 11, "asc");
static_assert(Desc[0] == 8 && Desc[1] == 4 && Desc[2] == 6 && Desc[3] == 2 && Desc[4] == 10 && Desc[5] == 12, "desc");
// place of an upper neighbour's slot among them
template <bool NINE>
constexpr int up_index(int s) {
  for (int u = 0; u < nn<NINE>(); ++u)
    if (up<NINE>(u) == s) return u;
  return -1;
}
constexpr int slot(int di, int dj) {
  for (int s = 0; s < NSLOT; ++s)
    if (Di[s] == di && Dj[s] == dj) return s;
  return -1;
}
// The products of a row's elimination, in order: with lower neighbour n's
// diagonal inverse (u = -1), then with those of its upper blocks u that meet a
// block `target` of the row.
struct Product {
  int n, u, target;
};
template <bool NINE>
struct Plan {
  Product p[6 * 7] = {};
  int count = 0;
  constexpr Plan() {
    for (int n = 0; n < nn<NINE>(); ++n) {
      p[count++] = {n, -1, low<NINE>(n)};
      for (int u = 0; u < nn<NINE>(); ++u) {
        const int t = slot(Di[low<NINE>(n)] + Di[up<NINE>(u)], Dj[low<NINE>(n)] + Dj[up<NINE>(u)]);
        if (t >= 0 && (!NINE || in_box(t))) p[count++] = {n, u, t};
      }
    }
  }
};
template <bool NINE>
constexpr Plan<NINE> plan;
// f(integral_constant) for 0 .. N - 1
template <class F, int... I>
__device__ __forceinline__ void each(F f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>()), ...);
}
}  // namespace ct

// Column groups of the apply and the layout of their factor records.
//
// Both passes of an apply run through the same steps: the descending one
// counts columns and rows from the other end (c' = GW - 1 - c and s = njc -
// 1 - j; c' = c and s = j ascending).  Step t = X + s + 2 c' solves row s of
// column c'; X steps come first in which only edge columns of the group
// before arrive (GC of them, none when one group holds the chunk).
//
// P lanes share a row of a cell, entry k of column c' on lanes P (c' NV + k) +
// h.  With P = 2, lane h = 0 takes the blocks of the own column (and of the
// oldest cell in reach of the column before), lane 1 those of the newest and
// middle cell of the column before, and each one half of the diagonal's row:
// so each has one block whose operand the step before solves, and one that was
// ready earlier.
//
// Per step and lane a record holds n1 floats in the pass without the diagonal
// (row k of the lane's blocks, the one with the newest operand first), n2 in
// the pass with it (its part of the diagonal's row last): float4 runs over the
// lanes, then single floats for the remainder, so a wave reads 16 bytes per
// lane, contiguous over lanes.  Records of cells or neighbours that do not
// exist are zero, which makes their values zero without a mask.  Four arrays:
// M^-1 ascending (L) and descending (U, D^-1), then M^-T ascending (U^T, D^-T)
// and descending (L^T), where a block's column is stored as a row at the cell
// that multiplies by it.
template <int NV, int W, bool NINE, int P>
struct Lay {
  static constexpr int B = NV * NV, NN = NINE ? 4 : 6;
  static constexpr int GCX = NINE ? 1 : 2, CAP = 64 / P / NV;
  static constexpr int NG = W <= CAP ? 1 : (W + CAP - 1) / CAP;
  static constexpr int GC = NG == 1 ? 0 : GCX, X = 2 * GC;
  static constexpr int GW = (W + NG - 1) / NG;  // columns of a group
  static constexpr int ROWS = GW * NV, LN = P * ROWS;  // rows of a step, lanes with one
  static constexpr int ND = (NV + P - 1) / P;          // entries of the diagonal's row on a lane
  static constexpr int n1 = NN / P * NV, n2 = n1 + ND;
  static constexpr int UN = 8;                  // steps in a block of the solving loop
  // steps whose records are in flight (they share the registers with the
  // operands)
  static constexpr int pd(int n) { return n <= 20 ? 8 : 4; }
  // neighbour n (ct::Asc, ct::Desc order): the lane that takes it and its
  // place there
  static constexpr int half(int n) { return P == 2 && (n == 1 || n == 2 || n == 5); }
  static constexpr int place(int n) { return P == 1 ? n : n == 2 || n == 3 ? 0 : n < 2 ? 1 : 2; }
  __host__ __device__ static int neighbour(int h, int place) {
    return P == 1 ? place : place == 0 ? (h ? 2 : 3) : place == 1 ? h : 4 + h;
  }
  static constexpr int rs(int n) { return (n * LN + 15) / 16 * 16; }  // floats of a step's record
  static constexpr int count(int a) { return a == 0 || a == 3 ? n1 : n2; }  // per lane, in array a
  static_assert(LN <= 64, "a group fits a wave");
  // steps of a pass, rounded up to the solving loop's blocks, and records
  // (the loop reads ahead)
  __host__ __device__ static int steps(int njc) { return (X + njc + 2 * (GW - 1) + UN - 1) / UN * UN; }
  __host__ __device__ static int nrec(int njc) { return steps(njc) + UN; }
  // float offset of array a (0-3)
  __host__ __device__ static size_t array(int a, int nchunk, int njc) {
    const size_t per = (size_t)nchunk * NG * nrec(njc);
    return per * (a == 0 ? 0 : a == 1 ? rs(n1) : a == 2 ? rs(n1) + rs(n2) : rs(n1) + 2 * rs(n2));
  }
  // one more record per chunk, for what the factorisation's idle lanes store
  __host__ __device__ static size_t spare(int chunk, int nchunk, int njc) {
    return (size_t)nchunk * NG * nrec(njc) * (2 * rs(n1) + 2 * rs(n2)) + (size_t)chunk * rs(n2);
  }
  __host__ __device__ static size_t floats(int nchunk, int njc) { return spare(nchunk, nchunk, njc); }
  // float of entry f on a lane inside a record of n floats per lane
  __device__ static unsigned in_record(int n, int lane, int f) {
    const int q = n / 4;
    return f < 4 * q ? (unsigned)((f / 4 * LN + lane) * 4 + (f & 3)) : (unsigned)(4 * q * LN + (f - 4 * q) * LN + lane);
  }
  // words of one link (edge values of one pass, all rows), of a pass's links, and
  // of all of them with their head (on whole lines)
  __host__ __device__ static size_t link(int njc) { return (size_t)njc * GC * NV; }
  __host__ __device__ static size_t pass_links(int nchunk, int njc) { return (size_t)nchunk * (NG - 1) * link(njc); }
  static size_t links(int nchunk, int njc) { return kSlotHead + (2 * pass_links(nchunk, njc) + 15) / 16 * 16; }
};

// Zeroes the records of M^-1 that the factorisation does not write, or writes
// in part: steps at both ends of a pass, and groups with absent columns.  One
// block per record.
template <int NV, int W, bool NINE, int P>
__global__ __launch_bounds__(256) void cilu_zero_kernel(int nic, int njc, int nchunk, float* rec) {
  using La = Lay<NV, W, NINE, P>;
  const int t = blockIdx.x, gg = blockIdx.y, s = t - La::X;
  const int wk = min(W, nic - gg / La::NG * W) - gg % La::NG * La::GW;
  if (wk >= La::GW && s >= 2 * (La::GW - 1) && s < njc) return;
  for (int a = 0; a < 2; ++a) {
    const int rs = La::rs(La::count(a));
    float* r = rec + La::array(a, nchunk, njc) + ((size_t)gg * La::nrec(njc) + t) * rs;
    for (int e = threadIdx.x; e < rs; e += 256) r[e] = 0.0f;
  }
}

// The records of M^-T from those of M^-1: row r of a cell's U^T and D^-T from
// the U blocks of its lower neighbours and its own D^-1, row r of L^T from the
// L blocks of its upper neighbours, zeros elsewhere.  One block per record.
// Written by the factorisation, they were half of the bytes that one CU per
// chunk had to move; here the whole chip does.
template <int NV, int W, bool NINE, int P>
__global__ __launch_bounds__(256) void cilu_transpose_kernel(int nic, int njc, int nchunk, float* rec) {
  using La = Lay<NV, W, NINE, P>;
  const int t = blockIdx.x, gg = blockIdx.y, chunk = gg / La::NG, c0 = gg % La::NG * La::GW, wk = min(W, nic - chunk * W);
  const int nrec = La::nrec(njc);
  // float of row `row`, half h, place f of cell (c, j) in array a
  auto from = [&](int a, int c, int j, int row, int h, int f) {
    const int n = La::count(a), g = c / La::GW, cl = c % La::GW;
    const bool asc = a == 0 || a == 2;
    const int c1 = asc ? cl : La::GW - 1 - cl, s = asc ? j : njc - 1 - j;
    return rec[La::array(a, nchunk, njc) + ((size_t)(chunk * La::NG + g) * nrec + La::X + s + 2 * c1) * La::rs(n) +
               La::in_record(n, P * (c1 * NV + row) + h, f)];
  };
#pragma unroll
  for (int a = 2; a < 4; ++a) {
    constexpr int N[2] = {La::n2, La::n1};
    const int n = N[a - 2], rs = La::rs(n);
    float* out = rec + La::array(a, nchunk, njc) + ((size_t)gg * nrec + t) * rs;
    for (int e = threadIdx.x; e < rs; e += 256) {
      // lane and float of the lane, as in Lay::in_record
      const int q4 = n / 4 * 4 * La::LN;
      const int lane = e < q4 ? e / 4 % La::LN : (e - q4) % La::LN;
      const int f = e < q4 ? e / 4 / La::LN * 4 + e % 4 : n / 4 * 4 + (e - q4) / La::LN;
      const int h = lane % P, row = lane / P % NV, c1 = lane / P / NV;
      const int s = t - La::X - 2 * c1, c = c0 + (a == 2 ? c1 : La::GW - 1 - c1), j = a == 2 ? s : njc - 1 - s;
      float v = 0.0f;
      if (f < n && c < wk && s >= 0 && s < njc) {
        if (f < La::n1) {
          const int place = f / NV, k = f % NV, nb = La::neighbour(h, place);
          const int slot = a == 2 ? ct::asc(nb) : ct::desc(nb);
          const int cn = c + ct::di(slot), jn = j + ct::dj(slot);
          if (cn >= 0 && cn < wk && jn >= 0 && jn < njc) v = from(a == 2 ? 1 : 0, cn, jn, k, h, place * NV + row);
        } else {
          const int q = h * La::ND + f - La::n1;
          if (q < NV) v = from(1, c, j, q, row / La::ND, La::n1 + row % La::ND);
        }
      }
      out[e] = v;
    }
  }
}

// Shape of the factorisation: a thread holds one row of a cell, CW cells to a
// wave.
template <int NV, int W, bool NINE>
struct Fac {
  static constexpr int NN = NINE ? 4 : 6, NS = NINE ? 9 : NSLOT;  // blocks of a row
  static constexpr int CW = 64 / NV, NW = (W + CW - 1) / CW;      // cells of a wave, waves
  static constexpr int N2 = (NS * NV + 1) / 2;                    // 16-byte words of a row
  // levels kept: a cell's lower neighbours lie on the three (13-point: four)
  // levels before its own
  static constexpr int NR = NINE ? 4 : 5;
  // the kept blocks hold FP32 values; where they fit as doubles nothing has to
  // be converted when they are read
  using R = std::conditional_t<NINE, double, float>;
  // block and cell strides: the cells of a wave read different banks
  static constexpr int BP = NINE ? (NV == 5 ? 26 : 18) : (NV == 5 ? 28 : 20);
  static constexpr int GP = 2 * NV * NV + (NV == 4 ? 2 : 0);
};

// Gathers the factorisation's operands into level order: for chunk, level L,
// 16-byte word e and row (c, r) of the level, entries 2 e and 2 e + 1 of row r
// of the blocks of I/dt - J at cell (i0 + c, L - 2c), slot after slot, or zero
// where the cell or the neighbour lies outside the chunk or the grid.  The rows
// of a level are contiguous, so the factorisation reads 16 bytes a thread, all
// used.  Read in place, a level's W cells lie on a diagonal of rows 2 ldi
// apart: every 8-byte read took its own line, used again only ~W levels later
// after L2 had evicted it.  Here all levels are gathered at once and the
// levels that share a line are read together.  Only the pattern's blocks: at
// 545x385 the box 0.44 ms, all 13 blocks 0.73.
template <int NV, int W, bool NINE>
__global__ __launch_bounds__(256) void cilu_gather_kernel(int nic, int njc, int ldi, int nlev, const double* idt,
                                                          const double* blocks, double2* ops, size_t total) {
  using Fa = Fac<NV, W, NINE>;
  constexpr int B = NV * NV;
  const size_t plane = (size_t)njc * ldi;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
    size_t u = t;
    const int row = (int)(u % (W * NV)), c = row / NV, r = row % NV;
    u /= W * NV;
    const int e = (int)(u % Fa::N2);
    u /= Fa::N2;
    const int L = (int)(u % (size_t)nlev), chunk = (int)(u / (size_t)nlev);
    const int i0 = chunk * W, wk = min(W, nic - i0), j = L - 2 * c;
    const size_t cell = (size_t)j * ldi + i0 + c;
    double v[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int f = 2 * e + x, s = f / NV, q = f % NV;
      const int cn = c + ct::di(s), jn = j + ct::dj(s);
      v[x] = 0.0;
      if (s < Fa::NS && c < wk && j >= 0 && j < njc && cn >= 0 && cn < wk && jn >= 0 && jn < njc) {
        v[x] = -blocks[(size_t)(s * B + r * NV + q) * plane + cell];
        if (s == 0 && r == q) v[x] += idt[cell];
      }
    }
    ops[t] = double2{v[0], v[1]};
  }
}

// 16-byte words of the gathered factorisation operands
template <int NV, int W, bool NINE>
static size_t cilu_ops(int nic, int njc) {
  const int nchunk = (nic + W - 1) / W, nlev = njc + 2 * W - 2;
  return (size_t)nchunk * nlev * Fac<NV, W, NINE>::N2 * W * NV;
}

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00027000);
}

// A record's n floats of a lane, in the layout of Lay::in_record.
template <int N, int LN>
__device__ __forceinline__ void put_record(float* rec, int lane, const float* v) {
  float* quads = rec + 4 * lane;
#pragma unroll
  for (int q = 0; q < N / 4; ++q)
    *reinterpret_cast<float4*>(quads + q * LN * 4) = float4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
  float* rest = rec + 4 * (N / 4) * LN + lane;
#pragma unroll
  for (int f = N / 4 * 4; f < N; ++f) rest[(f - 4 * (N / 4)) * LN] = v[f];
}

// Orders this wave's LDS accesses (a wave's LDS operations execute in issue
// order, so nothing is waited for).
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}

// Factorisation, one level after another, one work-group per chunk.  NINE:
// ILU(0) on the 3x3-box pattern (the +-2 blocks of A and their fill dropped;
// with the first-order Jacobian of lhs_order 1 those slots hold fill only),
// else on the 13-point stencil.
//
// Thread (c, r) holds row r of the blocks of its level's cell in column c.  A
// row is eliminated without the cell's other rows: it is multiplied by the
// lower neighbours' diagonal inverses and upper blocks, which an LDS ring keeps
// and the threads of a cell read together (a broadcast).  The diagonal block is
// inverted by Gauss-Jordan with partial pivoting on [D | I], a row a thread:
// rows stay where they are and carry the position that swapping would have
// given them.  The next level's operands are in flight meanwhile.  One barrier a
// level: the ring has room for the level that is written.
//
// What bounds it: a level, njc + 2 W - 2 times.  A wave issues some 1,600
// instructions for it (about 430 FP64 FMAs, the LDS reads that feed them, the
// pivots' exchanges), some 3 us, and one CU moves 59 KB of operands and 29 KB
// of records (nv 5, W 32), about 20 bytes/ns.  A level takes 5.3 us (nv 4:
// 3.3).  With a thread per block entry, two barriers per neighbour and one per
// pivot, every product read ten LDS words for five FMAs and a level took 14 us
// (6.0).  545x385 nv 5 6.35 -> 2.36 ms, and 0.15 for M^-T, which the whole chip
// writes afterwards; 97x65 nv 4 0.76 -> 0.42.
template <int NV, int W, bool NINE, int P>
__global__ __launch_bounds__((64 * Fac<NV, W, NINE>::NW)) __attribute__((amdgpu_waves_per_eu(1, 1))) void
cilu_factor_kernel(int nic, int njc, int nlev, const double2* ops, float* rec) {
  using La = Lay<NV, W, NINE, P>;
  using Fa = Fac<NV, W, NINE>;
  using R = typename Fa::R;
  constexpr int B = NV * NV, NR = Fa::NR, NN = Fa::NN, NS = Fa::NS, N2 = Fa::N2, CW = Fa::CW, ND = La::ND;
  // per level: diagonal inverse, then the upper blocks (ct::up order)
  __shared__ R ring[(NR * (1 + NN) * W + 1) * Fa::BP] __attribute__((aligned(16)));
  constexpr int kNone = NR * (1 + NN) * W;  // the block of an absent neighbour: zero
  // block b of column ci at the level `back` levels before level L
  auto block = [&](int L, int back, int b, int ci) {
    return (int)((((unsigned)(L + NR - back) % NR) * (1 + NN) + b) * W) + ci;
  };
  auto block_or_none = [&](bool there, int at) -> const R* {
    asm volatile("" : "+v"(at));  // a select, not a branch around the index
    return ring + (there ? at : kNone) * Fa::BP;
  };
  __shared__ double gj[Fa::NW * CW + 1][Fa::GP] __attribute__((aligned(16)));  // [D | I] by position; the last: idle lanes
  const int chunk = blockIdx.x, nchunk = gridDim.x, i0 = chunk * W, wk = min(W, nic - i0);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, cw = lane / NV, r = lane % NV;
  const int c = cw < CW ? wave * CW + cw : W, cc = min(c, W - 1);
  double* mat = gj[cw < CW ? wave * CW + cw : Fa::NW * CW];
  const int nrec = La::nrec(njc);
  // the record of cell (ci, jj) in array a, or the spare one (where all lanes take
  // the first place, so that they cost one store)
  auto record = [&](bool there, int a, int ci, int jj) {
    const int g = ci / La::GW, cl = ci % La::GW;
    const bool asc = a == 0 || a == 2;
    const int c1 = asc ? cl : La::GW - 1 - cl, s = asc ? jj : njc - 1 - jj;
    const size_t at = La::array(a, nchunk, njc) +
                      ((size_t)(chunk * La::NG + g) * nrec + La::X + s + 2 * c1) * La::rs(La::count(a));
    return rec + (there ? at : La::spare(chunk, nchunk, njc));
  };
  // lane of half h of row `row` of column ci
  auto lane_of = [&](bool asc, int ci, int row, int h) {
    const int cl = ci % La::GW;
    return P * ((asc ? cl : La::GW - 1 - cl) * NV + row) + h;
  };
  // (without a branch: a level is one block of code, or its products are not
  // scheduled as written)
  auto inside = [&](int ci, int jj) { return ((unsigned)ci < (unsigned)wk) & ((unsigned)jj < (unsigned)njc); };
  for (int e = threadIdx.x; e < (int)(sizeof(ring) / sizeof(R)); e += blockDim.x) ring[e] = R(0);

  const double2* op = ops + (size_t)chunk * nlev * N2 * (W * NV) + (cc * NV + r);
  double2 next[N2];  // the coming level's operands
  auto fetch = [&](int L) {
    const double2* from = op + (size_t)min(L, nlev - 1) * N2 * (W * NV);
#pragma unroll
    for (int e = 0; e < N2; ++e) next[e] = from[(size_t)e * (W * NV)];
  };
  fetch(0);
  // arrived before the loop: its wait for a level's operands then counts the
  // stores that follow them in the loop, and waits for none of those
#pragma unroll
  for (int e = N2 - 1; e >= 0; --e) asm volatile("" : "+v"(next[e].x), "+v"(next[e].y));
  lds_barrier();
  for (int L = 0; L < nlev; ++L) {
    const int j = L - 2 * c;
    const bool valid = inside(c, j);  // (the idle lanes' c = W is outside)
    double a[NS][NV];
#pragma unroll
    for (int f = 0; f < NS * NV; ++f) a[f / NV][f % NV] = f & 1 ? next[f / 2].y : next[f / 2].x;
    __builtin_amdgcn_sched_barrier(0);
    fetch(L + 1);

    // ---- elimination of the lower neighbours; a product's block is read while
    // the one before is formed.  An absent neighbour's blocks, and its block in
    // this row, are zero; so are the blocks that couple a neighbour to a cell
    // outside.
    R blk[2][B];
    double l[NV];
    constexpr int NP = ct::plan<NINE>.count;
    auto read = [&](auto at) {
      constexpr int i = decltype(at)::value;
      constexpr ct::Product pr = ct::plan<NINE>.p[i];
      constexpr int s = ct::low<NINE>(pr.n), di = ct::Di[s], dj = ct::Dj[s];
      const R* m = block_or_none(valid & inside(c + di, j + dj), block(L, -dj - 2 * di, 1 + pr.u, c + di));
#pragma unroll
      for (int k = 0; k < B; ++k) blk[i & 1][k] = m[k];
    };
    read(std::integral_constant<int, 0>());
    ct::each([&](auto at) {
      constexpr int i = decltype(at)::value;
      constexpr ct::Product pr = ct::plan<NINE>.p[i];
      // one wait for the whole block, before the next one's reads
#pragma unroll
      for (int k = B - 1; k >= 0; --k) asm volatile("" : "+v"(blk[i & 1][k]));
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (i + 1 < NP) read(std::integral_constant<int, i + 1>());
      double sum[NV];
#pragma unroll
      for (int q = 0; q < NV; ++q) sum[q] = 0.0;
#pragma unroll
      for (int k = 0; k < NV; ++k)
#pragma unroll
        for (int q = 0; q < NV; ++q) sum[q] += (pr.u < 0 ? a[pr.target][k] : l[k]) * (double)blk[i & 1][k * NV + q];
#pragma unroll
      for (int q = 0; q < NV; ++q) {
        if (pr.u < 0) a[pr.target][q] = l[q] = sum[q];
        else a[pr.target][q] -= sum[q];
        asm volatile("" : "+v"(a[pr.target][q]));  // formed here, not where it is used
      }
    }, std::make_integer_sequence<int, NP>());
    __builtin_amdgcn_sched_barrier(0);

    // ---- the level's L and U rows are final: the upper blocks into the ring,
    // both into this cell's records of M^-1
    float r0[P][La::n1], r1[P][La::n2];
#pragma unroll
    for (int n = 0; n < NN; ++n)
#pragma unroll
      for (int q = 0; q < NV; ++q) {
        r0[La::half(n)][La::place(n) * NV + q] = (float)a[ct::Asc[n]][q];
        r1[La::half(n)][La::place(n) * NV + q] = (float)a[ct::Desc[n]][q];
      }
    R* const cell = ring + block(L, 0, 0, cc) * Fa::BP;
    constexpr int kStep = W * Fa::BP;  // from one of a cell's blocks to the next
    if (c < W) {
#pragma unroll
      for (int n = 0; n < NN; ++n)
#pragma unroll
        for (int q = 0; q < NV; ++q)
          cell[(1 + ct::up_index<NINE>(ct::Desc[n])) * kStep + r * NV + q] =
              valid ? (R)r1[La::half(n)][La::place(n) * NV + q] : R(0);
    }
    double d[NV], id[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) { d[q] = a[0][q]; id[q] = q == r ? 1.0 : 0.0; }
    // Stores without a branch around them: where one may be skipped, the next
    // wait for a load waits for all of them.
    float* const to0 = record(valid, 0, cc, j);
#pragma unroll
    for (int h = 0; h < P; ++h) put_record<La::n1, La::LN>(to0, valid ? lane_of(true, cc, r, h) : 0, r0[h]);
    __builtin_amdgcn_sched_barrier(0);

    // ---- inverse of the factored diagonal block
    int pos = r;
#pragma unroll
    for (int p = 0; p < NV; ++p) {
#pragma unroll
      for (int q = p; q < NV; ++q) mat[pos * 2 * NV + q] = d[q];
#pragma unroll
      for (int q = 0; q < NV; ++q) mat[pos * 2 * NV + NV + q] = id[q];
      wave_order();
      double cp = mat[p * 2 * NV + p], best = fabs(cp);
      int piv = p;
#pragma unroll
      for (int rr = p + 1; rr < NV; ++rr) {
        const double x = mat[rr * 2 * NV + p], v = fabs(x);
        if (v > best) { best = v; piv = rr; cp = x; }
      }
      const double ip = 1.0 / cp, f = d[p];
      const double* prow = mat + piv * 2 * NV;
      const bool mine = pos == piv;
#pragma unroll
      for (int q = p + 1; q < NV; ++q) {
        const double x = prow[q] * ip;
        d[q] = mine ? x : f != 0.0 ? d[q] - f * x : d[q];
      }
#pragma unroll
      for (int q = 0; q < NV; ++q) {
        const double x = prow[NV + q] * ip;
        id[q] = mine ? x : f != 0.0 ? id[q] - f * x : id[q];
      }
      pos = mine ? p : pos == p ? piv : pos;
      wave_order();
    }
    if (c < W) {
#pragma unroll
      for (int q = 0; q < NV; ++q) cell[pos * NV + q] = valid ? (R)(float)id[q] : R(0);
    }
    wave_order();
#pragma unroll
    for (int q = 0; q < P * ND; ++q) {  // an odd row's second half ends in a zero
      r1[q / ND][La::n1 + q % ND] = q < NV ? (float)cell[r * NV + min(q, NV - 1)] : 0.0f;
    }
    float* const to1 = record(valid, 1, cc, j);
#pragma unroll
    for (int h = 0; h < P; ++h) put_record<La::n2, La::LN>(to1, valid ? lane_of(false, cc, r, h) : 0, r1[h]);
    lds_barrier();
  }
}

// How far the waves of a work-group have got in a pass: steps solved,
// right-hand-side rows loaded, edge rows received, rows taken out of the ring.
struct Progress {
  int step, loaded, edges, taken;
};
// LDS of one group's work-group: the solved values of the last kRing steps by
// step, column and component (edge columns first; idle lanes store to the
// column after the last), the right-hand sides of the steps to come, and how
// far each wave has got in either pass.
constexpr int kRing = 64;
template <int NV, int W, bool NINE, int P>
struct ApplyLds {
  using La = Lay<NV, W, NINE, P>;
  static constexpr int NVP = (NV + 1) & ~1;  // a cell's values, in 16-byte units
  static constexpr int NP = La::GCX + La::GW;
  double ring[kRing][NP + 1][NVP] __attribute__((aligned(16)));
  double x[kRing][La::ROWS + 1];  // the last place is always zero
  double tmp[La::GW + 1][8] __attribute__((aligned(16)));  // a row's halves at 0 and 4
  Progress pass[2];
  int stored;  // the first pass's stores are complete
};
__device__ __forceinline__ int lds_read(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_write(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_release() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local"); }
__device__ __forceinline__ void lds_acquire() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local"); }

constexpr int kAll = 1 << 29;  // a count that never holds the solving wave up
// The receiving wave of one pass: moves the edge rows the group before
// publishes into the ring.  One poll reads as many rows as fit the wave; a
// word is read as one 64-bit atomic and holds either a value or kNoValue, so
// nothing has to be ordered between words.  The one that fills a link runs, has
// run or will run (see the kernel), so the wait ends.  One that gives up, after `most`
// polls without a new row, fills the state of the links' head (see SlotHead).
template <int NV, int W, bool NINE, int P>
__device__ void cilu_receive(unsigned long long* links, unsigned long long* in, int njc, int most,
                             ApplyLds<NV, W, NINE, P>& sh, Progress& pr) {
  using La = Lay<NV, W, NINE, P>;
  constexpr int EN = La::GCX * NV, RP = 64 / EN;
  const int lane = threadIdx.x & 63, rr = lane / EN, gi = lane % EN / NV, k = lane % NV;
  int n = 0, polls = 0;
  while (n < njc) {
    // edge column gi's row s belongs to step s + X - 2 (1 + gi); its place
    // holds a value that is read up to three steps after its own
    const int row = n + rr, free = lds_read(&pr.step) + kRing - 8 - La::X;
    unsigned long long v = kNoValue;
    if (rr < RP && row < njc && row < free) v = slot_load(in + (size_t)row * EN + lane % EN);
    const unsigned long long missing = ~__ballot(v != kNoValue);
    const int rows = min(RP, (missing ? __builtin_ctzll(missing) : 64) / EN);
    if (rows == 0) {
      if (n < free && ++polls > most) break;  // a full ring is no failure
      continue;
    }
    polls = 0;
    if (rr < rows)
      sh.ring[(row + La::X - 2 * (1 + gi)) & (kRing - 1)][La::GCX - 1 - gi][k] = __longlong_as_double((long long)v);
    n += rows;
    lds_release();
    if (lane == 0) lds_write(&pr.edges, n < njc ? n : kAll);
  }
  if (n < njc) {  // never filled: every value that depends on it becomes NaN
    if (lane == 0) slots_lost(links);
    for (int e = lane; e < kRing * EN; e += 64) sh.ring[e / EN][e % EN / NV][e % NV] = __builtin_nan("");
    lds_release();
    if (lane == 0) lds_write(&pr.edges, kAll);
  }
}

// The storing wave of one pass: takes finished rows out of the ring, stores
// them to z (a row is contiguous in memory, a step's cells are not) and
// publishes the edge columns for the next group.  In the solving wave these
// stores held up the loads, whose waits run in issue order.  After a wait on a
// link that gave up in an earlier launch it stores NaN instead, until the next
// factorisation: values that came late may lie in the links.
template <int NV, int W, bool NINE, int P, bool ASC>
__device__ void cilu_store(double* z, int njc, int ldi, size_t plane, int col0, int wk, unsigned long long* out,
                           const unsigned long long* links, ApplyLds<NV, W, NINE, P>& sh, Progress& pr) {
  using La = Lay<NV, W, NINE, P>;
  constexpr int LAST = La::X + 2 * (La::GW - 1), RB = 4;
  const int lane = threadIdx.x & 63, k = lane % NV, c1 = lane / NV, c = ASC ? c1 : La::GW - 1 - c1;
  const int gi = La::GW - 1 - c1;
  const bool live = c1 < La::GW && c < wk, pub = out && c1 < La::GW && gi < La::GC;
  double* zl = z + (size_t)k * plane + col0 + (live ? c : 0);
  const bool lost = La::NG > 1 && slot_head(links).state != kNoValue;
  for (int n = 0; n < njc;) {
    const int rows = min(min(lds_read(&pr.step) - LAST, njc) - n, RB);
    if (rows <= 0) {
      __builtin_amdgcn_s_sleep(1);
      continue;
    }
    lds_acquire();
    double v[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r)
      v[r] = sh.ring[(La::X + n + r + 2 * c1) & (kRing - 1)][min(La::GCX + c1, ApplyLds<NV, W, NINE, P>::NP)][k];
#pragma unroll
    for (int r = 0; r < RB; ++r) v[r] = lost ? __builtin_nan("") : v[r];
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      if (r >= rows) break;
      if (pub)
        slot_store(out + ((size_t)(n + r) * La::GCX + gi) * NV + k, (unsigned long long)__double_as_longlong(v[r]));
      if (live) zl[(size_t)(ASC ? n + r : njc - 1 - n - r) * ldi] = v[r];
    }
    n += rows;
    lds_release();
    if (lane == 0) lds_write(&pr.taken, n < njc ? n : kAll);
  }
}

// The loading wave of one pass: brings the right-hand sides into LDS by step
// (a row's cells belong to steps two apart), LB rows at a time and one batch
// ahead, and reads one word of every 128-byte line of the records 16 to 32
// steps ahead of the solving wave, so that its loads find them in the XCD's
// L2 instead of memory (much further ahead, the groups of an XCD overflow it).
template <int NV, int W, bool NINE, int P, bool ASC, bool DIAG>
__device__ void cilu_load(const float* R, int njc, int ldi, size_t plane, int col0, int wk, const double* src,
                          ApplyLds<NV, W, NINE, P>& sh, Progress& pr) {
  using La = Lay<NV, W, NINE, P>;
  constexpr int RS = La::rs(DIAG ? La::n2 : La::n1), LB = 16, TAIL = 2 * (La::GW - 1);
  // a batch is fetched when the solving wave is at step s0 - (kRing - X - TAIL)
  constexpr int LEAD = kRing - La::X - TAIL - LB;
  const int lane = threadIdx.x & 63, k = lane % NV, c1 = lane / NV, c = ASC ? c1 : La::GW - 1 - c1;
  const int nrec = La::nrec(njc);
  const bool live = c1 < La::GW && c < wk;
  const double* sl = src + (size_t)k * plane + col0 + (live ? c : 0);
  double v[2][LB];
  float touch[LB];
  auto fetch = [&](int s0, int b) {
#pragma unroll
    for (int u = 0; u < LB; ++u) {
      const int s = min(max(s0 + u, 0), njc - 1);
      v[b][u] = sl[(size_t)(ASC ? s : njc - 1 - s) * ldi];
    }
#pragma unroll
    for (int u = 0; u < LB; ++u)
      touch[u] = R[(size_t)min(max(s0 + u - LEAD, 0), nrec - 1) * RS + min(lane * 32, RS - 1)];
  };
  // rows before the first are zero too: every place starts at zero
  for (int e = lane; e < kRing * (La::ROWS + 1); e += 64) (&sh.x[0][0])[e] = 0.0;
  fetch(0, 0);
  for (int s0 = 0; s0 < njc + TAIL; s0 += 2 * LB) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int s1 = s0 + b * LB;
#pragma unroll
      for (int u = 0; u < LB; ++u) asm volatile("" ::"v"(touch[u]));
      fetch(s1 + LB, b ^ 1);
      // the last place this batch writes must have been read
      while (lds_read(&pr.step) < La::X + s1 + LB - 1 + TAIL + 1 - kRing) __builtin_amdgcn_s_sleep(2);
#pragma unroll
      for (int u = 0; u < LB; ++u)
        if (lane < La::ROWS) sh.x[(La::X + s1 + u + 2 * c1) & (kRing - 1)][lane] = live && s1 + u < njc ? v[b][u] : 0.0;
      lds_release();
      if (lane == 0) lds_write(&pr.loaded, s1 + LB);
    }
  }
  if (lane == 0) lds_write(&pr.loaded, kAll);
}


// The value of the other lane of the pair.
__device__ __forceinline__ double pair_sum(double v) {
  constexpr int kSwap = 0xB1;  // quad_perm [1,0,3,2]
  return v + __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), kSwap, 0xF, 0xF, true),
                              __builtin_amdgcn_mov_dpp(__double2loint(v), kSwap, 0xF, 0xF, true));
}

// The solving wave of one pass, applying the diagonal inverse when DIAG.  The
// operand that the step before solves (own column, or newest cell of the
// column before) is read right after that step is stored; the other was read
// a step earlier, and its product (`base`) and the conversions of the coming
// step are formed while an LDS exchange is under way.  The wave issues one
// instruction every four cycles at best, so its instructions are what a step
// costs: everything that is not a factor, an FMA or an exchange with its
// neighbours is done by the other waves, and no step has a branch but the one
// that waits for them.
template <int NV, int W, bool NINE, bool DIAG>
__device__ __forceinline__ void cilu_solve_pairs(const float* R, int njc, ApplyLds<NV, W, NINE, 2>& sh, Progress& pr, bool up) {
  using La = Lay<NV, W, NINE, 2>;
  using A = ApplyLds<NV, W, NINE, 2>;
  constexpr int N = DIAG ? La::n2 : La::n1, RS = La::rs(N), NQ = N / 4, NREM = N % 4, PD = La::pd(N), UN = La::UN, ND = La::ND;
  static_assert(kRing % UN == 0 && UN % PD == 0, "a block does not wrap around the ring");
  const int lane = threadIdx.x & 63, h = lane & 1, row = min(lane >> 1, La::ROWS), k = row % NV, c1 = row / NV;
  const bool real = row < La::ROWS;
  const int pos = La::GCX + (real ? c1 : 0), wpos = real ? pos : A::NP;
  const int xrow = h ? La::ROWS : row, tk = k / ND * 4 + k % ND;  // the right-hand side is taken once
  const int T = La::steps(njc), rl = min(lane, La::LN - 1);
  // the records of a block of steps and of those that are loaded in it: a pass's
  // whole array may be beyond a buffer's 32-bit offsets
  auto block_of = [&](int t0) { return buffer_of(R + (size_t)t0 * RS, 2 * UN * RS * sizeof(float)); };
  auto rrec = block_of(0);
  const unsigned oq = rl * 16, or_ = (4 * NQ * La::LN + rl) * 4;
  u32x4 fq[PD][NQ > 0 ? NQ : 1];
  unsigned fr[PD][NREM > 0 ? NREM : 1];
  // the record's part that is used first is loaded last, so that one wait
  // covers the record
  int so = 0;  // the record that is loaded next, in the buffer
  auto fetch = [&](int u) {
#pragma unroll
    for (int q = 0; q < NREM; ++q) fr[u][q] = __builtin_amdgcn_raw_buffer_load_b32(rrec, or_ + q * La::LN * 4, so, 0);
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      if (q != NV / 4) fq[u][q] = __builtin_amdgcn_raw_buffer_load_b128(rrec, oq + q * La::LN * 16, so, 0);
    fq[u][NV / 4] = __builtin_amdgcn_raw_buffer_load_b128(rrec, oq + NV / 4 * La::LN * 16, so, 0);
    so += RS * 4;
  };
  auto factor = [&](int u, int e) -> double {  // entry e of the record in set u
    return e < 4 * NQ ? __uint_as_float(fq[u][e / 4 < NQ ? e / 4 : 0][e & 3])
                      : __uint_as_float(fr[u][e >= 4 * NQ ? e - 4 * NQ : 0]);
  };
#pragma unroll
  for (int u = 0; u < PD; ++u) {
    fetch(u);
    // in the loop's order: the wait for a load counts what was issued after
    // it on every path to it
    __builtin_amdgcn_sched_barrier(0);
  }
  int lim = 0;  // steps the other waves allow
  auto wait = [&](int t) {
    if (__builtin_expect(t < lim, 1)) return;
    do {
      // x is read one step early
      const int a = lds_read(&pr.loaded) + La::X - 1, b = up ? lds_read(&pr.edges) + 1 : kAll;
      const int c = lds_read(&pr.taken) + kRing + La::X;
      lim = __builtin_amdgcn_readfirstlane(min(min(a, b), c));
    } while (t >= lim);
    lds_acquire();
  };
  // operands of the coming step: the newest, the one ready earlier, the +-2
  // coupling's; ynext is the earlier one of the step after
  double xn[NV], ye[NV], ynext[NV], far[NV], fn[NV], fd[ND], x, base;
#pragma unroll
  for (int m = 0; m < NV; ++m) xn[m] = ye[m] = ynext[m] = far[m] = 0.0;
  auto early = [&](int u) {
    double p = x;
#pragma unroll
    for (int m = 0; m < NV; ++m) p -= factor(u, NV + m) * ye[m];
    if (!NINE) {
#pragma unroll
      for (int m = 0; m < NV; ++m) p -= factor(u, 2 * NV + m) * far[m];
    }
    base = p;
  };
  auto widen = [&](int u) {
#pragma unroll
    for (int m = 0; m < NV; ++m) fn[m] = factor(u, m);
    if (DIAG) {
#pragma unroll
      for (int m = 0; m < ND; ++m) fd[m] = factor(u, La::n1 + m);
    }
  };
  wait(1);
  x = sh.x[0][xrow];
  early(0);
  widen(0);
  x = sh.x[1][xrow];
  for (int t0 = 0; t0 < T; t0 += UN) {
    rrec = block_of(t0);
    so = PD * RS * 4;
    const int r0 = t0 & (kRing - 1), r1 = (t0 + UN) & (kRing - 1);
    // cell of the column before that is ynext at the block's first step
    const double* y0 = sh.ring[h ? r0 : (r0 - 1) & (kRing - 1)][pos - 1];
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int t = t0 + u, nx = (u + 1) % PD;
      double p = base, s = 0.0;
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        if (m & 1) s += fn[m] * xn[m];
        else p -= fn[m] * xn[m];
      }
      double r = pair_sum(p - s);
#pragma unroll
      for (int m = 0; m < NV; ++m) ye[m] = ynext[m];
      if (DIAG) {
        sh.tmp[c1][tk] = r;
        wave_order();
        double td[ND];
#pragma unroll
        for (int m = 0; m < ND; ++m) td[m] = sh.tmp[c1][4 * h + m];
        if (NINE) {
          __builtin_amdgcn_sched_barrier(0);
          early(nx);
        }
        r = 0.0;
#pragma unroll
        for (int m = 0; m < ND; ++m) r += fd[m] * td[m];
        r = pair_sum(r);
      }
      auto* cur = sh.ring[r0 + u];
      cur[wpos][k] = r;
      wave_order();
      if (u & 1) lds_write(&pr.step, t + 1);
      if (u & 1) wait(t + 2);  // for the next two steps
      const double* yn = u == 0 ? y0 : sh.ring[r0 + u - 1 + h][pos - 1];
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        xn[m] = cur[pos - h][m];
        ynext[m] = yn[m];
        if (!NINE) far[m] = sh.ring[(t - 1 - 2 * h) & (kRing - 1)][pos - 2 * h][m];
      }
      const double x2 = sh.x[u + 2 < UN ? r0 + u + 2 : r1 + u + 2 - UN][xrow];
      __builtin_amdgcn_sched_barrier(0);  // the reads go first: the next step starts with them
      if (!(DIAG && NINE)) early(nx);
      x = x2;
      widen(nx);
      fetch(u % PD);
    }
  }
}

// The same with one lane a row, which takes both operands of either kind.
template <int NV, int W, bool NINE, bool DIAG>
__device__ __forceinline__ void cilu_solve_rows(const float* R, int njc, ApplyLds<NV, W, NINE, 1>& sh, Progress& pr, bool up) {
  using La = Lay<NV, W, NINE, 1>;
  using A = ApplyLds<NV, W, NINE, 1>;
  constexpr int N = DIAG ? La::n2 : La::n1, RS = La::rs(N), NQ = N / 4, NREM = N % 4, PD = La::pd(N), UN = La::UN;
  static_assert(kRing % UN == 0 && UN % PD == 0, "a block does not wrap around the ring");
  const int lane = threadIdx.x & 63, row = min(lane, La::ROWS), k = row % NV, c1 = row / NV;
  const bool real = row < La::ROWS;
  const int pos = La::GCX + (real ? c1 : 0), wpos = real ? pos : A::NP;
  const int T = La::steps(njc), rl = min(lane, La::LN - 1);
  // the records of a block of steps and of those that are loaded in it: a pass's
  // whole array may be beyond a buffer's 32-bit offsets
  auto block_of = [&](int t0) { return buffer_of(R + (size_t)t0 * RS, 2 * UN * RS * sizeof(float)); };
  auto rrec = block_of(0);
  const unsigned oq = rl * 16, or_ = (4 * NQ * La::LN + rl) * 4;
  u32x4 fq[PD][NQ > 0 ? NQ : 1];
  unsigned fr[PD][NREM > 0 ? NREM : 1];
  int so = 0;  // the record that is loaded next, in the buffer
  auto fetch = [&](int u) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) fq[u][q] = __builtin_amdgcn_raw_buffer_load_b128(rrec, oq + q * La::LN * 16, so, 0);
#pragma unroll
    for (int q = 0; q < NREM; ++q) fr[u][q] = __builtin_amdgcn_raw_buffer_load_b32(rrec, or_ + q * La::LN * 4, so, 0);
    so += RS * 4;
  };
  auto factor = [&](int u, int e) -> double {  // entry e of the record in set u
    return e < 4 * NQ ? __uint_as_float(fq[u][e / 4 < NQ ? e / 4 : 0][e & 3])
                      : __uint_as_float(fr[u][e >= 4 * NQ ? e - 4 * NQ : 0]);
  };
#pragma unroll
  for (int u = 0; u < PD; ++u) {
    fetch(u);
    // in the loop's order: the wait for a load counts what was issued after
    // it on every path to it
    __builtin_amdgcn_sched_barrier(0);
  }
  int lim = 0;  // steps the other waves allow
  auto wait = [&](int t) {
    if (__builtin_expect(t < lim, 1)) return;
    do {
      // x is read one step early
      const int a = lds_read(&pr.loaded) + La::X - 1, b = up ? lds_read(&pr.edges) + 1 : kAll;
      const int c = lds_read(&pr.taken) + kRing + La::X;
      lim = __builtin_amdgcn_readfirstlane(min(min(a, b), c));
    } while (t >= lim);
    lds_acquire();
  };
  // the column before at its newest and middle cell in reach (its oldest is
  // in base); the own column's last two cells; the column two before; the
  // coming step's right-hand side, and it without the early couplings
  double xn[NV], vb[NV], xo[NV], xp[NV], far[NV], fo[NV], fn[NV], fd[NV], x, base;
#pragma unroll
  for (int m = 0; m < NV; ++m) xn[m] = vb[m] = xo[m] = xp[m] = far[m] = 0.0;
  auto early = [&](int u, const double* old, const double* mid, const double* own2) {
    double p = x, s = 0.0;
#pragma unroll
    for (int m = 0; m < NV; ++m) {
      p -= factor(u, m) * old[m];
      s += factor(u, NV + m) * mid[m];
    }
    if (!NINE) {
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        p -= factor(u, 4 * NV + m) * own2[m];
        s += factor(u, 5 * NV + m) * far[m];
      }
    }
    base = p - s;
  };
  auto widen = [&](int u) {
#pragma unroll
    for (int m = 0; m < NV; ++m) {
      fo[m] = factor(u, 3 * NV + m);
      fn[m] = factor(u, 2 * NV + m);
      if (DIAG) fd[m] = factor(u, La::n1 + m);
    }
  };
  wait(1);
  x = sh.x[0][row];
  early(0, vb, vb, xp);
  widen(0);
  x = sh.x[1][row];
  for (int t0 = 0; t0 < T; t0 += UN) {
    rrec = block_of(t0);
    so = PD * RS * 4;
    const int r0 = t0 & (kRing - 1), r1 = (t0 + UN) & (kRing - 1);
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int t = t0 + u, nx = (u + 1) % PD;
      double p = base, s = 0.0;
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        p -= fo[m] * xo[m];
        s += fn[m] * xn[m];
      }
      double r = p - s;
      if (DIAG) {
        sh.tmp[c1][k] = r;
        wave_order();
        double td[NV];
#pragma unroll
        for (int m = 0; m < NV; ++m) td[m] = sh.tmp[c1][m];
        if (NINE) {
          __builtin_amdgcn_sched_barrier(0);
          early(nx, vb, xn, xo);
        }
        r = 0.0;
#pragma unroll
        for (int m = 0; m < NV; ++m) r += fd[m] * td[m];
      }
      auto* cur = sh.ring[r0 + u];
      cur[wpos][k] = r;
      wave_order();
      if (u & 1) lds_write(&pr.step, t + 1);
      if (u & 1) wait(t + 2);  // for the next two steps
      double own2[NV], old[NV];
#pragma unroll
      for (int m = 0; m < NV; ++m) {
        old[m] = vb[m]; own2[m] = xo[m];
        vb[m] = xn[m];
        xo[m] = cur[pos][m];
        xn[m] = cur[pos - 1][m];
        if (!NINE) far[m] = sh.ring[(t - 3) & (kRing - 1)][pos - 2][m];
      }
      const double x2 = sh.x[u + 2 < UN ? r0 + u + 2 : r1 + u + 2 - UN][row];
      __builtin_amdgcn_sched_barrier(0);  // the reads go first: the next step starts with them
      if (!(DIAG && NINE)) early(nx, old, vb, own2);
      x = x2;
      widen(nx);
      fetch(u % PD);
    }
  }
}

template <int NV, int W, bool NINE, int P, bool DIAG>
__device__ __forceinline__ void cilu_solve(const float* R, int njc, ApplyLds<NV, W, NINE, P>& sh, Progress& pr, bool up) {
  if constexpr (P == 2) cilu_solve_pairs<NV, W, NINE, DIAG>(R, njc, sh, pr, up);
  else cilu_solve_rows<NV, W, NINE, DIAG>(R, njc, sh, pr, up);
}

// z = (LU)^-1 b, or (LU)^-T b when TR: the ascending and the descending pass, or
// one of them.  Wave 0 of a work-group solves one column group, wave 1 loads and
// wave 2 stores for it, and wave 3 receives the edge columns of the group before
// where a chunk has several.  Work-groups are dealt to the XCDs round-robin by
// index: the groups of a chunk sit on one XCD, consecutive in its order.
//
// Both passes in one launch: a group waits in the second for groups started after
// it, so its XCD must have room for all groups of a chunk (at most 6; the chunks
// before are complete and finish).  The host asks for that only where every CU
// of the device takes part.  A launch per pass needs no room (see
// sg_pass_order.hpp) and takes 1.5 to 2.5 us longer on small grids, 8 at 1409x641
// (448 us).
//
// What bounds it: a step of the solving wave, some 57 instructions of one wave
// and the LDS exchanges that link two steps, times njc + 2 W steps and a pass,
// and about 2 us per group and pass for its link.  Two lanes a row: 150-165 ns
// a step (nv 4: 120-150), one lane 200-215 (155-185; with its records beyond
// L2 290, as one CU takes about 18 bytes/ns from memory); with one work-group
// of nv W threads per chunk and a barrier per level it was 600.  Precond 7,
// W 32, M^-1 (M^-T alike), at first / one lane / two lanes: 97x65 nv 4 101 / 54
// / 51 us, 97x257 nv 5 - / 156 / 135, 705x257 - / 160 / 141, 1409x641 966 / 442
// / 576 (more groups than CUs).
enum { kAscending, kDescending, kBoth };
template <int NV, int W, bool NINE, int P, bool TR, int PASS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void cilu_apply_kernel(
    int nic, int njc, int ldi, int nchunk, const float* rec, unsigned long long* links, int most, const double* b,
    double* z) {
  using La = Lay<NV, W, NINE, P>;
  constexpr bool UP = PASS != kDescending, DOWN = PASS != kAscending;
  __shared__ ApplyLds<NV, W, NINE, P> sh;
  const PassGroup at = pass_group((int)blockIdx.x, La::NG, UP);
  const int chunk = at.chunk, g = at.group;
  if (chunk >= nchunk) return;
  const int i0 = chunk * W, wk = min(W, nic - i0) - g * La::GW;  // columns from this group on
  if (wk <= 0) return;
  const bool left = g > 0, right = wk > La::GW;
  // values of steps not yet solved, and the place after an odd row's last
  // entry, meet zero factors: they need to be finite
  double* zero = &sh.ring[0][0][0];
  for (int e = threadIdx.x; e < (int)(sizeof(sh.ring) / sizeof(double)); e += blockDim.x) zero[e] = 0.0;
  for (int e = threadIdx.x; e < (int)(sizeof(sh.tmp) / sizeof(double)); e += blockDim.x) (&sh.tmp[0][0])[e] = 0.0;
  if (threadIdx.x < 2)
    sh.pass[threadIdx.x] = {0, -La::X, 0, 0};  // not even the steps before the first row may start
  if (threadIdx.x == 0) sh.stored = 0;
  __syncthreads();
  const size_t plane = (size_t)njc * ldi, gr = (size_t)(chunk * La::NG + g) * La::nrec(njc);
  const float* R1 = rec + La::array(TR ? 2 : 0, nchunk, njc) + gr * La::rs(TR ? La::n2 : La::n1);
  const float* R2 = rec + La::array(TR ? 3 : 1, nchunk, njc) + gr * La::rs(TR ? La::n1 : La::n2);
  const int col0 = i0 + g * La::GW, wg = min(wk, La::GW);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Progress &up = sh.pass[0], &down = sh.pass[1];
  // link l of a pass joins groups l and l + 1
  const size_t lw = La::link(njc);
  unsigned long long* la = links + (size_t)chunk * (La::NG - 1) * lw;
  unsigned long long* ld = la + La::pass_links(nchunk, njc);
  // non-transposed: unit-lower L ascending, then D + U descending;
  // transposed: (D + U)^T ascending, then unit-lower L^T descending
  if (wave == 0) {
    if (UP) cilu_solve<NV, W, NINE, P, TR>(R1, njc, sh, up, left);
    if (DOWN) cilu_solve<NV, W, NINE, P, !TR>(R2, njc, sh, down, right);
  } else if (wave == 1) {
    if (UP) cilu_load<NV, W, NINE, P, true, TR>(R1, njc, ldi, plane, col0, wg, b, sh, up);
    if (PASS == kBoth) {
      // the second pass loads what the first stored, and reuses its LDS
      while (!lds_read(&sh.stored) || lds_read(&up.step) < La::steps(njc)) __builtin_amdgcn_s_sleep(1);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
    if (DOWN) cilu_load<NV, W, NINE, P, false, !TR>(R2, njc, ldi, plane, col0, wg, z, sh, down);
  } else if (wave == 2) {
    if (UP) cilu_store<NV, W, NINE, P, true>(z, njc, ldi, plane, col0, wg, right ? la + g * lw : nullptr, links, sh, up);
    if (PASS == kBoth) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      if ((threadIdx.x & 63) == 0) lds_write(&sh.stored, 1);
    }
    if (DOWN)
      cilu_store<NV, W, NINE, P, false>(z, njc, ldi, plane, col0, wg, left ? ld + (g - 1) * lw : nullptr, links, sh, down);
  } else {
    if (UP && left) cilu_receive<NV, W, NINE, P>(links, la + (g - 1) * lw, njc, most, sh, up);
    if (DOWN && right) {
      // the first pass is done with the edge columns' places
      if (PASS == kBoth)
        while (lds_read(&up.step) < La::steps(njc)) __builtin_amdgcn_s_sleep(1);
      cilu_receive<NV, W, NINE, P>(links, ld + g * lw, njc, most, sh, down);
    }
    // the links are empty for the next apply
    for (size_t e = threadIdx.x & 63; e < lw; e += 64) {
      if (UP && left) slot_store(la + (g - 1) * lw + e, kNoValue);
      if (DOWN && right) slot_store(ld + g * lw + e, kNoValue);
    }
  }
}

// The store of a factorisation: the links with their head, the records, the
// factorisation's operands.
template <int NV, int W, bool NINE, int P>
static size_t cilu_size_t(int nic, int njc) {
  using La = Lay<NV, W, NINE, P>;
  const int nchunk = (nic + W - 1) / W;
  return La::links(nchunk, njc) + La::floats(nchunk, njc) / 2 + 2 * cilu_ops<NV, W, NINE>(nic, njc);
}

template <int NV, int W, bool NINE, int P>
static hipError_t cilu_factor_t(int nic, int njc, int ldi, const double* idt, const double* blocks, double* store,
                                hipStream_t s) {
  using La = Lay<NV, W, NINE, P>;
  const int nchunk = (nic + W - 1) / W, nlev = njc + 2 * W - 2;
  const size_t total = cilu_ops<NV, W, NINE>(nic, njc), nl = La::links(nchunk, njc);
  float* rec = reinterpret_cast<float*>(store + nl);
  double2* ops = reinterpret_cast<double2*>(rec + La::floats(nchunk, njc));
  hipLaunchKernelGGL((cilu_zero_kernel<NV, W, NINE, P>), dim3(La::nrec(njc), nchunk * La::NG), dim3(256), 0, s, nic, njc,
                     nchunk, rec);
  const size_t nblk = std::min<size_t>((total + 255) / 256, (size_t)1 << 20);
  hipLaunchKernelGGL((cilu_gather_kernel<NV, W, NINE>), dim3((unsigned)nblk), dim3(256), 0, s, nic, njc, ldi, nlev, idt,
                     blocks, ops, total);
  hipLaunchKernelGGL((cilu_factor_kernel<NV, W, NINE, P>), dim3(nchunk), dim3(64 * Fac<NV, W, NINE>::NW), 0, s, nic, njc, nlev, ops,
                     rec);
  hipLaunchKernelGGL((cilu_transpose_kernel<NV, W, NINE, P>), dim3(La::nrec(njc), nchunk * La::NG), dim3(256), 0, s, nic,
                     njc, nchunk, rec);
  return reduce_slots_init(store, nl, s);
}

template <int NV, int W, bool NINE, int P>
static void cilu_apply_t(int nic, int njc, int ldi, double* store, const double* b, double* z, bool tr, bool apart,
                         int most, hipStream_t s) {
  using La = Lay<NV, W, NINE, P>;
  const int nchunk = (nic + W - 1) / W;
  const float* rec = reinterpret_cast<const float*>(store + La::links(nchunk, njc));
  unsigned long long* links = reinterpret_cast<unsigned long long*>(store) + kSlotHead;
  const dim3 grid(pass_blocks(nchunk, La::NG)), block(La::NG > 1 ? 256 : 192);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, s, nic, njc, ldi, nchunk, rec, links, most, b, z);
  };
  if constexpr (P == 1) {
    if (apart) {
      launch(tr ? cilu_apply_kernel<NV, W, NINE, P, true, kAscending> : cilu_apply_kernel<NV, W, NINE, P, false, kAscending>);
      launch(tr ? cilu_apply_kernel<NV, W, NINE, P, true, kDescending> : cilu_apply_kernel<NV, W, NINE, P, false, kDescending>);
      return;
    }
  }
  launch(tr ? cilu_apply_kernel<NV, W, NINE, P, true, kBoth> : cilu_apply_kernel<NV, W, NINE, P, false, kBoth>);
}

bool cilu_width_ok(int w) { return w == 8 || w == 16 || w == 24 || w == 32; }

// Lanes per row.  Two make a group's step cheaper, but its columns half as
// many, so there are twice as many groups, and with more groups than CUs some
// share one: 1409x641 (264) 576 us against 442.  One with a launch per pass,
// which is not where the time counts.
template <int NV, int W, bool NINE>
static int cilu_lanes(int nic, bool apart) {
  return !apart && (nic + W - 1) / W * Lay<NV, W, NINE, 2>::NG <= 256 ? 2 : 1;
}
template <int NV, int W, bool NINE>
static size_t cilu_size_w(int nic, int njc, bool apart) {
  return cilu_lanes<NV, W, NINE>(nic, apart) == 2 ? cilu_size_t<NV, W, NINE, 2>(nic, njc)
                                                  : cilu_size_t<NV, W, NINE, 1>(nic, njc);
}
template <int NV, int W, bool NINE, class... T>
static hipError_t cilu_factor_w(bool apart, int nic, T... a) {
  if (cilu_lanes<NV, W, NINE>(nic, apart) == 2) return cilu_factor_t<NV, W, NINE, 2>(nic, a...);
  return cilu_factor_t<NV, W, NINE, 1>(nic, a...);
}
template <int NV, int W, bool NINE>
static void cilu_apply_w(int nic, int njc, int ldi, double* store, const double* b, double* z, bool tr, bool apart,
                         int most, hipStream_t s) {
  if (cilu_lanes<NV, W, NINE>(nic, apart) == 2) cilu_apply_t<NV, W, NINE, 2>(nic, njc, ldi, store, b, z, tr, apart, most, s);
  else cilu_apply_t<NV, W, NINE, 1>(nic, njc, ldi, store, b, z, tr, apart, most, s);
}

template <bool NINE>
static hipError_t cilu_factor_n(int nic, int njc, int ldi, int nv, int w, bool apart, const double* idt,
                                const double* blocks, double* store, hipStream_t s) {
  if (nv == 5) {
    if (w == 8) return cilu_factor_w<5, 8, NINE>(apart, nic, njc, ldi, idt, blocks, store, s);
    if (w == 16) return cilu_factor_w<5, 16, NINE>(apart, nic, njc, ldi, idt, blocks, store, s);
    if (w == 24) return cilu_factor_w<5, 24, NINE>(apart, nic, njc, ldi, idt, blocks, store, s);
    return cilu_factor_w<5, 32, NINE>(apart, nic, njc, ldi, idt, blocks, store, s);
  }
  if (w == 8) return cilu_factor_w<4, 8, NINE>(apart, nic, njc, ldi, idt, blocks, store, s);
  if (w == 16) return cilu_factor_w<4, 16, NINE>(apart, nic, njc, ldi, idt, blocks, store, s);
  if (w == 24) return cilu_factor_w<4, 24, NINE>(apart, nic, njc, ldi, idt, blocks, store, s);
  return cilu_factor_w<4, 32, NINE>(apart, nic, njc, ldi, idt, blocks, store, s);
}

template <bool NINE>
static void cilu_apply_n(int nic, int njc, int ldi, int nv, int w, double* store, const double* b, double* z,
                         bool transpose, bool apart, int most, hipStream_t s) {
  if (nv == 5) {
    if (w == 8) cilu_apply_w<5, 8, NINE>(nic, njc, ldi, store, b, z, transpose, apart, most, s);
    else if (w == 16) cilu_apply_w<5, 16, NINE>(nic, njc, ldi, store, b, z, transpose, apart, most, s);
    else if (w == 24) cilu_apply_w<5, 24, NINE>(nic, njc, ldi, store, b, z, transpose, apart, most, s);
    else cilu_apply_w<5, 32, NINE>(nic, njc, ldi, store, b, z, transpose, apart, most, s);
  } else {
    if (w == 8) cilu_apply_w<4, 8, NINE>(nic, njc, ldi, store, b, z, transpose, apart, most, s);
    else if (w == 16) cilu_apply_w<4, 16, NINE>(nic, njc, ldi, store, b, z, transpose, apart, most, s);
    else if (w == 24) cilu_apply_w<4, 24, NINE>(nic, njc, ldi, store, b, z, transpose, apart, most, s);
    else cilu_apply_w<4, 32, NINE>(nic, njc, ldi, store, b, z, transpose, apart, most, s);
  }
}

template <bool NINE>
static size_t cilu_size_n(int nic, int njc, int nv, int w, bool apart) {
  if (nv == 5)
    return w == 8 ? cilu_size_w<5, 8, NINE>(nic, njc, apart)
                  : w == 16 ? cilu_size_w<5, 16, NINE>(nic, njc, apart)
                            : w == 24 ? cilu_size_w<5, 24, NINE>(nic, njc, apart) : cilu_size_w<5, 32, NINE>(nic, njc, apart);
  return w == 8 ? cilu_size_w<4, 8, NINE>(nic, njc, apart)
                : w == 16 ? cilu_size_w<4, 16, NINE>(nic, njc, apart)
                          : w == 24 ? cilu_size_w<4, 24, NINE>(nic, njc, apart) : cilu_size_w<4, 32, NINE>(nic, njc, apart);
}

size_t cilu_size(int nic, int njc, int nv, int w, bool nine, bool apart) {
  return nine ? cilu_size_n<true>(nic, njc, nv, w, apart) : cilu_size_n<false>(nic, njc, nv, w, apart);
}

hipError_t cilu_factor(int nic, int njc, int ldi, int nv, int w, bool nine, bool apart, const double* idt,
                       const double* blocks, double* store, hipStream_t s) {
  return nine ? cilu_factor_n<true>(nic, njc, ldi, nv, w, apart, idt, blocks, store, s)
              : cilu_factor_n<false>(nic, njc, ldi, nv, w, apart, idt, blocks, store, s);
}

hipError_t cilu_apply(int nic, int njc, int ldi, int nv, int w, bool nine, double* store, const double* b, double* z,
                      bool transpose, bool apart, int polls, hipStream_t s) {
  if (nine) cilu_apply_n<true>(nic, njc, ldi, nv, w, store, b, z, transpose, apart, polls, s);
  else cilu_apply_n<false>(nic, njc, ldi, nv, w, store, b, z, transpose, apart, polls, s);
  return hipGetLastError();
}

}  // namespace sg
