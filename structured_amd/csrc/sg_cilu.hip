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
// up to 6 (nv 5) or 8 (nv 4) columns, twice that on very wide grids, with one
// solving wave each: a column depends on earlier columns only, so the groups
// run as a pipeline, each on its own CU, and hand the solved values of their
// edge columns on through memory.
//
// Factors are stored in FP32 (the preconditioner only has to approximate
// A^-1; FGMRES runs in FP64) in the order the solving waves read them, see
// Lay below.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sg_linalg.hpp"

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
// The apply's neighbours, in the order of their records: lower ones for the
// ascending pass, upper ones for the descending pass, entry n of one being
// the opposite offset of entry n of the other.  0-2 are the column before
// (its oldest, middle and newest solved cell in reach), 3 the cell's own
// column, 4 and 5 the +-2 couplings of the 13-point stencil.
constexpr int Asc[6] = {5, 3, 7, 1, 9, 11};
constexpr int Desc[6] = {8, 4, 6, 2, 10, 12};
constexpr int slot(int di, int dj) {
  for (int s = 0; s < NSLOT; ++s)
    if (Di[s] == di && Dj[s] == dj) return s;
  return -1;
}
}  // namespace ct

// Factorisation, one level after another.  Thread (c, e) holds entry e of
// every stencil block of its cell's row in registers.  A row's lower
// neighbours lie on the four previous levels (L-1 .. L-4), whose factored
// diagonal inverses and upper blocks are kept in an LDS ring, so the level
// loop reads the 13 blocks of its own cells (gathered in level order by
// cilu_gather_kernel) from memory and nothing else; the elimination exchanges
// one 5x5 block per cell through LDS per lower neighbour.

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
  __host__ __device__ static size_t floats(int nchunk, int njc) {
    return (size_t)nchunk * NG * nrec(njc) * (2 * rs(n1) + 2 * rs(n2));
  }
  // float of entry f on a lane inside a record of n floats per lane
  __device__ static unsigned in_record(int n, int lane, int f) {
    const int q = n / 4;
    return f < 4 * q ? (unsigned)((f / 4 * LN + lane) * 4 + (f & 3)) : (unsigned)(4 * q * LN + (f - 4 * q) * LN + lane);
  }
  // words of one link (edge values of one pass, all rows) and of all links
  __host__ __device__ static size_t link(int njc) { return (size_t)njc * GC * NV; }
  static size_t links(int nchunk, int njc) { return 2 * (size_t)nchunk * (NG - 1) * link(njc); }
};

// Zeroes the records that the factorisation does not write, or writes in
// part: steps at both ends of a pass, and groups with absent columns.  One
// block per record.
template <int NV, int W, bool NINE, int P>
__global__ __launch_bounds__(256) void cilu_zero_kernel(int nic, int njc, int nchunk, float* rec) {
  using La = Lay<NV, W, NINE, P>;
  const int t = blockIdx.x, gg = blockIdx.y, s = t - La::X;
  const int wk = min(W, nic - gg / La::NG * W) - gg % La::NG * La::GW;
  if (wk >= La::GW && s >= 2 * (La::GW - 1) && s < njc) return;
  for (int a = 0; a < 4; ++a) {
    const int rs = La::rs(La::count(a));
    float* r = rec + La::array(a, nchunk, njc) + ((size_t)gg * La::nrec(njc) + t) * rs;
    for (int e = threadIdx.x; e < rs; e += 256) r[e] = 0.0f;
  }
}

// Gathers the factorisation's operands into level order: for chunk, level L,
// slot s, block entry e and column c, entry e of the block of I/dt - J in row
// (i0 + c, L - 2c) and neighbour slot s, or zero where the cell or the
// neighbour lies outside the chunk or the grid.  Consecutive columns are
// contiguous, so the factorisation reads a level's operands in runs of W
// doubles.  Read in place, a level's W cells lie on a diagonal of rows 2 ldi
// apart: every 8-byte read took its own line, used again only ~W levels later
// after L2 had evicted it.  Here all levels are gathered at once and the
// levels that share a line are read together.
template <int NV, int W>
__global__ __launch_bounds__(256) void cilu_gather_kernel(int nic, int njc, int ldi, int nlev, const double* idt,
                                                          const double* blocks, double* ops, size_t total) {
  constexpr int B = NV * NV;
  const size_t plane = (size_t)njc * ldi;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
    size_t u = t;
    const int c = (int)(u % W);
    u /= W;
    const int e = (int)(u % B);
    u /= B;
    const int s = (int)(u % NSLOT);
    u /= NSLOT;
    const int L = (int)(u % (size_t)nlev), chunk = (int)(u / (size_t)nlev);
    const int i0 = chunk * W, wk = min(W, nic - i0), j = L - 2 * c;
    const int cn = c + ct::Di[s], jn = j + ct::Dj[s];
    double v = 0.0;
    if (c < wk && j >= 0 && j < njc && cn >= 0 && cn < wk && jn >= 0 && jn < njc) {
      const size_t cell = (size_t)j * ldi + i0 + c;
      v = -blocks[(size_t)(s * B + e) * plane + cell];
      if (s == 0 && e / NV == e % NV) v += idt[cell];
    }
    ops[t] = v;
  }
}

// doubles of the gathered factorisation operands
static size_t cilu_ops_doubles(int nic, int njc, int nv, int w) {
  const int nchunk = (nic + w - 1) / w, nlev = njc + 2 * w - 2;
  return (size_t)nchunk * nlev * NSLOT * nv * nv * w;
}

// A link word that holds no value: a signalling NaN, which no arithmetic
// produces.
constexpr unsigned long long kEmpty = 0x7FF45347454D5054ull;
__global__ __launch_bounds__(256) void cilu_empty_kernel(unsigned long long* x, size_t n) {
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x)
    x[e] = kEmpty;
}

// NINE: ILU(0) on the 3x3-box pattern (the +-2 blocks of A and their fill
// dropped; with the first-order Jacobian of lhs_order 1 those slots hold
// fill only), else on the 13-point stencil.
template <int NV, int W, bool NINE, int P>
__global__ __launch_bounds__(W * NV * NV) void cilu_factor_kernel(int nic, int njc, int nlev, const double* ops,
                                                                  float* rec) {
  using La = Lay<NV, W, NINE, P>;
  constexpr int B = NV * NV, NR = 4, NN = ct::nn<NINE>();
  __shared__ float ring[NR][7][W][B];  // per level: diagonal inverse, then the six upper blocks (ct::Up order)
  __shared__ double Ab[W][B];
  __shared__ double Lb[W][B];
  __shared__ double cb[2][W][NV];
  const int chunk = blockIdx.x, i0 = chunk * W, wk = min(W, nic - i0);
  const int t = threadIdx.x, c = t / B, e = t % B, r = e / NV, q = e % NV;
  // float f of half h of row `row` of cell (cc, jj) in array a
  const int nchunk = gridDim.x, nrec = La::nrec(njc);
  auto put_at = [&](int a, int cc, int jj, int row, int h, int f, float v) {
    const int n = La::count(a), g = cc / La::GW, cl = cc % La::GW;
    const bool asc = a == 0 || a == 2;
    const int c1 = asc ? cl : La::GW - 1 - cl, s = asc ? jj : njc - 1 - jj;
    rec[La::array(a, nchunk, njc) + ((size_t)(chunk * La::NG + g) * nrec + La::X + s + 2 * c1) * La::rs(n) +
        La::in_record(n, P * (c1 * NV + row) + h, f)] = v;
  };
  auto put = [&](int a, int cc, int jj, int row, int n, int qq, float v) {  // neighbour n's entry qq
    put_at(a, cc, jj, row, La::half(n), La::place(n) * NV + qq, v);
  };
  auto put_diag = [&](int a, int cc, int jj, int row, int qq, float v) {
    put_at(a, cc, jj, row, qq / La::ND, La::n1 + qq % La::ND, v);
    // the second half of an odd row ends in a zero
    if (NV % P && qq == NV - 1) put_at(a, cc, jj, row, 1, La::n1 + La::ND - 1, 0.0f);
  };
  auto inside = [&](int cc, int jj) { return cc >= 0 && cc < wk && jj >= 0 && jj < njc; };
  for (int L = 0; L < nlev; ++L) {
    const int j = L - 2 * c;
    const bool valid = inside(c, j);
    // this row's 13 blocks of I/dt - J, gathered in level order (zero where
    // the cell or the neighbour is outside)
    const double* opl = ops + ((size_t)(chunk * nlev + L) * NSLOT * B + e) * W + c;
    double a[NSLOT];
#pragma unroll
    for (int s = 0; s < NSLOT; ++s) a[s] = opl[(size_t)s * B * W];
#pragma unroll
    for (int qi = 0; qi < NN; ++qi) {
      const int s = ct::low<NINE>(qi), di = ct::Di[s], dj = ct::Dj[s];
      const int cn = c + di, jn = j + dj;
      const bool nok = valid && inside(cn, jn);
      const int ln = (L + dj + 2 * di) & (NR - 1);  // the neighbour's level in the ring
      const int cs = nok ? cn : c;
      Ab[c][e] = a[s];
      lds_barrier();
      double l = 0.0;
      if (nok) {
#pragma unroll
        for (int k = 0; k < NV; ++k) l += Ab[c][r * NV + k] * (double)ring[ln][0][cs][k * NV + q];
      }
      a[s] = l;
      Lb[c][e] = l;
      lds_barrier();
      if (nok) {
#pragma unroll
        for (int ui = 0; ui < NN; ++ui) {
          const int ts = ct::up<NINE>(ui);
          const int ri = di + ct::Di[ts], rj = dj + ct::Dj[ts];
          const int su = ct::slot(ri, rj);
          if (su < 0 || (NINE && !ct::in_box(su)) || !inside(c + ri, j + rj)) continue;
          double sum = 0.0;
#pragma unroll
          for (int k = 0; k < NV; ++k) sum += Lb[c][r * NV + k] * (double)ring[ln][1 + ui][cs][k * NV + q];
          a[su] -= sum;
        }
      }
    }
    // the level's L and U blocks are final: store them (records of both
    // directions and ring).  A block goes to its own row's record and,
    // transposed, to that of the neighbour it couples to; absent neighbours
    // leave zeros in this cell's own records.
    const int lr = L & (NR - 1);
    if (valid) {
#pragma unroll
      for (int n = 0; n < NN; ++n) {
        const int sl = ct::Asc[n], su = ct::Desc[n];
        put(0, c, j, r, n, q, (float)a[sl]);
        put(1, c, j, r, n, q, (float)a[su]);
        const int cl = c + ct::Di[sl], jl = j + ct::Dj[sl], cu = c + ct::Di[su], ju = j + ct::Dj[su];
        const bool lok = inside(cl, jl), uok = inside(cu, ju);
        if (lok) put(3, cl, jl, q, n, r, (float)a[sl]);
        else put(2, c, j, q, n, r, 0.0f);
        if (uok) put(2, cu, ju, q, n, r, (float)a[su]);
        else put(3, c, j, q, n, r, 0.0f);
      }
    }
#pragma unroll
    for (int ui = 0; ui < NN; ++ui) ring[lr][1 + ui][c][e] = valid ? (float)a[ct::up<NINE>(ui)] : 0.0f;
    // inverse of the factored diagonal block: Gauss-Jordan with partial
    // pivoting on [D | I], column-parallel (thread e < 2 NV of a cell owns
    // column e; the pivot column is broadcast through LDS each step)
    Ab[c][e] = a[0];
    lds_barrier();
    double col[NV];
#pragma unroll
    for (int rr = 0; rr < NV; ++rr) col[rr] = (e < NV) ? Ab[c][rr * NV + e] : ((e - NV == rr) ? 1.0 : 0.0);
#pragma unroll
    for (int p = 0; p < NV; ++p) {
      if (e == p) {
#pragma unroll
        for (int rr = 0; rr < NV; ++rr) cb[p & 1][c][rr] = col[rr];
      }
      lds_barrier();
      double cp[NV];
#pragma unroll
      for (int rr = 0; rr < NV; ++rr) cp[rr] = cb[p & 1][c][rr];
      int piv = p;
      double best = fabs(cp[p]);
#pragma unroll
      for (int rr = p + 1; rr < NV; ++rr) {
        const double v = fabs(cp[rr]);
        if (v > best) { best = v; piv = rr; }
      }
#pragma unroll
      for (int rr = p + 1; rr < NV; ++rr) {
        const bool sw = piv == rr;
        const double x = cp[p], y = cp[rr], u = col[p], w = col[rr];
        cp[p] = sw ? y : x; cp[rr] = sw ? x : y;
        col[p] = sw ? w : u; col[rr] = sw ? u : w;
      }
      const double ip = 1.0 / cp[p];
      col[p] *= ip;
#pragma unroll
      for (int rr = 0; rr < NV; ++rr) {
        if (rr == p) continue;
        const double f = cp[rr];
        col[rr] = (f != 0.0) ? col[rr] - f * col[p] : col[rr];
      }
    }
    if (e >= NV && e < 2 * NV) {
#pragma unroll
      for (int rr = 0; rr < NV; ++rr) Lb[c][rr * NV + e - NV] = col[rr];
    }
    lds_barrier();
    const float dinv = valid ? (float)Lb[c][e] : 0.0f;
    if (valid) {
      put_diag(1, c, j, r, q, dinv);
      put_diag(2, c, j, q, r, dinv);
    }
    ring[lr][0][c][e] = dinv;
  }
}

// LDS of one group's work-group: the solved values of the last kRing steps by
// step, column and component (edge columns first; idle lanes store to the
// column after the last), the right-hand sides of the steps to come, and how
// far each wave has got.
constexpr int kRing = 64;
template <int NV, int W, bool NINE, int P>
struct ApplyLds {
  using La = Lay<NV, W, NINE, P>;
  static constexpr int NVP = (NV + 1) & ~1;  // a cell's values, in 16-byte units
  static constexpr int NP = La::GCX + La::GW;
  double ring[kRing][NP + 1][NVP] __attribute__((aligned(16)));
  double x[kRing][La::ROWS + 1];  // the last place is always zero
  double tmp[La::GW + 1][8] __attribute__((aligned(16)));  // a row's halves at 0 and 4
  // per pass: steps solved, right-hand-side rows loaded, edge rows received,
  // rows taken out of the ring, rows whose stores are complete
  int step[2], loaded[2], edges[2], taken[2], stored[2];
};
__device__ __forceinline__ int lds_read(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_write(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_release() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local"); }
__device__ __forceinline__ void lds_acquire() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local"); }
// Orders this wave's LDS accesses (a wave's LDS operations execute in issue
// order, so nothing is waited for).
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}

constexpr int kAll = 1 << 29;  // a count that never holds the solving wave up
// Polls without a new row before a link gives up (each takes about a
// microsecond, so several seconds).  The groups of a chunk are dispatched
// one after another, so the one that fills a link runs or has run, and the
// wait ends.
constexpr int kLinkPolls = 1 << 22;

// The receiving wave of one pass: moves the edge rows the group before
// publishes into the ring.  One poll reads as many rows as fit the wave; a
// word is read as one 64-bit atomic and holds either a value or kEmpty, so
// nothing has to be ordered between words.
template <int NV, int W, bool NINE, int P>
__device__ void cilu_receive(unsigned long long* in, int njc, ApplyLds<NV, W, NINE, P>& sh, int pass) {
  using La = Lay<NV, W, NINE, P>;
  constexpr int EN = La::GCX * NV, RP = 64 / EN;
  const int lane = threadIdx.x & 63, rr = lane / EN, gi = lane % EN / NV, k = lane % NV;
  int n = 0, polls = 0;
  while (n < njc) {
    // edge column gi's row s belongs to step s + X - 2 (1 + gi); its place
    // holds a value that is read up to three steps after its own
    const int row = n + rr, free = lds_read(&sh.step[pass]) + kRing - 8 - La::X;
    unsigned long long v = kEmpty;
    if (rr < RP && row < njc && row < free)
      v = __hip_atomic_load(in + (size_t)row * EN + lane % EN, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long missing = ~__ballot(v != kEmpty);
    const int rows = min(RP, (missing ? __builtin_ctzll(missing) : 64) / EN);
    if (rows == 0) {
      if (n < free && ++polls > kLinkPolls) break;  // a full ring is no failure
      continue;
    }
    polls = 0;
    if (rr < rows)
      sh.ring[(row + La::X - 2 * (1 + gi)) & (kRing - 1)][La::GCX - 1 - gi][k] = __longlong_as_double((long long)v);
    n += rows;
    lds_release();
    if (lane == 0) lds_write(&sh.edges[pass], n < njc ? n : kAll);
  }
  if (n < njc) {  // never filled: every value that depends on it becomes NaN
    for (int e = lane; e < kRing * EN; e += 64) sh.ring[e / EN][e % EN / NV][e % NV] = __builtin_nan("");
    lds_release();
    if (lane == 0) lds_write(&sh.edges[pass], kAll);
  }
}

// The storing wave of one pass: takes finished rows out of the ring, stores
// them to z (a row is contiguous in memory, a step's cells are not) and
// publishes the edge columns for the next group.  In the solving wave these
// stores held up the loads, whose waits run in issue order.
template <int NV, int W, bool NINE, int P, bool ASC>
__device__ void cilu_store(double* z, int njc, int ldi, size_t plane, int col0, int wk, unsigned long long* out,
                           ApplyLds<NV, W, NINE, P>& sh, int pass) {
  using La = Lay<NV, W, NINE, P>;
  constexpr int LAST = La::X + 2 * (La::GW - 1), RB = 4;
  const int lane = threadIdx.x & 63, k = lane % NV, c1 = lane / NV, c = ASC ? c1 : La::GW - 1 - c1;
  const int gi = La::GW - 1 - c1;
  const bool live = c1 < La::GW && c < wk, pub = out && c1 < La::GW && gi < La::GC;
  double* zl = z + (size_t)k * plane + col0 + (live ? c : 0);
  for (int n = 0; n < njc;) {
    const int rows = min(min(lds_read(&sh.step[pass]) - LAST, njc) - n, RB);
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
    for (int r = 0; r < RB; ++r) {
      if (r >= rows) break;
      if (pub)
        __hip_atomic_store(out + ((size_t)(n + r) * La::GCX + gi) * NV + k, (unsigned long long)__double_as_longlong(v[r]),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (live) zl[(size_t)(ASC ? n + r : njc - 1 - n - r) * ldi] = v[r];
    }
    n += rows;
    lds_release();
    if (lane == 0) lds_write(&sh.taken[pass], n < njc ? n : kAll);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  if (lane == 0) lds_write(&sh.stored[pass], 1);
}

// The loading wave of one pass: brings the right-hand sides into LDS by step
// (a row's cells belong to steps two apart), LB rows at a time and one batch
// ahead, and reads one word of every 128-byte line of the records 16 to 32
// steps ahead of the solving wave, so that its loads find them in the XCD's
// L2 instead of memory (much further ahead, the groups of an XCD overflow it).
template <int NV, int W, bool NINE, int P, bool ASC, bool DIAG>
__device__ void cilu_load(const float* R, int njc, int ldi, size_t plane, int col0, int wk, const double* src,
                          ApplyLds<NV, W, NINE, P>& sh, int pass) {
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
      while (lds_read(&sh.step[pass]) < La::X + s1 + LB - 1 + TAIL + 1 - kRing) __builtin_amdgcn_s_sleep(2);
#pragma unroll
      for (int u = 0; u < LB; ++u)
        if (lane < La::ROWS) sh.x[(La::X + s1 + u + 2 * c1) & (kRing - 1)][lane] = live && s1 + u < njc ? v[b][u] : 0.0;
      lds_release();
      if (lane == 0) lds_write(&sh.loaded[pass], s1 + LB);
    }
  }
  if (lane == 0) lds_write(&sh.loaded[pass], kAll);
}

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00027000);
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
__device__ __forceinline__ void cilu_solve_pairs(const float* R, int njc, ApplyLds<NV, W, NINE, 2>& sh, int pass, bool up) {
  using La = Lay<NV, W, NINE, 2>;
  using A = ApplyLds<NV, W, NINE, 2>;
  constexpr int N = DIAG ? La::n2 : La::n1, RS = La::rs(N), NQ = N / 4, NREM = N % 4, PD = La::pd(N), UN = La::UN, ND = La::ND;
  static_assert(kRing % UN == 0 && UN % PD == 0, "a block does not wrap around the ring");
  const int lane = threadIdx.x & 63, h = lane & 1, row = min(lane >> 1, La::ROWS), k = row % NV, c1 = row / NV;
  const bool real = row < La::ROWS;
  const int pos = La::GCX + (real ? c1 : 0), wpos = real ? pos : A::NP;
  const int xrow = h ? La::ROWS : row, tk = k / ND * 4 + k % ND;  // the right-hand side is taken once
  const int T = La::steps(njc), rl = min(lane, La::LN - 1);
  const auto rrec = buffer_of(R, (size_t)La::nrec(njc) * RS * sizeof(float));
  const unsigned oq = rl * 16, or_ = (4 * NQ * La::LN + rl) * 4;
  u32x4 fq[PD][NQ > 0 ? NQ : 1];
  unsigned fr[PD][NREM > 0 ? NREM : 1];
  // the record's part that is used first is loaded last, so that one wait
  // covers the record
  int so = 0;
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
      const int a = lds_read(&sh.loaded[pass]) + La::X - 1, b = up ? lds_read(&sh.edges[pass]) + 1 : kAll;
      const int c = lds_read(&sh.taken[pass]) + kRing + La::X;
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
      if (u & 1) lds_write(&sh.step[pass], t + 1);
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
__device__ __forceinline__ void cilu_solve_rows(const float* R, int njc, ApplyLds<NV, W, NINE, 1>& sh, int pass, bool up) {
  using La = Lay<NV, W, NINE, 1>;
  using A = ApplyLds<NV, W, NINE, 1>;
  constexpr int N = DIAG ? La::n2 : La::n1, RS = La::rs(N), NQ = N / 4, NREM = N % 4, PD = La::pd(N), UN = La::UN;
  static_assert(kRing % UN == 0 && UN % PD == 0, "a block does not wrap around the ring");
  const int lane = threadIdx.x & 63, row = min(lane, La::ROWS), k = row % NV, c1 = row / NV;
  const bool real = row < La::ROWS;
  const int pos = La::GCX + (real ? c1 : 0), wpos = real ? pos : A::NP;
  const int T = La::steps(njc), rl = min(lane, La::LN - 1);
  const auto rrec = buffer_of(R, (size_t)La::nrec(njc) * RS * sizeof(float));
  const unsigned oq = rl * 16, or_ = (4 * NQ * La::LN + rl) * 4;
  u32x4 fq[PD][NQ > 0 ? NQ : 1];
  unsigned fr[PD][NREM > 0 ? NREM : 1];
  int so = 0;
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
      const int a = lds_read(&sh.loaded[pass]) + La::X - 1, b = up ? lds_read(&sh.edges[pass]) + 1 : kAll;
      const int c = lds_read(&sh.taken[pass]) + kRing + La::X;
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
      if (u & 1) lds_write(&sh.step[pass], t + 1);
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
__device__ __forceinline__ void cilu_solve(const float* R, int njc, ApplyLds<NV, W, NINE, P>& sh, int pass, bool up) {
  if constexpr (P == 2) cilu_solve_pairs<NV, W, NINE, DIAG>(R, njc, sh, pass, up);
  else cilu_solve_rows<NV, W, NINE, DIAG>(R, njc, sh, pass, up);
}

// z = (LU)^-1 b, or (LU)^-T b when TR.  Wave 0 of a work-group solves one
// column group, wave 1 loads and wave 2 stores for it, and wave 3 receives
// the edge columns of the group before where a chunk has several.
// Work-groups are dealt to the XCDs round-robin by index: the groups of a
// chunk sit on one XCD, consecutive in its order, so a group's neighbours are
// dispatched with it.
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
template <int NV, int W, bool NINE, int P, bool TR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void cilu_apply_kernel(
    int nic, int njc, int ldi, int nchunk, const float* rec, unsigned long long* links, const double* b, double* z) {
  using La = Lay<NV, W, NINE, P>;
  __shared__ ApplyLds<NV, W, NINE, P> sh;
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int chunk = slot / La::NG * 8 + xcd, g = slot % La::NG;
  if (chunk >= nchunk) return;
  const int i0 = chunk * W, wk = min(W, nic - i0) - g * La::GW;  // columns from this group on
  if (wk <= 0) return;
  const bool left = g > 0, right = wk > La::GW;
  // values of steps not yet solved, and the place after an odd row's last
  // entry, meet zero factors: they need to be finite
  double* zero = &sh.ring[0][0][0];
  for (int e = threadIdx.x; e < (int)(sizeof(sh.ring) / sizeof(double)); e += blockDim.x) zero[e] = 0.0;
  for (int e = threadIdx.x; e < (int)(sizeof(sh.tmp) / sizeof(double)); e += blockDim.x) (&sh.tmp[0][0])[e] = 0.0;
  if (threadIdx.x < 2) {
    sh.step[threadIdx.x] = sh.edges[threadIdx.x] = sh.taken[threadIdx.x] = sh.stored[threadIdx.x] = 0;
    sh.loaded[threadIdx.x] = -La::X;  // not even the steps before the first row may start
  }
  __syncthreads();
  const size_t plane = (size_t)njc * ldi, gr = (size_t)(chunk * La::NG + g) * La::nrec(njc);
  const float* R1 = rec + La::array(TR ? 2 : 0, nchunk, njc) + gr * La::rs(TR ? La::n2 : La::n1);
  const float* R2 = rec + La::array(TR ? 3 : 1, nchunk, njc) + gr * La::rs(TR ? La::n1 : La::n2);
  const int col0 = i0 + g * La::GW, wg = min(wk, La::GW);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // link l of a pass joins groups l and l + 1
  const size_t lw = La::link(njc);
  unsigned long long* la = links + (size_t)chunk * (La::NG - 1) * lw;
  unsigned long long* ld = la + (size_t)nchunk * (La::NG - 1) * lw;
  // non-transposed: unit-lower L ascending, then D + U descending;
  // transposed: (D + U)^T ascending, then unit-lower L^T descending
  if (wave == 0) {
    cilu_solve<NV, W, NINE, P, TR>(R1, njc, sh, 0, left);
    cilu_solve<NV, W, NINE, P, !TR>(R2, njc, sh, 1, right);
  } else if (wave == 1) {
    cilu_load<NV, W, NINE, P, true, TR>(R1, njc, ldi, plane, col0, wg, b, sh, 0);
    // the second pass loads what the first stored, and reuses its LDS
    while (!lds_read(&sh.stored[0]) || lds_read(&sh.step[0]) < La::steps(njc)) __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    cilu_load<NV, W, NINE, P, false, !TR>(R2, njc, ldi, plane, col0, wg, z, sh, 1);
  } else if (wave == 2) {
    cilu_store<NV, W, NINE, P, true>(z, njc, ldi, plane, col0, wg, right ? la + g * lw : nullptr, sh, 0);
    cilu_store<NV, W, NINE, P, false>(z, njc, ldi, plane, col0, wg, left ? ld + (g - 1) * lw : nullptr, sh, 1);
  } else {
    if (left) cilu_receive<NV, W, NINE, P>(la + (g - 1) * lw, njc, sh, 0);
    if (right) {
      // the first pass is done with the edge columns' places
      while (lds_read(&sh.step[0]) < La::steps(njc)) __builtin_amdgcn_s_sleep(1);
      cilu_receive<NV, W, NINE, P>(ld + g * lw, njc, sh, 1);
    }
    // the links are empty for the next apply
    for (size_t e = threadIdx.x & 63; e < lw; e += 64) {
      if (left) __hip_atomic_store(la + (g - 1) * lw + e, kEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (right) __hip_atomic_store(ld + g * lw + e, kEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

template <int NV, int W, bool NINE, int P>
static size_t cilu_size_t(int nic, int njc) {
  using La = Lay<NV, W, NINE, P>;
  const int nchunk = (nic + W - 1) / W;
  return (La::floats(nchunk, njc) + 1) / 2 + La::links(nchunk, njc) + cilu_ops_doubles(nic, njc, NV, W);
}

template <int NV, int W, bool NINE, int P>
static void cilu_factor_t(int nic, int njc, int ldi, const double* idt, const double* blocks, double* store,
                          hipStream_t s) {
  using La = Lay<NV, W, NINE, P>;
  const int nchunk = (nic + W - 1) / W, nlev = njc + 2 * W - 2;
  const size_t total = cilu_ops_doubles(nic, njc, NV, W), nl = La::links(nchunk, njc);
  double* links = store + (La::floats(nchunk, njc) + 1) / 2;
  double* ops = links + nl;
  hipLaunchKernelGGL((cilu_zero_kernel<NV, W, NINE, P>), dim3(La::nrec(njc), nchunk * La::NG), dim3(256), 0, s, nic, njc,
                     nchunk, reinterpret_cast<float*>(store));
  const size_t nblk = std::min<size_t>((total + 255) / 256, (size_t)1 << 20);
  hipLaunchKernelGGL((cilu_gather_kernel<NV, W>), dim3((unsigned)nblk), dim3(256), 0, s, nic, njc, ldi, nlev, idt,
                     blocks, ops, total);
  hipLaunchKernelGGL((cilu_factor_kernel<NV, W, NINE, P>), dim3(nchunk), dim3(W * NV * NV), 0, s, nic, njc, nlev, ops,
                     reinterpret_cast<float*>(store));
  if (nl)
    hipLaunchKernelGGL(cilu_empty_kernel, dim3((unsigned)std::min<size_t>((nl + 255) / 256, 1024)), dim3(256), 0, s,
                       reinterpret_cast<unsigned long long*>(links), nl);
}

template <int NV, int W, bool NINE, int P>
static void cilu_apply_t(int nic, int njc, int ldi, double* store, const double* b, double* z, bool tr,
                         hipStream_t s) {
  using La = Lay<NV, W, NINE, P>;
  const int nchunk = (nic + W - 1) / W;
  const float* rec = reinterpret_cast<const float*>(store);
  unsigned long long* links = reinterpret_cast<unsigned long long*>(store + (La::floats(nchunk, njc) + 1) / 2);
  const dim3 grid((nchunk + 7) / 8 * 8 * La::NG), block(La::NG > 1 ? 256 : 192);
  if (tr)
    hipLaunchKernelGGL((cilu_apply_kernel<NV, W, NINE, P, true>), grid, block, 0, s, nic, njc, ldi, nchunk, rec, links, b,
                       z);
  else
    hipLaunchKernelGGL((cilu_apply_kernel<NV, W, NINE, P, false>), grid, block, 0, s, nic, njc, ldi, nchunk, rec, links,
                       b, z);
}

bool cilu_width_ok(int w) { return w == 8 || w == 16 || w == 24 || w == 32; }

// Lanes per row.  Two make a group's step cheaper, but its columns half as
// many, so there are twice as many groups, and with more groups than CUs some
// share one: 1409x641 (270) 576 us against 450.
template <int NV, int W, bool NINE>
static int cilu_lanes(int nic) {
  return (nic + W - 1) / W * Lay<NV, W, NINE, 2>::NG <= 256 ? 2 : 1;
}
template <int NV, int W, bool NINE>
static size_t cilu_size_w(int nic, int njc) {
  return cilu_lanes<NV, W, NINE>(nic) == 2 ? cilu_size_t<NV, W, NINE, 2>(nic, njc) : cilu_size_t<NV, W, NINE, 1>(nic, njc);
}
template <int NV, int W, bool NINE, class... T>
static void cilu_factor_w(int nic, T... a) {
  if (cilu_lanes<NV, W, NINE>(nic) == 2) cilu_factor_t<NV, W, NINE, 2>(nic, a...);
  else cilu_factor_t<NV, W, NINE, 1>(nic, a...);
}
template <int NV, int W, bool NINE, class... T>
static void cilu_apply_w(int nic, T... a) {
  if (cilu_lanes<NV, W, NINE>(nic) == 2) cilu_apply_t<NV, W, NINE, 2>(nic, a...);
  else cilu_apply_t<NV, W, NINE, 1>(nic, a...);
}

template <bool NINE>
static void cilu_factor_n(int nic, int njc, int ldi, int nv, int w, const double* idt, const double* blocks,
                          double* store, hipStream_t s) {
  if (nv == 5) {
    if (w == 8) cilu_factor_w<5, 8, NINE>(nic, njc, ldi, idt, blocks, store, s);
    else if (w == 16) cilu_factor_w<5, 16, NINE>(nic, njc, ldi, idt, blocks, store, s);
    else if (w == 24) cilu_factor_w<5, 24, NINE>(nic, njc, ldi, idt, blocks, store, s);
    else cilu_factor_w<5, 32, NINE>(nic, njc, ldi, idt, blocks, store, s);
  } else {
    if (w == 8) cilu_factor_w<4, 8, NINE>(nic, njc, ldi, idt, blocks, store, s);
    else if (w == 16) cilu_factor_w<4, 16, NINE>(nic, njc, ldi, idt, blocks, store, s);
    else if (w == 24) cilu_factor_w<4, 24, NINE>(nic, njc, ldi, idt, blocks, store, s);
    else cilu_factor_w<4, 32, NINE>(nic, njc, ldi, idt, blocks, store, s);
  }
}

template <bool NINE>
static void cilu_apply_n(int nic, int njc, int ldi, int nv, int w, double* store, const double* b, double* z,
                         bool transpose, hipStream_t s) {
  if (nv == 5) {
    if (w == 8) cilu_apply_w<5, 8, NINE>(nic, njc, ldi, store, b, z, transpose, s);
    else if (w == 16) cilu_apply_w<5, 16, NINE>(nic, njc, ldi, store, b, z, transpose, s);
    else if (w == 24) cilu_apply_w<5, 24, NINE>(nic, njc, ldi, store, b, z, transpose, s);
    else cilu_apply_w<5, 32, NINE>(nic, njc, ldi, store, b, z, transpose, s);
  } else {
    if (w == 8) cilu_apply_w<4, 8, NINE>(nic, njc, ldi, store, b, z, transpose, s);
    else if (w == 16) cilu_apply_w<4, 16, NINE>(nic, njc, ldi, store, b, z, transpose, s);
    else if (w == 24) cilu_apply_w<4, 24, NINE>(nic, njc, ldi, store, b, z, transpose, s);
    else cilu_apply_w<4, 32, NINE>(nic, njc, ldi, store, b, z, transpose, s);
  }
}

template <bool NINE>
static size_t cilu_size_n(int nic, int njc, int nv, int w) {
  if (nv == 5)
    return w == 8 ? cilu_size_w<5, 8, NINE>(nic, njc)
                  : w == 16 ? cilu_size_w<5, 16, NINE>(nic, njc)
                            : w == 24 ? cilu_size_w<5, 24, NINE>(nic, njc) : cilu_size_w<5, 32, NINE>(nic, njc);
  return w == 8 ? cilu_size_w<4, 8, NINE>(nic, njc)
                : w == 16 ? cilu_size_w<4, 16, NINE>(nic, njc)
                          : w == 24 ? cilu_size_w<4, 24, NINE>(nic, njc) : cilu_size_w<4, 32, NINE>(nic, njc);
}

size_t cilu_size(int nic, int njc, int nv, int w, bool nine) {
  return nine ? cilu_size_n<true>(nic, njc, nv, w) : cilu_size_n<false>(nic, njc, nv, w);
}

hipError_t cilu_factor(int nic, int njc, int ldi, int nv, int w, bool nine, const double* idt, const double* blocks,
                       double* store, hipStream_t s) {
  if (nine) cilu_factor_n<true>(nic, njc, ldi, nv, w, idt, blocks, store, s);
  else cilu_factor_n<false>(nic, njc, ldi, nv, w, idt, blocks, store, s);
  return hipGetLastError();
}

hipError_t cilu_apply(int nic, int njc, int ldi, int nv, int w, bool nine, double* store, const double* b, double* z,
                      bool transpose, hipStream_t s) {
  if (nine) cilu_apply_n<true>(nic, njc, ldi, nv, w, store, b, z, transpose, s);
  else cilu_apply_n<false>(nic, njc, ldi, nv, w, store, b, z, transpose, s);
  return hipGetLastError();
}

}  // namespace sg
