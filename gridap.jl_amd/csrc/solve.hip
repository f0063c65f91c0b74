// FP64 SpMV and preconditioned CG on the assembled matrix.
//
// Gridap solves AffineFEOperators with a direct LU (src/Algebra/LinearSolvers.jl:
// 249-274); this engine keeps the matrix in HBM and runs CG instead.  The matrix
// is symmetric (the assembled forms are), so the CSC arrays are read as CSR rows.
//
// One iteration is two kernels with a diagonal (or no) preconditioner and three
// with the factored FSAI preconditioner M = GᵀG:
//   spmv_dir      p' = z + β p and q = A p' in one pass (p' of the neighbours is
//                 formed on the fly from z and p), partials of p'·q;
//   update        x += α p', r -= α q, z = M r, partials of r·z and r·r  (diagonal M);
//   update_lower  x += α p', r' = r - α q, y = G r' (r' of the neighbours formed on
//                 the fly from r and q; r double-buffered), partials of r'·r';
//   upper_rz      z = Gᵀ y, partials of r'·z;
// G and Gᵀ are read from the solver's 16-slot row copy (weights with D^-1/2
// folded in, column indices), written with the factor.  When the free dofs form a
// full box of Q1 lattice nodes, the same iteration runs on stencil kernels with no
// column indices: A as 14 offset arrays (lower half, the upper mirrored), G as 14, Gᵀ read
// from G's arrays at the mirrored offsets.  Small systems (solve_small.hip) and boxes that
// fit the device's registers (solve_resident.hip) are solved in one launch instead.
// Reductions are deterministic and need no grid-wide synchronisation: a kernel
// writes one partial per block, and every block of the consuming kernel sums all
// of them in index order at its start (the same value everywhere); block 0 of
// spmv_dir publishes r·z for the next iteration's β.  The host sums the r·r
// partials itself at the convergence checks.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <mutex>

#include "gh_internal.h"

namespace gh {
namespace {

constexpr int kBlock = 512;
constexpr int kMaxParts = 1024;  // partial slots per reduced quantity (max blocks per grid)
constexpr int kApplyLanes = 4;   // lanes per row in the FSAI applications

// scalar slots
constexpr int kRz = 0;  // [0..1]: r·z, double-buffered by iteration parity
// convergence decided on the device: kStop = 0 (running), 1 (r·r met the threshold),
// 2 (r·r not finite); kStopIt = the iteration at whose start it was decided
constexpr int kStop = 5, kStopIt = 6, kBad = 7;

// One partial per block: part[blockIdx.x] = Σ_block v, for up to four quantities with one
// barrier (wave sums inside the vector unit, the wave sums by the first wave).
template <int N>
__device__ __forceinline__ void put_partials(const double (&v)[N], double *const (&part)[N]) {
  static_assert(N <= 4 && kBlock / 64 <= 16, "a row of 16 lanes per quantity");
  __shared__ double sums[N][16];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const double s = wave_sum(v[k]);
    if (lane == 0) sums[k][w] = s;
  }
  __syncthreads();
  if (w != 0) return;
  const int q = lane >> 4, i = lane & 15;
  const double s = row16_sum(q < N && i < kBlock / 64 ? sums[q < N ? q : 0][i] : 0.0);
#pragma unroll
  for (int k = 0; k < N; ++k)
    if (lane == 16 * k + 15) part[k][blockIdx.x] = s;
}
__device__ __forceinline__ void put_partial(double v, double *part) {
  const double a[1] = {v};
  double *const p[1] = {part};
  put_partials(a, p);
}

// Grids of the iteration kernels are capped at kPcgGrid blocks (grid-stride loops):
// every block of a consuming kernel re-reads all partials of its producer, so the
// partial count, not only the row count, sets the cost of a reduction.
constexpr int kPcgGrid = 1024;
static_assert(kPcgGrid <= kMaxParts, "partial slots");

// The loads an iteration kernel starts with, issued together: the stop flag and this
// thread's share of one or two partial arrays.  The kernel issues its first data loads
// next, so they are in flight while the reduction below runs: an iteration kernel of a
// small system is a chain of memory round trips (about 1 µs each), not bandwidth.
struct StartIn {
  double a = 0.0, b = 0.0, stop = 0.0;
};

__device__ __forceinline__ StartIn start_loads(const double *scal, const double *__restrict__ pa,
                                               const double *__restrict__ pb, int np) {
  constexpr int kPer = (kPcgGrid + kBlock - 1) / kBlock;  // partials per thread
  StartIn S;
  double va[kPer], vb[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int k = (int)threadIdx.x + u * kBlock;
    va[u] = k < np ? pa[k] : 0.0;
    vb[u] = pb && k < np ? pb[k] : 0.0;
  }
  S.stop = scal[kStop];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    S.a += va[u];
    S.b += vb[u];
  }
  return S;
}

// Σ of both partial arrays (fixed order, the same in every block) into S.a, S.b; true
// when an earlier kernel stopped the solve.  Thread 0's flag decides for the block.
// One barrier; sh holds 2 x kBlock/64 + 1 values and is reused by later reductions.
__device__ __forceinline__ bool start_sums(StartIn &S, double *sh) {
  constexpr int kW = kBlock / 64;
  static_assert(kW <= 16, "a row of 16 lanes per quantity");
  const double a = wave_sum(S.a), b = wave_sum(S.b);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    sh[w] = a;
    sh[kW + w] = b;
  }
  if (threadIdx.x == 0) sh[2 * kW] = S.stop;
  __syncthreads();
  const int q = lane >> 4, i = lane & 15;
  const double v = row16_sum(q < 2 && i < kW ? sh[kW * (q & 1) + i] : 0.0);
  S.a = lane_value(v, 15);
  S.b = lane_value(v, 31);
  return sh[2 * kW] != 0.0;
}
constexpr int kStartLds = 2 * (kBlock / 64) + 1;

// Convergence at the start of an iteration (after the first of a start): r·r of the
// previous update against thr = (rtol ‖b‖)²; true when the solve stops here (block 0
// records why and at which iteration).  Every block has summed the same partials in the
// same order, so every block takes the same decision.
// news (a word of pinned host memory, or null): the iteration that has begun, and
// kStopped when it is the one that stops.
constexpr uint64_t kStopped = uint64_t(1) << 32;
__device__ __forceinline__ bool iteration_stops(double *scal, uint64_t *news, double rr, int first,
                                                double thr, int it) {
  const bool stop = !first && (!(rr > thr) || !isfinite(rr));
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (stop) {
      scal[kStop] = isfinite(rr) ? 1.0 : 2.0;
      scal[kStopIt] = (double)it;
    }
    if (news)
      __hip_atomic_store(news, (stop ? kStopped : 0) | (uint32_t)it, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
  }
  return stop;
}

// Workgroups of the stencil product: two on each of 256 compute units, or one.  µs an
// iteration with 1024, 512 and 256: 84³ -, 26.9 and 29.5; 100³ 44.6, 42.4 and -; 160² x 50
// -, 55.8 and 56.7; 110³ -, 53.9 and 52.8; 140² x 80 -, 70.9 and 64.2; 128³ 98.0, 95.2 and 93.3.
constexpr unsigned kStencilGrid = 512;

inline unsigned grid_rows(int64_t rows, int rows_per_block) {
  return (unsigned)std::min<int64_t>(
      std::max<int64_t>((rows + rows_per_block - 1) / rows_per_block, 1), kPcgGrid);
}

// ---- CSR rows --------------------------------------------------------------------------
// L lanes take a row together, U entries per lane and turn (a turn is L·U consecutive
// entries: coalesced values and column indices, all loads of a turn in flight before the
// first is used).  L and U follow the mean row length (row_shape): one turn covers most
// rows, and a wave holds 64 / L rows, so short rows leave few lanes idle and long ones
// are no chain of dependent turns.  Eight lanes and one entry at a time, as before: 612 µs
// at 184 entries a row (vector Q2, 32³, 1.81 GB), 50 µs at 28 (P2, 40³ x 6 tetrahedra);
// now 385 µs (4.7 TB/s) and 31 µs.
// The SpMV runs one workgroup per tile of rows, however many (vector Q2: 451 µs with 4096
// workgroups, 385 µs with 50,700); the solver's kernels stay at kPcgGrid, whose partials
// every block re-reads.  Tiles go round-robin over the XCDs: the numbering puts the
// vertex dofs, whose rows are the longest, first, and contiguous slabs gave one XCD
// twice the work (P2: 79 µs).
template <int L, int U>
struct RowTurn {
  int32_t col[U];
  double v[U];
  int32_t left;  // entries of the row from this lane's first one on
  // entries p0 + sub + L·u of [.., p1); past the end: the row's last entry, for drop or add
  __device__ __forceinline__ void load(const int32_t *__restrict__ rv,
                                       const double *__restrict__ val, int32_t p0, int32_t p1) {
    const int32_t p = p0 + (int32_t)(threadIdx.x % L);
    left = p1 - p;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int32_t k = max(p + min(u * L, left - 1), 0);
      col[u] = rv[k];
      v[u] = val[k];
    }
  }
  // Weight 0 past the end: for finite vectors.
  __device__ __forceinline__ void drop() {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u * L >= left) v[u] = 0.0;
  }
  // s + entry u times g, for any g (0 times an infinite one would be NaN).
  __device__ __forceinline__ double add(double s, int u, double g) const {
    const double t = s + v[u] * g;
    return u * L < left ? t : s;
  }
};

template <int L>
__device__ __forceinline__ double row_sum(double s) {
#pragma unroll
  for (int o = L / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
  return s;
}

// y = A x (rows from the CSC of a symmetric A).
template <int L, int U>
__global__ __launch_bounds__(kBlock) void spmv_kernel(int n,
                                                      const int32_t *__restrict__ cp,
                                                      const int32_t *__restrict__ rv,
                                                      const double *__restrict__ val,
                                                      const double *__restrict__ x,
                                                      double *__restrict__ y) {
  const int row = blockIdx.x * (kBlock / L) + (int)threadIdx.x / L;
  double s = 0.0;
  if (row < n) {
    const int32_t p1 = cp[row + 1];
    for (int32_t p = cp[row]; p < p1; p += L * U) {
      RowTurn<L, U> R;
      R.load(rv, val, p, p1);
      double g[U];
#pragma unroll
      for (int u = 0; u < U; ++u) g[u] = x[R.col[u]];
#pragma unroll
      for (int u = 0; u < U; ++u) s = R.add(s, u, g[u]);
    }
  }
  s = row_sum<L>(s);
  if (row < n && threadIdx.x % L == 0) y[row] = s;
}

// Lanes per row and entries per lane and turn, by the mean row length (2-D Q1: 9, 3-D Q1
// and P2: 25-29, scalar Q2: 60, vector Q2: 150-190).  Measured around the choices, in µs:
// P2 4x8 32, 8x4 31, 8x6 37, 16x2 36, 16x3 42; 3-D Q1 (40³) 4.4, 4.3, 5.5, 5.4, 6.2;
// vector Q2 16x12 406, 32x4 385, 32x6 415, 32x8 400, 64x3 438, 64x6 518: entries past the
// row's end cost their issue slots, so a turn that covers every row is not the best.
// f(L, U) with both as compile-time constants.
template <class F>
void row_shape(int64_t nnz, int64_t n, F &&f) {
  const double m = (double)nnz / (double)std::max<int64_t>(n, 1);
  auto c = [](auto v) { return v; };
  using std::integral_constant;
  if (m <= 12) f(c(integral_constant<int, 4>{}), c(integral_constant<int, 3>{}));
  else if (m <= 32) f(c(integral_constant<int, 8>{}), c(integral_constant<int, 4>{}));
  else if (m <= 80) f(c(integral_constant<int, 16>{}), c(integral_constant<int, 5>{}));
  else f(c(integral_constant<int, 32>{}), c(integral_constant<int, 4>{}));
}

// The diagonal of a row by binary search (rows are sorted).
__global__ void diag_inv_kernel(int64_t n, const int32_t *__restrict__ cp,
                                const int32_t *__restrict__ rv, const double *__restrict__ val,
                                double *__restrict__ dinv) {
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  int lo = cp[j], hi = cp[j + 1];
  const int end = hi;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (rv[mid] < j) lo = mid + 1;
    else hi = mid;
  }
  const double d = lo < end && rv[lo] == j ? val[lo] : 0.0;
  dinv[j] = d != 0.0 ? 1.0 / d : 1.0;
}

// r = b - q; with a diagonal (or no) preconditioner also z = M r; partials of r·z,
// r·r, b·b.  The CSR kernels keep z and p interleaved (zp: z in .x, p in .y): they take
// {z, 0} here.
__global__ __launch_bounds__(kBlock) void init_kernel(int64_t n, const double *__restrict__ b,
                                                      const double *__restrict__ q,
                                                      const double *__restrict__ dinv,
                                                      int factored, double *__restrict__ r,
                                                      double *__restrict__ z,
                                                      double2 *__restrict__ zp,
                                                      double *__restrict__ part_rz,
                                                      double *__restrict__ part_rr,
                                                      double *__restrict__ part_bb) {
  double rz = 0.0, rr = 0.0, bb = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock) {
    const double ri = b[i] - q[i];
    r[i] = ri;
    if (!factored) {
      const double zi = dinv ? ri * dinv[i] : ri;
      if (zp) zp[i] = make_double2(zi, 0.0);
      else z[i] = zi;
      rz += ri * zi;
    }
    rr += ri * ri;
    bb += b[i] * b[i];
  }
  if (factored)
    put_partials({rr, bb}, {part_rr, part_bb});
  else
    put_partials({rr, bb, rz}, {part_rr, part_bb, part_rz});
}

// r·z of this iteration from its partials (published to scal[rz slot] by block 0);
// p' = z + β p, q = A p', partials of p'·q  (β = 0 on the first iteration of a start).
// z and p of a column come from one 16-byte gather, issued for the first row's first turn
// ahead of the reduction that gives β.  Both are finite, or the solve is lost anyway: the next
// check of r·r stops it.
template <int L, int U>
__global__ __launch_bounds__(kBlock) void spmv_dir_kernel(
    int n, int ntiles, const int32_t *__restrict__ cp, const int32_t *__restrict__ rv,
    const double *__restrict__ val, const double2 *__restrict__ zp, double2 *__restrict__ zpnew,
    double *__restrict__ q, double *scal, int par, int first,
    const double *__restrict__ part_rz, const double *__restrict__ part_rr, int np_rz, double thr,
    int it, uint64_t *news,
    double *__restrict__ part_pq) {
  __shared__ double sh[kStartLds];
  StartIn S = start_loads(scal, part_rz, first ? nullptr : part_rr, np_rz);
  const double rz_old = scal[kRz + (par ^ 1)];
  int t = blockIdx.x;
  RowTurn<L, U> R;
  double2 g[U], own{};
  int row = n;
  int32_t p = 0, p1 = 0;
  auto gather = [&] {
    R.load(rv, val, p, p1);
    R.drop();  // (add: up to 22 registers more, vector Q2 of 12x11x10 cells 3.06 -> 3.37 ms)
#pragma unroll
    for (int u = 0; u < U; ++u) g[u] = zp[R.col[u]];
  };
  auto open = [&](int tile) {  // a row's first turn
    row = tile * (kBlock / L) + (int)threadIdx.x / L;
    if (row >= n) return;
    p = cp[row];
    p1 = cp[row + 1];
    own = zp[row];
    gather();
  };
  if (t < ntiles) open(t);
  if (start_sums(S, sh)) return;
  const double rz = S.a;
  if (iteration_stops(scal, news, S.b, first, thr, it)) return;
  const double beta = first ? 0.0 : rz / rz_old;
  if (blockIdx.x == 0 && threadIdx.x == 0) scal[kRz + par] = rz;
  double dot = 0.0;
  while (t < ntiles) {
    double s = 0.0;
    if (row < n)
      for (;;) {
#pragma unroll
        for (int u = 0; u < U; ++u) s += R.v[u] * (g[u].x + beta * g[u].y);
        p += L * U;
        if (p >= p1) break;
        gather();
      }
    s = row_sum<L>(s);
    if (row < n && threadIdx.x % L == 0) {
      const double pn = own.x + beta * own.y;
      zpnew[row].y = pn;
      q[row] = s;
      dot += pn * s;
    }
    t += gridDim.x;
    if (t < ntiles) open(t);
  }
  put_partial(dot, part_pq);
}

// α = r·z / p'·q; x += α p'; r -= α q; z = M r beside p' (diagonal M or none); partials
// of r·z and r·r: the CSR kernels' form (interleaved z and p), loads ahead of the
// reduction that gives α
__global__ __launch_bounds__(kBlock) void update_zp_kernel(
    int64_t n, int par, const double *__restrict__ dinv, double *__restrict__ x,
    double *__restrict__ r, double2 *__restrict__ zp, const double *__restrict__ q,
    const double *scal, const double *__restrict__ part_pq, int np_pq,
    double *__restrict__ part_rz, double *__restrict__ part_rr) {
  __shared__ double sh[kStartLds];
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  double xi = 0.0, ri = 0.0, pi = 0.0, qi = 0.0, di = 1.0;
  auto load = [&] {
    pi = zp[i].y;
    qi = q[i];
    ri = r[i];
    xi = x[i];
    if (dinv) di = dinv[i];
  };
  StartIn S = start_loads(scal, part_pq, nullptr, np_pq);
  const double rz_now = scal[kRz + par];
  if (i < n) load();
  if (start_sums(S, sh)) return;
  const double alpha = rz_now / S.a;
  double rz = 0.0, rr = 0.0;
  while (i < n) {
    x[i] = xi + alpha * pi;
    ri -= alpha * qi;
    r[i] = ri;
    const double zi = dinv ? ri * di : ri;
    zp[i] = make_double2(zi, pi);
    rz += ri * zi;
    rr += ri * ri;
    i += stride;
    if (i < n) load();
  }
  put_partials({rz, rr}, {part_rz, part_rr});
}

// α = r·z / p'·q; x += α p'; r -= α q; z = M r (diagonal M or none); partials of
// r·z and r·r.  Two consecutive entries per thread (16-byte loads and stores: every
// vector starts 16-byte aligned); the first pair's loads are issued before the
// reduction that gives α.  One entry per thread and the reduction first: 6.9 µs at 64³,
// 24.6 µs at 128³; this form 5.9 and 22.9 µs (131 MB, 5.7 TB/s).
__global__ __launch_bounds__(kBlock) void update_kernel(
    int64_t n, int par, const double *__restrict__ dinv, double *__restrict__ x,
    double *__restrict__ r, double *__restrict__ z, const double *__restrict__ p,
    const double *__restrict__ q, const double *scal, const double *__restrict__ part_pq,
    int np_pq, double *__restrict__ part_rz, double *__restrict__ part_rr) {
  __shared__ double sh[kStartLds];
  const int64_t n2 = n / 2, stride = (int64_t)gridDim.x * kBlock;
  int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  double2 xi{}, ri{}, pi{}, qi{}, di{1.0, 1.0};
  auto load = [&](int64_t k) {
    pi = reinterpret_cast<const double2 *>(p)[k];
    qi = reinterpret_cast<const double2 *>(q)[k];
    ri = reinterpret_cast<const double2 *>(r)[k];
    xi = reinterpret_cast<const double2 *>(x)[k];
    if (dinv) di = reinterpret_cast<const double2 *>(dinv)[k];
  };
  StartIn S = start_loads(scal, part_pq, nullptr, np_pq);
  const double rz_now = scal[kRz + par];
  if (i < n2) load(i);
  if (start_sums(S, sh)) return;
  const double alpha = rz_now / S.a;
  double rz = 0.0, rr = 0.0;
  auto one = [&](double &xv, double &rv, double pv, double qv, double dv) {
    xv += alpha * pv;
    rv -= alpha * qv;
    const double zv = dinv ? rv * dv : rv;
    rz += rv * zv;
    rr += rv * rv;
    return zv;
  };
  while (i < n2) {
    double2 zi;
    zi.x = one(xi.x, ri.x, pi.x, qi.x, di.x);
    zi.y = one(xi.y, ri.y, pi.y, qi.y, di.y);
    reinterpret_cast<double2 *>(x)[i] = xi;
    reinterpret_cast<double2 *>(r)[i] = ri;
    reinterpret_cast<double2 *>(z)[i] = zi;
    i += stride;
    if (i < n2) load(i);
  }
  if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
    double xv = x[n - 1], rv = r[n - 1];
    z[n - 1] = one(xv, rv, p[n - 1], q[n - 1], dinv ? dinv[n - 1] : 1.0);
    x[n - 1] = xv;
    r[n - 1] = rv;
  }
  put_partials({rz, rr}, {part_rz, part_rr});
}

// G and Gᵀ are 16-slot rows (kFsaiEllSlots): 4 lanes per row, 4 slots per lane, one
// 16-byte load of weights and one of column indices per lane.
constexpr int kSlots = kFsaiEllSlots;
static_assert(kSlots == 4 * kApplyLanes, "4 slots per lane");

// α = r·z / p'·q; x += α p'; r' = r - α q; y = G r'; partials of r'·r'
__global__ __launch_bounds__(kBlock) void update_lower_kernel(
    int64_t n, int par, const float *__restrict__ ge, const int32_t *__restrict__ gi,
    double *__restrict__ x, const double *__restrict__ rold, double *__restrict__ rnew,
    const double2 *__restrict__ zp, const double *__restrict__ q, double *__restrict__ y,
    const double *scal, const double *__restrict__ part_pq, int np_pq,
    double *__restrict__ part_rr) {
  __shared__ double sh[kStartLds];
  StartIn S = start_loads(scal, part_pq, nullptr, np_pq);
  const double rz_now = scal[kRz + par];
  if (start_sums(S, sh)) return;
  const double alpha = rz_now / S.a;
  const int sub = threadIdx.x % kApplyLanes;
  const int64_t stride = (int64_t)gridDim.x * (kBlock / kApplyLanes);
  double rr = 0.0;
  for (int64_t row = (int64_t)blockIdx.x * (kBlock / kApplyLanes) + threadIdx.x / kApplyLanes;
       row < n; row += stride) {
    const float4 g = reinterpret_cast<const float4 *>(ge + row * kSlots)[sub];
    const int4 j = reinterpret_cast<const int4 *>(gi + row * kSlots)[sub];
    double s = (double)g.x * (rold[j.x] - alpha * q[j.x]);
    s += (double)g.y * (rold[j.y] - alpha * q[j.y]);
    s += (double)g.z * (rold[j.z] - alpha * q[j.z]);
    s += (double)g.w * (rold[j.w] - alpha * q[j.w]);
#pragma unroll
    for (int o = kApplyLanes / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (sub == 0) {
      y[row] = s;
      const double ri = rold[row] - alpha * q[row];
      rnew[row] = ri;
      x[row] += alpha * zp[row].y;
      rr += ri * ri;
    }
  }
  put_partial(rr, part_rr);
}

// y = G r (start of a solve)
__global__ __launch_bounds__(kBlock) void lower_kernel(int64_t n, const float *__restrict__ ge,
                                                       const int32_t *__restrict__ gi,
                                                       const double *__restrict__ r,
                                                       double *__restrict__ y) {
  const int sub = threadIdx.x % kApplyLanes;
  const int64_t stride = (int64_t)gridDim.x * (kBlock / kApplyLanes);
  for (int64_t row = (int64_t)blockIdx.x * (kBlock / kApplyLanes) + threadIdx.x / kApplyLanes;
       row < n; row += stride) {
    const float4 g = reinterpret_cast<const float4 *>(ge + row * kSlots)[sub];
    const int4 j = reinterpret_cast<const int4 *>(gi + row * kSlots)[sub];
    double s = (double)g.x * r[j.x] + (double)g.y * r[j.y] + (double)g.z * r[j.z] +
               (double)g.w * r[j.w];
#pragma unroll
    for (int o = kApplyLanes / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (sub == 0) y[row] = s;
  }
}

// z = Gᵀ y (beside p); partials of r·z.  START: p becomes 0 (start of a solve)
template <bool START>
__global__ __launch_bounds__(kBlock) void upper_rz_kernel(
    int64_t n, const float *__restrict__ ge, const int32_t *__restrict__ gi,
    const double *__restrict__ y, const double *__restrict__ r, double2 *__restrict__ zp,
    const double *scal, double *__restrict__ part_rz) {
  __shared__ double sh[kStartLds];
  StartIn S = start_loads(scal, nullptr, nullptr, 0);
  if (start_sums(S, sh)) return;
  const int sub = threadIdx.x % kApplyLanes;
  const int64_t stride = (int64_t)gridDim.x * (kBlock / kApplyLanes);
  double rz = 0.0;
  for (int64_t row = (int64_t)blockIdx.x * (kBlock / kApplyLanes) + threadIdx.x / kApplyLanes;
       row < n; row += stride) {
    const float4 g = reinterpret_cast<const float4 *>(ge + row * kSlots)[sub];
    const int4 j = reinterpret_cast<const int4 *>(gi + row * kSlots)[sub];
    double s = (double)g.x * y[j.x] + (double)g.y * y[j.y] + (double)g.z * y[j.z] +
               (double)g.w * y[j.w];
#pragma unroll
    for (int o = kApplyLanes / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (sub == 0) {
      if (START) zp[row] = make_double2(s, 0.0);
      else zp[row].x = s;
      rz += s * r[row];
    }
  }
  put_partial(rz, part_rz);
}

// ---- box lattice: stencil kernels ---------------------------------------------------
// Row i ↔ box node (x, y, z); neighbour offset o = (dx+1) + 3 (dy+1) + 9 (dz+1) has dof
// offset dx + m0 dy + m0 m1 dz, ascending in o.  The assembled lattice matrix is
// symmetric bit for bit (both entries of a pair sum the same cells in the same order),
// so A is held as its lower half a27[o·N + i], o ≤ 13 (zero where the neighbour is
// outside the box), and A(i, i + off(o)) for o > 13 is read as row i + off(o)'s entry
// at offset 26 − o.  G is g14[o·N + i] for o ≤ 13 (lower offsets); Gᵀ row i collects
// g14[o·N + i − off(o)] from the mirrored neighbours.

// a27 (lower half, o ≤ 13) from the CSR rows of the box-lattice matrix.  A lattice
// row holds exactly the neighbours that lie in the box, in ascending column order (the
// symbolic phase has verified the pattern), which is ascending offset order: the
// row's k-th entry belongs to the k-th in-box offset.  A block of kConvRows rows first stages its
// contiguous run of values in LDS with coalesced loads; then all lanes write array o
// together (coalesced, zeros outside the box written explicitly).  A row whose
// length differs from its in-box neighbour count is flagged.  32-bit indices
// (N < 2^31, checked by the caller).
constexpr int kConvRows = 128;

__global__ __launch_bounds__(kConvRows) void stencil_values_kernel(
    Box B, const int32_t *__restrict__ cp, const double *__restrict__ val,
    double *__restrict__ a27, int *__restrict__ bad) {
  __shared__ double sv[kConvRows * 27];
  const int n = (int)B.n;
  const int i0 = blockIdx.x * kConvRows;
  const int i1 = min(i0 + kConvRows, n);
  const int q0 = cp[i0], nq = cp[i1] - q0;
  if (nq > kConvRows * 27) {  // not a 27-point lattice matrix
    if (threadIdx.x == 0) atomicOr(bad, 1);
    return;
  }
  for (int k = threadIdx.x; k < nq; k += kConvRows) sv[k] = val[q0 + k];
  __syncthreads();
  const int i = i0 + (int)threadIdx.x;
  if (i >= n) return;
  const uint32_t vm = box_valid(B, i);
  int p = cp[i] - q0;
  const bool ok = cp[i + 1] - cp[i] == __popc(vm);
#pragma unroll
  for (int o = 0; o < 27; ++o) {
    double v = 0.0;
    if (((vm >> o) & 1u) && ok) v = sv[p++];
    if (o <= 13) a27[(size_t)o * n + i] = v;  // the upper half is read from the mirror
  }
  if (!ok) atomicOr(bad, 1);
}

// D^-1 of the box-lattice matrix from the centre array
__global__ void diag_inv_box_kernel(int64_t n, const double *__restrict__ a27,
                                    double *__restrict__ dinv) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double d = a27[13 * n + i];
  dinv[i] = d != 0.0 ? 1.0 / d : 1.0;
}

// The stencil kernels take tiles of kBlock consecutive rows, one row per thread.  The
// neighbours of a tile's rows are, per dz, one run of consecutive rows (kBlock +
// 2 (m0 + 1) of them; long rows, m0 > kBlock, take one run of kBlock + 2 per (dz, dy)),
// so the vector they multiply goes to LDS once per tile, zero outside [0, N), and each
// row then reads its neighbours there.  No mask is needed: a stored coefficient is zero
// where its neighbour leaves the box, and so is the mirrored one of an upper offset (when
// row j = i + off is a wrapped neighbour, row j's neighbour at -off leaves the box too);
// beyond the last row the run in LDS is zero, and the coefficient address stays inside
// the 14 arrays.  All 27 coefficient loads of a row are independent and issued together,
// ahead of the reduction that gives β.  A row used to load coefficient and vector inside
// the branch of each neighbour, 27 round trips one after the other: spmv_dir 22.5 µs at
// 64³ and 181 µs at 128³ (latency), now 10.2 and 66 µs (bandwidth: 294 MB, 4.5 TB/s; with
// the mirrored entries that miss L2 380 MB, 5.7 TB/s);
// update_lower 10.6 -> 7.8 µs, upper_rz 6.5 -> 4.8 µs at 64³.
// Each XCD sweeps a contiguous slab of the tiles in order, so the mirrored coefficients
// of the next plane are in its L2 when the plane itself reads them.
constexpr int kRunUnroll = 2;  // kBlock-strided loads of one run held in registers

// Where the runs of a tile start and how a row finds its neighbours in them.  Z0: the
// first dz of the runs, NZ: how many dz.
template <bool WIDE, int Z0, int NZ>
struct Runs {
  static constexpr int kRuns = WIDE ? 3 * NZ : NZ;
  int m0, m01, len;
  __device__ __forceinline__ explicit Runs(const Box &B)
      : m0((int)B.m0), m01((int)(B.m0 * B.m1)), len(run_len(B.m0)) {}
  __host__ __device__ static int run_len(int64_t m0) {
    return WIDE ? kBlock + 2 : kBlock + 2 * ((int)m0 + 1);
  }
  __device__ __forceinline__ int base(int i0, int d) const {
    return WIDE ? i0 + (Z0 + d / 3) * m01 + (d % 3 - 1) * m0 - 1 : i0 + (Z0 + d) * m01 - m0 - 1;
  }
  // LDS position of neighbour (dx, dy, dz) of the tile's row t
  __device__ __forceinline__ int at(int t, int dx, int dy, int dz) const {
    return WIDE ? (3 * (dz - Z0) + dy + 1) * len + 1 + dx + t
                : (dz - Z0) * len + (m0 + 1) + dy * m0 + dx + t;
  }
  __device__ __forceinline__ int at(int t, int o) const {
    return at(t, o % 3 - 1, (o / 3) % 3 - 1, o / 9 - 1);
  }
};

// The tiles of this block: first, end of the XCD's slab, step.
struct TileRange {
  int t, end, step;
};
__device__ __forceinline__ TileRange tile_range(int ntiles) {
  constexpr int kXcds = 8;
  const int x = blockIdx.x % kXcds, local = blockIdx.x / kXcds;
  const int q = ntiles / kXcds, r = ntiles % kXcds;
  const int beg = x * q + min(x, r);
  const int nb = ((int)gridDim.x - x + kXcds - 1) / kXcds;
  return {beg + local, beg + q + (x < r), nb};
}

// a[j] + c b[j] (b nullptr: a[j]) over the runs of a tile, zero outside [0, n); the loads
// and the LDS stores are two steps, so that the loads can be issued ahead of the
// reduction that gives c.
template <class R>
struct RunLoads {
  double va[R::kRuns][kRunUnroll], vb[R::kRuns][kRunUnroll];
  __device__ __forceinline__ void issue(const R &r, const double *__restrict__ a,
                                        const double *__restrict__ b, int i0, int n) {
#pragma unroll
    for (int d = 0; d < R::kRuns; ++d)
#pragma unroll
      for (int u = 0; u < kRunUnroll; ++u) {
        const int k = (int)threadIdx.x + u * kBlock, j = r.base(i0, d) + k;
        const bool in = k < r.len && j >= 0 && j < n;
        va[d][u] = in ? a[j] : 0.0;
        vb[d][u] = in && b ? b[j] : 0.0;
      }
  }
  __device__ __forceinline__ void store(const R &r, double *dst, const double *__restrict__ a,
                                        const double *__restrict__ b, double c, int i0, int n) {
#pragma unroll
    for (int d = 0; d < R::kRuns; ++d) {
#pragma unroll
      for (int u = 0; u < kRunUnroll; ++u) {
        const int k = (int)threadIdx.x + u * kBlock;
        if (k < r.len) dst[d * r.len + k] = va[d][u] + c * vb[d][u];
      }
      for (int k = (int)threadIdx.x + kRunUnroll * kBlock; k < r.len; k += kBlock) {
        const int j = r.base(i0, d) + k;
        const bool in = j >= 0 && j < n;
        dst[d * r.len + k] = (in ? a[j] : 0.0) + c * (in && b ? b[j] : 0.0);
      }
    }
  }
};

// Element i of a wave-uniform array: 32-bit byte offset (the box holds < 2^28 rows).
template <class T>
__device__ __forceinline__ T at32(const T *p, uint32_t i) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + i * (uint32_t)sizeof(T));
}

// stencil form of spmv_dir_kernel
template <bool WIDE>
__global__ __launch_bounds__(kBlock) void spmv_dir_box_kernel(
    Box B, int ntiles, const double *__restrict__ a27, const double *__restrict__ z,
    const double *__restrict__ pold, double *__restrict__ pnew, double *__restrict__ q,
    double *scal, int par, int first, const double *__restrict__ part_rz,
    const double *__restrict__ part_rr, int np_rz, double thr, int it,
    uint64_t *news, double *__restrict__ part_pq) {
  extern __shared__ __align__(16) double run[];
  __shared__ double sh[kStartLds];
  using R = Runs<WIDE, -1, 3>;
  const R runs(B);
  const int n = (int)B.n;
  const double *pb = first ? nullptr : pold;
  StartIn S = start_loads(scal, part_rz, first ? nullptr : part_rr, np_rz);
  const double rz_old = scal[kRz + (par ^ 1)];
  TileRange T = tile_range(ntiles);
  RunLoads<R> L;
  double a[27];
  auto loads = [&](int t) {
    const int i0 = t * kBlock;
    L.issue(runs, z, pb, i0, n);
    const uint32_t i = (uint32_t)min(i0 + (int)threadIdx.x, n - 1);
#pragma unroll
    for (int o = 0; o < 27; ++o)  // an upper offset's entry is row j's at the mirrored one
      a[o] = o <= 13 ? at32(a27 + (int64_t)o * n, i)
                     : at32(a27 + (int64_t)(26 - o) * n + box_off(B, o), i);
  };
  if (T.t < T.end) loads(T.t);
  if (start_sums(S, sh)) return;
  const double rz = S.a;
  if (iteration_stops(scal, news, S.b, first, thr, it)) return;
  const double beta = first ? 0.0 : rz / rz_old;
  if (blockIdx.x == 0 && threadIdx.x == 0) scal[kRz + par] = rz;
  double dot = 0.0;
  for (; T.t < T.end;) {
    const int i0 = T.t * kBlock, i = i0 + (int)threadIdx.x;
    L.store(runs, run, z, pb, beta, i0, n);
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int o = 0; o < 27; ++o) s += a[o] * run[runs.at(threadIdx.x, o)];
    const double pn = run[runs.at(threadIdx.x, 13)];
    if (i < n) {
      pnew[i] = pn;
      q[i] = s;
      dot += pn * s;
    }
    T.t += T.step;
    if (T.t < T.end) {
      loads(T.t);
      __syncthreads();  // the runs are read: the next tile's go in
    }
  }
  put_partial(dot, part_pq);
}

// stencil form of update_lower_kernel; START: y = G r only (start of a solve; rold = r)
template <bool WIDE, bool START>
__global__ __launch_bounds__(kBlock) void update_lower_box_kernel(
    Box B, int ntiles, int par, const float *__restrict__ g14, double *__restrict__ x,
    const double *__restrict__ rold, double *__restrict__ rnew, const double *__restrict__ p,
    const double *__restrict__ q, double *__restrict__ y, const double *scal,
    const double *__restrict__ part_pq, int np_pq, double *__restrict__ part_rr) {
  extern __shared__ __align__(16) double run[];
  __shared__ double sh[kStartLds];
  using R = Runs<WIDE, -1, 2>;
  const R runs(B);
  const int n = (int)B.n;
  const double *qb = START ? nullptr : q;
  StartIn S;
  double rz_now = 0.0;
  if (!START) {
    S = start_loads(scal, part_pq, nullptr, np_pq);
    rz_now = scal[kRz + par];
  }
  TileRange T = tile_range(ntiles);
  RunLoads<R> L;
  float g[14];
  double xi = 0.0, pi = 0.0;
  auto loads = [&](int t) {
    const int i0 = t * kBlock;
    L.issue(runs, rold, qb, i0, n);
    const uint32_t i = (uint32_t)min(i0 + (int)threadIdx.x, n - 1);
#pragma unroll
    for (int o = 0; o < 14; ++o) g[o] = at32(g14 + (int64_t)o * n, i);
    if (!START) {
      xi = at32(x, i);
      pi = at32(p, i);
    }
  };
  if (T.t < T.end) loads(T.t);
  double alpha = 0.0;
  if (!START) {
    if (start_sums(S, sh)) return;
    alpha = rz_now / S.a;
  }
  double rr = 0.0;
  for (; T.t < T.end;) {
    const int i0 = T.t * kBlock, i = i0 + (int)threadIdx.x;
    L.store(runs, run, rold, qb, -alpha, i0, n);
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int o = 0; o < 14; ++o) s += (double)g[o] * run[runs.at(threadIdx.x, o)];
    if (i < n) {
      y[i] = s;
      if (!START) {
        const double ri = run[runs.at(threadIdx.x, 13)];
        rnew[i] = ri;
        x[i] = xi + alpha * pi;
        rr += ri * ri;
      }
    }
    T.t += T.step;
    if (T.t < T.end) {
      loads(T.t);
      __syncthreads();
    }
  }
  if (!START) put_partial(rr, part_rr);
}

// z = Gᵀ y, partials of r·z; stencil form: entry (j, i) of G with j = i − off(o),
// o ≤ 13, sits at g14[o·N + j]
template <bool WIDE>
__global__ __launch_bounds__(kBlock) void upper_rz_box_kernel(
    Box B, int ntiles, const float *__restrict__ g14, const double *__restrict__ y,
    const double *__restrict__ r, double *__restrict__ z, const double *scal,
    double *__restrict__ part_rz) {
  extern __shared__ __align__(16) double run[];
  __shared__ double sh[kStartLds];
  using R = Runs<WIDE, 0, 2>;
  const R runs(B);
  const int n = (int)B.n;
  StartIn S = start_loads(scal, nullptr, nullptr, 0);
  TileRange T = tile_range(ntiles);
  RunLoads<R> L;
  float g[14];
  double ri = 0.0;
  auto loads = [&](int t) {
    const int i0 = t * kBlock;
    L.issue(runs, y, nullptr, i0, n);
    const uint32_t i = (uint32_t)min(i0 + (int)threadIdx.x, n - 1);
#pragma unroll
    for (int o = 0; o < 14; ++o) g[o] = at32(g14 + (int64_t)o * n - box_off(B, o), i);
    ri = at32(r, i);
  };
  if (T.t < T.end) loads(T.t);
  if (start_sums(S, sh)) return;
  double rz = 0.0;
  for (; T.t < T.end;) {
    const int i0 = T.t * kBlock, i = i0 + (int)threadIdx.x;
    L.store(runs, run, y, nullptr, 0.0, i0, n);
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int o = 13; o >= 0; --o) s += (double)g[o] * run[runs.at(threadIdx.x, 26 - o)];
    if (i < n) {
      z[i] = s;
      rz += s * ri;
    }
    T.t += T.step;
    if (T.t < T.end) {
      loads(T.t);
      __syncthreads();
    }
  }
  put_partial(rz, part_rz);
}

}  // namespace

void spmv_device(Ctx &c, const double *x, double *y) {
  row_shape(c.nnz, c.nfree, [&](auto L, auto U) {
    const int ntiles = (int)((c.nfree + kBlock / L() - 1) / (kBlock / L()));
    hipLaunchKernelGGL((spmv_kernel<L(), U()>), dim3((unsigned)std::max(ntiles, 1)),
                       dim3(kBlock), 0, c.stream, (int)c.nfree, c.colptr.get(), c.rowval.get(),
                       c.nzval.get(), x, y);
  });
  GH_CHECK_HIP(hipGetLastError());
}

namespace {
// Σ of np partials on the host (convergence checks only; fixed order).
double host_sum(const double *v, int np) {
  double a = 0.0;
  for (int k = 0; k < np; ++k) a += v[k];
  return a;
}
}  // namespace

namespace {

// Device vectors of one solve: the solution x (initial guess on entry) and b, the CG
// vectors, the diagonal inverse, partial sums (4 x kMaxParts) and scalars (8).
struct PcgBufs {
  double *x, *b, *r, *r2, *z, *p, *p2, *q, *y, *dinv, *part, *scal;
  double2 *zp, *zp2;  // the CSR form's interleaved z and p (two buffers)
};

__global__ void clear_stop_kernel(double *scal) {
  if (threadIdx.x < 2) scal[kStop + threadIdx.x] = 0.0;
}

// The solve on the given buffers.  box: the stencil form may be used (needs c.a27
// and, for FSAI, c.g14); timed: HIP events around the solve (device_ms), else 0.
void pcg_run(Ctx &c, const PcgBufs &V, int precond, double rtol, int maxit, bool allow_box,
             bool timed, gh_solve_stats *st) {
  const int64_t n = c.nfree;
  hipStream_t s = c.stream;
  const size_t nn = (size_t)std::max<int64_t>(n, 1);
  // the solve is timed from here: per-matrix preparation (D^-1, the stencil arrays)
  // included
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (timed) {
    e0 = c.timing_events()[0];
    e1 = c.timing_events()[1];
    GH_CHECK_HIP(hipEventRecord(e0, s));
  }
  HostCopy copy(c, !timed);
  uint64_t *news = copy.word();
  double *dinv = nullptr;
  const int factored = precond == GH_PRECOND_FSAI;
  // box lattice: stencil kernels (A as 14 offset arrays, G as 14), one thread per row
  // GRIDAP_HIP_STENCIL_PCG=0 runs the general (CSR) kernels on a box lattice too, so
  // the two forms can be compared on the same system
  const char *stencil_env = std::getenv("GRIDAP_HIP_STENCIL_PCG");
  bool box = allow_box && c.box && n > 0 && n < (int64_t(1) << 28) &&
             (!factored || c.g14.get() != nullptr) && !(stencil_env && stencil_env[0] == '0');
  const Box B{n, c.box_m[0], c.box_m[1], c.box_m[2]};
  if (box) {
    c.a27.resize((size_t)14 * nn);
    int *bad = reinterpret_cast<int *>(V.scal + kBad);
    GH_CHECK_HIP(hipMemsetAsync(bad, 0, sizeof(int), s));
    hipLaunchKernelGGL(stencil_values_kernel, dim3((unsigned)((n + kConvRows - 1) / kConvRows)),
                       dim3(kConvRows), 0, s, B, c.colptr.get(), c.nzval.get(), c.a27.get(),
                       bad);
    GH_CHECK_HIP(hipGetLastError());
    int hbad = 0;
    copy.down(&hbad, bad, sizeof(int));
    box = hbad == 0;
  }
  if (precond == GH_PRECOND_JACOBI) {
    if (box)
      hipLaunchKernelGGL(diag_inv_box_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                         n, c.a27.get(), V.dinv);
    else
      hipLaunchKernelGGL(diag_inv_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n,
                         c.colptr.get(), c.rowval.get(), c.nzval.get(), V.dinv);
    dinv = V.dinv;
  }
  if (factored)
    GH_REQUIRE(c.fsai_built, GH_ERR_STATE, "no FSAI factor for this matrix: call gh_fsai_build");
  double *scal = V.scal;
  double *part_pq = V.part, *part_rz = part_pq + kMaxParts;
  double *part_rr = part_rz + kMaxParts, *part_bb = part_rr + kMaxParts;
  double *rbuf[2] = {V.r, factored ? V.r2 : V.r};
  double *pbuf[2] = {V.p, V.p2};
  double2 *zpbuf[2] = {V.zp, V.zp2};
  const int ntiles = (int)((n + kBlock - 1) / kBlock);
  // the vector kernels: two entries per thread, one with the interleaved z and p
  const unsigned g_vec = grid_rows(box ? (n + 1) / 2 : n, kBlock);
  const unsigned g_box = grid_rows(n, kBlock);            // one tile per block and turn
  // the stencil product: the two workgroups a compute unit holds, so that every slab is swept
  // once in order; one where the matrix and the vectors (176 bytes a row) no longer stay in
  // the 256 MB cache, so that less of a plane's mirrored coefficients leaves L2 before the
  // plane needs them (kStencilGrid)
  unsigned g_spmv = std::min(g_box, n * 176 > 224000000 ? kStencilGrid / 2 : kStencilGrid);
  if (!box) row_shape(c.nnz, n, [&](auto L, auto) { g_spmv = grid_rows(n, kBlock / L()); });
  const unsigned g_apply = box ? g_box : grid_rows(n, kBlock / kApplyLanes);
  // the stencil kernels' form: one run per dz, or per (dz, dy) for long rows
  const bool wide = B.m0 > kBlock;
  const size_t run_bytes = sizeof(double) * (wide ? 3 * Runs<true, 0, 1>::run_len(B.m0)
                                                  : Runs<false, 0, 1>::run_len(B.m0));
  auto spmv_dir_box = [&](double *pold, double *pnew, int par, int first, int np_rz, double thr,
                          int itk) {
    auto kern = wide ? spmv_dir_box_kernel<true> : spmv_dir_box_kernel<false>;
    hipLaunchKernelGGL(kern, dim3(g_spmv), dim3(kBlock), 3 * run_bytes, s, B, ntiles, c.a27.get(),
                       V.z, pold, pnew, V.q, scal, par, first, part_rz, part_rr, np_rz, thr, itk,
                       news, part_pq);
  };
  auto lower_box = [&](bool start, int par, double *rold, double *rnew, double *pnew) {
    auto kern = wide ? (start ? update_lower_box_kernel<true, true>
                              : update_lower_box_kernel<true, false>)
                     : (start ? update_lower_box_kernel<false, true>
                              : update_lower_box_kernel<false, false>);
    hipLaunchKernelGGL(kern, dim3(g_box), dim3(kBlock), 2 * run_bytes, s, B, ntiles, par,
                       c.g14.get(), V.x, rold, rnew, pnew, V.q, V.y, scal, part_pq, (int)g_spmv,
                       part_rr);
  };
  auto upper_box = [&](double *r) {
    auto kern = wide ? upper_rz_box_kernel<true> : upper_rz_box_kernel<false>;
    hipLaunchKernelGGL(kern, dim3(g_box), dim3(kBlock), 2 * run_bytes, s, B, ntiles,
                       c.g14.get(), V.y, r, V.z, scal, part_rz);
  };
  // partial counts of each quantity, by producer
  const int np_rz = factored ? (int)g_apply : (int)g_vec;
  double hsum[kMaxParts + kPcgGrid];  // r·r and b·b: neighbours, g_vec <= kPcgGrid of each

  double bnorm = 1.0, relres = INFINITY;
  int it = 0, restarts = 0;
  bool converged = false;
  while (true) {
    // (re)start from the true residual r = b - A x
    spmv_device(c, V.x, V.q);
    hipLaunchKernelGGL(init_kernel, dim3(g_vec), dim3(kBlock), 0, s, n, V.b, V.q,
                       dinv, factored, rbuf[0], V.z, box ? nullptr : zpbuf[0], part_rz, part_rr,
                       part_bb);
    hipLaunchKernelGGL(clear_stop_kernel, dim3(1), dim3(64), 0, s, scal);
    if (factored && box) {
      lower_box(true, 0, rbuf[0], nullptr, nullptr);
      upper_box(rbuf[0]);
    } else if (factored) {
      hipLaunchKernelGGL(lower_kernel, dim3(g_apply), dim3(kBlock), 0, s, n, c.gle.get(),
                         c.gli.get(), rbuf[0], V.y);
      hipLaunchKernelGGL(upper_rz_kernel<true>, dim3(g_apply), dim3(kBlock), 0, s, n,
                         c.gue.get(), c.gui.get(), V.y, rbuf[0], zpbuf[0], scal, part_rz);
    }
    GH_CHECK_HIP(hipGetLastError());
    copy.down(hsum, part_rr, sizeof(double) * (kMaxParts + g_vec));
    const double bb = host_sum(hsum + kMaxParts, (int)g_vec);
    bnorm = std::sqrt(bb) > 0 ? std::sqrt(bb) : 1.0;
    relres = std::sqrt(host_sum(hsum, (int)g_vec)) / bnorm;
    if (relres <= rtol) {
      converged = true;
      break;
    }
    if (it >= maxit || restarts > 3) break;
    ++restarts;
    // each spmv_dir decides on the device whether the previous update met the tolerance,
    // and once it has, every later kernel returns at once
    const double thr = (rtol * bnorm) * (rtol * bnorm);
    int k = 0;  // iteration since this start: selects the buffers and scalar slots
    auto iteration = [&](int itk) {
      const int par = k & 1;
      double *pold = pbuf[par], *pnew = pbuf[par ^ 1];
      double2 *zpold = zpbuf[par], *zpnew = zpbuf[par ^ 1];
      if (box)
        spmv_dir_box(pold, pnew, par, k == 0 ? 1 : 0, np_rz, thr, itk);
      else
        row_shape(c.nnz, n, [&](auto L, auto U) {
          const int nt = (int)((n + kBlock / L() - 1) / (kBlock / L()));
          hipLaunchKernelGGL((spmv_dir_kernel<L(), U()>), dim3(g_spmv), dim3(kBlock), 0, s,
                             (int)n, nt, c.colptr.get(), c.rowval.get(), c.nzval.get(), zpold,
                             zpnew, V.q, scal, par, k == 0 ? 1 : 0, part_rz, part_rr, np_rz,
                             thr, itk, news, part_pq);
        });
      if (factored && box) {
        double *rold = rbuf[par], *rnew = rbuf[par ^ 1];
        lower_box(false, par, rold, rnew, pnew);
        upper_box(rnew);
      } else if (factored) {
        double *rold = rbuf[par], *rnew = rbuf[par ^ 1];
        hipLaunchKernelGGL(update_lower_kernel, dim3(g_apply), dim3(kBlock), 0, s, n, par,
                           c.gle.get(), c.gli.get(), V.x, rold, rnew, zpnew, V.q,
                           V.y, scal, part_pq, (int)g_spmv, part_rr);
        hipLaunchKernelGGL(upper_rz_kernel<false>, dim3(g_apply), dim3(kBlock), 0, s, n,
                           c.gue.get(), c.gui.get(), V.y, rnew, zpnew, scal, part_rz);
      } else if (!box) {
        hipLaunchKernelGGL(update_zp_kernel, dim3(g_vec), dim3(kBlock), 0, s, n, par, dinv,
                           V.x, rbuf[0], zpnew, V.q, scal, part_pq, (int)g_spmv, part_rz,
                           part_rr);
      } else {
        hipLaunchKernelGGL(update_kernel, dim3(g_vec), dim3(kBlock), 0, s, n, par, dinv,
                           V.x, rbuf[0], V.z, pnew, V.q, scal, part_pq,
                           (int)g_spmv, part_rz, part_rr);
      }
      ++k;
    };
    // The host enqueues at most kAhead iterations past the one that the device says it has
    // begun, and none once it has stopped: the device never waits for the host (a read-back
    // every 16 iterations left it idle for 18 µs each time), and little is enqueued in
    // vain.  Without the word, chunks of 16 and a read-back.
    constexpr int kAhead = 3, kChunk = 16;
    constexpr uint64_t kNoNews = ~uint64_t(0);
    bool stopped = false, ended = false;
    if (news) __atomic_store_n(news, kNoNews, __ATOMIC_RELAXED);  // the stream is idle
    for (int m = 0; it < maxit && !stopped; ++m) {
      iteration(it++);
      GH_CHECK_HIP(hipGetLastError());
      if (news) {
        for (unsigned spin = 1; !ended; ++spin) {
          const uint64_t v = __atomic_load_n(news, __ATOMIC_RELAXED);
          const int begun = v == kNoNews ? it - m - 2 : (int)(uint32_t)v;
          stopped = v != kNoNews && (v & kStopped);
          if (stopped) it = begun;  // iterations completed before the stop
          if (stopped || it - 1 - begun <= kAhead) break;
          __builtin_ia32_pause();
          if (spin % 4096 == 0) {
            const hipError_t e = hipStreamQuery(s);
            if (e == hipErrorNotReady) (void)hipGetLastError();
            else GH_CHECK_HIP(e);
            ended = e == hipSuccess;  // nothing more will come: read back below
          }
        }
      }
      if (!stopped && (it == maxit || ended || (!news && (m + 1) % kChunk == 0))) {
        double st2[2] = {0.0, 0.0};
        copy.down(st2, scal + kStop, sizeof(st2));
        stopped = st2[0] != 0.0;
        if (stopped) it = (int)st2[1];
        ended = false;
      }
    }
    // the true residual of the next start decides convergence (and, if the stopped
    // r·r was not finite, the restart count ends the solve)
  }
  float ms = 0.f;
  if (timed) {
    GH_CHECK_HIP(hipEventRecord(e1, s));
    GH_CHECK_HIP(hipEventSynchronize(e1));
    GH_CHECK_HIP(hipEventElapsedTime(&ms, e0, e1));
  } else {
    GH_CHECK_HIP(hipStreamSynchronize(s));
  }
  c.solve_form = box ? GH_SOLVE_STENCIL : GH_SOLVE_ROWS;
  st->iterations = it;
  st->converged = converged ? 1 : 0;
  st->rel_residual = relres;
  st->device_ms = ms;
}

}  // namespace

// Systems that the one-workgroup solve takes: at most 4096 rows, 40,960 entries and 64
// entries a row on average, boxes 1536 rows.  The rows are what a workgroup holds and not
// where it stops winning (4096 rows 3.9 µs an iteration and 9.4 in the general kernels: past
// them an iteration takes more than twice as long).  Past the entries one compute unit streams too
// much of the matrix (µs an iteration: 3-D Q1 39,304 entries 7.5, 50,653 14.6, 64,000 15.6,
// where the general kernels take 10 to 12); with longer rows a thread's serial share is too
// long (one workgroup and general kernels: 3-D Q2 of 41 a row 9.8 and 12.2; vector Q2 of
// 110 a row and 38,124 entries 11.5 and 10.0); larger boxes fit the resident solve (1000
// rows 182 and 252 µs a solve, 1728 297 and 284).  GRIDAP_HIP_SMALL_PCG=0 switches it off, and
// so does choosing between the other forms (GRIDAP_HIP_STENCIL_PCG).
constexpr int64_t kSmallMaxNnz = 40960, kSmallMaxRow = 64, kSmallMaxBox = 1536;
bool small_system(const Ctx &c, int precond) {
  const char *off = std::getenv("GRIDAP_HIP_SMALL_PCG");
  return (precond == GH_PRECOND_NONE || precond == GH_PRECOND_JACOBI) && c.nfree > 0 &&
         c.nfree <= (c.box ? kSmallMaxBox : kSmallMaxN) && c.nnz <= kSmallMaxNnz &&
         c.nnz <= kSmallMaxRow * c.nfree && !(off && off[0] == '0') &&
         !std::getenv("GRIDAP_HIP_STENCIL_PCG");
}

void pcg_device(Ctx &c, int precond, double rtol, int maxit, gh_solve_stats *st) {
  // a solve in one launch, timed like the general one; false: not taken.  The time of one
  // that gave up counts too, and so do its iterations (done).
  double spent = 0.0;
  int done = 0;
  auto timed = [&](auto &&solve) {
    float ms = 0.f;
    hipEvent_t *ev = c.timing_events();
    GH_CHECK_HIP(hipEventRecord(ev[0], c.stream));
    const bool taken = solve();
    GH_CHECK_HIP(hipEventRecord(ev[1], c.stream));
    GH_CHECK_HIP(hipEventSynchronize(ev[1]));
    GH_CHECK_HIP(hipEventElapsedTime(&ms, ev[0], ev[1]));
    spent += ms;
    st->device_ms = spent;
    return taken;
  };
  c.s_small.resize(std::max(kSmallWs, kResidentWs));
  if (small_system(c, precond) && timed([&] {
        HostCopy copy(c);
        return pcg_small(c, copy, precond, rtol, maxit, c.s_x.get(), c.s_b.get(),
                         c.s_small.get(), st);
      }))
    return;
  const size_t nn = (size_t)std::max<int64_t>(c.nfree, 1);
  for (auto *bf : {&c.s_r, &c.s_z, &c.s_q}) bf->resize(nn);
  // p and its second buffer, or the interleaved z and p of the CSR kernels
  for (auto *bf : {&c.s_p, &c.s_p2}) bf->resize(2 * nn);
  c.s_part.resize(4 * kMaxParts);
  c.s_scal.resize(8);
  if (precond == GH_PRECOND_JACOBI) c.s_dinv.resize(nn);
  if (precond == GH_PRECOND_FSAI) {
    c.s_y.resize(nn);
    c.s_r2.resize(nn);
  }
  const PcgBufs V{c.s_x.get(), c.s_b.get(), c.s_r.get(), c.s_r2.get(), c.s_z.get(),
                  c.s_p.get(), c.s_p2.get(), c.s_q.get(), c.s_y.get(), c.s_dinv.get(),
                  c.s_part.get(), c.s_scal.get(), (double2 *)c.s_p.get(),
                  (double2 *)c.s_p2.get()};
  const Box B{c.nfree, c.box_m[0], c.box_m[1], c.box_m[2]};
  if (c.box && resident_system(c, B, precond) &&
      (precond != GH_PRECOND_FSAI || (c.fsai_built && c.g14.get())) && timed([&] {
        return pcg_resident(c, B, precond, rtol, maxit, V.x, V.b, {V.r, V.p, V.z},
                            {V.p2, V.r2, V.y}, c.s_small.get(), st, &done);
      }))
    return;
  pcg_run(c, V, precond, rtol, maxit - done, true, true, st);
  st->iterations += done;
  st->device_ms += spent;
}

// ---- the solve that allocates nothing (gh_pcg_noalloc) ------------------------------
// Its vectors live in one fixed device array, `scratch`, which every GPU the library
// runs on holds until the process ends: x, b, r, q, D^-1 and two interleaved {z, p}, of
// at most GH_NOALLOC_MAX_N entries each (nine vectors), then the partial sums and the
// scalars.  Every call on one GPU shares that GPU's copy (calls that overlap on one GPU
// race), and nothing in it is read before the call writes it.
namespace {
constexpr size_t kNoAllocVec = (size_t)GH_NOALLOC_MAX_N;
constexpr size_t kNoAllocVecs = 9;
constexpr size_t kScratchDoubles = kNoAllocVecs * kNoAllocVec + 4 * (size_t)kMaxParts + 8;
__device__ __align__(256) double scratch[kScratchDoubles];

constexpr int kMaxDevices = 64;
double *g_scratch[kMaxDevices] = {};  // device address of `scratch` on each GPU
std::mutex g_scratch_mu;
}  // namespace

// Look up this GPU's address of `scratch` once (the calling thread has the device
// current).  Host code uses that address, never the array's name.
void scratch_init(int device) {
  GH_REQUIRE(device >= 0 && device < kMaxDevices, GH_ERR_ARG, "device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch[device]) return;
  void *p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || p == nullptr)
    throw Error(GH_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
  g_scratch[device] = static_cast<double *>(p);
}

void pcg_noalloc(Ctx &c, int precond, const double *b, double *x, double rtol, int maxit,
                 gh_solve_stats *st) {
  GH_REQUIRE(precond == GH_PRECOND_NONE || precond == GH_PRECOND_JACOBI, GH_ERR_UNSUPPORTED,
             "the allocation-free solve provides Jacobi or no preconditioner");
  GH_REQUIRE(c.nfree <= GH_NOALLOC_MAX_N, GH_ERR_ARG,
             "num_free_dofs exceeds GH_NOALLOC_MAX_N, the allocation-free solve's limit");
  double *base = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    base = c.device >= 0 && c.device < kMaxDevices ? g_scratch[c.device] : nullptr;
  }
  GH_REQUIRE(base, GH_ERR_STATE, "scratch address not set up for this device");
  const size_t n = (size_t)c.nfree;
  const size_t L = kNoAllocVec;
  double *part = base + kNoAllocVecs * L;
  const PcgBufs V{base, base + L, base + 2 * L, nullptr, nullptr, nullptr, nullptr, base + 3 * L,
                  nullptr, base + 4 * L, part, part + 4 * (size_t)kMaxParts,
                  (double2 *)(base + 5 * L), (double2 *)(base + 7 * L)};
  const auto t0 = std::chrono::steady_clock::now();
  HostCopy copy(c, true);
  copy.up(V.x, x, sizeof(double) * n);
  if (b)
    copy.up(V.b, b, sizeof(double) * n);
  else
    GH_CHECK_HIP(hipMemcpyAsync(V.b, c.b.get(), sizeof(double) * n, hipMemcpyDeviceToDevice,
                                c.stream));
  // the one-workgroup solve's workspace: the two {z, p}, which it does not need
  static_assert(kSmallWs <= 4 * kNoAllocVec * sizeof(double), "workspace");
  if (!(small_system(c, precond) &&
        pcg_small(c, copy, precond, rtol, maxit, V.x, V.b, (unsigned char *)V.zp, st)))
    pcg_run(c, V, precond, rtol, maxit, false, false, st);
  copy.down(x, V.x, sizeof(double) * n);
  copy.finish();
  st->device_ms =
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  st->precond_used = precond;
}

}  // namespace gh
