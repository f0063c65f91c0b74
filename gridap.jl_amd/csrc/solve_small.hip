// The whole PCG solve of a small system in one workgroup.
//
// A small system's iteration is launches and memory round trips, not work: two kernels
// and their gaps take 10 to 16 µs however small the matrix.  Here one workgroup of 512
// threads runs the solve: start residual, iterations, restarts and the stopping test, one
// launch and one read-back.  A thread owns rows t, t + 512, ... (R of them); p, x and D^-1
// live in LDS, r and the first E entries of every row in registers (R E is what the 256
// registers of 8 waves hold; with R = 8 the ninth entry, the last of a 2-D Q1 row, is in
// LDS), so consecutive threads read consecutive entries of p (no bank conflicts for lattice
// numberings) and a row's sum needs no other thread.  The entries past those of a slice of 64
// rows are copied once, lane by lane and column as 16 bits, to a workspace from which the
// wave streams them every iteration (10 bytes an entry, coalesced).  Bound by the LDS reads of p and the three barriers while the matrix fits the
// registers, else by what one compute unit draws from L2.  Microseconds an iteration, start-up
// included, here and in the general kernels: 2-D Q1 1024 rows 3.2 and 10.2, 4096 rows 3.9
// and 9.4; 3-D Q1 729 rows 5.7 and 15.7, 1728 rows 7.5 and 16.2; scalar Q2 729 rows 9.8
// and 14.2.  (1024 threads and sums through LDS permutes took 6.8 for the first: twice the
// waves at each barrier, half the registers.)  No form spills registers: gh_pcg_noalloc runs
// them, and the runtime would back scratch with device memory.  (Eight rows a thread at 2070
// and 4096 rows: nine entries in registers, 20 of them spilled, 4.3 and 4.2 µs; eight, and the
// ninth streamed, 3.8 and 4.4; the ninth in LDS 3.9 and 3.9.)
// Both dot products sum in a fixed order: the result is the same every time.
// One launch runs at most kPause iterations: past them the state goes to the workspace and
// the next launch takes it up, so that a solve that never ends on its own does not hold the
// device in one kernel.
#include <algorithm>
#include <cmath>

#include "gh_internal.h"

namespace gh {
namespace {

constexpr int kT = 512, kWaves = kT / 64;
constexpr int kMaxRows = 8;                      // rows per thread
static_assert(kSmallMaxN == kT * kMaxRows, "rows");

struct SmallArgs {
  int n, maxit, jacobi;
  double rtol;
  const int32_t *cp, *rv;
  const double *val, *b;
  double *x;        // initial guess in, solution out
  double *wv;       // streamed values and columns, kSmallStream each
  uint16_t *wc;
  double *state;    // r and p between launches, kSmallMaxN each
  int resume;
  double *out;      // {iterations, converged, relative residual, kDone..., and a paused
                    //  solve's rz, threshold and restarts}
};
constexpr int kOut = 7, kPause = 8192;
constexpr double kDone = 0, kDeclined = 1, kPaused = 2;

// Σ a and Σ b over the workgroup, the same in every thread.  One barrier: the sums of two
// calls in turn use different halves of sh (turn).
__device__ __forceinline__ void sum2(double &a, double &b, double *sh, int &turn) {
  static_assert(kWaves <= 16, "wave sums of a row");
  a = wave_sum(a);
  b = wave_sum(b);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double *s = sh + 32 * turn;
  turn ^= 1;
  if (lane == 0) {
    s[w] = a;
    s[16 + w] = b;
  }
  __syncthreads();
  // every wave sums the wave sums: a in lanes 0-15, b in lanes 16-31
  const double v = row16_sum((lane & 15) < kWaves ? s[lane & 31] : 0.0);
  a = lane_value(v, 15);
  b = lane_value(v, 31);
}

// X: entry E of every row (one more) in LDS too.
template <int R, int E, int X>
__global__ __launch_bounds__(kT) void small_pcg_kernel(const SmallArgs A) {
  extern __shared__ __align__(16) double lds[];
  __shared__ double sh[64];
  int turn = 0;
  __shared__ int width[kMaxRows * kWaves];
  const int t = threadIdx.x, lane = t & 63, n = A.n;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // uniform values in scalar registers
  double *pl = lds, *xl = lds + R * kT, *dl = lds + 2 * R * kT;
  double *vx = lds + 3 * R * kT;
  uint16_t *cx = reinterpret_cast<uint16_t *>(vx + R * kT);
  // matrix: first E entries of each row here, the rest to the stream
  double v[R][E];
  uint32_t col[R][(E + 1) / 2];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = t + k * kT;
    int len = i < n ? A.cp[i + 1] - A.cp[i] - E - X : 0;
    len = max(len, 0);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) len = max(len, __shfl_xor(len, o));
    if (lane == 0) width[k * kWaves + wave] = len;
  }
  __syncthreads();
  int base[R], wd[R], total = 0;
#pragma unroll
  for (int k = 0; k < R; ++k) base[k] = wd[k] = 0;
  for (int s = 0; s < R * kWaves; ++s) {
    const int w = __builtin_amdgcn_readfirstlane(width[s]);
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (s == k * kWaves + wave) {
        base[k] = total;
        wd[k] = w;
      }
    total += min(64 * w, kSmallStream);
    total = min(total, kSmallStream + 1);
  }
  if (total > kSmallStream) {  // rows too uneven for the slices: the general kernels solve it
    if (t == 0) A.out[3] = kDeclined;
    return;
  }
  double diag[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = t + k * kT;
    const int p0 = i < n ? A.cp[i] : 0, p1 = i < n ? A.cp[i + 1] : 0, last = max(p1 - 1, 0);
    diag[k] = 0.0;
    int j[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {  // past the end: the last entry with weight 0
      j[e] = A.rv[min(p0 + e, last)];
      v[k][e] = A.val[min(p0 + e, last)];
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const bool in = p0 + e < p1;
      v[k][e] = in ? v[k][e] : 0.0;
      j[e] = in ? j[e] : 0;
      diag[k] = in && j[e] == i ? v[k][e] : diag[k];
      col[k][e / 2] = e % 2 ? col[k][e / 2] | ((uint32_t)j[e] << 16) : (uint32_t)j[e];
    }
    if (X) {
      __builtin_amdgcn_sched_barrier(0);
      const bool in = p0 + E < p1;
      const int p = in ? p0 + E : last, jj = A.rv[p];
      const double a = A.val[p];
      vx[i] = in ? a : 0.0;
      cx[i] = (uint16_t)(in ? jj : 0);
      diag[k] = in && jj == i ? a : diag[k];
    }
#pragma unroll 4
    for (int e = 0; e < wd[k]; ++e) {
      const int p = min(p0 + E + X + e, last);
      const bool in = p0 + E + X + e < p1;
      const int jj = in ? A.rv[p] : 0;
      const double a = in ? A.val[p] : 0.0;
      diag[k] = in && jj == i ? a : diag[k];
      A.wv[base[k] + 64 * e + lane] = a;
      A.wc[base[k] + 64 * e + lane] = (uint16_t)jj;
    }
    __builtin_amdgcn_sched_barrier(0);  // one row's loads at a time: registers
  }
  double r[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = t + k * kT;
    xl[i] = i < n ? A.x[i] : 0.0;
    dl[i] = A.jacobi && diag[k] != 0.0 ? 1.0 / diag[k] : 1.0;
    r[k] = 0.0;
  }
  // q_k = (A p)_row, p in LDS (a lane's own stream entries: no barrier needed after the
  // copy above)
  auto spmv = [&](double (&q)[R]) {
#pragma unroll
    for (int k = 0; k < R; ++k) {
      double s = 0.0;
      // the columns are opaque here: LDS addresses hoisted out of the iteration loop would
      // take one register an entry
#pragma unroll
      for (int e = 0; e < (E + 1) / 2; ++e) asm volatile("" : "+v"(col[k][e]));
#pragma unroll
      for (int e = 0; e < E; ++e) s += v[k][e] * pl[(col[k][e / 2] >> (16 * (e % 2))) & 0xffffu];
      if (X) {
        int i = t + k * kT;  // its addresses formed here
        asm volatile("" : "+v"(i));
        s += vx[i] * pl[cx[i]];
      }
      int at = base[k] + lane, left = wd[k];
      asm volatile("" : "+v"(at), "+s"(left));
      constexpr int U = 8;
#pragma unroll 1
      for (; left >= U; left -= U, at += 64 * U) {
        double a[U];
        int j[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          a[u] = A.wv[at + 64 * u];
          j[u] = A.wc[at + 64 * u];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) s += a[u] * pl[j[u]];
      }
#pragma unroll 1
      for (; left > 0; --left, at += 64) s += A.wv[at] * pl[A.wc[at]];
      q[k] = s;
      __builtin_amdgcn_sched_barrier(0);  // one row's loads at a time: registers
    }
  };
  // Each turn multiplies by A once: a step of the recurrence, or (start) the true residual
  // r = b - A x of a (re)start.  One copy of the product keeps the registers in bounds.
  int it = 0, restarts = 0, converged = 0;
  double relres = INFINITY, how = kDone, rz = 0.0, rr = 0.0, thr = 0.0, none, q[R];
  bool start = !A.resume;
  if (start) {
#pragma unroll
    for (int k = 0; k < R; ++k) pl[t + k * kT] = xl[t + k * kT];
  } else {
    it = (int)A.out[0];
    rz = A.out[4];
    thr = A.out[5];
    restarts = (int)A.out[6];
#pragma unroll
    for (int k = 0; k < R; ++k) {
      r[k] = A.state[t + k * kT];
      pl[t + k * kT] = A.state[kSmallMaxN + t + k * kT];
    }
  }
  __syncthreads();
  const int until = A.maxit - it > kPause ? it + kPause : A.maxit;
  for (;;) {
    spmv(q);
    none = 0.0;
    if (start) {
      int t0 = t;  // addresses of b formed here: hoisted they would take registers all along
      asm volatile("" : "+v"(t0));
      double bb = 0.0;
      rr = 0.0;
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const int i = t0 + k * kT;
        const double bi = i < n ? A.b[i] : 0.0;
        r[k] = i < n ? bi - q[k] : 0.0;
        rr += r[k] * r[k];
        bb += bi * bi;
      }
      sum2(rr, bb, sh, turn);
      const double bnorm = sqrt(bb) > 0 ? sqrt(bb) : 1.0;
      relres = lane_value(sqrt(rr) / bnorm, 0);
      converged = relres <= A.rtol;
      if (converged || it >= A.maxit || restarts > 3) break;
      ++restarts;
      thr = lane_value((A.rtol * bnorm) * (A.rtol * bnorm), 0);
      rz = 0.0;
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const double z = dl[t + k * kT] * r[k];
        pl[t + k * kT] = z;
        rz += r[k] * z;
      }
      sum2(rz, none, sh, turn);  // and p is written
      start = false;
    } else {
      double pq = 0.0;
#pragma unroll
      for (int k = 0; k < R; ++k) pq += pl[t + k * kT] * q[k];
      sum2(pq, none, sh, turn);  // and every thread has read p
      const double alpha = lane_value(rz / pq, 0);
      double rzn = 0.0;
      rr = 0.0;
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const int i = t + k * kT;
        xl[i] += alpha * pl[i];
        r[k] -= alpha * q[k];
        q[k] = dl[i] * r[k];  // z
        rzn += r[k] * q[k];
        rr += r[k] * r[k];
      }
      sum2(rzn, rr, sh, turn);
      const double beta = lane_value(rzn / rz, 0);
      rz = rzn;
      ++it;
      // at the tolerance, not finite or at the limit: the true residual decides
      start = !(rr > thr) || !isfinite(rr) || it >= A.maxit;
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const int i = t + k * kT;
        pl[i] = start ? xl[i] : q[k] + beta * pl[i];
      }
      __syncthreads();
    }
    if (!start && it >= until) {
      how = kPaused;
#pragma unroll
      for (int k = 0; k < R; ++k) {
        A.state[t + k * kT] = r[k];
        A.state[kSmallMaxN + t + k * kT] = pl[t + k * kT];
      }
      break;
    }
  }
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = t + k * kT;
    if (i < n) A.x[i] = xl[i];
  }
  __syncthreads();  // A.out is read by every thread on a resumed start
  if (t == 0) {
    A.out[0] = it;
    A.out[1] = converged;
    A.out[2] = relres;
    A.out[3] = how;
    A.out[4] = rz;
    A.out[5] = thr;
    A.out[6] = restarts;
  }
}

template <int R, int E, int X = 0>
void launch(const SmallArgs &A, hipStream_t s) {
  auto kern = small_pcg_kernel<R, E, X>;
  constexpr size_t bytes = (sizeof(double) * (3 + X) + sizeof(uint16_t) * X) * R * kT;
  GH_CHECK_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)bytes));
  hipLaunchKernelGGL(kern, dim3(1), dim3(kT), bytes, s, A);
  GH_CHECK_HIP(hipGetLastError());
}

}  // namespace

// At most kSmallMaxN rows; the bound on the padded slices is checked by the kernel.
bool pcg_small(Ctx &c, HostCopy &copy, int precond, double rtol, int maxit, double *x,
               const double *b, unsigned char *ws, gh_solve_stats *st) {
  const int64_t n = c.nfree;
  double *at = reinterpret_cast<double *>(ws);
  SmallArgs A{};
  A.n = (int)n;
  A.maxit = maxit;
  A.jacobi = precond == GH_PRECOND_JACOBI;
  A.rtol = rtol;
  A.cp = c.colptr.get();
  A.rv = c.rowval.get();
  A.val = c.nzval.get();
  A.b = b;
  A.x = x;
  A.out = at;
  A.state = at + 16;
  A.wv = A.state + 2 * kSmallMaxN;
  A.wc = reinterpret_cast<uint16_t *>(A.wv + kSmallStream);
  static_assert(kOut <= 16 && sizeof(double) * (16 + 2 * kSmallMaxN + kSmallStream) +
                                      sizeof(uint16_t) * kSmallStream <= kSmallWs, "workspace");
  double h[kOut];
  do {
    if (n <= kT) launch<1, 60>(A, c.stream);
    else if (n <= 2 * kT) launch<2, 32>(A, c.stream);
    else if (n <= 4 * kT) launch<4, 18>(A, c.stream);
    else launch<8, 8, 1>(A, c.stream);
    copy.down(h, A.out, sizeof(h));
    A.resume = 1;
  } while (h[3] == kPaused);
  if (h[3] == kDeclined) return false;
  c.solve_form = GH_SOLVE_WORKGROUP;
  st->iterations = (int)h[0];
  st->converged = h[1] != 0.0;
  st->rel_residual = h[2];
  return true;
}

}  // namespace gh
