// PCG on a box lattice in one launch: the workgroups stay on their compute units for the
// whole solve and keep their rows' matrix in registers (and some in LDS).
//
// The two kernels of an iteration (solve.hip) read the stencil again every time, 28 MB at
// 64³, and pay two launches.  Here a workgroup owns rb consecutive rows, one per thread, with
// the 27 coefficients of the row in registers and x, r, z and D^-1 too (FSAI's G, 14 FP32
// values a row, comes from L2); per iteration only the vector that the stencil multiplies crosses
// workgroups.  It is published to memory, and every workgroup reads the runs its rows need
// (three of rb + 2 (m0 + 1) rows) into LDS, where the direction p of the runs is kept, so
// that z alone is exchanged: p = z + β p is formed for the neighbours' rows as well.
//
// Workgroups meet in exchanges: each stores its partial sums in its own slots, and every
// workgroup polls all slots and adds them in the same order: a barrier and the dot products
// in one, and every workgroup takes the same decisions.  Two an iteration: p·q, then r·z
// with r·r.  Published data and slots are relaxed agent-scope atomics, which the L2s of
// the eight XCDs keep coherent.
//
// Published vectors (z; with FSAI also r and y = G r on the way to z = Gᵀ y) need no
// barrier of their own: what is not published yet holds kEmpty, a NaN that no published
// value is, and a reader polls until it has a value.  z alternates between two buffers.
// With E1, E2 the exchanges of an iteration and z(k) the z published before E2(k):
//  - past E2(k) every workgroup has read z(k-1), r(k) and y(k) (they enter what it sent to
//    E1(k) and E2(k)), so each empties its own rows of them then;
//  - the emptying has completed (s_waitcnt) before the workgroup sends to E1(k+1);
//  - r, y and z(k+1) are published and read past E1(k+1): no reader finds an old value.
// On a (re)start, where there is no E1 between, the vectors are published with a wait
// and read past the exchange instead.
//
// Microseconds an iteration, launched kernels and here: Jacobi 63³ rows 17.1 and 10.2, 31³
// 11.9 and 6.9; FSAI 25.3 and 18.4, 17.5 and 12.0; rows past one a thread, in LDS: 65x64x65
// 19.6 and 15.8, 70³ 20.6 and 16.8.  (Barriers for the published vectors too: 10.7, 7.6, 22.6,
// 16.0.)  What bounds it: the trips through the fabric, 3 to 4 µs an exchange or published
// vector with 245 workgroups, 2 with 14.  Hence the largest workgroups that fit, 512 rows
// at least (31³ with barriers: 256 rows 8.3, 512 7.1, 1024 7.3).  16 waves leave a thread 128
// registers, of which the coefficients take 54: 28 values spill (FSAI 42, rows in LDS 88) to 20,
// 60 and 200 bytes of scratch.
//
// Every wait ends: a workgroup that waits longer than kArrive for the first exchange (some
// workgroups are not on the device: other work holds it) or kLost for a later one sets the
// abort word, which every waiting workgroup polls, and the launched kernels go on from the
// last iterate that reached memory.  Those group the dot products differently, so the last
// bits of a solution depend on which form ended it.  One launch runs at most kPause
// iterations, and holds the compute units that long (21 ms at 63³, 38 ms with FSAI).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "gh_internal.h"

namespace gh {
namespace {

constexpr int kMaxBlocks = 256, kMaxThreads = 1024, kMinRows = 512, kMaxWords = 3, kSets = 4;
constexpr uint64_t kEmpty = 0xfff7a11ce5107000ull;  // a NaN (see exchange)
constexpr int kStageRows = 128;  // rows whose values are staged at once
constexpr int kPause = 2048;
constexpr size_t kMaxLds = 150 * 1024;
constexpr uint64_t kArrive = 200000, kLost = 100000000;  // ticks of 10 ns
constexpr int kOut = 8;
constexpr double kNone = 0, kDone = 1, kPaused = 2;

struct ResidentArgs {
  Box B;
  int rb, maxit, jacobi, resume;
  double rtol;
  const int32_t *cp;
  const double *val, *b;
  const float *g14;
  double *x, *r, *p, *z;
  uint64_t *zpub, *rpub, *ypub;  // published z (two buffers), r and y
  // {kNone, kDone or kPaused, iterations, converged, relative residual; a paused solve's
  //  rz, beta, threshold, restarts}
  double *out;
  uint32_t *abort;  // the abort word, then the most iterations of this launch
  uint64_t *slots;  // [kSets][kMaxWords][kMaxBlocks]
};

// Words that cross workgroups.
__device__ __forceinline__ uint64_t get(const uint64_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store(uint64_t *p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void put(uint64_t *p, uint64_t v) {  // a value: never kEmpty
  store(p, v == kEmpty ? v - 1 : v);
}

// The value again, unknown to the compiler: what is computed from it is computed here and
// does not take a register from one turn of the solve to the next.
__device__ __forceinline__ int fresh(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// State of the waits: exchanges so far, and whether one of the workgroup's was given up.
struct Waits {
  uint32_t num;
  int *dead;  // LDS
};
// For a thread that polls: false when it is time to give up.
__device__ __forceinline__ bool keep_on(const ResidentArgs &A, const Waits &E, int spin,
                                        uint64_t t0, uint64_t limit) {
  if ((spin & 15) != 15) return true;
  if (wall_clock64() - t0 <= limit &&
      __hip_atomic_load(A.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
    return true;
  *E.dead = 1;
  return false;
}
// After a barrier: true when the workgroup gives up (and tells the others).
__device__ __forceinline__ bool gave_up(const ResidentArgs &A, const Waits &E) {
  if (!*E.dead) return false;
  if (threadIdx.x == 0)
    __hip_atomic_store(A.abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// One exchange: v becomes its sums over all workgroups.  False: aborted.  FLUSH: this
// workgroup's stores have completed before its sums are there.  during() runs between
// sending and waiting.  A slot that is not written yet holds kEmpty, so that a sum and the
// news that it is there are one word.  Of the four sets of slots, exchange num writes
// num % 4, and a workgroup past it empties its own slots of (num + 3) % 4: all have read
// those (exchange num - 1), as all have written num; and of two exchanges in turn one
// flushes, so the emptying has completed before this workgroup sends to num + 2, and
// whoever gets past that finds no old value in them.
template <int NS, bool FLUSH, class During>
__device__ __forceinline__ bool exchange(const ResidentArgs &A, Waits &E,
                                         double (&v)[NS ? NS : 1], During during) {
  constexpr int kW = NS ? NS : 1;
  __shared__ double mine[3][16], all[3][kMaxBlocks / 64];
  const int t = fresh(threadIdx.x), lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), nb = (int)gridDim.x;
  const uint32_t num = ++E.num;
  uint64_t *slot = A.slots + (size_t)(num % kSets) * kMaxWords * kMaxBlocks;
  uint64_t *last = A.slots + (size_t)((num + kSets - 1) % kSets) * kMaxWords * kMaxBlocks;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const double w = wave_sum(v[s]);
    if (lane == 0) mine[s][wave] = w;
  }
  if (FLUSH) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (wave == 0) {
    const int q = lane >> 4, i = lane & 15;
    double w = 0.0;
    if (NS) w = row16_sum(q < NS && i < (int)blockDim.x / 64 ? mine[q < NS ? q : 0][i] : 0.0);
    uint64_t word = 0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const uint64_t u = (uint64_t)__double_as_longlong(lane_value(w, 16 * s + 15));
      if (lane == s) word = u;
    }
    if (lane < kW) put(slot + (size_t)lane * kMaxBlocks + blockIdx.x, word);
  }
  during();
  if (wave < kMaxBlocks / 64) {
    uint64_t w[kW] = {};
    const uint64_t t0 = wall_clock64(), limit = num == 1 ? kArrive : kLost;
    for (int spin = 0; t < nb; ++spin) {
      bool here = true;
#pragma unroll
      for (int k = 0; k < kW; ++k) w[k] = get(slot + (size_t)k * kMaxBlocks + t);
#pragma unroll
      for (int k = 0; k < kW; ++k) here = here && w[k] != kEmpty;
      if (here || !keep_on(A, E, spin, t0, limit)) break;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const double sum = wave_sum(t < nb ? __longlong_as_double((long long)w[s]) : 0.0);
      if (lane == 0) all[s][wave] = sum;
    }
  }
  __syncthreads();
  if (wave == 0 && lane < kMaxWords)
    store(last + (size_t)lane * kMaxBlocks + blockIdx.x, kEmpty);
  if (gave_up(A, E)) return false;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < kMaxBlocks / 64; ++k)
      if (64 * k < nb) sum += all[s][k];
    v[s] = lane_value(sum, 0);
  }
  return true;
}
template <int NS>
__device__ __forceinline__ bool exchange(const ResidentArgs &A, Waits &E,
                                         double (&v)[NS ? NS : 1]) {
  return exchange<NS, true>(A, E, v, [] {});
}

// The runs of a workgroup's rows in LDS: run d holds rows i0 + (z0 + d) m0 m1 - m0 - 1 + k,
// k < len = rb + 2 (m0 + 1); zero outside [0, n).
struct Window {
  int n, m0, m01, i0, rb, len;
  __device__ __forceinline__ int at(int t, int o, int z0) const {  // row t's neighbour o
    return (o / 9 - 1 - z0) * len + m0 + 1 + ((o / 3) % 3 - 1) * m0 + (o % 3 - 1) + t;
  }
  // entry e of what run d reads (the own run: only the rows before and after the
  // workgroup's own): how many, position in the run, row
  __device__ __forceinline__ int count(int dz) const { return dz ? len : 2 * (m0 + 1); }
  __device__ __forceinline__ int pos(int dz, int e) const { return dz || e <= m0 ? e : e + rb; }
  __device__ __forceinline__ int row(int dz, int e) const {
    return i0 + dz * m01 - m0 - 1 + pos(dz, e);
  }
};

// A published vector into the runs z0 .. z0 + NZ - 1: issue() starts the loads, finish()
// polls what was not there and stores dst = value (copy) or value + beta dst; own rows: mine.
template <int NZ>
struct Halo {
  uint64_t v[NZ][2];
  __device__ __forceinline__ void issue(const Window &W, const uint64_t *src, int z0) {
    const int t = fresh(threadIdx.x);
#pragma unroll
    for (int d = 0; d < NZ; ++d)
#pragma unroll
      for (int u = 0; u < (z0 + d == 0 ? 1 : 2); ++u) {  // lanes past the end read one address
        const int j = W.row(z0 + d, min(t + u * (int)blockDim.x, W.count(z0 + d) - 1));
        v[d][u] = get(src + min(max(j, 0), W.n - 1));
      }
  }
  __device__ __forceinline__ bool missing(const Window &W, int z0) const {
    bool m = false;
#pragma unroll
    for (int d = 0; d < NZ; ++d)
#pragma unroll
      for (int u = 0; u < (z0 + d == 0 ? 1 : 2); ++u) m = m || v[d][u] == kEmpty;
    return m;
  }
  __device__ __forceinline__ void finish(const Window &W, const ResidentArgs &A, const Waits &E,
                                         const uint64_t *src, int z0, double *dst, bool copy,
                                         double beta, double mine) {
    if (missing(W, z0)) {
      const uint64_t t0 = wall_clock64();
      for (int spin = 0; missing(W, z0) && keep_on(A, E, spin, t0, kLost); ++spin) {
        __builtin_amdgcn_s_sleep(2);
        issue(W, src, z0);  // all again: one round trip however many are missing
      }
    }
    const int t = fresh(threadIdx.x), bd = blockDim.x;
#pragma unroll
    for (int d = 0; d < NZ; ++d) {
      double *run = dst + d * W.len;
      auto one = [&](int e, uint64_t w) {
        const int j = W.row(z0 + d, e), k = W.pos(z0 + d, e);
        const double x = j >= 0 && j < W.n ? __longlong_as_double((long long)w) : 0.0;
        run[k] = copy ? x : x + beta * run[k];
      };
      const int held = z0 + d == 0 ? 1 : 2;
#pragma unroll
      for (int u = 0; u < held; ++u)
        if (t + u * bd < W.count(z0 + d)) one(t + u * bd, v[d][u]);
      for (int e = t + held * bd; e < W.count(z0 + d); e += bd) {  // long lattice rows
        const uint64_t *p = src + min(max(W.row(z0 + d, e), 0), W.n - 1);
        const uint64_t t0 = wall_clock64();
        uint64_t w = get(p);
        for (int spin = 0; w == kEmpty && keep_on(A, E, spin, t0, kLost); ++spin) w = get(p);
        one(e, w);
      }
      if (z0 + d == 0) run[W.m0 + 1 + t] = mine;
    }
  }
};

template <bool FACT, bool EXTRA>
__global__ __launch_bounds__(kMaxThreads) void resident_pcg_kernel(const ResidentArgs A) {
  extern __shared__ __align__(16) double lds[];
  __shared__ int bad, dead;
  const int t = threadIdx.x, n = (int)A.B.n, bd = blockDim.x;
  Window W;
  W.n = n;
  W.m0 = (int)A.B.m0;
  W.m01 = (int)(A.B.m0 * A.B.m1);
  W.i0 = (int)blockIdx.x * A.rb;
  W.rb = A.rb;
  W.len = A.rb + 2 * (W.m0 + 1);
  double *run = lds, *rrun = lds + 3 * W.len, *yrun = lds + 5 * W.len;
  // EXTRA: rows past one per thread, their state and coefficients in LDS
  const int ext = EXTRA ? A.rb - bd : 0;
  double *xs = lds + max(3 * W.len, kStageRows * 27), *rs = xs + ext, *zs = rs + ext;
  double *ps = zs + ext, *ds = ps + ext, *as = ds + ext;
  const bool has2 = EXTRA && t < ext;
  const int i = W.i0 + t, ic = min(i, n - 1);
  const bool own = i < n, own2 = has2 && i + bd < n;
  // coefficients: rows are runs of nzval; a lattice row holds its in-box neighbours in
  // offset order
  double a[27];
  {
    const uint32_t vm = own ? box_valid(A.B, i) : 0;
    const int q0 = A.cp[ic], q1 = A.cp[ic + 1];
    const bool ok = !own || q1 - q0 == __popc(vm);
    if (t == 0) bad = 0;
    __syncthreads();
    if (!ok) bad = 1;
    uint32_t vm2 = 0;
    int q2 = 0;
    if (EXTRA && own2) {
      vm2 = box_valid(A.B, i + bd);
      q2 = A.cp[i + bd];
      if (A.cp[i + bd + 1] - q2 != __popc(vm2)) bad = 1;
    }
    for (int c0 = 0; c0 < A.rb; c0 += kStageRows) {
      const int r0 = min(W.i0 + c0, n), r1 = min(r0 + kStageRows, n);
      const int p0 = A.cp[r0], count = min(A.cp[r1] - p0, kStageRows * 27);
      __syncthreads();
      for (int k = t; k < count; k += bd) lds[k] = A.val[p0 + k];
      __syncthreads();
      if (t >= c0 && t < c0 + kStageRows) {
        int k = min(q0 - p0, kStageRows * 27 - 27);  // in bounds for other matrices too
        if (k < 0) k = 0;
#pragma unroll
        for (int o = 0; o < 27; ++o) {
          const bool in = (vm >> o) & 1u;
          a[o] = in ? lds[k] : 0.0;
          k += in ? 1 : 0;
        }
      }
      if (has2 && t + bd >= c0 && t + bd < c0 + kStageRows) {
        int k = max(min(q2 - p0, kStageRows * 27 - 27), 0);
        for (int o = 0; o < 27; ++o) {
          const bool in = (vm2 >> o) & 1u;
          as[o * ext + t] = in ? lds[k] : 0.0;
          k += in ? 1 : 0;
        }
        const double d = as[13 * ext + t];
        ds[t] = A.jacobi && d != 0.0 ? 1.0 / d : 1.0;
        xs[t] = own2 ? A.x[i + bd] : 0.0;
        rs[t] = zs[t] = ps[t] = 0.0;
      }
    }
    __syncthreads();
    if (bad) {  // not the lattice matrix: the general kernels take it
      if (t == 0)
        __hip_atomic_store(A.abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
  }
  const double dinv = A.jacobi && a[13] != 0.0 ? 1.0 / a[13] : 1.0;
  if (t == 0) dead = 0;
  Waits E{0, &dead};
  int turn = 1;  // the buffer of the last z
  double none[1], xi = own ? A.x[i] : 0.0, ri = 0.0, zi = 0.0, pi = 0.0;
  Halo<3> H;
  auto publish = [&](uint64_t *buf, double v, const double *v2) {
    const int j = W.i0 + fresh(t);
    if (own) put(buf + j, (uint64_t)__double_as_longlong(v));
    if (own2) put(buf + j + bd, (uint64_t)__double_as_longlong(v2[j - W.i0]));
  };
  auto zbuf = [&](int k) { return A.zpub + (k & 1 ? n : 0); };
  // r published: z = Gᵀ G r
  auto apply = [&] {
    float g[14];
    Halo<2> P;
    P.issue(W, A.rpub, -1);
    const int t1 = fresh(t), j1 = min(W.i0 + t1, n - 1);
#pragma unroll
    for (int o = 0; o < 14; ++o) g[o] = A.g14[(int64_t)o * n + j1];
    P.finish(W, A, E, A.rpub, -1, rrun, true, 0.0, ri);
    __syncthreads();
    if (gave_up(A, E)) return false;
    double y = 0.0;
#pragma unroll
    for (int o = 0; o < 14; ++o) y += (double)g[o] * rrun[W.at(t1, o, -1)];
    if (!own) y = 0.0;
    publish(A.ypub, y, nullptr);
    P.issue(W, A.ypub, 0);
    const int t2 = fresh(t), j2 = min(W.i0 + t2, n - 1);
#pragma unroll
    for (int o = 0; o < 14; ++o) g[o] = A.g14[(int64_t)o * n + j2 - box_off(A.B, o)];
    P.finish(W, A, E, A.ypub, 0, yrun, true, 0.0, y);
    __syncthreads();
    if (gave_up(A, E)) return false;
    zi = 0.0;
#pragma unroll
    for (int o = 13; o >= 0; --o) zi += (double)g[o] * yrun[W.at(t2, 26 - o, 0)];
    if (!own) zi = 0.0;
    return true;
  };
  // past the exchange that follows the publication of z: the buffers of the next turn
  auto empty = [&](bool other) {
    if (!own) return;
    const int j = W.i0 + fresh(t);
    if (other) store(zbuf(turn + 1) + j, kEmpty);
    if (other && own2) store(zbuf(turn + 1) + j + bd, kEmpty);
    if (FACT) {
      store(A.rpub + j, kEmpty);
      store(A.ypub + j, kEmpty);
    }
  };
  int it = 0, restarts = 0, converged = 0;
  double relres = INFINITY, rz = 0.0, thr = 0.0, beta = 0.0, how = kDone;
  bool start = !A.resume, first = false;
  if (start) {
    publish(zbuf(++turn), xi, xs);
    if (!exchange<0>(A, E, none)) return;
  } else {
    it = (int)A.out[1];
    rz = A.out[4];
    beta = A.out[5];
    thr = A.out[6];
    restarts = (int)A.out[7];
    if (own) {
      ri = A.r[i];
      pi = A.p[i];
      zi = A.z[i];
    }
    if (own2) {
      rs[t] = A.r[i + bd];
      ps[t] = A.p[i + bd];
      zs[t] = A.z[i + bd];
    }
    publish(zbuf(++turn), pi, ps);
    if (!exchange<0>(A, E, none)) return;
    H.issue(W, zbuf(turn), -1);
    H.finish(W, A, E, zbuf(turn), -1, run, true, 0.0, pi);
    publish(zbuf(++turn), zi, zs);
    if (!exchange<0>(A, E, none)) return;
    empty(true);
  }
  H.issue(W, zbuf(turn), -1);
  // (from memory: as an argument of the kernel it costs registers, 2% of every iteration)
  const int pause = __builtin_amdgcn_readfirstlane((int)A.abort[1]);
  const int until = A.maxit - it > pause ? it + pause : A.maxit;
  // each turn multiplies by A once: a step of the recurrence, or (start) the true residual
  for (;;) {
    pi = start ? xi : first ? zi : zi + beta * pi;
    H.finish(W, A, E, zbuf(turn), -1, run, start || first, beta, pi);
    if (has2) {
      const int e = fresh(t);
      ps[e] = start ? xs[e] : first ? zs[e] : zs[e] + beta * ps[e];
      run[W.at(e + bd, 13, -1)] = ps[e];
    }
    __syncthreads();
    if (gave_up(A, E)) return;
    double q = 0.0;
    const int t1 = fresh(t);
#pragma unroll
    for (int o = 0; o < 27; ++o) q += a[o] * run[W.at(t1, o, -1)];
    if (!own) q = 0.0;
    double q2 = 0.0;
    if (own2) {
      const int e = fresh(t);
#pragma unroll 9
      for (int o = 0; o < 27; ++o) q2 += as[o * ext + e] * run[W.at(e + bd, o, -1)];
    }
    if (start) {
      const double bi = own ? A.b[W.i0 + fresh(t)] : 0.0;
      ri = bi - q;
      zi = dinv * ri;
      double v[3] = {ri * ri, bi * bi, zi * ri};
      if (own2) {
        const int e = fresh(t);
        const double b2 = A.b[W.i0 + e + bd], r2 = b2 - q2, z2 = ds[e] * r2;
        rs[e] = r2;
        zs[e] = z2;
        v[0] += r2 * r2;
        v[1] += b2 * b2;
        v[2] += z2 * r2;
      }
      publish(FACT ? A.rpub : zbuf(++turn), FACT ? ri : zi, zs);
      if (!exchange<3>(A, E, v)) return;
      const double bnorm = sqrt(v[1]) > 0 ? sqrt(v[1]) : 1.0;
      relres = lane_value(sqrt(v[0]) / bnorm, 0);
      converged = relres <= A.rtol;
      if (converged || it >= A.maxit || restarts > 3) break;
      rz = v[2];
      if (FACT) {
        if (!apply()) return;
        publish(zbuf(++turn), zi, nullptr);
        double w[1] = {zi * ri};
        if (!exchange<1>(A, E, w)) return;
        rz = w[0];
      }
      H.issue(W, zbuf(turn), -1);
      empty(true);
      ++restarts;
      thr = lane_value((A.rtol * bnorm) * (A.rtol * bnorm), 0);
      first = true;
      start = false;
      beta = 0.0;  // for a pause right here: the next p is z, p itself still holds x
    } else {
      double pq[1] = {pi * q};
      if (own2) pq[0] += ps[fresh(t)] * q2;
      if (!exchange<1>(A, E, pq)) return;
      const double alpha = lane_value(rz / pq[0], 0);
      xi += alpha * pi;
      ri -= alpha * q;
      zi = dinv * ri;
      if (FACT) {
        publish(A.rpub, ri, nullptr);
        if (!apply()) return;
      }
      double v[2] = {ri * ri, zi * ri};
      if (own2) {
        const int e = fresh(t);
        xs[e] += alpha * ps[e];
        const double r2 = rs[e] - alpha * q2, z2 = ds[e] * r2;
        rs[e] = r2;
        zs[e] = z2;
        v[0] += r2 * r2;
        v[1] += z2 * r2;
      }
      publish(zbuf(++turn), zi, zs);
      if (!exchange<2, false>(A, E, v, [&] { H.issue(W, zbuf(turn), -1); })) return;
      beta = lane_value(v[1] / rz, 0);
      rz = v[1];
      ++it;
      first = false;
      // at the tolerance, not finite or at the limit: the true residual decides
      start = !(v[0] > thr) || !isfinite(v[0]) || it >= A.maxit;
      empty(!start);
      if (start) {
        publish(zbuf(++turn), xi, xs);
        if (!exchange<0>(A, E, none)) return;
        H.issue(W, zbuf(turn), -1);
      }
    }
    if (!start && it >= until) {
      how = kPaused;
      if (own) {
        const int j = W.i0 + fresh(t);
        A.r[j] = ri;
        A.p[j] = pi;
        A.z[j] = zi;
      }
      if (own2) {
        const int e = fresh(t), j = W.i0 + e + bd;
        A.r[j] = rs[e];
        A.p[j] = ps[e];
        A.z[j] = zs[e];
      }
      break;
    }
  }
  if (own) A.x[W.i0 + fresh(t)] = xi;
  if (own2) A.x[W.i0 + bd + fresh(t)] = xs[t];
  if (blockIdx.x == 0 && t == 0) {
    A.out[0] = how;
    A.out[1] = it;
    A.out[2] = converged;
    A.out[3] = relres;
    A.out[4] = rz;
    A.out[5] = beta;
    A.out[6] = thr;
    A.out[7] = restarts;
  }
}

// Before each launch: no exchange has happened, nothing is published or aborted.
__global__ void resident_clear_kernel(ResidentArgs A, int pause, bool abort) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < kSets * kMaxWords * kMaxBlocks) A.slots[k] = kEmpty;
  if (k < (int)A.B.n) {
    A.zpub[k] = A.zpub[k + A.B.n] = kEmpty;
    if (A.rpub) A.rpub[k] = A.ypub[k] = kEmpty;
  }
  if (k == 0) {
    A.abort[0] = abort;
    A.abort[1] = (uint32_t)pause;
    A.out[0] = kNone;
  }
}

// rb rows per workgroup, one per thread up to 1024; without FSAI the rows past that are
// kept in LDS (5 vectors and 27 coefficients each) while it lasts.
struct Shape {
  int rb, threads, blocks;
  size_t lds;
};
Shape shape(const Box &B, int cus, bool fact) {
  const int64_t nb = std::min(cus, kMaxBlocks);
  const int64_t rb = std::max<int64_t>(((B.n + nb - 1) / nb + 63) / 64 * 64, kMinRows);
  const int64_t threads = std::min<int64_t>(rb, kMaxThreads);
  const int64_t runs = std::max<int64_t>((fact ? 7 : 3) * (rb + 2 * (B.m0 + 1)), kStageRows * 27);
  return {(int)std::min<int64_t>(rb, INT32_MAX), (int)threads, (int)((B.n + rb - 1) / rb),
          sizeof(double) * (size_t)(runs + 32 * (rb - threads))};
}

int compute_units(int device) {
  int v = 0;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
    return 0;
  return v;
}

// One resident solve per device at a time: two that each hold a part of the device
// would wait for each other until both give up.
constexpr int kMaxDevices = 64;
std::atomic<bool> g_busy[kMaxDevices];
struct Turn {
  std::atomic<bool> *flag = nullptr;
  explicit Turn(int device) {
    if (device < 0 || device >= kMaxDevices) return;
    bool idle = false;
    if (g_busy[device].compare_exchange_strong(idle, true)) flag = &g_busy[device];
  }
  ~Turn() {
    if (flag) flag->store(false);
  }
};

}  // namespace

bool resident_system(const Ctx &c, const Box &B, int precond) {
  const char *off = std::getenv("GRIDAP_HIP_RESIDENT_PCG");
  if ((off && off[0] == '0') || std::getenv("GRIDAP_HIP_STENCIL_PCG")) return false;
  const int cus = compute_units(c.device);
  if (cus < 1 || B.n < 1) return false;
  const Shape S = shape(B, cus, precond == GH_PRECOND_FSAI);
  return (S.rb == S.threads || precond != GH_PRECOND_FSAI) && S.lds <= kMaxLds;
}

bool pcg_resident(Ctx &c, const Box &B, int precond, double rtol, int maxit, double *x,
                  const double *b, double *const (&state)[3], double *const (&pub)[3],
                  unsigned char *ws, gh_solve_stats *st, int *done) {
  *done = 0;
  static_assert(sizeof(double) * (kOut + 8) + sizeof(uint64_t) * kSets * kMaxWords * kMaxBlocks <=
                    kResidentWs, "workspace");
  Turn turn(c.device);
  if (!turn.flag) return false;
  const bool fact = precond == GH_PRECOND_FSAI;
  const Shape S = shape(B, compute_units(c.device), fact);
  ResidentArgs A{};
  A.B = B;
  A.rb = S.rb;
  A.maxit = maxit;
  A.jacobi = precond == GH_PRECOND_JACOBI;
  int pause = kPause;
  if (const char *env = std::getenv("GRIDAP_HIP_RESIDENT_PAUSE"))
    pause = std::min(std::max(std::atoi(env), 1), kPause);
  A.rtol = rtol;
  A.cp = c.colptr.get();
  A.val = c.nzval.get();
  A.b = b;
  A.g14 = fact ? c.g14.get() : nullptr;
  A.x = x;
  A.r = state[0];
  A.p = state[1];
  A.z = state[2];
  A.zpub = reinterpret_cast<uint64_t *>(pub[0]);
  A.rpub = fact ? reinterpret_cast<uint64_t *>(pub[1]) : nullptr;
  A.ypub = fact ? reinterpret_cast<uint64_t *>(pub[2]) : nullptr;
  A.out = reinterpret_cast<double *>(ws);
  A.abort = reinterpret_cast<uint32_t *>(A.out + kOut);
  A.slots = reinterpret_cast<uint64_t *>(A.out + kOut + 8);
  auto kern = fact ? resident_pcg_kernel<true, false>
              : S.rb > S.threads ? resident_pcg_kernel<false, true>
                                 : resident_pcg_kernel<false, false>;
  GH_CHECK_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)S.lds));
  // for tests: in the launch of this number the last workgroup's rows never come, and whoever
  // waits finds the abort word set
  const char *env = std::getenv("GRIDAP_HIP_RESIDENT_GIVE_UP");
  const int lose = env && S.blocks > 1 ? std::atoi(env) : -1;
  const int64_t clear = std::max<int64_t>(B.n, kSets * kMaxWords * kMaxBlocks);
  double h[kOut + 1];
  for (int launch = 0;; ++launch) {
    hipLaunchKernelGGL(resident_clear_kernel, dim3((unsigned)((clear + 255) / 256)), dim3(256), 0,
                       c.stream, A, pause, launch == lose);
    hipLaunchKernelGGL(kern, dim3((unsigned)S.blocks - (launch == lose)),
                       dim3((unsigned)S.threads), S.lds, c.stream, A);
    GH_CHECK_HIP(hipGetLastError());
    HostCopy copy(c);
    copy.down(h, A.out, sizeof(h));
    uint32_t aborted;
    std::memcpy(&aborted, h + kOut, sizeof(aborted));
    if (aborted || h[0] == kNone) return false;
    if (h[0] != kPaused) break;
    *done = (int)h[1];
    A.resume = 1;
  }
  c.solve_form = GH_SOLVE_RESIDENT;
  st->iterations = (int)h[1];
  st->converged = h[2] != 0.0;
  st->rel_residual = h[3];
  return true;
}

}  // namespace gh
