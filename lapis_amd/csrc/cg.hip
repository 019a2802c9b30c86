// Conjugate gradients on the device: the solver examples/pcg_solve.py:52-101
// lowers to, with its scalars kept in device memory between kernels.
//
// Reference iteration (one pass of the scf.while, :74-98):
//   Ap = A p ; pAp = p.Ap ; rz = r.z ; alpha = rz/pAp
//   x = 1*x + alpha*p ; r = 1*r + (-alpha)*Ap ; rr = r.r
//   relres = sqrt(rr)/sqrt(r0.r0) ; leave if !(relres > tol) or i == maxiter
//   z = r*dinv ; rz' = r.z ; beta = rz'/rz ; p = 1*z + beta*p ; i = i+1
// r.z at the top of an iteration is the rz' of the one before (same vectors), so
// it is carried instead of recomputed; without a preconditioner z is r and rz' is rr.
//
// A dot product never needs a launch of its own: the vector kernel that produces the
// operands leaves one partial per block, and EVERY block of the next vector kernel
// adds those partials (at most 2048 doubles, from L2) in index order before it
// starts, so all blocks hold the same bits of alpha, beta and relres.  Kernel
// boundaries do the ordering; no block needs a device-scope fence (on a multi-XCD
// part such a fence writes back and invalidates L2, and two thousand of them per
// kernel cost more than the vector pass itself).  The iteration number is a kernel
// argument (the host knows which iteration it is queueing); scalars that one kernel
// both reads and replaces (r.z) are kept twice, indexed by iteration parity.
//
// x is needed by nobody until the solve ends, so x += alpha p is made by the kernel
// that reads p anyway to replace it (p = z + beta p), not by the one that updates r, and
// there for two iterations at once: odd iterations leave their p where it is (the next p
// goes into a second buffer), even ones add the alpha p of both, x being read and written
// half as often.  The pass that decides to leave adds what is owed and makes no new p.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <mutex>
#include <vector>

#include "blas1.hpp"
#include "common.hpp"
#include "plan.hpp"
#include "rowsplit_fix.hpp"

namespace lapis {

struct CgState {
  double pAp;      // p . Ap of the last iteration (diagnostic)
  double rz[2];    // r . z entering iteration i is rz[i & 1]
  double rr;       // r . r after the update
  double initres;  // sqrt(r0 . r0)
  double relres;
  double alpha[2]; // r.z / p.Ap of iteration i is alpha[i & 1]
  unsigned long long done_iter;  // 0 while iterating, then the reference's counter i at exit (it starts at 1)
  unsigned long long maxiter;
  double tol;
};

// What the device writes into pinned host memory.
struct CgProgress {
  unsigned long long iter;  // last iteration whose convergence test was made; kLeft is set when it left
  double relres;            // of the iteration that left
};
constexpr unsigned long long kLeft = 1ull << 63;

__device__ __forceinline__ double block_sum_256d(double v, double *lds4) {
  v = group_sum<64>(v);
  if ((threadIdx.x & 63) == 0) lds4[threadIdx.x >> 6] = v;
  __syncthreads();
  const double total = ((lds4[0] + lds4[1]) + lds4[2]) + lds4[3];
  __syncthreads();
  return total;
}

// The exit mark, read once per block: block 0 of the kernel that makes the convergence
// test sets it while other blocks of the same kernel may still be starting, and
// every thread of a block has to take the same way past the barriers below.
__device__ __forceinline__ unsigned long long block_done_iter(const CgState *st) {
  __shared__ unsigned long long seen;
  if (threadIdx.x == 0) seen = st->done_iter;
  __syncthreads();
  const unsigned long long d = seen;
  __syncthreads();
  return d;
}

// Sum of partials[0..count) in a fixed order, by one block of 256 threads.
__device__ __forceinline__ double ordered_total(const double *partials, int count, double *lds4) {
  double s = 0.0;
  for (int i = threadIdx.x; i < count; i += 256) s = s + partials[i];
  return block_sum_256d(s, lds4);
}

// The vector passes below walk their arrays two doubles (one 128-bit access) per
// thread and trip when every array is 16-byte aligned (`vec`), element by element
// otherwise; an odd last element is taken by the scalar tail.
#define CG_GRID_STRIDE(i, first, count) \
  for (long long i = (first) + (long long)blockIdx.x * 256 + threadIdx.x; i < (count); i += (long long)gridDim.x * 256)

__device__ __forceinline__ v2d ld2(const double *p, long long i) { return reinterpret_cast<const v2d *>(p)[i]; }
__device__ __forceinline__ void st2(double *p, long long i, v2d v) { reinterpret_cast<v2d *>(p)[i] = v; }

// r0 = b, p0 = r0*dinv (or r0), x0 = 0; block partials of r0.r0 and r0.z0.
__global__ __launch_bounds__(256) void cg_init_kernel(long long n, const double *__restrict__ b,
                                                      const double *__restrict__ dinv, double *__restrict__ x,
                                                      double *__restrict__ r, double *__restrict__ p,
                                                      double *__restrict__ partials, int divide) {
  __shared__ double lds4[4];
  double rr = 0.0, rz = 0.0;
  CG_GRID_STRIDE(i, 0, n) {
    const double ri = b[i];
    const double zi = dinv ? (divide ? ri / dinv[i] : ri * dinv[i]) : ri;
    r[i] = ri;
    p[i] = zi;
    x[i] = 0.0;
    rr = rr + ri * ri;
    rz = rz + ri * zi;
  }
  const double brr = block_sum_256d(rr, lds4);
  const double brz = block_sum_256d(rz, lds4);
  if (threadIdx.x == 0) {
    partials[blockIdx.x] = brr;
    partials[kDotMaxBlocks + blockIdx.x] = brz;
  }
}

// block partials of p . Ap
__global__ __launch_bounds__(256) void cg_pap_kernel(long long n, const double *__restrict__ p,
                                                     const double *__restrict__ Ap, double *__restrict__ partials,
                                                     int vec) {
  __shared__ double lds4[4];
  double acc = 0.0;
  const long long nv = vec ? n / 2 : 0;
  CG_GRID_STRIDE(i, 0, nv) {
    const v2d a = ld2(p, i), b = ld2(Ap, i);
    acc = acc + a.x * b.x;
    acc = acc + a.y * b.y;
  }
  CG_GRID_STRIDE(i, 2 * nv, n) acc = acc + p[i] * Ap[i];
  const double bsum = block_sum_256d(acc, lds4);
  if (threadIdx.x == 0) partials[blockIdx.x] = bsum;
}

// Sums of `count` partial sums in at most kReducedPartials parts, a part per block, each in a fixed order.
constexpr int kReducedPartials = 64;
__global__ __launch_bounds__(256) void cg_reduce_partials_kernel(int count, const double *__restrict__ in,
                                                                 double *__restrict__ out) {
  __shared__ double lds4[4];
  const int per = (count + (int)gridDim.x - 1) / (int)gridDim.x;
  const int first = (int)blockIdx.x * per;
  const double sum = ordered_total(in + first, min(per, count - first), lds4);
  if (threadIdx.x == 0) out[blockIdx.x] = sum;
}

// The same partials when Ap came from the row-split SpMV kernel with its fix-up left out
// and the chunk sums of p[r]*Ap[r] over uncut rows taken (`chunk_pap`): thread t of a
// block completes the row cut at chunk boundary c (if that boundary is the first to cut
// it), adds that row's p[r]*Ap[r], and adds chunk c's sum.  Neither vector is read in
// full again.  Chunks and boundaries are dealt to blocks and lanes in a fixed order.
template <int CH>
__global__ __launch_bounds__(256) void cg_pap_fix_kernel(int nchunks, int chunks_per_block,
                                                         const double *__restrict__ p, double *Ap,
                                                         const double *__restrict__ chunk_pap,
                                                         double *__restrict__ partials,
                                                         const int *__restrict__ pos,
                                                         const int *__restrict__ chunk_row,
                                                         const double *__restrict__ part_first,
                                                         const double *__restrict__ part_last) {
  __shared__ double lds4[4];
  const long long c0 = (long long)blockIdx.x * chunks_per_block;
  const long long c1 = std::min<long long>(nchunks, c0 + chunks_per_block);
  double acc = 0.0;
  for (long long base = c0; base < c1; base += 256) {
    const long long c = base + threadIdx.x;
    const bool mine = c < c1;
    bool owner;
    int r;
    const double total = rowsplit_row_total<double, CH>((mine && c >= 1) ? c : nchunks, nchunks, pos, chunk_row,
                                                        part_first, part_last, owner, r);
    if (owner) {
      Ap[r] = total;
      acc = acc + p[r] * total;
    }
    if (mine) acc = acc + chunk_pap[c];
  }
  const double bsum = block_sum_256d(acc, lds4);
  if (threadIdx.x == 0) partials[blockIdx.x] = bsum;
}

// z = r dinv, r / dinv or r
enum { kNoPrec = 0, kMultiply = 1, kDivide = 2 };
template <int PREC>
__device__ __forceinline__ double preconditioned(double r, double d) {
  return PREC == kDivide ? r / d : PREC == kMultiply ? r * d : r;
}

// r -= alpha Ap ; block partials of r.r and, preconditioned, of r.z.   alpha = r.z / p.Ap with p.Ap summed here
// from the partials the p.Ap kernel left; block 0 keeps alpha for the kernel that updates x and p.
// Ap is read here for the last time: it goes through streaming accesses, so that it does not
// push p, which the next SpMV gathers from, out of the caches.
template <int PREC>
__global__ __launch_bounds__(256) void cg_update_r_kernel(long long n, const double *__restrict__ Ap,
                                                          double *__restrict__ r, const double *__restrict__ dinv,
                                                          CgState *st, unsigned long long iter, int count,
                                                          const double *__restrict__ pap_partials,
                                                          double *__restrict__ rr_partials,
                                                          double *__restrict__ rz_partials, int vec) {
  __shared__ double lds4[4];
  if (block_done_iter(st)) return;
  const double pAp = ordered_total(pap_partials, count, lds4);
  const double alpha = st->rz[iter & 1] / pAp;
  const double malpha = -alpha;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->pAp = pAp;
    st->alpha[iter & 1] = alpha;
  }
  double rr = 0.0, rz = 0.0;
  const long long nv = vec ? n / 2 : 0;
  CG_GRID_STRIDE(i, 0, nv) {
    const v2d av = load_stream(reinterpret_cast<const v2d *>(Ap) + i);
    v2d rv = ld2(r, i), dv = {0.0, 0.0};
    if (PREC) dv = ld2(dinv, i);
    rv.x = rv.x + av.x * malpha;
    rv.y = rv.y + av.y * malpha;
    st2(r, i, rv);
    rr = rr + rv.x * rv.x;
    rr = rr + rv.y * rv.y;
    if (PREC) {
      rz = rz + rv.x * preconditioned<PREC>(rv.x, dv.x);
      rz = rz + rv.y * preconditioned<PREC>(rv.y, dv.y);
    }
  }
  CG_GRID_STRIDE(i, 2 * nv, n) {
    const double rt = Ap[i] * malpha;
    const double ri = r[i] + rt;
    r[i] = ri;
    rr = rr + ri * ri;
    if (PREC) rz = rz + ri * preconditioned<PREC>(ri, dinv[i]);
  }
  const double brr = block_sum_256d(rr, lds4);
  if (threadIdx.x == 0) rr_partials[blockIdx.x] = brr;
  if (PREC) {
    const double brz = block_sum_256d(rz, lds4);
    if (threadIdx.x == 0) rz_partials[blockIdx.x] = brz;
  }
}

// The convergence test of examples/pcg_solve.py:84-90, made by every block from the
// r.r partials: leave when !(relres > tol) or i == maxiter.  Block 0 records the exit, and tells the host how far
// the device is (relaxed stores to pinned memory: nothing waits for them, and the host reads relres after it has
// waited for the stream).
__device__ __forceinline__ bool cg_continues(CgState *st, CgProgress *host, unsigned long long iter, double rr) {
  const double relres = sqrt(rr) / st->initres;
  const bool go_on = (relres > st->tol) && (iter != st->maxiter);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->rr = rr;
    st->relres = relres;
    if (!go_on) {
      st->done_iter = iter;
      host->relres = relres;
    }
    __hip_atomic_store(&host->iter, go_on ? iter : iter | kLeft, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  return go_on;
}

// Elementwise pieces of the masked operator and of the moment right-hand sides
// (examples/hitting_times.py:73-93, :166-177, :181-198).
// mode 0: out = (d*t - out) * m     (end of plpt; t = mask*x, out holds A t)
// mode 1: out = (d*t + out) * m     (right-hand side of the second moment; t = mom1, out holds A mom1)
__global__ __launch_bounds__(256) void masked_combine_kernel(long long n, int mode, const double *__restrict__ d,
                                                             const double *__restrict__ t,
                                                             const double *__restrict__ m, double *out) {
  CG_GRID_STRIDE(i, 0, n) {
    const double t1 = d[i] * t[i];
    const double t2 = mode == 0 ? t1 - out[i] : t1 + out[i];
    out[i] = t2 * m[i];
  }
}

__global__ __launch_bounds__(256) void normalize_mom2_kernel(long long n, const double *__restrict__ m1,
                                                             const double *__restrict__ m2, double *__restrict__ out) {
  CG_GRID_STRIDE(i, 0, n) {
    const double sq = m1[i] * m1[i];
    out[i] = sqrt(m2[i] - sq);
  }
}

// Convergence test; p_next = z + beta p with beta = (new r.z) / (old r.z) and z made from r; in even iterations
// x += alpha' p' + alpha p, with the p' and alpha' of the iteration before (p_next overwrites p').
// Every block makes the test, from the r.r partials.  The pass that leaves (the exit mark may already name this very
// iteration) adds to x what is owed to it and makes no p; passes queued behind it find an older mark and touch
// nothing.  x and r go through streaming accesses: they are touched for the last time in this iteration and must not
// push p out of the caches.
template <int PREC, bool EVEN>
__global__ __launch_bounds__(256) void cg_update_xp_kernel(long long n, const double *__restrict__ r,
                                                           const double *__restrict__ dinv, const double *__restrict__ p,
                                                           double *__restrict__ other, double *__restrict__ x, CgState *st,
                                                           CgProgress *host, unsigned long long iter, int count,
                                                           const double *__restrict__ rr_partials,
                                                           const double *__restrict__ rz_partials, int vec) {
  __shared__ double lds4[4];
  const unsigned long long mark = block_done_iter(st);
  if (mark != 0 && mark != iter) return;
  const double rr = ordered_total(rr_partials, count, lds4);
  const double rz_new = PREC ? ordered_total(rz_partials, count, lds4) : rr;
  const bool go_on = cg_continues(st, host, iter, rr);
  const double alpha = st->alpha[iter & 1], alpha_before = st->alpha[(iter + 1) & 1];
  const long long nv = vec ? n / 2 : 0;
  if (!go_on) {
    CG_GRID_STRIDE(i, 0, nv) {
      const v2d pv = ld2(p, i);
      v2d xv = load_stream(reinterpret_cast<const v2d *>(x) + i);
      if (EVEN) {
        const v2d qv = ld2(other, i);
        xv.x = xv.x + qv.x * alpha_before;
        xv.y = xv.y + qv.y * alpha_before;
      }
      xv.x = xv.x + pv.x * alpha;
      xv.y = xv.y + pv.y * alpha;
      store_stream(reinterpret_cast<v2d *>(x) + i, xv);
    }
    CG_GRID_STRIDE(i, 2 * nv, n) {
      double xi = x[i];
      if (EVEN) xi = xi + other[i] * alpha_before;
      x[i] = xi + p[i] * alpha;
    }
    return;
  }
  const double beta = rz_new / st->rz[iter & 1];
  if (blockIdx.x == 0 && threadIdx.x == 0) st->rz[(iter + 1) & 1] = rz_new;
  CG_GRID_STRIDE(i, 0, nv) {
    v2d zv = load_stream(reinterpret_cast<const v2d *>(r) + i);
    if (PREC) {
      const v2d dv = load_stream(reinterpret_cast<const v2d *>(dinv) + i);
      zv.x = preconditioned<PREC>(zv.x, dv.x);
      zv.y = preconditioned<PREC>(zv.y, dv.y);
    }
    const v2d pv = ld2(p, i);
    if (EVEN) {
      const v2d qv = ld2(other, i);
      v2d xv = load_stream(reinterpret_cast<const v2d *>(x) + i);
      xv.x = xv.x + qv.x * alpha_before;
      xv.y = xv.y + qv.y * alpha_before;
      xv.x = xv.x + pv.x * alpha;
      xv.y = xv.y + pv.y * alpha;
      store_stream(reinterpret_cast<v2d *>(x) + i, xv);
    }
    v2d nv2;
    nv2.x = zv.x + pv.x * beta;
    nv2.y = zv.y + pv.y * beta;
    st2(other, i, nv2);
  }
  CG_GRID_STRIDE(i, 2 * nv, n) {
    const double zi = preconditioned<PREC>(r[i], PREC ? dinv[i] : 1.0);
    const double pi = p[i];
    if (EVEN) {
      const double xi = x[i] + other[i] * alpha_before;
      x[i] = xi + pi * alpha;
    }
    other[i] = zi + pi * beta;
  }
}

// One block, once per solve: the scalars of the initial residual.
__global__ __launch_bounds__(256) void cg_init_scalar_kernel(int count, const double *__restrict__ partials,
                                                             CgState *st, unsigned long long maxiter, double tol) {
  __shared__ double lds4[4];
  const double trr = ordered_total(partials, count, lds4);
  const double trz = ordered_total(partials + kDotMaxBlocks, count, lds4);
  if (threadIdx.x == 0) {
    st->initres = sqrt(trr);
    st->rz[1] = trz;  // the first iteration is i = 1
    st->done_iter = 0;
    st->maxiter = maxiter;
    st->tol = tol;
  }
}

// ---- small systems: the whole solve in one launch -------------------------------------------------
//
// On a system of a few ten thousand rows an iteration of the kernels above is launches and gaps (6 launches,
// 25 us per iteration at 16 384 rows, of which the data of an iteration is worth 1 us; 6.3 us here: a whole solve of 40
// iterations 1.50 -> 0.27 ms, 490 000 rows 2.20 -> 0.68 ms).  What bounds it: two exchanges with the sums and barriers
// around them, 2.5 us each across 32 workgroups, and a dependent trip past L2 for every four entries of a row, 0.6 us each
// (16 384 rows of 3, 5, 7, 9 and 13 entries: 5.65, 6.25, 6.24, 6.79 and 7.34 us; one workgroup of 512 rows: 4.2 to 5.4).  Here one workgroup per
// compute unit keeps a stretch of rows for the whole solve: their entries in LDS, their r, x, p and dinv in
// registers.  What the others need goes through memory: z (r where there is no preconditioner) and p, and two
// exchanges per iteration, each a sum over the workgroups and a barrier in one:
//     p = z + beta p (own rows) ; Ap = A p, with p of the gathered columns made on the way from z and the previous p
//   exchange p.Ap -> alpha
//     x += alpha p ; r -= alpha Ap ; z = r dinv
//   exchange r.r, r.z -> convergence test, beta
// An exchange is one hop: workgroup g writes its partial sums, each half tagged with the exchange's number, into
// its slot, and every workgroup reads all slots until all carry the number.  Slots alternate between two sets:
// a set is written again only after every workgroup has been through the exchange between.  p alternates
// between two buffers for the same reason.
// Shared words are written and read with agent-scope accesses (past the L2s, which are not coherent across the
// XCDs); a wavefront waits for its own stores before its workgroup's slot is written.  Every wait is bounded: a
// workgroup whose wait runs out (the others were not resident) gives up, so do all, and the host takes the
// kernels above instead.  A launch makes at most `budget` iterations; the host continues from what it left.
constexpr int kSmallMaxBlocks = 256;
constexpr int kSmallThreads = 512;
constexpr int kSmallMaxRowsPerThread = 4;
constexpr int kSmallLdsBytes = 150 * 1024;

struct CgSmallResult {
  unsigned long long done_iter;  // the reference's counter at exit, 0 when the budget ended first
  double relres;
  double rz, beta, initres;  // where the next launch goes on
  unsigned fault;
  unsigned pad;
};

struct CgSmallArgs {
  int n, rows, blocks;  // rows per workgroup, workgroups
  int entries;          // LDS room for entries of a workgroup
  const int *pos, *crd;
  const double *val, *b, *dinv;
  double *x, *r, *z, *p0, *p1;
  unsigned long long *slots;  // [2][kSmallMaxBlocks][4]
  unsigned epoch;             // number of the first exchange
  int resume;
  unsigned long long iter0;  // iterations made by earlier launches
  unsigned long long maxiter, budget;
  double tol, rz, beta, initres;
  int spins;           // polls of an exchange before it gives up
  CgSmallResult *out;  // host memory
};

__device__ __forceinline__ double shared_load(const double *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void shared_store(double *p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Sums v0 and v1 over all threads of all workgroups, in a fixed order; false when the wait ran out.
// lds: 2 * 8 + 2 * kSmallMaxBlocks doubles.
template <int V>
__device__ __forceinline__ bool small_exchange(const CgSmallArgs &a, unsigned epoch, double (&v)[V], double *lds) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double *part = lds + 16;
#pragma unroll
  for (int i = 0; i < V; ++i) v[i] = group_sum<64>(v[i]);
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < V; ++i) lds[i * 8 + wave] = v[i];
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's z and p are where the others read them
  __syncthreads();
  unsigned long long *set = a.slots + (size_t)(epoch & 1) * kSmallMaxBlocks * 4;
  if (tid < 2 * V) {
    double sum = 0.0;
    for (int w = 0; w < kSmallThreads / 64; ++w) sum = sum + lds[(tid >> 1) * 8 + w];
    const unsigned long long bits = __builtin_bit_cast(unsigned long long, sum);
    const unsigned half = (unsigned)(tid & 1 ? bits >> 32 : bits);
    __hip_atomic_store(set + (size_t)blockIdx.x * 4 + tid, ((unsigned long long)epoch << 32) | half, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
  bool ok = true;
  if (tid < a.blocks) {
    unsigned long long w[2 * V] = {};
    ok = false;
    for (int spin = 0; spin < a.spins; ++spin) {
      ok = true;
#pragma unroll
      for (int i = 0; i < 2 * V; ++i)
        w[i] = __hip_atomic_load(set + (size_t)tid * 4 + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int i = 0; i < 2 * V; ++i) ok = ok && (unsigned)(w[i] >> 32) == epoch;
      if (ok) break;
    }
#pragma unroll
    for (int i = 0; i < V; ++i)
      part[i * kSmallMaxBlocks + tid] =
          __builtin_bit_cast(double, (w[2 * i] & 0xffffffffull) | (w[2 * i + 1] << 32));
  }
  ok = __syncthreads_and(ok);
#pragma unroll
  for (int i = 0; i < V; ++i) {
    double sum = 0.0;
    for (int g = lane; g < a.blocks; g += 64) sum = sum + part[i * kSmallMaxBlocks + g];
    v[i] = group_sum<64>(sum);
  }
  __syncthreads();  // the next exchange writes the same LDS
  return ok;
}

template <int RPT, bool PRE>
__global__ __launch_bounds__(kSmallThreads) void cg_small_kernel(CgSmallArgs a) {
  extern __shared__ __align__(16) unsigned char small_lds[];
  __shared__ double xlds[16 + 2 * kSmallMaxBlocks];
  double *lval = reinterpret_cast<double *>(small_lds);
  int *lcrd = reinterpret_cast<int *>(lval + a.entries);
  const int tid = threadIdx.x;
  const int row0 = blockIdx.x * a.rows;
  const int rows_here = min(a.rows, a.n - row0);
  const int first = a.pos[row0], last = a.pos[row0 + rows_here];
  for (int j = tid; j < last - first; j += kSmallThreads) {
    lval[j] = a.val[first + j];
    lcrd[j] = a.crd[first + j];
  }
  double r[RPT], x[RPT], p[RPT], z[RPT], d[RPT];
  int lo[RPT], hi[RPT];
  double sums[2] = {0.0, 0.0};
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int k = tid + i * kSmallThreads;
    const bool have = k < rows_here;
    const int row = row0 + k;
    lo[i] = have ? a.pos[row] - first : 0;
    hi[i] = have ? a.pos[row + 1] - first : 0;
    d[i] = have && PRE ? a.dinv[row] : 1.0;
    p[i] = 0.0;
    if (a.resume) {
      r[i] = have ? a.r[row] : 0.0;
      x[i] = have ? a.x[row] : 0.0;
      z[i] = PRE ? r[i] * d[i] : r[i];
      p[i] = have ? shared_load((a.iter0 & 1 ? a.p1 : a.p0) + row) : 0.0;
    } else {
      r[i] = have ? a.b[row] : 0.0;
      x[i] = 0.0;
      z[i] = PRE ? r[i] * d[i] : r[i];
      if (have) shared_store(a.z + row, z[i]);
      sums[0] = sums[0] + r[i] * r[i];
      sums[1] = sums[1] + r[i] * z[i];
    }
  }
  unsigned epoch = a.epoch;
  double rz = a.rz, beta = a.beta, initres = a.initres;
  bool ok = true;
  if (a.resume) {
    __syncthreads();  // the entries are in LDS
  } else {
    ok = small_exchange<2>(a, epoch++, sums, xlds);
    initres = sqrt(sums[0]);
    rz = sums[1];
  }
  double relres = 0.0;
  unsigned long long iter = a.iter0, done = 0;
  bool first_pass = !a.resume;
  while (ok && iter - a.iter0 < a.budget) {
    ++iter;  // the reference's counter of this pass
    double *pnew = iter & 1 ? a.p1 : a.p0;
    const double *pold = iter & 1 ? a.p0 : a.p1;
    double Ap[RPT];
    double pAp[1] = {0.0};
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int k = tid + i * kSmallThreads;
      if (first_pass) {
        p[i] = z[i];
      } else {
        const double pt = p[i] * beta;
        p[i] = z[i] + pt;
      }
      if (k < rows_here) shared_store(pnew + row0 + k, p[i]);
      double acc = 0.0;
      for (int j = lo[i]; j < hi[i]; j += 4) {  // four entries' z and p in flight, summed in ascending order
        double zj[4], pj[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int c = lcrd[min(j + u, hi[i] - 1)];
          zj[u] = shared_load(a.z + c);
          pj[u] = first_pass ? 0.0 : shared_load(pold + c);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (j + u < hi[i]) {
            const double pt = pj[u] * beta;
            const double pv = first_pass ? zj[u] : zj[u] + pt;
            acc = acc + lval[j + u] * pv;
          }
        }
      }
      Ap[i] = acc;
      pAp[0] = pAp[0] + p[i] * acc;
    }
    if (!(ok = small_exchange<1>(a, epoch++, pAp, xlds))) break;
    const double alpha = rz / pAp[0];
    const double malpha = -alpha;
    sums[0] = sums[1] = 0.0;
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int k = tid + i * kSmallThreads;
      const double xt = p[i] * alpha;
      x[i] = x[i] + xt;
      const double rt = Ap[i] * malpha;
      r[i] = r[i] + rt;
      z[i] = PRE ? r[i] * d[i] : r[i];
      if (k < rows_here) shared_store(a.z + row0 + k, z[i]);
      sums[0] = sums[0] + r[i] * r[i];
      sums[1] = sums[1] + r[i] * z[i];
    }
    if (!(ok = small_exchange<2>(a, epoch++, sums, xlds))) break;
    relres = sqrt(sums[0]) / initres;
    beta = sums[1] / rz;
    rz = sums[1];
    first_pass = false;
    if (!(relres > a.tol) || iter == a.maxiter) {
      done = iter;
      break;
    }
  }
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int k = tid + i * kSmallThreads;
    if (ok && k < rows_here) {
      a.x[row0 + k] = x[i];
      if (!done) a.r[row0 + k] = r[i];
    }
  }
  if (tid == 0 && (blockIdx.x == 0 || !ok)) {
    if (!ok) {
      __hip_atomic_store(&a.out->fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    } else {
      a.out->done_iter = done;
      a.out->relres = relres;
      a.out->rz = rz;
      a.out->beta = beta;
      a.out->initres = initres;
    }
  }
}

}  // namespace lapis

using namespace lapis;

namespace {

// Scratch of one solve: device memory for the scalars, partial sums and exchange slots, and a word of pinned
// host memory the device reports to.  A solve takes one for its duration (it synchronises its stream before it
// returns), so a scratch is never shared; at most kKeptScratch are kept, until lapis_hip_finalize.
struct CgScratch {
  int device = 0;
  CgState *state = nullptr;
  double *partials = nullptr;
  unsigned long long *slots = nullptr;
  unsigned epoch = 1;  // slots carry smaller numbers only
  CgProgress *progress = nullptr;
  CgSmallResult *host_result = nullptr;
  void *device_block = nullptr, *host_block = nullptr;
  double *parts = nullptr;  // p.Ap in more parts than every block can add up
  size_t parts_capacity = 0;
  unsigned lds_raised = 0;  // one-launch kernels (a bit per rows of a thread) that may take kSmallLdsBytes on this device
};
constexpr int kKeptScratch = 8;
std::mutex g_cg_mutex;
std::vector<CgScratch *> g_cg_scratch;

constexpr size_t kSlotWords = 2 * (size_t)kSmallMaxBlocks * 4;

void free_scratch(CgScratch *s) {
  if (s->device_block) (void)hipFree(s->device_block);
  if (s->parts) (void)hipFree(s->parts);
  if (s->host_block) (void)hipHostFree(s->host_block);
  delete s;
}

hipError_t take_scratch(CgScratch **out, hipStream_t st) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  {
    std::lock_guard<std::mutex> lock(g_cg_mutex);
    for (size_t i = 0; i < g_cg_scratch.size(); ++i) {
      if (g_cg_scratch[i]->device != dev) continue;
      *out = g_cg_scratch[i];
      g_cg_scratch.erase(g_cg_scratch.begin() + (ptrdiff_t)i);
      return hipSuccess;
    }
  }
  CgScratch *s = new CgScratch();
  s->device = dev;
  const size_t partial_bytes = sizeof(double) * 3 * kDotMaxBlocks;
  e = hipMalloc(&s->device_block, 256 + partial_bytes + 8 * kSlotWords);
  if (e == hipSuccess) e = hipHostMalloc(&s->host_block, 4096, hipHostMallocDefault);
  if (e == hipSuccess) {
    char *base = static_cast<char *>(s->device_block);
    s->state = reinterpret_cast<CgState *>(base);
    s->partials = reinterpret_cast<double *>(base + 256);
    s->slots = reinterpret_cast<unsigned long long *>(base + 256 + partial_bytes);
    s->progress = static_cast<CgProgress *>(s->host_block);
    s->host_result = reinterpret_cast<CgSmallResult *>(static_cast<char *>(s->host_block) + 512);
    // no slot carries the number of an exchange before that exchange writes it
    if (lapis_hip_fill_f64((int64_t)kSlotWords, 0.0, reinterpret_cast<double *>(s->slots), st) != LAPIS_HIP_OK)
      e = hipErrorUnknown;
  }
  if (e != hipSuccess) {
    free_scratch(s);
    return e;
  }
  *out = s;
  return hipSuccess;
}

constexpr size_t kKeptParts = (size_t)1 << 19;

hipError_t parts_of(CgScratch *s, size_t count, double **out) {
  if (s->parts_capacity < count) {
    if (s->parts) (void)hipFree(s->parts);
    s->parts = nullptr;
    s->parts_capacity = 0;
    const hipError_t e = hipMalloc(&s->parts, sizeof(double) * count);
    if (e != hipSuccess) return e;
    s->parts_capacity = count;
  }
  *out = s->parts;
  return hipSuccess;
}

void give_scratch(CgScratch *s) {
  if (s->parts_capacity > kKeptParts) {
    (void)hipFree(s->parts);
    s->parts = nullptr;
    s->parts_capacity = 0;
  }
  {
    std::lock_guard<std::mutex> lock(g_cg_mutex);
    if ((int)g_cg_scratch.size() < kKeptScratch) {
      g_cg_scratch.push_back(s);
      return;
    }
  }
  free_scratch(s);
}
}  // namespace

namespace lapis {
void cg_release_scratch() {
  std::lock_guard<std::mutex> lock(g_cg_mutex);
  for (CgScratch *s : g_cg_scratch) free_scratch(s);
  g_cg_scratch.clear();
}
}  // namespace lapis

namespace {
static_assert(sizeof(CgState) <= 256, "the state sits in the first 256 bytes of the scratch");

// Rows per workgroup of the one-launch solve, 0 when the system is not for it: it has to fit the chip with a
// workgroup per compute unit, every workgroup's entries its LDS, and rows are walked by one thread each.
int small_rows(const lapis_hip_csr_plan *plan, int64_t n, int *entries) {
  const lapis_hip_csr_stats &s = plan->stats;
  if (n < 1 || s.nnz < 1 || s.max_row_len > 64) return 0;
  const int cus = std::min(device_cu_count(), kSmallMaxBlocks);
  // fewer workgroups make a cheaper exchange: 256^2 rows of 5 take 327 us (41 iterations) with 512 rows each, 425 with 256
  const int64_t rows = std::max<int64_t>(kSmallThreads, ceil_div(n, cus));
  if (rows > (int64_t)kSmallThreads * kSmallMaxRowsPerThread) return 0;
  if (rows * s.max_row_len * 12 > kSmallLdsBytes) return 0;
  *entries = (int)((rows * s.max_row_len + 1) & ~(int64_t)1);
  return (int)rows;
}

template <int RPT>
hipError_t launch_small_rpt(const CgSmallArgs &a, CgScratch *scratch, size_t lds, hipStream_t st) {
  const void *kernel = reinterpret_cast<const void *>(a.dinv ? cg_small_kernel<RPT, true> : cg_small_kernel<RPT, false>);
  const unsigned bit = 1u << (2 * RPT + (a.dinv ? 1 : 0));
  if (!(scratch->lds_raised & bit)) {  // a setting of the device's, as the scratch is
    const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kSmallLdsBytes);
    if (e != hipSuccess) return e;
    scratch->lds_raised |= bit;
  }
  // A cooperative launch: the workgroups of one solve are resident together whatever other streams run (8 us more
  // per solve than a plain launch).
  CgSmallArgs copy = a;
  void *params[] = {&copy};
  return hipLaunchCooperativeKernel(kernel, dim3(a.blocks), dim3(kSmallThreads), params, (unsigned)lds, st);
}

hipError_t launch_small(const CgSmallArgs &a, CgScratch *scratch, hipStream_t st) {
  const char *off = getenv("LAPIS_HIP_CG_ONE_LAUNCH");  // "0": as on a device that refuses the launch
  if (off && off[0] == '0') return hipErrorNotSupported;
  const size_t lds = (size_t)a.entries * 12;
  switch ((int)ceil_div(a.rows, kSmallThreads)) {
    case 1: return launch_small_rpt<1>(a, scratch, lds, st);
    case 2: return launch_small_rpt<2>(a, scratch, lds, st);
    case 3: return launch_small_rpt<3>(a, scratch, lds, st);
    default: return launch_small_rpt<4>(a, scratch, lds, st);
  }
}

// What the solver applies as A and as the preconditioner.
//   mask == nullptr: A p is the SpMV, z = r * prec (prec may be null: z = r)      examples/pcg_solve.py:52-101
//   mask != nullptr: A p is plpt, y = mask*(d*(mask*p) - A (mask*p)), z = r / d   examples/hitting_times.py:97-149
// work holds 4 vectors (5 with a mask), `stride` apart.
int pcg_run(lapis_hip_csr_plan *plan, int64_t n, const int32_t *pos, const int32_t *crd, const double *val,
            const double *b, const double *dinv, const double *mask, double tol, uint64_t maxiter, double *x,
            uint64_t *iters, double *relres, double *work, lapis_hip_stream_t stream) {
  LAPIS_CHECK_INIT();
  LAPIS_REQUIRE(n >= 0, "pcg: negative size");
  LAPIS_REQUIRE(iters && relres, "pcg: null iters/relres output");
  hipStream_t st = as_stream(stream);
  if (n == 0) {
    // r0.r0 = 0: relres is 0/0 = NaN, `relres > tol` is false, the loop leaves at i = 1
    *iters = 1;
    *relres = std::nan("");
    return LAPIS_HIP_OK;
  }
  LAPIS_REQUIRE(pos && b && x, "pcg: null positions, right-hand side or solution");
  const char *what = mask ? "pcg_masked" : "pcg";

  int rc = LAPIS_HIP_OK;
  lapis_hip_csr_plan *own_plan = nullptr;
  double *own_work = nullptr;
  int64_t stride = n;  // distance between the four work vectors
  CgScratch *scratch = nullptr;
  double *chunk_pap = nullptr;  // p.Ap per chunk or per workgroup of the SpMV, where every block cannot add up that many
  bool finished = false;

  // one-exit cleanup
  auto cleanup = [&]() {
    if (own_plan) lapis_hip_csr_plan_destroy(own_plan);
    if (own_work) (void)hipFree(own_work);
    if (scratch) {
      if (!finished) (void)hipStreamSynchronize(st);  // an error left work queued on the scratch
      give_scratch(scratch);
    }
  };
#define PCG_TRY(expr)                                                                          \
  do {                                                                                         \
    hipError_t e_ = (expr);                                                                    \
    if (e_ != hipSuccess) {                                                                    \
      cleanup();                                                                               \
      return set_error(LAPIS_HIP_ERR_RUNTIME, "pcg: %s failed: %s", #expr, hipGetErrorString(e_)); \
    }                                                                                          \
  } while (0)
#define PCG_RC(expr)      \
  do {                    \
    rc = (expr);          \
    if (rc != LAPIS_HIP_OK) { \
      cleanup();          \
      return rc;          \
    }                     \
  } while (0)

  if (!plan) {
    int32_t nnz32 = 0;
    PCG_TRY(hipMemcpyAsync(&nnz32, pos + n, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    PCG_TRY(hipStreamSynchronize(st));
    PCG_RC(lapis_hip_csr_plan_create(&own_plan, n, n, nnz32, pos, crd, 8, stream));
    plan = own_plan;
    PCG_RC(check_planned(what, plan, n, n, pos, crd, val, 8));
    // the column-blocked copy costs about as much as 40 SpMVs of such a matrix: build it
    // only when the iteration limit allows it to pay back
    if (maxiter >= 64) PCG_RC(lapis_hip_csr_plan_analyze(own_plan, crd, val, 8, stream));
  } else {
    // the kernels below size their LDS and their grids by the plan: refused before the first of them
    PCG_RC(check_planned(what, plan, n, n, pos, crd, val, 8));
  }
  if (!work) {
    // own scratch: an even stride keeps all four vectors 16-byte aligned
    stride = (n + 1) & ~(int64_t)1;
    PCG_TRY(hipMalloc(&own_work, sizeof(double) * (mask ? 5 : 4) * (size_t)stride));
    work = own_work;
  }
  double *r = work, *p_odd = work + 2 * stride, *p_even = work + stride, *Ap = work + 3 * stride;  // p of odd, even iterations
  double *tmp = mask ? work + 4 * stride : nullptr;
  PCG_TRY(take_scratch(&scratch, st));
  if (!mask && maxiter != 0 && x != b) {  // x != b: what gives up after x is written starts again from b
    int entries = 0;
    const int rows = small_rows(plan, n, &entries);
    if (rows) {
      CgSmallArgs a{};
      a.n = (int)n;
      a.rows = rows;
      a.blocks = (int)ceil_div(n, rows);
      a.entries = entries;
      a.pos = pos;
      a.crd = crd;
      a.val = val;
      a.b = b;
      a.dinv = dinv;
      a.x = x;
      a.r = r;
      a.z = work + stride;
      a.p0 = work + 2 * stride;
      a.p1 = work + 3 * stride;
      a.slots = scratch->slots;
      a.maxiter = maxiter;
      a.budget = 4096;
      a.tol = tol;
      const char *spins = getenv("LAPIS_HIP_CG_SPINS");  // tests of what happens when a wait runs out
      a.spins = spins ? atoi(spins) : 1 << 18;
      a.out = scratch->host_result;
      for (;;) {
        if (scratch->epoch > 0xf0000000u) {  // start over before the numbers wrap
          PCG_RC(lapis_hip_fill_f64((int64_t)kSlotWords, 0.0, reinterpret_cast<double *>(scratch->slots), stream));
          scratch->epoch = 1;
        }
        a.epoch = scratch->epoch;
        scratch->epoch += 2 * (unsigned)a.budget + 2;
        scratch->host_result->fault = 0;
        // A launch that is refused (a device or a process that takes no cooperative launches, workgroups that do not
        // fit) and workgroups that were not resident together: the kernels below start from the beginning.
        if (launch_small(a, scratch, st) != hipSuccess) {
          (void)hipGetLastError();
          break;
        }
        PCG_TRY(hipStreamSynchronize(st));
        const CgSmallResult &got = *scratch->host_result;
        if (got.fault) break;
        if (got.done_iter != 0) {
          *iters = got.done_iter;
          *relres = got.relres;
          finished = true;
          cleanup();
          return LAPIS_HIP_OK;
        }
        a.resume = 1;
        a.iter0 += a.budget;
        a.rz = got.rz;
        a.beta = got.beta;
        a.initres = got.initres;
      }
    }
  }
  CgState *state = scratch->state;
  double *partials = scratch->partials;
  const bool row_chunks = !mask && plan->runs_rowchunk();
  const int xy_blocks = row_chunks ? rowchunk_xy_blocks(plan) : 0;
  if (xy_blocks > kDotMaxBlocks) PCG_TRY(parts_of(scratch, (size_t)xy_blocks, &chunk_pap));
  if (!mask && !row_chunks && plan->stats.kernel == LAPIS_HIP_SPMV_NNZSPLIT && plan->nchunks > 1)
    PCG_TRY(parts_of(scratch, (size_t)plan->nchunks, &chunk_pap));

  const int grid = dot_grid(n);
  const int prec = !dinv ? kNoPrec : mask ? kDivide : kMultiply;
  const int vec = (aligned16(x) && aligned16(r) && aligned16(p_odd) && aligned16(p_even) && aligned16(Ap) && (!dinv || aligned16(dinv))) ? 1 : 0;
  volatile CgProgress *progress = scratch->progress;
  progress->iter = 0;
  progress->relres = 0.0;
  hipLaunchKernelGGL(cg_init_kernel, dim3(grid), dim3(256), 0, st, (long long)n, b, dinv, x, r, p_odd, partials,
                     mask ? 1 : 0);
  hipLaunchKernelGGL(cg_init_scalar_kernel, dim3(1), dim3(256), 0, st, grid, partials, state,
                     (unsigned long long)maxiter, tol);
  PCG_TRY(hipGetLastError());
  double *pap_partials = partials, *rr_partials = partials + kDotMaxBlocks, *rz_partials = partials + 2 * kDotMaxBlocks;
  // The host stays a few iterations ahead of the device, which tells it how far it is: enough that the device never
  // waits for a launch (about 100 us of work), few enough that little is left queued when it leaves -- such passes
  // find the exit mark and return at once, the product of long-row kernels excepted.
  const double iteration_us = ((double)plan->stats.nnz * 12.0 + (double)n * 100.0) / 5e6;
  const uint64_t ahead = (uint64_t)std::min(32.0, 2.0 + 100.0 / (iteration_us + 4.0));
  uint64_t launched = 0;
  while (!finished) {
    if (maxiter == 0 || launched < maxiter) {
      const unsigned long long iter = ++launched;  // the reference's counter for this pass
      double *p = iter & 1 ? p_odd : p_even, *other = iter & 1 ? p_even : p_odd;
      int pap_count = grid;
      int deferred = 0;  // chunk length when the SpMV left its cut rows to the p.Ap kernel
      if (row_chunks) {
        // Ap = A p and p.Ap in one pass
        PCG_RC(launch_rowchunk_xy<double>(plan, crd, val, p, Ap, st, chunk_pap ? chunk_pap : pap_partials, false, &pap_count,
                                          &state->done_iter));
        if (chunk_pap) {
          hipLaunchKernelGGL(cg_reduce_partials_kernel, dim3(kReducedPartials), dim3(256), 0, st, pap_count, chunk_pap,
                             pap_partials);
          pap_count = kReducedPartials;
        }
      } else if (mask) {
        // plpt: tmp = mask*p ; Ap = A tmp ; Ap = (d*tmp - Ap)*mask
        PCG_RC(lapis_hip_mult_f64(n, p, mask, tmp, stream));
        PCG_RC(spmv_overwrite_f64(plan, n, n, pos, crd, val, tmp, Ap, stream));
        hipLaunchKernelGGL(masked_combine_kernel, dim3(grid), dim3(256), 0, st, (long long)n, 0, dinv, tmp, mask, Ap);
      } else {
        // Ap = A p: the reference zero-fills Ap and accumulates (examples/pcg_solve.py:12-19)
        PCG_RC(spmv_overwrite_f64(plan, n, n, pos, crd, val, p, Ap, stream, chunk_pap ? &deferred : nullptr,
                                  chunk_pap));
      }
      if (deferred) {
        // one thread per chunk, at most kDotMaxBlocks blocks
        const int nchunks = plan->nchunks;
        const int per_block = (int)std::max<int64_t>(256, ceil_div(ceil_div(nchunks, kDotMaxBlocks), 256) * 256);
        pap_count = (int)ceil_div(nchunks, per_block);
#define PCG_PAP_FIX(CH)                                                                                         \
  hipLaunchKernelGGL(cg_pap_fix_kernel<CH>, dim3(pap_count), dim3(256), 0, st, nchunks, per_block, p, Ap,        \
                     (const double *)chunk_pap, pap_partials, pos, (const int *)plan->chunk_row,                \
                     (const double *)plan->part_first, (const double *)plan->part_last)
        switch (deferred) {
          case 512: PCG_PAP_FIX(512); break;
          case 1024: PCG_PAP_FIX(1024); break;
          case 2048: PCG_PAP_FIX(2048); break;
          default:
            cleanup();
            return set_error(LAPIS_HIP_ERR_RUNTIME, "pcg: no p.Ap kernel for chunks of %d non-zeros", deferred);
        }
#undef PCG_PAP_FIX
      } else if (!row_chunks) {
        hipLaunchKernelGGL(cg_pap_kernel, dim3(grid), dim3(256), 0, st, (long long)n, p, Ap, pap_partials, vec);
      }
#define PCG_UPDATES(PREC)                                                                                           \
  hipLaunchKernelGGL(cg_update_r_kernel<PREC>, dim3(grid), dim3(256), 0, st, (long long)n, Ap, r, dinv, state, iter, \
                     pap_count, pap_partials, rr_partials, rz_partials, vec);                                       \
  hipLaunchKernelGGL((iter & 1 ? cg_update_xp_kernel<PREC, false> : cg_update_xp_kernel<PREC, true>), dim3(grid),    \
                     dim3(256), 0, st, (long long)n, r, dinv, p, other, x, state, scratch->progress, iter, grid,     \
                     rr_partials, rz_partials, vec)
      if (prec == kNoPrec) {
        PCG_UPDATES(kNoPrec);
      } else if (prec == kMultiply) {
        PCG_UPDATES(kMultiply);
      } else {
        PCG_UPDATES(kDivide);
      }
#undef PCG_UPDATES
      PCG_TRY(hipGetLastError());
    }
    // wait until no more than `ahead` iterations are queued, or, past the last one, until all are done
    const bool last = maxiter != 0 && launched == maxiter;
    const uint64_t want = last ? launched : launched > ahead ? launched - ahead : 0;
    bool drained = false;
    for (unsigned spin = 1;; ++spin) {
      const unsigned long long at = progress->iter;
      finished = (at & kLeft) != 0;
      if (finished || at >= want || drained) break;
      __builtin_ia32_pause();
      if (spin % 65536 == 0) {  // a stream that failed, or ended without a word, ends the wait
        const hipError_t e = hipStreamQuery(st);
        if (e == hipErrorNotReady)
          (void)hipGetLastError();
        else
          PCG_TRY(e);
        drained = e == hipSuccess;
      }
    }
    if (finished || last || drained) {
      PCG_TRY(hipStreamSynchronize(st));
      const unsigned long long at = progress->iter;
      if (!(at & kLeft)) {
        // iteration `maxiter` always raises the flag, so this is unreachable unless the state was corrupted
        finished = true;
        cleanup();
        return set_error(LAPIS_HIP_ERR_RUNTIME, "pcg: %llu iterations queued and the device never reported an exit",
                         (unsigned long long)launched);
      }
      finished = true;
      *iters = at & ~kLeft;
      *relres = progress->relres;
    }
  }
  cleanup();
#undef PCG_TRY
#undef PCG_RC
  return LAPIS_HIP_OK;
}

}  // namespace

extern "C" int lapis_hip_pcg_f64_i32(lapis_hip_csr_plan *plan, int64_t n, const int32_t *pos, const int32_t *crd,
                                     const double *val, const double *b, const double *dinv, double tol,
                                     uint64_t maxiter, double *x, uint64_t *iters, double *relres, double *work,
                                     lapis_hip_stream_t stream) {
  return pcg_run(plan, n, pos, crd, val, b, dinv, nullptr, tol, maxiter, x, iters, relres, work, stream);
}

extern "C" int lapis_hip_pcg_masked_f64_i32(lapis_hip_csr_plan *plan, int64_t n, const int32_t *pos,
                                            const int32_t *crd, const double *val, const double *b,
                                            const double *mask, const double *d, double tol, uint64_t maxiter,
                                            double *x, uint64_t *iters, double *relres, double *work,
                                            lapis_hip_stream_t stream) {
  LAPIS_REQUIRE(n == 0 || (mask && d), "pcg_masked: null mask or diagonal");
  return pcg_run(plan, n, pos, crd, val, b, d, mask, tol, maxiter, x, iters, relres, work, stream);
}

extern "C" int lapis_hip_mht_f64_i32(lapis_hip_csr_plan *plan, int64_t n, int64_t nnz, const int32_t *pos,
                                     const int32_t *crd, double *val, const double *mask, const double *d,
                                     double alpha, double tol, uint64_t maxiter, double *mom1, double *mom2,
                                     lapis_hip_stream_t stream) {
  LAPIS_CHECK_INIT();
  LAPIS_REQUIRE(n >= 0 && nnz >= 0, "mht: negative size");
  if (n == 0) return LAPIS_HIP_OK;
  LAPIS_REQUIRE(pos && mask && d && mom1 && mom2 && (nnz == 0 || (crd && val)), "mht: null argument");
  hipStream_t st = as_stream(stream);
  double *bbuf = nullptr;
  LAPIS_HIP_TRY(hipMalloc(&bbuf, sizeof(double) * (size_t)n));
  uint64_t its = 0;
  double res = 0.0;
  int rc = lapis_hip_scale_f64(nnz, alpha, val, stream);  // scale_csr, in place
  // a column-blocked copy inside the caller's plan still holds the unscaled values
  if (rc == LAPIS_HIP_OK && plan) rc = lapis_hip_csr_plan_update_values(plan, val, 8, stream);
  if (rc == LAPIS_HIP_OK) rc = lapis_hip_mult_f64(n, d, mask, bbuf, stream);
  if (rc == LAPIS_HIP_OK)
    rc = lapis_hip_pcg_masked_f64_i32(plan, n, pos, crd, val, bbuf, mask, d, tol, maxiter, mom1, &its, &res, nullptr,
                                      stream);
  if (rc == LAPIS_HIP_OK) rc = spmv_overwrite_f64(plan, n, n, pos, crd, val, mom1, bbuf, stream);
  if (rc == LAPIS_HIP_OK) {
    hipLaunchKernelGGL(masked_combine_kernel, dim3(dot_grid(n)), dim3(256), 0, st, (long long)n, 1, d,
                       (const double *)mom1, mask, bbuf);
    if (hipGetLastError() != hipSuccess) rc = set_error(LAPIS_HIP_ERR_RUNTIME, "mht: kernel launch failed");
  }
  if (rc == LAPIS_HIP_OK)
    rc = lapis_hip_pcg_masked_f64_i32(plan, n, pos, crd, val, bbuf, mask, d, tol, maxiter, mom2, &its, &res, nullptr,
                                      stream);
  (void)hipStreamSynchronize(st);
  (void)hipFree(bbuf);
  return rc;
}

extern "C" int lapis_hip_normalize_mom2_f64(int64_t n, const double *mom1, const double *mom2, double *out,
                                            lapis_hip_stream_t stream) {
  LAPIS_CHECK_INIT();
  LAPIS_REQUIRE(n >= 0, "normalize_mom2: negative size");
  if (n == 0) return LAPIS_HIP_OK;
  LAPIS_REQUIRE(mom1 && mom2 && out, "normalize_mom2: null argument");
  hipLaunchKernelGGL(normalize_mom2_kernel, dim3(dot_grid(n)), dim3(256), 0, as_stream(stream), (long long)n, mom1,
                     mom2, out);
  LAPIS_LAUNCH_CHECK();
  return LAPIS_HIP_OK;
}
