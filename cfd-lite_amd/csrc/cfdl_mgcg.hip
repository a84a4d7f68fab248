// cfdl_mgcg.hip -- multigrid-preconditioned conjugate gradients for the
// pressure-correction system on MI355X (an extension: the reference solves
// that system with the 4-subdomain Gauss-Seidel solver of
// src/modules/mod_solver.f90:124-189; its stop rule, rms residual at most a
// tenth of the initial one or nit iterations, :271-322, is kept).
//
// Design:
//  * Conjugate gradients in FP64 on the mesh CSR as it stands (ap, anb, b of
//    calc_coef_p, no copies), vectors in the global cell order.  Every dot
//    product and norm is a blocked reduction of fixed shape: block x of 256
//    lanes owns a contiguous chunk, lane t sums its strided elements in
//    order (1024 threads compute them), the lanes combine as
//    s[t] += s[t+h] for h = 128, 64 (LDS) and 32 .. 1 (wavefront shuffles),
//    and the last block to finish (a ticket counter) combines the block sums
//    in the same way and does the scalar work (alpha, beta, the stop test)
//    in the same launch.  So each CG iteration is four launches besides the
//    preconditioner, and the result does not depend on scheduling.
//  * The preconditioner is one V-cycle of agglomeration multigrid (the
//    hierarchy of cfdl_mg.cpp): Galerkin coarse operators summed once per
//    solve from lists (no atomics), one forward colour Gauss-Seidel sweep
//    before and one backward after each coarse correction, so the operator
//    is symmetric.  Every level is stored in its colours' order (struct Lev;
//    level 0 is a copy of the system, in FP32 for the mixed variant), so a
//    colour reads its rows and nothing between them; the forward sweep starts
//    from zero without reading zeros and leaves the last colours' residuals;
//    the prolongation skips the colour the backward sweep computes first.
//    Levels of more than kCoarseMax nodes run as grid-wide launches (one per
//    colour, the small trailing colours in one); the small levels below run
//    inside one workgroup of 1024 threads, with their values in LDS and each
//    colour's rows loaded while the one before computes.  In the mixed variant
//    the V-cycle runs in FP32; CG, its residual and the stop test stay FP64.
//    A V-cycle at 128^3 in FP32 took 329 us with the levels in mesh order and
//    176 us so; at 80 x 100 x 72 in FP64 (up to nine colours a level) 636 us
//    and 321 us.
//  * All kernels read the solve's active flag and return at once when it is
//    clear, so the host can queue an iteration before knowing whether the
//    previous one stopped the solve.
//  * Grouped solves (mgcg_solve_group) run the same steps for up to
//    kMaxGroup independent systems, one launch per step for all of them:
//    the launch's blocks are split into per-system ranges, each system keeps
//    its own vectors, reductions and stop test, so its results are those of
//    a solve alone, bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <type_traits>
#include <vector>

#include "cfdl_group.h"
#include "cfdl_internal.h"

namespace cfdl {

namespace {

#define MGCHK(x)                                                                    \
  do {                                                                              \
    hipError_t e_ = (x);                                                            \
    if (e_ != hipSuccess) {                                                         \
      set_error(std::string(#x) + ": " + hipGetErrorString(e_));                    \
      return CFDL_EHIP;                                                             \
    }                                                                               \
  } while (0)

constexpr int kRed = 256;          // lanes of a blocked sum
// Threads of a reduction block.  The blocked sums fix 256 lanes a block and
// 4,096 elements a block, which is 2 wavefronts a SIMD on a 128^3 mesh: too
// few loads in flight.  Four lane groups compute the elements of a block, its
// 256 lanes add them in order (blocked_acc).  With the partials passed without
// fences (put_part), at 128^3: A p with p.q 78 -> 35 us, the update 57 -> 22
// us, r.z 36 -> 9 us.
constexpr int kRedThreads = 1024;
constexpr int kRedSeg = 16 * kRed;  // elements staged in LDS at a time
constexpr int kMaxRedBlocks = 1024;
constexpr int kBlk = 256;          // lanes per block of the grid-wide V-cycle kernels
constexpr int kCoarseMax = 4096;   // levels at most this large run in one workgroup
constexpr int kCoarseThreads = 1024;
constexpr int kCoarseSweeps = 10;  // forward + backward sweep pairs on the coarsest level

// control block of one solve
struct CgCtl {
  int it, active, ticket, nit;
  double res_i, res_f, res_max, target, rho, rho_old, alpha, beta;
};

// blocked reduction shape of an n-element vector
struct Red {
  int n, nblk, chunk;
};
Red red_of(int n) {
  int nb = (n + 4095) / 4096;
  nb = nb < 1 ? 1 : (nb > kMaxRedBlocks ? kMaxRedBlocks : nb);
  return Red{n, nb, (n + nb - 1) / nb};
}

// s[t] += s[t+h], h = 128, 64 in LDS, then 32 .. 1 by shuffles in wave 0;
// v from threads 0 .. 255, the block's sum in thread 0 (the pairing of an LDS
// tree)
__device__ inline double tree_sum(double v, double *s) {
  const int t = threadIdx.x;
  if (t < kRed) s[t] = v;
  __syncthreads();
  if (t < 128) s[t] = s[t] + s[t + 128];
  __syncthreads();
  double x = 0.0;
  if (t < 64) {
    x = s[t] + s[t + 64];
#pragma unroll
    for (int h = 32; h >= 1; h >>= 1) x = x + __shfl_down(x, h, 64);
  }
  __syncthreads();
  return x;
}
// the maximum over all kRedThreads threads (the same in any order), in thread 0
__device__ inline double block_max(double v, double *s) {
  const int t = threadIdx.x;
#pragma unroll
  for (int h = 32; h >= 1; h >>= 1) v = fmax(v, __shfl_down(v, h, 64));
  if (t % 64 == 0) s[t / 64] = v;
  __syncthreads();
  if (t == 0)
    for (int w = 1; w < kRedThreads / 64; w++) v = fmax(v, s[w]);
  __syncthreads();
  return v;
}

// Lane t's sum (threads 0 .. 255) of f(i) over i = lo + t, lo + t + 256, ... <
// hi, in that order from 0: all threads of the block evaluate f, once per i,
// into LDS (s: kRedSeg doubles), a segment at a time, and the lanes add.
template <typename F>
__device__ inline double blocked_acc(int lo, int hi, double *s, F f) {
  const int t = threadIdx.x;
  double acc = 0.0;
  for (int base = lo; base < hi; base += kRedSeg) {
    const int n = min(kRedSeg, hi - base);
#pragma unroll
    for (int j = 0; j < kRedSeg / kRedThreads; j++) {
      const int o = t + j * kRedThreads;
      if (o < n) s[o] = f(base + o);
    }
    __syncthreads();
    if (t < kRed)
      for (int o = t; o < n; o += kRed) acc = acc + s[o];
    __syncthreads();
  }
  return acc;
}

// Block partials pass through memory at agent scope (stores and loads that
// bypass the XCD's L2), so no block needs a fence: a fence writes back and
// invalidates an L2, per wavefront that executes it, which took longer than
// the sums (with 16 wavefronts a block each of the three kernels took 100 to
// 130 us more at 128^3).
__device__ inline void put_part(double *part, double v) {
  __hip_atomic_store(part, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline double get_part(const double *part) {
  return __hip_atomic_load(part, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Returns true in every thread of the last block to arrive, which then sees
// the partials of all blocks.  Thread 0 wrote this block's; it waits until
// they are in memory before it takes the ticket.
__device__ inline bool arrive_last(CgCtl *c, int nblk) {
  __shared__ int last;
  if (threadIdx.x == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    last = __hip_atomic_fetch_add(&c->ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           nblk - 1;
  }
  __syncthreads();
  return last;
}
// the last block's sum of the nblk partials part[k * stride]
__device__ inline double final_sum(const double *part, int nblk, int stride, double *s) {
  double acc = 0.0;
  if (threadIdx.x < kRed)
    for (int i = threadIdx.x; i < nblk; i += kRed) acc = acc + get_part(part + i * stride);
  return tree_sum(acc, s);
}
__device__ inline double final_max(const double *part, int nblk, int stride, double *s) {
  double acc = 0.0;
  for (int i = threadIdx.x; i < nblk; i += kRedThreads) acc = fmax(acc, get_part(part + i * stride));
  return block_max(acc, s);
}

// ---------------------------------------------------------------------------
// CG kernels.  Each step is a device body run by block bx of the system's own
// grid (bx = blockIdx.x for a solve alone; the block's index inside the
// system's range in a grouped launch) and two thin kernels around it.
// ---------------------------------------------------------------------------

// acc + sum over row i of anb * x[nbr], in CSR order; a six-entry
// (hexahedral) row issues all its loads before the sum
__device__ inline double csr_sum(const int *__restrict__ row, const int *__restrict__ nbr,
                                 const double *__restrict__ anb, const double *__restrict__ x,
                                 int i, double acc) {
  const int r0 = row[i], r1 = row[i + 1];
  if (r1 - r0 == 6) {
    int c[6];
    double a[6], v[6];
#pragma unroll
    for (int k = 0; k < 6; k++) {
      c[k] = nbr[r0 + k];
      a[k] = anb[r0 + k];
    }
#pragma unroll
    for (int k = 0; k < 6; k++) v[k] = x[c[k]];
#pragma unroll
    for (int k = 0; k < 6; k++) acc = acc + a[k] * v[k];
    return acc;
  }
  for (int k = r0; k < r1; k++) acc = acc + anb[k] * x[nbr[k]];
  return acc;
}

// r = b + sum anb phi_nb - ap phi, also as rt in the V-cycle's numbering
// (pos) and type; res_i, target and the active flag from rms(r)
template <typename T>
__device__ inline void d_cg_init(int bx, Red R, const int *__restrict__ row,
                                 const int *__restrict__ nbr, const int *__restrict__ pos,
                                 const double *__restrict__ ap, const double *__restrict__ anb,
                                 const double *__restrict__ b, const double *__restrict__ phi,
                                 double *__restrict__ r, T *__restrict__ rt, CgCtl *c,
                                 double *part, int nit) {
  __shared__ double s[kRedSeg];
  const int lo = bx * R.chunk, hi = min(lo + R.chunk, R.n);
  const double acc = blocked_acc(lo, hi, s, [&](int i) {
    double v = csr_sum(row, nbr, anb, phi, i, b[i]);
    v = v - ap[i] * phi[i];
    r[i] = v;
    rt[pos[i]] = static_cast<T>(v);
    return v * v;
  });
  const double bs = tree_sum(acc, s);
  if (threadIdx.x == 0) put_part(part + bx, bs);
  if (!arrive_last(c, R.nblk)) return;
  const double rr = final_sum(part, R.nblk, 1, s);
  if (threadIdx.x == 0) {
    const double ri = sqrt(rr / static_cast<double>(R.n));
    c->res_i = ri;
    c->res_f = ri;
    c->target = ri / 10.0;
    c->res_max = 0.0;
    c->it = 0;
    c->nit = nit;
    c->rho_old = 0.0;
    c->active = (0 < nit && ri > c->target) ? 1 : 0;
    c->ticket = 0;
  }
}

// rho = r.z, beta = rho / rho_old (0 on the first iteration)
template <typename T>
__device__ inline void d_cg_rz(int bx, Red R, const double *__restrict__ r,
                               const T *__restrict__ z, const int *__restrict__ pos, CgCtl *c,
                               double *part) {
  __shared__ double s[kRedSeg];
  if (!c->active) return;
  const int lo = bx * R.chunk, hi = min(lo + R.chunk, R.n);
  const double acc =
      blocked_acc(lo, hi, s, [&](int i) { return r[i] * static_cast<double>(z[pos[i]]); });
  const double bs = tree_sum(acc, s);
  if (threadIdx.x == 0) put_part(part + bx, bs);
  if (!arrive_last(c, R.nblk)) return;
  const double rho = final_sum(part, R.nblk, 1, s);
  if (threadIdx.x == 0) {
    c->rho = rho;
    c->beta = c->it == 0 ? 0.0 : rho / c->rho_old;
    c->ticket = 0;
  }
}

// p = z, or z + beta p (element i)
template <typename T>
__device__ inline void d_cg_p(int i, int n, const T *__restrict__ z, const int *__restrict__ pos,
                              double *__restrict__ p, const CgCtl *c) {
  if (i >= n || !c->active) return;
  const double zi = static_cast<double>(z[pos[i]]);
  if (c->it == 0)
    p[i] = zi;
  else
    p[i] = zi + c->beta * p[i];
}

// q = ap p - sum anb p_nb, sigma = p.q, alpha = rho / sigma (a breakdown,
// sigma or rho not positive, ends the solve)
__device__ inline void d_cg_spmv(int bx, Red R, const int *__restrict__ row,
                                 const int *__restrict__ nbr, const double *__restrict__ ap,
                                 const double *__restrict__ anb, const double *__restrict__ p,
                                 double *__restrict__ q, CgCtl *c, double *part) {
  __shared__ double s[kRedSeg];
  if (!c->active) return;
  const int lo = bx * R.chunk, hi = min(lo + R.chunk, R.n);
  const double acc = blocked_acc(lo, hi, s, [&](int i) {
    const double sm = csr_sum(row, nbr, anb, p, i, 0.0);
    const double pi = p[i], qi = ap[i] * pi - sm;
    q[i] = qi;
    return pi * qi;
  });
  const double bs = tree_sum(acc, s);
  if (threadIdx.x == 0) put_part(part + bx, bs);
  if (!arrive_last(c, R.nblk)) return;
  const double sigma = final_sum(part, R.nblk, 1, s);
  if (threadIdx.x == 0) {
    if (!(sigma > 0.0) || !(c->rho > 0.0))
      c->active = 0;
    else
      c->alpha = c->rho / sigma;
    c->ticket = 0;
  }
}

// phi += alpha p, r -= alpha q (also as rt for the next V-cycle); rms and max
// |r|; the iteration count and the stop test
template <typename T>
__device__ inline void d_cg_update(int bx, Red R, double *__restrict__ phi,
                                   const double *__restrict__ p, const double *__restrict__ q,
                                   const int *__restrict__ pos, double *__restrict__ r,
                                   T *__restrict__ rt, CgCtl *c, double *part) {
  __shared__ double s[kRedSeg];
  if (!c->active) return;
  const double alpha = c->alpha;
  const int lo = bx * R.chunk, hi = min(lo + R.chunk, R.n);
  double mx = 0.0;
  const double acc = blocked_acc(lo, hi, s, [&](int i) {
    phi[i] = phi[i] + alpha * p[i];
    const double v = r[i] - alpha * q[i];
    r[i] = v;
    rt[pos[i]] = static_cast<T>(v);
    mx = fmax(mx, fabs(v));
    return v * v;
  });
  const double bs = tree_sum(acc, s), bm = block_max(mx, s);
  if (threadIdx.x == 0) {
    put_part(part + 2 * bx, bs);
    put_part(part + 2 * bx + 1, bm);
  }
  if (!arrive_last(c, R.nblk)) return;
  const double rr = final_sum(part, R.nblk, 2, s);
  const double rm = final_max(part + 1, R.nblk, 2, s);
  if (threadIdx.x == 0) {
    c->it = c->it + 1;
    c->res_f = sqrt(rr / static_cast<double>(R.n));
    c->res_max = rm;
    c->rho_old = c->rho;
    c->active = (c->it < c->nit && c->res_f > c->target) ? 1 : 0;
    c->ticket = 0;
  }
}

__device__ inline void d_cg_log(const CgCtl *c, LogLine *log, int *nlog, const LogLine &tmpl) {
  const int k = *nlog;
  if (k >= kLogCap) return;
  LogLine l = tmpl;
  l.it = c->it;
  l.res_i = c->res_i;
  l.res_f = c->res_f;
  l.res_max = c->res_max;
  log[k] = l;
  *nlog = k + 1;
}

template <typename T>
__global__ void __launch_bounds__(kRedThreads)
k_cg_init(Red R, const int *__restrict__ row, const int *__restrict__ nbr,
          const int *__restrict__ pos, const double *__restrict__ ap,
          const double *__restrict__ anb, const double *__restrict__ b,
          const double *__restrict__ phi, double *__restrict__ r, T *__restrict__ rt, CgCtl *c,
          double *part, int nit) {
  d_cg_init<T>(xcd_block(), R, row, nbr, pos, ap, anb, b, phi, r, rt, c, part, nit);
}
template <typename T>
__global__ void __launch_bounds__(kRedThreads)
k_cg_rz(Red R, const double *__restrict__ r, const T *__restrict__ z, const int *__restrict__ pos,
        CgCtl *c, double *part) {
  d_cg_rz<T>(xcd_block(), R, r, z, pos, c, part);
}
template <typename T>
__global__ void k_cg_p(int n, const T *__restrict__ z, const int *__restrict__ pos,
                       double *__restrict__ p, const CgCtl *c) {
  d_cg_p<T>(xcd_block() * blockDim.x + threadIdx.x, n, z, pos, p, c);
}
__global__ void __launch_bounds__(kRedThreads)
k_cg_spmv(Red R, const int *__restrict__ row, const int *__restrict__ nbr,
          const double *__restrict__ ap, const double *__restrict__ anb,
          const double *__restrict__ p, double *__restrict__ q, CgCtl *c, double *part) {
  d_cg_spmv(xcd_block(), R, row, nbr, ap, anb, p, q, c, part);
}
template <typename T>
__global__ void __launch_bounds__(kRedThreads)
k_cg_update(Red R, double *__restrict__ phi, const double *__restrict__ p,
            const double *__restrict__ q, const int *__restrict__ pos, double *__restrict__ r,
            T *__restrict__ rt, CgCtl *c, double *part) {
  d_cg_update<T>(xcd_block(), R, phi, p, q, pos, r, rt, c, part);
}
__global__ void k_cg_log(const CgCtl *c, LogLine *log, int *nlog, LogLine tmpl) {
  if (threadIdx.x == 0 && blockIdx.x == 0) d_cg_log(c, log, nlog, tmpl);
}

// ---------------------------------------------------------------------------
// V-cycle kernels on one level (T = double or float)
// ---------------------------------------------------------------------------
// One level as the kernels see it (device pointers).  Its nodes are numbered
// by colour: colour c is the positions cbeg[c] .. cbeg[c] + ccnt[c] - 1 (on
// the grid-wide levels a colour starts at a multiple of 64; the positions in
// between belong to no node), so a colour's rows, values and results are
// contiguous.  In the mesh order the rows of two colours alternate and every
// cache line of the matrix was fetched for each of them.  Rows are stored in
// slices of 64 positions, entry-major: entry k of position p is at
// mg_entry(p) + 64 k.  Row sums keep the entries' CSR order, so the numbering
// changes no bit.
template <typename T>
struct Lev {
  int n, npad, nnz, ncol;
  int uni;    // entries of every row, 0 if they differ
  int fin;    // first position of the final nodes, -1 if they are no such range
  int ctail;  // colours from this one on share one workgroup (ncol: none do)
  int kmax;   // longest row
  const int *cbeg, *ccnt;  // per colour
  const int *sptr;         // first entry of each slice (not uni)
  // row length; bit 15: a final node, whose neighbours all have lower colours,
  // so that a forward sweep leaves its row sum final
  const unsigned short *info;
  const int *col;  // position of the neighbour; npad + halo on level 0
  const int *agg, *mptr, *mem, *iptr, *ilist, *gptr, *glist, *gpos;
  T *ap, *anb, *b, *x, *t;  // t: residual after the forward sweep
};
constexpr int kTailNodes = 1024;

template <typename T>
__device__ inline int mg_entry(const Lev<T> &L, int p) {
  return (L.uni ? (p >> 6) * 64 * L.uni : L.sptr[p >> 6]) + (p & 63);
}
template <typename T>
__device__ inline bool mg_final(const Lev<T> &L, int p) {
  return L.fin >= 0 ? p >= L.fin : (L.info[p] >> 15) != 0;
}

// acc + sum over row p of anb * val(neighbour), in entry order.  Loads go out
// in groups of six or eight before their part of the sum; a short row's group
// repeats its last entry and leaves it out of the sum.
template <typename T, typename V>
__device__ inline T row_sum(const Lev<T> &L, int e, int len, T acc, V val) {
  if (L.uni == 6) {
    int c[6];
    T a[6], v[6];
#pragma unroll
    for (int k = 0; k < 6; k++) {
      c[k] = L.col[e + 64 * k];
      a[k] = L.anb[e + 64 * k];
    }
#pragma unroll
    for (int k = 0; k < 6; k++) v[k] = val(c[k]);
#pragma unroll
    for (int k = 0; k < 6; k++) acc = acc + a[k] * v[k];
    return acc;
  }
  for (int k0 = 0; k0 < len; k0 += 8) {
    int c[8];
    T a[8], v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int q = e + 64 * min(k0 + k, len - 1);
      c[k] = L.col[q];
      a[k] = L.anb[q];
    }
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = val(c[k]);
#pragma unroll
    for (int k = 0; k < 8; k++) acc = k0 + k < len ? acc + a[k] * v[k] : acc;
  }
  return acc;
}

// Level 0: the system's coefficients into the level's numbering and type, one
// thread per mesh cell g (its row is read whole; a colour's entries are
// written next to each other).
template <typename T>
__device__ inline void d_mg_copy0(int g, const Lev<T> &L, const int *__restrict__ pos,
                                  const int *__restrict__ row, const double *__restrict__ ap,
                                  const double *__restrict__ anb) {
  if (g >= L.n) return;
  const int p = pos[g], e = mg_entry(L, p), r0 = row[g], r1 = row[g + 1];
  L.ap[p] = static_cast<T>(ap[g]);
  if (r1 - r0 == 6) {  // the loads go out before the stores
    double v[6];
#pragma unroll
    for (int k = 0; k < 6; k++) v[k] = anb[r0 + k];
#pragma unroll
    for (int k = 0; k < 6; k++) L.anb[e + 64 * k] = static_cast<T>(v[k]);
    return;
  }
  for (int k = r0; k < r1; k++) L.anb[e + 64 * (k - r0)] = static_cast<T>(anb[k]);
}

// Galerkin operator of the next level: thread g < C.npad sums the diagonal of
// the aggregate at position g (members' ap in order, minus the inside entries
// in order), thread C.npad + s sums coarse slot s (its list of fine entries in
// order)
template <typename T>
__device__ inline void d_mg_galerkin(int g, const Lev<T> &F, const Lev<T> &C) {
  if (g < C.npad) {
    T acc = static_cast<T>(0);
    for (int q = F.mptr[g]; q < F.mptr[g + 1]; q++) acc = acc + F.ap[F.mem[q]];
    for (int q = F.iptr[g]; q < F.iptr[g + 1]; q++) acc = acc - F.anb[F.ilist[q]];
    C.ap[g] = acc;
  } else if (g < C.npad + C.nnz) {
    const int sl = g - C.npad;
    T acc = static_cast<T>(0);
    for (int q = F.gptr[sl]; q < F.gptr[sl + 1]; q++) acc = acc + F.anb[F.glist[q]];
    C.anb[C.gpos[sl]] = acc;
  }
}

// Gauss-Seidel sweeps by colour, x_i = (b_i + sum anb x_nb) / ap_i.
// kFwd0: the forward sweep from x = 0, which reads no x it has not written:
// later colours and halos count as the zeros they stand for, and colour 0 is
// (b_i + 0) / ap_i without its row (0 anb = 0: the coefficients are finite,
// or cg_init's residual is not and the solve never starts).  Final nodes
// leave their residual in t for the restriction.  kFwd, kBwd: from x as it is.
enum { kFwd0 = 0, kFwd = 1, kBwd = 2 };
// A node's row as it is loaded before its neighbours' values: where it is, its
// scalars, and its first K entries (a short row's last one again; K = 6 for
// levels of six entries a row).  What a launch of one colour takes is a chain
// of loads (the slice's start; the entries; the neighbours' values; the store)
// and not its bytes, so the chain holds nothing else: the colour's range comes
// as arguments, and the solve's flag is on its way with the first loads (mean
// over the levels: 80 x 100 x 72 in FP64 5.83 -> 5.62 us, the 96^3 channel in
// FP32 5.68 -> 5.37 us; 34 and 30 such launches a V-cycle).
template <typename T, int K>
struct MgRow {
  int e, info, c[K];
  T b, ap, a[K];
};
// a value that the compiler must have here, so that its load stays ahead of
// the branch below
__device__ inline void have(int &x) { asm volatile("" : "+v"(x)); }

template <typename T, int K>
__device__ inline void mg_place(const Lev<T> &L, int p, MgRow<T, K> &r) {
  r.e = mg_entry(L, p);
  r.info = K == 6 ? 6 : L.info[p];
  r.b = L.b[p];
  r.ap = L.ap[p];
}
template <typename T, int K>
__device__ inline void mg_entries(const Lev<T> &L, MgRow<T, K> &r) {
  const int last = max((r.info & 0x7fff) - 1, 0);
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int q = r.e + 64 * (K == 6 ? k : min(k, last));
    r.c[k] = L.col[q];
    r.a[k] = L.anb[q];
  }
}
// the node's update; its row's entries beyond the first K come in groups of K
template <typename T, int K>
__device__ inline void mg_node(const Lev<T> &L, int p, int c0, int mode, const MgRow<T, K> &r) {
  const T zero = static_cast<T>(0);
  const int len = K == 6 ? 6 : r.info & 0x7fff;
  auto val = [&](int q) { return mode != kFwd0 || q < c0 ? L.x[q] : zero; };
  T v[K], s = r.b;
#pragma unroll
  for (int k = 0; k < K; k++) v[k] = val(r.c[k]);
#pragma unroll
  for (int k = 0; k < K; k++) s = k < len ? s + r.a[k] * v[k] : s;
  for (int k0 = K; k0 < len; k0 += K) {
    int c[K];
    T a[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int q = r.e + 64 * min(k0 + k, len - 1);
      c[k] = L.col[q];
      a[k] = L.anb[q];
    }
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = val(c[k]);
#pragma unroll
    for (int k = 0; k < K; k++) s = k0 + k < len ? s + a[k] * v[k] : s;
  }
  const T x = s / r.ap;
  L.x[p] = x;
  if (mode == kFwd0 && (K == 6 ? mg_final(L, p) : (r.info >> 15) != 0)) L.t[p] = s - r.ap * x;
}
// the first colour of a forward sweep from zero
template <typename T>
__device__ inline void mg_first(const Lev<T> &L, int p, int info, T b, T ap) {
  const T s = info & 0x7fff ? b + static_cast<T>(0) : b, x = s / ap;
  L.x[p] = x;
  if (L.uni == 6 ? mg_final(L, p) : (info >> 15) != 0) L.t[p] = s - ap * x;
}
template <typename T, int K>
__device__ inline void mg_colour(const Lev<T> &L, int p, int c, int c0, int mode, int active) {
  MgRow<T, K> r;
  mg_place(L, p, r);
  if (mode == kFwd0 && c == 0) {
    have(r.info);
    if (active) mg_first(L, p, r.info, r.b, r.ap);
    return;
  }
  if (K == 6) {
    mg_entries(L, r);
#pragma unroll
    for (int k = 0; k < K; k++) have(r.c[k]);
    if (active) mg_node(L, p, c0, mode, r);
  } else {
    have(r.e);
    have(r.info);
    if (!active) return;
    mg_entries(L, r);
    mg_node(L, p, c0, mode, r);
  }
}
// Step q of a sweep: colour q (positions c0 .. c0 + cnt - 1), or, at q =
// ctail, the remaining colours one after the other in one workgroup (greedy
// colourings end in a few colours of a few nodes, where a launch of its own
// costs more than its work), one node a thread at a time, whose row is loaded
// while the nodes before it compute.
template <typename T>
__device__ inline void d_mg_sweep(int bx, const Lev<T> &L, int q, int c0, int cnt, int mode,
                                  const CgCtl *ctl) {
  const int active = ctl->active;
  if (cnt >= 0) {
    const int t = bx * blockDim.x + threadIdx.x;
    if (t >= cnt) return;
    if (L.uni == 6)
      mg_colour<T, 6>(L, c0 + t, q, c0, mode, active);
    else
      mg_colour<T, 8>(L, c0 + t, q, c0, mode, active);
    return;
  }
  if (!active) return;
  const int nt = blockDim.x;
  auto colour = [&](int i) { return mode == kBwd ? L.ncol - 1 - (i - L.ctail) : i; };
  auto load = [&](int beg, int n, int t, MgRow<T, 8> &r) {
    if (t >= n) return;
    mg_place(L, beg + t, r);
    mg_entries(L, r);
  };
  int i = L.ctail, t0 = 0, beg = L.cbeg[colour(i)], n = L.ccnt[colour(i)];
  MgRow<T, 8> A, B;
  load(beg, n, threadIdx.x, A);
  while (i < L.ncol) {
    int ni = i, nt0 = t0 + nt, nbeg = beg, nn = n;
    if (nt0 >= n) {
      ni = i + 1;
      nt0 = 0;
      if (ni < L.ncol) {
        nbeg = L.cbeg[colour(ni)];
        nn = L.ccnt[colour(ni)];
      }
    }
    if (ni < L.ncol) load(nbeg, nn, nt0 + static_cast<int>(threadIdx.x), B);
    const int t = t0 + static_cast<int>(threadIdx.x);
    if (t < n) mg_node(L, beg + t, beg, mode, A);
    if (ni != i) __syncthreads();
    A = B;
    i = ni;
    t0 = nt0;
    beg = nbeg;
    n = nn;
  }
}

// Residual b_i + sum anb x_nb - ap_i x_i of the nodes the forward sweep has
// not left it for.  A pass of its own in position order: the restriction takes
// its members from all over the level, and rows gathered that way (4 lines of
// 128 bytes for 24 used) cost more than the pass and its t together (mean over
// the three grid-wide levels at 128^3 in FP32: 31 us fused, 7 + 7 us split).
template <typename T>
__device__ inline int mg_open(const Lev<T> &F) {
  return F.fin >= 0 ? F.fin : F.npad;
}
template <typename T>
__device__ inline void mg_residual(const Lev<T> &F, int p) {
  if (mg_final(F, p)) return;
  const int len = F.uni == 6 ? 6 : F.info[p] & 0x7fff;
  F.t[p] = row_sum(F, mg_entry(F, p), len, F.b[p], [&](int q) { return F.x[q]; }) - F.ap[p] * F.x[p];
}
template <typename T>
__device__ inline void d_mg_residual(int p, int n, const Lev<T> &F, const CgCtl *ctl) {
  const int active = ctl->active;
  if (p >= n) return;
  if (F.uni == 6) {
    if (active) mg_residual(F, p);
    return;
  }
  MgRow<T, 8> r;
  mg_place(F, p, r);
  have(r.e);
  have(r.info);
  if (!active || r.info >> 15) return;
  F.t[p] = row_sum(F, r.e, r.info & 0x7fff, r.b, [&](int q) { return F.x[q]; }) - r.ap * F.x[p];
}
// restriction to position I: the sum of its members' residuals in order, from zero
template <typename T>
__device__ inline void mg_restrict(int I, int q0, int q1, const Lev<T> &F, T *bC) {
  T acc = static_cast<T>(0);
  for (; q0 < q1; q0 += 8) {
    int m[8];
    T v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) m[k] = F.mem[min(q0 + k, q1 - 1)];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = F.t[m[k]];
#pragma unroll
    for (int k = 0; k < 8; k++) acc = q0 + k < q1 ? acc + v[k] : acc;
  }
  bC[I] = acc;
}
template <typename T>
__device__ inline void d_mg_restrict(int I, int n, const Lev<T> &F, T *bC, const CgCtl *ctl) {
  const int active = ctl->active;
  if (I >= n) return;
  int q0 = F.mptr[I], q1 = F.mptr[I + 1];
  have(q0);
  have(q1);
  if (active) mg_restrict(I, q0, q1, F, bC);
}

// Prolongation x_i += x_C(agg_i), for every colour but the last: the backward
// sweep computes that one first, from the others alone.
template <typename T>
__device__ inline int mg_prolonged(const Lev<T> &F) {
  return F.cbeg[F.ncol - 1];
}
template <typename T>
__device__ inline void d_mg_prolong(int i, int n, const Lev<T> &F, const T *__restrict__ xc,
                                    const CgCtl *ctl) {
  const int active = ctl->active;
  if (i >= n) return;
  int g = F.agg[i];
  have(g);
  if (active) F.x[i] = F.x[i] + xc[g];
}

// The small levels lc .. nlev-1 of the V-cycle in one workgroup: the same
// sweeps, restrictions and prolongations as the grid-wide kernels, with a
// barrier where those have a kernel boundary.  lv[lc].b is the restricted
// residual.  The levels' x and the coarser ones' b live in LDS (coarse_lds
// bytes, host), so a colour's only global loads are its rows, which depend on
// nothing before them.
// A level of that workgroup: x, b, and the tables of colours and slices in LDS.
template <typename T>
struct WgLev {
  Lev<T> L;
  const int *cbeg, *ccnt, *sptr;  // sptr has one more entry, the total
};
// A node's row as loaded ahead of its turn: the first kAhead entries (a short
// row's last one again), its scalars and what the rest needs.
constexpr int kAhead = 8;
template <typename T>
struct WgRow {
  int p, e, info, c[kAhead];
  T a[kAhead], b, ap;
};
template <typename T>
__device__ inline void wg_load(const WgLev<T> &W, int p, bool on, WgRow<T> &r) {
  const Lev<T> &L = W.L;
  r.p = on ? p : -1;
  if (!on) return;
  const int s0 = W.sptr[p >> 6], last = (W.sptr[(p >> 6) + 1] - s0) / 64 - 1;
  r.e = s0 + (p & 63);
  r.info = L.info[p];
  r.b = L.b[p];
  r.ap = L.ap[p];
#pragma unroll
  for (int k = 0; k < kAhead; k++) {
    const int q = r.e + 64 * max(min(k, last), 0);
    r.c[k] = L.col[q];
    r.a[k] = L.anb[q];
  }
}
// the row's sum from acc and the node's update: mg_node on a loaded row
template <typename T>
__device__ inline void wg_node(const WgLev<T> &W, const WgRow<T> &r, int c0, int mode) {
  const Lev<T> &L = W.L;
  if (r.p < 0) return;
  const T zero = static_cast<T>(0);
  const int len = r.info & 0x7fff;
  T v[kAhead], acc = r.b;
#pragma unroll
  for (int k = 0; k < kAhead; k++)
    v[k] = mode != kFwd0 || r.c[k] < c0 ? L.x[r.c[k]] : zero;
#pragma unroll
  for (int k = 0; k < kAhead; k++) acc = k < len ? acc + r.a[k] * v[k] : acc;
  for (int k = kAhead; k < len; k++) {
    const int q = L.col[r.e + 64 * k];
    acc = acc + L.anb[r.e + 64 * k] * (mode != kFwd0 || q < c0 ? L.x[q] : zero);
  }
  const T x = acc / r.ap;
  L.x[r.p] = x;
  if (mode == kFwd0 && (r.info >> 15)) L.t[r.p] = acc - r.ap * x;
}
// A sweep: the colours in chunks of one node a thread, a barrier after each
// colour; a chunk's rows are loaded while the one before computes, so a
// colour waits for LDS and its division, not for memory.
template <typename T>
__device__ void wg_sweep(const WgLev<T> &W, int mode) {
  const int ncol = W.L.ncol, nt = blockDim.x;
  int i = 0, t0 = 0;
  auto colour = [&](int j) { return mode == kBwd ? ncol - 1 - j : j; };
  auto load = [&](int j, int t, WgRow<T> &r) {
    const int c = colour(j), q = t + threadIdx.x;
    wg_load(W, W.cbeg[c] + q, q < W.ccnt[c], r);
  };
  WgRow<T> A, B;
  load(0, 0, A);
  while (i < ncol) {
    const int c = colour(i);
    int ni = i, nt0 = t0 + nt;
    if (nt0 >= W.ccnt[c]) ni = i + 1, nt0 = 0;
    if (ni < ncol) load(ni, nt0, B);
    wg_node(W, A, W.cbeg[c], mode);
    if (ni != i) __syncthreads();
    A = B;
    i = ni;
    t0 = nt0;
  }
}
// kCoarseSweeps symmetric sweep pairs from x = 0 on a coarsest level of at
// most 64 nodes by one wavefront, whose LDS accesses complete in program
// order: lane p holds the row of node p in registers (K entries).  The colour
// at a turn is computed once: its second value would come from the same
// neighbour values.
template <typename T, int K>
__device__ void wave_coarsest(const Lev<T> &Z, const T *bz, T *xs) {
  const int p = threadIdx.x, n = Z.n;
  const int pc = min(p, n - 1), len = p < n ? Z.info[pc] & 0x7fff : 0, e = mg_entry(Z, pc);
  int c[K];
  T a[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int q = e + 64 * min(k, max(len - 1, 0));
    c[k] = len > 0 ? Z.col[q] : 0;
    a[k] = len > 0 ? Z.anb[q] : static_cast<T>(0);
  }
  const T b = bz[pc], ap = Z.ap[pc];
  int mine = -1;  // the lane's colour
  for (int q = 0; q < Z.ncol; q++)
    if (p >= Z.cbeg[q] && p < Z.cbeg[q] + Z.ccnt[q]) mine = q;
  auto colour = [&](int q) {
    if (q == mine) {
      T v[K], acc = b;
#pragma unroll
      for (int k = 0; k < K; k++) v[k] = xs[c[k]];
#pragma unroll
      for (int k = 0; k < K; k++) acc = k < len ? acc + a[k] * v[k] : acc;
      xs[p] = acc / ap;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  if (p < n) xs[p] = static_cast<T>(0);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  colour(0);
  for (int k = 0; k < kCoarseSweeps; k++) {
    for (int q = 1; q < Z.ncol; q++) colour(q);
    for (int q = Z.ncol - 2; q >= 0; q--) colour(q);
  }
}
template <typename T>
__device__ inline void d_mg_coarse(const Lev<T> *__restrict__ lv, int lc, int nlev,
                                   const CgCtl *ctl) {
  extern __shared__ double dyn_lds[];
  if (!ctl->active) return;
  // each level's view: x (and below lc, b) and its tables in LDS
  T *at = reinterpret_cast<T *>(dyn_lds);
  int *tab = reinterpret_cast<int *>(at);
  {
    int reals = 0;
    for (int i = lc; i < nlev; i++) reals += (i == lc ? 1 : 2) * lv[i].npad;
    tab = reinterpret_cast<int *>(at + reals);
  }
  auto level = [&](int l) {
    WgLev<T> W;
    T *q = at;
    int *k = tab;
    for (int i = lc; i < l; i++) {
      q += (i == lc ? 1 : 2) * lv[i].npad;
      k += 2 * lv[i].ncol + (lv[i].npad + 63) / 64 + 1;
    }
    W.L = lv[l];
    W.L.x = q;
    if (l > lc) W.L.b = q + W.L.npad;
    W.cbeg = k;
    W.ccnt = k + W.L.ncol;
    W.sptr = k + 2 * W.L.ncol;
    return W;
  };
  for (int l = lc; l < nlev; l++) {
    const WgLev<T> W = level(l);
    int *k = const_cast<int *>(W.cbeg);
    for (int i = threadIdx.x; i < W.L.ncol; i += blockDim.x) {
      k[i] = W.L.cbeg[i];
      k[W.L.ncol + i] = W.L.ccnt[i];
    }
    for (int i = threadIdx.x; i <= (W.L.npad + 63) / 64; i += blockDim.x)
      k[2 * W.L.ncol + i] = W.L.sptr[i];
  }
  __syncthreads();
  for (int l = lc; l < nlev - 1; l++) {
    const WgLev<T> F = level(l), C = level(l + 1);
    wg_sweep(F, kFwd0);
    for (int p = threadIdx.x; p < mg_open(F.L); p += blockDim.x) mg_residual(F.L, p);
    __syncthreads();
    for (int I = threadIdx.x; I < C.L.npad; I += blockDim.x)
      mg_restrict(I, F.L.mptr[I], F.L.mptr[I + 1], F.L, C.L.b);
    __syncthreads();
  }
  const WgLev<T> Z = level(nlev - 1);
  if (Z.L.n <= 64 && Z.L.kmax <= 20) {
    if (threadIdx.x < 64) {
      if (Z.L.kmax <= 6)
        wave_coarsest<T, 6>(Z.L, Z.L.b, Z.L.x);
      else if (Z.L.kmax <= 12)
        wave_coarsest<T, 12>(Z.L, Z.L.b, Z.L.x);
      else
        wave_coarsest<T, 20>(Z.L, Z.L.b, Z.L.x);
    }
    __syncthreads();
  } else {
    for (int k = 0; k < kCoarseSweeps; k++) {
      wg_sweep(Z, k == 0 ? kFwd0 : kFwd);
      wg_sweep(Z, kBwd);
    }
  }
  for (int l = nlev - 2; l >= lc; l--) {
    const WgLev<T> F = level(l);
    const T *xc = level(l + 1).L.x;
    const int n = F.cbeg[F.L.ncol - 1];
    for (int i = threadIdx.x; i < n; i += blockDim.x) F.L.x[i] = F.L.x[i] + xc[F.L.agg[i]];
    __syncthreads();
    wg_sweep(F, kBwd);
  }
  const Lev<T> F = level(lc).L;
  for (int i = threadIdx.x; i < F.npad; i += blockDim.x) lv[lc].x[i] = F.x[i];
}

template <typename T>
__global__ void k_mg_copy0(Lev<T> L, const int *__restrict__ pos, const int *__restrict__ row,
                           const double *__restrict__ ap, const double *__restrict__ anb) {
  d_mg_copy0<T>(xcd_block() * blockDim.x + threadIdx.x, L, pos, row, ap, anb);
}
template <typename T>
__global__ void k_mg_galerkin(Lev<T> F, Lev<T> C) {
  d_mg_galerkin<T>(blockIdx.x * blockDim.x + threadIdx.x, F, C);
}
template <typename T>
__global__ void __launch_bounds__(1024)
k_mg_sweep(Lev<T> L, int q, int c0, int cnt, int mode, const CgCtl *ctl) {
  d_mg_sweep<T>(xcd_block(), L, q, c0, cnt, mode, ctl);
}
template <typename T>
__global__ void k_mg_residual(Lev<T> F, int n, const CgCtl *ctl) {
  d_mg_residual<T>(xcd_block() * blockDim.x + threadIdx.x, n, F, ctl);
}
template <typename T>
__global__ void k_mg_restrict(Lev<T> F, int n, T *bC, const CgCtl *ctl) {
  d_mg_restrict<T>(xcd_block() * blockDim.x + threadIdx.x, n, F, bC, ctl);
}
template <typename T>
__global__ void k_mg_prolong(Lev<T> F, int n, const T *__restrict__ xc, const CgCtl *ctl) {
  d_mg_prolong<T>(xcd_block() * blockDim.x + threadIdx.x, n, F, xc, ctl);
}
template <typename T>
__global__ void __launch_bounds__(kCoarseThreads)
k_mg_coarse(const Lev<T> *__restrict__ lv, int lc, int nlev, const CgCtl *ctl) {
  d_mg_coarse<T>(lv, lc, nlev, ctl);
}

// ---------------------------------------------------------------------------
// Grouped kernels: one launch runs a step for every system of a group.  Each
// system's descriptor (device memory) holds its vectors, its control block
// and its levels.
// ---------------------------------------------------------------------------
template <typename T>
struct MgSlot {
  Red R;
  int ne, nit, nlev, lc;
  const int *row, *nbr, *pos;
  const double *ap, *anb, *b;
  double *phi, *r, *p, *q, *part;
  T *rt, *z;              // level 0's right-hand side and values
  CgCtl *ctl;
  const Lev<T> *lv;       // device levels
  LogLine *log;
  int *nlog;
  LogLine tmpl;
  uint64_t serial;  // the solver's
};

template <typename T>
__global__ void g_mg_copy0(GroupMap g, const MgSlot<T> *__restrict__ S) {
  int bx;
  const MgSlot<T> &x = S[group_slot(g, bx)];
  const Lev<T> L = x.lv[0];
  d_mg_copy0<T>(bx * blockDim.x + threadIdx.x, L, x.pos, x.row, x.ap, x.anb);
}
template <typename T>
__global__ void g_mg_galerkin(GroupMap g, const MgSlot<T> *__restrict__ S, int l) {
  int bx;
  const MgSlot<T> &x = S[group_slot(g, bx, true)];
  const Lev<T> F = x.lv[l], C = x.lv[l + 1];
  d_mg_galerkin<T>(bx * blockDim.x + threadIdx.x, F, C);
}
template <typename T>
__global__ void __launch_bounds__(kRedThreads) g_cg_init(GroupMap g, const MgSlot<T> *__restrict__ S) {
  int bx;
  const MgSlot<T> &x = S[group_slot(g, bx)];
  d_cg_init<T>(bx, x.R, x.row, x.nbr, x.pos, x.ap, x.anb, x.b, x.phi, x.r, x.rt, x.ctl, x.part,
               x.nit);
}
// step i of a sweep of level l, or of the system's coarsest level for l < 0
// (backward: counted from the last step)
template <typename T>
__global__ void __launch_bounds__(1024)
g_mg_sweep(GroupMap g, const MgSlot<T> *__restrict__ S, int l, int i, int mode) {
  int bx;
  const MgSlot<T> &x = S[group_slot(g, bx)];
  const Lev<T> L = x.lv[l < 0 ? x.nlev - 1 : l];
  const int nstep = L.ctail < L.ncol ? L.ctail + 1 : L.ncol, q = mode == kBwd ? nstep - 1 - i : i;
  const bool tail = q >= L.ctail;
  d_mg_sweep<T>(bx, L, q, tail ? 0 : L.cbeg[q], tail ? -1 : L.ccnt[q], mode, x.ctl);
}
template <typename T>
__global__ void g_mg_residual(GroupMap g, const MgSlot<T> *__restrict__ S, int l) {
  int bx;
  const MgSlot<T> &x = S[group_slot(g, bx)];
  const Lev<T> F = x.lv[l];
  d_mg_residual<T>(bx * blockDim.x + threadIdx.x, mg_open(F), F, x.ctl);
}
template <typename T>
__global__ void g_mg_restrict(GroupMap g, const MgSlot<T> *__restrict__ S, int l) {
  int bx;
  const MgSlot<T> &x = S[group_slot(g, bx)];
  const Lev<T> F = x.lv[l];
  d_mg_restrict<T>(bx * blockDim.x + threadIdx.x, x.lv[l + 1].npad, F, x.lv[l + 1].b, x.ctl);
}
template <typename T>
__global__ void g_mg_prolong(GroupMap g, const MgSlot<T> *__restrict__ S, int l) {
  int bx;
  const MgSlot<T> &x = S[group_slot(g, bx)];
  const Lev<T> F = x.lv[l];
  d_mg_prolong<T>(bx * blockDim.x + threadIdx.x, mg_prolonged(F), F, x.lv[l + 1].x, x.ctl);
}
template <typename T>
__global__ void __launch_bounds__(kCoarseThreads)
g_mg_coarse(GroupMap g, const MgSlot<T> *__restrict__ S) {
  int bx;
  const MgSlot<T> &x = S[group_slot(g, bx)];
  d_mg_coarse<T>(x.lv, x.lc, x.nlev, x.ctl);
}
template <typename T>
__global__ void __launch_bounds__(kRedThreads) g_cg_rz(GroupMap g, const MgSlot<T> *__restrict__ S) {
  int bx;
  const MgSlot<T> &x = S[group_slot(g, bx)];
  d_cg_rz<T>(bx, x.R, x.r, x.z, x.pos, x.ctl, x.part);
}
template <typename T>
__global__ void g_cg_p(GroupMap g, const MgSlot<T> *__restrict__ S) {
  int bx;
  const MgSlot<T> &x = S[group_slot(g, bx)];
  d_cg_p<T>(bx * blockDim.x + threadIdx.x, x.ne, x.z, x.pos, x.p, x.ctl);
}
template <typename T>
__global__ void __launch_bounds__(kRedThreads) g_cg_spmv(GroupMap g, const MgSlot<T> *__restrict__ S) {
  int bx;
  const MgSlot<T> &x = S[group_slot(g, bx)];
  d_cg_spmv(bx, x.R, x.row, x.nbr, x.ap, x.anb, x.p, x.q, x.ctl, x.part);
}
template <typename T>
__global__ void __launch_bounds__(kRedThreads) g_cg_update(GroupMap g, const MgSlot<T> *__restrict__ S) {
  int bx;
  const MgSlot<T> &x = S[group_slot(g, bx)];
  d_cg_update<T>(bx, x.R, x.phi, x.p, x.q, x.pos, x.r, x.rt, x.ctl, x.part);
}
// the active flags of systems 0 .. n-1, and their log lines at the end
template <typename T>
__global__ void g_cg_flags(int n, const MgSlot<T> *__restrict__ S, int *flags) {
  const int k = threadIdx.x;
  if (k < n) flags[k] = S[k].ctl->active;
}
template <typename T>
__global__ void g_cg_log(int n, const MgSlot<T> *__restrict__ S) {
  const int k = threadIdx.x;
  if (k < n) d_cg_log(S[k].ctl, S[k].log, S[k].nlog, S[k].tmpl);
}

inline int nb(int n, int b) { return (n + b - 1) / b; }

}  // namespace
// device copy of the hierarchy and the solve's work vectors
struct MgCgSolver {
  const uint64_t serial = next_serial();
  int fp32 = 0, ne = 0, nbf = 0, nlev = 0, lc = 0;
  size_t coarse_lds = 0;  // LDS of the workgroup that runs levels lc ..
  std::vector<void *> mem;
  std::vector<std::vector<int>> cbeg, ccnt;  // first position and nodes per level and colour (host)
  std::vector<int> open, prolonged;    // positions of d_mg_residual and d_mg_prolong, per level
  // the levels for one real type (host copies of the device descriptors)
  std::vector<Lev<double>> lvd;
  std::vector<Lev<float>> lvf;
  Lev<double> *d_lvd = nullptr;
  Lev<float> *d_lvf = nullptr;
  const int *pos = nullptr;  // level 0's position of each cell
  double *r = nullptr, *p = nullptr, *q = nullptr, *part = nullptr;
  CgCtl *ctl = nullptr;
  int *hflag = nullptr;  // pinned
  hipEvent_t ev[2] = {nullptr, nullptr};
  int launches = 0;

  ~MgCgSolver() {
    for (void *m : mem) (void)hipFree(m);
    if (hflag) (void)hipHostFree(hflag);
    for (auto &e : ev)
      if (e) (void)hipEventDestroy(e);
  }
  template <typename X>
  int alloc(X **p, size_t n) {
    void *v = nullptr;
    hipError_t e = hipMalloc(&v, sizeof(X) * (n > 0 ? n : 1));
    if (e != hipSuccess) {
      set_error(std::string("hipMalloc (multigrid): ") + hipGetErrorString(e));
      return CFDL_ENOMEM;
    }
    mem.push_back(v);
    *p = static_cast<X *>(v);
    return CFDL_OK;
  }
  template <typename X>
  int upload(const std::vector<X> &v, const X **out) {
    X *d = nullptr;
    if (int rc = alloc(&d, v.size())) return rc;
    if (!v.empty()) MGCHK(hipMemcpy(d, v.data(), sizeof(X) * v.size(), hipMemcpyHostToDevice));
    *out = d;
    return CFDL_OK;
  }
};

#define MGCALL(x)          \
  do {                     \
    int rc_ = (x);         \
    if (rc_) return rc_;   \
  } while (0)

namespace {
template <typename T>
std::vector<Lev<T>> &host_levels(MgCgSolver *s);
template <>
std::vector<Lev<double>> &host_levels<double>(MgCgSolver *s) { return s->lvd; }
template <>
std::vector<Lev<float>> &host_levels<float>(MgCgSolver *s) { return s->lvf; }
template <typename T>
Lev<T> *&dev_levels(MgCgSolver *s);
template <>
Lev<double> *&dev_levels<double>(MgCgSolver *s) { return s->d_lvd; }
template <>
Lev<float> *&dev_levels<float>(MgCgSolver *s) { return s->d_lvf; }

// One level's numbering by colour and its sliced rows (struct Lev).
struct Numbering {
  std::vector<int> pos;              // position of each node
  std::vector<int> cbeg, ccnt;       // per colour
  std::vector<int> sptr, slot;       // slice starts; entry of each CSR slot
  std::vector<unsigned short> info;  // per position
  int npad = 0, nent = 0, uni = 0, fin = -1, kmax = 0;
};
// align: positions a colour's start is rounded up to (64, or 1 inside the
// workgroup-only levels, whose coarsest is one node a lane)
int number_level(const MgLevel &H, int align, bool level0, Numbering *out) {
  Numbering &N = *out;
  N.pos.assign(H.n, 0);
  std::vector<int> node;
  for (int c = 0; c < H.ncol; c++) {
    while (static_cast<int>(node.size()) % align) node.push_back(-1);
    N.cbeg.push_back(static_cast<int>(node.size()));
    N.ccnt.push_back(H.cptr[c + 1] - H.cptr[c]);
    for (int q = H.cptr[c]; q < H.cptr[c + 1]; q++) {
      N.pos[H.cperm[q]] = static_cast<int>(node.size());
      node.push_back(H.cperm[q]);
    }
  }
  while (static_cast<int>(node.size()) % align) node.push_back(-1);
  N.npad = static_cast<int>(node.size());
  bool six = level0;
  int64_t at = 0;
  N.info.assign(N.npad, 0);
  for (int p0 = 0; p0 < N.npad; p0 += 64) {
    int k = 0;
    for (int p = p0; p < std::min(p0 + 64, N.npad); p++)
      if (node[p] >= 0) k = std::max(k, H.row[node[p] + 1] - H.row[node[p]]);
    N.sptr.push_back(static_cast<int>(at));
    at += 64 * int64_t{k};
  }
  if (at > 0x7fffffff) {
    set_error("mgcg_create: level too large");
    return CFDL_EINVAL;
  }
  N.nent = static_cast<int>(at);
  N.sptr.push_back(N.nent);
  N.slot.assign(H.nnz, 0);
  for (int c = 0, p = 0; p < N.npad; p++) {
    const int i = node[p];
    if (i < 0) continue;
    while (c + 1 < H.ncol && p >= N.cbeg[c + 1]) c++;
    const int len = H.row[i + 1] - H.row[i];
    if (len > 0x7fff) {
      set_error("mgcg_create: row of more than 32767 entries");
      return CFDL_EINVAL;
    }
    six = six && len == 6;
    bool final = true;
    for (int k = H.row[i]; k < H.row[i + 1]; k++) {
      N.slot[k] = N.sptr[p >> 6] + 64 * (k - H.row[i]) + (p & 63);
      if (H.col[k] < H.n && N.pos[H.col[k]] >= N.cbeg[c]) final = false;
    }
    N.info[p] = static_cast<unsigned short>(len | (final ? 0x8000 : 0));
    N.kmax = std::max(N.kmax, len);
  }
  if (six) N.uni = 6;  // every slice then holds 6 entries a position
  // the final nodes as a range at the end, when they are one
  int f = N.npad;
  while (f > 0 && (node[f - 1] < 0 || (N.info[f - 1] >> 15))) f--;
  bool range = true;
  for (int p = 0; p < f && range; p++) range = node[p] < 0 || !(N.info[p] >> 15);
  if (range) N.fin = f;
  return CFDL_OK;
}

template <typename T>
int fill_levels(MgCgSolver *s, const MgHier &h) {
  std::vector<Lev<T>> &lv = host_levels<T>(s);
  lv.assign(s->nlev, Lev<T>{});
  std::vector<Numbering> num(s->nlev);
  for (int l = 0; l < s->nlev; l++)
    MGCALL(number_level(h.lv[l], l < s->lc ? 64 : 1, l == 0, &num[l]));
  auto zeroed = [&](T **p, size_t n) -> int {
    MGCALL(s->alloc(p, n));
    MGCHK(hipMemset(*p, 0, sizeof(T) * (n > 0 ? n : 1)));
    return CFDL_OK;
  };
  for (int l = 0; l < s->nlev; l++) {
    const MgLevel &H = h.lv[l];
    const Numbering &N = num[l];
    Lev<T> &L = lv[l];
    L.n = H.n;
    L.npad = N.npad;
    L.nnz = H.nnz;
    L.ncol = H.ncol;
    L.uni = N.uni;
    L.fin = N.fin;
    L.kmax = N.kmax;
    // the tail: the trailing colours of together at most kTailNodes nodes,
    // if they are at least two
    int tail = H.ncol, left = 0;
    while (tail > 1 && left + N.ccnt[tail - 1] <= kTailNodes) left += N.ccnt[--tail];
    L.ctail = H.ncol - tail >= 2 ? tail : H.ncol;
    s->cbeg.push_back(N.cbeg);
    s->ccnt.push_back(N.ccnt);
    s->prolonged.push_back(N.cbeg[H.ncol - 1]);
    s->open.push_back(N.fin >= 0 ? N.fin : N.npad);
    std::vector<int> col(N.nent + 64, 0);  // an empty slice's loads stay inside
    for (int i = 0; i < H.n; i++)
      for (int k = H.row[i]; k < H.row[i + 1]; k++)
        col[N.slot[k]] = H.col[k] < H.n ? N.pos[H.col[k]] : N.npad + (H.col[k] - H.n);
    MGCALL(s->upload(N.cbeg, &L.cbeg));
    MGCALL(s->upload(N.ccnt, &L.ccnt));
    MGCALL(s->upload(N.sptr, &L.sptr));
    MGCALL(s->upload(N.info, &L.info));
    MGCALL(s->upload(col, &L.col));
    MGCALL(zeroed(&L.ap, N.npad));
    MGCALL(zeroed(&L.anb, N.nent + 64));
    MGCALL(zeroed(&L.b, N.npad));
    MGCALL(zeroed(&L.x, N.npad + (l == 0 ? s->nbf : 0)));
    MGCALL(zeroed(&L.t, N.npad));
    if (l > 0) MGCALL(s->upload(N.slot, &L.gpos));
    if (l == 0) MGCALL(s->upload(N.pos, &s->pos));
    if (l + 1 == s->nlev) continue;
    const Numbering &C = num[l + 1];
    const MgLevel &HC = h.lv[l + 1];
    std::vector<int> agg(N.npad, 0), at(C.npad, -1), mptr(1, 0), mem, iptr(1, 0), ilist;
    for (int i = 0; i < H.n; i++) agg[N.pos[i]] = C.pos[H.agg[i]];
    for (int g = 0; g < HC.n; g++) at[C.pos[g]] = g;
    for (int p = 0; p < C.npad; p++) {
      const int g = at[p];
      for (int q = g < 0 ? 0 : H.mptr[g]; g >= 0 && q < H.mptr[g + 1]; q++)
        mem.push_back(N.pos[H.mem[q]]);
      for (int q = g < 0 ? 0 : H.iptr[g]; g >= 0 && q < H.iptr[g + 1]; q++)
        ilist.push_back(N.slot[H.ilist[q]]);
      mptr.push_back(static_cast<int>(mem.size()));
      iptr.push_back(static_cast<int>(ilist.size()));
    }
    std::vector<int> glist(H.glist.size());
    for (size_t q = 0; q < glist.size(); q++) glist[q] = N.slot[H.glist[q]];
    MGCALL(s->upload(agg, &L.agg));
    MGCALL(s->upload(mptr, &L.mptr));
    MGCALL(s->upload(mem, &L.mem));
    MGCALL(s->upload(iptr, &L.iptr));
    MGCALL(s->upload(ilist, &L.ilist));
    MGCALL(s->upload(H.gptr, &L.gptr));
    MGCALL(s->upload(glist, &L.glist));
  }
  for (int l = s->lc; l < s->nlev; l++)
    s->coarse_lds += sizeof(T) * (l == s->lc ? 1 : 2) * static_cast<size_t>(num[l].npad) +
                     sizeof(int) * (num[l].cbeg.size() * 2 + num[l].sptr.size());
  MGCALL(s->alloc(&dev_levels<T>(s), s->nlev));
  MGCHK(hipMemcpy(dev_levels<T>(s), lv.data(), sizeof(Lev<T>) * s->nlev, hipMemcpyHostToDevice));
  return CFDL_OK;
}

// steps of a sweep (d_mg_sweep), and the blocks of blk threads of step i
// counted in the sweep's direction
template <typename T>
int sweep_steps(const Lev<T> &L) {
  return L.ctail < L.ncol ? L.ctail + 1 : L.ncol;
}
template <typename T>
int sweep_blocks(const MgCgSolver *s, int l, const Lev<T> &L, int i, int mode, int blk) {
  const int n = sweep_steps(L), q = mode == kBwd ? n - 1 - i : i;
  return i >= n ? 0 : q < L.ctail ? nb(s->ccnt[l][q], blk) : 1;
}

// one V-cycle: z = M r on level 0 (lv[0].b = r, lv[0].x = z)
template <typename T>
int vcycle(MgCgSolver *s, hipStream_t st) {
  const std::vector<Lev<T>> &lv = host_levels<T>(s);
  const CgCtl *ctl = s->ctl;
  const int nlev = s->nlev, lc = s->lc;
  auto sweep = [&](int l, int mode) {
    const Lev<T> &L = lv[l];
    const int n = sweep_steps(L);
    for (int i = 0; i < n; i++) {
      const int q = mode == kBwd ? n - 1 - i : i;
      const bool tail = q >= L.ctail;
      const dim3 g(sweep_blocks(s, l, L, i, mode, kBlk)), b(tail ? kTailNodes : kBlk);
      hipLaunchKernelGGL(k_mg_sweep<T>, g, b, 0, st, L, q, tail ? 0 : s->cbeg[l][q],
                         tail ? -1 : s->ccnt[l][q], mode, ctl);
      s->launches++;
    }
  };
  // grid-wide levels 0 .. lc-1 (the coarsest among them, if no small
  // levels follow, smoothed in place)
  const int top = lc < nlev ? lc : nlev - 1;
  for (int l = 0; l < top; l++) {
    sweep(l, kFwd0);
    if (s->open[l] > 0)
      hipLaunchKernelGGL(k_mg_residual<T>, dim3(nb(s->open[l], kBlk)), dim3(kBlk), 0, st, lv[l],
                         s->open[l], ctl);
    hipLaunchKernelGGL(k_mg_restrict<T>, dim3(nb(lv[l + 1].npad, kBlk)), dim3(kBlk), 0, st, lv[l],
                       lv[l + 1].npad, lv[l + 1].b, ctl);
    s->launches += 2;
  }
  if (lc < nlev) {
    hipLaunchKernelGGL(k_mg_coarse<T>, dim3(1), dim3(kCoarseThreads), s->coarse_lds, st,
                       static_cast<const Lev<T> *>(dev_levels<T>(s)), lc, nlev, ctl);
    s->launches++;
  } else {
    for (int k = 0; k < kCoarseSweeps; k++) {
      sweep(nlev - 1, k == 0 ? kFwd0 : kFwd);
      sweep(nlev - 1, kBwd);
    }
  }
  for (int l = top - 1; l >= 0; l--) {
    if (s->prolonged[l] > 0) {
      hipLaunchKernelGGL(k_mg_prolong<T>, dim3(nb(s->prolonged[l], kBlk)), dim3(kBlk), 0, st,
                         lv[l], s->prolonged[l], static_cast<const T *>(lv[l + 1].x), ctl);
      s->launches++;
    }
    sweep(l, kBwd);
  }
  MGCHK(hipGetLastError());
  return CFDL_OK;
}
}  // namespace

int mgcg_create(const MgHier &h, int nbf, int fp32, MgCgSolver **out) {
  std::unique_ptr<MgCgSolver> s(new MgCgSolver());
  s->fp32 = fp32 ? 1 : 0;
  s->nlev = static_cast<int>(h.lv.size());
  if (s->nlev < 1 || h.lv[0].n < 1) {
    set_error("mgcg_create: empty hierarchy");
    return CFDL_EINVAL;
  }
  s->ne = h.lv[0].n;
  s->nbf = nbf;
  // the small levels that run in one workgroup: the trailing levels (below
  // level 0) of at most kCoarseMax nodes whose x, b and tables fit 64 KB of LDS
  s->lc = s->nlev;
  size_t below = 0, real = fp32 ? sizeof(float) : sizeof(double);
  while (s->lc - 1 >= 1 && h.lv[s->lc - 1].n <= kCoarseMax &&
         below + real * h.lv[s->lc - 1].n <= 57344) {
    s->lc--;
    below += 2 * real * h.lv[s->lc].n;
  }
  const int ne = s->ne, nall = ne + nbf;
  MGCALL(s->alloc(&s->r, ne));
  MGCALL(s->alloc(&s->q, ne));
  MGCALL(s->alloc(&s->p, nall));
  MGCALL(s->alloc(&s->part, 2 * kMaxRedBlocks));
  MGCALL(s->alloc(&s->ctl, 1));
  MGCHK(hipMemset(s->ctl, 0, sizeof(CgCtl)));
  MGCHK(hipMemset(s->p, 0, sizeof(double) * nall));
  MGCALL(s->fp32 ? fill_levels<float>(s.get(), h) : fill_levels<double>(s.get(), h));
  MGCHK(hipHostMalloc(reinterpret_cast<void **>(&s->hflag), 2 * sizeof(int), hipHostMallocDefault));
  MGCHK(hipEventCreateWithFlags(&s->ev[0], hipEventDisableTiming));
  MGCHK(hipEventCreateWithFlags(&s->ev[1], hipEventDisableTiming));
  *out = s.release();
  return CFDL_OK;
}

void mgcg_destroy(MgCgSolver *s) { delete s; }

void mgcg_stats(const MgCgSolver *s, int *launches, int *levels) {
  if (launches) *launches = s ? s->launches : 0;
  if (levels) *levels = s ? s->nlev : 0;
}

namespace {
template <typename T>
int solve(MgCgSolver *s, const MgCgSystem &sys, hipStream_t st) {
  const int ne = s->ne;
  const Red R = red_of(ne);
  std::vector<Lev<T>> &lv = host_levels<T>(s);
  T *rt = lv[0].b;
  const T *z = lv[0].x;
  s->launches = 0;
  hipLaunchKernelGGL(k_mg_copy0<T>, dim3(nb(ne, kBlk)), dim3(kBlk), 0, st, lv[0], s->pos, sys.row,
                     sys.ap, sys.anb);
  for (int l = 0; l + 1 < s->nlev; l++)
    hipLaunchKernelGGL(k_mg_galerkin<T>, dim3(nb(lv[l + 1].npad + lv[l + 1].nnz, kBlk)), dim3(kBlk),
                       0, st, lv[l], lv[l + 1]);
  hipLaunchKernelGGL(k_cg_init<T>, dim3(R.nblk), dim3(kRedThreads), 0, st, R, sys.row, sys.nbr,
                     s->pos, sys.ap, sys.anb, sys.b, static_cast<const double *>(sys.phi), s->r, rt,
                     s->ctl, s->part, sys.nit);
  MGCHK(hipGetLastError());
  const double *r = s->r, *p = s->p, *q = s->q;
  int *act = &s->ctl->active;
  // Iteration k is queued before the host reads the flag after iteration
  // k-1, so the GPU never waits for the host; an iteration queued after the
  // stop exits at once.
  for (int it = 0; it < sys.nit; it++) {
    MGCALL(vcycle<T>(s, st));
    hipLaunchKernelGGL(k_cg_rz<T>, dim3(R.nblk), dim3(kRedThreads), 0, st, R, r, z, s->pos, s->ctl,
                       s->part);
    hipLaunchKernelGGL(k_cg_p<T>, dim3(nb(ne, kBlk)), dim3(kBlk), 0, st, ne, z, s->pos, s->p,
                       static_cast<const CgCtl *>(s->ctl));
    hipLaunchKernelGGL(k_cg_spmv, dim3(R.nblk), dim3(kRedThreads), 0, st, R, sys.row, sys.nbr,
                       sys.ap, sys.anb, p, s->q, s->ctl, s->part);
    hipLaunchKernelGGL(k_cg_update<T>, dim3(R.nblk), dim3(kRedThreads), 0, st, R, sys.phi, p, q,
                       s->pos, s->r, rt, s->ctl, s->part);
    s->launches += 4;
    MGCHK(hipGetLastError());
    MGCHK(hipMemcpyAsync(&s->hflag[it & 1], act, sizeof(int), hipMemcpyDeviceToHost, st));
    MGCHK(hipEventRecord(s->ev[it & 1], st));
    if (it > 0) {
      MGCHK(hipEventSynchronize(s->ev[(it - 1) & 1]));
      if (!s->hflag[(it - 1) & 1]) break;
    }
  }
  LogLine tmpl{};
  std::memcpy(tmpl.name, sys.name, 8);
  hipLaunchKernelGGL(k_cg_log, dim3(1), dim3(64), 0, st, static_cast<const CgCtl *>(s->ctl),
                     sys.log, sys.nlog, tmpl);
  MGCHK(hipGetLastError());
  return CFDL_OK;
}
}  // namespace

int mgcg_solve(MgCgSolver *s, const MgCgSystem &sys, void *stream) {
  if (!s || sys.ne != s->ne || sys.nbf != s->nbf) {
    set_error("mgcg_solve: system does not match the hierarchy");
    return CFDL_EINVAL;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  return s->fp32 ? solve<float>(s, sys, st) : solve<double>(s, sys, st);
}

// ---------------------------------------------------------------------------
// Grouped solves
// ---------------------------------------------------------------------------
namespace {
// A grouped solve between its phases (host side): the systems, their
// descriptors as uploaded, and the launch shape.
template <typename T>
struct GroupRun {
  std::vector<MgCgSolver *> ss;
  std::vector<MgSlot<T>> h;
  int n = 0, blk = 256, maxtop = 0, maxlev = 0, nitmax = 0;
};
}  // namespace

struct MgGroup {
  int fp32 = 0;            // precision of the current run
  GroupRun<double> rd;
  GroupRun<float> rf;
  void *slots = nullptr;  // device MgSlot<T>[kMaxGroup]
  int *flags = nullptr;   // device active flags
  int *hflags = nullptr;  // pinned, two sets of kMaxGroup
  hipEvent_t ev[2] = {nullptr, nullptr};
  // The composition whose descriptors are on the device, with the solvers'
  // serial numbers: launch shapes come from their host tables (colours, sizes
  // of levels), and a later solver may get a destroyed one's addresses.
  std::vector<char> key;
  int launches = 0;
  ~MgGroup() {
    if (slots) (void)hipFree(slots);
    if (flags) (void)hipFree(flags);
    if (hflags) (void)hipHostFree(hflags);
    for (auto &e : ev)
      if (e) (void)hipEventDestroy(e);
  }
};

int mgcg_group_create(MgGroup **out) {
  std::unique_ptr<MgGroup> g(new MgGroup());
  const size_t bytes = sizeof(MgSlot<double>) > sizeof(MgSlot<float>) ? sizeof(MgSlot<double>)
                                                                       : sizeof(MgSlot<float>);
  MGCHK(hipMalloc(&g->slots, bytes * kMaxGroup));
  MGCHK(hipMalloc(reinterpret_cast<void **>(&g->flags), sizeof(int) * kMaxGroup));
  MGCHK(hipHostMalloc(reinterpret_cast<void **>(&g->hflags), 2 * sizeof(int) * kMaxGroup,
                      hipHostMallocDefault));
  MGCHK(hipEventCreateWithFlags(&g->ev[0], hipEventDisableTiming));
  MGCHK(hipEventCreateWithFlags(&g->ev[1], hipEventDisableTiming));
  *out = g.release();
  return CFDL_OK;
}

void mgcg_group_destroy(MgGroup *g) { delete g; }

namespace {
template <typename T>
GroupRun<T> &run_of(MgGroup *G);
template <>
GroupRun<double> &run_of<double>(MgGroup *G) { return G->rd; }
template <>
GroupRun<float> &run_of<float>(MgGroup *G) { return G->rf; }

// The solve of mgcg_solve for n systems at once, in phases: begin (descriptors
// uploaded when they changed; synchronises then, so it runs outside any graph
// capture), setup (level 0's copies, Galerkin operators, initial residual),
// one iteration at a time (V-cycle and CG step, then the
// systems' active flags copied to a host slot), finish (the log lines).
// Every launch covers the systems that take part in its step; each system
// runs exactly its own sequence of steps (a system with fewer levels or
// colours sits out the launches it has no part in), so its arithmetic is
// that of a solve alone.
template <typename T>
int group_begin(MgGroup *G, MgCgSolver *const *ss, const MgCgSystem *sys, int n, hipStream_t st,
                int blk, int *changed) {
  GroupRun<T> &R = run_of<T>(G);
  R.ss.assign(ss, ss + n);
  R.n = n;
  R.blk = blk;
  R.h.assign(n, MgSlot<T>{});
  std::memset(static_cast<void *>(R.h.data()), 0, sizeof(MgSlot<T>) * n);  // the key compares bytes
  R.maxtop = R.maxlev = R.nitmax = 0;
  for (int k = 0; k < n; k++) {
    MgCgSolver *s = ss[k];
    MgSlot<T> &x = R.h[k];
    x.R = red_of(s->ne);
    x.ne = s->ne;
    x.nit = sys[k].nit;
    x.nlev = s->nlev;
    x.lc = s->lc;
    x.row = sys[k].row;
    x.nbr = sys[k].nbr;
    x.ap = sys[k].ap;
    x.anb = sys[k].anb;
    x.b = sys[k].b;
    x.phi = sys[k].phi;
    x.r = s->r;
    x.p = s->p;
    x.q = s->q;
    x.part = s->part;
    x.pos = s->pos;
    x.rt = host_levels<T>(s)[0].b;
    x.z = host_levels<T>(s)[0].x;
    x.ctl = s->ctl;
    x.lv = dev_levels<T>(s);
    x.log = sys[k].log;
    x.nlog = sys[k].nlog;
    x.serial = s->serial;
    std::memcpy(x.tmpl.name, sys[k].name, 8);
    R.maxtop = std::max(R.maxtop, s->lc < s->nlev ? s->lc : s->nlev - 1);
    R.maxlev = std::max(R.maxlev, s->nlev);
    R.nitmax = std::max(R.nitmax, sys[k].nit);
  }
  // the descriptors go to the device when the composition changes
  const char *kb = reinterpret_cast<const char *>(R.h.data());
  std::vector<char> key(kb, kb + sizeof(MgSlot<T>) * n);
  key.push_back(static_cast<char>(sizeof(T)));
  *changed = key != G->key;
  if (*changed) {
    MGCHK(hipStreamSynchronize(st));
    MGCHK(hipMemcpy(G->slots, R.h.data(), sizeof(MgSlot<T>) * n, hipMemcpyHostToDevice));
    G->key.swap(key);
  }
  G->launches = 0;
  return CFDL_OK;
}

// the launch shapes of a run
template <typename T>
struct GroupShape {
  GroupRun<T> &R;
  GroupMap g{};
  std::vector<int> ids, cnt;
  explicit GroupShape(GroupRun<T> &r) : R(r), ids(r.n), cnt(r.n) {
    for (int k = 0; k < R.n; k++) ids[k] = k;
  }
  // one grouped launch: blocks_of(k) blocks for system k (0 = sits out)
  template <typename F>
  int map(F blocks_of) {
    for (int k = 0; k < R.n; k++) cnt[k] = blocks_of(k);
    return group_map(g, ids.data(), cnt.data(), R.n);
  }
  int top_of(int k) const {
    return R.ss[k]->lc < R.ss[k]->nlev ? R.ss[k]->lc : R.ss[k]->nlev - 1;
  }
};

template <typename T>
int group_setup(MgGroup *G, hipStream_t st) {
  GroupRun<T> &R = run_of<T>(G);
  GroupShape<T> sh(R);
  const MgSlot<T> *S = static_cast<const MgSlot<T> *>(G->slots);
  const int blk = R.blk;
  int nbk = 0;
  nbk = sh.map([&](int k) { return nb(R.ss[k]->ne, blk); });
  hipLaunchKernelGGL(g_mg_copy0<T>, dim3(nbk), dim3(blk), 0, st, sh.g, S);
  G->launches++;
  for (int l = 0; l + 1 < R.maxlev; l++) {
    nbk = sh.map([&](int k) {
      if (l + 1 >= R.ss[k]->nlev) return 0;
      const Lev<T> &C = host_levels<T>(R.ss[k])[l + 1];
      return nb(C.npad + C.nnz, blk);
    });
    if (nbk > 0) {
      hipLaunchKernelGGL(g_mg_galerkin<T>, dim3(nbk), dim3(blk), 0, st, sh.g, S, l);
      G->launches++;
    }
  }
  nbk = sh.map([&](int k) { return R.h[k].R.nblk; });
  hipLaunchKernelGGL(g_cg_init<T>, dim3(nbk), dim3(kRedThreads), 0, st, sh.g, S);
  G->launches++;
  MGCHK(hipGetLastError());
  return CFDL_OK;
}

template <typename T>
int group_iteration(MgGroup *G, hipStream_t st, int slot) {
  GroupRun<T> &R = run_of<T>(G);
  GroupShape<T> sh(R);
  const MgSlot<T> *S = static_cast<const MgSlot<T> *>(G->slots);
  const int n = R.n, blk = R.blk;
  // a sweep of level l (l < 0: the coarsest level of systems without small
  // levels)
  auto sweep = [&](int l, int mode) {
    auto level_of = [&](int k) { return l < 0 ? R.ss[k]->nlev - 1 : l; };
    auto part = [&](int k) { return l < 0 ? R.ss[k]->lc == R.ss[k]->nlev : l < sh.top_of(k); };
    int steps = 0;
    for (int k = 0; k < n; k++)
      if (part(k)) steps = std::max(steps, sweep_steps(host_levels<T>(R.ss[k])[level_of(k)]));
    for (int i = 0; i < steps; i++) {
      const int nbk = sh.map([&](int k) {
        const int lk = level_of(k);
        return part(k) ? sweep_blocks(R.ss[k], lk, host_levels<T>(R.ss[k])[lk], i, mode, blk) : 0;
      });
      if (nbk > 0) {
        hipLaunchKernelGGL(g_mg_sweep<T>, dim3(nbk), dim3(blk), 0, st, sh.g, S, l, i, mode);
        G->launches++;
      }
    }
  };
  int nbk = 0;
  // V-cycle
  for (int l = 0; l < R.maxtop; l++) {
    sweep(l, kFwd0);
    nbk = sh.map([&](int k) { return l < sh.top_of(k) ? nb(R.ss[k]->open[l], blk) : 0; });
    if (nbk > 0) {
      hipLaunchKernelGGL(g_mg_residual<T>, dim3(nbk), dim3(blk), 0, st, sh.g, S, l);
      G->launches++;
    }
    nbk = sh.map([&](int k) {
      return l < sh.top_of(k) ? nb(host_levels<T>(R.ss[k])[l + 1].npad, blk) : 0;
    });
    if (nbk > 0) {
      hipLaunchKernelGGL(g_mg_restrict<T>, dim3(nbk), dim3(blk), 0, st, sh.g, S, l);
      G->launches++;
    }
  }
  nbk = sh.map([&](int k) { return R.ss[k]->lc < R.ss[k]->nlev ? 1 : 0; });
  if (nbk > 0) {
    size_t lds = 0;
    for (int k = 0; k < n; k++) lds = std::max(lds, R.ss[k]->coarse_lds);
    hipLaunchKernelGGL(g_mg_coarse<T>, dim3(nbk), dim3(kCoarseThreads), lds, st, sh.g, S);
    G->launches++;
  }
  bool any_flat = false;
  for (int k = 0; k < n; k++) any_flat = any_flat || R.ss[k]->lc == R.ss[k]->nlev;
  if (any_flat)
    for (int r = 0; r < kCoarseSweeps; r++) {
      sweep(-1, r == 0 ? kFwd0 : kFwd);
      sweep(-1, kBwd);
    }
  for (int l = R.maxtop - 1; l >= 0; l--) {
    nbk = sh.map([&](int k) { return l < sh.top_of(k) ? nb(R.ss[k]->prolonged[l], blk) : 0; });
    if (nbk > 0) {
      hipLaunchKernelGGL(g_mg_prolong<T>, dim3(nbk), dim3(blk), 0, st, sh.g, S, l);
      G->launches++;
    }
    sweep(l, kBwd);
  }
  // CG
  nbk = sh.map([&](int k) { return R.h[k].R.nblk; });
  hipLaunchKernelGGL(g_cg_rz<T>, dim3(nbk), dim3(kRedThreads), 0, st, sh.g, S);
  const GroupMap gR = sh.g;
  nbk = sh.map([&](int k) { return nb(R.ss[k]->ne, blk); });
  hipLaunchKernelGGL(g_cg_p<T>, dim3(nbk), dim3(blk), 0, st, sh.g, S);
  hipLaunchKernelGGL(g_cg_spmv<T>, dim3(gR.b0[gR.n]), dim3(kRedThreads), 0, st, gR, S);
  hipLaunchKernelGGL(g_cg_update<T>, dim3(gR.b0[gR.n]), dim3(kRedThreads), 0, st, gR, S);
  hipLaunchKernelGGL(g_cg_flags<T>, dim3(1), dim3(kMaxGroup), 0, st, n, S, G->flags);
  G->launches += 5;
  MGCHK(hipGetLastError());
  MGCHK(hipMemcpyAsync(G->hflags + slot * kMaxGroup, G->flags, sizeof(int) * n,
                       hipMemcpyDeviceToHost, st));
  return CFDL_OK;
}

template <typename T>
int group_finish(MgGroup *G, hipStream_t st) {
  GroupRun<T> &R = run_of<T>(G);
  const MgSlot<T> *S = static_cast<const MgSlot<T> *>(G->slots);
  hipLaunchKernelGGL(g_cg_log<T>, dim3(1), dim3(kMaxGroup), 0, st, R.n, S);
  G->launches++;
  MGCHK(hipGetLastError());
  for (MgCgSolver *s : R.ss) s->launches = G->launches;
  return CFDL_OK;
}
}  // namespace

int mgcg_group_begin(MgGroup *G, MgCgSolver *const *s, const MgCgSystem *sys, int n, void *stream,
                     int block, int *changed) {
  if (!G || !s || !sys || n < 1 || n > kMaxGroup) {
    set_error("mgcg_solve_group: 1 .. " + std::to_string(kMaxGroup) + " systems");
    return CFDL_EINVAL;
  }
  if (block < 64 || block > 1024 || block % 64 != 0) {
    set_error("mgcg_solve_group: block must be a multiple of 64 in 64 .. 1024");
    return CFDL_EINVAL;
  }
  for (int k = 0; k < n; k++) {
    if (!s[k] || sys[k].ne != s[k]->ne || sys[k].nbf != s[k]->nbf) {
      set_error("mgcg_solve_group: system " + std::to_string(k) + " does not match its hierarchy");
      return CFDL_EINVAL;
    }
    if (s[k]->fp32 != s[0]->fp32) {
      set_error("mgcg_solve_group: the systems of a group share one preconditioner precision");
      return CFDL_EINVAL;
    }
    for (int j = 0; j < k; j++)
      if (s[j] == s[k]) {
        set_error("mgcg_solve_group: a solver appears twice in the group");
        return CFDL_EINVAL;
      }
  }
  int dummy = 0;
  if (!changed) changed = &dummy;
  hipStream_t st = static_cast<hipStream_t>(stream);
  G->fp32 = s[0]->fp32;
  return G->fp32 ? group_begin<float>(G, s, sys, n, st, block, changed)
                 : group_begin<double>(G, s, sys, n, st, block, changed);
}

int mgcg_group_setup(MgGroup *G, void *stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  return G->fp32 ? group_setup<float>(G, st) : group_setup<double>(G, st);
}

int mgcg_group_iteration(MgGroup *G, void *stream, int slot) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  return G->fp32 ? group_iteration<float>(G, st, slot) : group_iteration<double>(G, st, slot);
}

int mgcg_group_finish(MgGroup *G, void *stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  return G->fp32 ? group_finish<float>(G, st) : group_finish<double>(G, st);
}

int mgcg_group_nit(const MgGroup *G) { return G->fp32 ? G->rf.nitmax : G->rd.nitmax; }

bool mgcg_group_any_active(const MgGroup *G, int slot) {
  const int n = G->fp32 ? G->rf.n : G->rd.n;
  const int *f = G->hflags + slot * kMaxGroup;
  for (int k = 0; k < n; k++)
    if (f[k]) return true;
  return false;
}

int mgcg_solve_group(MgGroup *G, MgCgSolver *const *s, const MgCgSystem *sys, int n,
                     void *stream, int block) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  MGCALL(mgcg_group_begin(G, s, sys, n, stream, block, nullptr));
  MGCALL(mgcg_group_setup(G, stream));
  // iteration it is queued before the host reads the flags after it-1
  for (int it = 0; it < mgcg_group_nit(G); it++) {
    MGCALL(mgcg_group_iteration(G, stream, it & 1));
    MGCHK(hipEventRecord(G->ev[it & 1], st));
    if (it > 0) {
      MGCHK(hipEventSynchronize(G->ev[(it - 1) & 1]));
      if (!mgcg_group_any_active(G, (it - 1) & 1)) break;
    }
  }
  return mgcg_group_finish(G, stream);
}

}  // namespace cfdl
