// gf_solve_common.hpp -- definitions shared by the solver translation units:
// launch helpers, the device-resident solver scalars, the workgroup-to-element
// mapping of the 3-D element kernels and declarations of their launchers.
// The 3-D kernels themselves are in gf_k3d.hpp and are compiled once per
// element order in the gf_k3d_n*.hip translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "gf_boxdss.hpp"
#include "gf_internal.hpp"
#include "gf_kernels.hpp"
#include "gf_pen3.hpp"

namespace gfs {

using gf::kThreads;
using gf::Shape;

inline int nblocks(size_t n, int per = kThreads) {
  size_t b = (n + per - 1) / per;
  if (b > 65536) b = 65536;
  return (int)std::max<size_t>(b, 1);
}

// Solver scalars of one system: 0 rho, 2 beta, 3 rnorm, 4 rtol, 6 iter,
// 7 maxit, 8 done, 9 first, 10 volume, 11 n, 12 rho of the previous iteration
// (1 and 5 are not used; without them a kernel's loads of the set are slower:
// 416 iterations on 10x9x6 terrain elements, p = 6, 7.65 ms against 7.48).  On
// the device a system has kCGScal doubles: two such sets (of kCGSet doubles),
// read and written alternately by the apply kernels of consecutive iterations,
// and the step length alpha at kCGAlpha.
enum { S_RHO = 0, S_BETA = 2, S_RNORM, S_RTOL, S_ITER = 6, S_MAXIT, S_DONE, S_FIRST, S_VOL, S_N,
       S_RHOM, S_COUNT };
constexpr int kCGSet = 16, kCGAlpha = 2 * kCGSet, kCGScal = 40;

#define GRID_LOOP(g, n)                                                     \
  for (size_t g = blockIdx.x * (size_t)blockDim.x + threadIdx.x; g < (n); \
       g += (size_t)gridDim.x * blockDim.x)

struct StageArgs {
  const double *uin[3];
  const double *kprev[3];
  double bh;
  double *acc[3];
  const double *accsrc[3];
  double ch;
  double *kout[3];
  const double *D, *W, *edx, *ejac, *imass;
  double nu;
  size_t nelems;
};

// Arguments of the adjoint stage kernel (k_burgers_adj3).
struct Adj3Args {
  const double *u[3], *y[3];
  double *abar[3], *lin[3], *yo[3];
  const double *imass, *W, *edx, *ejac;
  double hc, hb, nu;
  gf::BoxTopo topo;
  size_t nelems, imstride;
};

inline gf::PenD<double> pend_d(gf_mesh *m) {
  gf::PenD<double> p;
  for (int c = 0; c < 3; c++) {
    p.R[c] = m->pDR[c];
    p.C[c] = m->pDC[c];
  }
  return p;
}
inline gf::PenD<float> pend_f(gf_mesh *m) {
  gf::PenD<float> p;
  for (int c = 0; c < 3; c++) {
    p.R[c] = m->pDR32[c];
    p.C[c] = m->pDC32[c];
  }
  return p;
}

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own
// L2).  Grids of the element kernels are a multiple of kXCD workgroups and
// are renumbered so that each XCD walks one contiguous range of elements:
// neighbouring elements, whose shared faces the gather kernels read, then
// run on the same XCD close together in time.
constexpr int kXCD = 8;
inline int xcd_grid(size_t nblocks) { return (int)((nblocks + kXCD - 1) / kXCD * kXCD); }
// rev: each XCD walks its range from the end.
__device__ __forceinline__ size_t xcd_block(bool rev = false) {
  const size_t per = gridDim.x / kXCD, at = blockIdx.x / kXCD;
  return (size_t)(blockIdx.x % kXCD) * per + (rev ? per - 1 - at : at);
}

// Copies the 512 doubles at g (an element, 4 KB) to LDS at l with four
// 16-byte global-to-LDS loads per lane (global_load_lds_dwordx4: lane L's 16
// bytes land at l + 16 L, so l gets g's layout), half the instructions of
// per-column 8-byte loads and no registers holding the data in flight.  l
// must be the same for the whole wave; the compiler waits for the copy before
// the first LDS read after the next barrier.
__device__ __forceinline__ void lds_copy512(const double *__restrict__ g, double *l, int lane) {
#pragma unroll
  for (int q = 0; q < 4; q++)
    __builtin_amdgcn_global_load_lds((const void *)(g + q * 128 + 2 * lane),
                                     (__attribute__((address_space(3))) void *)(l + q * 128), 16,
                                     0, 0);
}

// Grid-stride loop over [0, n) with the blocks renumbered by xcd_block (the
// grid a multiple of kXCD): each XCD walks contiguous ranges.
#define XCD_GRID_LOOP(g, n)                                                 \
  for (size_t g = xcd_block() * blockDim.x + threadIdx.x; g < (n);         \
       g += (size_t)gridDim.x * blockDim.x)

// Thread/element mapping shared by the 3-D element kernels.
template <int N, typename P = gf::Pen3<N>>
struct ColIdx {
  int el, i, j, r;
  size_t e;
  bool active;
  __device__ __forceinline__ ColIdx(size_t nelems, bool rev = false)
      : ColIdx(nelems, rev, (int)threadIdx.x) {}
  __device__ __forceinline__ ColIdx(size_t nelems, bool rev, int tid) {
    using C = P;
    el = tid / C::N2;
    r = tid - el * C::N2;
    i = r % N;
    j = r / N;
    size_t eg = xcd_block(rev) * C::EPB + el;
    active = el < C::EPB && eg < nelems;
    e = active ? eg : (nelems - 1);
  }
};

// Control of a CG iteration, an argument of its kernels.  An iteration is
//   apply   rho, beta, norm and stopping test from the previous update's
//           partial sums; x += alpha w (the previous step), w = z + beta w,
//           q = A w and the partial sums of w.q
//   (DSS    where q is assembled by a pass of its own)
//   update  alpha from the apply's partial sums; r -= alpha DSS(q) and the
//           partial sums of r.z and of the norm
// The scalars are formed in the kernels that use them: every block sums all
// partials of its system in the same order (a few KB from L2), so no
// one-block reduction kernel runs between the two, and the system's first
// block stores the results.  x is advanced in the apply, which reads w
// anyway: 9 passes over the fields an iteration instead of 10.
// Place of a block of a batched mesh: its system s (elements e0 .. e1, blocks
// b0 .. b0 + nb) and its number lb there.
struct CGSegBlock {
  int s, lb, nb, b0;
  int64_t e0, e1;
};

struct CGCtl {
  double *scal;           // kCGScal doubles per system
  const CGSegBlock *blk;  // batched mesh (nseg > 0): nblk blocks
  int nseg, nblk;
  size_t nelems;
  int nbA, nbU;          // blocks of the apply and update kernels (nseg == 0)
  double *partA, *partU; // w.q per apply block; (r.z, norm) per update block
  int par, init;         // set read by this iteration's apply; first iteration
  int stream;            // the vectors exceed the Infinity Cache (see launch_cg_apply3p)
  int normtype;
  double *resid;         // residual history, or null
  double *mirror;        // mapped host memory, kCGSet doubles per system,
  double epoch;          // written when the system is done, S_DONE = epoch
};

struct CGApply3Args {
  CGCtl c;
  const void *r, *dinv;
  // Jacobi table: elements with deq[e] read dtab (one element's values) in
  // place of dinv; null: dinv everywhere
  const void *dtab;
  const unsigned char *deq;
  void *x, *w, *q;
  const void *W, *edx, *ejac, *qf, *mask;
  double p;
  double qs;  // mass-term scalar when qf is NULL (0: no mass term)
  gf::BoxTopo topo;  // with tmask: mask formed from the box faces (mask NULL)
  int tmask;
};

// Member of element e: the s with eoff[s] <= e < eoff[s+1] (binary search
// over the nseg+1 offsets; e past the end maps to the last member).
__device__ __forceinline__ int seg_of(const int64_t *__restrict__ eoff, int nseg, size_t e) {
  int lo = 0, hi = nseg;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if ((size_t)eoff[mid] <= e) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Workgroups of kThreads that loop over `chunks` pieces of work, at most
// `cap`, every one with the same number of pieces or one less.
inline int loop_blocks(size_t chunks, size_t cap) {
  const size_t rounds = std::max<size_t>(1, (chunks + cap - 1) / cap);
  return xcd_grid(std::max<size_t>(1, (chunks + rounds - 1) / rounds));
}

// Element mapping of the 3-D CG kernels: workgroups of kThreads (four waves),
// N^2 threads per element.  WAVE: an element's threads lie in one wave, which
// works EW elements and orders its own LDS accesses, so the workgroup's waves
// run apart; else the workgroup works EPB elements between barriers and loses
// fewer lanes.  A wave where it fills (N = 2, 3, 4, 8), and at N = 7 (49 of 64
// lanes): an iteration at 20^3, p = 6 takes 68 us in FP64 and 41 in FP32
// against 71 and 43 between barriers.  At N = 5 (50 lanes) 24^3 takes 47.6
// against 43.9, at N = 6 (36 lanes) 88 against 62.  Threads without an
// element (lane false) idle: they follow threads of another element through
// the barriers and store nothing, in memory or in LDS.
template <int N>
struct CGShape {
  static constexpr int N2 = N * N;
  static constexpr bool WAVE = 64 / N2 * N2 > 56 || N == 7;
  static constexpr int EW = WAVE ? 64 / N2 : 0;
  static constexpr int EPB = WAVE ? kThreads / 64 * EW : kThreads / N2;
  static constexpr bool FULL = EPB * N2 == kThreads;
  int el, r, i, j;
  bool lane;
  __device__ __forceinline__ CGShape() {
    int t = (int)threadIdx.x, e0 = 0;
    if constexpr (WAVE) {
      e0 = (t >> 6) * EW;
      t &= 63;
    }
    constexpr int ACT = WAVE ? EW * N2 : EPB * N2;
    lane = t < ACT;
    if (!lane) t -= ACT;
    el = t / N2;
    r = t - el * N2;
    el += e0;
    i = r % N;
    j = r / N;
  }
  // lane, a compile-time constant where no thread idles
  __device__ __forceinline__ auto own() const {
    if constexpr (FULL) return std::true_type();
    else return lane;
  }
};

#define GF_DISPATCH_N3(NV, FN, ...)                   \
  [&]() -> int {                                      \
    switch (NV) {                                     \
      case 2: return FN<2>(__VA_ARGS__);              \
      case 3: return FN<3>(__VA_ARGS__);              \
      case 4: return FN<4>(__VA_ARGS__);              \
      case 5: return FN<5>(__VA_ARGS__);              \
      case 6: return FN<6>(__VA_ARGS__);              \
      case 7: return FN<7>(__VA_ARGS__);              \
      case 8: return FN<8>(__VA_ARGS__);              \
      case 9: return FN<9>(__VA_ARGS__);              \
      case 10: return FN<10>(__VA_ARGS__);            \
      default: return GF_ERR_UNSUPPORTED;             \
    }                                                 \
  }()

constexpr int kUpdBlocks = 1024;

template <typename A>
__device__ __forceinline__ double finish_norm(int normtype, double v, const A &scal) {
  switch (normtype) {
    case GF_NORM_INF: return v;
    case GF_NORM_EUC: return sqrt(v / scal[S_N]);
    case GF_NORM_L2: return sqrt(v / scal[S_VOL]);
    case GF_NORM_L1: return v / scal[S_VOL];
    default: return sqrt(v);
  }
}

// System of a block and the block's place in it (b: the block, nb: blocks of
// a single system).  ok is false for a padding block of a batched mesh.
struct CGBlock {
  int s, lb, nb, b0;
  size_t e0, e1;
  double *st;
  bool ok;
  __device__ __forceinline__ CGBlock(const CGCtl &c, int b, int nb_) {
    s = 0;
    lb = b;
    nb = nb_;
    b0 = 0;
    e0 = 0;
    e1 = c.nelems;
    ok = true;
    if (c.nseg > 0) {
      ok = b < c.nblk;
      const CGSegBlock v = c.blk[ok ? b : 0];
      s = v.s;
      lb = v.lb;
      nb = v.nb;
      b0 = v.b0;
      e0 = (size_t)v.e0;
      e1 = (size_t)v.e1;
    }
    st = c.scal + (size_t)s * kCGScal;
  }
};

// A block's walk over the chunks (of CH elements) of its system.  A single
// system's chunks are split in one contiguous range per XCD, over which the
// XCD's blocks move together; reversed, the walk runs from the range's end:
// the update kernel, walking backwards, starts with the elements the apply
// kernel left in the caches last, and the next apply with those the update
// left.
struct CGWalk {
  int64_t c, step, lo, hi;
  __device__ __forceinline__ CGWalk(const CGCtl &ctl, const CGBlock &b, int CH, bool rev) {
    const int64_t n = (int64_t)((b.e1 - b.e0 + CH - 1) / CH);
    int64_t at = b.lb, per = b.nb;
    lo = 0;
    hi = n;
    if (ctl.nseg == 0) {
      const int64_t x = blockIdx.x % kXCD;
      lo = x * n / kXCD;
      hi = (x + 1) * n / kXCD;
      at = blockIdx.x / kXCD;
      per = gridDim.x / kXCD;
    }
    c = rev ? hi - 1 - at : lo + at;
    step = rev ? -per : per;
  }
  __device__ __forceinline__ bool in() const { return c >= lo && c < hi; }
  __device__ __forceinline__ void next() { c += step; }
};

// Sums (or, for w with wmax, the maximum) over the block of v and w, to
// every thread.
__device__ __forceinline__ void block_all2(double &v, double &w, bool wmax, double *sred) {
  v = gf::wave_sum(v);
  w = wmax ? gf::wave_max(w) : gf::wave_sum(w);
  const int wid = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sred[2 * wid] = v;
    sred[2 * wid + 1] = w;
  }
  __syncthreads();
  v = sred[0];
  w = sred[1];
  for (int k = 1; k < (int)(blockDim.x >> 6); k++) {
    v += sred[2 * k];
    w = wmax ? fmax(w, sred[2 * k + 1]) : w + sred[2 * k + 1];
  }
  __syncthreads();  // sred is free again
}

// Head of an apply kernel: the scalars of this iteration (the recurrences and
// stopping rule of gcg.ipp:297-335: continue while iter < maxit and
// rnorm > rtol) from the previous update's partials.  The constructor issues
// every load (a kernel starts with cold caches: one trip to memory, in which
// the caller's first element loads travel too), finish() uses them.
// run false: the system was done before; xonly: it is done now, and only
// x += alpha w is left.
struct CGHead {
  static constexpr int NP = 4;  // partial pairs per thread loaded ahead
  double P[S_COUNT], al;
  double2 pv[NP];
  const double2 *pu;
  int n;
  double beta, alpha;
  bool run, first, xonly;
  __device__ __forceinline__ CGHead(const CGCtl &c, const CGBlock &b) {
    const double *p = b.st + kCGSet * c.par;
#pragma unroll
    for (int k = 0; k < S_COUNT; k++) P[k] = p[k];
    al = b.st[kCGAlpha];
    pu = (const double2 *)c.partU + b.b0;
    n = c.init ? 0 : (c.nseg > 0 ? b.nb : c.nbU);
#pragma unroll
    for (int k = 0; k < NP; k++) {
      const int i = threadIdx.x + k * kThreads;
      pv[k] = i < n ? pu[i] : make_double2(0.0, 0.0);
    }
  }
  __device__ __forceinline__ void finish(const CGCtl &c, const CGBlock &b, double *sred) {
    double *Q = b.st + kCGSet * (c.par ^ 1);
    const bool lead = b.lb == 0 && threadIdx.x == 0;
    double *mir = c.mirror ? c.mirror + (size_t)b.s * kCGSet : nullptr;
    beta = alpha = 0.0;
    first = xonly = false;
    run = P[S_DONE] == 0.0;
    if (run && c.init) {
      beta = P[S_BETA];
      first = P[S_FIRST] != 0.0;
    }
    if (!run || c.init) {
      if (lead) {
#pragma unroll
        for (int k = 0; k < S_COUNT; k++) Q[k] = P[k];
        if (!run && mir) mirror(mir, c.epoch);
      }
      return;
    }
    const bool inf = c.normtype == GF_NORM_INF;
    double rho = 0.0, nr = 0.0;
    for (int i = threadIdx.x + NP * kThreads; i < n; i += kThreads) {
      const double2 t = pu[i];
      rho += t.x;
      nr = inf ? fmax(nr, t.y) : nr + t.y;
    }
#pragma unroll
    for (int k = 0; k < NP; k++) {
      rho += pv[k].x;
      nr = inf ? fmax(nr, pv[k].y) : nr + pv[k].y;
    }
    block_all2(rho, nr, inf, sred);
    beta = rho / P[S_RHO];
    alpha = al;
    const double rn = finish_norm(c.normtype, nr, P);
    const int it = (int)P[S_ITER] + 1;
    xonly = !(it < (int)P[S_MAXIT] && rn > P[S_RTOL]);
    if (lead) {
      P[S_RHOM] = P[S_RHO];
      P[S_RHO] = rho;
      P[S_BETA] = beta;
      P[S_RNORM] = rn;
      P[S_ITER] = it;
      P[S_FIRST] = 0.0;
      P[S_DONE] = xonly ? 1.0 : 0.0;
#pragma unroll
      for (int k = 0; k < S_COUNT; k++) Q[k] = P[k];
      if (c.resid) c.resid[it - 1] = rn;
      if (xonly && mir) mirror(mir, c.epoch);
    }
  }
  __device__ __forceinline__ void mirror(double *mir, double epoch) const {
#pragma unroll
    for (int k = 0; k < S_COUNT; k++)
      if (k != S_DONE) mir[k] = P[k];
    mir[S_DONE] = epoch;
  }
};

// Head of an update kernel: alpha = rho / (w.q) from the apply's partials;
// the loads in the constructor, as above.
struct CGAlphaHead {
  static constexpr int NP = 4;
  double done, rho, pv[NP];
  const double *pa;
  int n;
  __device__ __forceinline__ CGAlphaHead(const CGCtl &c, const CGBlock &b) {
    const double *Q = b.st + kCGSet * (c.par ^ 1);
    done = Q[S_DONE];
    rho = Q[S_RHO];
    pa = c.partA + b.b0;
    n = c.nseg > 0 ? b.nb : c.nbA;
#pragma unroll
    for (int k = 0; k < NP; k++) {
      const int i = threadIdx.x + k * kThreads;
      pv[k] = i < n ? pa[i] : 0.0;
    }
  }
  // false when the system is done
  __device__ __forceinline__ bool finish(const CGBlock &b, double *sred, double &alpha) {
    if (done != 0.0) return false;
    double v = 0.0, w = 0.0;
    for (int i = threadIdx.x + NP * kThreads; i < n; i += kThreads) v += pa[i];
#pragma unroll
    for (int k = 0; k < NP; k++) v += pv[k];
    block_all2(v, w, false, sred);
    alpha = rho / v;
    if (b.lb == 0 && threadIdx.x == 0) b.st[kCGAlpha] = alpha;
    return true;
  }
};

// One node's contributions to r.z and to the norm.
template <int NORM>
__device__ __forceinline__ void cg_accum(double rv, double z, double im, const double *mass,
                                         size_t g, double &rho, double &nrm) {
  rho += rv * z * im;
  if (NORM == GF_NORM_INF) nrm = fmax(nrm, fabs(rv));
  else if (NORM == GF_NORM_EUC) nrm += rv * rv;
  else if (NORM == GF_NORM_L2) nrm += mass[g] * rv * rv;
  else if (NORM == GF_NORM_L1) nrm += mass[g] * fabs(rv);
  else nrm += rv * rv * im;
}

template <typename T>
struct CGVecs {
  T *x, *r, *w, *q;
  const T *dinv, *mask, *qf;
  const T *dtab;               // Jacobi table (CGApply3Args), or null
  const unsigned char *deq;
  const gf::BoxTopo *topos;    // boxes of a batched mesh's systems, or null
  const T *imult;  // 1/multiplicity in the recurrence precision (exact in FP64)
  const void *D, *W, *edx, *ejac;
  const void *G[6];  // T node metrics and lumped mass (meshes with node metrics)
  const void *mass;
  double p;
  double qs;  // mass-term scalar when qf is NULL
};




// Launchers of the 3-D element kernels (gf_k3d.hpp), one instantiation per
// element order N = 2..10 in the gf_k3d_n*.hip translation units.
template <int N>
int launch_stage3p(gf_mesh *m, const StageArgs &a);
template <int N>
int launch_advect3p(gf_mesh *m, const double *p, const double *const *v, double *po);
template <int N>
int launch_grad3p(gf_mesh *m, const double *p, double *const *o, const double *edx);
template <int N>
int launch_stage3b(gf_mesh *m, double *const *uin, double *const *kp, double *const *acc,
                   double *const *kout, double bh, double ca, double cb, double nu, int in,
                   int accm);
template <int N>
int launch_rk_out_box(gf_mesh *m, double *const *u, double *const *acc);
template <int N>
int launch_adj3(gf_mesh *m, const Adj3Args &a, int mode);
template <int N>
int launch_stage_input(gf_mesh *m, const double *const *u, double *const *k, double *const *v,
                       double bh, int cont);
template <int N>
int helm3c_d(gf_mesh *m, double p, const double *pf, const double *qf, double qs, const double *u,
             double *uo);
template <int N>
int helm3c_f(gf_mesh *m, float p, const float *qf, float qs, const float *u, float *uo);
template <int N>
int cgapply3c_d(gf_mesh *m, const CGApply3Args &a);
template <int N>
int cgapply3c_f(gf_mesh *m, const CGApply3Args &a);
template <typename T, int NORM, int N>
int launch_update_box_n(gf_mesh *m, const CGCtl &c, const CGVecs<T> &v);
// Blocks of the 3-D apply and box update kernels on a mesh of N points.
template <typename T, int N>
int cg_blocks3(size_t nelems);

}  // namespace gfs
