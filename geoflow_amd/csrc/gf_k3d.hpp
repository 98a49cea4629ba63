// gf_k3d.hpp -- 3-D regular-element kernels (pencil form, gf_pen3.hpp) and
// their launchers: Helmholtz apply, CG apply and update, Burgers RK stages
// and the structured-box RK output.  Included by the gf_k3d_n*.hip
// translation units, each of which instantiates the launchers for some
// element orders (GF_K3D_INSTANTIATE).
#pragma once

#include <type_traits>

#include "gf_solve_common.hpp"

namespace gfs {

// ---------------------------------------------------------------------------
// Pencil-form 3-D kernels (see gf_pen3.hpp): Helmholtz apply and CG apply.
// ---------------------------------------------------------------------------
template <int N, typename T>
__global__ __launch_bounds__(gf::Pen3<N>::THREADS) void k_helm3p(
    const T *__restrict__ u, T *__restrict__ uo, gf::PenD<T> D, const T *__restrict__ W,
    const T *__restrict__ edx, const T *__restrict__ ejac, T p, const T *__restrict__ pf,
    const T *__restrict__ qf, T qs, size_t nelems) {
  using S = gf::Pen3<N>;
  __shared__ T su[S::EPB][S::SZ], sd[S::EPB][S::SZ];
  ColIdx<N> t(nelems);
  const size_t col = t.e * S::NN + t.r;
  T ru[N];
#pragma unroll
  for (int k = 0; k < N; k++) ru[k] = u[col + k * S::N2];
  const T jac = ejac[t.e];
  const T f0 = edx[t.e * 3], f1 = edx[t.e * 3 + 1], f2 = edx[t.e * 3 + 2];
  auto post = [&](int k, T Lu, T M, T, T) {
    if (!t.active) return;
    T acc = Lu;
    if (!pf && p != T(1)) acc *= p;
    if (qf) {
      T tq = M * ru[k];
      tq *= qf[col + k * S::N2];
      acc += tq;
    } else if (qs != T(0)) {
      T tq = M * ru[k];
      if (qs != T(1)) tq *= qs;
      acc += tq;
    }
    uo[col + k * S::N2] = acc;
  };
  gf::pen_op3<N, T, false>(ru, su[t.el], sd[t.el], (T *)nullptr, D, W, t.i, t.j, W[t.i], W[t.j],
                           jac, f0 * f0,
                           f1 * f1, f2 * f2, pf ? pf + t.e * S::NN : (const T *)nullptr,
                           gf::NoPenCB(), gf::NoPenCB(), gf::NoPenCB(), post);
}

// CG apply (see CGCtl), 3-D pencil form: x += alpha w, w = z + beta w, then
// q = A w on the element (unassembled) and the partial sums of w.q.  Because
// w is continuous and zero where masked, sum_j w_j (DSS q)_j imult_j equals
// sum_j w_j q_j over local nodes, so the dot product of gcg.ipp:307-308 is
// formed before the assembly; the Dirichlet mask is applied to q here (it is
// constant over each coincidence group, so DSS(q) mask = DSS(q mask)).
// NT: x and w, which this kernel alone reads and writes, bypass the caches
// (see launch_cg_apply3p).
template <int N, typename T, bool NT>
__global__ __launch_bounds__(kThreads) void k_cg_apply3p(CGApply3Args a) {
  using S = gf::Pen3<N>;
  using C = CGShape<N>;
  __shared__ T sl[C::EPB][2][S::SZ];
  __shared__ double sred[2 * (kThreads / 64)];
  const CGBlock b(a.c, (int)xcd_block(), a.c.nbA);
  if (!b.ok) return;
  const T *__restrict__ r = (const T *)a.r, *__restrict__ dinv = (const T *)a.dinv;
  const T *__restrict__ dtab = (const T *)a.dtab, *__restrict__ W = (const T *)a.W;
  const T *__restrict__ edx = (const T *)a.edx, *__restrict__ ejac = (const T *)a.ejac;
  const T *__restrict__ qf = (const T *)a.qf, *__restrict__ mask = (const T *)a.mask;
  T *__restrict__ x = (T *)a.x, *__restrict__ w = (T *)a.w, *__restrict__ qv = (T *)a.q;
  const C t;
  const T p = (T)a.p, qs = (T)a.qs;
  CGHead h(a.c, b);
  T rv[N], dv[N], wv[N], xv[N], jac, f0, f1, f2;
  size_t e, col;
  bool act;
  // the element of a chunk: all its loads; the Jacobi values from the table
  // where the element's equal it
  auto load = [&](int64_t c) {
    const size_t eg = b.e0 + (size_t)c * C::EPB + t.el;
    act = t.own() && eg < b.e1;
    e = eg < b.e1 ? eg : b.e1 - 1;
    col = e * S::NN + t.r;
    const T *dsrc = dinv ? ((dtab && a.deq[e]) ? dtab + t.r : dinv + col) : nullptr;
#pragma unroll
    for (int q = 0; q < N; q++) {
      const size_t g = col + q * S::N2;
      rv[q] = r[g];
      wv[q] = NT ? __builtin_nontemporal_load(w + g) : w[g];
      xv[q] = NT ? __builtin_nontemporal_load(x + g) : x[g];
    }
#pragma unroll
    for (int q = 0; q < N; q++) dv[q] = dsrc ? dsrc[q * S::N2] : T(1);
    jac = ejac[e];
    f0 = edx[e * 3];
    f1 = edx[e * 3 + 1];
    f2 = edx[e * 3 + 2];
  };
  CGWalk k(a.c, b, C::EPB, false);
  if (k.in()) load(k.c);
  const T wi = W[t.i], wj = W[t.j];
  h.finish(a.c, b, sred);
  if (!h.run) return;
  const T beta = (T)h.beta, alpha = (T)h.alpha;
  double dot = 0.0;
  while (k.in()) {
    T ru[N];
    const size_t ce = e, cc = col;
    const bool ca = act;
    const T cj = jac, c0 = f0 * f0, c1 = f1 * f1, c2 = f2 * f2;
#pragma unroll
    for (int q = 0; q < N; q++) {
      const T z = dinv ? dv[q] * rv[q] : rv[q];
      ru[q] = h.first ? z : beta * wv[q] + z;
    }
    if (ca) {
#pragma unroll
      for (int q = 0; q < N; q++) {
        const size_t g = cc + q * S::N2;
        const T xn = xv[q] + alpha * wv[q];
        if (!a.c.init) {
          if (NT) __builtin_nontemporal_store(xn, x + g);
          else x[g] = xn;
        }
        if (!h.xonly) {
          if (NT) __builtin_nontemporal_store(ru[q], w + g);
          else w[g] = ru[q];
        }
      }
    }
    k.next();
    if (k.in()) load(k.c);  // in flight while this element is worked
    if (h.xonly) continue;
    int ec[3] = {0, 0, 0};
    if (a.tmask) gf::box_elem_coords(a.topo, ce, ec);
    auto post = [&](int q, T Lu, T M, T, T) {
      if (!ca) return;
      const size_t g = cc + q * S::N2;
      T acc = Lu;
      if (p != T(1)) acc *= p;
      if (qf) {
        T tq = M * ru[q];
        tq *= qf[g];
        acc += tq;
      } else if (qs != T(0)) {
        T tq = M * ru[q];
        if (qs != T(1)) tq *= qs;
        acc += tq;
      }
      if (mask) acc *= mask[g];
      else if (a.tmask && gf::box_masked(a.topo, N, ec, t.i, t.j, q)) acc *= T(0);
      qv[g] = acc;
      dot += (double)ru[q] * (double)acc;
    };
    gf::pen_op3<N, T, false, C::WAVE>(ru, sl[t.el][0], sl[t.el][1], (T *)nullptr, gf::PenD<T>(), W,
                                      t.i, t.j, wi, wj, cj, c0, c1, c2, (const T *)nullptr,
                                      gf::NoPenCB(), gf::NoPenCB(), gf::NoPenCB(), post, t.own());
  }
  if (h.xonly) return;
  const double bs = gf::block_reduce<false>(dot, sred);
  if (threadIdx.x == 0) a.c.partA[b.b0 + b.lb] = bs;
}

// Fused Burgers stage, 3-D pencil form (see k_burgers_stage for the contract).
// The x- and y-derivative factors of the advection term are carried to the
// column owner through LDS, so every node's advection is summed in the
// reference order ((ux rx) u0 + (uy ry) u1) + (uz rz) u2 (gadvect.ipp:58-100).
template <int N>
__global__ __launch_bounds__(gf::Pen3<N>::THREADS) __attribute__((amdgpu_waves_per_eu(N <= 8 ? 3 : 1)))
void k_burgers_stage3p(
    StageArgs a, gf::PenD<double> Dp) {
  using S = gf::Pen3<N>;
  __shared__ double su[S::EPB][S::SZ], sd[S::EPB][S::SZ], sx[S::EPB][S::SZ];
  ColIdx<N> t(a.nelems);
  const size_t col = t.e * S::NN + t.r;
  // the inverse mass of the column, read once for all components
  double im[N];
#pragma unroll
  for (int k = 0; k < N; k++) im[k] = a.imass[col + k * S::N2];
  double ru[3][N];
#pragma unroll
  for (int c = 0; c < 3; c++) {
#pragma unroll
    for (int k = 0; k < N; k++) {
      const size_t g = col + k * S::N2;
      const double ui = a.uin[c][g];
      double v = ui;
      if (a.kprev[c]) {
        const double kp = a.kprev[c][g];
        v = ui + a.bh * kp;
        if (a.acc[c] && t.active) a.acc[c][g] = a.accsrc[c][g] + kp * a.ch;
      }
      ru[c][k] = v;
    }
  }
  const double jac = a.ejac[t.e];
  const double wa = a.W[t.i], wb = a.W[t.j];
  const double rx = a.edx[t.e * 3], ry = a.edx[t.e * 3 + 1], rz = a.edx[t.e * 3 + 2];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    // the z pass's derivatives, kept for the advection term
    double uzs[N];
    auto zcb = [&](int k, double uz, double) { uzs[k] = uz; };
    auto xcb = [&](int, double ux, double) { return ux * rx; };
    auto ycb = [&](int, double uy, double) { return uy * ry; };
    double *kout = a.kout[c];
    auto post = [&](int k, double L, double M, double hx, double hy) {
      if (!t.active) return;
      const size_t g = col + k * S::N2;
      const double uz = uzs[k];
      double po = hx * ru[0][k];
      po += hy * ru[1][k];
      po += (uz * rz) * ru[2][k];
      const double adv = po * M;
      if (a.nu != 1.0) L *= a.nu;
      const double urhs = -1.0 * L + -1.0 * adv;
      kout[g] = im[k] * urhs;
    };
    gf::pen_op3<N, double, true>(ru[c], su[t.el], sd[t.el], sx[t.el], Dp, a.W, t.i, t.j, wa, wb, jac,
                                 rx * rx, ry * ry, rz * rz, (const double *)nullptr, xcb, ycb, zcb,
                                 post);
    __syncthreads();  // the next component reuses the LDS buffers
  }
}

// First derivatives of a field on regular 3-D elements in one pass, the
// element in the pencil layout of pen_op3 (z derivative in the column's
// registers, x and y through LDS):
//   ADV 0  o0, o1, o2 = d_x p, d_y p, d_z p (GMTK::grad, gmtk.ipp:2883-2892;
//          edx NULL: reference-space derivatives, compute_grefderivs)
//   ADV 1  o0 = M (((d_x p) v0 + (d_y p) v1) + (d_z p) v2), GAdvect::apply
//          (gadvect.ipp:57-99)
//   ADV 2  the same, where a velocity component may be missing (NULL): its term
//          is left out, for its derivative may be infinite or NaN (a form of its
//          own: with the tests in every call the operators of 21x17x13, p = 5
//          took 40.6 us together against 39.3)
// Memory bound: four fields for the gradient, five for the advection (the
// composed advection moved 23).  At 24^3, p = 7: gradient 34 us against 43 of
// the LDS form k_grad, advection 41.5 us (6.8 TB/s) against 242 composed; at
// 21x17x13, p = 5: 8.1 against 9.7 us and 8.5 against 51 us.
template <int N, int ADV>
__global__ __launch_bounds__(gf::Pen3<N>::THREADS) void k_grad3p(
    const double *__restrict__ p, const double *__restrict__ v0, const double *__restrict__ v1,
    const double *__restrict__ v2, double *__restrict__ o0, double *__restrict__ o1,
    double *__restrict__ o2, const double *__restrict__ W, const double *__restrict__ edx,
    const double *__restrict__ ejac, size_t nelems) {
  using S = gf::Pen3<N>;
  constexpr int NV = ADV ? N : 1;
  const bool h0 = ADV != 2 || v0, h1 = ADV != 2 || v1, h2 = ADV != 2 || v2;
  __shared__ double su[S::EPB][S::SZ], sd[S::EPB][S::SZ];
  ColIdx<N> t(nelems);
  const size_t col = t.e * S::NN + t.r;
  double rp[N], vx[NV], vy[NV], vz[NV];
#pragma unroll
  for (int k = 0; k < N; k++) rp[k] = p[col + k * S::N2];
  // the velocities' loads are in flight while p is differentiated
  if constexpr (ADV != 0) {
#pragma unroll
    for (int k = 0; k < N; k++) {
      const size_t g = col + k * S::N2;
      vx[k] = h0 ? v0[g] : 0.0;
      vy[k] = h1 ? v1[g] : 0.0;
      vz[k] = h2 ? v2[g] : 0.0;
    }
  }
  const double rx = edx ? edx[t.e * 3] : 1.0, ry = edx ? edx[t.e * 3 + 1] : 1.0,
               rz = edx ? edx[t.e * 3 + 2] : 1.0;
  double *u = su[t.el], *d = sd[t.el];
#pragma unroll
  for (int k = 0; k < N; k++) u[S::at(t.i, t.j, k)] = rp[k];
  double dz[N], x[N], y[N];
  gf::gll_apply<N, false>(rp, dz);
  __syncthreads();
  // x pencil (j, k) = (t.i, t.j) to sd, y pencil (i, k) back into su
#pragma unroll
  for (int m = 0; m < N; m++) x[m] = u[S::at(m, t.i, t.j)];
  gf::gll_apply<N, false>(x, y);
#pragma unroll
  for (int m = 0; m < N; m++) d[S::at(m, t.i, t.j)] = y[m];
#pragma unroll
  for (int m = 0; m < N; m++) x[m] = u[S::at(t.i, m, t.j)];
  gf::gll_apply<N, false>(x, y);
  __syncthreads();
#pragma unroll
  for (int m = 0; m < N; m++) u[S::at(t.i, m, t.j)] = y[m];
  __syncthreads();
  if (!t.active) return;
  if constexpr (ADV != 0) {
    const double jac = ejac[t.e], wi = W[t.i], wj = W[t.j];
#pragma unroll
    for (int k = 0; k < N; k++) {
      const int q = S::at(t.i, t.j, k);
      double a = h0 ? (d[q] * rx) * vx[k] : 0.0;
      if (h1) a += (u[q] * ry) * vy[k];
      if (h2) a += (dz[k] * rz) * vz[k];
      o0[col + k * S::N2] = a * (((W[k] * wj) * wi) * jac);
    }
  } else {
#pragma unroll
    for (int k = 0; k < N; k++) {
      const int q = S::at(t.i, t.j, k);
      const size_t g = col + k * S::N2;
      o0[g] = d[q] * rx;
      o1[g] = u[q] * ry;
      o2[g] = dz[k] * rz;
    }
  }
}

template <int N>
int launch_advect3p(gf_mesh *m, const double *p, const double *const *v, double *po) {
  using S = gf::Pen3<N>;
  const int nb = xcd_grid((m->nelems + S::EPB - 1) / S::EPB);
  auto *k = v[0] && v[1] && v[2] ? k_grad3p<N, 1> : k_grad3p<N, 2>;
  hipLaunchKernelGGL(k, dim3(nb), dim3(S::THREADS), 0, m->ctx->stream, p, v[0], v[1], v[2], po,
                     (double *)nullptr, (double *)nullptr, m->W[0], m->edx, m->ejac, m->nelems);
  GF_LAUNCH_CHECK(m->ctx);
  return GF_OK;
}
template <int N>
int launch_grad3p(gf_mesh *m, const double *p, double *const *o, const double *edx) {
  using S = gf::Pen3<N>;
  const int nb = xcd_grid((m->nelems + S::EPB - 1) / S::EPB);
  hipLaunchKernelGGL((k_grad3p<N, 0>), dim3(nb), dim3(S::THREADS), 0, m->ctx->stream, p,
                     (const double *)nullptr, (const double *)nullptr, (const double *)nullptr, o[0],
                     o[1], o[2], m->W[0], edx, m->ejac, m->nelems);
  GF_LAUNCH_CHECK(m->ctx);
  return GF_OK;
}

template <int N>
int launch_stage3p(gf_mesh *m, const StageArgs &a) {
  using S = gf::Pen3<N>;
  int nb = xcd_grid((m->nelems + S::EPB - 1) / S::EPB);
  hipLaunchKernelGGL((k_burgers_stage3p<N>), dim3(nb), dim3(S::THREADS), 0, m->ctx->stream, a,
                     pend_d(m));
  GF_LAUNCH_CHECK(m->ctx);
  return GF_OK;
}

// ---------------------------------------------------------------------------
// Burgers RK on a structured box (mesh->has_box): the GGFX Smooth S of the
// stage derivatives, of the final-stage input and of the step output is
// formed by gather in the kernels that consume them (gf_boxdss.hpp) instead
// of separate DSS passes.  Stage derivatives are stored unsmoothed.
//
// S is linear, so step_b's output S(uin + sum_s c_s h S(K_s))
// (gexrk_stepper.ipp:251-341) is S(uin + sum_s c_s h K_s) with the
// unsmoothed own K_s, and one gather at the end serves the whole sum.  A
// stage has its own K_s in registers and the previous one in its halo, so
// the accumulator is touched in every second stage only.
//
// Copies of a node differ in the accumulator, so its Smooth rounds where
// step_b's, of equal copies, is exact.  RK4 has no more error for it: four
// additions to the state in either order (rms against extended precision, 4
// steps at 4x3x3, p = 7: 1.67e-16 of the field, 1.75e-16 in step_b's order).  At
// orders 2 and 3, with two additions, it would have (1.31e-16 against 1.25e-16): they
// accumulate the increments alone (ACC 5) and add the state once, in the last
// stage (ACC 2 and 6: 1.09e-16).  It is read once more for that: at 32^3, p = 7
// RK2 652 -> 676 us a step, RK3 1102 -> 1115 (RK4 that way 1415 -> 1438).  A Smooth
// corrected to one rounding instead left 1.28e-16 and cost 2-4 % at all sizes.
//   IN  stage input
//     0  v = uin                        (first stage from a state)
//     1  v = uin + bh S(kp)
//     2  v = S(uin + bh S(kp))          (step_b's smoothed final-stage input,
//                                        for a state that may be discontinuous)
//     3  v = S(kp), kp the finished accumulator of the previous step: the
//        step output, stored to `acc` (the state), is this stage's input
//   ACC  accumulation after the operator
//     0  none                           K -> kout
//     1  acc = uin + ca kp + cb K       K -> kout
//     2  acc = uin + (ca kp + cb K)     (last stage: K is not stored)
//     3  acc = acc + ca kp + cb K       (last stage)
//     4  acc = v                        K -> kout  (stage states of the adjoint)
//     5  acc = ca kp                    K -> kout
//     6  acc = uin + (acc + cb K)       (last stage)
//        (RK3, whose second stage has no weight)
//   SP  a third of the workgroup's threads to each component, which exchange
//       the stage input through LDS; else a thread does all three in turn.
//       The same operations (stage_split_max says which runs)
// Group sums are pairwise (x, then y, then z), exact for equal members of
// groups of 2, 4 and 8, so S leaves a continuous state as it is and IN 1 and
// IN 2 agree bit for bit on it.
//
// Stages that do not accumulate (every second one of RK4) walk the elements
// backwards and start with what the stage before left in the Infinity Cache
// (32^3, p = 5 817 -> 791 us a step, p = 7 1402 -> 1389).
//
// Bound by memory: at 32^3, p = 7 an RK4 step moves 42 fields of 134 MB; the
// form whose every stage smoothed into the accumulator moved 54 and gathered
// uin too in the last one.  Stages (IN, ACC) = (3,0) 346, (1,1) 420, (1,0)
// 312, (1,3) 373 us, 3.5-4.3 TB/s where copies beyond the Infinity Cache have
// 4.6-5.3; before, 392 + 543 + 459 + 601 us.
// ---------------------------------------------------------------------------
template <int N, int IN, int ACC, bool SP>
__global__ __launch_bounds__((gf::PenStage<N, SP>::THREADS)) __attribute__((amdgpu_waves_per_eu(N <= 8 ? 2 : 1)))
void k_burgers_stage3b(
    const double *__restrict__ ui0, const double *__restrict__ ui1, const double *__restrict__ ui2,
    const double *__restrict__ kp0, const double *__restrict__ kp1, const double *__restrict__ kp2,
    double *ac0, double *ac1, double *ac2, double *__restrict__ ko0, double *__restrict__ ko1,
    double *__restrict__ ko2, const double *__restrict__ imass, const double *__restrict__ W,
    const double *__restrict__ edx, const double *__restrict__ ejac, gf::PenD<double> Dp,
    double bh, double ca, double cb, double nu, gf::BoxTopo topo, size_t nelems, size_t imstride) {
  using S = gf::PenStage<N, SP>;
  using H = gf::Halo<N>;
  constexpr bool KP = IN != 0, GU = IN == 2, UIN = IN != 3;
  constexpr bool LAST = ACC == 2 || ACC == 3 || ACC == 6;
  static_assert(KP || ACC == 0, "the first stage accumulates nothing");
  static_assert(IN != 3 || ACC == 0, "an output stage is a first stage");
  // N = 8: an element is one wave and its own values go straight to LDS
  // (lds_copy512), behind kp's halo; else they pass through registers
  constexpr bool L8 = N == 8 && !SP;
  constexpr int UOFF = H::SIZE, AOFF = UOFF + 512;
  constexpr int HL = !KP ? 0
                         : (GU ? 2 * H::SIZE
                               : H::SIZE + (L8 && UIN ? 512 : 0)) + (L8 && ACC == 3 ? 512 : 0);
  // per element: the halos, then (the same memory) the three element buffers
  constexpr int NSL = HL > 3 * S::SZ ? HL : 3 * S::SZ;
  constexpr int NC = SP ? 3 : 1, TPC = S::EPB * S::N2;
  __shared__ double sl[NC * S::EPB * NSL];
  const double *uin[3] = {ui0, ui1, ui2};
  const double *kp[3] = {kp0, kp1, kp2};
  double *acc[3] = {ac0, ac1, ac2};
  double *kout[3] = {ko0, ko1, ko2};
  const int cs = SP ? (int)threadIdx.x / TPC : 0;
  ColIdx<N, S> t(nelems, ACC == 0, SP ? (int)threadIdx.x - cs * TPC : (int)threadIdx.x);
  const size_t col = t.e * S::NN + t.r;
  double *hk = sl + (cs * S::EPB + t.el) * NSL;
  double im[N];
#pragma unroll
  for (int k = 0; k < N; k++) im[k] = imass[t.e * imstride + t.r + (size_t)k * S::N2];
  // KR: kp is read again for the sum, where to keep it costs a wave (RK2 at 9^3,
  // p = 7 25.0 us a step against 26.6, p = 9 51.6 against 63)
  constexpr bool KR = ACC == 2 && N == (SP ? 8 : 10), RA = ACC >= 1 && ACC <= 3 && !KR;
  // SP: this thread's component, else all three
  double rv[SP ? 1 : 3][N], ra[RA && !SP ? 3 : 1][RA ? N : 1];
  constexpr bool AU = ACC == 2 || ACC == 6;  // the state is added in the end
  auto pick = [&](auto *const (&p)[3]) { return cs == 0 ? p[0] : (cs == 1 ? p[1] : p[2]); };
  if constexpr (KP) {
    int ec[3];
    gf::box_elem_coords(topo, t.e, ec);
    const gf::BoxElemDeltas de = gf::box_elem_deltas(topo, N, ec);
    const int l = t.r;
    const int64_t ebase = (int64_t)t.e * S::NN;
    double *hu = hk + UOFF;
    double *ha = hk + (GU ? 2 * H::SIZE : AOFF);
    const gf::HaloSum<N> hs(de, t.i, t.j);
    gf::static_for<0, SP ? 1 : 3>([&](auto cc) {
      constexpr int c = decltype(cc)::value;
      const double *kpc = SP ? pick(kp) : kp[c], *uic = SP ? pick(uin) : uin[c];
      double *acl = SP ? pick(acc) : acc[c];
      if (c > 0) __syncthreads();  // the previous component's group sums have read LDS
      // every load of the component is issued before the first LDS store
      double ko[N], uo[N], ao[N];
      if constexpr (L8) {
        lds_copy512(kpc + ebase, hk, l);
        if (UIN) lds_copy512(uic + ebase, hu, l);
        if (ACC == 3) lds_copy512(acl + ebase, ha, l);
      } else {
#pragma unroll
        for (int k = 0; k < N; k++) ko[k] = kpc[col + (size_t)k * S::N2];
        if (UIN) {
#pragma unroll
          for (int k = 0; k < N; k++) uo[k] = uic[col + (size_t)k * S::N2];
        }
        if (ACC == 3) {
#pragma unroll
          for (int k = 0; k < N; k++) ao[k] = acl[col + (size_t)k * S::N2];
        }
      }
      gf::HaloRim<N, double> Lk, Lu;
      Lk.issue(kpc, de, ebase, l);
      if (GU) Lu.issue(uic, de, ebase, l);
      Lk.store(hk, l);
      if (GU) Lu.store(hu, l);
      if constexpr (!L8) {
#pragma unroll
        for (int k = 0; k < N; k++) {
          hk[l + S::N2 * k] = ko[k];
          if (GU) hu[l + S::N2 * k] = uo[k];
        }
      }
      __syncthreads();
      gf::static_for<0, N>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        const int own = l + S::N2 * k;
        const double inv = hs.template inv_k<k>();  // Smooth: Sum / count, exact
        const double kown = L8 ? hk[own] : ko[k];
        const double ks = hs.template sum<k>(hk, kown) * inv;
        double v;
        if constexpr (IN == 3) {
          v = ks;
          if (t.active) acl[col + (size_t)k * S::N2] = v;
        } else {
          const double u = L8 ? hu[own] : uo[k];
          v = fma(bh, ks, u);
          // the members only: an absent partner's zero would add bh ks
          if (GU)
            v = hs.template sum<k>(hu, u, [&](double w, bool on) {
              return on ? fma(bh, ks, w) : 0.0;
            }) * inv;
          if constexpr (ACC == 1) ra[c][k] = fma(ca, kown, u);
          if constexpr (ACC == 2 && RA) ra[c][k] = ca * kown;
          if constexpr (ACC == 3) ra[c][k] = fma(ca, kown, L8 ? ha[own] : ao[k]);
          if constexpr (ACC == 5) {
            if (t.active) acl[col + (size_t)k * S::N2] = ca * kown;
          }
        }
        // the value is formed here, node by node: without this the compiler
        // interleaves the sums of many nodes and keeps their operands live
        // (354 registers instead of 154 at N = 8, IN 1, ACC 0)
        asm volatile("" : "+v"(v));
        if constexpr (ACC == 4) {
          if (t.active) acl[col + (size_t)k * S::N2] = v;
        }
        rv[c][k] = v;
      });
    });
    __syncthreads();  // the element buffers below reuse the halo area
  } else {
#pragma unroll
    for (int c = 0; c < (SP ? 1 : 3); c++) {
      const double *uic = SP ? pick(uin) : uin[c];
#pragma unroll
      for (int k = 0; k < N; k++) rv[c][k] = uic[col + (size_t)k * S::N2];
    }
  }
  // the velocity of the column
  double va[SP ? 3 : 1][N];
  if constexpr (SP) {
#pragma unroll
    for (int k = 0; k < N; k++) hk[t.r + S::N2 * k] = rv[0][k];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int k = 0; k < N; k++) va[c][k] = sl[(c * S::EPB + t.el) * NSL + t.r + S::N2 * k];
    __syncthreads();
  }
  auto vel = [&](int c, int k) { return SP ? va[SP ? c : 0][k] : rv[SP ? 0 : c][k]; };
  double *su = hk, *sd = hk + S::SZ, *sx = hk + 2 * S::SZ;
  const double jac = ejac[t.e];
  const double wa = W[t.i], wb = W[t.j];
  const double rx = edx[t.e * 3], ry = edx[t.e * 3 + 1], rz = edx[t.e * 3 + 2];
#pragma unroll
  for (int c = 0; c < (SP ? 1 : 3); c++) {
    // the z pass's derivatives, kept for the advection term
    double uzs[N];
    auto zcb = [&](int k, double uz, double) { uzs[k] = uz; };
    auto xcb = [&](int, double ux, double) { return ux * rx; };
    double *ko = SP ? pick(kout) : kout[c], *ac = SP ? pick(acc) : acc[c];
    const double *uic = SP ? pick(uin) : uin[c];
    // operands of the sum, read again (kept over the operator, the state and the
    // accumulator cost N = 9 a wave: RK3 at 16^3 317 us a step against 253) and on
    // their way while the y pencil is worked
    const double *kpc = SP ? pick(kp) : kp[c];
    double us[AU ? N : 1], as[ACC == 6 || KR ? N : 1];
    auto ycb = [&](int j, double uy, double) {
      if constexpr (AU) us[j] = uic[col + (size_t)j * S::N2];
      if constexpr (ACC == 6 || KR) as[j] = (KR ? kpc : ac)[col + (size_t)j * S::N2];
      return uy * ry;
    };
    auto post = [&](int k, double L, double M, double hx, double hy) {
      if (!t.active) return;
      const size_t g = col + k * S::N2;
      // contractions written out: every form of the stage rounds alike
      const double po =
          fma(uzs[k] * rz, vel(2, k), fma(hy, vel(1, k), hx * vel(0, k)));
      if (nu != 1.0) L *= nu;
      const double urhs = fma(-po, M, -L);
      const double K = im[k] * urhs;
      if (!LAST) ko[g] = K;
      if constexpr (ACC == 1 || ACC == 3) ac[g] = fma(cb, K, ra[c][k]);
      if constexpr (AU) {
        double a;
        if constexpr (RA) a = ra[c][k];
        else a = ACC == 6 ? as[k] : ca * as[k];
        ac[g] = us[k] + fma(cb, K, a);
      }
    };
    gf::pen_op3<N, double, true>(rv[c], su, sd, sx, Dp, W, t.i, t.j, wa, wb, jac, rx * rx, ry * ry,
                                 rz * rz, (const double *)nullptr, xcb, ycb, zcb, post);
    if (!SP) __syncthreads();  // the next component reuses the LDS buffers
  }
}

// Step output on a structured box: u = S(acc), the Smooth by gather through
// the LDS halo, with the operations of the fused form (IN 3 above).
template <int N>
__global__ __launch_bounds__(gf::PenS<N>::THREADS) void k_rk_out_halo(
    double *__restrict__ u0, double *__restrict__ u1, double *__restrict__ u2,
    const double *__restrict__ a0, const double *__restrict__ a1, const double *__restrict__ a2,
    gf::BoxTopo topo, size_t nelems) {
  using S = gf::PenS<N>;
  using H = gf::Halo<N>;
  __shared__ double sl[S::EPB * H::SIZE];
  double *u[3] = {u0, u1, u2};
  const double *acc[3] = {a0, a1, a2};
  ColIdx<N, gf::PenS<N>> t(nelems);
  double *hk = sl + t.el * H::SIZE;
  const int l = t.r;
  const int64_t ebase = (int64_t)t.e * S::NN;
  int ec[3];
  gf::box_elem_coords(topo, t.e, ec);
  const gf::BoxElemDeltas de = gf::box_elem_deltas(topo, N, ec);
  const gf::HaloSum<N> hs(de, t.i, t.j);
  gf::static_for<0, 3>([&](auto cc) {
    constexpr int c = decltype(cc)::value;
    __syncthreads();  // the previous component's sums have read LDS
    gf::HaloRim<N, double> L;
    if constexpr (N == 8) {
      lds_copy512(acc[c] + ebase, hk, l);
      L.issue(acc[c], de, ebase, l);
    } else {
      double ao[N];
#pragma unroll
      for (int k = 0; k < N; k++) ao[k] = acc[c][ebase + l + S::N2 * k];
      L.issue(acc[c], de, ebase, l);
#pragma unroll
      for (int k = 0; k < N; k++) hk[l + S::N2 * k] = ao[k];
    }
    L.store(hk, l);
    __syncthreads();
    gf::static_for<0, N>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      const double s = hs.template sum<k>(hk, hk[l + S::N2 * k]);
      if (t.active) u[c][ebase + l + S::N2 * k] = s * hs.template inv_k<k>();
    });
  });
}

template <int N, int IN, int ACC, bool SP>
int launch_stage3b_h(gf_mesh *m, double *const *uin, double *const *kp, double *const *acc,
                     double *const *kout, double bh, double ca, double cb, double nu) {
  using S = gf::PenStage<N, SP>;
  const int nb = xcd_grid((m->nelems + S::EPB - 1) / S::EPB);
  auto at = [](double *const *p, int c) { return p ? p[c] : nullptr; };
  hipLaunchKernelGGL((k_burgers_stage3b<N, IN, ACC, SP>), dim3(nb), dim3(S::THREADS), 0,
                     m->ctx->stream, at(uin, 0), at(uin, 1), at(uin, 2), at(kp, 0), at(kp, 1),
                     at(kp, 2), at(acc, 0), at(acc, 1), at(acc, 2), at(kout, 0), at(kout, 1),
                     at(kout, 2), m->imass_el ? m->imass_el : m->imass, m->W[0], m->edx, m->ejac,
                     pend_d(m), bh, ca, cb, nu, m->box, m->nelems,
                     m->imass_el ? (size_t)0 : (size_t)S::NN);
  GF_LAUNCH_CHECK(m->ctx);
  return GF_OK;
}

template <int N>
int launch_stage3b(gf_mesh *m, double *const *uin, double *const *kp, double *const *acc,
                   double *const *kout, double bh, double ca, double cb, double nu, int in,
                   int accm) {
  const bool sp = m->nelems <= stage_split_max(N);
#define GF_STAGE(I, A)                                                                         \
  if (in == I && accm == A)                                                                    \
  return sp ? launch_stage3b_h<N, I, A, true>(m, uin, kp, acc, kout, bh, ca, cb, nu)           \
            : launch_stage3b_h<N, I, A, false>(m, uin, kp, acc, kout, bh, ca, cb, nu)
  GF_STAGE(0, 0);
  GF_STAGE(3, 0);
  GF_STAGE(1, 0);
  GF_STAGE(1, 1);
  GF_STAGE(1, 2);
  GF_STAGE(1, 3);
  GF_STAGE(1, 4);
  GF_STAGE(1, 5);
  GF_STAGE(1, 6);
  GF_STAGE(2, 2);
  GF_STAGE(2, 3);
  GF_STAGE(2, 6);
#undef GF_STAGE
  return gf_set_err(m->ctx, GF_ERR_ARG, "stage3b: unsupported stage form");
}

template <int N>
int launch_rk_out_box(gf_mesh *m, double *const *u, double *const *acc) {
  using S = gf::PenS<N>;
  hipLaunchKernelGGL(k_rk_out_halo<N>, dim3(xcd_grid((m->nelems + S::EPB - 1) / S::EPB)),
                     dim3(S::THREADS), 0, m->ctx->stream, u[0], u[1], u[2], acc[0], acc[1], acc[2],
                     m->box, m->nelems);
  GF_LAUNCH_CHECK(m->ctx);
  return GF_OK;
}

// ---------------------------------------------------------------------------
// Adjoint of the Burgers right-hand side on regular 3-D elements, and of the
// RK step's stages on structured boxes.  With z_c = Minv w_c,
//   y_j = -( sum_d D_d^T [ M (nu r_d^2 D_d z_j + r_d u_d z_j) ]
//            + sum_c (r_j D_j u_c) M z_c )
// is (dF/du)^T w (see gf_adjoint.hip): the viscous term and the transported
// quantity share one transposed contraction per direction, and the element's
// three components are worked together.  On a box the Smooths of the step's
// adjoint are formed by gather, as in k_burgers_stage3b:
//   MODE
//     0  w = y; lam (`yo`) += (dF/du)^T w
//     1  last stage: abar = S(y), y = dJ/du_{n+1}; w = hc abar; yo = y_s
//     2  after it: w = hc abar + hb S(y); lin = abar + S(y) (the final-stage
//        input is smoothed); yo = y_s
//     3  w as in 2; lin += y; yo = y_s
//     4  first stage: w as in 2; yo = lin + y + y_0 = dJ/du_n
//     5  first stage of two: w as in 2; yo = abar + S(y) + y_0
// abar is smooth, so S(hc abar + hb y) is hc abar + hb S(y).  Bound by memory
// and latency like the forward stage: 9-18 fields a stage.  12^3, p = 6: a
// step's adjoint takes 193 us with its stage states; composed (a
// derivative, a product and an update for every pair of components, a DSS
// pass for every smoothed field) 1750.
// ---------------------------------------------------------------------------
template <int N, int MODE>
__global__ __launch_bounds__(gf::Pen3<N>::THREADS) __attribute__((amdgpu_waves_per_eu(N <= 8 ? 2 : 1)))
void k_burgers_adj3(Adj3Args a) {
  using S = gf::Pen3<N>;
  using H = gf::Halo<N>;
  constexpr bool G = MODE != 0, FIN = MODE >= 4;
  constexpr int NSL = G && H::SIZE > 5 * S::SZ ? H::SIZE : 5 * S::SZ;
  __shared__ double sl[S::EPB * NSL];
  ColIdx<N> t(a.nelems);
  const size_t col = t.e * S::NN + t.r;
  const int64_t ebase = (int64_t)t.e * S::NN;
  double *hk = sl + t.el * NSL;
  double rz[3][N], rl[FIN ? 3 : 1][FIN ? N : 1];
  {
    double im[N];
#pragma unroll
    for (int k = 0; k < N; k++) im[k] = a.imass[t.e * a.imstride + t.r + (size_t)k * S::N2];
    if constexpr (G) {
      int ec[3];
      gf::box_elem_coords(a.topo, t.e, ec);
      const gf::BoxElemDeltas de = gf::box_elem_deltas(a.topo, N, ec);
      const gf::HaloSum<N> hs(de, t.i, t.j);
      gf::static_for<0, 3>([&](auto cc) {
        constexpr int c = decltype(cc)::value;
        const double *__restrict__ y = a.y[c];
        __syncthreads();  // the previous component's sums have read LDS
        double yo[N], ab[N], li[N];
#pragma unroll
        for (int k = 0; k < N; k++) yo[k] = y[col + (size_t)k * S::N2];
        gf::HaloRim<N, double> L;
        L.issue(y, de, ebase, t.r);
#pragma unroll
        for (int k = 0; k < N; k++) {
          if (MODE >= 2) ab[k] = a.abar[c][col + (size_t)k * S::N2];
          if (MODE == 3 || MODE == 4) li[k] = a.lin[c][col + (size_t)k * S::N2];
        }
#pragma unroll
        for (int k = 0; k < N; k++) hk[t.r + S::N2 * k] = yo[k];
        L.store(hk, t.r);
        __syncthreads();
        gf::static_for<0, N>([&](auto kc) {
          constexpr int k = decltype(kc)::value;
          const size_t g = col + (size_t)k * S::N2;
          double s = hs.template sum<k>(hk, yo[k]) * hs.template inv_k<k>();
          asm volatile("" : "+v"(s));  // node by node (see k_burgers_stage3b)
          double w;
          if constexpr (MODE == 1) {
            if (t.active) a.abar[c][g] = s;
            w = a.hc * s;
          } else {
            w = fma(a.hb, s, a.hc * ab[k]);
            if constexpr (MODE == 2) {
              if (t.active) a.lin[c][g] = ab[k] + s;
            }
            if constexpr (MODE == 3) {
              if (t.active) a.lin[c][g] = li[k] + yo[k];
            }
            if constexpr (MODE == 4) rl[c][k] = li[k] + yo[k];
            if constexpr (MODE == 5) rl[c][k] = ab[k] + s;
          }
          rz[c][k] = im[k] * w;
        });
      });
      __syncthreads();  // the element buffers below reuse the halo
    } else {
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int k = 0; k < N; k++) rz[c][k] = im[k] * a.y[c][col + (size_t)k * S::N2];
    }
  }
  // element buffers: u_0, u_1, u_2, and two for the passes
  double *U[3] = {hk, hk + S::SZ, hk + 2 * S::SZ}, *su = hk + 3 * S::SZ, *sd = hk + 4 * S::SZ;
  const double cab = (a.W[t.j] * a.W[t.i]) * a.ejac[t.e];  // M = W[k] cab on the thread's pencils
  const double r_[3] = {a.edx[t.e * 3], a.edx[t.e * 3 + 1], a.edx[t.e * 3 + 2]};
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int k = 0; k < N; k++) U[c][S::at(t.i, t.j, k)] = a.u[c][col + (size_t)k * S::N2];
  // element (pencil node m) of the thread's pencil along direction d
  auto at = [&](int d, int m) {
    return d == 0 ? S::at(m, t.i, t.j) : (d == 1 ? S::at(t.i, m, t.j) : S::at(t.i, t.j, m));
  };
  gf::static_for<0, 3>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    // T = sum_c (r_j D_j u_c) M z_c at the column's nodes: the derivatives on
    // the pencils of direction j, through sd to the column
    double T[N], p[N], d[N];
#pragma unroll
    for (int k = 0; k < N; k++) su[S::at(t.i, t.j, k)] = rz[j][k];
    gf::static_for<0, 3>([&](auto cc) {
      constexpr int c = decltype(cc)::value;
      if (c == 0 || j != 2) __syncthreads();  // U and su are written; sd has been read
#pragma unroll
      for (int m = 0; m < N; m++) p[m] = U[c][at(j, m)];
      gf::gll_apply<N, false>(p, d);
      if constexpr (j != 2) {
#pragma unroll
        for (int m = 0; m < N; m++) sd[at(j, m)] = d[m];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < N; k++) d[k] = sd[S::at(t.i, t.j, k)];
      }
#pragma unroll
      for (int k = 0; k < N; k++) {
        const double v = (a.W[k] * cab) * rz[c][k];
        T[k] = c == 0 ? d[k] * v : fma(d[k], v, T[k]);
        asm volatile("" : "+v"(T[k]));
      }
    });
#pragma unroll
    for (int k = 0; k < N; k++) T[k] *= r_[j];
    if (j != 2) __syncthreads();  // sd has been read
    // sum_d D_d^T [ M (nu r_d^2 D_d z_j + r_d u_d z_j) ]: z on the column,
    // x and y on their pencils
    gf::static_for<0, 3>([&](auto dc) {
      constexpr int dd = 2 - decltype(dc)::value;  // z, y, x
      double f[N];
      const double nr = a.nu * (r_[dd] * r_[dd]);
#pragma unroll
      for (int m = 0; m < N; m++) p[m] = dd == 2 ? rz[j][m] : su[at(dd, m)];
      gf::gll_apply<N, false>(p, f);
#pragma unroll
      for (int m = 0; m < N; m++)
        f[m] = (a.W[m] * cab) * fma(nr, f[m], (r_[dd] * U[dd][at(dd, m)]) * p[m]);
      gf::gll_apply<N, true>(f, d);
      if constexpr (dd == 2) {
#pragma unroll
        for (int k = 0; k < N; k++) {
          T[k] += d[k];
          asm volatile("" : "+v"(T[k]));
        }
      } else if constexpr (dd == 1) {
#pragma unroll
        for (int m = 0; m < N; m++) sd[at(1, m)] = d[m];
        __syncthreads();
      } else {
#pragma unroll
        for (int m = 0; m < N; m++) sd[at(0, m)] += d[m];
        __syncthreads();
      }
    });
#pragma unroll
    for (int k = 0; k < N; k++) {
      const size_t g = col + (size_t)k * S::N2;
      const double y = -(sd[S::at(t.i, t.j, k)] + T[k]);
      if (t.active) {
        if (MODE == 0) a.yo[j][g] += y;
        else if (FIN) a.yo[j][g] = rl[FIN ? j : 0][FIN ? k : 0] + y;
        else a.yo[j][g] = y;
      }
    }
  });
}

// The final-stage input of a step on a structured box: v = S(u + bh S(k)), or
// u + bh S(k) on a continuous u (SM false), where the two agree bit for bit.
template <int N, bool SM>
__global__ __launch_bounds__(gf::Pen3<N>::THREADS) void k_stage_input_halo(
    const double *__restrict__ u0, const double *__restrict__ u1, const double *__restrict__ u2,
    const double *__restrict__ k0, const double *__restrict__ k1, const double *__restrict__ k2,
    double *__restrict__ v0, double *__restrict__ v1, double *__restrict__ v2, double bh,
    gf::BoxTopo topo, size_t nelems) {
  using S = gf::Pen3<N>;
  using H = gf::Halo<N>;
  __shared__ double sl[S::EPB * (SM ? 2 : 1) * H::SIZE];
  const double *u[3] = {u0, u1, u2}, *kf[3] = {k0, k1, k2};
  double *v[3] = {v0, v1, v2};
  ColIdx<N> t(nelems);
  double *hk = sl + t.el * (SM ? 2 : 1) * H::SIZE, *hu = hk + H::SIZE;
  const int64_t ebase = (int64_t)t.e * S::NN;
  int ec[3];
  gf::box_elem_coords(topo, t.e, ec);
  const gf::BoxElemDeltas de = gf::box_elem_deltas(topo, N, ec);
  const gf::HaloSum<N> hs(de, t.i, t.j);
  gf::static_for<0, 3>([&](auto cc) {
    constexpr int c = decltype(cc)::value;
    __syncthreads();  // the previous component's sums have read LDS
    double ko[N], uo[N];
    gf::HaloRim<N, double> Lk, Lu;
#pragma unroll
    for (int k = 0; k < N; k++) ko[k] = kf[c][ebase + t.r + S::N2 * k];
#pragma unroll
    for (int k = 0; k < N; k++) uo[k] = u[c][ebase + t.r + S::N2 * k];
    Lk.issue(kf[c], de, ebase, t.r);
    if (SM) Lu.issue(u[c], de, ebase, t.r);
#pragma unroll
    for (int k = 0; k < N; k++) {
      hk[t.r + S::N2 * k] = ko[k];
      if (SM) hu[t.r + S::N2 * k] = uo[k];
    }
    Lk.store(hk, t.r);
    if (SM) Lu.store(hu, t.r);
    __syncthreads();
    gf::static_for<0, N>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      const double inv = hs.template inv_k<k>();
      const double ks = hs.template sum<k>(hk, ko[k]) * inv;
      double r = fma(bh, ks, uo[k]);
      if (SM)
        r = hs.template sum<k>(hu, uo[k], [&](double w, bool on) {
          return on ? fma(bh, ks, w) : 0.0;
        }) * inv;
      asm volatile("" : "+v"(r));  // node by node (see k_burgers_stage3b)
      if (t.active) v[c][ebase + t.r + S::N2 * k] = r;
    });
  });
}

template <int N>
int launch_adj3(gf_mesh *m, const Adj3Args &a, int mode) {
  using S = gf::Pen3<N>;
  const dim3 nb(xcd_grid((m->nelems + S::EPB - 1) / S::EPB)), nt(S::THREADS);
  switch (mode) {
    case 0: hipLaunchKernelGGL((k_burgers_adj3<N, 0>), nb, nt, 0, m->ctx->stream, a); break;
    case 1: hipLaunchKernelGGL((k_burgers_adj3<N, 1>), nb, nt, 0, m->ctx->stream, a); break;
    case 2: hipLaunchKernelGGL((k_burgers_adj3<N, 2>), nb, nt, 0, m->ctx->stream, a); break;
    case 3: hipLaunchKernelGGL((k_burgers_adj3<N, 3>), nb, nt, 0, m->ctx->stream, a); break;
    case 4: hipLaunchKernelGGL((k_burgers_adj3<N, 4>), nb, nt, 0, m->ctx->stream, a); break;
    default: hipLaunchKernelGGL((k_burgers_adj3<N, 5>), nb, nt, 0, m->ctx->stream, a); break;
  }
  GF_LAUNCH_CHECK(m->ctx);
  return GF_OK;
}
template <int N>
int launch_stage_input(gf_mesh *m, const double *const *u, double *const *k, double *const *v,
                       double bh, int cont) {
  using S = gf::Pen3<N>;
  const dim3 nb(xcd_grid((m->nelems + S::EPB - 1) / S::EPB)), nt(S::THREADS);
  if (cont)
    hipLaunchKernelGGL((k_stage_input_halo<N, false>), nb, nt, 0, m->ctx->stream, u[0], u[1], u[2],
                       k[0], k[1], k[2], v[0], v[1], v[2], bh, m->box, m->nelems);
  else
    hipLaunchKernelGGL((k_stage_input_halo<N, true>), nb, nt, 0, m->ctx->stream, u[0], u[1], u[2],
                       k[0], k[1], k[2], v[0], v[1], v[2], bh, m->box, m->nelems);
  GF_LAUNCH_CHECK(m->ctx);
  return GF_OK;
}

template <int N, typename T>
int launch_helm3p(gf_mesh *m, T p, const T *pf, const T *qf, T qs, const T *u, T *uo,
                  const gf::PenD<T> &D, const T *W, const T *edx, const T *ejac) {
  using S = gf::Pen3<N>;
  int nb = xcd_grid((m->nelems + S::EPB - 1) / S::EPB);
  hipLaunchKernelGGL((k_helm3p<N, T>), dim3(nb), dim3(S::THREADS), 0, m->ctx->stream, u, uo, D, W,
                     edx, ejac, p, pf, qf, qs, m->nelems);
  GF_LAUNCH_CHECK(m->ctx);
  return GF_OK;
}

// Blocks of the 3-D CG kernels: as many as are resident at once (FP64 8
// waves a CU by registers, FP32 16).  Twice as many in FP64: 20^3, p = 6
// 76 us an iteration against 71, 16^3, p = 7 50 against 43.
template <typename T, int N>
int cg_blocks3(size_t nelems) {
  constexpr int EPB = CGShape<N>::EPB;
  return loop_blocks((nelems + EPB - 1) / EPB, sizeof(T) == 8 ? 512 : 1024);
}

// stream: the solve's vectors do not fit the 256 MB Infinity Cache.  Then x
// and w, read and written by this kernel only, are marked non-temporal, so
// that the cache keeps r and q for the update kernel (which walks backwards).
template <int N, typename T>
int launch_cg_apply3p(gf_mesh *m, const CGApply3Args &a) {
  if (a.c.stream)
    hipLaunchKernelGGL((k_cg_apply3p<N, T, true>), dim3(a.c.nbA), dim3(kThreads), 0, m->ctx->stream,
                       a);
  else
    hipLaunchKernelGGL((k_cg_apply3p<N, T, false>), dim3(a.c.nbA), dim3(kThreads), 0,
                       m->ctx->stream, a);
  GF_LAUNCH_CHECK(m->ctx);
  return GF_OK;
}

template <int N>
int helm3c_d(gf_mesh *m, double p, const double *pf, const double *qf, double qs, const double *u,
             double *uo) {
  return launch_helm3p<N, double>(m, p, pf, qf, qs, u, uo, pend_d(m), m->W[0], m->edx, m->ejac);
}
template <int N>
int helm3c_f(gf_mesh *m, float p, const float *qf, float qs, const float *u, float *uo) {
  return launch_helm3p<N, float>(m, p, (const float *)nullptr, qf, qs, u, uo, pend_f(m), m->W32,
                                 m->edx32, m->ejac32);
}
template <int N>
int cgapply3c_d(gf_mesh *m, const CGApply3Args &a) { return launch_cg_apply3p<N, double>(m, a); }
template <int N>
int cgapply3c_f(gf_mesh *m, const CGApply3Args &a) { return launch_cg_apply3p<N, float>(m, a); }

// CG update on structured boxes (see CGCtl): q arrives unassembled, straight
// from the apply, and is assembled here through the LDS halo of each element
// (gf_boxdss.hpp), so no DSS pass runs in between; r -= alpha DSS(q), and the
// partial sums of r.z / (group size) and of the norm.  All copies of a node
// sum its group in the same order, so r stays continuous bit for bit.  topos:
// the box of each system of a batched mesh.
template <typename T, int NORM, int N>
__global__ __launch_bounds__(kThreads) void k_cg_update_halo(
    CGCtl c, T *__restrict__ r, const T *__restrict__ qv, const T *__restrict__ dinv,
    const double *__restrict__ mass, gf::BoxTopo topo1, const gf::BoxTopo *__restrict__ topos,
    const T *__restrict__ dtab, const unsigned char *__restrict__ deq) {
  using S = gf::Pen3<N>;
  using C = CGShape<N>;
  using H = gf::Halo<N>;
  __shared__ T sl[C::EPB][H::SIZE];
  __shared__ double sred[2 * (kThreads / 64)];
  const CGBlock b(c, (int)xcd_block(), c.nbU);
  if (!b.ok) return;
  CGAlphaHead h(c, b);
  const gf::BoxTopo topo = topos ? topos[b.s] : topo1;
  const C t;
  T *hl = sl[t.el];
  T qo[N], ro[N], dv[N];
  gf::HaloRim<N, T> L;
  gf::BoxElemDeltas de;
  size_t col;
  bool act;
  auto load = [&](int64_t ch) {
    const size_t el = (size_t)ch * C::EPB + t.el, nel = b.e1 - b.e0;
    act = t.own() && el < nel;
    const size_t le = el < nel ? el : nel - 1, e = b.e0 + le;
    col = e * S::NN + t.r;
    int ec[3];
    gf::box_elem_coords(topo, le, ec);
    de = gf::box_elem_deltas(topo, N, ec);
    const T *dsrc = dinv ? ((dtab && deq[e]) ? dtab + t.r : dinv + col) : nullptr;
#pragma unroll
    for (int q = 0; q < N; q++) qo[q] = qv[col + q * S::N2];
    L.issue(qv, de, (int64_t)(e * S::NN), t.r);
#pragma unroll
    for (int q = 0; q < N; q++) ro[q] = r[col + q * S::N2];
#pragma unroll
    for (int q = 0; q < N; q++) dv[q] = dsrc ? dsrc[q * S::N2] : T(1);
  };
  CGWalk k(c, b, C::EPB, true);
  if (k.in()) load(k.c);
  double alpha64;
  if (!h.finish(b, sred, alpha64)) return;
  const T alpha = (T)alpha64;
  double rho = 0.0, nrm = 0.0;
  while (k.in()) {
    gf::elem_sync<C::WAVE>();  // the previous element's sums have read LDS
#pragma unroll
    for (int q = 0; q < N; q++)
      if (t.own()) hl[t.r + S::N2 * q] = qo[q];
    if (t.own()) L.store(hl, t.r);
    gf::elem_sync<C::WAVE>();
    const gf::HaloSum<N> hs(de, t.i, t.j);
    gf::static_for<0, N>([&](auto kc) {
      constexpr int q = decltype(kc)::value;
      const T s = hs.template sum<q>(hl, qo[q]);
      T rn = ro[q] + (-alpha) * s;
      asm volatile("" : "+v"(rn));  // node by node (see k_burgers_stage3b)
      const size_t g = col + q * S::N2;
      if (act) {
        r[g] = rn;
        cg_accum<NORM>((double)rn, dinv ? (double)(dv[q] * rn) : (double)rn, hs.template inv_k<q>(), mass,
                       g, rho, nrm);
      }
    });
    k.next();
    if (k.in()) load(k.c);
  }
  const double ra = gf::block_reduce<false>(rho, sred);
  const double rb = NORM == GF_NORM_INF ? gf::block_reduce<true>(nrm, sred)
                                        : gf::block_reduce<false>(nrm, sred);
  if (threadIdx.x == 0) ((double2 *)c.partU)[b.b0 + b.lb] = make_double2(ra, rb);
}

template <typename T, int NORM, int N>
int launch_update_box_n(gf_mesh *m, const CGCtl &c, const CGVecs<T> &v) {
  hipLaunchKernelGGL((k_cg_update_halo<T, NORM, N>), dim3(c.nbU), dim3(kThreads), 0,
                     m->ctx->stream, c, v.r, v.q, v.dinv, m->mass, m->box, v.topos, v.dtab, v.deq);
  GF_LAUNCH_CHECK(m->ctx);
  return GF_OK;
}

}  // namespace gfs

#define GF_K3D_UPD(T, N) \
  template int cg_blocks3<T, N>(size_t); \
  template int launch_update_box_n<T, GF_NORM_INF, N>(gf_mesh *, const CGCtl &, const CGVecs<T> &); \
  template int launch_update_box_n<T, GF_NORM_EUC, N>(gf_mesh *, const CGCtl &, const CGVecs<T> &); \
  template int launch_update_box_n<T, GF_NORM_L2, N>(gf_mesh *, const CGCtl &, const CGVecs<T> &); \
  template int launch_update_box_n<T, GF_NORM_L1, N>(gf_mesh *, const CGCtl &, const CGVecs<T> &); \
  template int launch_update_box_n<T, GF_NORM_ASSEMBLED_L2, N>(gf_mesh *, const CGCtl &, const CGVecs<T> &);

#define GF_K3D_INSTANTIATE(N)                                                                \
  template int launch_stage3p<N>(gf_mesh *, const StageArgs &);                              \
  template int launch_advect3p<N>(gf_mesh *, const double *, const double *const *, double *); \
  template int launch_grad3p<N>(gf_mesh *, const double *, double *const *, const double *);  \
  template int launch_stage3b<N>(gf_mesh *, double *const *, double *const *, double *const *, \
                                 double *const *, double, double, double, double, int, int); \
  template int launch_rk_out_box<N>(gf_mesh *, double *const *, double *const *);             \
  template int launch_adj3<N>(gf_mesh *, const Adj3Args &, int);                             \
  template int launch_stage_input<N>(gf_mesh *, const double *const *, double *const *,      \
                                     double *const *, double, int);                          \
  template int helm3c_d<N>(gf_mesh *, double, const double *, const double *, double,         \
                           const double *, double *);                                        \
  template int helm3c_f<N>(gf_mesh *, float, const float *, float, const float *, float *);   \
  template int cgapply3c_d<N>(gf_mesh *, const CGApply3Args &);                              \
  template int cgapply3c_f<N>(gf_mesh *, const CGApply3Args &);                              \
  GF_K3D_UPD(float, N)                                                                       \
  GF_K3D_UPD(double, N)
