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

template <int N, typename T>
__global__ __launch_bounds__(gf::Pen3<N>::THREADS) void k_cg_apply3p(
    const T *__restrict__ r, const T *__restrict__ dinv, T *__restrict__ w, T *__restrict__ qv,
    gf::PenD<T> Dp, const T *__restrict__ W, const T *__restrict__ edx,
    const T *__restrict__ ejac, const T *__restrict__ qf, T qs, const T *__restrict__ mask, double pd,
    const double *__restrict__ scal, double *__restrict__ part, size_t nelems, gf::BoxTopo topo,
    int tmask, const int64_t *__restrict__ seg_eoff, int nseg, const double *__restrict__ sscal,
    const T *__restrict__ dtab, const unsigned char *__restrict__ deq) {
  using S = gf::Pen3<N>;
  __shared__ T su[S::EPB][S::SZ], sd[S::EPB][S::SZ];
  __shared__ double sred[S::THREADS > 64 ? S::THREADS : 64];
  ColIdx<N> t(nelems);
  // batched mesh: each element's member scalars; an element of a member
  // that has converged computes nothing it stores, and the partial sums are
  // kept per element so that each member's are one contiguous range
  if (nseg > 0) {
    scal = sscal + kSegScal * seg_of(seg_eoff, nseg, t.e);
    if (scal[S_DONE] != 0.0) {
      if (S::EPB == 1) return;  // the whole workgroup
      t.active = false;
    }
  } else if (scal[S_DONE] != 0.0) {
    return;
  }
  const bool first = scal[S_FIRST] != 0.0;
  const T beta = (T)scal[S_BETA];
  const size_t col = t.e * S::NN + t.r;
  const T jac = ejac[t.e];
  const T f0 = edx[t.e * 3], f1 = edx[t.e * 3 + 1], f2 = edx[t.e * 3 + 2];
  // all loads of the column first, then the stores of w; the Jacobi values
  // from the table where the element's equal it
  const T *dsrc = dinv ? ((dtab && deq[t.e]) ? dtab + t.r : dinv + col) : nullptr;
  T ru[N], dv[N], wv[N];
#pragma unroll
  for (int k = 0; k < N; k++) {
    const size_t g = col + k * S::N2;
    ru[k] = r[g];
    dv[k] = dsrc ? dsrc[k * S::N2] : T(1);
    wv[k] = first ? T(0) : w[g];
  }
#pragma unroll
  for (int k = 0; k < N; k++) {
    const T z = dinv ? dv[k] * ru[k] : ru[k];
    ru[k] = first ? z : beta * wv[k] + T(1) * z;
  }
  if (t.active) {
#pragma unroll
    for (int k = 0; k < N; k++) w[col + k * S::N2] = ru[k];
  }
  double dot = 0.0;
  const T p = (T)pd;
  int ec[3] = {0, 0, 0};
  if (tmask) gf::box_elem_coords(topo, t.e, ec);
  auto post = [&](int k, T Lu, T M, T, T) {
    if (!t.active) return;
    const size_t g = col + k * S::N2;
    T acc = Lu;
    if (p != T(1)) acc *= p;
    if (qf) {
      T tq = M * ru[k];
      tq *= qf[g];
      acc += tq;
    } else if (qs != T(0)) {
      T tq = M * ru[k];
      if (qs != T(1)) tq *= qs;
      acc += tq;
    }
    if (mask) acc *= mask[g];
    else if (tmask && gf::box_masked(topo, N, ec, t.i, t.j, k)) acc *= T(0);
    qv[g] = acc;
    dot += (double)ru[k] * (double)acc;
  };
  gf::pen_op3<N, T, false>(ru, su[t.el], sd[t.el], (T *)nullptr, Dp, W, t.i, t.j, W[t.i],
                           W[t.j], jac, f0 * f0, f1 * f1, f2 * f2, (const T *)nullptr,
                           gf::NoPenCB(), gf::NoPenCB(), gf::NoPenCB(), post);
  if (nseg > 0) {
    // per-element partials: the element's lanes, summed in lane order
    sred[threadIdx.x] = dot;
    __syncthreads();
    if (t.r == 0 && t.active) {
      double v = 0.0;
      for (int q2 = 0; q2 < S::N2; q2++) v += sred[t.el * S::N2 + q2];
      part[t.e] = v;
    }
    return;
  }
  double bs = gf::block_reduce<false>(dot, sred);
  if (threadIdx.x == 0) part[blockIdx.x] = bs;
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
//   ADV false  o0, o1, o2 = d_x p, d_y p, d_z p (GMTK::grad, gmtk.ipp:2883-2892;
//              edx NULL: reference-space derivatives, compute_grefderivs)
//   ADV true   o0 = M (((d_x p) v0 + (d_y p) v1) + (d_z p) v2), GAdvect::apply
//              (gadvect.ipp:57-99); a missing velocity component is zero
// Memory bound: four fields for the gradient, five for the advection (the
// composed advection moved 23).  At 24^3, p = 7: gradient 34 us against 43 of
// the LDS form k_grad, advection 41.5 us (6.8 TB/s) against 242 composed; at
// 21x17x13, p = 5: 8.1 against 9.7 us and 8.5 against 51 us.
template <int N, bool ADV>
__global__ __launch_bounds__(gf::Pen3<N>::THREADS) void k_grad3p(
    const double *__restrict__ p, const double *__restrict__ v0, const double *__restrict__ v1,
    const double *__restrict__ v2, double *__restrict__ o0, double *__restrict__ o1,
    double *__restrict__ o2, const double *__restrict__ W, const double *__restrict__ edx,
    const double *__restrict__ ejac, size_t nelems) {
  using S = gf::Pen3<N>;
  constexpr int NV = ADV ? N : 1;
  __shared__ double su[S::EPB][S::SZ], sd[S::EPB][S::SZ];
  ColIdx<N> t(nelems);
  const size_t col = t.e * S::NN + t.r;
  double rp[N], vx[NV], vy[NV], vz[NV];
#pragma unroll
  for (int k = 0; k < N; k++) rp[k] = p[col + k * S::N2];
  // the velocities' loads are in flight while p is differentiated
  if constexpr (ADV) {
#pragma unroll
    for (int k = 0; k < N; k++) {
      const size_t g = col + k * S::N2;
      vx[k] = v0 ? v0[g] : 0.0;
      vy[k] = v1 ? v1[g] : 0.0;
      vz[k] = v2 ? v2[g] : 0.0;
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
  if constexpr (ADV) {
    const double jac = ejac[t.e], wi = W[t.i], wj = W[t.j];
#pragma unroll
    for (int k = 0; k < N; k++) {
      const int q = S::at(t.i, t.j, k);
      double a = (d[q] * rx) * vx[k];
      a += (u[q] * ry) * vy[k];
      a += (dz[k] * rz) * vz[k];
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
  hipLaunchKernelGGL((k_grad3p<N, true>), dim3(nb), dim3(S::THREADS), 0, m->ctx->stream, p, v[0],
                     v[1], v[2], po, (double *)nullptr, (double *)nullptr, m->W[0], m->edx, m->ejac,
                     m->nelems);
  GF_LAUNCH_CHECK(m->ctx);
  return GF_OK;
}
template <int N>
int launch_grad3p(gf_mesh *m, const double *p, double *const *o, const double *edx) {
  using S = gf::Pen3<N>;
  const int nb = xcd_grid((m->nelems + S::EPB - 1) / S::EPB);
  hipLaunchKernelGGL((k_grad3p<N, false>), dim3(nb), dim3(S::THREADS), 0, m->ctx->stream, p,
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
//     2  acc = uin + ca kp + cb K       (last stage: K is not stored)
//     3  acc = acc + ca kp + cb K       (last stage)
// Group sums are pairwise (x, then y, then z), exact for equal members of
// groups of 2, 4 and 8, so S leaves a continuous state as it is and IN 1 and
// IN 2 agree bit for bit on it.
//
// Bound by memory: at 32^3, p = 7 an RK4 step moves 42 fields of 134 MB; the
// form whose every stage smoothed into the accumulator moved 54 and gathered
// uin too in the last one.  Stages (IN, ACC) = (3,0) 358, (1,1) 424, (1,0)
// 338, (1,3) 399 us, 3.6-3.8 TB/s where a copy of this size has 4.7; before,
// 392 + 543 + 459 + 601 us.  19x14x11, p = 5 (RK3): 27 + 27 + 22 us against
// 39 + 41 + 27, where the members were loaded node by node.
// ---------------------------------------------------------------------------
template <int N, int IN, int ACC>
__global__ __launch_bounds__(gf::Pen3<N>::THREADS) __attribute__((amdgpu_waves_per_eu(N <= 8 ? 2 : 1)))
void k_burgers_stage3b(
    const double *__restrict__ ui0, const double *__restrict__ ui1, const double *__restrict__ ui2,
    const double *__restrict__ kp0, const double *__restrict__ kp1, const double *__restrict__ kp2,
    double *ac0, double *ac1, double *ac2, double *__restrict__ ko0, double *__restrict__ ko1,
    double *__restrict__ ko2, const double *__restrict__ imass, const double *__restrict__ W,
    const double *__restrict__ edx, const double *__restrict__ ejac, gf::PenD<double> Dp,
    double bh, double ca, double cb, double nu, gf::BoxTopo topo, size_t nelems, size_t imstride) {
  using S = gf::Pen3<N>;
  using H = gf::Halo<N>;
  constexpr bool KP = IN != 0, GU = IN == 2, UIN = IN != 3;
  static_assert(KP || ACC == 0, "the first stage accumulates nothing");
  static_assert(IN != 3 || ACC == 0, "an output stage is a first stage");
  // N = 8: an element is one wave and its own values go straight to LDS
  // (lds_copy512), behind kp's halo; else they pass through registers
  constexpr bool L8 = N == 8;
  constexpr int UOFF = H::SIZE, AOFF = UOFF + 512;
  constexpr int HL = !KP ? 0
                         : (GU ? 2 * H::SIZE
                               : H::SIZE + (L8 && UIN ? 512 : 0)) + (L8 && ACC == 3 ? 512 : 0);
  // per element: the halos, then (the same memory) the three element buffers
  constexpr int NSL = HL > 3 * S::SZ ? HL : 3 * S::SZ;
  __shared__ double sl[S::EPB * NSL];
  const double *uin[3] = {ui0, ui1, ui2};
  const double *kp[3] = {kp0, kp1, kp2};
  double *acc[3] = {ac0, ac1, ac2};
  double *kout[3] = {ko0, ko1, ko2};
  ColIdx<N> t(nelems);
  const size_t col = t.e * S::NN + t.r;
  double *hk = sl + t.el * NSL;
  double im[N];
#pragma unroll
  for (int k = 0; k < N; k++) im[k] = imass[t.e * imstride + t.r + (size_t)k * S::N2];
  double ru[3][N], ra[ACC ? 3 : 1][ACC ? N : 1];
  if constexpr (KP) {
    int ec[3];
    gf::box_elem_coords(topo, t.e, ec);
    const gf::BoxElemDeltas de = gf::box_elem_deltas(topo, N, ec);
    const int l = t.r;
    const int64_t ebase = (int64_t)t.e * S::NN;
    double *hu = hk + UOFF;
    double *ha = hk + (GU ? 2 * H::SIZE : AOFF);
    const gf::HaloCol<N> hc(de, t.i, t.j);
    gf::static_for<0, 3>([&](auto cc) {
      constexpr int c = decltype(cc)::value;
      __syncthreads();  // the previous component's group sums have read LDS
      // every load of the component is issued before the first LDS store
      double ko[N], uo[N], ao[N];
      if constexpr (L8) {
        lds_copy512(kp[c] + ebase, hk, l);
        if (UIN) lds_copy512(uin[c] + ebase, hu, l);
        if (ACC == 3) lds_copy512(acc[c] + ebase, ha, l);
      } else {
#pragma unroll
        for (int k = 0; k < N; k++) ko[k] = kp[c][col + (size_t)k * S::N2];
        if (UIN) {
#pragma unroll
          for (int k = 0; k < N; k++) uo[k] = uin[c][col + (size_t)k * S::N2];
        }
        if (ACC == 3) {
#pragma unroll
          for (int k = 0; k < N; k++) ao[k] = acc[c][col + (size_t)k * S::N2];
        }
      }
      gf::HaloRim<N, double> Lk, Lu;
      Lk.issue(kp[c], de, ebase, l);
      if (GU) Lu.issue(uin[c], de, ebase, l);
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
        constexpr bool ZF = k == 0 || k == N - 1;  // groups of up to 8, else 4
        const int own = l + S::N2 * k;
        int ad[8];
        const int cnt = gf::halo_order<N, k>(hc, de, ad);
        const double inv = gf::box_inv(cnt);  // Smooth: Sum / count, exact
        auto sum = [&](auto &&val) {
          double s = (val(ad[0]) + val(ad[1])) + (val(ad[2]) + val(ad[3]));
          if (ZF) s = s + ((val(ad[4]) + val(ad[5])) + (val(ad[6]) + val(ad[7])));
          return s * inv;
        };
        const double kown = L8 ? hk[own] : ko[k];
        const double ks = sum([&](int q) { return hk[q]; });
        double v;
        if constexpr (IN == 3) {
          v = ks;
          if (t.active) acc[c][col + (size_t)k * S::N2] = v;
        } else {
          const double u = L8 ? hu[own] : uo[k];
          v = fma(bh, ks, u);
          // the members only: an absent partner's zero slot would add bh ks
          if (GU) v = sum([&](int q) { return q == H::ZERO ? 0.0 : fma(bh, ks, hu[q]); });
          if constexpr (ACC == 1 || ACC == 2) ra[c][k] = fma(ca, kown, u);
          if constexpr (ACC == 3) ra[c][k] = fma(ca, kown, L8 ? ha[own] : ao[k]);
        }
        // the value is formed here, node by node: without this the compiler
        // interleaves the sums of many nodes and keeps their operands live
        // (354 registers instead of 154 at N = 8, IN 1, ACC 0)
        asm volatile("" : "+v"(v));
        ru[c][k] = v;
      });
    });
    __syncthreads();  // the element buffers below reuse the halo area
  } else {
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int k = 0; k < N; k++) ru[c][k] = uin[c][col + (size_t)k * S::N2];
  }
  double *su = hk, *sd = hk + S::SZ, *sx = hk + 2 * S::SZ;
  const double jac = ejac[t.e];
  const double wa = W[t.i], wb = W[t.j];
  const double rx = edx[t.e * 3], ry = edx[t.e * 3 + 1], rz = edx[t.e * 3 + 2];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    // the z pass's derivatives, kept for the advection term
    double uzs[N];
    auto zcb = [&](int k, double uz, double) { uzs[k] = uz; };
    auto xcb = [&](int, double ux, double) { return ux * rx; };
    auto ycb = [&](int, double uy, double) { return uy * ry; };
    double *ko = kout[c], *ac = acc[c];
    auto post = [&](int k, double L, double M, double hx, double hy) {
      if (!t.active) return;
      const size_t g = col + k * S::N2;
      // contractions written out: every form of the stage rounds alike
      const double po =
          fma(uzs[k] * rz, ru[2][k], fma(hy, ru[1][k], hx * ru[0][k]));
      if (nu != 1.0) L *= nu;
      const double urhs = fma(-po, M, -L);
      const double K = im[k] * urhs;
      if (ACC < 2) ko[g] = K;
      if (ACC) ac[g] = fma(cb, K, ra[ACC ? c : 0][ACC ? k : 0]);
    };
    gf::pen_op3<N, double, true>(ru[c], su, sd, sx, Dp, W, t.i, t.j, wa, wb, jac, rx * rx, ry * ry,
                                 rz * rz, (const double *)nullptr, xcb, ycb, zcb, post);
    __syncthreads();  // the next component reuses the LDS buffers
  }
}

// Step output on a structured box: u = S(acc), the Smooth by gather through
// the LDS halo, with the operations of the fused form (IN 3 above).
template <int N>
__global__ __launch_bounds__(gf::Pen3<N>::THREADS) void k_rk_out_halo(
    double *__restrict__ u0, double *__restrict__ u1, double *__restrict__ u2,
    const double *__restrict__ a0, const double *__restrict__ a1, const double *__restrict__ a2,
    gf::BoxTopo topo, size_t nelems) {
  using S = gf::Pen3<N>;
  using H = gf::Halo<N>;
  __shared__ double sl[S::EPB * H::SIZE];
  double *u[3] = {u0, u1, u2};
  const double *acc[3] = {a0, a1, a2};
  ColIdx<N> t(nelems);
  double *hk = sl + t.el * H::SIZE;
  const int l = t.r;
  const int64_t ebase = (int64_t)t.e * S::NN;
  int ec[3];
  gf::box_elem_coords(topo, t.e, ec);
  const gf::BoxElemDeltas de = gf::box_elem_deltas(topo, N, ec);
  const gf::HaloCol<N> hc(de, t.i, t.j);
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
      constexpr bool ZF = k == 0 || k == N - 1;
      int ad[8];
      const int cnt = gf::halo_order<N, k>(hc, de, ad);
      double s = (hk[ad[0]] + hk[ad[1]]) + (hk[ad[2]] + hk[ad[3]]);
      if (ZF) s = s + ((hk[ad[4]] + hk[ad[5]]) + (hk[ad[6]] + hk[ad[7]]));
      if (t.active) u[c][ebase + l + S::N2 * k] = s * gf::box_inv(cnt);
    });
  });
}

template <int N, int IN, int ACC>
int launch_stage3b_h(gf_mesh *m, double *const *uin, double *const *kp, double *const *acc,
                     double *const *kout, double bh, double ca, double cb, double nu) {
  using S = gf::Pen3<N>;
  const int nb = xcd_grid((m->nelems + S::EPB - 1) / S::EPB);
  auto at = [](double *const *p, int c) { return p ? p[c] : nullptr; };
  hipLaunchKernelGGL((k_burgers_stage3b<N, IN, ACC>), dim3(nb), dim3(S::THREADS), 0,
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
#define GF_STAGE(I, A) \
  if (in == I && accm == A) return launch_stage3b_h<N, I, A>(m, uin, kp, acc, kout, bh, ca, cb, nu)
  GF_STAGE(0, 0);
  GF_STAGE(3, 0);
  GF_STAGE(1, 0);
  GF_STAGE(1, 1);
  GF_STAGE(1, 2);
  GF_STAGE(1, 3);
  GF_STAGE(2, 2);
  GF_STAGE(2, 3);
#undef GF_STAGE
  return gf_set_err(m->ctx, GF_ERR_ARG, "stage3b: unsupported stage form");
}

template <int N>
int launch_rk_out_box(gf_mesh *m, double *const *u, double *const *acc) {
  using S = gf::Pen3<N>;
  hipLaunchKernelGGL(k_rk_out_halo<N>, dim3(xcd_grid((m->nelems + S::EPB - 1) / S::EPB)),
                     dim3(S::THREADS), 0, m->ctx->stream, u[0], u[1], u[2], acc[0], acc[1], acc[2],
                     m->box, m->nelems);
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

template <int N, typename T>
int launch_cg_apply3p(gf_mesh *m, const CGApply3Args &a) {
  using S = gf::Pen3<N>;
  int nb = xcd_grid((m->nelems + S::EPB - 1) / S::EPB);
  gf::PenD<T> Dp;
  for (int c = 0; c < 3; c++) {
    Dp.R[c] = (const T *)a.DR[c];
    Dp.C[c] = (const T *)a.DC[c];
  }
  hipLaunchKernelGGL((k_cg_apply3p<N, T>), dim3(nb), dim3(S::THREADS), 0, m->ctx->stream,
                     (const T *)a.r, (const T *)a.dinv, (T *)a.w, (T *)a.q, Dp, (const T *)a.W,
                     (const T *)a.edx, (const T *)a.ejac, (const T *)a.qf, (T)a.qs, (const T *)a.mask, a.p,
                     (const double *)a.scal, a.part, a.nelems, a.topo, a.tmask, a.seg_eoff, a.nseg,
                     (const double *)a.sscal, (const T *)a.dtab, a.deq);
  GF_LAUNCH_CHECK(m->ctx);
  return GF_OK;
}

// Number of workgroups (= partial sums) the 3-D column apply launches.
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

// u3 = uin + bh*k ; acc = accsrc + ch*k   (final-stage input of step_b, :315-320)

// k_cg_update on a structured box: q arrives unassembled (straight from the
// apply) and is assembled here by gather (gf_boxdss.hpp), in the GGFX order,
// so no DSS pass runs between the apply and the update.  The multiplicity
// weight is 1/(group size), which equals GGFX::get_imult.  Work is split in
// chunks of whole elements so that an element's box coordinates are formed
// once per chunk (and are wave-uniform when a chunk is one element).
template <typename T, int NORM, int N, typename I>
__global__ __launch_bounds__(kThreads) void k_cg_update_box(
    T *__restrict__ x, const T *__restrict__ w, T *__restrict__ r, const T *__restrict__ qv,
    const T *__restrict__ dinv, const double *__restrict__ mass, gf::BoxTopo topo, double *scal,
    double *__restrict__ part, size_t nelems) {
  constexpr int NN = N * N * N;
  constexpr int CE = NN >= kThreads ? 1 : kThreads / NN;  // elements per chunk
  constexpr int CN = CE * NN;                              // nodes per chunk
  constexpr int QPC = (CN + kThreads - 1) / kThreads;      // nodes per thread per chunk
  // chunks per batch: every load of a batch is issued before its first
  // store, so a batch should keep enough bytes in flight (FP32 takes two)
  constexpr int BC = (sizeof(T) == 4 && QPC <= 2) ? 2 : 1;
  constexpr int NQ = BC * QPC;
  __shared__ double sred[kThreads / 64];
  if (scal[S_DONE] != 0.0) return;
  const T alpha = (T)scal[S_ALPHA];
  double rho = 0.0, nrm = 0.0;
  // each (XCD-renumbered) block walks a contiguous range of chunks
  const size_t nchunks = (nelems + CE - 1) / CE;
  const size_t cpb = (nchunks + gridDim.x - 1) / gridDim.x;
  const size_t c0 = xcd_block() * cpb, c1 = c0 + cpb < nchunks ? c0 + cpb : nchunks;
  // box coordinates of the walk's next element (chunks of one element)
  int ecw[3] = {0, 0, 0};
  if (CE == 1) gf::box_elem_coords(topo, c0, ecw);
  for (size_t c = c0; c < c1; c += BC) {
    I gs[NQ];
    T dv[NQ], xo[NQ], wo[NQ], ro[NQ], qm[NQ][8];
    int cnt[NQ];
    bool ok[NQ];
#pragma unroll
    for (int bc = 0; bc < BC; bc++) {
      const size_t cc = c + bc;
      int ec0[3];
      if (CE == 1) {
        ec0[0] = ecw[0];
        ec0[1] = ecw[1];
        ec0[2] = ecw[2];
        gf::box_elem_next(topo, ecw);
      } else {
        gf::box_elem_coords(topo, cc * CE, ec0);
      }
      const gf::BoxElemDeltas d0 = gf::box_elem_deltas(topo, N, ec0);  // uniform when CE == 1
#pragma unroll
      for (int qq = 0; qq < QPC; qq++) {
        const int s = bc * QPC + qq;
        const int q = qq * kThreads + (int)threadIdx.x;
        const int el = CE == 1 ? 0 : q / NN;
        const int rr = CE == 1 ? q : q - el * NN;
        const size_t e = cc * CE + el;
        ok[s] = cc < c1 && q < CN && e < nelems;
        gf::BoxElemDeltas de = d0;
        if (CE > 1 && el) {
          int ec[3];
          gf::box_elem_coords(topo, e, ec);
          de = gf::box_elem_deltas(topo, N, ec);
        }
        const int i = rr % N, j = (rr / N) % N, k = rr / (N * N);
        // out-of-range slots read node 0 (always valid) and are not stored
        const I g = ok[s] ? (I)(e * NN + rr) : (I)0;
        gs[s] = g;
        I mem[8];
        if (ok[s]) {
          cnt[s] = gf::box_members<I>(de, N, g, i, j, k, mem);
        } else {
          cnt[s] = 1;
#pragma unroll
          for (int m2 = 0; m2 < 8; m2++) mem[m2] = (I)0;
        }
        dv[s] = dinv ? dinv[g] : T(1);
        xo[s] = x[g];
        wo[s] = w[g];
        ro[s] = r[g];
        gf::box_load8m<I, T>(qv, mem, cnt[s], qm[s]);
      }
    }
#pragma unroll
    for (int s = 0; s < NQ; s++) {
      if (!ok[s]) continue;
      const I g = gs[s];
      const T qa = gf::box_sum8z<T>(qm[s], cnt[s]);
      const T xv = (T)1 * xo[s] + alpha * wo[s];
      x[g] = xv;
      const T rv = (T)1 * ro[s] + (-alpha) * qa;
      r[g] = rv;
      const T z = dinv ? dv[s] * rv : rv;
      const double im = gf::box_inv(cnt[s]);
      rho += (double)rv * (double)z * im;
      const double rd = (double)rv;
      if (NORM == GF_NORM_INF) nrm = fmax(nrm, fabs(rd));
      else if (NORM == GF_NORM_EUC) nrm += rd * rd;
      else if (NORM == GF_NORM_L2) nrm += mass[g] * rd * rd;
      else if (NORM == GF_NORM_L1) nrm += mass[g] * fabs(rd);
      else nrm += rd * rd * im;
    }
  }
  double a = gf::block_reduce<false>(rho, sred);
  double b = NORM == GF_NORM_INF ? gf::block_reduce<true>(nrm, sred)
                                 : gf::block_reduce<false>(nrm, sred);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = a;
    part[2 * blockIdx.x + 1] = b;
  }
}

// 16-byte vector of T (4 floats or 2 doubles).
template <typename T>
struct Vec16;
template <>
struct Vec16<float> {
  using V = float4;
  static constexpr int R = 4;
  __device__ static float get(const V &v, int n) {
    return n == 0 ? v.x : (n == 1 ? v.y : (n == 2 ? v.z : v.w));
  }
  __device__ static void set(V &v, int n, float a) {
    if (n == 0) v.x = a;
    else if (n == 1) v.y = a;
    else if (n == 2) v.z = a;
    else v.w = a;
  }
};
template <>
struct Vec16<double> {
  using V = double2;
  static constexpr int R = 2;
  __device__ static double get(const V &v, int n) { return n == 0 ? v.x : v.y; }
  __device__ static void set(V &v, int n, double a) {
    if (n == 0) v.x = a;
    else v.y = a;
  }
};

// True when k_cg_update_boxv handles order N in precision T: a node row
// splits into at least two 16-byte runs and a workgroup holds whole elements.
template <typename T, int N>
constexpr bool boxv_ok() {
  return N % Vec16<T>::R == 0 && N > Vec16<T>::R &&
         kThreads % (N * N * N / Vec16<T>::R) == 0;
}

// k_cg_update_box with each lane working a run of R = 16/sizeof(T)
// consecutive nodes along x (one 16-byte load or store per vector), so the
// wave issues a quarter (FP32) or half (FP64) of the memory instructions.
// The group of a node is the product of its partner choices per direction:
// the run's y, z and yz partners are runs of the neighbouring elements at the
// same x offset (16-byte loads), and only the run's first or last node can
// have an x partner (scalar loads).  Members are summed in the order
// (z side, y side, x side), lower side first, where the lower side of a
// direction is the copy with the smaller global index; because the element
// index dominates the global index, that order is the ascending order of the
// group's global indices, GGFX's summation order (ggfx.hpp:346-443), so the
// result equals k_cg_update_box's bit for bit.
template <typename T, int NORM, int N, typename I>
__global__ __launch_bounds__(kThreads) void k_cg_update_boxv(
    T *__restrict__ x, const T *__restrict__ w, T *__restrict__ r, const T *__restrict__ qv,
    const T *__restrict__ dinv, const double *__restrict__ mass, gf::BoxTopo topo, double *scal,
    double *__restrict__ part, size_t nelems, const T *__restrict__ dtab,
    const unsigned char *__restrict__ deq) {
  using VT = Vec16<T>;
  using V = typename VT::V;
  constexpr int R = VT::R;
  constexpr int NN = N * N * N;
  constexpr int RPR = N / R;           // runs per node row
  constexpr int RPE = NN / R;          // runs per element
  constexpr int EPP = kThreads / RPE;  // elements per workgroup pass
  __shared__ double sred[kThreads / 64];
  if (scal[S_DONE] != 0.0) return;
  const T alpha = (T)scal[S_ALPHA];
  double rho = 0.0, nrm = 0.0;
  const int el = (int)threadIdx.x / RPE, rr = (int)threadIdx.x - el * RPE;
  const int ir = rr % RPR, j = (rr / RPR) % N, k = rr / (RPR * N);
  const int i0 = ir * R;
  // the run node that can have an x partner: the row's first or last node
  const int xn = ir == 0 ? 0 : (ir == RPR - 1 ? R - 1 : -1);
  const size_t npass = (nelems + EPP - 1) / EPP;
  const size_t ppb = (npass + gridDim.x - 1) / gridDim.x;
  const size_t c0 = xcd_block() * ppb, c1 = c0 + ppb < npass ? c0 + ppb : npass;
  for (size_t c = c0; c < c1; c++) {
    const size_t e = c * EPP + el;
    if (e >= nelems) continue;
    int ec[3];
    gf::box_elem_coords(topo, e, ec);
    const gf::BoxElemDeltas d = gf::box_elem_deltas(topo, N, ec);
    const I g0 = (I)(e * NN) + (I)(k * N * N + j * N + i0);
    const I dy = j == 0 ? (I)d.lo[1] : (j == N - 1 ? (I)d.hi[1] : (I)0);
    const I dz = k == 0 ? (I)d.lo[2] : (k == N - 1 ? (I)d.hi[2] : (I)0);
    const I dx = xn == 0 ? (I)d.lo[0] : (xn == R - 1 ? (I)d.hi[0] : (I)0);
    const bool py = dy != 0, pz = dz != 0, px = dx != 0;
    // every load of the run before its first store
    const V xo = *(const V *)(x + g0);
    const V wo = *(const V *)(w + g0);
    const V ro = *(const V *)(r + g0);
    V dv;
    if (dinv)  // the Jacobi values from the table where the element's equal it
      dv = (dtab && deq[e]) ? *(const V *)(dtab + (g0 - (I)(e * NN))) : *(const V *)(dinv + g0);
    const V q0 = *(const V *)(qv + g0);
    V qy = {}, qz = {}, qyz = {};
    if (py) qy = *(const V *)(qv + g0 + dy);
    if (pz) qz = *(const V *)(qv + g0 + dz);
    if (py && pz) qyz = *(const V *)(qv + g0 + dy + dz);
    T sx = T(0), sxy = T(0), sxz = T(0), sxyz = T(0);
    if (px) {
      const I gx = g0 + (I)xn + dx;
      sx = qv[gx];
      if (py) sxy = qv[gx + dy];
      if (pz) sxz = qv[gx + dz];
      if (py && pz) sxyz = qv[gx + dy + dz];
    }
    // the partner side is the lower one when its offset is negative
    const bool ysw = dy < 0, zsw = dz < 0, xsw = dx < 0;
    V xv, rv;
#pragma unroll
    for (int n = 0; n < R; n++) {
      // t[side z][side y][side x], side 0 = own copy, 1 = partner
      T t[2][2][2];
      t[0][0][0] = VT::get(q0, n);
      t[0][1][0] = VT::get(qy, n);
      t[1][0][0] = VT::get(qz, n);
      t[1][1][0] = VT::get(qyz, n);
      const bool hx = (n == 0 || n == R - 1) && n == xn && px;
      t[0][0][1] = hx ? sx : T(0);
      t[0][1][1] = hx ? sxy : T(0);
      t[1][0][1] = hx ? sxz : T(0);
      t[1][1][1] = hx ? sxyz : T(0);
      const bool xs = hx && xsw;
      // canonical order: lower side first in z, then y, then x; absent
      // partners contribute +0 (see box_sum8z)
      T sum = T(0);
#pragma unroll
      for (int cz = 0; cz < 2; cz++)
#pragma unroll
        for (int cy = 0; cy < 2; cy++)
#pragma unroll
          for (int cx = 0; cx < 2; cx++) {
            const int sz = cz ^ (int)zsw, sy = cy ^ (int)ysw, sxi = cx ^ (int)xs;
            sum = sum + t[sz][sy][sxi];
          }
      const int cnt = (1 + (int)py) * (1 + (int)pz) * (1 + (int)hx);
      const T qa = cnt == 1 ? t[0][0][0] : sum;
      const T xn1 = (T)1 * VT::get(xo, n) + alpha * VT::get(wo, n);
      VT::set(xv, n, xn1);
      const T rn1 = (T)1 * VT::get(ro, n) + (-alpha) * qa;
      VT::set(rv, n, rn1);
      const T z = dinv ? VT::get(dv, n) * rn1 : rn1;
      const double im = gf::box_inv(cnt);
      rho += (double)rn1 * (double)z * im;
      const double rd = (double)rn1;
      if (NORM == GF_NORM_INF) nrm = fmax(nrm, fabs(rd));
      else if (NORM == GF_NORM_EUC) nrm += rd * rd;
      else if (NORM == GF_NORM_L2) nrm += mass[g0 + n] * rd * rd;
      else if (NORM == GF_NORM_L1) nrm += mass[g0 + n] * fabs(rd);
      else nrm += rd * rd * im;
    }
    *(V *)(x + g0) = xv;
    *(V *)(r + g0) = rv;
  }
  double a = gf::block_reduce<false>(rho, sred);
  double b = NORM == GF_NORM_INF ? gf::block_reduce<true>(nrm, sred)
                                 : gf::block_reduce<false>(nrm, sred);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = a;
    part[2 * blockIdx.x + 1] = b;
  }
}

template <typename T, int NORM, int N>
int launch_update_box_n(gf_mesh *m, CGVecs<T> &v, double *part) {
  if constexpr (boxv_ok<T, N>()) {
    if (m->ndof < ((size_t)1 << 31))
      hipLaunchKernelGGL((k_cg_update_boxv<T, NORM, N, int32_t>), dim3(kUpdBlocks), dim3(kThreads),
                         0, m->ctx->stream, v.x, v.w, v.r, v.q, v.dinv, m->mass, m->box, m->scal,
                         part, m->nelems, v.dtab, v.deq);
    else
      hipLaunchKernelGGL((k_cg_update_boxv<T, NORM, N, int64_t>), dim3(kUpdBlocks), dim3(kThreads),
                         0, m->ctx->stream, v.x, v.w, v.r, v.q, v.dinv, m->mass, m->box, m->scal,
                         part, m->nelems, v.dtab, v.deq);
    return GF_OK;
  }
  // 32-bit node indices whenever every index of the mesh fits
  if (m->ndof < ((size_t)1 << 31))
    hipLaunchKernelGGL((k_cg_update_box<T, NORM, N, int32_t>), dim3(kUpdBlocks), dim3(kThreads), 0,
                       m->ctx->stream, v.x, v.w, v.r, v.q, v.dinv, m->mass, m->box, m->scal, part,
                       m->nelems);
  else
    hipLaunchKernelGGL((k_cg_update_box<T, NORM, N, int64_t>), dim3(kUpdBlocks), dim3(kThreads), 0,
                       m->ctx->stream, v.x, v.w, v.r, v.q, v.dinv, m->mass, m->box, m->scal, part,
                       m->nelems);
  return GF_OK;
}

}  // namespace gfs

#define GF_K3D_UPD(T, N)                                                              \
  template int launch_update_box_n<T, GF_NORM_INF, N>(gf_mesh *, CGVecs<T> &, double *); \
  template int launch_update_box_n<T, GF_NORM_EUC, N>(gf_mesh *, CGVecs<T> &, double *); \
  template int launch_update_box_n<T, GF_NORM_L2, N>(gf_mesh *, CGVecs<T> &, double *);  \
  template int launch_update_box_n<T, GF_NORM_L1, N>(gf_mesh *, CGVecs<T> &, double *);  \
  template int launch_update_box_n<T, GF_NORM_ASSEMBLED_L2, N>(gf_mesh *, CGVecs<T> &, double *);

#define GF_K3D_INSTANTIATE(N)                                                                \
  template int launch_stage3p<N>(gf_mesh *, const StageArgs &);                              \
  template int launch_advect3p<N>(gf_mesh *, const double *, const double *const *, double *); \
  template int launch_grad3p<N>(gf_mesh *, const double *, double *const *, const double *);  \
  template int launch_stage3b<N>(gf_mesh *, double *const *, double *const *, double *const *, \
                                 double *const *, double, double, double, double, int, int); \
  template int launch_rk_out_box<N>(gf_mesh *, double *const *, double *const *);             \
  template int helm3c_d<N>(gf_mesh *, double, const double *, const double *, double,         \
                           const double *, double *);                                        \
  template int helm3c_f<N>(gf_mesh *, float, const float *, float, const float *, float *);   \
  template int cgapply3c_d<N>(gf_mesh *, const CGApply3Args &);                              \
  template int cgapply3c_f<N>(gf_mesh *, const CGApply3Args &);                              \
  GF_K3D_UPD(float, N)                                                                       \
  GF_K3D_UPD(double, N)
