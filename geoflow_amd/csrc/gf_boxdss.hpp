// gf_boxdss.hpp -- direct stiffness summation by gather on a structured box.
//
// On a box grid (elements in x-fastest linear order, x/y/z element counts
// ne[], optional periodicity per direction) the GGFX coincidence group of a
// node follows from its position alone: in each direction a node with index
// 0 also lives at index N-1 of the previous element, and one with index N-1
// at index 0 of the next element (wrapping around when that direction is
// periodic).  The group is the product of these per-direction choices, at
// most 8 nodes.  A consumer kernel can therefore assemble a local vector on
// the fly ("gather"): every copy of a shared node reads all members of its
// group, through a halo of its element in LDS, and sums them in pairs along x,
// then y, then z (HaloSum).  GGFX::doOp accumulates a group in ascending
// global index (std::accumulate from 0 over the sorted members,
// src/cdg/comm/ggfx.hpp:346-443), so the two agree to rounding.  All copies
// compute the same sum, so the result stays continuous, and no separate DSS
// pass or index array is needed.  gf_mesh_create enables this only after checking
// on the host that the groups it produces equal the GGFX groups of the mesh.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace gf {

struct BoxTopo {
  int ne[3];     // elements per direction
  int per[3];    // 1 if the direction is periodic
  int fmask[6];  // 1 if the nodes of face x0,x1,y0,y1,z0,z1 are masked (Dirichlet-type)
};

// Boundary mask of node (i,j,k) (N per direction) of the element at box
// coordinates ec[]: 0 on a masked domain face, else 1 -- the mask of
// GGrid::init_bc_info for a box whose face types are fmask[].
__host__ __device__ __forceinline__ bool box_masked(const BoxTopo &t, int N, const int (&ec)[3],
                                                    int i, int j, int k) {
  const int nc[3] = {i, j, k};
  bool mk = false;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    mk = mk || (nc[d] == 0 && ec[d] == 0 && t.fmask[2 * d]);
    mk = mk || (nc[d] == N - 1 && ec[d] == t.ne[d] - 1 && t.fmask[2 * d + 1]);
  }
  return mk;
}

// Box coordinates (ex, ey, ez) of element e (32-bit division whenever the
// operands fit, which avoids the long 64-bit division sequence).
__host__ __device__ __forceinline__ void box_elem_coords(const BoxTopo &t, size_t e, int (&ec)[3]) {
  const size_t nxy = (size_t)t.ne[0] * t.ne[1];
  if (e < ((size_t)1 << 32) && nxy < ((size_t)1 << 32)) {
    const uint32_t e32 = (uint32_t)e, nx = (uint32_t)t.ne[0], n2 = (uint32_t)nxy;
    const uint32_t z = e32 / n2, rem = e32 - z * n2, y = rem / nx;
    ec[2] = (int)z;
    ec[1] = (int)y;
    ec[0] = (int)(rem - y * nx);
    return;
  }
  ec[2] = (int)(e / nxy);
  const size_t rem = e - (size_t)ec[2] * nxy;
  ec[1] = (int)(rem / (size_t)t.ne[0]);
  ec[0] = (int)(rem - (size_t)ec[1] * t.ne[0]);
}

// Advances box coordinates to those of the next element in linear order.
__host__ __device__ __forceinline__ void box_elem_next(const BoxTopo &t, int (&ec)[3]) {
  if (++ec[0] == t.ne[0]) {
    ec[0] = 0;
    if (++ec[1] == t.ne[1]) {
      ec[1] = 0;
      ++ec[2];
    }
  }
}

// Members of the group of node (i,j,k) (N nodes per direction) of the element
// at box coordinates ec[], whose own global index is gself; written to g[] in
// ascending order, g[m] = SIZE_MAX for m >= count; returns the count.
//
// In direction d the partner differs from the node by the index offset
// delta_d (0 if there is none).  Global indices are e*N^3 + k*N^2 + j*N + i
// with e = ex + nx*(ey + ny*ez), i.e. lexicographic in (ez,ey,ex,k,j,i), so
// the non-zero |delta_d| sorted in decreasing order are superincreasing (each
// exceeds the sum of the smaller ones).  With lo the smallest member, member
// m = lo + sum_s bit_s(m) |delta|_(s) therefore increases with m.
__host__ __device__ __forceinline__ int box_group(const BoxTopo &t, int N, const int (&ec)[3],
                                                  size_t gself, int i, int j, int k,
                                                  size_t (&g)[8]) {
  const int nc[3] = {i, j, k};
  const int64_t NN = (int64_t)N * N * N;
  const int64_t es[3] = {NN, (int64_t)t.ne[0] * NN, (int64_t)t.ne[0] * t.ne[1] * NN};
  const int64_t ns[3] = {1, N, (int64_t)N * N};
  int64_t lo = (int64_t)gself;
  int64_t a[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    int64_t dl = 0;
    if (nc[d] == 0 && (ec[d] > 0 || t.per[d])) {
      const int oe = ec[d] > 0 ? ec[d] - 1 : t.ne[d] - 1;
      dl = (int64_t)(oe - ec[d]) * es[d] + (int64_t)(N - 1) * ns[d];
    } else if (nc[d] == N - 1 && (ec[d] < t.ne[d] - 1 || t.per[d])) {
      const int oe = ec[d] < t.ne[d] - 1 ? ec[d] + 1 : 0;
      dl = (int64_t)(oe - ec[d]) * es[d] - (int64_t)(N - 1) * ns[d];
    }
    lo += dl < 0 ? dl : 0;
    a[d] = dl < 0 ? -dl : dl;
  }
  // decreasing magnitudes (absent directions, 0, last)
  auto cs = [](int64_t &x, int64_t &y) {
    const int64_t h = x > y ? x : y, l = x > y ? y : x;
    x = h;
    y = l;
  };
  cs(a[0], a[1]);
  cs(a[1], a[2]);
  cs(a[0], a[1]);
  const int na = (a[0] != 0) + (a[1] != 0) + (a[2] != 0);
  const int cnt = 1 << na;
#pragma unroll
  for (int m = 0; m < 8; m++) {
    int64_t v = lo;
    if (na >= 1) v += ((m >> (na - 1)) & 1) ? a[0] : 0;
    if (na >= 2) v += ((m >> (na - 2)) & 1) ? a[1] : 0;
    if (na >= 3) v += (m & 1) ? a[2] : 0;
    g[m] = m < cnt ? (size_t)v : SIZE_MAX;
  }
  return cnt;
}

// Partner offsets of one element: in direction d a node with index 0 has its
// partner at offset lo[d] (index N-1 of the previous element), a node with
// index N-1 at hi[d] (index 0 of the next element); 0 where there is none.
// They depend only on the element, so kernels form them once per element.
struct BoxElemDeltas {
  int64_t lo[3], hi[3];
};

__host__ __device__ __forceinline__ BoxElemDeltas box_elem_deltas(const BoxTopo &t, int N,
                                                                  const int (&ec)[3]) {
  const int64_t NN = (int64_t)N * N * N;
  const int64_t es[3] = {NN, (int64_t)t.ne[0] * NN, (int64_t)t.ne[0] * t.ne[1] * NN};
  const int64_t ns[3] = {1, N, (int64_t)N * N};
  BoxElemDeltas d;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    d.lo[c] = 0;
    d.hi[c] = 0;
    if (ec[c] > 0 || t.per[c]) {
      const int oe = ec[c] > 0 ? ec[c] - 1 : t.ne[c] - 1;
      d.lo[c] = (int64_t)(oe - ec[c]) * es[c] + (int64_t)(N - 1) * ns[c];
    }
    if (ec[c] < t.ne[c] - 1 || t.per[c]) {
      const int oe = ec[c] < t.ne[c] - 1 ? ec[c] + 1 : 0;
      d.hi[c] = (int64_t)(oe - ec[c]) * es[c] - (int64_t)(N - 1) * ns[c];
    }
  }
  return d;
}

// Members of the group of node (i,j,k) with global index gself, from the
// element's partner offsets; ascending in g[0..count), count returned, and
// *own the slot of gself itself.  Same construction as box_group
// (superincreasing magnitudes), in index type I (int32_t when every index of
// the mesh fits, else int64_t), written without branches or per-slot
// selects: the non-zero magnitudes in ascending order b0 <= b1 <= b2 (0 where
// absent) weight bits 0, 1, 2 of the slot number, so slot m is
// lo + (m&1) b0 + (m&2) b1 + (m&4) b2, and the node's own slot has the bits of
// the directions whose partner lies below it.  Slots past the count repeat
// members (their weights are 0) and are never read.
template <typename I>
__host__ __device__ __forceinline__ int box_members_own(const BoxElemDeltas &d, int N, I gself,
                                                        int i, int j, int k, I (&g)[8], int *own) {
  static_assert(std::is_signed<I>::value, "partner offsets are signed");
  using U = typename std::make_unsigned<I>::type;
  const int nc[3] = {i, j, k};
  I lo = gself;
  U key[3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const I dl = nc[c] == 0 ? (I)d.lo[c] : (nc[c] == N - 1 ? (I)d.hi[c] : (I)0);
    lo += dl < 0 ? dl : (I)0;
    // 2 magnitude + (partner below) - 2 as unsigned: an absent direction
    // (magnitude 0) wraps to the largest key and sorts last; magnitudes are
    // distinct, so the sign bit never decides the order
    key[c] = ((((U)(dl < 0 ? -dl : dl)) << 1) | (U)(dl < 0)) - (U)2;
  }
  auto cs = [](U &x, U &y) {
    const U l = x < y ? x : y, h = x < y ? y : x;
    x = l;
    y = h;
  };
  cs(key[0], key[1]);
  cs(key[1], key[2]);
  cs(key[0], key[1]);
  const I b0 = (I)((key[0] + (U)2) >> 1), b1 = (I)((key[1] + (U)2) >> 1),
          b2 = (I)((key[2] + (U)2) >> 1);
  *own = (int)(key[0] & 1) | ((int)(key[1] & 1) << 1) | ((int)(key[2] & 1) << 2);
  const int na = (b0 != 0) + (b1 != 0) + (b2 != 0);
  const I l1 = lo + b1;
  g[0] = lo;
  g[1] = lo + b0;
  g[2] = l1;
  g[3] = l1 + b0;
  g[4] = lo + b2;
  g[5] = g[4] + b0;
  g[6] = l1 + b2;
  g[7] = g[6] + b0;
  return 1 << na;
}

template <typename I>
__host__ __device__ __forceinline__ int box_members(const BoxElemDeltas &d, int N, I gself, int i,
                                                    int j, int k, I (&g)[8]) {
  int own;
  return box_members_own<I>(d, N, gself, i, j, k, g, &own);
}

// ---------------------------------------------------------------------------
// Element halo in LDS for a gather Smooth (N^2 threads per element, thread
// l = a + N b owning the column (a, b, .)).  Instead of each node loading its
// group members from global memory -- loads under per-lane conditions, each
// waited for in turn -- the element's threads load its own values and every
// partner value it can need with unconditional loads, all in flight
// together, and the group sums read LDS.  Layout (values of T):
//   own values       [0, N^3)     i + N j + N^2 k
//   faces            FACE + N^2 f + p + N q, f = 2 d + s (d the face
//                    direction, s = 1 for the upper face), (p, q) the node's
//                    other two indices in increasing direction order
//   edges            EDGE + N e + r, e = 4 pd + 2 s1 + s2 for the direction
//                    pair pd (0: xy, 1: xz, 2: yz) with sides s1, s2, r the
//                    node's third index
//   corners          CORNER + sx + 2 sy + 4 sz
//   zeros            [ZERO, SIZE): +0, read for absent partners; as many as
//                    the stride of a column's face slots spans
// A halo slot holds the value at the partner node across that face, edge
// or corner (the offsets of box_elem_deltas added up); where the element has
// no partner the offset is 0, the slot holds an own value and is never read.
// ---------------------------------------------------------------------------
template <int N>
struct Halo {
  static constexpr int N2 = N * N, FACE = N * N * N, EDGE = FACE + 6 * N2,
                       CORNER = EDGE + 12 * N, ZERO = CORNER + 8, NZ = N * (N - 1) + 1,
                       SIZE = ZERO + NZ;
  static constexpr int ER = (12 * N + N2 - 1) / N2;  // edge rounds per thread
  static constexpr int CR = (8 + N2 - 1) / N2;       // corner rounds
  static constexpr int RQ = 6 + ER + CR;             // partner loads per thread
};

// f(std::integral_constant<int, B>), ..., f(std::integral_constant<int, E-1>):
// a loop whose index is a compile-time constant in the body.
template <int B, int E, typename F>
__host__ __device__ __forceinline__ void static_for(F &&f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

__device__ __forceinline__ int64_t halo_delta(const BoxElemDeltas &de, int d, int s) {
  return s ? de.hi[d] : de.lo[d];
}

// Offset from the element's first node read by load q (0 .. RQ-1) of thread
// l and the LDS slot it fills (-1: the thread has nothing to load in this
// round; it reads the element's first node instead, so every load is
// unconditional and in bounds).
template <int N>
__device__ __forceinline__ int64_t halo_src(const BoxElemDeltas &de, int l, int q, int *slot) {
  using H = Halo<N>;
  if (q < 6) {  // faces: the node's own offset is a function of l per face
    const int d = q >> 1, s = q & 1, p = l % N, r = l / N;
    const int own = d == 0 ? N * l + (N - 1) * s
                           : (d == 1 ? p + H::N2 * r + N * (N - 1) * s : l + H::N2 * (N - 1) * s);
    *slot = H::FACE + H::N2 * q + l;
    return own + halo_delta(de, d, s);
  }
  if (q < 6 + H::ER) {  // edges
    const int x = (q - 6) * H::N2 + l, e = x / N, r = x - e * N;
    if (e >= 12) {
      *slot = -1;
      return 0;
    }
    // pair pd: 0 (x, y), 1 (x, z), 2 (y, z), sides s1, s2; selects only,
    // so no array is indexed by a lane-dependent value
    const int pd = e >> 2, s1 = (e >> 1) & 1, s2 = e & 1;
    const int e1 = s1 ? N - 1 : 0, e2 = s2 ? N - 1 : 0;
    const int c0 = pd == 2 ? r : e1;
    const int c1 = pd == 0 ? e2 : (pd == 1 ? r : e1);
    const int c2 = pd == 0 ? r : e2;
    const int64_t dx = halo_delta(de, 0, s1), dy1 = halo_delta(de, 1, s1),
                  dy2 = halo_delta(de, 1, s2), dz = halo_delta(de, 2, s2);
    *slot = H::EDGE + x;
    return c0 + N * c1 + H::N2 * c2 + (pd == 0 ? dx + dy2 : (pd == 1 ? dx + dz : dy1 + dz));
  }
  const int c = (q - 6 - H::ER) * H::N2 + l;
  if (c >= 8) {  // corners
    *slot = -1;
    return 0;
  }
  const int sx = c & 1, sy = (c >> 1) & 1, sz = c >> 2;
  *slot = H::CORNER + c;
  return (N - 1) * (sx + N * sy + H::N2 * sz) + halo_delta(de, 0, sx) + halo_delta(de, 1, sy) +
         halo_delta(de, 2, sz);
}

// The partner values of field u for the element at ebase: RQ loads per
// thread into registers (halo_src), then their LDS slots in the halo hl and
// the zero slot; the element's own values, hl[0, N^3), are copied separately.
template <int N, typename T>
struct HaloRim {
  static constexpr int RQ = Halo<N>::RQ;
  T hv[RQ];
  int slot[RQ];
  __device__ __forceinline__ void issue(const T *__restrict__ u, const BoxElemDeltas &de,
                                        int64_t ebase, int l) {
#pragma unroll
    for (int q = 0; q < RQ; q++) hv[q] = u[ebase + halo_src<N>(de, l, q, &slot[q])];
  }
  __device__ __forceinline__ void store(T *hl, int l) const {
#pragma unroll
    for (int q = 0; q < RQ; q++)
      if (slot[q] >= 0) hl[slot[q]] = hv[q];
    if (l < Halo<N>::NZ) hl[Halo<N>::ZERO + l] = T(0);
  }
};

// True when halo_order's canonical order is GGFX's on this box at N nodes
// per direction: every partner offset in x smaller than every one in y, and
// the x and y ones together smaller than every z one (superincreasing in x,
// y, z).  An offset is the element stride less N - 1 node strides between
// neighbours, (ne - 1) element strides plus N - 1 node strides across a
// periodic wrap, and N - 1 node strides within an element that is its own
// periodic neighbour (ne = 1).
__host__ __device__ __forceinline__ bool box_halo_ok(const BoxTopo &t, int N) {
  const int64_t NN = (int64_t)N * N * N, ns[3] = {1, N, (int64_t)N * N};
  const int64_t es[3] = {NN, (int64_t)t.ne[0] * NN, (int64_t)t.ne[0] * t.ne[1] * NN};
  int64_t below = 0;  // sum of the largest offsets of the lower directions
  bool ok = true;
  for (int d = 0; d < 3; d++) {
    int64_t mn, mx;
    if (t.ne[d] == 1) {
      if (!t.per[d]) continue;  // no partners in this direction
      mn = mx = (N - 1) * ns[d];
    } else {
      mn = es[d] - (N - 1) * ns[d];
      mx = t.per[d] ? (int64_t)(t.ne[d] - 1) * es[d] + (N - 1) * ns[d] : mn;
    }
    ok = ok && below < mn;
    below += mx;
  }
  return ok;
}

// Per-thread constants of the group sums of the column (i, j, .): which x and
// y partners exist, whether they lie below, and the k-independent parts of
// their halo addresses (the zero slot where a partner is absent).
template <int N>
struct HaloCol {
  using H = Halo<N>;
  int i, j, xon, yon, nx, ny;
  int ax0, ay0, axy0;  // + k * (N xon), + k * (N yon), + k * (xon & yon)
  __device__ __forceinline__ HaloCol(const BoxElemDeltas &de, int i_, int j_) : i(i_), j(j_) {
    const int sx = i == N - 1, sy = j == N - 1;
    const int64_t dx = i == 0 ? de.lo[0] : (i == N - 1 ? de.hi[0] : 0);
    const int64_t dy = j == 0 ? de.lo[1] : (j == N - 1 ? de.hi[1] : 0);
    xon = dx != 0;
    yon = dy != 0;
    nx = dx < 0;
    ny = dy < 0;
    ax0 = xon ? H::FACE + H::N2 * sx + j : H::ZERO;
    ay0 = yon ? H::FACE + H::N2 * (2 + sy) + i : H::ZERO;
    axy0 = (xon & yon) ? H::EDGE + N * (2 * sx + sy) : H::ZERO;
  }
};

// The group of node (i, j, K) as halo addresses in canonical order (the layout's
// statement in GGFX's terms; the kernels sum with HaloSum) -- lower
// side first in z, then in y, then in x, the lower side of a direction being
// the copy with the smaller global index -- over the 2 x 2 (x 2 on the z
// faces) crossings, an absent partner's terms reading the zero slot, which
// adds +0 and leaves every sum as it is.  Every copy of a node
// has the same order.  Where box_halo_ok holds it is ascending global index,
// GGFX's order.  Returns the count of the group.
template <int N, int K>
__device__ __forceinline__ int halo_order(const HaloCol<N> &c, const BoxElemDeltas &de,
                                          int (&a)[8]) {
  using H = Halo<N>;
  const int own = c.i + N * c.j + H::N2 * K;
  const int ax = c.ax0 + K * N * c.xon, ay = c.ay0 + K * N * c.yon;
  const int axy = c.axy0 + K * (c.xon & c.yon);
  // within a y row, lower x first; then lower y row first
  const int l0 = c.nx ? ax : own, u0 = c.nx ? own : ax;
  const int l1 = c.nx ? axy : ay, u1 = c.nx ? ay : axy;
  int p[4] = {c.ny ? l1 : l0, c.ny ? u1 : u0, c.ny ? l0 : l1, c.ny ? u0 : u1};
  int zon = 0, nz = 0;
  int q[4] = {H::ZERO, H::ZERO, H::ZERO, H::ZERO};
  if (K == 0 || K == N - 1) {
    const int64_t dz = K == 0 ? de.lo[2] : de.hi[2];
    zon = dz != 0;
    nz = dz < 0;
    const int sz = K == N - 1, sx = c.i == N - 1, sy = c.j == N - 1;
    const int bz = zon ? H::FACE + H::N2 * (4 + sz) + c.i + N * c.j : H::ZERO;
    const int bxz = (zon & c.xon) ? H::EDGE + N * (4 + 2 * sx + sz) + c.j : H::ZERO;
    const int byz = (zon & c.yon) ? H::EDGE + N * (8 + 2 * sy + sz) + c.i : H::ZERO;
    const int bxyz = (zon & c.xon & c.yon) ? H::CORNER + sx + 2 * sy + 4 * sz : H::ZERO;
    const int m0 = c.nx ? bxz : bz, n0 = c.nx ? bz : bxz;
    const int m1 = c.nx ? bxyz : byz, n1 = c.nx ? byz : bxyz;
    q[0] = c.ny ? m1 : m0;
    q[1] = c.ny ? n1 : n0;
    q[2] = c.ny ? m0 : m1;
    q[3] = c.ny ? n0 : n1;
  }
#pragma unroll
  for (int m = 0; m < 4; m++) {
    a[m] = nz ? q[m] : p[m];
    a[4 + m] = nz ? p[m] : q[m];
  }
  return (1 + c.xon) * (1 + c.yon) * (1 + zon);
}

// Group sums of a column (i, j, .) from the halo:
//   (own + X) + (Y + XY)  [+ ((Z + XZ) + (YZ + XYZ)) on the z faces],
// X the x partner's value and so on, zeros where there is none.  Each copy of
// a node has the same pairs, at most exchanged, so all copies get the same
// sum bit for bit whatever the partners' order; the sums of 2, 4 and 8 equal
// values are exact.  A column's slots lie at fixed strides from one address
// per partner kind (absent partners: the zeros), so no address is formed per
// node.  Choosing the members' slots in GGFX order node by node instead took
// more instructions than the operator at small orders: RK3 on 19x14x11, p = 5
// 75 us a step against 66, FP32 CG at 20^3, p = 6 41 us an iteration against 37.
template <int N>
struct HaloSum {
  using H = Halo<N>;
  int x, y, xy, z[2], xz[2], yz[2], xyz[2];
  bool xon, yon, zon[2];
  double inv;  // 1 / (group size) off the z faces
  __device__ __forceinline__ HaloSum(const BoxElemDeltas &de, int i, int j) {
    const int sx = i == N - 1, sy = j == N - 1;
    xon = (i == 0 && de.lo[0] != 0) || (sx && de.hi[0] != 0);
    yon = (j == 0 && de.lo[1] != 0) || (sy && de.hi[1] != 0);
    const bool both = xon && yon;
    x = xon ? H::FACE + H::N2 * sx + j : H::ZERO;
    y = yon ? H::FACE + H::N2 * (2 + sy) + i : H::ZERO;
    xy = both ? H::EDGE + N * (2 * sx + sy) : H::ZERO;
#pragma unroll
    for (int s = 0; s < 2; s++) {
      zon[s] = (s ? de.hi[2] : de.lo[2]) != 0;
      z[s] = zon[s] ? H::FACE + H::N2 * (4 + s) + i + N * j : H::ZERO;
      xz[s] = zon[s] && xon ? H::EDGE + N * (4 + 2 * sx + s) + j : H::ZERO;
      yz[s] = zon[s] && yon ? H::EDGE + N * (8 + 2 * sy + s) + i : H::ZERO;
      xyz[s] = zon[s] && both ? H::CORNER + sx + 2 * sy + 4 * s : H::ZERO;
    }
    inv = (xon ? 0.5 : 1.0) * (yon ? 0.5 : 1.0);
  }
  // 1 / (group size) of node K, exact
  template <int K>
  __device__ __forceinline__ double inv_k() const {
    if (K == 0 || K == N - 1) return zon[K != 0] ? 0.5 * inv : inv;
    return inv;
  }
  // sum over the group of node K of f(value, present)
  template <int K, typename T, typename F>
  __device__ __forceinline__ T sum(const T *h, T own, F &&f) const {
    T s = (f(own, true) + f(h[x + K * N], xon)) +
          (f(h[y + K * N], yon) + f(h[xy + K], xon && yon));
    if constexpr (K == 0 || K == N - 1) {
      constexpr int e = K != 0;
      s = s + ((f(h[z[e]], zon[e]) + f(h[xz[e]], zon[e] && xon)) +
               (f(h[yz[e]], zon[e] && yon) + f(h[xyz[e]], zon[e] && xon && yon)));
    }
    return s;
  }
  template <int K, typename T>
  __device__ __forceinline__ T sum(const T *h, T own) const {
    return sum<K>(h, own, [](T v, bool) { return v; });
  }
};

// HaloCol, halo_order and box_halo_ok state the halo's layout in GGFX's terms,
// and are run by the CPU checks of the halo; no kernel uses them.  The N = 8
// instances under their own names.
constexpr int kHalo8 = Halo<8>::SIZE;
constexpr int kHalo8Zero = Halo<8>::ZERO;
template <typename T>
using Halo8Rim = HaloRim<8, T>;
using Halo8Col = HaloCol<8>;
__host__ __device__ __forceinline__ bool box_halo8_ok(const BoxTopo &t) {
  return box_halo_ok(t, 8);
}
template <int K>
__device__ __forceinline__ int halo8_order(const Halo8Col &c, const BoxElemDeltas &de,
                                           int (&a)[8]) {
  return halo_order<8, K>(c, de, a);
}

}  // namespace gf
