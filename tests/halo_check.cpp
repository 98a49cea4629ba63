// CPU check of the element halo (gf_boxdss.hpp) at every order N = 2..10: the
// halo of each element is filled with global node indices thread by thread
// (own values, HaloRim), and for every node the slots of halo_order, absent
// partners skipped, must be the members of box_group, in an order that every
// copy of the node shares and that is ascending wherever box_halo_ok says so;
// only the z faces may use the last four terms.  With random values in place of
// the indices, HaloSum's group sums must be the same bit for bit at every copy
// of a node and equal the members' sum to rounding, eight equal members must
// average to themselves, and inv_k must be 1 / (group size).  Exit status 0 when
// everything holds.
#define __host__
#define __device__
#define __forceinline__ inline
#define HIP_INCLUDE_HIP_HIP_RUNTIME_H
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <map>
#include <vector>

#include "gf_boxdss.hpp"

template <int N>
size_t check_sums(const gf::BoxTopo &t) {
  using H = gf::Halo<N>;
  const size_t nel = (size_t)t.ne[0] * t.ne[1] * t.ne[2], nn = (size_t)N * N * N, n = nel * nn;
  std::vector<double> u(n), hl(H::SIZE), ones(H::SIZE);
  unsigned r = 12345;
  for (double &v : u) {
    r = r * 1664525u + 1013904223u;
    v = (double)r / 4294967296.0 - 0.5;
  }
  size_t wrong = 0;
  std::map<size_t, double> sums;
  for (size_t e = 0; e < nel; e++) {
    int ec[3];
    gf::box_elem_coords(t, e, ec);
    const gf::BoxElemDeltas de = gf::box_elem_deltas(t, N, ec);
    for (size_t q = 0; q < nn; q++) hl[q] = u[e * nn + q];
    for (int l = 0; l < N * N; l++) {
      gf::HaloRim<N, double> L;
      L.issue(u.data(), de, (int64_t)(e * nn), l);
      L.store(hl.data(), l);
    }
    for (size_t q = 0; q < H::SIZE; q++) ones[q] = (int)q < H::ZERO ? u[0] : 0.0;
    for (int l = 0; l < N * N; l++) {
      const int i = l % N, j = l / N;
      const gf::HaloSum<N> hs(de, i, j);
      gf::static_for<0, N>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        const size_t q = e * nn + i + N * j + (size_t)N * N * k;
        size_t g[8];
        const int cnt = gf::box_group(t, N, ec, q, i, j, k, g);
        double ref = 0.0;
        for (int s = 0; s < cnt; s++) ref += u[g[s]];
        const double v = hs.template sum<k>(hl.data(), u[q]);
        int np = 0;
        hs.template sum<k>(hl.data(), u[q], [&](double w, bool on) {
          np += on;
          return on ? w : 0.0;
        });
        auto it = sums.find(g[0]);
        if (it == sums.end()) sums[g[0]] = v;
        else wrong += !(it->second == v);
        wrong += !(std::fabs(v - ref) <= 1e-15) || np != cnt ||
                 hs.template inv_k<k>() != 1.0 / cnt ||
                 hs.template sum<k>(ones.data(), u[0]) * hs.template inv_k<k>() != u[0];
      });
    }
  }
  return wrong;
}

template <int N>
size_t check(const gf::BoxTopo &t) {
  using H = gf::Halo<N>;
  const size_t nel = (size_t)t.ne[0] * t.ne[1] * t.ne[2], nn = (size_t)N * N * N, n = nel * nn;
  std::vector<double> gid(n), hl(H::SIZE);
  for (size_t q = 0; q < n; q++) gid[q] = (double)q;
  const bool hok = gf::box_halo_ok(t, N);
  size_t wrong = 0;
  std::map<size_t, std::vector<size_t>> order;  // by the group's smallest member
  for (size_t e = 0; e < nel; e++) {
    int ec[3];
    gf::box_elem_coords(t, e, ec);
    const gf::BoxElemDeltas de = gf::box_elem_deltas(t, N, ec);
    for (double &h : hl) h = -1.0;
    for (size_t q = 0; q < nn; q++) hl[q] = gid[e * nn + q];
    for (int l = 0; l < N * N; l++) {
      int slot;
      for (int q = 0; q < H::RQ; q++) {  // every load in bounds
        const int64_t o = (int64_t)(e * nn) + gf::halo_src<N>(de, l, q, &slot);
        wrong += o < 0 || o >= (int64_t)n || slot >= H::ZERO;
      }
      if (wrong) return wrong;
      gf::HaloRim<N, double> L;
      L.issue(gid.data(), de, (int64_t)(e * nn), l);
      L.store(hl.data(), l);
    }
    for (int l = 0; l < N * N; l++) {
      const int i = l % N, j = l / N;
      const gf::HaloCol<N> hc(de, i, j);
      gf::static_for<0, N>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        size_t g[8];
        const int cnt =
            gf::box_group(t, N, ec, e * nn + i + N * j + (size_t)N * N * k, i, j, k, g);
        int ad[8];
        bool ok = gf::halo_order<N, k>(hc, de, ad) == cnt && hl[H::ZERO] == 0.0;
        std::vector<size_t> m;
        for (int s = 0; s < 8; s++) {
          if (ad[s] == H::ZERO) continue;
          ok = ok && ad[s] >= 0 && ad[s] < H::ZERO && hl[ad[s]] >= 0.0 &&
               (s < 4 || k == 0 || k == N - 1);
          m.push_back((size_t)hl[ad[s]]);
        }
        ok = ok && (int)m.size() == cnt;
        if (hok) ok = ok && std::equal(m.begin(), m.end(), g);
        auto it = order.find(g[0]);
        if (it == order.end()) order[g[0]] = m;
        else ok = ok && it->second == m;
        std::sort(m.begin(), m.end());
        ok = ok && (int)m.size() == cnt && std::equal(m.begin(), m.end(), g);
        wrong += !ok;
      });
    }
  }
  return wrong + check_sums<N>(t);
}

int main() {
  const int nes[][3] = {{3, 3, 3}, {1, 1, 1}, {2, 1, 3}, {1, 3, 2}, {3, 2, 1}, {2, 2, 2}, {1, 1, 2}};
  int bad = 0;
  for (const auto &ne : nes)
    for (int per = 0; per < 2; per++) {
      gf::BoxTopo t = {};
      for (int d = 0; d < 3; d++) {
        t.ne[d] = ne[d];
        t.per[d] = per;
      }
      const size_t w[] = {check<2>(t), check<3>(t), check<4>(t), check<5>(t), check<6>(t),
                          check<7>(t), check<8>(t), check<9>(t), check<10>(t)};
      for (int k = 0; k < 9; k++)
        if (w[k]) {
          printf("N=%d ne=%d,%d,%d per=%d: %zu wrong\n", k + 2, ne[0], ne[1], ne[2], per, w[k]);
          bad++;
        }
    }
  return bad ? 1 : 0;
}
