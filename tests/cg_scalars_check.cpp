// CPU check of the CG driver's reading of its final scalars (gf_solve.hip), run
// against a stand-in for the HIP runtime that this program defines and
// libgeoflow_hip.so binds to.  Kernels are not run.  The stand-in of the apply
// kernel that ends the iteration shows its done flags in the mapped mirror at
// once, as a kernel that is still running may, and the scalars beside them only
// when the stream has been waited for (or an event recorded behind the kernel):
// a driver that reads them on sight of the flags reads those of before.
//   cg_scalars_check single|batched fp64|mixed
// Exit status 0 when every result is that of the scalars the kernels left.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "geoflow_hip.h"
#include "gf_solve_common.hpp"

using gfs::CGCtl;
using gfs::kCGSet;

namespace {

constexpr int kEnd = 6;            // the apply that finds the iteration done: in the second batch
const double kRhom = 4.0, kRho32 = 3.0, kRnorm = 1e-3;  // of system 0; system s adds s

struct Pending {
  long seq;
  std::function<void()> write;
};
// kernels by their host stubs, filled by the library before main's statics exist
std::map<const void *, std::string> &names() {
  static std::map<const void *, std::string> m;
  return m;
}
std::vector<Pending> pending;
std::vector<double> betas;  // S_BETA of every cycle's first apply, system 0
long seq = 0;
int loops = 0, fin = 0;
int nsys = 1;

void complete(long upto) {
  std::vector<Pending> rest;
  for (auto &p : pending) {
    if (p.seq <= upto) p.write();
    else rest.push_back(p);
  }
  pending.swap(rest);
}
struct Event {
  long seq = 0;
};

// iterations of system s in its n-th cycle
int iters(int s, int n) { return 5 + 2 * s + n; }

void apply(const CGCtl &c) {
  static int it = 0;
  static double epoch = 0.0;
  if (c.epoch != epoch) {
    epoch = c.epoch;
    it = 0;
    loops++;
    betas.push_back(c.scal[kCGSet * c.par + gfs::S_BETA]);
  }
  if (++it != kEnd) return;
  double *m = c.mirror;
  const double e = c.epoch;
  const int n = loops;
  for (int s = 0; s < nsys; s++) m[s * kCGSet + gfs::S_DONE] = e;
  double *resid = c.resid;
  pending.push_back({seq, [=]() {
                       for (int s = 0; s < nsys; s++) {
                         double *p = m + s * kCGSet;
                         p[gfs::S_ITER] = iters(s, n);
                         p[gfs::S_RNORM] = kRnorm * (1 + s);
                         p[gfs::S_RHOM] = kRhom + s;
                       }
                       for (int k = 0; resid && k < iters(0, n); k++) resid[k] = 100.0 + k;
                     }});
}

}  // namespace

extern "C" {
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 0, hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static double scratch[1 << 16];
  return *p = scratch, hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return ""; }
hipError_t hipMalloc(void **p, size_t n) { return *p = calloc(1, n + 64), hipSuccess; }
hipError_t hipFree(void *p) { return free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = calloc(1, n + 64), hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return complete(++seq), hipSuccess; }
hipError_t hipDeviceSynchronize() { return complete(++seq), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  complete(++seq);
  return memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
  ++seq;
  if (k == hipMemcpyDeviceToHost) complete(seq);  // pageable: the call waits
  return memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  return ++seq, memset(d, v, n), hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t) new Event, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete (Event *)e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return ((Event *)e)->seq = ++seq, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { return complete(((Event *)e)->seq), hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.f, hipSuccess; }

static dim3 cfg_grid, cfg_block;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) {
  return cfg_grid = g, cfg_block = b, hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *s) {
  *g = cfg_grid;
  *b = cfg_block;
  *sh = 0;
  *s = nullptr;
  return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) {
  static void *h = nullptr;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *,
                           void *, dim3 *, dim3 *, int *) {
  names()[f] = name;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t) {
  ++seq;
  const std::string &k = names()[f];
  auto has = [&](const char *s) { return k.find(s) != std::string::npos; };
  // both argument structures begin with the control
  if (has("k_cg_apply")) apply(*(const CGCtl *)args[0]);
  // set-up reductions: (rho, norm) = (3, 1), the residual gone after two cycles
  const double norm = loops < 2 ? 1.0 : 0.0;
  if (has("k_setup_fin_seg")) {
    const int ns = *(const int *)args[2];
    double *out = *(double *const *)args[4];
    for (int s = 0; s < ns; s++) {
      out[2 * s] = kRho32;
      out[2 * s + 1] = norm;
    }
  } else if (has("k_setup_fin")) {
    double *out = *(double *const *)args[3];
    out[0] = kRho32;
    out[1] = norm;
  }
  return hipSuccess;
}
}

#define REQUIRE(c)                                                \
  do {                                                            \
    if (!(c)) {                                                   \
      printf("%s:%d: %s does not hold\n", __FILE__, __LINE__, #c); \
      return 1;                                                   \
    }                                                             \
  } while (0)

int main(int argc, char **argv) {
  if (argc != 3) return 2;
  const bool batched = !strcmp(argv[1], "batched"), mixed = !strcmp(argv[2], "mixed");
  nsys = batched ? 2 : 1;
  gf_ctx *ctx = nullptr;
  REQUIRE(gf_ctx_create(0, nullptr, &ctx) == GF_OK);
  // two elements of order 1 whose nodes are all their own groups
  const int nel = 2, n = nel * 8;
  double xi[2], w[2], D[4], dx[3 * nel], jac[nel];
  REQUIRE(gf_gll_basis(1, xi, w, D) == GF_OK);
  std::vector<int64_t> offs(n + 1), mem(n);
  for (int k = 0; k < n; k++) offs[k] = mem[k] = k;
  offs[n] = n;
  for (double &v : dx) v = 2.0;
  for (double &v : jac) v = 0.125;
  gf_mesh_desc d;
  memset(&d, 0, sizeof(d));
  d.dim = 3;
  d.gtype = GF_GE_REGULAR;
  d.nelems = nel;
  for (int k = 0; k < 3; k++) {
    d.N[k] = 2;
    d.D[k] = D;
    d.W[k] = w;
  }
  d.elem_dxidx = dx;
  d.elem_jac = jac;
  d.ggfx_offs = offs.data();
  d.ggfx_members = mem.data();
  gf_mesh *m = nullptr;
  REQUIRE(gf_mesh_create(ctx, &d, &m) == GF_OK);
  const int64_t eoff[3] = {0, 1, 2};
  if (batched) REQUIRE(gf_mesh_set_segments(m, 2, eoff) == GF_OK);

  std::vector<double> b(n, 1.0), x(n, 0.0), resid(64, 0.0);
  gf_cg_params prm;
  memset(&prm, 0, sizeof(prm));
  prm.maxit = 50;
  prm.tol = 1e-2;
  prm.normtype = GF_NORM_INF;
  prm.precision = mixed ? 1 : 0;
  prm.p_scalar = prm.q_scalar = 1.0;
  prm.resid = resid.data();
  gf_cg_result res;
  REQUIRE(gf_cg_solve(m, &prm, b.data(), nullptr, x.data(), &res) == GF_OK);

  const int cycles = mixed ? 2 : 1;
  REQUIRE(loops == cycles);
  int want[2] = {0, 0};
  for (int k = 1; k <= cycles; k++)
    for (int s = 0; s < 2; s++) want[s] += iters(s, k);
  REQUIRE(res.iters == want[nsys - 1]);
  if (!mixed) REQUIRE(res.rnorm == kRnorm * nsys);
  if (!mixed && !batched)
    for (int k = 0; k < 64; k++) REQUIRE(resid[k] == (k < want[0] ? 100.0 + k : 0.0));
  if (mixed) {  // the direction is kept across cycles: beta = rho / rho of before
    REQUIRE(betas.size() == 2 && betas[0] == 0.0);
    REQUIRE(betas[1] == kRho32 / kRhom);
  }
  if (batched) {
    int its[2];
    double rn[2], rn0[2];
    REQUIRE(gf_cg_member_results(m, 2, its, rn, rn0) == GF_OK);
    for (int s = 0; s < 2; s++) REQUIRE(its[s] == want[s]);
    if (!mixed) REQUIRE(rn[0] == kRnorm && rn[1] == 2 * kRnorm);
  }
  gf_mesh_destroy(m);
  gf_ctx_destroy(ctx);
  return 0;
}
