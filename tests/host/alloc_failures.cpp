// The library's host code (psdns_api.hip, sgs_api.hip) on a stand-in for the
// HIP runtime whose device memory is host memory and whose n-th allocation can
// be made to fail.  The kernel launchers that matter here check that every
// pointer they are given lies in a live allocation; the others do nothing.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include <hip/hip_runtime.h>

#include "psdns_gpu.h"
#include "psdns_internal.h"
#include "psdns_sgs.h"
#include "sgs_internal.h"

static std::map<char*, size_t> live;
static int countdown = -1;  // allocations until the one that fails (-1: none)
static int bad = 0, launches = 0;

static void check(bool ok, const char* what) {
  if (!ok) {
    std::printf("FAIL: %s\n", what);
    bad++;
  }
}
static bool alive(const void* p, size_t bytes) {
  auto it = live.upper_bound((char*)p);
  if (!p || it == live.begin()) return false;
  --it;
  return (char*)p + bytes <= it->first + it->second;
}

extern "C" {
static hipError_t get(void** p, size_t n) {
  if (countdown >= 0 && countdown-- == 0) return hipErrorOutOfMemory;
  *p = std::calloc(n ? n : 1, 1);
  live[(char*)*p] = n ? n : 1;
  return hipSuccess;
}
static hipError_t put(void* p) {
  if (!p) return hipSuccess;
  if (!live.erase((char*)p)) return hipErrorInvalidValue;
  std::free(p);
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) { return get(p, n); }
hipError_t hipFree(void* p) { return put(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return get(p, n); }
hipError_t hipHostFree(void* p) { return put(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipGetSymbolAddress(void** p, const void* s) { return *p = const_cast<void*>(s), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = nullptr, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { return *t = 0.f, hipSuccess; }
}

namespace psdns {
int launch_y_grad(const Ctx& c, const void* phi, void* yw, int nv, int) {
  launches++;
  const size_t slot = 2 * sizeof(double) * (size_t)c.geo.na * c.geo.n;
  check(alive(yw, 2 * nv * slot) && phi, "launch_y_grad: the gradient cylinder");
  return 0;
}
int launch_pass(const Ctx& c, Pass p, int a0, int a1) {
  const size_t n = c.geo.n, xi = 2 * sizeof(double) * n * n * c.geo.max_al_x;
  if (p == Pass::ZInv && a1 == 2) check(alive(c.xi, 3 * a0 * xi), "z pass: the gradient z pencils");
  if (p == Pass::XC2R) check(alive(c.xi, a0 * xi) && alive(c.ux, a0 * n * n * n * sizeof(double)), "x pass: the gradient");
  return 0;
}
void launch_ek_force(const Ctx& c, int, int, const EkInf&, double* terms, double* ek, double* out) {
  launches++;
  check(c.nforce > 0 && alive(c.force_list, sizeof(int2) * c.nforce), "force list");
  check(alive(terms, 12 * (size_t)c.nforce), "force list terms");
  check(alive(ek, 64 * sizeof(double)) && alive(out, sizeof(double)), "energies");
}
namespace sgs {
void launch_invariants(hipStream_t, int, const void* A, size_t P, double, float* lam, float* T) {
  launches++;
  check(alive(A, 9 * P * sizeof(double)) && alive(lam, 5 * P * sizeof(float)) && alive(T, 24 * P * sizeof(float)),
        "invariants: the gradient");
}
}  // namespace sgs
}  // namespace psdns

static psdns_ctx* context(int n) {
  psdns_params p{};
  p.nx = p.ny = p.nz = n;
  p.prec = 8;
  p.kshift = 1;
  p.viscos = 0.01;
  psdns_ctx* c = nullptr;
  check(psdns_create(&p, &c) == PSDNS_OK, "psdns_create");
  int na = 0, mx = 0;
  psdns_geometry(c, &na, &mx);
  std::vector<double> u((size_t)2 * 3 * na * n, 0.0);
  check(psdns_put_state(c, u.data(), 0) == PSDNS_OK, "psdns_put_state");
  return c;
}

// features(): each of its buffers fails once; the next call is whole
static void features() {
  for (int k = 0; k < 3; k++) {
    psdns_ctx* c = context(32);
    psdns_sgs* m = nullptr;
    check(psdns_sgs_create(32, 0, &m) == PSDNS_OK, "psdns_sgs_create");
    countdown = k;
    check(psdns_sgs_features(m, c) == PSDNS_ENOMEM, "features without memory");
    countdown = -1;
    launches = 0;
    check(psdns_sgs_features(m, c) == PSDNS_OK && launches == 2, "features after a failed call");
    const size_t held = live.size();
    check(psdns_sgs_features(m, c) == PSDNS_OK && live.size() == held, "features once more");
    psdns_sgs_destroy(m);
    psdns_destroy(c);
    check(live.empty(), "memory left");
  }
}

// the forcing list: a longer one fails, the former one is asked for again
static void force_list() {
  for (int k = 0; k < 2; k++) {
    psdns_ctx* c = context(32);
    double ek[64];
    check(psdns_ek_shell(c, 4, ek) == PSDNS_OK, "ek_shell");
    countdown = k;
    check(psdns_ek_shell(c, 5, ek) != PSDNS_OK, "ek_shell without memory");
    countdown = -1;
    launches = 0;
    check(psdns_ek_shell(c, 4, ek) == PSDNS_OK && launches == 1, "ek_shell after a failed call");
    check(psdns_ek_shell(c, 5, ek) == PSDNS_OK && launches == 2, "ek_shell, the longer list");
    psdns_destroy(c);
    check(live.empty(), "memory left");
  }
}

int main(int argc, char** argv) {
  if (argc > 1 && !std::strcmp(argv[1], "features")) features();
  else if (argc > 1 && !std::strcmp(argv[1], "force_list")) force_list();
  else return 2;
  std::printf("%s\n", bad ? "failures" : "ok");
  return bad != 0;
}
