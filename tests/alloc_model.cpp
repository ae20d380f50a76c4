// The create calls of the 1D and BGK contexts against host allocations that fail one after another: every
// failure is FR_E_NOMEM, no exception leaves the C entry; when the ensemble's loop is captured anew; and the
// sizes of launches.  The HIP runtime is a stand-in that succeeds.
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "../include/fr.h"

extern "C" {
typedef void *P;
int hipGetDeviceCount(int *n) { return *n = 1, 0; }
int hipGetDevice(int *d) { return *d = 0, 0; }
int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int *v, int, int) { return *v = 256, 0; }
int hipMalloc(P *p, size_t) { return *p = std::malloc(8), 0; }
int hipHostMalloc(P *p, size_t, unsigned) { return *p = std::malloc(8), 0; }
int hipFree(P p) { return std::free(p), 0; }
int hipHostFree(P p) { return std::free(p), 0; }
int hipMemcpy(P, const void *, size_t, int) { return 0; }
int hipMemcpyAsync(P, const void *, size_t, int, P) { return 0; }
int hipMemset(P, int, size_t) { return 0; }
int hipMemsetAsync(P, int, size_t, P) { return 0; }
int hipStreamCreateWithFlags(P *s, unsigned) { return *s = std::malloc(8), 0; }
int hipStreamDestroy(P s) { return std::free(s), 0; }
int hipStreamSynchronize(P) { return 0; }
int hipStreamWaitEvent(P, P, unsigned) { return 0; }
int hipStreamGetDevice(P, int *d) { return *d = 0, 0; }
int hipStreamBeginCapture(P, int) { return 0; }
int hipStreamEndCapture(P, P *) { return 0; }
int captures = 0;
int hipGraphInstantiate(P *g, P, P *, char *, size_t) { return ++captures, *g = &captures, 0; }
int hipGraphExecDestroy(P) { return 0; }
int hipGraphDestroy(P) { return 0; }
int hipGraphLaunch(P, P) { return 0; }
int hipEventCreate(P *e) { return *e = std::malloc(8), 0; }
int hipEventCreateWithFlags(P *e, unsigned) { return *e = std::malloc(8), 0; }
int hipEventDestroy(P e) { return std::free(e), 0; }
int hipEventRecord(P, P) { return 0; }
int hipEventSynchronize(P) { return 0; }
float elapsed = 1e6f;  // every timing beats the last one
int hipEventElapsedTime(float *ms, P, P) { return *ms = --elapsed, 0; }
int hipPointerGetAttributes(P, const void *) { return 1; }
int hipGetSymbolAddress(P *p, const void *) { return *p = std::malloc(8), 0; }
void __hipRegisterVar(P *, P, char *, char *, int, size_t, int, int) {}
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int last_error = 0;
int hipGetLastError(void) {
  const int e = last_error;
  return last_error = 0, e;
}
const char *hipGetErrorString(int) { return ""; }
struct Dim { unsigned x, y, z; };
// a launch has fewer than 2^32 threads
int hipLaunchKernel(const void *, Dim g, Dim b, P *, size_t, P) {
  return last_error = (unsigned long long)g.x * b.x < 1ull << 32 ? 0 : 9;
}
Dim grid, block;
unsigned __hipPushCallConfiguration(Dim g, Dim b, size_t, P) { return grid = g, block = b, 0; }
int __hipPopCallConfiguration(Dim *g, Dim *b, size_t *lds, P *st) { return *g = grid, *b = block, *lds = 0, *st = nullptr, 0; }
P *__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(P *) {}
void __hipRegisterFunction(P *, const void *, char *, const char *, int, P, P, P, P, int *) {}
}

static long countdown = -1;  // allocations until one fails, -1: none does
static bool thrown = false;

void *operator new(size_t n) {
  if (countdown >= 0 && countdown-- == 0) {
    thrown = true;
    throw std::bad_alloc();
  }
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

// call() with its first, second, ... allocation failing, until it runs through; returns the faults
template <class F>
static int each(const char *name, F &&call) {
  int bad = 0;
  for (long k = 0;; ++k) {
    thrown = false;
    countdown = k;
    const int rc = call();
    countdown = -1;
    if (!thrown) {
      std::printf("%s: %ld allocations, rc %d\n", name, k, rc);
      return bad + (rc != FR_OK) + (k == 0);
    }
    if (rc != FR_E_NOMEM) std::printf("FAIL %s: allocation %ld gives %d\n", name, k, rc), ++bad;
  }
}

int main() {
  std::setvbuf(stdout, nullptr, _IONBF, 0);
  int bad = 0;
  fr1d_desc d1{};
  d1.equation = FR_EQ_EULER, d1.ncell = 1000, d1.deg = 2, d1.dx = 1e-3, d1.gamma = 1.4;
  bad += each("fr1d_create", [&] {
    fr1d_ctx *c = nullptr;
    const int rc = fr1d_create(&c, &d1);
    fr1d_destroy(c);
    return rc;
  });
  std::vector<int> n(300, 400), deg(300, 3);
  std::vector<double> dx(300, 0.01);
  bad += each("fr_ens_create", [&] {
    fr_ens_ctx *c = nullptr;
    const int rc = fr_ens_create(&c, 300, n.data(), deg.data(), dx.data(), 1.4, FR_FLUX_HLL, FR_BC1_PERIOD);
    fr_ens_destroy(c);
    return rc;
  });
  // a captured loop of register-resident steps outlives a new mapping of the launches per stage
  for (int path : {FR1D_PATH_AUTO, FR1D_PATH_BATCHED}) {
    fr_ens_ctx *c = nullptr;
    int choice = -1;
    bool ok = fr_ens_create(&c, 300, n.data(), deg.data(), dx.data(), 1.4, FR_FLUX_HLL, FR_BC1_PERIOD) == FR_OK;
    ok = ok && fr_ens_set_path(c, path) == FR_OK;
    captures = 0;
    for (int r = 0; r < 2; ++r) ok = ok && fr_ens_run_graph(c, FR_ENS_FILTER, 1e-3, 3, 1, nullptr, nullptr) == FR_OK;
    ok = ok && captures == 1 && fr_ens_autotune(c, 1e-3, &choice) == FR_OK && choice == 14;
    ok = ok && fr_ens_run_graph(c, FR_ENS_FILTER, 1e-3, 3, 1, nullptr, nullptr) == FR_OK;
    ok = ok && captures == (path == FR1D_PATH_AUTO ? 1 : 2);
    fr_ens_destroy(c);
    if (!ok) std::printf("FAIL path %d: %d captures\n", path, captures), ++bad;
  }
  std::vector<double> v(64, 1.0), tau(2, 0.1);
  for (int cells : {8, 80}) {  // 80 x 80 x 64 x 64 velocities: the path of large states
    fr_bgk_desc d{};
    d.nx = d.ny = cells, d.deg = 2, d.nu = d.nv = 64, d.nmem = 2, d.dx = d.dy = 0.1, d.gamma = 2.0;
    d.u = d.v = d.wu = d.wv = v.data(), d.tau = tau.data();
    bad += each("fr_bgk_create", [&] {
      fr_bgk_ctx *c = nullptr;
      const int rc = fr_bgk_create(&c, &d);
      fr_bgk_destroy(c);
      return rc;
    });
  }
  {  // 2^30 points in planes of 2^27, four velocities: every launch of a step within the runtime's limit
    fr_bgk_desc d{};
    d.nx = 8192, d.ny = 4096, d.deg = 1, d.nu = d.nv = 2, d.nmem = 8, d.dx = d.dy = 0.1, d.gamma = 2.0;
    std::vector<double> taus(8, 0.1);
    d.u = d.v = d.wu = d.wv = v.data(), d.tau = taus.data();
    fr_bgk_ctx *c = nullptr;
    const bool ok = fr_bgk_create(&c, &d) == FR_OK && fr_bgk_step(c, 1e-3, 1) == FR_OK;
    fr_bgk_destroy(c);
    if (!ok) std::printf("FAIL fr_bgk_step of 2^30 points\n"), ++bad;
  }
  {  // a strip of two million rows of cells, p = 2: 72 million rows of values between the two layouts
    fr2d_desc d{};
    d.nx = 1, d.ny = 2000000, d.deg = 2, d.gamma = 1.4, d.iJ11 = d.iJ22 = 1.0;
    fr2d_ctx *c = nullptr;
    double u = 0.0;
    const bool ok = fr2d_create(&c, &d) == FR_OK && fr2d_set_state_dev(c, &u) == FR_OK &&
                    fr2d_get_state_dev(c, &u) == FR_OK;
    fr2d_destroy(c);
    if (!ok) std::printf("FAIL 2D state copies of 72 million rows\n"), ++bad;
  }
  fr_bgk1d_desc d{};
  d.nx = 20, d.deg = 2, d.nu = 64, d.nmem = 2, d.dx = 0.1, d.gamma = 3.0;
  d.u = d.w = v.data(), d.tau = tau.data();
  bad += each("fr_bgk1d_create", [&] {
    fr_bgk1d_ctx *c = nullptr;
    const int rc = fr_bgk1d_create(&c, &d);
    fr_bgk1d_destroy(c);
    return rc;
  });
  fr_bgk1d_ctx *c = nullptr;
  bad += fr_bgk1d_create(&c, &d) != FR_OK;
  std::vector<double> w(20 * 3 * 3 * 2);
  bad += each("fr_bgk1d_moments", [&] { return fr_bgk1d_moments(c, w.data()); });
  fr_bgk1d_destroy(c);
  return bad;
}
