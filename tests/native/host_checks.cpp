// Host code of libscn_hip.so with the HIP runtime's calls replaced by the ones below: no GPU is used, kernels are counted and not run.
// Usage: host_checks NAME; prints "ok" and returns 0, or says which check failed.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../include/scn_hip.h"
#include "../../sparseconvnet_amd/csrc/conv_common.h"

static int mallocs, fail_malloc = -1, launches;  // fail_malloc: that many succeed, the next two fail (the library tries twice)
static bool fail_launch, capturing;
static hipError_t last = hipSuccess;

extern "C" {
hipError_t hipMalloc(void **p, size_t bytes) {
  if (fail_malloc >= 0 && (mallocs == fail_malloc || mallocs == fail_malloc + 1)) {
    mallocs++;
    return last = hipErrorOutOfMemory;
  }
  mallocs++;
  *p = calloc(1, bytes);
  return hipSuccess;
}
hipError_t hipFree(void *p) { return free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
  *p = calloc(1, bytes);
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)malloc(8), hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) { return a->device = 0, hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
  launches++;
  return fail_launch ? last = hipErrorLaunchFailure : hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = (hipEvent_t)malloc(8), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
  return *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone, hipSuccess;
}
}

#define CHECK(x)                                            \
  do {                                                      \
    if (!(x)) {                                             \
      printf("%s:%d: %s\n", __FILE__, __LINE__, #x);        \
      exit(1);                                              \
    }                                                       \
  } while (0)

using namespace scn;

// A failed allocation is reported by its own error and not once more by the next launch.
static void failed_allocation() {
  mallocs = 0;
  fail_malloc = 0;
  bool threw = false;
  try {
    pool_alloc(5000, POOL_COMPUTE);
  } catch (const std::exception &) {
    threw = true;
  }
  fail_malloc = -1;
  CHECK(threw && mallocs == 2 && hipGetLastError() == hipSuccess);
}

static void add_level(Metadata &m, int64_t side, int64_t n) {
  Level &l = m.levels[SizeKey{side, side, side}];
  l.n = n;
  l.npad = round_up(n, 64);
}

// A table is kept for later calls only once the kernel that fills it has been launched, and a level nobody asked about yet does not
// fail the call.
static void identity_tables() {
  for (int ok = 0; ok < 8; ok++) {  // how many allocations succeed: two per table, four tables
    Metadata m;
    m.dim = 3;
    add_level(m, 64, 5000), add_level(m, 32, 90000), add_level(m, 16, 700), add_level(m, 8, 30);
    mallocs = launches = 0;
    fail_malloc = ok;
    bool threw = false;
    try {
      Table &t = identity_table(m, 90000, nullptr);
      CHECK(t.n == 90000 && t.nbr.p && t.gmask.p && launches == 1);
    } catch (const std::exception &) {
      threw = true;
    }
    fail_malloc = -1;
    CHECK(threw == (ok < 2));
    if (threw) CHECK(m.ident.empty() && launches == 0);
    for (auto &e : m.ident) CHECK(e.second.nbr.p && e.second.gmask.p);
    const int before = launches;
    for (int64_t n : {90000, 5000, 700, 30}) {
      const bool had = m.ident.count(n);
      Table &t = identity_table(m, n, nullptr);
      CHECK(t.n == n && t.K == 1 && t.nbr.p && t.gmask.p);
      CHECK(had || launches > before);
    }
    m.ident.clear();
    scn_release_cache();  // the next round allocates again
  }
  Metadata m;
  m.dim = 3;
  add_level(m, 16, 700);
  fail_launch = true;
  bool threw = false;
  try {
    identity_table(m, 5000, nullptr);
  } catch (const std::exception &) {
    threw = true;
  }
  fail_launch = false;
  CHECK(threw && m.ident.empty());
}

// Calls whose tables, operands or scratch k_conv_wave cannot read are refused, whatever else they are: forward or gradient, either operand type.
static void wave_refuses() {
  Metadata m;
  Table t;
  t.n = 3000, t.npad = 3008;
  t.gmask.reserve(188);
  const float *in = (const float *)4096;
  for (bool bf16 : {false, true})
    for (bool gradient : {false, true}) {
      m.bf16 = bf16;
      const int n_in = 32;
      for (int K : {1, 8, 27, 32}) {
        t.K = K;
        CHECK(conv_wave_serves(m, t, in, 3000, n_in, 32, gradient) == !(bf16 && gradient));
        for (int64_t rows : {(int64_t)0, (int64_t)1 << 24, (int64_t)1 << 31}) CHECK(!conv_wave_serves(m, t, in, rows, n_in, 32, gradient));
        CHECK(!conv_wave_serves(m, t, in + 1, 3000, n_in, 32, gradient));
        CHECK(!conv_wave_serves(m, t, in, 3000, 33, 32, gradient) && !conv_wave_serves(m, t, in, 3000, 30, 32, gradient));
        m.fixed_scratch = (unsigned char *)&m;
        CHECK(!conv_wave_serves(m, t, in, 3000, n_in, 32, gradient));
        m.fixed_scratch = nullptr;
        Table bare;
        bare.n = t.n, bare.npad = t.npad, bare.K = K;
        CHECK(!conv_wave_serves(m, bare, in, 3000, n_in, 32, gradient));
      }
      for (int K : {33, 49, 64, 125}) {
        t.K = K;
        for (int64_t n : {500, 3000, 300001}) {
          t.n = n;
          for (int planes : {8, 20, 32, 48, 64, 128})
            for (int out : {8, 32, 40, 48, 64}) CHECK(!conv_wave_serves(m, t, in, n, planes, out, gradient));
        }
        t.n = 3000;
      }
    }
}

// A handle that dies while its stream is captured launches nothing into the graph, and its counts are read later all the same.
static void counts_under_capture() {
  double macs = 0;
  CHECK(scn_take_released_macs(&macs) == 0);
  for (bool captured : {false, true}) {
    scn_metadata *h = scn_md_create(3);
    Metadata &m = *reinterpret_cast<Metadata *>(h);  // the handle's first member
    m.consumer_known = true;
    auto c = std::make_shared<Counts>();
    c->K = 3, c->slots = 2;
    c->dev.reserve(6);
    for (int i = 0; i < 6; i++) c->dev.p[i] = 10 + i;  // 75 rules
    for (double per_rule : {4.0, 6.0}) m.pending_macs.emplace_back(c, per_rule);
    m.macs_settled = 5;
    launches = 0;
    capturing = captured;
    scn_md_destroy(h);
    capturing = false;
    CHECK(launches == (captured ? 0 : 1));
    if (captured) {
      CHECK(scn_take_released_macs(&macs) == 0 && macs == 75 * 10.0 + 5);
      CHECK(scn_take_released_macs(&macs) == 0 && macs == 0);
    } else {  // (the kernel that adds them up did not run)
      CHECK(scn_take_released_macs(&macs) == 0);
    }
  }
  for (int i = 0; i < 400; i++) {  // read on the way when many have gathered
    scn_metadata *h = scn_md_create(3);
    Metadata &m = *reinterpret_cast<Metadata *>(h);
    m.consumer_known = true;
    auto c = std::make_shared<Counts>();
    c->K = 1;
    c->dev.reserve(1);
    c->dev.p[0] = 2;
    m.pending_macs.emplace_back(c, 1.0);
    std::weak_ptr<Counts> seen = c;
    c.reset();
    capturing = i < 300;
    scn_md_destroy(h);
    capturing = false;
    if (i == 0) CHECK(!seen.expired());
  }
  CHECK(scn_take_released_macs(&macs) == 0 && macs == 300 * 2.0 - 100);  // (the launches of the other hundred, which did not run, left their -1)
}

int main(int argc, char **argv) {
  const char *name = argc > 1 ? argv[1] : "";
  if (!strcmp(name, "failed_allocation")) failed_allocation();
  else if (!strcmp(name, "identity_tables")) identity_tables();
  else if (!strcmp(name, "wave_refuses")) wave_refuses();
  else if (!strcmp(name, "counts_under_capture")) counts_under_capture();
  else return printf("no check of that name\n"), 2;
  printf("ok\n");
  return 0;
}
