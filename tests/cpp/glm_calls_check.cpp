// Host check of the evaluation calls (stan_amd/csrc/capi_glm.cpp) against a
// stand-in HIP runtime: device memory is host memory, a stream is a thread
// that works its queue off, and the kernels are replaced by a function of
// theta that is as simple as it is different from point to point.  The
// stand-in shows what the hardware shows rarely or never: stores that reach
// the host in another order than they were issued, work that is still queued
// when a call returns, and allocations that fail.
//   glm_calls_check <scenario>   prints "ok" or what went wrong
#include <malloc.h>

#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <deque>
#include <functional>
#include <map>

#include "../../stan_amd/csrc/capi_glm.cpp"

namespace {

// ---- the stand-in runtime -------------------------------------------------

struct stream_queue {
  std::mutex mu;
  std::condition_variable cv;
  std::deque<std::function<void()>> q;
  size_t pending = 0;
  bool stop = false;
  std::thread th;
  stream_queue() : th([this] { work(); }) {}
  ~stream_queue() {
    {
      std::lock_guard<std::mutex> l(mu);
      stop = true;
    }
    cv.notify_all();
    th.join();
  }
  void work();
  void push(std::function<void()> f) {
    std::lock_guard<std::mutex> l(mu);
    q.push_back(std::move(f));
    ++pending;
    cv.notify_all();
  }
  void wait() {
    std::unique_lock<std::mutex> l(mu);
    cv.wait(l, [this] { return pending == 0; });
  }
};

hipError_t g_last = hipSuccess;  // what hipGetLastError returns, once
int g_delay_us = 0;          // before every queued operation
int g_late_us = 3000;        // before the late words of a single evaluation
bool g_fail_launch = false;  // kernel launches are refused
bool g_no_store = false;     // kernels run and store nothing
bool g_fail_pinned = false;  // no pinned memory
size_t g_limit = SIZE_MAX, g_used = 0;  // device memory
std::map<void*, size_t> g_dev;
int g_pinned_calls = 0;

void pause_us(int us) {
  if (us > 0) std::this_thread::sleep_for(std::chrono::microseconds(us));
}

void stream_queue::work() {
  std::unique_lock<std::mutex> l(mu);
  while (true) {
    cv.wait(l, [this] { return stop || !q.empty(); });
    if (q.empty()) return;
    std::function<void()> f = std::move(q.front());
    q.pop_front();
    l.unlock();
    pause_us(g_delay_us);
    f();
    l.lock();
    --pending;
    cv.notify_all();
  }
}

stream_queue* queue_of(hipStream_t s) { return reinterpret_cast<stream_queue*>(s); }

// the stand-in density: distinct for every theta and parameter
double value(const double* th, int D) {
  double s = 0;
  for (int i = 0; i < D; ++i) s += (i + 1) * th[i];
  return s;
}
double slope(const double* th, int i) { return 2.0 * th[i] + i; }

void store(double* out, size_t i, double v) {
  __atomic_store_n(reinterpret_cast<uint64_t*>(out + i), *reinterpret_cast<uint64_t*>(&v),
                   __ATOMIC_RELAXED);
}

// one chain's outputs; the words of `late` reach the host after the others
void put(const double* th, double* out, int D, size_t late0, size_t late1) {
  if (g_no_store) return;
  const double status = std::fabs(th[0]) < 1e100 ? 0.0 : 1.0;
  const auto one = [&](size_t i) {
    store(out, i, i == 0 ? value(th, D) : i == static_cast<size_t>(D) + 1 ? status : slope(th, i - 1));
  };
  for (size_t i = D + 2; i-- > 0;)
    if (i < late0 || i >= late1) one(i);
  if (late0 < late1) pause_us(g_late_us);
  for (size_t i = late0; i < late1; ++i) one(i);
}

}  // namespace

extern "C" {

hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(static_cast<void*>(p), 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return std::exchange(g_last, hipSuccess); }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipMalloc(void** p, size_t n) {
  *p = nullptr;
  if (n > g_limit - std::min(g_limit, g_used)) return g_last = hipErrorOutOfMemory;
  *p = std::calloc(1, std::max<size_t>(n, 1));
  g_dev[*p] = n;
  g_used += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  g_used -= g_dev[p];
  g_dev.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = nullptr;
  if (g_fail_pinned) return g_last = hipErrorOutOfMemory;
  ++g_pinned_calls;
  *p = std::calloc(1, n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  queue_of(st)->push([=] { std::memcpy(d, s, n); });
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
  queue_of(st)->push([=] { std::memset(d, v, n); });
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  return *s = reinterpret_cast<hipStream_t>(new stream_queue), hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { return queue_of(s)->wait(), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return delete queue_of(s), hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = nullptr, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }

}  // extern "C"

namespace sx {

int noalloc_setup(int) { return SX_OK; }

tile_geom make_geom(int64_t N, int64_t K, int L, int smax) {
  tile_geom g;
  g.L = L;
  for (g.lgL = 0; (1 << g.lgL) < L;) ++g.lgL;
  g.R = 64 / L;
  g.S = static_cast<int>((K + L - 1) / L);
  g.smax = smax;
  g.T = (N + g.R - 1) / g.R;
  return g;
}
hipError_t launch_tile_x_f64(const double*, double*, int64_t, int64_t, const tile_geom&,
                             hipStream_t) {
  return hipSuccess;
}
hipError_t launch_split_x(const double*, uint16_t*, uint16_t*, int64_t, int64_t, int64_t, int64_t,
                          hipStream_t) {
  return hipSuccess;
}
hipError_t launch_prep_y(const void*, float*, int, int64_t, int64_t, hipStream_t) {
  return hipSuccess;
}
// points and results of a batch, one chain after the other
static hipError_t batch(const double* theta, int64_t ts, double* out, int64_t os, int D, int C,
                        double* scratch, int64_t per_chain, hipStream_t s, size_t late0 = 0,
                        size_t late1 = 0) {
  if (g_fail_launch) return hipErrorInvalidValue;
  if (const hipError_t e = hipGetLastError()) return e;  // a launch's own check
  queue_of(s)->push([=] {
    for (int c = 0; c < C; ++c) {
      for (int64_t i = 0; i < per_chain; ++i) scratch[c * per_chain + i] = c;
      put(theta + c * ts, out + c * os, D, late0, late1);
    }
  });
  return hipSuccess;
}
hipError_t launch_pass_f64(int, const tile_geom&, const pass_args& a, int blocks, int,
                           hipStream_t s, bool) {
  return batch(a.theta, a.theta_stride, a.out, a.out_stride, a.D, a.chains, a.partials,
               static_cast<int64_t>(a.E) * blocks, s);
}
hipError_t launch_eval_f64(int, const tile_geom&, const pass_args& a, const double* h_theta, int,
                           int, hipStream_t s) {
  if (g_fail_launch) return hipErrorInvalidValue;
  if (const hipError_t e = hipGetLastError()) return e;
  const std::vector<double> th(h_theta, h_theta + a.D);  // carried by the launch
  double* out = a.out;
  queue_of(s)->push([=] { put(th.data(), out, static_cast<int>(th.size()), 2, 4); });
  return hipSuccess;
}
hipError_t launch_mfma_pass(int, const double* theta, int64_t D, int C, const mx_args&,
                            const pass_args& pa, hipStream_t s) {
  return batch(theta, D, pa.out, pa.out_stride, static_cast<int>(D), C, nullptr, 0, s);
}
// To the host, the z gradients of the launch before the last are the last to
// arrive: nothing between the two launches publishes them to it.
hipError_t launch_hier(const hier_args& a, bool, hipStream_t s, bool host_out) {
  const size_t z0 = 2 * static_cast<size_t>(a.K) + 3, z1 = static_cast<size_t>(a.D) + 1;
  return batch(a.theta, a.theta_stride, a.out, a.out_stride, a.D, a.chains, a.cpart, a.E, s,
               host_out ? z0 : 0, host_out ? z1 : 0);
}

}  // namespace sx

// ---- scenarios -------------------------------------------------------------

namespace {

int g_bad = 0;
#define CHECK(cond)                                                  \
  do {                                                               \
    if (!(cond) && ++g_bad < 10)                                     \
      std::printf("line %d: %s (%s)\n", __LINE__, #cond, sx_last_error()); \
  } while (0)

sx_glm* make(int family, int64_t N, int64_t K, int64_t J, int precision) {
  std::vector<double> X(N * K, 0.5), yd(N, 1.0);
  std::vector<int32_t> yi(N, 1);
  std::vector<int64_t> off(J + 1);
  for (int64_t j = 0; j <= J; ++j) off[j] = N * j / std::max<int64_t>(J, 1);
  sx_glm* m = nullptr;
  const void* y = family == SX_NORMAL ? static_cast<const void*>(yd.data()) : yi.data();
  CHECK(sx_glm_create(&m, family, X.data(), y, N, K, J ? off.data() : nullptr, J, precision,
                      nullptr, 0) == SX_OK);
  return m;
}

std::vector<double> points(int64_t C, int64_t D, int seed) {
  std::vector<double> th(C * D);
  for (size_t i = 0; i < th.size(); ++i) th[i] = 0.25 * seed + 0.001 * (i % 977) + 1e-6 * i;
  return th;
}

void check_chain(const double* th, int D, double lp, const double* g) {
  CHECK(lp == value(th, D));
  for (int i = 0; i < D; ++i) CHECK(g[i] == slope(th, i));
}

void check_batch(sx_glm* m, int64_t C, int seed, int64_t from = 0) {
  const std::vector<double> th = points(C, m->D, seed);
  std::vector<double> lp(C), g(C * m->D);
  CHECK(sx_glm_logp_grad_batch(m, th.data(), C, 1, 1, lp.data(), g.data()) == SX_OK);
  for (int64_t c = from; c < C; ++c)
    check_chain(th.data() + c * m->D, static_cast<int>(m->D), lp[c], g.data() + c * m->D);
}

void check_single(sx_glm* m, int seed) {
  const std::vector<double> th = points(1, m->D, seed);
  double lp = 0;
  std::vector<double> g(m->D);
  CHECK(sx_glm_logp_grad(m, th.data(), 1, 1, &lp, g.data()) == SX_OK);
  check_chain(th.data(), static_cast<int>(m->D), lp, g.data());
}

// Single evaluations return this call's results, whatever the order in which
// the words reach the host.
void single_fresh() {
  sx_glm* h = make(SX_HIER_LOGIT, 400, 3, 50, SX_FP64);
  sx_glm* m = make(SX_NORMAL, 300, 7, 0, SX_FP64);
  for (int i = 1; i <= 4; ++i) {
    check_single(h, i);
    check_single(m, i);
  }
  sx_glm_destroy(h);
  sx_glm_destroy(m);
}

// A device that takes longer than the host watches its words for.
void single_slow() {
  sx_glm* h = make(SX_HIER_LOGIT, 60, 2, 5, SX_FP64);
  sx_glm* m = make(SX_LOGIT, 60, 3, 0, SX_FP64);
  g_delay_us = 20000;
  for (int i = 1; i <= 2; ++i) {
    check_single(h, i);
    check_single(m, i);
  }
  // a launch that stores nothing is an error, not the last call's result
  g_no_store = true;
  double lp = 0;
  std::vector<double> g(h->D), th = points(1, h->D, 3);
  CHECK(sx_glm_logp_grad(h, th.data(), 1, 1, &lp, g.data()) == SX_EDEVICE);
  CHECK(sx_glm_logp_grad(m, th.data(), 1, 1, &lp, g.data()) == SX_EDEVICE);
  g_no_store = false;
  g_delay_us = 0;
  check_single(h, 4);
  check_single(m, 4);
  sx_glm_destroy(h);
  sx_glm_destroy(m);
}

// A call that fails leaves nothing queued: its points may be freed, its
// buffers used again.
void failed_calls_drain() {
  g_delay_us = 5000;
  for (int prec : {SX_FP64, SX_FP32}) {
    sx_glm* h = make(SX_HIER_LOGIT, 90, 3, 30, prec);
    for (int64_t C : {1, 3, 100, 2000}) {  // below, between and above the pinned buffer's limits
      std::vector<double> th = points(C, h->D, 1), lp(C), g(C * h->D);
      g_fail_launch = true;
      CHECK(sx_glm_logp_grad_batch(h, th.data(), C, 1, 1, lp.data(), g.data()) == SX_EDEVICE);
      CHECK(queue_of(h->stream)->pending == 0);
      if (C == 1) {
        CHECK(sx_glm_logp_grad(h, th.data(), 1, 1, lp.data(), g.data()) == SX_EDEVICE);
        CHECK(queue_of(h->stream)->pending == 0);
      }
      g_fail_launch = false;
      check_batch(h, C, 2);
    }
    check_single(h, 3);
    sx_glm_destroy(h);
  }
  sx_glm* m = make(SX_LOGIT, 64, 4, 0, SX_FP64);
  for (int64_t C : {1, 2, 3000}) {
    std::vector<double> th = points(C, m->D, 1), lp(C), g(C * m->D);
    g_fail_launch = true;
    CHECK(sx_glm_logp_grad_batch(m, th.data(), C, 1, 1, lp.data(), g.data()) == SX_EDEVICE);
    CHECK(queue_of(m->stream)->pending == 0);
    g_fail_launch = false;
    check_batch(m, C, 2);
  }
  sx_glm_destroy(m);
}

// Calls that need no memory of their own, or less, still run where memory is
// refused: FP64 batches of a logistic or normal model in smaller slabs and
// in the end chain by chain, every batch without a pinned buffer.
void refused_memory() {
  g_late_us = 0;
  for (int family : {SX_LOGIT, SX_NORMAL}) {
    // a chain's partials 4 KB (blocks = T / 4), its points and results less
    sx_glm* m = make(family, 64 * 4 * 60, 5, 0, SX_FP64);
    const size_t per = sizeof(double) * (m->K + 3) * m->blocks;
    for (size_t room : {size_t(0), per, 3 * per, 20 * per, 400 * per}) {
      g_limit = g_used + room;
      check_batch(m, 37, 1);
      check_batch(m, 1200, 2);
      check_batch(m, 3, 3);
      check_single(m, 4);
    }
    g_limit = SIZE_MAX;
    check_batch(m, 1500, 5);
    CHECK(m->bpart_cap == 1024);  // with memory, slabs of full size again
    sx_glm_destroy(m);
  }
  sx_glm* models[] = {make(SX_HIER_LOGIT, 90, 3, 30, SX_FP32), make(SX_HIER_LOGIT, 90, 3, 30, SX_FP64),
                      make(SX_LOGIT, 64, 4, 0, SX_BF16X2), make(SX_LOGIT, 64, 4, 0, SX_FP64)};
  for (sx_glm* m : models) {
    g_fail_pinned = true;
    for (int64_t C : {1, 2, 40, 2000, 9000}) check_batch(m, C, 1);
    g_fail_pinned = false;
    for (int64_t C : {2, 2000}) check_batch(m, C, 2);
    sx_glm_destroy(m);
  }
}

// Batches between the pinned buffers' limits keep no host memory: a buffer
// held by the context costs its first call the page faults, where memory
// that the allocator hands from one call to the next has its pages.
void nothing_kept() {
  sx_glm* h = make(SX_HIER_LOGIT, 90, 3, 30, SX_FP32);
  sx_glm* b = make(SX_LOGIT, 64, 40, 0, SX_BF16X2);
  sx_glm* m = make(SX_LOGIT, 64, 40, 0, SX_FP64);
  for (sx_glm* x : {h, b, m}) {
    check_batch(x, 5000, 1);  // device buffers for the largest batch
    const struct mallinfo2 a = mallinfo2();
    check_batch(x, 300, 2);
    check_batch(x, 350, 3);
    const struct mallinfo2 z = mallinfo2();
    const long kept = static_cast<long>(z.uordblks + z.hblkhd) - static_cast<long>(a.uordblks + a.hblkhd);
    if (kept > 4096 || kept < -4096) std::printf("kept %ld bytes\n", kept), ++g_bad;
    sx_glm_destroy(x);
  }
}

// Small batches pin no memory in the call: the context has it from its
// creation (one allocation per buffer, whatever its size).
void small_batches_pin_nothing() {
  sx_glm* models[] = {make(SX_HIER_LOGIT, 90, 3, 30, SX_FP32), make(SX_HIER_LOGIT, 90, 3, 30, SX_FP64),
                      make(SX_LOGIT, 64, 4, 0, SX_BF16X2), make(SX_NORMAL, 64, 4, 0, SX_FP64)};
  for (sx_glm* x : models) {
    const int before = g_pinned_calls;
    for (int64_t C : {1, 2, 60, 7}) {
      check_batch(x, C, static_cast<int>(C));
      check_single(x, 3);
    }
    const int64_t largest = 65535 / (8 * (x->D + 2));  // below 64 KB
    check_batch(x, largest, 5);
    if (g_pinned_calls != before) std::printf("pinned %d times\n", g_pinned_calls - before), ++g_bad;
    sx_glm_destroy(x);
  }
}

// Batches report the last chain with a domain error, give every such chain
// -inf, and leave the gradient of a chain at a non-finite point alone (a
// mixed-precision or hierarchical batch evaluates it).
void batch_errors() {
  struct {
    sx_glm* m;
    bool checked;
  } models[] = {{make(SX_HIER_LOGIT, 90, 3, 30, SX_FP32), false},
                {make(SX_LOGIT, 64, 40, 0, SX_BF16X2), false},
                {make(SX_NORMAL, 64, 40, 0, SX_FP64), true}};
  for (auto& x : models) {
    const int D = static_cast<int>(x.m->D);
    for (int64_t C : {2, 300, 9000}) {
      std::vector<double> th = points(C, D, 1), lp(C, 7.0), g(C * D, 7.0);
      th[0] = 1e200;  // an overflow
      if (x.checked) th[(C - 1) * D + 3] = NAN;
      CHECK(sx_glm_logp_grad_batch(x.m, th.data(), C, 1, 1, lp.data(), g.data()) == SX_EDOMAIN);
      const std::string said = sx_last_error();
      CHECK((said.find("parameter 3 is not finite") != std::string::npos) == x.checked);
      CHECK(lp[0] == -INFINITY && g[1] == slope(th.data(), 1));
      if (x.checked)
        for (int i = 0; i < D; ++i) CHECK(g[(C - 1) * D + i] == 7.0);
      CHECK((lp[C - 1] == -INFINITY) == x.checked);
      for (int64_t c = 1; c + 1 < C; ++c) check_chain(&th[c * D], D, lp[c], &g[c * D]);
      std::vector<double> lp2(C);
      CHECK(sx_glm_logp_grad_batch(x.m, th.data(), C, 1, 1, lp2.data(), nullptr) == SX_EDOMAIN);
      CHECK(lp == lp2);
      check_batch(x.m, C, 2);
    }
    sx_glm_destroy(x.m);
  }
}

// Which batches take the several-chains FP64 pass: on either side of each
// line where it was measured against the single-chain pass.
void chains_rule() {
  struct {
    int family;
    int64_t N;
    int K, L, C;
    bool fits;
  } cases[] = {
      {SX_LOGIT, 200003, 60, 2, 32, true},   {SX_LOGIT, 1000000, 100, 4, 8, true},
      {SX_LOGIT, 10000000, 100, 4, 7, false}, {SX_LOGIT, 1000000, 100, 8, 32, false},
      {SX_NORMAL, 1000000, 200, 8, 32, false},
      // groups of eight with few chains
      {SX_LOGIT, 900000, 1, 1, 10, false},   {SX_LOGIT, 900000, 1, 1, 16, true},
      {SX_LOGIT, 3728270, 2, 1, 9, false},   {SX_LOGIT, 745654, 10, 1, 10, false},
      {SX_LOGIT, 300000, 10, 1, 11, true},   {SX_LOGIT, 300000, 10, 1, 17, true},
      {SX_LOGIT, 240000, 32, 1, 9, true},    {SX_LOGIT, 200000, 32, 1, 9, false},
      {SX_NORMAL, 900000, 10, 1, 9, true},   {SX_NORMAL, 700000, 10, 1, 9, false},
      // work
      {SX_LOGIT, 53000, 20, 1, 8, true},     {SX_LOGIT, 52000, 20, 1, 8, false},
      {SX_LOGIT, 25000, 64, 2, 8, true},     {SX_LOGIT, 24000, 64, 2, 8, false},
      {SX_LOGIT, 25000, 127, 4, 8, true},    {SX_LOGIT, 24000, 127, 4, 8, false},
      // the forms the GPU tests compare bit for bit with single evaluations
      {SX_LOGIT, 120011, 9, 1, 8, true},     {SX_LOGIT, 70001, 13, 1, 11, true},
      {SX_LOGIT, 61007, 37, 2, 17, true},    {SX_LOGIT, 60005, 60, 4, 8, true},
      {SX_LOGIT, 33333, 63, 4, 13, true},    {SX_LOGIT, 21000, 128, 4, 16, true},
      {SX_LOGIT, 66000, 29, 4, 33, true},    {SX_LOGIT, 20001, 32, 1, 18, true},
      {SX_LOGIT, 100033, 17, 2, 8, true},    {SX_LOGIT, 400001, 3, 2, 12, true},
      {SX_LOGIT, 32003, 101, 4, 8, true},    {SX_LOGIT, 236001, 32, 1, 9, true},
      {SX_NORMAL, 1700003, 4, 1, 10, true},
  };
  for (const auto& c : cases) {
    sx::tile_geom g = sx::make_geom(c.N, c.K, c.L, 32);
    sx::pass_args a{};
    a.N = c.N;
    a.K = c.K;
    a.chains = c.C;
    if (sx::chains_pass_fits(c.family, g, a, 256) != c.fits || sx::chains_pass_fits(c.family, g, a, 64))
      std::printf("family %d N %ld K %d L %d chains %d\n", c.family, static_cast<long>(c.N), c.K, c.L, c.C),
          ++g_bad;
  }
}

// The row splits that are timed: every tile in one of them, each count once,
// and half, one and two per CU among them where the rows suffice.
void split_targets() {
  for (int64_t tiles : {1, 7, 8, 63, 255, 256, 257, 1506, 6250, 6251, 31250, 99999})
    for (int cus : {0, 64, 228, 256, 304}) {
      sx_glm m;
      m.Np = 32 * tiles;
      std::vector<int> splits;
      for (int t : sx::mx_split_targets(&m, cus)) {
        const int s = sx::mx_splits(&m, t);
        CHECK(t >= 1 && s >= 8 && s <= 512 && s % 8 == 0);
        CHECK((tiles + s - 1) / s * s >= tiles);
        for (int o : splits) CHECK(o != s);
        splits.push_back(s);
      }
      // a whole number of tiles per split rounds the count down, by less
      // than one tile's worth, and a multiple of 8 up
      for (int want : {cus / 2, cus, 2 * cus})
        if (want >= 8 && want <= 512 && tiles >= 100 * want) {
          bool near = false;
          for (int s : splits) near |= s > want - want / 50 - 1 && s <= want + 7;
          CHECK(near);
        }
    }
}

}  // namespace

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "single_fresh") single_fresh();
  else if (what == "single_slow") single_slow();
  else if (what == "failed_calls_drain") failed_calls_drain();
  else if (what == "refused_memory") refused_memory();
  else if (what == "nothing_kept") nothing_kept();
  else if (what == "small_batches_pin_nothing") small_batches_pin_nothing();
  else if (what == "batch_errors") batch_errors();
  else if (what == "chains_rule") chains_rule();
  else if (what == "split_targets") split_targets();
  else return std::printf("unknown scenario\n"), 2;
  if (!g_bad) std::printf("ok\n");
  return g_bad != 0;
}
