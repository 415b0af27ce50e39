// Checks of the library that need control over the runtime's allocations and
// copies: this program defines hipMalloc and a few other functions itself, so that
// the library's calls come here first, can be counted, and can be made to fail on
// the host as they do when the device is full.  Nothing is launched that the
// library would not launch.
//
//   native_check SCENARIO
//
// prints its steps and, if every one holds, "ok SCENARIO" (status 0).
#include "cc4s_ccsd.h"
#include "contract.hpp"

#include <dlfcn.h>
#include <errno.h>
#include <hip/hip_runtime.h>
#include <pthread.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <random>
#include <string>
#include <thread>
#include <utility>
#include <vector>

// ---------------------------------------------------------------------------
// the runtime's functions
// ---------------------------------------------------------------------------

namespace {
std::mutex g_lock;
std::map<void *, size_t> g_sizes;
size_t g_held = 0;           // bytes of device memory
size_t g_total = 0;          // bytes the device has; 0: what it really has
long g_fail_at = 0;          // the allocation that fails, counted from arm(); 0: none
long g_count = 0;
bool g_failed = false;
long g_threads = -1;         // threads that may still be created; -1: any number
struct Copy {
  const void *dst, *src;
  size_t bytes;
};
bool g_record = false;
std::vector<Copy> g_copies;  // while g_record
std::vector<size_t> g_allocations;  // while g_record
std::atomic<long> g_launches{0};

template <typename F>
F real(const char *name) {
  return reinterpret_cast<F>(dlsym(RTLD_NEXT, name));
}

void arm(long fail_at) {
  std::lock_guard<std::mutex> l(g_lock);
  g_fail_at = fail_at;
  g_count = 0;
  g_failed = false;
}
size_t held() {
  std::lock_guard<std::mutex> l(g_lock);
  return g_held;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t bytes) {
  static const auto f = real<hipError_t (*)(void **, size_t)>("hipMalloc");
  {
    std::lock_guard<std::mutex> l(g_lock);
    ++g_count;
    if (g_record) g_allocations.push_back(bytes);
    if ((g_fail_at && g_count == g_fail_at) || (g_total && g_held + bytes > g_total)) {
      g_failed = true;
      *p = nullptr;
      return hipErrorOutOfMemory;
    }
  }
  const hipError_t e = f(p, bytes);
  if (e == hipSuccess) {
    std::lock_guard<std::mutex> l(g_lock);
    g_sizes[*p] = bytes;
    g_held += bytes;
  }
  return e;
}
hipError_t hipFree(void *p) {
  static const auto f = real<hipError_t (*)(void *)>("hipFree");
  const hipError_t e = f(p);
  std::lock_guard<std::mutex> l(g_lock);
  auto it = g_sizes.find(p);
  if (it != g_sizes.end()) {
    g_held -= it->second;
    g_sizes.erase(it);
  }
  return e;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind kind,
                          hipStream_t stream) {
  static const auto f =
      real<hipError_t (*)(void *, const void *, size_t, hipMemcpyKind, hipStream_t)>("hipMemcpyAsync");
  {
    std::lock_guard<std::mutex> l(g_lock);
    if (g_record) g_copies.push_back({dst, src, bytes});
  }
  return f(dst, src, bytes, kind, stream);
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds,
                           hipStream_t stream) {
  static const auto r =
      real<hipError_t (*)(const void *, dim3, dim3, void **, size_t, hipStream_t)>("hipLaunchKernel");
  ++g_launches;
  return r(f, grid, block, args, lds, stream);
}
int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*run)(void *), void *arg) noexcept {
  static const auto f = real<int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *)>(
      "pthread_create");
  {
    std::lock_guard<std::mutex> l(g_lock);
    if (g_threads == 0) return EAGAIN;
    if (g_threads > 0) --g_threads;
  }
  return f(t, a, run, arg);
}
hipError_t hipMemGetInfo(size_t *free_bytes, size_t *total_bytes) {
  static const auto f = real<hipError_t (*)(size_t *, size_t *)>("hipMemGetInfo");
  std::lock_guard<std::mutex> l(g_lock);
  if (!g_total) return f(free_bytes, total_bytes);
  *free_bytes = g_total > g_held ? g_total - g_held : 0;
  *total_bytes = g_total;
  return hipSuccess;
}
}

namespace {

// ---------------------------------------------------------------------------
// problems
// ---------------------------------------------------------------------------

#define CHECK(cond)                                                        \
  do {                                                                     \
    if (!(cond)) {                                                         \
      std::printf("FAILED %s:%d %s\n", __FILE__, __LINE__, #cond);         \
      std::fflush(stdout);                                                 \
      std::_Exit(1);                                                       \
    }                                                                      \
  } while (0)

void step(const std::string &what) {
  std::printf("%s\n", what.c_str());
  std::fflush(stdout);
}

struct Problem {
  bool cplx;
  int64_t o, v, G;
  std::vector<double> gamma, eps, T1, T2;  // complex interleaved where complex
  int es() const { return cplx ? 2 : 1; }
  size_t n1() const { return size_t(o) * v * es(); }
  size_t n2() const { return size_t(o) * o * v * v * es(); }
};

// a Hermitian (real field: symmetric) vertex and amplitudes with T_abij = T_baji,
// both exactly
Problem problem(bool cplx, int64_t o, int64_t v, int64_t G, unsigned seed) {
  Problem p{cplx, o, v, G, {}, {}, {}, {}};
  const int64_t n = o + v;
  std::mt19937_64 rng(seed);
  std::normal_distribution<double> d;
  p.gamma.assign(2 * G * n * n, 0.0);
  for (int64_t q = 0; q < n; ++q)
    for (int64_t r = 0; r <= q; ++r)
      for (int64_t g = 0; g < G; ++g) {
        const double re = 0.1 * d(rng) / std::sqrt(double(G)), im = 0.1 * d(rng) / std::sqrt(double(G));
        double *x = &p.gamma[2 * (g + G * (q + n * r))], *y = &p.gamma[2 * (g + G * (r + n * q))];
        x[0] = y[0] = re;
        x[1] = q == r && cplx ? 0.0 : im;
        y[1] = cplx ? -x[1] : x[1];
      }
  for (int64_t q = 0; q < n; ++q) p.eps.push_back(q < o ? -1.0 - 0.1 * q : 0.5 + 0.05 * q);
  for (size_t k = 0; k < p.n1(); ++k) p.T1.push_back(0.05 * d(rng));
  p.T2.assign(p.n2(), 0.0);
  const int es = p.es();
  for (int64_t a = 0; a < v; ++a)
    for (int64_t b = 0; b < v; ++b)
      for (int64_t i = 0; i < o; ++i)
        for (int64_t j = 0; j < o; ++j)
          for (int c = 0; c < es; ++c) {
            double &x = p.T2[es * (a + v * (b + v * (i + o * j))) + c];
            double &y = p.T2[es * (b + v * (a + v * (j + o * i))) + c];
            if (a + v * i <= b + v * j) x = y = 0.05 * d(rng);
          }
  return p;
}

struct Context {
  cc4s_ccsd_context *c = nullptr;
  Context(const Problem &p, const std::function<void(cc4s_ccsd_params &)> &set = {}) {
    cc4s_ccsd_params q;
    cc4s_ccsd_default_params(&q);
    q.field = p.cplx ? CC4S_FIELD_COMPLEX : CC4S_FIELD_REAL;
    q.No = p.o;
    q.Nv = p.v;
    q.NG = p.G;
    if (set) set(q);
    CHECK(cc4s_ccsd_create(&q, &c) == 0);
  }
  ~Context() { cc4s_ccsd_destroy(c); }
  operator cc4s_ccsd_context *() const { return c; }
};

using Out = std::pair<std::vector<double>, std::vector<double>>;  // R1, R2

int residuum(cc4s_ccsd_context *c, const Problem &p, Out &r) {
  r.first.assign(p.n1(), 0.0);
  r.second.assign(p.n2(), 0.0);
  return cc4s_ccsd_residuum(c, p.T1.data(), p.T2.data(), r.first.data(), r.second.data());
}
double rel(const std::vector<double> &a, const std::vector<double> &b) {
  double d = 0, m = 0;
  for (size_t k = 0; k < a.size(); ++k) {
    if (!std::isfinite(a[k])) return HUGE_VAL;
    d = std::max(d, std::fabs(a[k] - b[k]));
    m = std::max(m, std::fabs(b[k]));
  }
  return d / m;
}

// several slices of the ladder, the last one short
Problem mixed_problem() { return problem(true, 5, 23, 40, 3); }
void mixed(cc4s_ccsd_params &q) { q.precision = CC4S_PRECISION_MIXED; }

// ---------------------------------------------------------------------------
// scenarios
// ---------------------------------------------------------------------------

// A split residuum in which one allocation after the other fails leaves nothing
// behind: the next one on the same context is that of a fresh context, bit for bit.
void failed_split_pass() {
  setenv("CC4S_MIXED_MIN_FLOPS", "0", 1);  // every contraction is split
  const Problem p = mixed_problem();
  Problem other = p;  // what the failing pass is given: large dressed vertices
  for (double &x : other.T1) x *= 1e3;
  Out ref, r;
  {
    Context c(p, mixed);
    CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
    CHECK(residuum(c, p, ref) == 0);
  }
  long n = 0;
  for (bool failed = true; failed;) {
    Context c(p, mixed);
    CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
    arm(++n);
    const int rc = residuum(c, other, r);
    failed = g_failed;
    arm(0);
    if (!failed) break;
    step("allocation " + std::to_string(n) + (rc ? ": " : " passed over") +
         (rc ? cc4s_ccsd_last_error(c) : ""));
    CHECK(residuum(c, p, r) == 0);
    CHECK(r.first == ref.first && r.second == ref.second);
  }
  CHECK(n > 10);
}

// After a split pass that failed, the FP64 gradient is that of a fresh context.
void failed_split_pass_then_gradient() {
  setenv("CC4S_MIXED_MIN_FLOPS", "0", 1);
  const Problem p = mixed_problem();
  const size_t n = size_t(2) * p.G * (p.o + p.v) * (p.o + p.v);
  std::vector<double> ref(n), grad(n);
  Out r;
  for (long fail_at : {0L, 1L, 4L, 9L}) {
    Context c(p, mixed);
    CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
    CHECK(cc4s_ccsd_set_amplitudes(c, p.T1.data(), p.T2.data()) == 0);
    arm(fail_at);
    const int rc = fail_at % 2 ? cc4s_ccsd_iterate(c, nullptr) : residuum(c, p, r);
    CHECK(rc == (g_failed ? 1 : 0) && g_failed == (fail_at > 0));
    arm(0);
    step("allocation " + std::to_string(fail_at));
    CHECK(cc4s_ccsd_energy_grad_backward(c, nullptr, 0, (fail_at ? grad : ref).data(), 0, nullptr,
                                         CC4S_PRECISION_FP64) == 0);
    if (fail_at) CHECK(grad == ref);
  }
}

// New inputs whose allocations fail leave a context that refuses to go on, and takes
// inputs again.
void failed_inputs() {
  const Problem p = problem(true, 3, 9, 12, 4), q = problem(true, 3, 9, 12, 5);
  Out ref, r;
  {
    Context c(p);
    CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
    CHECK(residuum(c, p, ref) == 0);
  }
  long n = 0;
  for (bool failed = true; failed;) {
    Context c(p);
    CHECK(cc4s_ccsd_set_inputs(c, q.gamma.data(), q.eps.data()) == 0);
    CHECK(residuum(c, q, r) == 0);
    arm(++n);
    const int rc = cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data());
    failed = g_failed;
    arm(0);
    CHECK(rc == (failed ? 1 : 0));
    if (!failed) break;
    step("allocation " + std::to_string(n));
    CHECK(residuum(c, p, r) == 1);
    CHECK(cc4s_ccsd_iterate(c, nullptr) == 1);
    CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
    CHECK(residuum(c, p, r) == 0);
    CHECK(r == ref);
  }
  CHECK(n > 10);
}

// sizes at which the resident pair integrals are most of what a context holds (about
// 160 MB complex, 80 real, against 30 and 15 without them)
Problem resident_problem(bool cplx) { return problem(cplx, 5, 64, 24, 6); }
constexpr size_t kMiB = size_t(1) << 20;
constexpr size_t kReserve = size_t(6) << 30;  // what the library leaves free for a pass
void slabs(cc4s_ccsd_params &q) { q.integrals_slice_size = q.No; }  // the default's slices
constexpr double kTol = 1e-12;  // of one FP64 residuum in two orders of summation

// device memory one residuum leaves a context with, and the residuum
size_t held_after(const Problem &p, const std::function<void(cc4s_ccsd_params &)> &set, Out &r) {
  Context c(p, set);
  CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
  CHECK(residuum(c, p, r) == 0);
  return held();
}

// Where the resident integrals do not fit, the slab ladder gives what it gives where
// it is asked for.
void small_device() {
  for (bool cplx : {true, false}) {
    const Problem p = resident_problem(cplx);
    Out resident, slab, r;
    const size_t with = held_after(p, {}, resident), without = held_after(p, slabs, slab);
    step("held with " + std::to_string(with / kMiB) + " MiB, without " +
         std::to_string(without / kMiB));
    CHECK(with > 2 * without && rel(resident.first, slab.first) < kTol &&
          rel(resident.second, slab.second) < kTol);
    g_total = kReserve + with;  // less than twice what they need is free
    CHECK(held_after(p, {}, r) <= without);
    g_total = 0;
    CHECK(r == slab);
  }
}

// An allocation that fails while the resident integrals are formed, or later in the
// pass, costs the integrals and not the pass, and nothing of them stays allocated.
void failed_formation() {
  for (bool cplx : {true, false}) {
    const Problem p = resident_problem(cplx);
    Out ref, r;
    const size_t without = held_after(p, slabs, ref);
    bool started = false;
    long n = 0, done = 0;
    for (bool failed = true; failed;) {
      Context c(p);
      CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
      arm(++n);
      int rc = residuum(c, p, r);
      failed = g_failed;
      arm(0);
      if (!failed) break;
      step("allocation " + std::to_string(n) + (rc ? " fails" : " passed over"));
      if (rc) {
        CHECK(!started);  // before the first of the integrals' only
        continue;
      }
      started = true;
      ++done;
      CHECK(rel(r.first, ref.first) < kTol && rel(r.second, ref.second) < kTol);
      CHECK(held() <= without + 16 * kMiB);
      CHECK(residuum(c, p, r) == 0);
      CHECK(rel(r.first, ref.first) < kTol && rel(r.second, ref.second) < kTol);
    }
    CHECK(done > 6);
  }
}

// (T) goes on with fewer hole triples at a time where little memory is free.
void triples_little_memory() {
  const Problem p = resident_problem(true);
  double ref = 0, e = 0;
  for (size_t room : {size_t(0), 60 * kMiB, 40 * kMiB}) {
    Context c(p, slabs);
    CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
    CHECK(cc4s_ccsd_set_amplitudes(c, p.T1.data(), p.T2.data()) == 0);
    g_total = room ? held() + room : 0;  // the ppph integrals take 20 MiB of it
    step("room " + std::to_string(room / kMiB));
    CHECK(cc4s_ccsd_triples(c, room ? &e : &ref) == 0);
    if (room) CHECK(std::fabs(e - ref) <= kTol * std::fabs(ref));
    g_total = 0;
  }
}

// The integrals that one context keeps do not take room from another context's
// history or from the context's own later calls: they are given back.
void given_back() {
  const Problem p = resident_problem(true);
  const size_t n = size_t(2) * p.G * (p.o + p.v) * (p.o + p.v);
  Out ref, r;
  double triples_ref = 0, triples = 0;
  std::vector<double> grad_ref(n), grad(n);
  {
    Context c(p, slabs);
    CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
    CHECK(cc4s_ccsd_set_amplitudes(c, p.T1.data(), p.T2.data()) == 0);
    CHECK(residuum(c, p, ref) == 0);
    CHECK(cc4s_ccsd_triples(c, &triples_ref) == 0);
    CHECK(cc4s_ccsd_energy_grad_backward(c, nullptr, 0, grad_ref.data(), 0, nullptr,
                                         CC4S_PRECISION_FP64) == 0);
  }
  auto right = [&](cc4s_ccsd_context *c) {
    CHECK(residuum(c, p, r) == 0);
    CHECK(rel(r.first, ref.first) < kTol && rel(r.second, ref.second) < kTol);
  };
  auto resident = [&](cc4s_ccsd_context *c) {  // a pass that forms them
    g_total = 0;
    CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
    CHECK(cc4s_ccsd_set_amplitudes(c, p.T1.data(), p.T2.data()) == 0);
    const size_t before = held();
    right(c);
    CHECK(held() > before + 100 * kMiB);
  };
  Context a(p);
  resident(a);
  step("another context's history");
  {
    const size_t before = held();
    size_t other = 0;
    {
      Context b(p);
      CHECK(cc4s_ccsd_set_inputs(b, p.gamma.data(), p.eps.data()) == 0);
      other = held() - before;
    }
    g_total = before + kReserve + other - kMiB;  // the history is short of 1 MiB
    Context b(p);
    CHECK(cc4s_ccsd_set_inputs(b, p.gamma.data(), p.eps.data()) == 0);
    cc4s_ccsd_iteration it;
    CHECK(cc4s_ccsd_iterate(b, &it) == 0);
    CHECK(it.diis_placement == 0 && held() < before);
    right(a);
    right(b);
  }
  resident(a);
  step("new inputs");
  g_total = held() + 40 * kMiB;
  CHECK(cc4s_ccsd_set_inputs(a, p.gamma.data(), p.eps.data()) == 0);
  right(a);
  resident(a);
  step("(T)");
  g_total = held() + 4 * kMiB;  // the ppph integrals take 20 MiB
  CHECK(cc4s_ccsd_triples(a, &triples) == 0);
  CHECK(std::fabs(triples - triples_ref) <= kTol * std::fabs(triples_ref));
  right(a);
  resident(a);
  step("gradient");
  g_total = held() + kMiB / 4;
  CHECK(cc4s_ccsd_energy_grad_backward(a, nullptr, 0, grad.data(), 0, nullptr,
                                       CC4S_PRECISION_FP64) == 0);
  CHECK(rel(grad, grad_ref) < kTol);
  right(a);
  g_total = 0;
}

// A context that forms its integrals again and again on one thread, and on another
// thread contexts whose history needs their room: both stay right.
void given_back_between_threads() {
  const Problem p = problem(true, 4, 40, 16, 7), q = problem(true, 10, 40, 16, 8);
  auto long_history = [](cc4s_ccsd_params &x) { x.max_residua = 11; };
  Out refp, refq, r;
  const size_t base = held();
  const size_t without = held_after(p, slabs, refp);
  const size_t resident = held_after(p, {}, r) - without;
  held_after(q, slabs, refq);
  size_t other = 0;
  {
    Context b(q, long_history);
    CHECK(cc4s_ccsd_set_inputs(b, q.gamma.data(), q.eps.data()) == 0);
    other = held() - base;
  }
  step("integrals " + std::to_string(resident / kMiB) + " MiB, the other context " +
       std::to_string(other / kMiB));
  CHECK(other > resident + 4 * kMiB);
  // the history is short of 3 MiB beside the integrals
  g_total = kReserve + without + resident + other - 3 * kMiB;
  std::thread first([&] {
    Context a(p);
    Out x;
    for (int n = 0; n < 12; ++n) {
      CHECK(cc4s_ccsd_set_inputs(a, p.gamma.data(), p.eps.data()) == 0);
      for (int k = 0; k < 3; ++k) {
        CHECK(residuum(a, p, x) == 0);
        CHECK(rel(x.first, refp.first) < kTol && rel(x.second, refp.second) < kTol);
      }
    }
  });
  std::thread second([&] {
    Out x;
    for (int n = 0; n < 12; ++n) {
      Context b(q, long_history);
      CHECK(cc4s_ccsd_set_inputs(b, q.gamma.data(), q.eps.data()) == 0);
      cc4s_ccsd_iteration it;
      CHECK(cc4s_ccsd_iterate(b, &it) == 0);
      CHECK(it.diis_placement == 0);
      CHECK(residuum(b, q, x) == 0);
      CHECK(rel(x.first, refq.first) < kTol && rel(x.second, refq.second) < kTol);
    }
  });
  first.join();
  second.join();
  g_total = 0;
}

// 17 MiB of amplitudes, any bytes: over the ring's threshold, a short last chunk
Problem transfer_problem() {
  Problem p{true, 7, 151, 2, {}, {}, {}, {}};
  std::mt19937_64 rng(9);
  for (size_t k = 0; k < p.n1(); ++k) p.T1.push_back(double(rng()));
  for (size_t k = 0; k < p.n2(); ++k) p.T2.push_back(double(rng()));
  return p;
}

// The caller's pinned memory is copied at once, not through the ring.
void pinned_copies() {
  const Problem p = transfer_problem();
  const size_t b1 = p.n1() * 8, b2 = p.n2() * 8;
  double *h1 = nullptr, *h2 = nullptr;
  CHECK(hipHostMalloc(reinterpret_cast<void **>(&h1), b1, hipHostMallocDefault) == hipSuccess);
  CHECK(hipHostMalloc(reinterpret_cast<void **>(&h2), b2, hipHostMallocDefault) == hipSuccess);
  std::memcpy(h1, p.T1.data(), b1);
  std::memcpy(h2, p.T2.data(), b2);
  Context c(p);
  g_record = true;
  CHECK(cc4s_ccsd_set_amplitudes(c, h1, h2) == 0);
  std::memset(h2, 0, b2);
  CHECK(cc4s_ccsd_get_amplitudes(c, h1, h2) == 0);
  g_record = false;
  int up = 0, down = 0;
  for (const Copy &x : g_copies) {
    up += x.src == h2 && x.bytes == b2;
    down += x.dst == h2 && x.bytes == b2;
  }
  CHECK(up == 1 && down == 1);
  CHECK(std::memcmp(h1, p.T1.data(), b1) == 0 && std::memcmp(h2, p.T2.data(), b2) == 0);
  CHECK(hipHostFree(h1) == hipSuccess && hipHostFree(h2) == hipSuccess);
}

// Copies of pageable memory with the threads that the system grants, and with none.
void copies_without_threads() {
  const Problem p = transfer_problem();
  Context c(p);
  std::vector<double> T1(p.n1()), T2(p.n2());
  for (long granted : {-1L, 0L, 1L, 3L}) {
    for (int up = 0; up < 2; ++up) {
      step(std::to_string(granted) + (up ? " up" : " down"));
      T2.assign(p.n2(), 0.0);
      g_threads = up ? granted : -1;
      CHECK(cc4s_ccsd_set_amplitudes(c, p.T1.data(), p.T2.data()) == 0);
      g_threads = up ? -1 : granted;
      CHECK(cc4s_ccsd_get_amplitudes(c, T1.data(), T2.data()) == 0);
      g_threads = -1;
      CHECK(T1 == p.T1 && T2 == p.T2);
    }
  }
}

// A small gradient takes its two products in one launch, beside the weights and the
// dots of two blocks in two launches each.
void gradient_launches() {
  const Problem p = problem(true, 3, 12, 30, 4);
  const size_t n = size_t(2) * p.G * (p.o + p.v) * (p.o + p.v);
  std::vector<double> grad(n), S(p.G);
  Context c(p);
  CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
  CHECK(cc4s_ccsd_set_amplitudes(c, p.T1.data(), p.T2.data()) == 0);
  long before = 0;
  for (int k = 0; k < 2; ++k) {  // the second call has its plans
    before = g_launches;
    CHECK(cc4s_ccsd_energy_grad_backward(c, nullptr, 0, grad.data(), 0, S.data(),
                                         CC4S_PRECISION_FP64) == 0);
  }
  step(std::to_string(g_launches - before) + " launches");
  CHECK(g_launches - before > 0 && g_launches - before <= 6);
}

// New inputs allocate nothing that they do not keep.
void inputs_keep_what_they_allocate() {
  for (bool cplx : {true, false}) {
    const Problem p = problem(cplx, 2, 5, 4, 4);  // no partial sums, whose buffer grows
    Context c(p);
    const size_t before = g_sizes.size();
    arm(0);
    CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
    step(std::to_string(g_count) + " allocations, " + std::to_string(g_sizes.size() - before) + " kept");
    CHECK(size_t(g_count) == g_sizes.size() - before);
  }
}

// Calls repeated on a context allocate nothing on the device.
void no_allocations() {
  const Problem p = problem(true, 3, 9, 12, 4), q2 = problem(true, 3, 9, 12, 5);
  for (int method : {CC4S_METHOD_CCSD, CC4S_METHOD_DRCCD}) {
    Context c(p, [&](cc4s_ccsd_params &q) { q.method = method; });
    Out r;
    std::vector<double> T1(p.n1()), T2(p.n2());
    CHECK(cc4s_ccsd_set_inputs(c, p.gamma.data(), p.eps.data()) == 0);
    for (int n = 0; n < 2; ++n) {
      arm(0);  // counts from here
      const Problem &t = n ? q2 : p;
      CHECK(cc4s_ccsd_set_amplitudes(c, t.T1.data(), t.T2.data()) == 0);
      CHECK(cc4s_ccsd_iterate(c, nullptr) == 0);
      CHECK(residuum(c, t, r) == 0);
      CHECK(cc4s_ccsd_get_amplitudes(c, T1.data(), T2.data()) == 0);
      step("method " + std::to_string(method) + ": " + std::to_string(g_count) + " allocations");
    }
    CHECK(g_count == 0);
  }
}

// ---------------------------------------------------------------------------
// contraction kernels
// ---------------------------------------------------------------------------

using namespace cc4s_amd;
using Z = std::complex<double>;

// C = alpha op(A) op(B) + beta op(D) on the host for some rows
struct Product {
  bool cplx;
  int64_t M, N, K;
  std::vector<Z> A, B, D;  // [m][k], [n][k], [m][n]
  Product(bool c, int64_t m, int64_t n, int64_t k) : cplx(c), M(m), N(n), K(k) {
    std::mt19937_64 rng(m + 3 * n + 7 * k);
    std::uniform_real_distribution<double> d(-1, 1);
    for (std::vector<Z> *x : {&A, &B, &D}) {
      x->resize(x == &A ? M * K : x == &B ? N * K : M * N);
      for (Z &z : *x) z = Z(d(rng), c ? d(rng) : 0.0);
    }
  }
  Z at(int64_t m, int64_t n, double alpha, bool conjA, bool conjB, double beta, bool conjD) const {
    const double fa = conjA ? -1 : 1, fb = conjB ? -1 : 1;
    const Z *a = &A[m * K], *b = &B[n * K];
    double re = 0, im = 0;
    for (int64_t k = 0; k < K; ++k) {
      re += a[k].real() * b[k].real() - fa * fb * a[k].imag() * b[k].imag();
      im += fb * a[k].real() * b[k].imag() + fa * a[k].imag() * b[k].real();
    }
    const Z d = beta == 0.0 ? Z() : conjD ? std::conj(D[m * N + n]) : D[m * N + n];
    return Z(alpha * re, alpha * im) + beta * d;
  }
  // Largest error of C over every `step`-th row and the last, in units of what
  // rounding allows: partial sums of K products of numbers up to one grow as sqrt(K)
  // / 3, their sqrt(K) roundings come to about K 2^-53 / 5, the largest of 10^5
  // elements to four or five times that, two orders of summation and the three-product
  // form's larger terms to four times more; and a few roundings at the end.
  double error(const std::vector<Z> &C, int64_t ld, int64_t step, double alpha, bool conjA,
               bool conjB, double beta, bool conjD) const {
    double e = 0;
    for (int64_t m = 0; m < M; m = m == M - 1 ? M : std::min(m + step, M - 1))
      for (int64_t n = 0; n < N; ++n) {
        const double x = std::abs(C[m * ld + n] - at(m, n, alpha, conjA, conjB, beta, conjD));
        if (!(x < HUGE_VAL)) return HUGE_VAL;
        e = std::max(e, x);
      }
    return e / ((8.0 * K + 16.0) * 0x1p-53);
  }
};
std::vector<double> packed(const std::vector<Z> &x, bool cplx) {
  std::vector<double> r;
  for (const Z &z : x) {
    r.push_back(z.real());
    if (cplx) r.push_back(z.imag());
  }
  return r;
}
template <typename T>
DeviceBuffer upload(const std::vector<T> &x) {
  DeviceBuffer b(x.size() * sizeof(T));
  CHECK(hipMemcpy(b.get(), x.data(), x.size() * sizeof(T), hipMemcpyHostToDevice) == hipSuccess);
  return b;
}

// Every tile of the GETT kernel, in every orientation, whole, with K split and with
// the last tiles cut along K (the fourth part of four then has no k left), at sizes
// that are no multiple of any tile, rows longer than what is used of them.
void gett_tiles() {
  const int64_t M = 323, N = 261;
  const int tiles[2][3][2] = {{{128, 128}, {64, 64}, {32, 32}}, {{128, 64}, {64, 64}, {32, 32}}};
  hipStream_t st;
  CHECK(hipStreamCreate(&st) == hipSuccess);
  for (int64_t K : {131, 70, 17, 1})
    for (bool cplx : {false, true}) {
      const Product P(cplx, M, N, K);
      const int64_t Kpad = (K + 15) / 16 * 16 + 80;  // whole stages, and five further
      const int64_t lk = K + 3, lm = M + 5, ln = N + 7;
      auto spread = [&](const std::vector<Z> &x, int64_t rows, int64_t cols, int64_t ld, bool turn) {
        std::vector<Z> r((turn ? cols : rows) * ld, Z(NAN, NAN));
        for (int64_t i = 0; i < rows; ++i)
          for (int64_t j = 0; j < cols; ++j) r[turn ? j * ld + i : i * ld + j] = x[i * cols + j];
        return packed(r, cplx);
      };
      auto table = [&](int64_t n, int64_t pad, int64_t stride) {
        std::vector<int64_t> t(std::max(n, pad), 0);
        for (int64_t i = 0; i < n; ++i) t[i] = i * stride;
        return upload(t);
      };
      const DeviceBuffer D = upload(spread(P.D, M, N, ln, false));
      const DeviceBuffer rowC = table(M, 0, ln), colC = table(N, 0, 1);
      for (int orient = 0; orient < 4; ++orient) {
        const bool ak = orient & 2, bk = orient & 1;
        const DeviceBuffer A = upload(spread(P.A, M, K, ak ? lk : lm, !ak)),
                           B = upload(spread(P.B, N, K, bk ? lk : ln, !bk));
        const DeviceBuffer rowA = table(M, 0, ak ? lk : 1), colA = table(K, Kpad, ak ? 1 : lm),
                           rowB = table(K, Kpad, bk ? 1 : ln), colB = table(N, 0, bk ? lk : 1);
        double worst = 0;
        for (int t = 0; t < 3; ++t) {
          const int64_t BM = tiles[cplx][t][0], BN = tiles[cplx][t][1];
          const int64_t count = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
          struct Mode {
            int splits, cut;
            bool add, other;  // beta, to another tensor
          };
          for (const Mode mode : {Mode{1, 1, false, false}, Mode{1, 1, true, false},
                                  Mode{3, 1, true, true}, Mode{1, 2, true, false},
                                  Mode{1, 4, true, true}, Mode{40, 1, false, false}}) {
            const int64_t full = count - count / 3;
            GettLaunch L;
            L.field = cplx ? Field::Complex : Field::Real;
            L.A = A.get();
            L.B = B.get();
            // C starts as D where that is added in place, as NaN where it is not read
            DeviceBuffer C = upload(mode.add && !mode.other
                                        ? spread(P.D, M, N, ln, false)
                                        : std::vector<double>(M * ln * (cplx ? 2 : 1), NAN));
            L.C = C.get();
            L.rowA = rowA.as<int64_t>();
            L.colA = colA.as<int64_t>();
            L.rowB = rowB.as<int64_t>();
            L.colB = colB.as<int64_t>();
            L.rowC = rowC.as<int64_t>();
            L.colC = colC.as<int64_t>();
            L.M = M;
            L.N = N;
            L.K = K;
            L.splits = mode.splits;
            L.tile = t;
            if (mode.cut > 1) {
              L.full_tiles = full;
              L.tail_splits = mode.cut;
            }
            const size_t parts = mode.splits > 1 ? size_t(mode.splits) * M * N
                                 : mode.cut > 1  ? size_t(mode.cut) * (count - full) * BM * BN
                                                 : 0;
            DeviceBuffer W = upload(std::vector<double>(parts * (cplx ? 2 : 1) + 1, NAN));
            L.W = W.get();
            L.alpha = 0.75;
            L.beta = mode.add ? -0.5 : 0.0;
            L.conjA = cplx && t != 1;
            L.conjB = cplx && mode.add;
            L.a_kcontig = ak;
            L.b_kcontig = bk;
            if (mode.other) {
              L.D = D.get();
              L.rowD = rowC.as<int64_t>();
              L.colD = colC.as<int64_t>();
              L.conjD = cplx;
            }
            launch_gett(L, st);
            std::vector<double> h(M * ln * (cplx ? 2 : 1));
            CHECK(hipStreamSynchronize(st) == hipSuccess);
            CHECK(hipMemcpy(h.data(), C.get(), h.size() * 8, hipMemcpyDeviceToHost) == hipSuccess);
            std::vector<Z> z(M * ln);
            for (int64_t i = 0; i < M * ln; ++i) z[i] = cplx ? Z(h[2 * i], h[2 * i + 1]) : Z(h[i], 0);
            const double e = P.error(z, ln, 7, L.alpha, L.conjA, L.conjB, L.beta, L.conjD);
            if (e > 1.0)
              step("tile " + std::to_string(t) + " splits " + std::to_string(mode.splits) + " cut " +
                   std::to_string(mode.cut) + " error " + std::to_string(e));
            worst = std::max(worst, e);
          }
        }
        std::printf("K %d %s orientation %d: %.2f\n", int(K), cplx ? "complex" : "real", orient, worst);
        std::fflush(stdout);
        CHECK(worst <= 1.0);
      }
    }
  CHECK(hipStreamDestroy(st) == hipSuccess);
}

// Sizes that the planner sends to each tile, whole, split and cut, in every
// orientation: that it does, and the products.
void gett_planner() {
  enum { Whole, Split, Cut };
  struct Size {
    bool cplx;
    int64_t M, N, K;
    const char *tile;
    int mode;
  };
  hipStream_t st;
  CHECK(hipStreamCreate(&st) == hipSuccess);
  for (const Size &x : std::vector<Size>{{false, 1677, 3921, 40, "", Whole},
                                         {false, 3861, 2128, 695, "", Cut},
                                         {false, 3512, 304, 40, "_t64", Whole},
                                         {false, 679, 366, 502, "_t64", Split},
                                         {false, 3886, 798, 183, "_t64", Cut},
                                         {false, 442, 357, 44, "_t32", Whole},
                                         {false, 365, 314, 999, "_t32", Split},
                                         {true, 2058, 748, 574, "", Whole},
                                         {true, 2226, 329, 1159, "", Split},
                                         {true, 2400, 1089, 755, "", Cut},
                                         {true, 864, 1187, 40, "_t64", Whole},
                                         {true, 565, 478, 655, "_t64", Split},
                                         {true, 1111, 1862, 185, "_t64", Cut},
                                         {true, 352, 546, 53, "_t32", Whole},
                                         {true, 307, 335, 709, "_t32", Split},
                                         {true, 305, 3310, 194, "_t32", Cut}}) {
    const Field f = x.cplx ? Field::Complex : Field::Real;
    const Product P(x.cplx, x.M, x.N, x.K);
    const size_t result = size_t(x.M) * x.N * scalar_bytes(f);
    auto turned = [&](const std::vector<Z> &y, int64_t rows) {
      std::vector<Z> r(y.size());
      const int64_t cols = y.size() / rows;
      for (int64_t i = 0; i < rows; ++i)
        for (int64_t j = 0; j < cols; ++j) r[j * rows + i] = y[i * cols + j];
      return packed(r, x.cplx);
    };
    for (int orient = 0; orient < 4; ++orient) {
      const bool ak = orient & 2, bk = orient & 1;
      // first index fastest: "km" is k-contiguous; C is "nm", n-contiguous
      DeviceBuffer A = upload(ak ? packed(P.A, x.cplx) : turned(P.A, x.M)),
                   B = upload(bk ? packed(P.B, x.cplx) : turned(P.B, x.N)), C(result);
      const View a = ak ? dense_view(A.get(), f, "km", {x.K, x.M}) : dense_view(A.get(), f, "mk", {x.M, x.K}),
                 b = bk ? dense_view(B.get(), f, "kn", {x.K, x.N}) : dense_view(B.get(), f, "nk", {x.N, x.K});
      ContractionEngine E(st);
      E.set_profiling(true);
      g_allocations.clear();
      g_record = true;
      E.contract(0.75, a, b, 0.0, dense_view(C.get(), f, "nm", {x.N, x.M}));
      g_record = false;
      const std::string name = std::string("gett_") + (x.cplx ? "c64" : "f64") + (ak ? "_ak" : "_am") +
                               (bk ? "_bk" : "_bn") + x.tile;
      CHECK(E.timings().size() == 1 && E.timings().count(name) == 1);
      // the offset tables' chunk, and the partial sums if there are any: of whole
      // results, or of whole tiles
      CHECK(g_allocations.size() == (x.mode == Whole ? 1 : 2));
      if (x.mode != Whole) CHECK((g_allocations[1] % result == 0) == (x.mode == Split));
      std::vector<double> h(size_t(x.M) * x.N * (x.cplx ? 2 : 1));
      CHECK(hipMemcpy(h.data(), C.get(), result, hipMemcpyDeviceToHost) == hipSuccess);
      std::vector<Z> z(size_t(x.M) * x.N);
      for (size_t i = 0; i < z.size(); ++i) z[i] = x.cplx ? Z(h[2 * i], h[2 * i + 1]) : Z(h[i], 0);
      const double e = P.error(z, x.N, x.M / 40, 0.75, false, false, 0.0, false);
      std::printf("%s %d x %d x %d: %.2f\n", name.c_str(), int(x.M), int(x.N), int(x.K), e);
      std::fflush(stdout);
      CHECK(e <= 1.0);
    }
  }
  CHECK(hipStreamDestroy(st) == hipSuccess);
}

const std::map<std::string, void (*)()> kScenarios = {
    {"gett_tiles", gett_tiles},
    {"gett_planner", gett_planner},
    {"no_allocations", no_allocations},
    {"gradient_launches", gradient_launches},
    {"inputs_keep_what_they_allocate", inputs_keep_what_they_allocate},
    {"pinned_copies", pinned_copies},
    {"copies_without_threads", copies_without_threads},
    {"given_back_between_threads", given_back_between_threads},
    {"small_device", small_device},
    {"failed_formation", failed_formation},
    {"given_back", given_back},
    {"triples_little_memory", triples_little_memory},
    {"failed_inputs", failed_inputs},
    {"failed_split_pass_then_gradient", failed_split_pass_then_gradient},
    {"failed_split_pass", failed_split_pass},
};

}  // namespace

int main(int argc, char **argv) {
  const auto it = kScenarios.find(argc > 1 ? argv[1] : "");
  if (it == kScenarios.end()) {
    for (const auto &s : kScenarios) std::printf("%s\n", s.first.c_str());
    return 2;
  }
  it->second();
  std::printf("ok %s\n", argv[1]);
  return 0;
}
