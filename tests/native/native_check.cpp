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

const std::map<std::string, void (*)()> kScenarios = {
    {"no_allocations", no_allocations},
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
