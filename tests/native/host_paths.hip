// The library's host paths on a CPU: its sources compiled for the host alone and
// linked against the stand-in HIP runtime below.  Device memory is host memory,
// copies are made at once, kernels are only noted, except that the solver's test
// kernels report the iteration at which a solve is to converge.  A chosen runtime
// call can be made to fail, so that every error path of an entry point runs.
//
// One scenario per run: host_paths <scenario>; exit code 0 and a last line "ok".
#include <stdio.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <functional>
#include <map>
#include <new>
#include <set>
#include <string>
#include <vector>

#include "../../cvc_amd/csrc/dslash.hip"
#include "../../cvc_amd/csrc/solver.hip"

namespace fake {

// ---------------------------------------------------------------- state
std::map<void *, size_t> dev, pinned;          // live allocations
std::set<void *> events, streams;
std::map<const void *, std::string> &names() {   // kernels by host stub (registered before main)
  static std::map<const void *, std::string> n;
  return n;
}
struct Copies {                                // device-to-host copies of a stream
  long issued = 0, ended = 0;
};
std::map<void *, Copies> to_host;
std::map<void *, std::pair<void *, long>> recorded;   // event: stream, copies issued before it
struct Launch {
  std::string name;
  dim3 grid, block;
  std::vector<uint32_t> cols;                  // k_copy_columns: columns of both sets, first ones, count
};
std::vector<Launch> launches;
hipError_t last = hipSuccess;
long allocs = 0, fail_alloc = 0;               // allocation number that fails (0: none)
size_t capacity = SIZE_MAX, used = 0;          // device memory
long calls = 0, fail_call = 0;                 // any runtime call that can fail, allocations among them
long news = 0, fail_new = 0;                   // the library's host allocations on the main thread
thread_local bool counted = false;
struct Own {                                   // the stand-in's own allocations are not counted
  bool was = counted;
  Own() { counted = false; }
  ~Own() { counted = was; }
};

// convergence that the solver's kernels report
int conv_it = 3, conv_rhs = 1 << 30;           // columns below conv_rhs converge at iteration conv_it

hipError_t call() { return ++calls == fail_call ? last = hipErrorUnknown : hipSuccess; }
hipError_t alloc(std::map<void *, size_t> &live, void **p, size_t n) {
  const Own own;
  if (++calls == fail_call || ++allocs == fail_alloc || (&live == &dev && n > capacity - used)) return last = hipErrorOutOfMemory;
  *p = calloc(n ? n : 1, 1);
  live[*p] = n;
  if (&live == &dev) used += n;
  return hipSuccess;
}
hipError_t release(std::map<void *, size_t> &live, void *p) {
  if (!p) return hipSuccess;
  if (!live.count(p)) {
    fprintf(stderr, "free of %p, which is not allocated\n", p);
    abort();
  }
  if (&live == &dev) used -= live[p];
  live.erase(p);
  free(p);
  return hipSuccess;
}

template <typename T> T arg(void **a, int k) { return *(T *)a[k]; }

void kernel(const std::string &n, dim3 grid, void **a) {
  using namespace cvchip;
  const bool test = n.find("k_sc_test") != std::string::npos, beta = n.find("k_sc_beta") != std::string::npos;
  if (test || beta) {
    RhsState *st = arg<RhsState *>(a, 0);
    RhsMirror *m = arg<RhsMirror *>(a, 1);
    const int it = arg<int>(a, beta ? 5 : 4), mixed = beta ? arg<int>(a, 6) : 0;
    for (int r = 0; r < (int)grid.x; r++) {
      if (!mixed && it >= conv_it && r < conv_rhs && !st[r].done) st[r].done = 1, st[r].iter = it;
      st[r].upd = mixed && !st[r].done && (it == 1 || it == conv_it);
      m[r].norm = m[r].normb = 1.;
      m[r].done = st[r].done;
      m[r].upd = st[r].upd;
      m[r].seq = it + 1;
    }
  }
  if (n.find("k_sc_reliable") != std::string::npos) {
    RhsState *st = arg<RhsState *>(a, 0);
    const int N = arg<int>(a, 2), it = arg<int>(a, 3);
    for (int r = 0; r < N && r < conv_rhs; r++)
      if (it >= conv_it && !st[r].done) st[r].done = 1, st[r].iter = it;
  }
}

}  // namespace fake

// ---------------------------------------------------------------- the runtime
using namespace fake;
extern "C" {
hipError_t hipMalloc(void **p, size_t n) { return alloc(dev, p, n); }
hipError_t hipFree(void *p) { return release(dev, p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return alloc(pinned, p, n); }
hipError_t hipHostFree(void *p) { return release(pinned, p); }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError(void) {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static char buf[1 << 21];
  return *p = buf, hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  if (const hipError_t e_ = call()) return e_;
  const Own own;
  *s = (hipStream_t)malloc(1);
  streams.insert(*s);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return streams.erase(s), to_host.erase(s), free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  if (const hipError_t e_ = call()) return e_;
  const Own own;
  to_host[s].ended = to_host[s].issued;
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return call(); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  if (const hipError_t e_ = call()) return e_;
  const Own own;
  *e = (hipEvent_t)malloc(1);
  events.insert(*e);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return events.erase(e), recorded.erase(e), free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (const hipError_t e_ = call()) return e_;
  const Own own;
  recorded[e] = {s, to_host[s].issued};
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  if (const hipError_t e_ = call()) return e_;
  const Own own;
  const auto r = recorded[e];
  if (r.second > to_host[r.first].ended) to_host[r.first].ended = r.second;
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) { return *t = 0.f, hipSuccess; }
// (what kernels alone would use stays zero, so that large sets are never touched)
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t q) {
  if (const hipError_t e_ = call()) return e_;
  const Own own;
  if (k == hipMemcpyDeviceToHost) to_host[q].issued++;
  if (k != hipMemcpyDeviceToDevice) memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) {
  if (const hipError_t e_ = call()) return e_;
  if (n < (size_t)1 << 20) memset(p, v, n);
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t, hipStream_t) {
  if (const hipError_t e_ = call()) return e_;
  const Own own;
  launches.push_back({names()[f], g, b, {}});
  if (names()[f].find("k_copy_columns") != std::string::npos)
    for (int k = 3; k < 8; k++) launches.back().cols.push_back(arg<uint32_t>(a, k));
  kernel(names()[f], g, a);
  return hipSuccess;
}
struct Config {
  dim3 g, b;
  size_t lds;
  hipStream_t s;
};
static Config config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) { return config = {g, b, lds, s}, hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
  *g = config.g, *b = config.b, *lds = config.lds, *s = config.s;
  return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) {
  static void *m;
  return &m;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
  names()[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}

void *operator new(size_t n) {
  if (counted && ++news == fail_new) throw std::bad_alloc();
  void *p = malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

// ---------------------------------------------------------------- scenarios
#define CHECK(cond, ...)                                                \
  do {                                                                  \
    if (!(cond)) {                                                      \
      fprintf(stderr, "%s:%d: %s: ", __FILE__, __LINE__, #cond);        \
      fprintf(stderr, __VA_ARGS__);                                     \
      fprintf(stderr, " (last error: %s)\n", cvchip_last_error());      \
      exit(1);                                                          \
    }                                                                   \
  } while (0)

struct Ctx {
  cvchip_ctx *c = nullptr;
  size_t V;
  std::vector<double> gauge;
  explicit Ctx(int T, int X, int Y, int Z) : V((size_t)T * X * Y * Z), gauge(72 * V) {
    const int d[4] = {T, X, Y, Z};
    const double bc[4] = {1, 0, 0, 0};
    CHECK(!cvchip_ctx_create(&c, d, bc, 0.15, 0.01), "create");
    CHECK(!cvchip_set_gauge(c, gauge.data()), "gauge");
  }
  ~Ctx() {
    cvchip_ctx_destroy(c);
    CHECK(dev.empty() && pinned.empty() && events.empty() && streams.empty(),
          "left behind: %zu device, %zu pinned, %zu events, %zu streams", dev.size(), pinned.size(), events.size(),
          streams.size());
  }
};

static int solve(Ctx &x, int nrhs, int prec, unsigned flags, cvchip_stats *st = nullptr, bool her = true) {
  std::vector<double> b(24 * x.V * nrhs), y(b.size());
  cvchip_stats s;
  return (her ? cvchip_invert_Qtm_her : cvchip_invert_Qtm)(x.c, y.data(), b.data(), nrhs, 1e-20, 20, prec, 0.1, flags,
                                                           st ? st : &s);
}

// scratch that does not fit beside the context's idle buffers takes their place, and
// one that does not fit at all leaves no error for the next call to find
static void scratch() {
  using namespace cvchip;
  int (*const ensure[3])(cvchip_ctx *, size_t) = {ensure_stage, ensure_red, ensure_red2};
  for (auto f : ensure) {
    Ctx x(4, 2, 2, 4);
    Field idle;
    CHECK(!field_alloc(x.c, idle, 60, CVCHIP_PREC_F64), "field");
    field_free(idle);
    capacity = used;
    CHECK(!f(x.c, idle.bytes / 2), "scratch beside idle buffers");
    CHECK(f(x.c, 4 * idle.bytes) == CVCHIP_ERR_OOM, "scratch beyond the device");
    capacity = SIZE_MAX;
    CHECK(hipGetLastError() == hipSuccess, "error left behind");
  }
}

// a solve none of whose allocations fails works after one that lacked any of them
static void solver_buffers() {
  for (long k = 1;; k++) {
    fprintf(stderr, "allocation %ld refused\n", k);
    Ctx x(4, 2, 2, 4);
    fail_alloc = allocs + k;
    const int rc = solve(x, 3, CVCHIP_PREC_F64, 0);
    const bool reached = allocs >= fail_alloc;
    fail_alloc = 0;
    CHECK(reached ? rc < 0 : rc >= 0, "allocation %ld: %d", k, rc);
    CHECK(solve(x, 3, CVCHIP_PREC_F64, 0) >= 0, "solve after allocation %ld failed", k);
    if (!reached) break;
  }
}

// Entry points that solve, on small sets; the host arrays are made once.
struct Entry {
  const char *name;
  std::function<int(Ctx &)> call;
};
static std::vector<Entry> entries() {
  static std::vector<double> conn(1 << 16), force(1 << 16), store(1 << 20), b(1 << 14), y(1 << 14);
  static double contact[8], L, dmu;
  static double *props[120];
  static const int src[4] = {1, 0, 1, 2}, mom[3] = {0, 1, 0};
  for (int k = 0; k < 120; k++) props[k] = &store[4096 * k];
  std::vector<Entry> v;
  for (int her = 0; her < 2; her++)
    for (unsigned f : {0u, CVCHIP_SOLVE_LAGGED, CVCHIP_SOLVE_EO})
      for (int prec = 0; prec < 3; prec++)
        v.push_back({her ? "invert_Qtm_her" : "invert_Qtm", [=](Ctx &x) {
                       cvchip_stats st;
                       return (her ? cvchip_invert_Qtm_her : cvchip_invert_Qtm)(x.c, y.data(), b.data(), 2, 1e-20, 20, prec,
                                                                                0.1, f, &st);
                     }});
  v.push_back({"Q_phi", [](Ctx &x) { return cvchip_Q_phi(x.c, y.data(), b.data(), 0.1, 0); }});
  v.push_back({"scalar_product", [](Ctx &x) { return cvchip_scalar_product_co(x.c, contact, y.data(), b.data()); }});
  v.push_back({"cvc_source", [](Ctx &x) { return cvchip_cvc_source(x.c, conn.data(), contact, src, 1e-20, 20, 0, 0.1, nullptr); }});
  v.push_back({"cvc_propagators", [](Ctx &x) { return cvchip_cvc_propagators(x.c, props, src, 1e-20, 20, 1, 0.1, nullptr); }});
  v.push_back({"p2gg_source", [](Ctx &x) {
                 return cvchip_p2gg_source(x.c, conn.data(), contact, src, 1, 5, mom, 1, 1e-20, 20, 2, 0.1, nullptr);
               }});
  v.push_back({"cvc_gradient", [](Ctx &x) {
                 return cvchip_cvc_gradient(x.c, src, 2., 1e-20, 20, 0, 0.1, &L, &dmu, force.data(), nullptr);
               }});
  return v;
}

// Every entry point with each of its `count`ed events refused in turn: the call ends
// (an error, or a result where there is another way), the context is as it was, the
// same call then works, and nothing is left allocated.
static void refuse_each(long &count, long &fail, const char *what, const std::vector<Entry> &list, int T = 2, int L = 2,
                        int LZ = 4) {
  for (const Entry &e : list)
    for (long k = 1;; k++) {
      std::string at = std::string(e.name) + ", " + what + " " + std::to_string(k);
      Ctx x(T, L, L, LZ);
      fail = count + k;
      const int rc = e.call(x);
      const bool reached = count >= fail;
      fail = 0;
      CHECK(reached || rc >= 0, "%s: %d", at.c_str(), rc);
      CHECK(x.c->mu == 0.01 && !x.c->op_mask && !x.c->red_off, "%s: context changed", at.c_str());
      const Copies q = x.c->copy_stream ? to_host[x.c->copy_stream] : Copies();
      CHECK(q.ended == q.issued, "%s: %ld pieces still on their way", at.c_str(), q.issued - q.ended);
      CHECK(hipGetLastError() == hipSuccess || rc >= 0, "%s: error left behind (returned %d)", at.c_str(), rc);
      CHECK(e.call(x) >= 0, "%s: the same call again", at.c_str());
      launches.clear();
      if (!reached) break;
    }
}
static void refused_calls() { refuse_each(calls, fail_call, "call", entries()); }
static void refused_host_memory() {
  std::vector<Entry> list = entries();
  list.pop_back();   // (cvc_gradient)
  counted = true;
  refuse_each(news, fail_new, "host allocation", list);
}

// the contraction of a lattice whose conn leaves in pieces (16 MB)
static void streamed_conn() {
  static std::vector<double> conn((size_t)32 << 16);
  static double contact[8];
  static const int src[4] = {1, 0, 1, 2};
  refuse_each(calls, fail_call, "call", {{"field_cvc_contract", [](Ctx &x) {
                cvchip_field *up = nullptr, *dn = nullptr;
                int rc = cvchip_field_create(x.c, 60, CVCHIP_PREC_F64, &up);
                if (!rc) rc = cvchip_field_create(x.c, 60, CVCHIP_PREC_F64, &dn);
                if (!rc) rc = cvchip_field_cvc_contract(x.c, conn.data(), contact, up, dn, src);
                cvchip_field_destroy(up);
                cvchip_field_destroy(dn);
                return rc;
              }}}, 16, 16, 16);
}

// A whole source on a device that holds the twelve-column solves but not the sixty-column
// ones: the sources are solved one by one, and that takes no more memory than if the
// larger solve had not been tried.
static void one_by_one() {
  static std::vector<double> conn(32 << 12);
  static double contact[8];
  static const int src[4] = {1, 0, 1, 2};
  const size_t set12 = (size_t)2304 * 4096, set60 = 5 * set12;
  // up and dn, b and x, the hermitian solver's nine sets; the links, scratch
  const size_t enough = 2 * set60 + 11 * set12 + ((size_t)14 << 20);
  Ctx x(8, 8, 8, 8);
  capacity = enough;
  launches.clear();
  const int rc = cvchip_cvc_source(x.c, conn.data(), contact, src, 1e-20, 20, 0, 0.1, nullptr);
  capacity = SIZE_MAX;
  CHECK(rc >= 0, "whole source: %d", rc);
  int k = 0;
  for (const Launch &l : launches) {
    if (l.cols.empty()) continue;
    const uint32_t s = 12u * (uint32_t)(k / 2 % 5);
    const std::vector<uint32_t> in = {12, 60, 0, s, 12}, out = {60, 12, s, 0, 12};
    CHECK(l.cols == (k % 2 ? out : in), "copy of columns %d", k);
    k++;
  }
  CHECK(k == 20, "%d copies of columns", k);
}

// A whole source whose third set of twelve does not converge: the statistics cover the
// two before it.
static void unconverged_source() {
  static std::vector<double> conn(32 << 6);
  static double contact[8];
  static const int src[4] = {1, 0, 1, 2};
  for (int prec = 0; prec < 3; prec++) {
    Ctx x(4, 2, 2, 4);
    cvchip_stats st;
    CHECK(cvchip_cvc_source(x.c, conn.data(), contact, src, 1e-20, 20, prec, 0.1, &st) >= 0, "converging source");
    CHECK(st.converged == 120 && st.iterations == 10 * (conv_it + 1), "%d, %d iterations", st.converged, st.iterations);
    conv_rhs = 30;   // of each solve's sixty
    const int rc = cvchip_cvc_source(x.c, conn.data(), contact, src, 1e-20, 20, prec, 0.1, &st);
    conv_rhs = 1 << 30;
    CHECK(rc == CVCHIP_ERR_NOCONV, "%d", rc);
    CHECK(st.converged == 24 && st.iterations == 2 * (conv_it + 1) && st.dslash_calls > 0, "%d converged, %d iterations, %d applications",
          st.converged, st.iterations, st.dslash_calls);
  }
}

// dslash_calls is the number of operator applications launched: on small lattices one of
// them goes out before the test that ends the solve, one more before a reliable update.
static void counted_applications() {
  for (int prec = 0; prec < 3; prec++) {
    Ctx x(4, 2, 2, 4);
    cvchip_stats st;
    launches.clear();
    CHECK(solve(x, 2, prec, 0, &st, false) >= 0, "solve");
    int n = 0;
    for (const Launch &l : launches) n += l.name.find("k_dslash") != std::string::npos;
    CHECK(n > 2 * st.iterations && st.dslash_calls == n, "precision %d: %d of %d applications counted", prec,
          st.dslash_calls, n);
  }
}

// The automatic columns of the multi-rhs operator keep the extents that a caller gives in
// bits 8-15 and 20-23 of the policy.
static void column_extents() {
  using namespace cvchip;
  Ctx x(8, 12, 12, 8);
  for (int eo = 0; eo < 2; eo++)
    for (int K : {1, 2, 4})
      for (int N : {8, 12, 48})
        for (int yb : {0, 1, 2, 6, 12})
          for (int bx : {0, 1, 3, 12}) {
            CHECK(!cvchip_ctx_set_dslash_policy(x.c, 5 | yb << 8 | bx << 20), "policy");
            const Traversal t = plan_traversal(x.c, N, eo, K);
            CHECK(t.mode == 4 && (!yb || t.yb == (unsigned)yb) && (!bx || t.bx == (unsigned)bx),
                  "N %d, yb %d, bx %d: mode %d, columns %u x %u", N, yb, bx, t.mode, t.bx, t.yb);
          }
}

// The multi-rhs operator's blocks waste few lanes: over the sites of a run, at most a
// quarter more than the least that any count from half a full block up takes.
static void block_lanes() {
  using namespace cvchip;
  for (uint32_t N = 8; N <= 128; N++)
    for (uint32_t len : {64, 96, 120, 128, 160, 192, 198, 255, 256, 285, 324, 396, 400, 512, 576, 1024}) {
      auto lanes = [&](uint32_t S) { return (len + S - 1) / S * ((S * N + 63) / 64 * 64); };
      const uint32_t full = 256 / N, S = op_sites((int)N, len, 1 << 24);
      uint32_t least = ~0u;
      for (uint32_t s = (full + 1) / 2; s <= full; s++) least = std::min(least, lanes(s));
      CHECK(S >= 1 && S <= full && 4 * lanes(S) <= 5 * least, "N %u, run of %u: %u sites, %u lanes, not %u", N, len, S,
            lanes(S), least);
    }
}

// The FP32 operator marches in t where the XCDs share its patches evenly and its sets do
// not stay in the caches.
static void march_rule() {
  using namespace cvchip;
  struct Case {
    int T, LX, LY, LZ, N, K, march;
  };
  for (const Case &k : {Case{32, 32, 32, 32, 12, 2, 1}, {64, 32, 32, 32, 8, 2, 1}, {32, 32, 16, 16, 20, 2, 1},
                        {24, 32, 32, 20, 16, 2, 1}, {18, 16, 32, 18, 20, 2, 1}, {16, 32, 16, 16, 20, 2, 0},
                        {64, 48, 48, 48, 12, 2, 0}, {20, 40, 40, 40, 16, 2, 0}, {32, 36, 32, 32, 12, 2, 0},
                        {32, 32, 32, 32, 24, 2, 0}, {64, 32, 32, 32, 7, 2, 0}, {64, 32, 32, 32, 12, 1, 0},
                        {64, 32, 32, 32, 12, 4, 0}}) {
    cvchip_ctx c;
    c.lat = Lattice{k.T, k.LX, k.LY, k.LZ, (int64_t)k.T * k.LX * k.LY * k.LZ};
    const Traversal t = plan_traversal(&c, k.N, false, k.K);
    CHECK((t.mode == 6) == (k.march == 1), "%d %d %d %d, %d rhs, K %d: mode %d", k.T, k.LX, k.LY, k.LZ, k.N, k.K, t.mode);
    CHECK(plan_traversal(&c, k.N, true, k.K).mode != 6, "even/odd");
  }
}

int main(int argc, char **argv) {
  const std::map<std::string, void (*)()> all = {{"scratch", scratch}, {"solver_buffers", solver_buffers},
                                                {"refused_calls", refused_calls}, {"refused_host_memory", refused_host_memory},
                                                {"streamed_conn", streamed_conn}, {"one_by_one", one_by_one},
                                                {"unconverged_source", unconverged_source},
                                                {"counted_applications", counted_applications},
                                                {"column_extents", column_extents},
                                                {"block_lanes", block_lanes}, {"march_rule", march_rule}};
  const auto it = argc == 2 ? all.find(argv[1]) : all.end();
  if (it == all.end()) return 2;
  it->second();
  puts("ok");
  return 0;
}
