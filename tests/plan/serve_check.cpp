// Host-only check of the RSQF serving loop's memory (gqf_rsqf_serve, its
// executor and the workers kept between runs) on a model of the device: this
// program defines the HIP calls that the loop makes, over a device of a given
// size whose buffers are numbers only, and the library's calls, which take
// the workspace that they report.  Built with hipcc for the host alone by
// tests/test_serve_memory.py; one scenario a run, "<name> ok" when it holds.
#include "../../gpuquotientfilters_amd/csrc/gqf_serve.hip"

#include <cstdarg>
#include <cstring>
#include <map>

// ---------------------------------------------------------------- the device
static std::mutex g_mu;
static std::map<uintptr_t, size_t> g_mem;
static size_t g_used = 0, g_max = 0, g_cap = (size_t)1 << 50;
static uintptr_t g_next = 0x10000;
static int g_refused = 0;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (g_used + n > g_cap) {
    ++g_refused;
    return hipErrorOutOfMemory;
  }
  g_mem[g_next] = n;
  *p = reinterpret_cast<void*>(g_next);
  g_next += (n + 255) & ~(size_t)255;
  g_used += n;
  g_max = std::max(g_max, g_used);
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(g_mu);
  auto i = g_mem.find(reinterpret_cast<uintptr_t>(p));
  if (i == g_mem.end()) return hipErrorInvalidValue;
  g_used -= i->second;
  g_mem.erase(i);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
// (no device code in this program)
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipUnregisterFatBinary(void**) {}
}

// ---------------------------------------------------------------- the library
struct Stream {
  void* ws = nullptr;
  size_t cap = 0;
};
static char g_err[512];
namespace gqf {
void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}
gqf_status hip_fail(hipError_t e, const char* what, const char*, int) {
  set_error("%s", what);
  return e == hipErrorOutOfMemory ? GQF_ERR_NOMEM : GQF_ERR_HIP;
}
size_t ws_alloc_bytes(size_t n) { return n; }
gqf_status ws_trim(gqf_stream s) {
  Stream* x = static_cast<Stream*>(s);
  if (x->ws) (void)hipFree(x->ws);
  x->ws = nullptr;
  x->cap = 0;
  return GQF_OK;
}
ProfScope::ProfScope(const char*, hipStream_t, double, const uint32_t*, double) {}
ProfScope::~ProfScope() {}
gqf_status rsqf_lookup_call(const gqf_rsqf&, int, const uint32_t*, int32_t*, gqf_stream, float*, bool) { return GQF_OK; }
}  // namespace gqf
constexpr size_t WS = 16;  // workspace bytes per key of an update
constexpr int SLOW = 777;  // an insert of so many keys takes 30 ms
static gqf_status update(gqf_stream s, int n) {
  Stream* x = static_cast<Stream*>(s);
  if (n == SLOW) std::this_thread::sleep_for(std::chrono::milliseconds(30));
  if (WS * (size_t)n <= x->cap) return GQF_OK;
  (void)ws_trim(s);
  if (hipMalloc(&x->ws, WS * (size_t)n) != hipSuccess) return GQF_ERR_NOMEM;
  x->cap = WS * (size_t)n;
  return GQF_OK;
}
extern "C" {
const char* gqf_last_error(void) { return g_err; }
gqf_status gqf_stream_create(gqf_stream* out) {
  *out = new Stream();
  return GQF_OK;
}
gqf_status gqf_stream_destroy(gqf_stream s) {
  (void)ws_trim(s);
  delete static_cast<Stream*>(s);
  return GQF_OK;
}
gqf_status gqf_stream_workspace_bytes(gqf_stream s, size_t* n) {
  *n = static_cast<Stream*>(s)->cap;
  return GQF_OK;
}
uint32_t gqf_rsqf_num_blocks(unsigned) { return 1; }
size_t gqf_rsqf_table_bytes(unsigned, unsigned) { return 0; }
size_t gqf_rsqf_workspace_bytes(gqf_rsqf, int op, int n, int) { return op == GQF_OP_LOOKUP ? 0 : WS * (size_t)n; }
gqf_status gqf_rsqf_insert(gqf_rsqf, int n, const uint32_t*, int32_t*, gqf_stream s, float*) { return update(s, n); }
gqf_status gqf_rsqf_delete(gqf_rsqf, int n, const uint32_t*, gqf_stream s, float*) { return update(s, n); }
}

// ---------------------------------------------------------------- scenarios
constexpr size_t MB = (size_t)1 << 20;
// One coalesced call of `parts` lookups, `keys` keys in all, per filter: a
// slow insert first, behind which they queue up.
struct Run {
  std::vector<gqf_request> reqs;
  gqf_serve_stats stats{};
  gqf_status st;
  size_t max_used;  // of the device, during the run
  Run(int filters, size_t keys, int parts, size_t budget) {
    std::vector<gqf_rsqf> f((size_t)filters);
    for (gqf_rsqf& x : f) {
      std::memset(&x, 0, sizeof(x));
      x.qbits = 20, x.rbits = 8, x.numBlocks = 1;
      *reinterpret_cast<void**>(&x.blocks) = reinterpret_cast<void*>(0x100);
    }
    auto add = [&](int fl, int op, int n) {
      gqf_request r;
      std::memset(&r, 0, sizeof(r));
      r.filter = fl, r.op = op, r.n = n;
      r.d_keys = reinterpret_cast<const uint32_t*>(0x1000000);
      r.d_out = reinterpret_cast<int32_t*>(0x1000000);
      reqs.push_back(r);
    };
    for (int i = 0; i < filters; ++i) add(i, GQF_OP_INSERT, SLOW);
    for (int k = 0; k < parts; ++k)
      for (int i = 0; i < filters; ++i) add(i, GQF_OP_LOOKUP, (int)(keys / (size_t)parts));
    gqf_serve_config cfg;
    std::memset(&cfg, 0, sizeof(cfg));
    cfg.hbm_budget = budget, cfg.coalesce = 1, cfg.max_batch = 1 << 30;
    g_max = g_used;
    st = gqf_rsqf_serve(f.data(), filters, reqs.data(), (int)reqs.size(), &cfg, &stats);
    max_used = g_max;
  }
  bool all_ok() const {
    for (const gqf_request& r : reqs)
      if (r.status != GQF_OK) return false;
    return st == GQF_OK;
  }
  bool one_call(int filters) const {  // a filter's lookups in one
    for (size_t i = (size_t)filters; i + (size_t)filters < reqs.size(); ++i)
      if (reqs[i].call != reqs[i + (size_t)filters].call) return false;
    return true;
  }
};
#define CHECK(x)                                                                                              \
  do {                                                                                                        \
    if (!(x)) {                                                                                               \
      std::printf("FAIL %s (max %zu MB, refused %d, %s)\n", #x, g_max / MB, g_refused, g_err);               \
      return 1;                                                                                               \
    }                                                                                                         \
  } while (0)

// A coalesced call whose buffers of exactly its keys fit the budget is one call.
static int exact() {
  const size_t keys = 590 * MB / 8;
  Run a(1, keys, 4, 600 * MB);
  CHECK(a.all_ok() && a.one_call(1));
  CHECK(a.max_used <= 600 * MB && a.stats.peak_bytes <= 600 * MB);
  (void)serve_release_idle();
  CHECK(g_used == 0);
  Run b(1, 100 * MB / 8, 4, 600 * MB);  // with room to spare: buffers for half as many keys again
  CHECK(b.all_ok() && b.one_call(1) && b.max_used >= 150 * MB - 64 && b.stats.peak_bytes >= b.max_used);
  return 0;
}

// Three filters' workers stay after a run; a later run's gather buffers fit the
// device only without them.
static int refused() {
  Run a(3, 60 * MB / 8, 4, (size_t)1 << 40);
  CHECK(a.all_ok() && g_used >= 150 * MB);
  g_cap = 250 * MB;
  Run b(1, 120 * MB / 8, 4, (size_t)1 << 40);
  CHECK(b.all_ok() && b.one_call(1) && g_refused >= 1);
  (void)serve_release_idle();
  Run c(1, 240 * MB / 8, 4, (size_t)1 << 40);  // buffers for exactly these keys
  CHECK(c.all_ok() && c.one_call(1));
  return 0;
}

// A run with fewer filters than the one before: the workers that it does not
// take count, and are given up when the budget needs their bytes.
static int idle() {
  Run a(3, 60 * MB / 8, 4, (size_t)1 << 40);
  CHECK(a.all_ok() && g_used >= 150 * MB);
  Run b(1, 100 * MB / 8, 4, 800 * MB);  // there is room: they stay
  CHECK(b.all_ok() && b.one_call(1));
  CHECK(b.stats.peak_bytes >= b.max_used && b.max_used <= 800 * MB && b.max_used >= 230 * MB);
  Run c(1, 590 * MB / 8, 4, 600 * MB);
  CHECK(c.all_ok() && c.one_call(1));
  CHECK(c.max_used <= 600 * MB && c.stats.peak_bytes <= 600 * MB);
  (void)serve_release_idle();
  Run d(3, 60 * MB / 8, 4, (size_t)1 << 40);
  Run e(1, 4 * MB / 8, 4, 100 * MB);  // a tight budget, below what stayed
  CHECK(d.all_ok() && e.all_ok());
  CHECK(e.stats.peak_bytes <= 100 * MB && g_used <= 100 * MB);
  return 0;
}

int main(int argc, char** argv) {
  const std::string name = argc > 1 ? argv[1] : "";
  int rc = 2;
  if (name == "exact") rc = exact();
  if (name == "refused") rc = refused();
  if (name == "idle") rc = idle();
  (void)serve_release_idle();
  if (rc == 0 && g_used != 0) {
    std::printf("FAIL %zu bytes left\n", g_used);
    rc = 1;
  }
  if (rc == 0) std::printf("%s ok\n", name.c_str());
  return rc;
}
