// What the library's host code asks of the HIP runtime, without a GPU: this
// program defines the runtime functions libwfx.so imports, so that the library
// binds to them, and runs the C-ABI over them.  Device memory is host memory
// filled with 0xff when allocated (a NaN in every double), memory copies and
// fills are done, kernels are noted by name and not run but for the few below.
// Usage: host_calls_check LIBRARY CHECK; prints what is wrong, exit code 0 if
// nothing is.
#include <dlfcn.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../include/wfx.h"

namespace {

struct Dim3 {
  uint32_t x, y, z;
};
struct Kernel {
  std::string name;
  int device;
  void *stream;
  bool captured;
};

std::mutex mu;
std::map<const void *, std::string> kernel_names;
std::vector<Kernel> launched;
std::function<void(const std::string &, void **)> on_launch;
int current = 0;  // device
int wanted = -1;  // >= 0: what follows the current device has to meet this one
bool capturing = false;
std::map<void *, size_t> pinned;  // bytes
size_t pinned_limit = SIZE_MAX;   // a larger request fails
int last_error = 0;
std::atomic<int> wrong{0};

#define EXPECT(cond, ...)      \
  do {                         \
    if (!(cond)) {             \
      ++wrong;                 \
      std::printf(__VA_ARGS__); \
      std::printf("\n");       \
    }                          \
  } while (0)

// an allocation, an event or work on the null stream: where the current device is
void at_current(const char *what, const std::string &name = "") {
  EXPECT(wanted < 0 || current == wanted, "%s %s on device %d, the context is on %d", what, name.c_str(), current, wanted);
}
bool is(const std::string &name, const char *kernel) { return name.find(kernel) != std::string::npos; }
template <typename T>
T arg(void **args, int k) {
  T v;
  std::memcpy(&v, args[k], sizeof(T));
  return v;
}

thread_local struct {
  Dim3 grid, block;
  size_t shmem;
  void *stream;
} pushed;

}  // namespace

extern "C" {
void **__hipRegisterFatBinary(const void *) {
  static void *modules = nullptr;
  return &modules;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *) {
  kernel_names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shmem, void *stream) {
  pushed = {grid, block, shmem, stream};
  return 0;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *shmem, void **stream) {
  *grid = pushed.grid;
  *block = pushed.block;
  *shmem = pushed.shmem;
  *stream = pushed.stream;
  return 0;
}
int hipLaunchKernel(const void *host, Dim3, Dim3, void **args, size_t, void *stream) {
  std::lock_guard<std::mutex> l(mu);
  const std::string &name = kernel_names[host];
  launched.push_back({name, current, stream, capturing});
  if (!stream) at_current("kernel", name);
  if (on_launch) on_launch(name, args);
  return 0;
}
int hipGetDeviceCount(int *n) {
  *n = 2;
  return 0;
}
int hipGetDevice(int *d) {
  *d = current;
  return 0;
}
int hipSetDevice(int d) {
  current = d;
  return 0;
}
int hipMalloc(void **p, size_t bytes) {
  *p = std::aligned_alloc(256, (bytes + 255) / 256 * 256);
  std::memset(*p, 0xff, bytes);
  at_current("hipMalloc");
  return 0;
}
int hipFree(void *p) {
  std::free(p);
  return 0;
}
int hipHostMalloc(void **p, size_t bytes, unsigned) {
  std::lock_guard<std::mutex> l(mu);
  if (bytes > pinned_limit) return last_error = 2;
  *p = std::aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
  pinned[*p] = bytes;
  return 0;
}
int hipHostFree(void *p) {
  std::lock_guard<std::mutex> l(mu);
  pinned.erase(p);
  std::free(p);
  return 0;
}
int hipMemset(void *p, int v, size_t bytes) {
  std::memset(p, v, bytes);
  return 0;
}
int hipMemcpy(void *d, const void *s, size_t bytes, int) {
  std::memcpy(d, s, bytes);
  return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t bytes, int, void *) {
  std::memcpy(d, s, bytes);
  return 0;
}
int hipGetSymbolAddress(void **p, const void *) {
  static char scratch[1 << 20];
  *p = scratch;
  return 0;
}
int hipGetLastError() {
  std::lock_guard<std::mutex> l(mu);
  const int e = last_error;
  last_error = 0;
  return e;
}
const char *hipGetErrorString(int) { return "error"; }
int hipDeviceSynchronize() {
  at_current("hipDeviceSynchronize");
  return 0;
}
int hipStreamSynchronize(void *s) {
  if (!s) at_current("hipStreamSynchronize");
  return 0;
}
int hipStreamWaitEvent(void *, void *, unsigned) { return 0; }
int hipStreamCreate(void **s) {
  *s = std::malloc(1);
  return 0;
}
int hipStreamDestroy(void *s) {
  std::free(s);
  return 0;
}
int hipStreamIsCapturing(void *, int *status) {
  *status = capturing ? 1 : 0;
  return 0;
}
int hipStreamBeginCapture(void *, int) {
  capturing = true;
  return 0;
}
int hipStreamEndCapture(void *, void **graph) {
  capturing = false;
  *graph = std::malloc(1);
  return 0;
}
int hipGraphInstantiate(void **exec, void *, void **, char *, size_t) {
  *exec = std::malloc(1);
  return 0;
}
int hipGraphLaunch(void *, void *) { return 0; }
int hipGraphDestroy(void *g) {
  std::free(g);
  return 0;
}
int hipGraphExecDestroy(void *g) {
  std::free(g);
  return 0;
}
int hipEventCreateWithFlags(void **e, unsigned) {
  *e = std::malloc(1);
  at_current("hipEventCreate");
  return 0;
}
int hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void *e) {
  std::free(e);
  return 0;
}
int hipEventRecord(void *, void *s) {
  if (!s) at_current("hipEventRecord");
  return 0;
}
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *) {
  *ms = 1.0f;
  return 0;
}
}  // extern "C"

namespace {

void *library;
template <typename F>
F *entry(const char *name) {
  void *p = dlsym(library, name);
  if (!p) {
    std::printf("%s is not exported\n", name);
    std::exit(2);
  }
  return reinterpret_cast<F *>(p);
}
// CALL(wfx_set_dt, c, dt): the entry point, which has to succeed
#define CALL(fn, ...)                                                                                              \
  do {                                                                                                             \
    const int rc = entry<decltype(fn)>(#fn)(__VA_ARGS__);                                                          \
    EXPECT(rc == 0, "%s returned %d: %s", #fn, rc, entry<decltype(wfx_last_error)>("wfx_last_error")());           \
  } while (0)

// nx x ny x nz hexahedra (tets: six tetrahedra each) and, with stray, a node of
// no element behind them
struct Box {
  std::vector<double> x;
  std::vector<int> el;
  int nodes, elems, n;
  explicit Box(int size, bool stray = false) : Box(size, size, size, false, stray) {}
  Box(int nx, int ny, int nz, bool tets = false, bool stray = false) : n(tets ? 4 : 8) {
    const int mx = nx + 1, my = ny + 1;
    for (int k = 0; k <= nz; ++k)
      for (int j = 0; j <= ny; ++j)
        for (int i = 0; i <= nx; ++i) x.insert(x.end(), {0.1 * i, 0.1 * j, 0.1 * k});
    const int part[6][4] = {{0, 1, 3, 5}, {1, 2, 3, 5}, {0, 5, 3, 4}, {4, 5, 3, 7}, {5, 6, 3, 7}, {5, 2, 3, 6}};
    for (int k = 0; k < nz; ++k)
      for (int j = 0; j < ny; ++j)
        for (int i = 0; i < nx; ++i) {
          const int a = (k * my + j) * mx + i, b = a + mx * my;
          const int h[8] = {a, a + 1, a + mx + 1, a + mx, b, b + 1, b + mx + 1, b + mx};
          if (!tets) el.insert(el.end(), h, h + 8);
          for (int t = 0; tets && t < 6; ++t)
            for (int q : part[t]) el.push_back(h[q]);
        }
    if (stray) x.insert(x.end(), {50.0, 50.0, 50.0});
    nodes = (int)x.size() / 3;
    elems = (int)el.size() / n;
  }
};

wfx_ctx *domain(const Box &b, int precision = WFX_FP64) {
  wfx_ctx *c = nullptr;
  CALL(wfx_create, &c, precision);
  CALL(wfx_set_mesh, c, b.nodes, b.elems, b.n, b.x.data(), b.el.data());
  CALL(wfx_set_density, c, 7850.0);
  CALL(wfx_set_material, c, WFX_BILINEAR, 200e9, 0.3, 7850.0, 300e6, 1e9, 0.0);
  CALL(wfx_set_dt, c, 1e-6);
  return c;
}

// Every entry of the step length's cotangent the gradient sums with a per-step
// time step is one a kernel wrote or was cleared: a node of no element is in no
// cluster, so that no cluster kernel writes its entry.
void adjoint_stray() {
  const Box b(3, true);
  wfx_ctx *c = domain(b);
  const int reaction[2] = {0, 1}, stray = b.nodes - 1;
  for (int d = 0; d < 3; ++d) CALL(wfx_add_bc_vel_node, c, stray, d, 0.0);
  CALL(wfx_allocate_bcs, c);
  CALL(wfx_set_reaction_nodes, c, reaction, 2);
  CALL(wfx_set_cfl, c, 0.3);
  CALL(wfx_init, c, nullptr);
  int summed = 0;
  on_launch = [&](const std::string &name, void **args) {
    if (!is(name, "a_cfl_apply")) return;
    ++summed;
    const double *dtb = arg<const double *>(args, 4);
    EXPECT(dtb[stray] == 0.0, "the cotangent of the step length sums %g for the node of no element", dtb[stray]);
  };
  const int n = 3;
  std::vector<double> hist(n), bar(n, 1.0), grad(3);
  CALL(wfx_adjoint_forward, c, n, 2, hist.data(), nullptr);
  CALL(wfx_adjoint_backward, c, bar.data(), grad.data(), nullptr, nullptr, nullptr, nullptr);
  EXPECT(summed == n, "the cotangent of the step length was summed %d times in %d steps", summed, n);
  CALL(wfx_destroy, c);
}

// The nodal mean densities a phase-2 call reads belong to the present
// densities: formed by an earlier kernel that ran, not by one that a capture
// only recorded; once per captured run.
void densities_captured() {
  const Box b(3);
  void *stream = nullptr;
  hipStreamCreate(&stream);
  wfx_ctx *c = domain(b);
  CALL(wfx_init, c, nullptr);
  CALL(wfx_step_fused, c, 3, nullptr, stream);
  const std::vector<double> rho(b.elems, 7000.0);
  CALL(wfx_set_field, c, "rho", rho.data(), (long)rho.size());
  const auto formed = [&](bool captured) {
    return std::count_if(launched.begin(), launched.end(), [&](const Kernel &k) {
      return k.captured == captured && is(k.name, "f0_vsum0");
    });
  };
  launched.clear();
  CALL(wfx_graph_capture, c, 4, 0, stream);
  EXPECT(formed(true) == 1, "the means are formed %ld times in a captured run", (long)formed(true));
  CALL(wfx_fused_phase, c, 1, 0, stream);
  CALL(wfx_fused_phase, c, 2, 0, stream);
  EXPECT(formed(false) == 1, "phase 2 after a capture reads the means of the densities before it");
  CALL(wfx_fused_phase, c, 2, 0, stream);
  EXPECT(formed(false) == 1, "two phase-2 calls form the means %ld times", (long)formed(false));
  // the caller's own capture: each replay meets the densities of its time
  launched.clear();
  hipStreamBeginCapture(stream, 0);
  CALL(wfx_fused_phase, c, 2, 0, stream);
  void *graph = nullptr;
  hipStreamEndCapture(stream, &graph);
  EXPECT(formed(true) == 1, "a captured phase 2 does not form the means");
  CALL(wfx_destroy, c);
}

// A uniform density needs no means: a run does not read the densities for them,
// and forms them once the densities may differ.
void densities_uniform() {
  const Box b(3);
  int formed = 0;
  on_launch = [&](const std::string &name, void **args) {
    if (is(name, "k_scan_elem")) {  // what it finds here
      unsigned long long *scan = arg<unsigned long long *>(args, 3);
      const double rho = 7850.0;
      scan[0] = scan[1] = 0;
      std::memcpy(&scan[2], &rho, 8);
      std::memcpy(&scan[3], &rho, 8);
    }
    if (is(name, "f0_vsum0")) formed += arg<const double *>(args, 7) != nullptr;
  };
  wfx_ctx *c = domain(b);
  CALL(wfx_init, c, nullptr);
  CALL(wfx_step_fused, c, 1, nullptr, nullptr);
  CALL(wfx_fused_phase, c, 2, 0, nullptr);
  EXPECT(formed == 0, "means of a uniform density were formed");
  CALL(wfx_calc_elem_density, c, nullptr);
  CALL(wfx_fused_phase, c, 2, 0, nullptr);
  EXPECT(formed == 1, "means formed %d times after the densities changed", formed);
  CALL(wfx_step_fused, c, 1, nullptr, nullptr);
  EXPECT(formed == 2, "a run did not form the means");
  CALL(wfx_destroy, c);
}

// Calls without a stream work whichever device is current, on the context's
// own, and leave the current one; so do the allocations of calls with a stream.
void other_device(int precision) {
  const Box b(4), large(60);  // large: more than one chunk of the transfers
  void *stream = nullptr;
  hipStreamCreate(&stream);
  for (int own = 0; own < 2; ++own) {
    wanted = -1;
    current = own;
    wfx_ctx *c = domain(b, precision), *l = domain(large, precision);
    current = 1 - own;
    wanted = own;
    std::vector<double> v(3 * b.nodes), e(b.elems, 5e7), w(3 * large.nodes);
    CALL(wfx_set_density, c, 7000.0);
    CALL(wfx_set_material, c, WFX_BILINEAR, 200e9, 0.3, 7850.0, 300e6, 1e9, 0.0);
    CALL(wfx_set_elem_sy0, c, e.data(), b.elems);
    CALL(wfx_set_elem_tangent, c, e.data(), b.elems);
    CALL(wfx_set_temperature, c, 30.0);
    CALL(wfx_set_elem_temperature, c, e.data(), b.elems);
    CALL(wfx_set_dt, c, 1e-6);
    CALL(wfx_init, c, stream);
    CALL(wfx_get_field, c, "x", v.data(), (long)v.size());
    CALL(wfx_set_field, c, "v", v.data(), (long)v.size());
    CALL(wfx_set_field, c, "rho", e.data(), (long)e.size());
    CALL(wfx_get_field, l, "x", w.data(), (long)w.size());
    CALL(wfx_set_field, l, "x", w.data(), (long)w.size());
    const int nodes[2] = {0, 1};
    CALL(wfx_set_reaction_nodes, c, nodes, 2);
    std::vector<double> hist(4);
    CALL(wfx_step_fused, c, 4, hist.data(), stream);
    CALL(wfx_destroy, c);
    CALL(wfx_destroy, l);
    EXPECT(current == 1 - own, "the current device is %d, the caller's was %d", current, 1 - own);
  }
}

// the transfer kernels of a real field in double, on the host
void run_transfers(const std::string &name, void **args) {
  const bool out = is(name, "k_field_outIdLb0E");
  if (!out && !is(name, "k_field_inIdLb0E")) return;
  const long k0 = arg<long>(args, 0), n = arg<long>(args, 1), cnt = arg<long>(args, 3);
  const int rows = arg<int>(args, 2);
  const int *perm = arg<const int *>(args, 4);
  double *p = arg<double *>(args, 5), *q = arg<double *>(args, 6);  // source, destination
  for (long t = 0; t < n; ++t) {
    const long i = (k0 + t) / rows, r = (k0 + t) % rows, at = r * cnt + (perm ? perm[i] : i);
    if (out) q[t] = p[at];
    else q[at] = p[t];
  }
}

size_t pinned_bytes() {
  size_t b = 0;
  for (const auto &p : pinned) b += p.second;
  return b;
}

// The pinned memory of the transfers: what transfers at the same time need, not
// what every context once needed; none after the last context.
void pinned_memory() {
  const Box b(60);  // 680,943 nodal values: two chunks
  std::vector<double> v(3 * b.nodes);
  wfx_ctx *c[6];
  for (auto &q : c) {
    q = domain(b);
    CALL(wfx_get_field, q, "x", v.data(), (long)v.size());
    CALL(wfx_get_field, q, "T", v.data(), (long)b.nodes);
    EXPECT(pinned_bytes() <= (68u << 20), "%zu MiB of pinned memory", pinned_bytes() >> 20);
  }
  for (auto &q : c) CALL(wfx_destroy, q);
  EXPECT(pinned.empty(), "%zu MiB of pinned memory without a context", pinned_bytes() >> 20);
}

// Transfers by each way (kernels, copies, the ring), without memory for the ring,
// and from several threads
void transfers() {
  on_launch = run_transfers;
  for (const int n : {1, 7, 8, 12, 13, 30, 60}) {  // 192 B to 5.4 MB of positions
    const Box m(n);
    wfx_ctx *c = domain(m);
    std::vector<double> x(m.x.size());
    CALL(wfx_get_field, c, "x", x.data(), (long)x.size());
    EXPECT(x == m.x, "%d^3: the positions read differ from the mesh's", n);
    CALL(wfx_destroy, c);
  }
  const Box b(60);
  const auto back_and_forth = [&](wfx_ctx *c, int seed) {
    std::vector<double> v(3 * b.nodes), w(v.size(), 0.0);
    for (size_t i = 0; i < v.size(); ++i) v[i] = (double)(i * 7 + seed);
    CALL(wfx_set_field, c, "v", v.data(), (long)v.size());
    CALL(wfx_get_field, c, "v", w.data(), (long)w.size());
    EXPECT(v == w, "a field set and read back differs");
  };
  pinned_limit = 4u << 20;
  wfx_ctx *c = domain(b);
  back_and_forth(c, 1);
  CALL(wfx_destroy, c);
  pinned_limit = SIZE_MAX;
  wfx_ctx *d[6];
  for (auto &q : d) q = domain(b);
  std::vector<std::thread> th;
  for (int t = 0; t < 6; ++t)
    th.emplace_back([&, t] {
      for (int k = 0; k < 8; ++k) back_and_forth(d[t], 10 * t + k);
    });
  for (auto &t : th) t.join();
  EXPECT(pinned_bytes() <= (4u * 68 << 20), "%zu MiB of pinned memory kept", pinned_bytes() >> 20);
  for (auto &q : d) CALL(wfx_destroy, q);
  EXPECT(pinned.empty(), "%zu MiB of pinned memory without a context", pinned_bytes() >> 20);
}

// Which passes a run of seven steps takes: all of its steps but the last in the
// solo pass, or in the paired ones, or every step in the separate ones (as the
// last step's nodal update always is).  An odd run's paired steps all go to the
// other set of buffers.
enum Passes { SEPARATE, PAIRED, SOLO };
void expect_passes(const char *what, wfx_ctx *c, Passes want) {
  const int n = 7;
  launched.clear();
  CALL(wfx_step_fused, c, n, nullptr, nullptr);
  const auto count = [](const char *kernel) {
    return (int)std::count_if(launched.begin(), launched.end(), [&](const Kernel &k) { return is(k.name, kernel); });
  };
  const int solo = count("f_solo"), pair = count("f41_cluster"), node = count("f4_node"), sums = count("f2_nodal"),
            elem = count("f3_cluster");
  double clusters = 0.0;
  CALL(wfx_get_param, c, "cluster_count", &clusters);
  const bool ok = want == SOLO     ? solo == 1 && pair == 0 && node == 1 && sums == 0 && elem == 1
                  : want == PAIRED ? solo == 0 && pair == n - 1 && node == 1 && sums == 0 && elem == n
                                   : solo == 0 && pair == 0 && node == n && sums == n && elem == n;
  EXPECT(ok, "%s, %g clusters: solo pass %d, paired node passes %d, node passes %d, nodal sums %d, element passes %d",
         what, clusters, solo, pair, node, sums, elem);
}
// cells along x, y and z, precision, clusters of the plan (0: any), passes
struct LineCase {
  int x, y, z;
  bool tets;
  int precision, clusters;
  Passes want;
};
void passes_by_size() {
  const LineCase cases[] = {
      {1, 1, 1, false, WFX_FP64, 1, SOLO},          {1, 1, 1, false, WFX_FP32_MIXED, 1, PAIRED},
      {16, 4, 4, false, WFX_FP64, 1, SOLO},         {17, 4, 4, false, WFX_FP64, 2, PAIRED},
      {20, 20, 20, false, WFX_FP64, 35, PAIRED},    {40, 40, 40, false, WFX_FP64, 250, PAIRED},
      {40, 40, 41, false, WFX_FP64, 264, SEPARATE}, {40, 40, 40, false, WFX_FP32_MIXED, 250, PAIRED},
      {48, 51, 50, false, WFX_FP32_MIXED, 480, PAIRED}, {49, 49, 49, false, WFX_FP32_MIXED, 574, SEPARATE},
      {3, 3, 4, true, WFX_FP64, 1, SOLO},           {20, 20, 20, true, WFX_FP64, 0, PAIRED},
      {27, 27, 27, true, WFX_FP64, 0, SEPARATE},    {27, 27, 27, true, WFX_FP32_MIXED, 0, PAIRED},
      {28, 28, 28, true, WFX_FP32_MIXED, 515, SEPARATE}};
  for (const LineCase &q : cases) {
    const Box b(q.x, q.y, q.z, q.tets);
    wfx_ctx *c = domain(b, q.precision);
    CALL(wfx_init, c, nullptr);
    double clusters = 0.0;
    CALL(wfx_get_param, c, "cluster_count", &clusters);
    EXPECT(q.clusters == 0 || clusters == q.clusters, "%d x %d x %d, precision %d: %g clusters", q.x, q.y, q.z,
           q.precision, clusters);
    char what[64];
    std::snprintf(what, sizeof(what), "%d x %d x %d %s, precision %d", q.x, q.y, q.z, q.tets ? "tets" : "hexa",
                  q.precision);
    expect_passes(what, c, q.want);
    CALL(wfx_destroy, c);
  }
}
void passes_by_option() {
  for (const int precision : {WFX_FP64, WFX_FP32_MIXED})
    for (const bool small : {true, false}) {
      const int n = small ? 2 : 9;
      const Passes solo = small && precision == WFX_FP64 ? SOLO : PAIRED;
      const Box hexa(n), tets(n, n, n, true), stray(n, true);
      const auto fresh = [&](const Box &b) {
        wfx_ctx *c = domain(b, precision);
        CALL(wfx_init, c, nullptr);
        return c;
      };
      wfx_ctx *c = fresh(hexa);
      expect_passes("plain", c, solo);
      CALL(wfx_set_cfl, c, 0.3);
      expect_passes("per-step time step", c, PAIRED);
      CALL(wfx_set_cfl, c, 0.0);
      expect_passes("fixed time step again", c, solo);
      CALL(wfx_set_thermal, c, 1, 50.0, 460.0, 0.9);
      expect_passes("thermal", c, PAIRED);
      CALL(wfx_set_thermal_expansion, c, 1e-5);
      expect_passes("thermal expansion", c, SEPARATE);
      CALL(wfx_destroy, c);
      c = fresh(tets);
      expect_passes("tetrahedra", c, solo);
      const double die[9] = {0, 0, 9, 9, 0, 9, 0, 9, 9}, moving[9] = {0, 0, -1, 0, 0, -1, 0, 0, -1};
      const int tri[3] = {0, 2, 1};
      CALL(wfx_set_rigid_mesh, c, 3, die, moving, 1, tri, nullptr);
      expect_passes("contact", c, PAIRED);
      CALL(wfx_destroy, c);
      c = fresh(stray);
      expect_passes("a node of no element", c, SEPARATE);
      CALL(wfx_destroy, c);
    }
  // above 256 clusters, FP32-mixed: only what fits two work-groups on a CU
  for (const bool tets : {false, true}) {
    wfx_ctx *c = domain(tets ? Box(24, 24, 24, true) : Box(44, 44, 44), WFX_FP32_MIXED);
    CALL(wfx_init, c, nullptr);
    expect_passes("more than 256 clusters, plain", c, PAIRED);
    CALL(wfx_set_cfl, c, 0.3);
    expect_passes("more than 256 clusters, per-step time step", c, tets ? PAIRED : SEPARATE);
    CALL(wfx_set_cfl, c, 0.0);
    CALL(wfx_set_thermal, c, 1, 50.0, 460.0, 0.9);
    expect_passes("more than 256 clusters, thermal", c, tets ? PAIRED : SEPARATE);
    CALL(wfx_destroy, c);
  }
  // 34 elements around an axis: more than the paired tables hold of a node
  Box fan(0);
  const int m = 34;
  fan.x.clear();
  for (int k = 0; k < 2; ++k) {
    fan.x.insert(fan.x.end(), {0.0, 0.0, 0.1 * k});
    for (int q = 0; q < m; ++q)
      fan.x.insert(fan.x.end(), {std::cos(6.283185307179586 * q / m), std::sin(6.283185307179586 * q / m), 0.1 * k});
  }
  for (int q = 0; q < 17; ++q)
    for (int half = 0; half < 2; ++half) {  // wedges as hexahedra with an edge of no length
      const int a = 2 * q + half, b = (a + 1) % m;
      fan.el.insert(fan.el.end(), {0, 1 + a, 1 + b, 0, m + 1, m + 2 + a, m + 2 + b, m + 1});
    }
  fan.nodes = 2 * (m + 1);
  fan.elems = m;
  wfx_ctx *c = domain(fan);
  CALL(wfx_init, c, nullptr);
  expect_passes("a node of 34 elements", c, SEPARATE);
  CALL(wfx_destroy, c);
}

}  // namespace

int main(int argc, char **argv) {
  const std::map<std::string, void (*)()> checks = {
      {"adjoint_stray", adjoint_stray},
      {"densities_captured", densities_captured},
      {"densities_uniform", densities_uniform},
      {"passes_by_size", passes_by_size},
      {"passes_by_option", passes_by_option},
      {"pinned_memory", pinned_memory},
      {"transfers", transfers},
      {"other_device_fp64", [] { other_device(WFX_FP64); }},
      {"other_device_mixed", [] { other_device(WFX_FP32_MIXED); }},
  };
  if (argc != 3 || !checks.count(argv[2])) return 2;
  library = dlopen(argv[1], RTLD_NOW);
  if (!library) {
    std::printf("%s\n", dlerror());
    return 2;
  }
  if (kernel_names.empty()) {  // the library bound to the HIP runtime itself
    std::printf("the library did not register its kernels here\n");
    return 2;
  }
  checks.at(argv[2])();
  return wrong ? 1 : 0;
}
