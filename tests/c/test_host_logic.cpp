// The library's host side on a stand-in for the HIP runtime: device memory is host memory with a limit, kernels
// are recorded and do nothing, a captured stream's launches become its graph's.  Defined here, the runtime's
// entry points come before libamdhip64's for libptq2 too.
//
// Checked: memory that a large mesh runs faster with (Box::xtile, the slots of A12 and the diagonal) never
// makes a call fail that fits without it, is a sixteenth of the device at most, and is in no graph that may
// outlive it; A12 and the diagonal run without slots under capture; the point projection needs no more than
// its sort and the nodal values.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "ptq2.h"
#include "ptq2_ctx.h"
#include "ptq2_solver.h"

namespace {
struct Launch {
  std::string name;
  hipStream_t stream;
  const void *xtile;  // of the passes that take one
};
struct Config {
  dim3 grid, block;
  size_t shmem;
  hipStream_t stream;
};
struct State {
  size_t limit = SIZE_MAX, used = 0, peak = 0, total = SIZE_MAX;
  std::map<void *, size_t> mem;
  std::map<const void *, std::string> kernels;
  std::vector<Launch> launches;
  std::map<hipStream_t, std::vector<Launch>> capture;
  Config config;
  int handles = 0;
};
State &S() {
  static State s;
  return s;
}
}  // namespace

extern "C" {
void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
  S().kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) {
  S().config = Config{g, b, m, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, hipStream_t *s) {
  const Config &c = S().config;
  *g = c.grid;
  *b = c.block;
  *m = c.shmem;
  *s = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t s) {
  Launch l{S().kernels[f], s, nullptr};
  if (l.name.find("k_a11_fp64_t") != std::string::npos || l.name.find("k_stokes_fp64") != std::string::npos)
    l.xtile = static_cast<const ptq2::Box *>(args[0])->xtile;
  auto c = S().capture.find(s);
  (c == S().capture.end() ? S().launches : c->second).push_back(l);
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
  *p = nullptr;
  if (S().used + n > S().limit) return hipErrorOutOfMemory;
  *p = calloc(n, 1);  // pages are taken when written
  S().mem[*p] = n;
  S().used += n;
  S().peak = std::max(S().peak, S().used);
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  auto m = S().mem.find(p);
  if (m == S().mem.end()) return hipErrorInvalidValue;
  S().used -= m->second;
  S().mem.erase(m);
  free(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *avail, size_t *total) {
  *avail = S().limit - S().used;
  *total = S().total;
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static char scratch[256];
  *p = scratch;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in"; }
static void *handle() { return (void *)(uintptr_t)(0x1000 + 16 * ++S().handles); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = (hipStream_t)handle();
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c) {
  if (!s && !S().capture.empty()) return hipErrorStreamCaptureImplicit;
  *c = S().capture.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  S().capture[s];
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) {
  *g = (hipGraph_t) new std::vector<Launch>(S().capture[s]);
  S().capture.erase(s);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
  *e = (hipGraphExec_t) new std::vector<Launch>(*(std::vector<Launch> *)g);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete (std::vector<Launch> *)g;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  delete (std::vector<Launch> *)e;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  for (const Launch &l : *(std::vector<Launch> *)e) S().launches.push_back(l);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = (hipEvent_t)handle();
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 0.01f;
  return hipSuccess;
}
}

namespace {
int bad = 0;
void expect(bool ok, const char *what, int line) {
  if (ok) return;
  std::printf("line %d: %s\n", line, what);
  bad++;
}
#define EXPECT(x) expect((x), #x, __LINE__)

int count(const char *name) {
  int n = 0;
  for (const Launch &l : S().launches) n += l.name.find(name) != std::string::npos;
  return n;
}
// whether the recorded FP64 passes had tiles: 1 all, 0 none, -1 some or no pass at all
int tiles() {
  int n = 0, with = 0;
  for (const Launch &l : S().launches)
    if (l.name.find("k_a11_fp64_t") != std::string::npos || l.name.find("k_stokes_fp64") != std::string::npos) {
      n++;
      with += l.xtile != nullptr;
    }
  return n && with == n ? 1 : (n && !with ? 0 : -1);
}

struct Mesh {
  int m[3];
  std::vector<double> coords, eta;
  std::vector<uint8_t> mask;
  int64_t nvel, npres;
  Mesh(int mx, int my, int mz) : m{mx, my, mz} {
    const int64_t N[3] = {2 * mx + 1, 2 * my + 1, 2 * mz + 1};
    nvel = 3 * N[0] * N[1] * N[2];
    npres = 4 * (int64_t)mx * my * mz;
    coords.assign(nvel, 0.5);
    mask.assign(nvel, 0);
    for (int64_t i = 0; i < 3 * N[0]; i++) mask[i] = 1;
    eta.assign(27 * (size_t)mx * my * mz, 1.0);
  }
  ptq2_ctx *make() const {
    ptq2_ctx *c = nullptr;
    EXPECT(ptq2_create(&c, 0) == PTQ2_OK);
    EXPECT(ptq2_setup_mesh(c, m[0], m[1], m[2], coords.data(), nullptr, mask.data()) == PTQ2_OK);
    EXPECT(ptq2_set_viscosity(c, eta.data(), 0, 0) == PTQ2_OK);
    return c;
  }
};

// every operator once on device vectors (the addresses are never read); the first failure's code
int all_operators(ptq2_ctx *c) {
  double v[1];
  const unsigned f = PTQ2_DEVICE | PTQ2_MATMULT;
  for (int rc : {ptq2_a11_apply(c, v, v + 1, f), ptq2_stokes_apply(c, v, v, v, v, f), ptq2_a12_apply(c, v, v, f),
                 ptq2_a11_diag(c, v, f), ptq2_a21_apply(c, v, v, f),
                 ptq2_stokes_residual(c, v, v, v, nullptr, nullptr, v, v, PTQ2_DEVICE),
                 ptq2_a11_apply(c, v, v + 1, f | PTQ2_FP32), ptq2_stokes_apply(c, v, v, v, v, f | PTQ2_FP32),
                 ptq2_a11_apply(c, v, v + 1, f | PTQ2_STOREDGEO)})
    if (rc) return rc;
  return PTQ2_OK;
}
size_t spare_of(int64_t nb) { return 8 * (size_t)(nb * (ptq2::FACEVALS + 3 * ptq2::TCS)); }

void operators_at_the_limit() {
  const Mesh m(1, 1, 32768);  // 8192 bricks of one column
  const size_t spare = spare_of(8192);
  S().peak = 0;
  ptq2_ctx *c = m.make();
  EXPECT(all_operators(c) == PTQ2_OK);
  EXPECT(tiles() == 1);
  const size_t all = S().peak;
  ptq2_destroy(&c);
  EXPECT(S().used == 0);
  // room for everything but the spare memory: it is taken at the set-up and given back
  S().limit = all - spare;
  S().launches.clear();
  c = m.make();
  EXPECT(all_operators(c) == PTQ2_OK);
  S().launches.clear();
  double v[1];
  EXPECT(ptq2_a11_apply(c, v, v + 1, PTQ2_DEVICE) == PTQ2_OK && tiles() == 0);
  EXPECT(ptq2_a12_apply(c, v, v, PTQ2_DEVICE) == PTQ2_OK && count("k_a12") > 1);
  ptq2_destroy(&c);
  EXPECT(S().used == 0);
  S().limit = SIZE_MAX;
  // a device of which it would be more than a sixteenth
  S().total = 16 * spare - 16;
  S().launches.clear();
  c = m.make();
  EXPECT(ptq2_a11_apply(c, v, v + 1, PTQ2_DEVICE) == PTQ2_OK && tiles() == 0);
  ptq2_destroy(&c);
  // of two contexts, the one that comes first has it; the other has it once the first is gone
  S().total = 16 * spare;
  c = m.make();
  ptq2_ctx *d = m.make();
  S().launches.clear();
  EXPECT(ptq2_a11_apply(d, v, v + 1, PTQ2_DEVICE) == PTQ2_OK && tiles() == 0);
  S().launches.clear();
  EXPECT(ptq2_a11_apply(c, v, v + 1, PTQ2_DEVICE) == PTQ2_OK && tiles() == 1);
  ptq2_destroy(&c);
  EXPECT(ptq2_setup_mesh(d, 1, 1, 32768, m.coords.data(), nullptr, nullptr) == PTQ2_OK);
  EXPECT(ptq2_set_viscosity(d, m.eta.data(), 1, 0) == PTQ2_OK);
  S().launches.clear();
  EXPECT(ptq2_a11_apply(d, v, v + 1, PTQ2_DEVICE) == PTQ2_OK && tiles() == 1);
  ptq2_destroy(&d);
  S().total = SIZE_MAX;
}

void operators_under_capture() {
  const Mesh m(1, 1, 32768);
  ptq2_ctx *c = m.make();
  double v[1];
  EXPECT(all_operators(c) == PTQ2_OK);
  hipStream_t s = (hipStream_t)ptq2_get_stream(c);
  S().launches.clear();
  hipGraph_t g;
  (void)hipStreamBeginCapture(s, hipStreamCaptureModeGlobal);
  EXPECT(ptq2_a11_apply(c, v, v + 1, PTQ2_DEVICE) == PTQ2_OK);
  EXPECT(ptq2_stokes_apply(c, v, v, v, v, PTQ2_DEVICE) == PTQ2_OK);
  EXPECT(ptq2_a12_apply(c, v, v, PTQ2_DEVICE) == PTQ2_OK);
  EXPECT(ptq2_a11_diag(c, v, PTQ2_DEVICE) == PTQ2_OK);
  (void)hipStreamEndCapture(s, &g);
  EXPECT(S().launches.empty());
  S().launches = *(std::vector<Launch> *)g;
  EXPECT(tiles() == 0 && count("k_a12") > 1 && count("k_diag") > 1 && count("k_gather") == 2);
  S().launches.clear();
  EXPECT(all_operators(c) == PTQ2_OK);
  EXPECT(tiles() == 1 && count("k_a12") == 1 && count("k_diag") == 1);
  (void)hipGraphDestroy(g);
  // another stream's capture does not change what a call on the null stream runs
  (void)hipStreamBeginCapture((hipStream_t)0x10, hipStreamCaptureModeThreadLocal);
  EXPECT(ptq2_set_stream(c, nullptr) == PTQ2_OK);
  S().launches.clear();
  EXPECT(all_operators(c) == PTQ2_OK);
  EXPECT(tiles() == 1 && count("k_a12") == 1 && count("k_diag") == 1);
  (void)hipStreamEndCapture((hipStream_t)0x10, &g);
  (void)hipGraphDestroy(g);
  ptq2_destroy(&c);
}

// The projection where only the sort's buffers and the nodal values fit: what it needed before it had a
// workspace of its own.
void projection_at_the_limit() {
  const Mesh m(4, 4, 2048);
  const int64_t ne = 32768, np = 8 * ne, nn = m.nvel / 3;
  std::vector<double> xi(3 * np, 0.0), v(np, 1.0), out(27 * ne);
  std::vector<int32_t> wil(np, 0);
  for (int dev = 0; dev < 2; dev++) {
    ptq2_ctx *c = m.make();
    const unsigned f = dev ? PTQ2_DEVICE : 0;
    const auto project = [&] {
      S().launches.clear();
      return ptq2_project_points_q1(c, np, xi.data(), wil.data(), v.data(), v.data(), out.data(), out.data(), f);
    };
    const size_t before = S().used;
    // the sort's keys, order and positions, its own scratch (at least keys and values), offsets, nodal values, staging
    const size_t need = (size_t)np * (12 + 8) + 8 * (size_t)(ne + 1) + 16 * (size_t)nn +
                        (dev ? 0 : (size_t)np * (24 + 4 + 16) + 2 * 27 * 8 * (size_t)ne);
    EXPECT(project() == PTQ2_OK && count("k_points_sums") == 1 && count("k_points_to_nodesILb0") == 1);
    const size_t kept = S().used - before;
    // a second call may use what the first one kept; without room the nodes sum the points themselves
    S().limit = before + need + (1 << 20);
    EXPECT(project() == PTQ2_OK && (dev || count("k_points_to_nodesILb1") == 1));
    EXPECT(ptq2_setup_mesh(c, 4, 4, 2048, m.coords.data(), nullptr, m.mask.data()) == PTQ2_OK);
    EXPECT(project() == PTQ2_OK && count("k_points_to_nodesILb1") == 1);
    // and an apply's buffers take the place of what it kept
    S().limit = SIZE_MAX;
    EXPECT(project() == PTQ2_OK && S().used >= before + kept);
    EXPECT(ptq2_set_viscosity(c, m.eta.data(), 3, 0) == PTQ2_OK);
    S().limit = S().used;
    double d[1];
    EXPECT(ptq2_a11_apply(c, d, d + 1, PTQ2_DEVICE) == PTQ2_OK);
    S().limit = SIZE_MAX;
    ptq2_destroy(&c);
    EXPECT(S().used == 0);
  }
}

void hierarchy_at_the_limit() {
  const Mesh m(128, 128, 32);  // 8192 bricks
  const size_t spare = spare_of(8192);
  ptq2_mg_opts o;
  ptq2_mg_default_opts(&o);
  o.nlevels = 5;
  o.fp32_smoother = 0;
  o.esteig_its = 1;
  o.autotune = 0;
  double v[1];
  for (int graph = 0; graph < 2; graph++) {
    o.use_graph = graph;
    S().peak = 0;
    ptq2_ctx *c = m.make();
    ptq2_mg *mg = nullptr;
    EXPECT(ptq2_mg_create(&mg, c, &o) == PTQ2_OK);
    const size_t all = S().peak;
    S().launches.clear();
    EXPECT(ptq2_mg_vcycle(mg, v, v) == PTQ2_OK && count("k_a11_fp64_t") > 0);
    const auto fine = [&](bool with) {  // the fine level's passes have tiles, or none has
      int n = 0;
      for (const Launch &l : S().launches) n += l.xtile != nullptr;
      return with ? n > 0 : n == 0;
    };
    EXPECT(fine(true));
    // the Krylov vectors find no room beside the spare memory: V-cycles go on without it
    const size_t had = S().used;
    S().limit = had + 4 * 8 * (size_t)m.nvel - spare / 2;
    int it;
    EXPECT(ptq2_mg_solve(mg, v, v, 1e-3, 1, 1, &it, nullptr, nullptr) == PTQ2_OK);
    S().limit = SIZE_MAX;
    S().launches.clear();
    EXPECT(ptq2_mg_vcycle(mg, v, v) == PTQ2_OK && count("k_a11_fp64_t") > 0 && fine(false));
    ptq2_mg_destroy(&mg);
    ptq2_destroy(&c);
    EXPECT(S().used == 0);
    // the set-up itself, where it fits without
    S().limit = all - spare / 2;
    c = m.make();
    EXPECT(ptq2_mg_create(&mg, c, &o) == PTQ2_OK);
    S().launches.clear();
    EXPECT(ptq2_mg_vcycle(mg, v, v) == PTQ2_OK && fine(false));
    ptq2_mg_destroy(&mg);
    ptq2_destroy(&c);
    EXPECT(S().used == 0);
    S().limit = SIZE_MAX;
  }
}
// The kernels that the autotuner compares do the same work: on a level of overlapping blocks, whose apply is
// complete, the others are launched with their face pass.
void autotuner_compares_like_with_like() {
  for (int m : {8, 64}) {
    const Mesh mesh(m, m, m);
    ptq2_ctx *c = mesh.make();
    ptq2_mg_opts o;
    ptq2_mg_default_opts(&o);
    o.nlevels = m == 8 ? 2 : 4;
    o.esteig_its = 1;
    S().launches.clear();
    ptq2_mg *mg = nullptr;
    EXPECT(ptq2_mg_create(&mg, c, &o) == PTQ2_OK);
    // up to 16^3 elements (5 blocks per axis) every level is one of overlapping blocks; 64^3 and 32^3 are not
    int with = 0, without = 0, own = 0;
    const std::vector<Launch> &l = S().launches;
    for (size_t i = 0; i + 1 < l.size(); i++) {
      own += l[i].name.find("k_a11_fp32_own") != std::string::npos;
      if (l[i].name.find("k_a11_fp32") == std::string::npos || l[i].name.find("_own") != std::string::npos) continue;
      const bool face = l[i + 1].name.find("k_gather_faces") != std::string::npos;
      (face ? with : without)++;
    }
    EXPECT(own > 0 && with > 0);
    EXPECT(m == 8 ? without == 0 : without > 0);
    ptq2_mg_destroy(&mg);
    ptq2_destroy(&c);
  }
}
}  // namespace

int main() {
  operators_at_the_limit();
  operators_under_capture();
  projection_at_the_limit();
  hierarchy_at_the_limit();
  autotuner_compares_like_with_like();
  if (bad) return 1;
  std::printf("host logic ok\n");
  return 0;
}
