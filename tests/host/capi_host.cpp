// The C-ABI's host logic (pelephysics_amd/csrc/capi.hip) without a GPU: the HIP
// runtime and the mechanism launchers are restated here as recorders, so that
// what a call allocates, clears, launches and returns can be looked at.
//
//   capi_host SCENARIO   prints "key value" lines
//
// Device memory is host memory from a pool in which a freed block is the next
// one handed out (oldest first), as a device allocator may do.  Kernels do not
// run but for zero_ints; reduce_stats hands over a preset result unless `deliver`
// is off.
#include "../../pelephysics_amd/csrc/capi.hip"

#include <deque>
#include <map>

namespace fake {
constexpr size_t BLOCK = 1 << 20;
std::deque<char*> freed;
int malloc_fails_in = -1;  // allocations until one fails (-1: none)
int captures = 0, replays = 0;
bool deliver = true;
unsigned long long result[NSTAT] = {};
const void *acc = nullptr;           // reduce_stats' accumulators of the last call
bool acc_clear = false;              // and whether they were zero then
char symbol[1024];                   // the device scratch's address (never dereferenced)
// last integrator launch
std::string launched;
int mode = -1, ncells = -1;
ppc::CellStats st{};
ppc::ReactParamsDev P{};

hipError_t react_1d(int m, const ppc::ReactParamsDev& p, double*, const double*, double*, const double*, double,
                    int n, ppc::CellStats s, int, hipStream_t) {
  launched = "lane_1d", mode = m, ncells = n, st = s, P = p;
  return hipSuccess;
}
hipError_t react_box(int m, const ppc::ReactParamsDev& p, const ppc::BoxArgs&, double, int n, ppc::CellStats s, int,
                     hipStream_t) {
  launched = "lane_box", mode = m, ncells = n, st = s, P = p;
  return hipSuccess;
}
hipError_t batched_1d(int m, const ppc::ReactParamsDev& p, double*, const double*, double*, const double*, double,
                      ppc::QueueArgs q, ppc::CellStats s, hipStream_t) {
  launched = "group_1d", mode = m, ncells = q.ncells, st = s, P = p;
  return hipSuccess;
}
hipError_t group_fixed(int, const ppc::ReactParamsDev&, double*, const double*, double*, const double*,
                       const ppc::BoxArgs*, double, int, int, ppc::CellStats, hipStream_t) {
  return hipErrorNotSupported;
}
hipError_t adjoint(const ppc::ReactParamsDev&, const ppc::AdjointArgs&, hipStream_t) { return hipSuccess; }
hipError_t flatten(const ppc::FlatArgs&, int, hipStream_t) { return hipSuccess; }
hipError_t mech_eval(int, const double*, const double*, int, double*, hipStream_t) { return hipSuccess; }
long long no_rows(int) { return 0; }
long long lane_rows(int) { return 5000; }
long long group_rows(int cpw) { return cpw == 4 ? 52 : (cpw == 2 ? 30 : 0); }
long long wide_rows(int cpw) { return cpw == 1 ? 20 : 0; }

// 20 species; a workspace of the one-lane kernels and group kernels as asked
MechLauncher mech(const char* name, bool lane_ws, bool groups) {
  MechLauncher L{};
  L.name = name, L.ns = 20, L.nr = 30, L.batched_ok = 1;
  L.react_1d = &react_1d, L.react_box = &react_box, L.batched_1d = &batched_1d, L.group_fixed = &group_fixed;
  L.adjoint_1d = &adjoint, L.flatten = &flatten, L.mech_eval = &mech_eval;
  L.ws_rows = lane_ws ? &lane_rows : &no_rows;
  L.group_ws_rows = groups ? &group_rows : &no_rows;
  return L;
}
}  // namespace fake

// The mechanisms: "heptane_lu_88sk" with a workspace of the one-lane kernels,
// "dodecane_lu" without group kernels, "LuEthylene_qss" with the widest groups
// only, the others with groups of 16 and 32 lanes and no such workspace.
namespace ppc {
#define PPC_MECH(M)                                                                   \
  const MechLauncher* launcher_##M() {                                                \
    static const MechLauncher L = [] {                                                \
      const std::string name = #M;                                                    \
      MechLauncher l = fake::mech(#M, name == "heptane_lu_88sk", name != "dodecane_lu"); \
      if (name == "LuEthylene_qss") l.group_ws_rows = &fake::wide_rows;               \
      return l;                                                                       \
    }();                                                                              \
    return &L;                                                                        \
  }
#include "../../pelephysics_amd/csrc/inst/registry.inc"
#undef PPC_MECH
const MechLauncher* manifold_launcher(int) { return nullptr; }
}  // namespace ppc

// ---------------------------------------------------- the HIP runtime --
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  *p = nullptr;
  if (fake::malloc_fails_in >= 0 && fake::malloc_fails_in-- == 0) return hipErrorOutOfMemory;
  if (n > fake::BLOCK) return hipErrorOutOfMemory;
  if (fake::freed.empty()) {
    *p = std::malloc(fake::BLOCK);
  } else {
    *p = fake::freed.front();
    fake::freed.pop_front();
  }
  std::memset(*p, 0xab, fake::BLOCK);
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (p) fake::freed.push_back((char*)p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return (*p = std::calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 2; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = fake::symbol; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)fake::symbol; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { *t = 1.f; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)fake::symbol; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { ++fake::captures; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = (hipGraph_t)fake::symbol; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { *e = (hipGraphExec_t)fake::symbol; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { ++fake::replays; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

static dim3 cfg_grid, cfg_block;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) { cfg_grid = g, cfg_block = b; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
  *g = cfg_grid, *b = cfg_block, *m = 0, *s = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
  if (f == (const void*)&reduce_stats) {
    const unsigned long long* acc = *(unsigned long long**)args[7];
    fake::acc = acc;
    fake::acc_clear = true;
    for (int i = 0; i <= NSTAT; ++i) fake::acc_clear = fake::acc_clear && acc[i] == 0;
    unsigned long long* host = *(unsigned long long**)args[8];
    if (fake::deliver)
      for (int i = 0; i < NSTAT; ++i) host[i] = fake::result[i];
  } else if (f == (const void*)&zero_ints) {
    std::memset(*(int**)args[0], 0, sizeof(int) * (size_t)(*(int*)args[1]));
  }
  return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, uint3*, uint3*, dim3*, dim3*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
}

// --------------------------------------------------------- scenarios --
namespace {

double buf[1 << 16];  // stands for every device array; kernels do not run

pp_chem* handle(const char* name, int mode, long long workspace_bytes = 0) {
  pp_chem_config c;
  pp_chem* h = nullptr;
  if (pp_chem_config_init(&c, name, mode, 2) != 0) std::abort();
  c.workspace_bytes = workspace_bytes;
  std::printf("create %d\n", pp_chem_create(&c, &h));
  return h;
}

int call_1d(pp_chem* h, int n) {
  double dt = 1e-5, t = 0;
  return pp_chem_react_1d(h, buf, buf, buf, buf, &dt, &t, n, 1, nullptr);
}
int call_chained(pp_chem* h, int n, int calls) {
  double dt = 1e-5, t = 0;
  return pp_chem_react_1d_chained(h, buf, buf, buf, buf, &dt, &t, n, calls, nullptr);
}
int call_noalloc(pp_chem* h, int n) {
  double dt = 1e-5, t = 0;
  return pp_chem_react_1d_noalloc(h, buf, buf, buf, buf, &dt, &t, n, nullptr);
}
int call_box(pp_chem* h, int n) {
  pp_array4 a{};
  a.p = buf, a.jstride = n, a.kstride = n, a.nstride = n, a.ncomp = 20;
  a.end[0] = n, a.end[1] = a.end[2] = 1;
  const int lo[3] = {0, 0, 0}, hi[3] = {n - 1, 0, 0};
  double dt = 1e-5, t = 0;
  return pp_chem_react_box(h, lo, hi, &a, &a, &a, &a, &a, &a, nullptr, &dt, &t, nullptr);
}

// a call's statistics do not arrive: an error, and the next call is sound again
void undelivered() {
  pp_chem* h = handle("drm19", PP_CHEM_RK64);
  fake::result[0] = 800;  // 8 steps a cell
  std::printf("first %d\nclear_at_first %d\n", call_1d(h, 100), (int)fake::acc_clear);
  fake::deliver = false;
  h->d_red[0] = 5, h->d_red[NSTAT] = 3;  // what such a call leaves behind
  std::printf("undelivered %d\n", call_1d(h, 100));
  fake::deliver = true;
  std::printf("next %d\nclear_at_next %d\n", call_1d(h, 100), (int)fake::acc_clear);
}

// two handles' calls without allocation share no accumulators
void noalloc_shared() {
  pp_chem *a = handle("drm19", PP_CHEM_RK64), *b = handle("drm19", PP_CHEM_RK64);
  call_noalloc(a, 100);
  const void* first = fake::acc;
  call_noalloc(b, 100);
  std::printf("shared %d\n", (int)(first == fake::acc));
}

// counters that grew between two chained calls, at the address they had: the
// captured launches hold their old layout
void graph_counters() {
  pp_chem* h = handle("drm19", PP_CHEM_BDF_ADAPTIVE_MIXED);
  call_chained(h, 100, 3);
  const int* nrhs = fake::st.nrhs;
  const void* cnt = h->d_cnt;
  std::printf("captures %d\n", fake::captures);
  call_1d(h, 200);
  std::printf("same_address %d\n", (int)(cnt == h->d_cnt));
  call_chained(h, 100, 3);
  std::printf("same_layout %d\n", (int)(nrhs == fake::st.nrhs));
  std::printf("captures_after_growth %d\n", fake::captures);
  call_chained(h, 100, 3);
  std::printf("captures_again %d\n", fake::captures);
}

// an allocation that fails while a buffer grows: the next call that fitted
// before allocates again
void failed_growth(int which) {
  pp_chem* h = handle("drm19", which == 2 ? PP_CHEM_BDF : PP_CHEM_BDF_ADAPTIVE);
  const auto call = [&](int n) {
    double dt = 1e-5, t = 0, g[4] = {};
    switch (which) {
      case 1: return pp_chem_react_1d(h, buf, buf, buf, buf, &dt, &t, n, 0, nullptr);
      case 2: return pp_chem_adjoint_1d(h, buf, buf, n, 1, dt, 0, 1, g, buf, nullptr);
      default: return call_1d(h, n);
    }
  };
  std::printf("before %d\n", call(10));
  // counters: the first or the second of their two; staging and checkpoints: their one
  if (which == 1) call_1d(h, 20);  // the counters have grown already
  fake::malloc_fails_in = which == 3 ? 1 : 0;
  std::printf("failed %d\n", call(20));
  fake::malloc_fails_in = -1;
  std::printf("after %d\n", call(10));
  std::printf("counters %d\n", (int)(which == 2 || (h->d_cnt && h->d_order)));
  std::printf("staging %d\n", (int)(which != 1 || h->d_stage));
  std::printf("checkpoints %d\n", (int)(which != 2 || h->d_ckpt));
}

// a mechanism without group kernels: the batched forms and ReactorCvode run on
// the one-lane-per-cell kernels of the adaptive BDF
void no_groups(int mode) {
  pp_chem* h = handle("dodecane_lu", mode);
  const auto say = [&](const char* what, int r) {
    std::printf("%s %d\n%s_kernel %s\n%s_adaptive %d\n", what, r, what, fake::launched.c_str(), what,
                (int)(fake::mode == ppc::MODE_ADAPTIVE && fake::P.adapt.fc_rhs == (mode == PP_CHEM_CVODE)));
  };
  fake::launched = "none";
  say("react_1d", call_1d(h, 10));
  say("box", call_box(h, 10));
  say("chained", call_chained(h, 10, 2));
  say("noalloc", call_noalloc(h, 10));
  std::printf("rows %lld\n", pp_chem_workspace_rows(h));
}

// cells per wave of a call, where the caller leaves them to the library
void group_size() {
  for (const char* name : {"drm19", "LuEthylene_qss"}) {
    pp_chem* h = handle(name, PP_CHEM_BDF_BATCHED_FP64);
    for (int n : {1, 10000}) {
      const int r = call_1d(h, n);
      std::printf("%s_%d %d\n", name, n, r == 0 ? fake::P.adapt.group : r);
    }
  }
}

// workspace_bytes below one wave's workspace
void small_workspace() {
  pp_chem* h = handle("drm19", PP_CHEM_BDF_ADAPTIVE_MIXED, 1000);
  std::printf("small_mechanism %d\n", call_1d(h, 100));
  std::printf("workspace_lanes %lld\n", fake::P.ws_lanes);
  h = handle("drm19", PP_CHEM_CVODE, 1000);
  std::printf("small_mechanism_cvode %d\n", call_box(h, 100));
  h = handle("heptane_lu_88sk", PP_CHEM_BDF_ADAPTIVE_MIXED, 1000);
  std::printf("large_mechanism %d\n", call_1d(h, 100));
  pp_chem_config c;
  pp_chem_config_init(&c, "drm19_table", PP_CHEM_BDF_ADAPTIVE_MIXED, 2);
  c.workspace_bytes = 1000;
  c.batched_cells_per_wave = 4;
  pp_chem_create(&c, &h);
  std::printf("named_group %d\n", call_1d(h, 100));
}

}  // namespace

int main(int argc, char** argv) {
  const std::string s = argc > 1 ? argv[1] : "";
  if (s == "undelivered") undelivered();
  else if (s == "noalloc_shared") noalloc_shared();
  else if (s == "graph_counters") graph_counters();
  else if (s.rfind("failed_growth", 0) == 0) failed_growth(s.back() - '0');
  else if (s.rfind("no_groups", 0) == 0) no_groups(s.back() - '0');
  else if (s == "group_size") group_size();
  else if (s == "small_workspace") small_workspace();
  else return 2;
  return 0;
}
