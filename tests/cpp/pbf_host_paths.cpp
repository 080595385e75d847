// Host paths of libpbf.so without a GPU: this program defines the HIP runtime
// calls that the library makes (its definitions come before libamdhip64's).
// Device memory is host memory, kernels do not run, and every launch and copy is
// checked: a pointer it hands over has to lie in a live allocation, and the
// arrays of a neighbor view have to be as long as the kernels read them. A chosen
// allocation can be made to fail, a stream to say that it is being captured, and
// the counters of a call to report what the test wants. Run by
// tests/test_host_paths.py with the name of a scenario; prints one line per
// violation and exits 1 if there is any.
#include <cxxabi.h>
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "../../physika-old_amd/csrc/pbf_internal.h"
#include "pbf.h"

namespace {

struct Kernel {
  std::string name;                 // without template arguments and namespace
  std::string full;                 // demangled
  std::vector<std::string> params;  // types
};

struct Launch {
  std::string name, full;
  unsigned block;
  pbf::NbrView nv;  // where the kernel's first parameter is one
  bool view;
};

constexpr long kNever = -1000000;

struct State {
  std::map<const void*, Kernel> kernels;
  std::map<const char*, size_t> live;
  size_t bytes = 0, peak = 0;
  long mallocs = 0, fail_at = kNever;  // fail_at: the malloc (0-based) that fails
  size_t fail_over = SIZE_MAX;     // every malloc of more bytes fails
  long copy_fail_at = kNever;  // copies left until one fails
  hipError_t last = hipSuccess;
  int capturing = 0;        // hipStreamIsCapturing: 0 no, 1 yes, 2 an error
  unsigned long long list_need = 0, calls = 0, uneven = 0, pairs = 0;
  bool graph = false;  // between hipStreamBeginCapture and hipStreamEndCapture
  std::vector<Launch> launches, recorded;  // recorded: by the last graph
  std::vector<std::string> ops;  // launches, copies and waits, in order
  std::map<const void*, long> searched;  // buffer of a search -> serial of the neighbor pass that last wrote it
  long searches = 0, exported = -1;      // exported: the search that the last export read
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
  int violations = 0;
};

State& S() {
  static State* s = new State();
  return *s;
}

void violation(const char* fmt, ...) {
  va_list a;
  va_start(a, fmt);
  std::printf("VIOLATION ");
  std::vprintf(fmt, a);
  std::printf("\n");
  va_end(a);
  ++S().violations;
}

// Bytes from p to the end of its live allocation (0: in none).
size_t room(const void* p) {
  auto it = S().live.upper_bound(static_cast<const char*>(p));
  if (it == S().live.begin()) return 0;
  --it;
  const char* q = static_cast<const char*>(p);
  return q < it->first + it->second ? (size_t)(it->first + it->second - q) : 0;
}

void need(const Kernel& k, const char* what, const void* p, size_t bytes) {
  if (bytes > 0 && room(p) < bytes)
    violation("%s: %s at %p needs %zu bytes, has %zu", k.name.c_str(), what, p, bytes, room(p));
}

void check_view(const Kernel& k, const pbf::NbrView& v) {
  const size_t n = (size_t)v.n, waves = (n + 63) / 64;
  need(k, "ssid", v.ssid, 4 * n);
  need(k, "win", v.win, sizeof(pbf::SceneWin));
  need(k, "cell_start", v.cell_start, 8);
  need(k, "xn", v.xn, 16 * (n + pbf::kXnPad));
  need(k, "nbr_cnt", v.nbr_cnt, 4 * n);
  need(k, "cnt_a", v.cnt_a, 2 * n);
  need(k, "list_base", v.list_base, 8 * waves);
  need(k, "list_jbase", v.list_jbase, 4 * waves);
  need(k, "list_mode", v.list_mode, 4 * waves);
  need(k, "mask_base", v.mask_base, 8 * waves);
  need(k, "stage", v.stage, sizeof(int) * pbf::kStageInts * waves);
  need(k, "counters", v.counters, 8 * pbf::kDeviceCounters);
  // the lists, and the two chunks that a lane pair reads ahead of the wave's words
  need(k, "list", v.list, 2 * (64 * waves * (size_t)v.list_per + pbf::kListPad));
}

// The arrays that a search leaves for the passes and the export.
std::vector<const void*> outputs(const pbf::NbrView& v) {
  return {v.list,       v.nbr_cnt,   v.xn,        v.ssid, v.list_base, v.list_jbase,
          v.list_mode,  v.mask_base, v.mask,      v.cnt_a, v.stage,    v.win,
          v.cell_start};
}

void launched(const void* f, dim3 block, void** args) {
  const Kernel& k = S().kernels[f];
  Launch l{k.name, k.full, block.x, {}, false};
  for (size_t i = 0; i < k.params.size(); ++i) {
    const std::string& t = k.params[i];
    if (t == "pbf::NbrView") {
      l.nv = *static_cast<pbf::NbrView*>(args[i]);
      l.view = true;
      check_view(k, l.nv);
    } else if (!t.empty() && t.back() == '*') {
      const void* p = *static_cast<void**>(args[i]);
      if (p && room(p) == 0) violation("%s: argument %zu (%s) points at no allocation: %p", k.name.c_str(), i, t.c_str(), p);
    }
  }
  if (S().graph) {
    S().recorded.push_back(l);
    return;
  }
  S().launches.push_back(l);
  S().ops.push_back(k.name);
  if (S().capturing == 1) return;
  if (k.name == "k_neighbors" || k.name == "k_neighbors_small") {
    for (const void* p : outputs(l.nv)) S().searched[p] = S().searches;
    ++S().searches;
  }
  if (k.name == "k_csr_fill") {
    S().exported = S().searched.count(l.nv.list) ? S().searched[l.nv.list] : -1;
    for (const void* p : outputs(l.nv))
      if (!S().searched.count(p) || S().searched[p] != S().exported) violation("k_csr_fill: arrays of different searches");
  }
  if (k.name == "k_wave_stats") {  // the counters of the call
    auto* host = *static_cast<unsigned long long**>(args[4]);
    for (int c = 0; c < pbf::C_COUNT; ++c) host[c] = 0;
    host[pbf::C_LIST_NEED] = S().list_need;
    host[pbf::C_CALLS] = ++S().calls;
    host[pbf::C_UNEVEN] = S().uneven;
    host[pbf::C_PAIRS] = S().pairs;
  }
}

void copied(const void* dst, const void* src, size_t bytes, hipMemcpyKind kind) {
  if (kind != hipMemcpyDeviceToHost && room(dst) < bytes) violation("copy of %zu bytes past its target", bytes);
  if (kind != hipMemcpyHostToDevice && room(src) < bytes) violation("copy of %zu bytes past its source", bytes);
  std::memmove(dst ? const_cast<void*>(dst) : nullptr, src, bytes);
}

Kernel parse(const char* mangled) {
  int status = 0;
  char* d = abi::__cxa_demangle(mangled, nullptr, nullptr, &status);
  Kernel k;
  k.full = status == 0 ? d : mangled;
  std::free(d);
  // parameters: the last balanced (...) of the text, split at its commas
  size_t open = k.full.rfind(')');
  int depth = 0;
  for (; open != std::string::npos; --open) {
    depth += k.full[open] == ')' ? 1 : (k.full[open] == '(' ? -1 : 0);
    if (depth == 0 || open == 0) break;
  }
  std::string head = k.full.substr(0, open), arg;
  depth = 0;
  for (size_t i = open + 1; i + 1 < k.full.size(); ++i) {
    const char c = k.full[i];
    depth += c == '<' || c == '(' ? 1 : (c == '>' || c == ')' ? -1 : 0);
    if (c == ',' && depth == 0) {
      k.params.push_back(arg);
      arg.clear();
    } else if (!(c == ' ' && arg.empty())) {
      arg += c;
    }
  }
  if (!arg.empty()) k.params.push_back(arg);
  head = head.substr(0, head.find('<'));
  const size_t at = head.rfind(':');
  k.name = at == std::string::npos ? head : head.substr(at + 1);
  if (k.name.rfind("void ", 0) == 0) k.name = k.name.substr(5);
  return k;
}

}  // namespace

// -- the HIP runtime --------------------------------------------------------
extern "C" {
void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  S().kernels[f] = parse(name);
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t st) {
  S().grid = g;
  S().block = b;
  S().shared = m;
  S().stream = st;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* st) {
  *g = S().grid;
  *b = S().block;
  *m = S().shared;
  *st = S().stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3 b, void** args, size_t, hipStream_t) {
  launched(f, b, args);
  return hipSuccess;
}
hipError_t hipExtLaunchKernel(const void* f, dim3, dim3 b, void** args, size_t, hipStream_t, hipEvent_t, hipEvent_t,
                              int) {
  launched(f, b, args);
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t bytes) {
  *p = nullptr;
  const long k = S().mallocs++;
  if (k == S().fail_at || bytes > S().fail_over) {
    return S().last = hipErrorOutOfMemory;
  }
  *p = std::calloc(bytes ? bytes : 1, 1);
  S().live[static_cast<char*>(*p)] = bytes;
  S().bytes += bytes;
  S().peak = std::max(S().peak, S().bytes);
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  auto it = S().live.find(static_cast<char*>(p));
  if (it == S().live.end()) {
    violation("free of %p, which is no live allocation", p);
    return hipErrorInvalidValue;
  }
  S().bytes -= it->second;
  S().live.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = std::calloc(bytes, 1);
  S().live[static_cast<char*>(*p)] = bytes;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  if (!p) return hipSuccess;
  S().live.erase(static_cast<char*>(p));
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
  *d = h;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  return hipMalloc(p, 2 * (size_t)PBF_NOALLOC_MAX_PARTICLES * 16 + 4096);
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t bytes, hipMemcpyKind kind, hipStream_t) {
  if (S().copy_fail_at != kNever && S().copy_fail_at-- == 0) return S().last = hipErrorUnknown;
  copied(d, s, bytes, kind);
  S().ops.push_back("copy");
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t bytes, hipMemcpyKind kind) {
  return hipMemcpyAsync(d, s, bytes, kind, nullptr);
}
hipError_t hipMemset(void* d, int v, size_t bytes) {
  if (room(d) < bytes) violation("memset of %zu bytes past its target", bytes);
  else std::memset(d, v, bytes);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t bytes, hipStream_t) { return hipMemset(d, v, bytes); }
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "host");
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* v, const void*, int, size_t) {
  *v = 4;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
  S().ops.push_back("wait");
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
  if (S().capturing == 2) return S().last = hipErrorStreamCaptureImplicit;
  *s = S().capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  S().graph = true;
  S().recorded.clear();
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  S().graph = false;
  *g = reinterpret_cast<hipGraph_t>(8);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *x = reinterpret_cast<hipGraphExec_t>(8);
  S().ops.push_back("instantiate");
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
  for (const Launch& l : S().recorded) S().launches.push_back(l);
  S().ops.push_back("replay");
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(8);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) {
  S().ops.push_back("wait");
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = S().last;
  S().last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "an error of the test"; }
}  // extern "C"

namespace {

// -- scenarios --------------------------------------------------------------
pbf_params small_params() {
  pbf_params p;
  pbf_params_default(&p);
  p.smoothing_length = 0.1f;  // a small grid
  p.sampling_distance = 0.04f;
  return p;
}

template <class T> T* device(size_t n) {
  void* p = nullptr;
  const long keep = S().fail_at;
  const size_t over = S().fail_over;
  S().fail_at = kNever;
  S().fail_over = SIZE_MAX;
  --S().mallocs;
  (void)hipMalloc(&p, sizeof(T) * n);
  S().fail_at = keep;
  S().fail_over = over;
  return static_cast<T*>(p);
}

struct Arrays {
  float *x, *v, *rho;
  double *dx, *dv;
  int *index, *elems;
  explicit Arrays(size_t n)
      : x(device<float>(3 * n)), v(device<float>(3 * n)), rho(device<float>(n)), dx(device<double>(3 * n)),
        dv(device<double>(3 * n)), index(device<int>(n)), elems(device<int>(n)) {}
};

void expect(bool ok, const char* what) {
  if (!ok) violation("%s", what);
}

// Every allocation of a sequence of calls fails once; each call is repeated
// until it gets through. No launch may see a pointer to nothing.
void failed_allocations(const std::vector<std::function<int(pbf_ctx*, Arrays&)>>& calls, unsigned flags) {
  long total = 1;
  for (long f = -1; f < total; ++f) {
    Arrays a(3000);
    pbf_params p = small_params();
    p.flags = flags;
    S().list_need = 96;
    pbf_ctx* c = nullptr;
    if (pbf_create(&p, &c) != PBF_OK) std::abort();
    const long start = S().mallocs;
    S().fail_at = f < 0 ? kNever : start + f;
    for (size_t k = 0; k < calls.size(); ++k) {
      int st = PBF_OK;
      for (int attempt = 0; attempt < 3; ++attempt)
        if ((st = calls[k](c, a)) == PBF_OK) break;
      if (st != PBF_OK) violation("call %zu with allocation %ld failing: %s", k, f, pbf_last_error(c));
    }
    if (f < 0) total = S().mallocs - start;
    S().fail_at = kNever;
    pbf_destroy(c);
    S().searched.clear();
  }
  std::printf("%ld allocations\n", total);
}

int step(pbf_ctx* c, Arrays& a, int n) { return pbf_step(c, a.x, a.v, a.rho, n, 1, nullptr); }

int dense(pbf_ctx* c, Arrays& a, int n, unsigned long long slots) {  // the next call's lists grow
  S().list_need = slots;
  const int st = step(c, a, n);
  S().list_need = 96;
  return st;
}

void list_reservation() {
  failed_allocations({[](pbf_ctx* c, Arrays& a) { return step(c, a, 500); },
                      [](pbf_ctx* c, Arrays& a) { return step(c, a, 2000); },
                      [](pbf_ctx* c, Arrays& a) { return dense(c, a, 2000, 400); },
                      [](pbf_ctx* c, Arrays& a) { return step(c, a, 2000); }},
                     0);
}

int forward(pbf_ctx* c, Arrays& a, bool f64, int n, int nsteps, int every) {
  return f64 ? pbf_rollout_forward_f64(c, a.dx, a.dv, nullptr, nullptr, 1, n, nsteps, every, nullptr)
             : pbf_rollout_forward(c, a.x, a.v, a.rho, nullptr, 1, n, nsteps, every, nullptr);
}

int backward(pbf_ctx* c, Arrays& a, bool f64) {
  return f64 ? pbf_rollout_backward_f64(c, a.dx, a.dv, nullptr) : pbf_rollout_backward(c, a.x, a.v, nullptr);
}

// A reverse that ran out of memory is not tried again: the next forward records
// into the slots that are there.
int backward_once(pbf_ctx* c, Arrays& a, bool f64) {
  const int st = backward(c, a, f64);
  return st == PBF_ERR_ALLOC ? PBF_OK : st;
}

void tape_slots() {
  for (bool f64 : {false, true})
    for (bool again : {false, true})
      failed_allocations({[=](pbf_ctx* c, Arrays& a) { return forward(c, a, f64, 1500, 5, 3); },
                          [=](pbf_ctx* c, Arrays& a) { return again ? backward(c, a, f64) : backward_once(c, a, f64); },
                          [=](pbf_ctx* c, Arrays& a) { return forward(c, a, f64, 1500, 5, 3); },
                          [=](pbf_ctx* c, Arrays& a) { return backward(c, a, f64); },
                          [=](pbf_ctx* c, Arrays& a) { return forward(c, a, !f64, 1500, 3, 3); },
                          [=](pbf_ctx* c, Arrays& a) { return backward(c, a, !f64); }},
                         0);
}

long exported(pbf_ctx* c, Arrays& a) {  // the search that step_neighbors exports
  long long total = 0;
  S().exported = -1;
  if (pbf_step_neighbors(c, a.index, a.elems, 0, &total, nullptr) != PBF_OK) violation("step_neighbors: %s", pbf_last_error(c));
  return S().exported;
}

void last_search() {
  for (bool f64 : {false, true})
    for (int every : {1, 2, 3, 5, 9}) {
      Arrays a(3000);
      pbf_params p = small_params();
      pbf_ctx* c = nullptr;
      if (pbf_create(&p, &c) != PBF_OK) std::abort();
      S().list_need = 96;
      long last = 0;
      for (int round = 0; round < 3; ++round) {
        expect(forward(c, a, f64, 1500, 5, every) == PBF_OK, "forward");
        last = S().searches - 1;
        expect(exported(c, a) == last, "lists after a forward");
        if (round < 2) expect(backward(c, a, f64) == PBF_OK, "reverse");
      }
      // a captured call that has not been replayed
      S().capturing = 1;
      expect(step(c, a, 1500) == PBF_OK, "captured step");
      S().capturing = 0;
      expect(exported(c, a) == last, "lists before the first replay");
      expect(backward(c, a, f64) == PBF_OK, "reverse");
      expect(step(c, a, 1500) == PBF_OK, "step");
      expect(exported(c, a) == S().searches - 1, "lists of the step");
      pbf_destroy(c);
      S().searched.clear();
    }
}

// A forward or a reverse that fails on its way leaves no lists to export, or
// whole ones.
void failed_rollout() {
  for (bool f64 : {false, true})
    for (long f = 0; f < 60; ++f) {
      Arrays a(3000);
      pbf_params p = small_params();
      pbf_ctx* c = nullptr;
      if (pbf_create(&p, &c) != PBF_OK) std::abort();
      S().list_need = 96;
      expect(forward(c, a, f64, 1500, 4, 2) == PBF_OK && backward(c, a, f64) == PBF_OK, "rollout");
      expect(step(c, a, 700) == PBF_OK, "step");
      for (bool reverse : {false, true}) {
        S().copy_fail_at = f;
        const int st = reverse ? backward(c, a, f64) : forward(c, a, f64, 1500, 4, 2);
        S().copy_fail_at = kNever;
        expect(S().last == hipSuccess, "an error left for the next call");
        S().last = hipSuccess;
        long long total = 0;
        S().exported = -1;
        if (pbf_step_neighbors(c, a.index, a.elems, 0, &total, nullptr) == PBF_OK) {
          expect(!reverse || st != PBF_OK, "lists after a reverse");
          expect(S().exported == S().searches - 1, "lists after a failed call");
        }
        if (!reverse && st != PBF_OK) expect(forward(c, a, f64, 1500, 4, 2) == PBF_OK, "forward again");
      }
      pbf_destroy(c);
      S().searched.clear();
    }
}

// Steps recorded by a forward (or run again by a reverse): where recording is off a
// forward records none, and the reverse runs its segment again.
void unrecorded_forward() {
  auto taped = [] {
    int k = 0;
    for (const Launch& l : S().launches) k += l.name == "k_copy_cells";
    S().launches.clear();
    return k;
  };
  for (bool f64 : {false, true}) {
    Arrays a(3000);
    pbf_params p = small_params();
    pbf_ctx* c = nullptr;
    if (pbf_create(&p, &c) != PBF_OK) std::abort();
    S().list_need = 96;
    taped();
    // a first rollout, recorded ones, one that is not, a recorded one again
    const int on[] = {1, 1, 0, 0, 1}, want[] = {0, 2, 0, 0, 2};
    for (int k = 0; k < 5; ++k) {
      expect(pbf_rollout_record(c, on[k]) == PBF_OK, "pbf_rollout_record");
      expect(forward(c, a, f64, 1500, 5, 3) == PBF_OK && taped() == want[k], "steps that the forward records");
      expect(exported(c, a) == S().searches - 1, "lists of the forward");
      if (k == 2) continue;  // nothing follows
      S().launches.clear();
      expect(backward(c, a, f64) == PBF_OK && taped() == 5 - want[k], "steps that the reverse runs");
    }
    expect(pbf_rollout_record(nullptr, 1) == PBF_ERR_INVALID, "null context");
    pbf_destroy(c);
    S().searched.clear();
  }
}

// A call on a stream that HIP says nothing about (the null stream while another one
// is captured) is not taken for a captured one: the forwards after it record again.
void unknown_capture() {
  for (bool f64 : {false, true}) {
    Arrays a(3000);
    pbf_params p = small_params();
    pbf_ctx* c = nullptr;
    if (pbf_create(&p, &c) != PBF_OK) std::abort();
    S().list_need = 96;
    expect(forward(c, a, f64, 1500, 5, 3) == PBF_OK && backward(c, a, f64) == PBF_OK, "rollout");
    for (int state : {2, 1}) {
      S().capturing = state;
      expect(step(c, a, 1500) == PBF_OK, "step");
      S().capturing = 0;
      expect(S().last == hipSuccess, "an error left for the next call");
      S().launches.clear();
      expect(forward(c, a, f64, 1500, 5, 3) == PBF_OK, "forward");
      int taped = 0;
      for (const Launch& l : S().launches) taped += l.name == "k_copy_cells";
      expect(taped == (state == 2 ? 2 : 0), "steps that the forward records");
      expect(backward(c, a, f64) == PBF_OK, "reverse");
    }
    pbf_destroy(c);
    S().searched.clear();
  }
}

// Frames replayed from a graph that was captured when the scene was even look at the
// counts again once it is uneven; the graph stays otherwise.
void replays_of_uneven_scenes() {
  Arrays a(300000);
  pbf_params p = small_params();
  pbf_ctx* c = nullptr;
  if (pbf_create(&p, &c) != PBF_OK) std::abort();
  S().list_need = 96;
  auto frames = [&](unsigned long long uneven_after) {  // how many passes look at the counts
    S().launches.clear();
    S().ops.clear();
    S().uneven = uneven_after;
    expect(pbf_step(c, a.x, a.v, a.rho, 280000, 4, nullptr) == PBF_OK, "frames");
    int look = 0, passes = 0;
    for (const Launch& l : S().launches)
      if (l.name == "k_density_lambda") ++passes, look += l.nv.maybe_uneven;
    expect(passes == 20, "passes of four frames");
    return look;
  };
  auto captures = [&] {
    int k = 0;
    for (const std::string& op : S().ops) k += op == "instantiate";
    return k;
  };
  expect(step(c, a, 280000) == PBF_OK, "a frame");  // says that the scene is even
  S().uneven = 1;
  expect(step(c, a, 280000) == PBF_OK, "a frame");
  expect(frames(1) == 0 && captures() == 1, "an even scene");
  expect(frames(2) == 0 && captures() == 0, "the scene turns uneven during the call");
  expect(frames(2) == 20 && captures() == 1, "an uneven scene");
  expect(frames(1) == 20 && captures() == 0, "it turns even again");
  expect(frames(1) == 10 && captures() == 0, "the graph's frames still look, the others do not");
  pbf_destroy(c);
}

// The row starts are in the caller's array when the call returns: nothing is copied
// after its last wait, counted by this call or by one before.
void blocking_export() {
  Arrays a(3000);
  pbf_params p = small_params();
  pbf_ctx* c = nullptr;
  if (pbf_create(&p, &c) != PBF_OK) std::abort();
  expect(step(c, a, 1500) == PBF_OK, "step");
  for (int call = 0; call < 3; ++call) {
    long long total = 0;
    S().ops.clear();
    expect(pbf_step_neighbors(c, a.index, call < 2 ? nullptr : a.elems, 0, &total, nullptr) == PBF_OK, "export");
    bool copied = false, open = false;
    for (const std::string& op : S().ops) {
      copied |= op == "copy";
      open = op == "copy" || (open && op != "wait");
    }
    expect(copied && !open, "a copy after the last wait");
  }
  pbf_destroy(c);
}

// The weights that a viscosity solve keeps: bounded in bytes, reserved with the
// other buffers, and not asked for again in every step once there is no room.
void viscosity_weights() {
  constexpr size_t limit = 192u << 20;
  auto kept = [] {  // whether the last step kept them
    for (auto l = S().launches.rbegin(); l != S().launches.rend(); ++l)
      if (l->name == "k_viscosity") return l->full.find("VisWeights)2") != std::string::npos;
    return false;
  };
  Arrays a(300000);
  pbf_params p = small_params();
  p.flags = PBF_FLAG_VISCOSITY;
  for (int slots : {96, 200, 400, 800, 1600})
    for (int n : {2000, 30000, 65536, 190000}) {
      p.list_slots = slots;
      pbf_ctx* c = nullptr;
      if (pbf_create(&p, &c) != PBF_OK) std::abort();
      expect(pbf_reserve(c, 190000) == PBF_OK, "reserve");
      pbf_params none = p;
      none.flags = 0;
      size_t without = S().bytes;
      {  // the context without weights
        pbf_ctx* d = nullptr;
        const size_t before = S().bytes;
        if (pbf_create(&none, &d) != PBF_OK || pbf_reserve(d, 190000) != PBF_OK) std::abort();
        without = S().bytes - before;
        pbf_destroy(d);
      }
      const size_t all = S().bytes;
      const long mallocs = S().mallocs;
      expect(step(c, a, n) == PBF_OK && step(c, a, n) == PBF_OK, "step");
      const size_t bytes = (size_t)((n + 63) / 64) * (slots / 8) * 128 * 16;
      expect(kept() == (bytes <= limit), "weights kept up to the limit");
      if (slots == 96) expect(S().mallocs == mallocs, "weights reserved");
      pbf_destroy(c);
      expect(all - S().bytes <= without + limit, "weights within the limit");
    }
  // viscosity switched on after the reservation
  p.list_slots = 0;
  p.flags = 0;
  pbf_ctx* c = nullptr;
  if (pbf_create(&p, &c) != PBF_OK || pbf_reserve(c, 30000) != PBF_OK) std::abort();
  p.flags = PBF_FLAG_VISCOSITY;
  expect(pbf_set_params(c, &p) == PBF_OK, "set_params");
  long mallocs = S().mallocs;
  S().list_need = 96;
  expect(step(c, a, 20000) == PBF_OK && kept(), "step");
  expect(S().mallocs == mallocs, "weights reserved with the parameters");
  pbf_destroy(c);
  // no room for them
  p.flags = 0;
  if (pbf_create(&p, &c) != PBF_OK || pbf_reserve(c, 30000) != PBF_OK) std::abort();
  p.flags = PBF_FLAG_VISCOSITY;
  S().fail_over = 1000;
  expect(pbf_set_params(c, &p) == PBF_OK, "set_params");
  mallocs = S().mallocs;
  for (int k = 0; k < 3; ++k) expect(step(c, a, 20000) == PBF_OK && !kept(), "step without weights");
  expect(S().mallocs == mallocs, "no allocation tried in a step");
  S().fail_over = SIZE_MAX;
  expect(pbf_reserve(c, 30000) == PBF_OK && step(c, a, 20000) == PBF_OK && kept(), "room again");
  pbf_destroy(c);
}

// Threads per workgroup of the PBD passes: 64 for lane pairs by default, what the
// caller sets otherwise; settings read and set again change nothing, and the
// autotuner's default (its choice here: all settings take the same time) is the
// context's.
void pass_blocks() {
  Arrays a(300000);
  pbf_params p = small_params();
  auto block = [&](pbf_ctx* c, int n) {
    S().launches.clear();
    expect(step(c, a, n) == PBF_OK, "step");
    unsigned b = 0;
    for (const Launch& l : S().launches)
      if (l.name == "k_density_lambda2" || l.name == "k_displacement2" || l.name == "k_density_lambda" ||
          l.name == "k_displacement") {
        if (b && b != l.block) violation("two block sizes");
        b = l.block;
      }
    return (int)b;
  };
  for (int smin : {0, -1}) {
    p.stage_min_particles = smin;
    pbf_ctx* c = nullptr;
    if (pbf_create(&p, &c) != PBF_OK) std::abort();
    expect(block(c, 2000) == 64, "the default, lane pairs");
    if (smin == 0) expect(block(c, 280000) == 256, "the default, one lane");
    pbf_tuning t;
    expect(pbf_get_tuning(c, &t) == PBF_OK && t.pass_block == 256 && pbf_set_tuning(c, &t) == PBF_OK, "round trip");
    expect(block(c, 2000) == 64, "the default set again");
    for (int lanes : {0, 2, 1})
      for (int stage : {-1, 1})
        for (int b : {64, 128, 256, 512}) {
          t = pbf_tuning{b, stage, 0, lanes};
          expect(pbf_set_tuning(c, &t) == PBF_OK && block(c, 2000) == b, "a block that the caller set");
        }
    pbf_params q = p;
    q.list_slots = 400;
    expect(pbf_set_tuning(c, &(t = pbf_tuning{256, 0, 0, 0})) == PBF_OK, "the defaults");
    pbf_ctx* wide = nullptr;
    if (pbf_create(&q, &wide) != PBF_OK) std::abort();
    for (int n : {2000, 65536, 80000, 131000, 200000})
      for (int row : {300, 200}) {  // of 400 slots
        S().pairs = (unsigned long long)row * (unsigned)n;
        (void)block(wide, n);  // says how long the rows are
        const bool even = row == 300 && (n == 65536 || n >= 131000);
        expect(block(wide, n) == (even ? 256 : 64), "the default, lane pairs with long lists");
      }
    S().pairs = 0;
    pbf_destroy(wide);
    expect(pbf_set_tuning(c, &t) == PBF_OK && block(c, 2000) == 64, "back to the defaults");
    pbf_tune_report r;
    S().launches.clear();
    expect(pbf_autotune(c, a.x, a.v, nullptr, 1, 2000, 1, nullptr, &r, nullptr) == PBF_OK, "autotune");
    expect(r.best.pass_block == 256 && r.best.stage_min_particles == 0, "its choice");
    bool pair256 = false;
    for (const Launch& l : S().launches) pair256 |= l.name == "k_density_lambda2" && l.block == 256;
    expect(pair256, "it times lane pairs in workgroups of 256");
    expect(block(c, 2000) == 64, "its default is the context's");
    pbf_destroy(c);
  }
}

const std::map<std::string, void (*)()> kScenarios = {
    {"pass_blocks", pass_blocks},
    {"viscosity_weights", viscosity_weights},
    {"blocking_export", blocking_export},
    {"unrecorded_forward", unrecorded_forward},
    {"unknown_capture", unknown_capture},
    {"replays_of_uneven_scenes", replays_of_uneven_scenes},
    {"last_search", last_search},
    {"failed_rollout", failed_rollout},
    {"tape_slots", tape_slots},
    {"list_reservation", list_reservation},
};

}  // namespace

int main(int argc, char** argv) {
  auto it = kScenarios.find(argc > 1 ? argv[1] : "");
  if (it == kScenarios.end()) return std::printf("no such scenario\n"), 2;
  it->second();
  std::printf("%s: %zu launches, %d violations\n", argv[1], S().launches.size(), S().violations);
  return S().violations ? 1 : 0;
}
