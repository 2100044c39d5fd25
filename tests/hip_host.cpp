// The part of the HIP runtime the library calls, on host memory: for tests of
// its host code without a GPU.  Device memory is host memory with a limit on
// the bytes held at a time; an error stays to be read by hipGetLastError, as
// in the real runtime.  Kernels do not run, with two exceptions:
//   k_gmres_ctl, op 0   marks every instance converged, so that a solve ends;
//   k_mlp_pass          checks the buffers of a gradient's arguments: each has
//                       to lie in live memory with room for all of its rows.
// A captured graph keeps its launches and repeats them when it is launched.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "glhip_dev.hpp"
#include "mlp_dev.hpp"

namespace {

std::map<const char *, size_t> live;  // address -> bytes
size_t used = 0, limit = SIZE_MAX;
hipError_t last = hipSuccess;
std::map<const void *, std::string> kernels;
std::map<std::string, long long> launches;
long long bad = 0, captures = 0;
bool capturing = false;
using Graph = std::vector<std::function<void()>>;
Graph recorded;
struct Config {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
} config;

hipError_t ret(hipError_t e)
{
  if (e != hipSuccess) last = e;
  return e;
}

bool holds(const void *p, size_t n)
{
  auto it = live.upper_bound((const char *)p);
  if (it == live.begin()) return false;
  --it;
  return (const char *)p + n <= it->first + it->second;
}

void run_pass(const glh::mlp::PassArgs &A)
{
  if (!A.lpart) return;  // inference
  const size_t rows = A.n_rows, W = A.width;
  bool ok = holds(A.X, 24) && holds(A.T, sizeof(float) * A.n_out) && holds(A.H[0], rows * 2 * A.F * 2);
  for (int l = 0; l < A.depth; ++l)
    ok = ok && holds(A.H[l + 1], rows * W * 2) && holds(A.Z[l], rows * W * 4) && holds(A.dZ[l], rows * W * 2);
  ok = ok && holds(A.dZ[A.depth], rows * glh::mlp::MLP_OUTP * 2);
  if (!ok) ++bad;
}

template <typename T>
void run_ctl(const glh::GmresCtl<T> &C, int op)
{
  if (op != 0) return;
  for (int i = 0; i < C.S; ++i) C.conv[i] = 1;
}

}  // namespace

extern "C" {

// ------------------------------------------------------------ for the tests
void hh_limit(size_t bytes) { limit = bytes; }
size_t hh_used() { return used; }
long long hh_bad() { return bad; }
long long hh_captures() { return captures; }
long long hh_launches(const char *name)
{
  long long n = 0;
  for (auto &k : launches)
    if (k.first.find(name) != std::string::npos) n += k.second;
  return n;
}

// --------------------------------------------------------------- the runtime
hipError_t hipMalloc(void **p, size_t n)
{
  *p = nullptr;
  if (used + n > limit) return ret(hipErrorOutOfMemory);
  *p = std::calloc(n, 1);
  live[(const char *)*p] = n;
  used += n;
  return hipSuccess;
}
hipError_t hipFree(void *p)
{
  if (!p) return hipSuccess;
  auto it = live.find((const char *)p);
  if (it == live.end()) return ret(hipErrorInvalidValue);
  used -= it->second;
  live.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return (*p = std::calloc(n, 1)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p)
{
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *)
{
  static std::vector<double> scratch(glh::SCRATCH_DOUBLES);
  *p = scratch.data();
  return hipSuccess;
}
hipError_t hipGetLastError()
{
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetDeviceCount(int *n)
{
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
  *s = (hipStream_t)std::malloc(1);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
  std::free((void *)s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
  *e = (hipEvent_t)std::malloc(1);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e)
{
  std::free((void *)e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
  *ms = 1.f;
  return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
  capturing = true;
  ++captures;
  recorded.clear();
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
  capturing = false;
  *g = (hipGraph_t) new Graph(recorded);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g)
{
  delete (Graph *)g;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t)
{
  *e = (hipGraphExec_t) new Graph(*(Graph *)g);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e)
{
  delete (Graph *)e;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t)
{
  for (auto &f : *(Graph *)e) f();
  return hipSuccess;
}

void **__hipRegisterFatBinary(const void *)
{
  static void *one;
  return &one;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *)
{
  kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s)
{
  config = Config{g, b, sh, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *s)
{
  *g = config.grid;
  *b = config.block;
  *sh = config.shared;
  *s = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3, void **args, size_t, hipStream_t)
{
  if (g.x == 0 || g.y == 0 || g.z == 0) return ret(hipErrorInvalidValue);
  const std::string name = kernels[f];
  std::function<void()> run = [name] { ++launches[name]; };
  if (name.find("k_mlp_pass") != std::string::npos) {
    const auto A = *(const glh::mlp::PassArgs *)args[0];
    run = [name, A] {
      ++launches[name];
      run_pass(A);
    };
  } else if (name.find("k_gmres_ctl") != std::string::npos) {
    const auto C = *(const glh::GmresCtl<double> *)args[0];  // (the fields used are the same in FP32)
    const int op = *(const int *)args[1];
    run = [name, C, op] {
      ++launches[name];
      run_ctl(C, op);
    };
  }
  if (capturing) recorded.push_back(run);
  else run();
  return hipSuccess;
}

}  // extern "C"
