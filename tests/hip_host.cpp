// A stand-in for the HIP runtime on host memory, for tests of the library's
// host code without a GPU: allocations, copies, streams and events behave (each
// of them belongs to a device), kernels are recorded by name and do nothing,
// except the library's plain copy kernel. Loaded with RTLD_GLOBAL before the
// library, so that the library's HIP calls bind to it.
#include <cxxabi.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>

namespace {

struct Owned { int device; };          // a stream or an event
struct Dim { unsigned x, y, z; };

enum { kOk = 0, kInvalidHandle = 400 };

thread_local int device = 0, lastError = 0;
thread_local long newBudget = -1;      // operator new calls until one fails; < 0: never
thread_local Dim callGrid, callBlock;
thread_local size_t callShared;
thread_local void *callStream;
std::mutex mutex;
std::map<const void *, std::string> &names() { static std::map<const void *, std::string> m; return m; }
std::string &launches() { static std::string s; return s; }

int note(int e)
{
  if (e) lastError = e;
  return e;
}

int allocate(void **p, size_t n)
{
  *p = std::calloc(n ? n : 1, 1);
  return *p ? kOk : note(2);
}

int make(Owned **o)
{
  *o = static_cast<Owned *>(std::malloc(sizeof(Owned)));
  (*o)->device = device;
  return kOk;
}

}  // namespace

void *operator new(size_t n)
{
  if (newBudget >= 0 && newBudget-- == 0) throw std::bad_alloc();
  void *p = std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {

// ---- for the tests
void rt_set_device(int d) { device = d; }
int rt_device() { return device; }
void rt_fail_new(long after) { newBudget = after; }
void rt_clear()
{
  std::lock_guard<std::mutex> lock(mutex);
  launches().clear();
}
// one line per launch: name, grid x
const char *rt_launches()
{
  std::lock_guard<std::mutex> lock(mutex);
  return launches().c_str();
}

// ---- the runtime
int hipGetDevice(int *d) { *d = device; return kOk; }
int hipSetDevice(int d) { device = d; return kOk; }
const char *hipGetErrorString(int) { return "stand-in runtime error"; }
int hipGetLastError()
{
  const int e = lastError;
  lastError = kOk;
  return e;
}
int hipMalloc(void **p, size_t n) { return allocate(p, n); }
int hipFree(void *p) { std::free(p); return kOk; }
int hipHostMalloc(void **p, size_t n, unsigned) { return allocate(p, n); }
int hipHostFree(void *p) { std::free(p); return kOk; }
int hipMemcpy(void *d, const void *s, size_t n, int) { std::memcpy(d, s, n); return kOk; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, Owned *) { std::memcpy(d, s, n); return kOk; }
int hipMemset(void *d, int v, size_t n) { std::memset(d, v, n); return kOk; }
int hipGetSymbolAddress(void **p, const void *)
{
  static void *scratch = std::calloc(size_t(64) << 20, 1);
  *p = scratch;
  return kOk;
}
int hipStreamCreate(Owned **s) { return make(s); }
int hipStreamDestroy(Owned *s) { std::free(s); return kOk; }
int hipStreamSynchronize(Owned *) { return kOk; }
int hipStreamWaitEvent(Owned *, Owned *, unsigned) { return kOk; }
int hipEventCreate(Owned **e) { return make(e); }
int hipEventCreateWithFlags(Owned **e, unsigned) { return make(e); }
int hipEventDestroy(Owned *e) { std::free(e); return kOk; }
// an event is recorded on a stream of its own device only
int hipEventRecord(Owned *e, Owned *s) { return note(e->device == s->device ? kOk : kInvalidHandle); }
int hipEventSynchronize(Owned *) { return kOk; }
int hipEventElapsedTime(float *ms, Owned *, Owned *) { *ms = 0.0f; return kOk; }
int hipStreamBeginCapture(Owned *, int) { return kOk; }
int hipStreamEndCapture(Owned *s, void **g) { *g = s; return kOk; }
int hipGraphInstantiate(void **x, void *g, void *, char *, size_t) { *x = g; return kOk; }
int hipGraphDestroy(void *) { return kOk; }
int hipGraphExecDestroy(void *) { return kOk; }
int hipGraphLaunch(void *, Owned *) { return kOk; }

void **__hipRegisterFatBinary(const void *)
{
  static void *handle;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
  int status = 0;
  char *d = abi::__cxa_demangle(name, nullptr, nullptr, &status);
  names()[f] = status == 0 ? d : name;
  std::free(d);
}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t shared, void *stream)
{
  callGrid = grid; callBlock = block; callShared = shared; callStream = stream;
  return kOk;
}
int __hipPopCallConfiguration(Dim *grid, Dim *block, size_t *shared, void **stream)
{
  *grid = callGrid; *block = callBlock; *shared = callShared; *stream = callStream;
  return kOk;
}
// a kernel is launched on a stream of the current device only
int hipLaunchKernel(const void *f, Dim grid, Dim, void **args, size_t, Owned *s)
{
  if (s->device != device) return note(kInvalidHandle);
  const std::string &name = names()[f];
  if (name.find("store_kernel(") != std::string::npos)
    std::memcpy(*(double **) args[0], *(const double **) args[1], *(size_t *) args[2] * sizeof(double));
  std::lock_guard<std::mutex> lock(mutex);
  const std::string space = "(anonymous namespace)::";
  const size_t at = name.find(space), from = at == std::string::npos ? 0 : at + space.size();
  launches() += name.substr(from, name.find('(', from) - from) + " " + std::to_string(grid.x) + "\n";
  return kOk;
}

}  // extern "C"
