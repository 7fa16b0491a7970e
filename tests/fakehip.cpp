// A stand-in for the HIP runtime on the CPU, for tests of the device library's
// host code: device memory is heap memory, launches are queued and logged.
// k_host_copy is carried out (when a wait or a blocking copy drains the queue),
// the other kernels are not.  Loaded with RTLD_GLOBAL before libdrnhip.so, in a
// process of its own, it serves every HIP function that the library calls.
#include <cxxabi.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
std::recursive_mutex mu;
std::map<const void*, std::string> kernels;  // host stub -> demangled device name
std::map<char*, size_t> device, pinned;
std::vector<std::function<void()>> queue;
std::map<void*, size_t> events;  // event -> operations queued before it
std::map<void*, double> event_ms;
size_t done = 0;                 // operations carried out
long fail_after = -1;            // device allocations and blocking copies until one fails, -1: none
int fail_pinned = 0;
thread_local int last_error = 0;
std::string journal;
double clock_ms = 0;
struct Config {
  uint32_t grid[3], block[3];
  size_t shared;
  void* stream;
};
thread_local std::vector<Config> config;

typedef std::lock_guard<std::recursive_mutex> Lock;
void run_to(size_t n) {
  for (; done < n; ++done) queue[done]();
}
void drain() { run_to(queue.size()); }

bool fails() {
  if (fail_after > 0) --fail_after;
  else if (fail_after == 0) {
    fail_after = -1;
    return true;
  }
  return false;
}

bool inside(const std::map<char*, size_t>& m, const void* p) {
  auto it = m.upper_bound((char*)p);
  if (it == m.begin()) return false;
  --it;
  return (char*)p < it->first + it->second;
}
int allocate(std::map<char*, size_t>& m, void** p, size_t n) {
  *p = aligned_alloc(256, (n + 511) / 256 * 256);
  memset(*p, 0xCB, (n + 511) / 256 * 256);
  m[(char*)*p] = n;
  return 0;
}
int release(std::map<char*, size_t>& m, void* p) {
  drain();
  if (p && m.erase((char*)p)) free(p);
  return 0;
}

template <typename E>
void host_copy(E* arr, uint64_t vs, uint64_t n, uint64_t e0, uint32_t cnt, E* host, bool to_host) {
  for (uint64_t q = 0; q < cnt; ++q) {
    const uint64_t v = (e0 + q) / n, l = (e0 + q) % n;
    if (to_host)
      host[q] = arr[v * vs + l];
    else
      arr[v * vs + l] = host[q];
  }
}
}  // namespace

extern "C" {
struct dim3_ {
  uint32_t x, y, z;
};

// the tests' controls
void fake_fail_after(long n) { fail_after = n; }
void fake_fail_pinned(int on) { fail_pinned = on; }
void fake_clear() {
  Lock l(mu);
  journal.clear();
}
const char* fake_journal() {
  static std::string copy;
  Lock l(mu);
  copy = journal;
  return copy.c_str();
}
int fake_is_device(void* p) {
  Lock l(mu);
  return inside(device, p);
}
void* fake_device_alloc(size_t n) {
  Lock l(mu);
  void* p;
  allocate(device, &p, n);
  return p;
}
void* fake_pinned_alloc(size_t n) {
  Lock l(mu);
  void* p;
  allocate(pinned, &p, n);
  return p;
}

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  int st = 0;
  char* d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
  kernels[f] = st == 0 ? d : name;
  free(d);
}
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t shared, void* stream) {
  config.push_back(Config{{g.x, g.y, g.z}, {b.x, b.y, b.z}, shared, stream});
  return 0;
}
int __hipPopCallConfiguration(dim3_* g, dim3_* b, size_t* shared, void** stream) {
  const Config c = config.back();
  config.pop_back();
  *g = dim3_{c.grid[0], c.grid[1], c.grid[2]};
  *b = dim3_{c.block[0], c.block[1], c.block[2]};
  *shared = c.shared;
  *stream = c.stream;
  return 0;
}

// one journal line per launch: its name, its grid and its first two arguments
int hipLaunchKernel(const void* f, dim3_ g, dim3_, void** args, size_t, void*) {
  Lock l(mu);
  const std::string& name = kernels[f];
  const size_t p = name.find("drn::");
  std::string s = p == std::string::npos ? name : name.substr(p + 5);
  s = s.substr(0, s.find('('));
  char line[160];
  uint64_t a0, a1;
  if (s.compare(0, 10, "k_exchange") == 0 || s.compare(0, 4, "k_ls") == 0) {  // a count, then a list
    a0 = *(uint32_t*)args[0];
    a1 = *(uint64_t*)args[1];
  } else {
    a0 = *(uint64_t*)args[0];
    a1 = *(uint64_t*)args[1];
  }
  snprintf(line, sizeof(line), "\t%u\t%llu\t%llu\n", g.x, (unsigned long long)a0, (unsigned long long)a1);
  journal += s + line;
  if (s.compare(0, 11, "k_host_copy") == 0) {
    const bool to_host = s.find("true") != std::string::npos;
    const bool wide64 = s.find("unsigned long") != std::string::npos;
    void *arr = *(void**)args[0], *host = *(void**)args[5];
    const uint64_t vs = *(uint64_t*)args[1], n = *(uint64_t*)args[2], e0 = *(uint64_t*)args[3];
    const uint32_t cnt = *(uint32_t*)args[4];
    queue.push_back([=] {
      if (wide64)
        host_copy((uint64_t*)arr, vs, n, e0, cnt, (uint64_t*)host, to_host);
      else
        host_copy((uint32_t*)arr, vs, n, e0, cnt, (uint32_t*)host, to_host);
    });
  }
  clock_ms += 1.0;
  return 0;
}

int hipGetDeviceCount(int* n) {
  *n = 1;
  return 0;
}
int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int* v, int, int) {
  *v = 256;
  return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 4;
  return 0;
}
const char* hipGetErrorString(int e) { return e ? "injected" : "none"; }
int hipGetLastError() {
  const int e = last_error;
  last_error = 0;
  return e;
}
int hipGetSymbolAddress(void** p, const void*) {
  static char word[64];
  *p = word;
  return 0;
}

int hipMalloc(void** p, size_t n) {
  Lock l(mu);
  *p = nullptr;
  return fails() ? 2 : allocate(device, p, n);
}
int hipFree(void* p) {
  Lock l(mu);
  return release(device, p);
}
int hipHostMalloc(void** p, size_t n, unsigned) {
  Lock l(mu);
  if (fail_pinned) {
    *p = nullptr;
    return last_error = 2;
  }
  return allocate(pinned, p, n);
}
int hipHostFree(void* p) {
  Lock l(mu);
  return release(pinned, p);
}
int hipHostGetDevicePointer(void** d, void* h, unsigned) {
  *d = h;
  return 0;
}
// hipPointerAttribute_t begins with the memory type: unregistered 0, host 1, device 2
int hipPointerGetAttributes(int* a, const void* p) {
  Lock l(mu);
  *a = inside(device, p) ? 2 : inside(pinned, p) ? 1 : 0;
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
  Lock l(mu);
  if (fails()) return 1;
  drain();
  memcpy(d, s, n);
  return 0;
}
// pinned or device memory: when the queue comes to it; pageable: at once
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*) {
  Lock l(mu);
  char line[64];
  snprintf(line, sizeof(line), "memcpy\t%zu\t%d\t0\n", n, kind);
  journal += line;
  queue.push_back([=] { memcpy(d, s, n); });
  if (!(inside(device, d) || inside(pinned, d)) || !(inside(device, s) || inside(pinned, s))) drain();
  return 0;
}
int hipMemset(void* d, int v, size_t n) {
  Lock l(mu);
  drain();
  memset(d, v, n);
  return 0;
}

int hipStreamCreateWithFlags(void** s, unsigned) {
  *s = malloc(1);
  return 0;
}
int hipStreamDestroy(void* s) {
  free(s);
  return 0;
}
int hipStreamSynchronize(void*) {
  Lock l(mu);
  drain();
  return 0;
}
int hipEventCreate(void** e) {
  *e = malloc(1);
  return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e) {
  free(e);
  return 0;
}
int hipEventRecord(void* e, void*) {
  Lock l(mu);
  events[e] = queue.size();
  event_ms[e] = clock_ms;
  return 0;
}
int hipEventSynchronize(void* e) {
  Lock l(mu);
  run_to(events[e]);
  return 0;
}
int hipEventElapsedTime(float* ms, void* a, void* b) {
  *ms = (float)(event_ms[b] - event_ms[a]);
  return 0;
}
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) {
  *g = malloc(1);
  return 0;
}
int hipGraphInstantiate(void** e, void*, void*, char*, size_t) {
  *e = malloc(1);
  return 0;
}
int hipGraphDestroy(void* g) {
  free(g);
  return 0;
}
int hipGraphExecDestroy(void* e) {
  free(e);
  return 0;
}
int hipGraphLaunch(void*, void*) { return 0; }
}
