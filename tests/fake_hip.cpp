// A HIP runtime without a device, preloaded in front of the real one by
// fakehip.py, so that the library's host code runs on the CPU.  Device memory
// is host memory; copies are made; of the kernels only k_fill is carried out
// (after a look at its range), the others are written to the log.
//   FAKE_HIP_LOG      the log: one line per launch, symbol upload and fault
//   FAKE_HIP_ELAPSED  what hipEventElapsedTime returns, in turn (ms)
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Dim3 { uint32_t x, y, z; };
std::map<const void*, std::string> names;
std::map<char*, size_t> blocks;
struct Config { Dim3 g, b; size_t sh; void* st; };
std::vector<Config> configs;
FILE* out() {
  static FILE* f = [] {
    const char* p = std::getenv("FAKE_HIP_LOG");
    FILE* o = p ? std::fopen(p, "w") : stderr;
    setvbuf(o, nullptr, _IOLBF, 1 << 12);
    return o;
  }();
  return f;
}
int take(void** p, size_t n) {
  *p = std::calloc(n ? n : 1, 1);
  if (*p) blocks[(char*)*p] = n;
  return *p ? 0 : 2;
}
int drop(void* p) {
  if (p && !blocks.erase((char*)p)) std::fprintf(out(), "fault free of an address that is no allocation\n");
  std::free(p);
  return 0;
}
void fill(const Dim3& g, const Dim3& b, void** args) {
  char* p = *(char**)args[0];
  const long n = *(long*)args[1], lanes = (long)g.x * b.x, m = n < lanes ? n : lanes;
  const double v = *(double*)args[2];
  auto it = blocks.upper_bound(p);
  if (it == blocks.begin()) { std::fprintf(out(), "fault fill outside all allocations\n"); return; }
  --it;
  const size_t off = p - it->first;
  if (off + 8 * m > it->second) {
    std::fprintf(out(), "fault fill of %ld doubles at byte %zu of %zu\n", m, off, it->second);
    return;
  }
  if (lanes < n) std::fprintf(out(), "fault grid of %ld lanes for a fill of %ld\n", lanes, n);
  std::fprintf(out(), "fill %zu %ld %zu\n", off, n, it->second);
  for (long k = 0; k < m; k++) ((double*)p)[k] = v;
}
}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  names[f] = name;
}
void __hipRegisterVar(void**, void* v, char*, char* name, int, size_t, int, int) { names[v] = name; }
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t sh, void* st) {
  configs.push_back({g, b, sh, st});
  return 0;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* sh, void** st) {
  const Config c = configs.back();
  configs.pop_back();
  *g = c.g; *b = c.b; *sh = c.sh; *st = c.st;
  return 0;
}
int hipLaunchKernel(const void* f, Dim3 g, Dim3 b, void** args, size_t, void*) {
  const std::string& n = names[f];
  std::fprintf(out(), "launch %s %u %u %u %u\n", n.c_str(), g.x, g.y, g.z, b.x);
  if (n == "_Z6k_fillPdld") fill(g, b, args);
  return 0;
}
int hipMalloc(void** p, size_t n) { return take(p, n); }
int hipFree(void* p) { return drop(p); }
int hipHostMalloc(void** p, size_t n, unsigned) { return take(p, n); }
int hipHostFree(void* p) { return drop(p); }
int hipMemcpy(void* d, const void* s, size_t n, int) { std::memmove(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { std::memmove(d, s, n); return 0; }
int hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void*) { std::memset(d, v, n); return 0; }
int hipMemcpyToSymbol(const void* sym, const void* s, size_t n, size_t, int) {
  std::fprintf(out(), "symbol %s %zu %d\n", names[sym].c_str(), n, *(const int*)s);
  return 0;
}
int hipMemcpyToSymbolAsync(const void* sym, const void* s, size_t n, size_t o, int k, void*) {
  return hipMemcpyToSymbol(sym, s, n, o, k);
}
int hipEventElapsedTime(float* ms, void*, void*) {
  static std::vector<float> v = [] {
    std::vector<float> w;
    for (const char* p = std::getenv("FAKE_HIP_ELAPSED"); p && *p;) {
      char* e;
      w.push_back(std::strtof(p, &e));
      p = *e ? e + 1 : e;
    }
    if (w.empty()) w.push_back(1.f);
    return w;
  }();
  static size_t k = 0;
  *ms = v[k++ % v.size()];
  return 0;
}
static int handle(void** h) { *h = (void*)(uintptr_t)0x10; return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { return handle(s); }
int hipEventCreate(void** e) { return handle(e); }
int hipEventCreateWithFlags(void** e, unsigned) { return handle(e); }
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) { return handle(g); }
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) { return handle(x); }
int hipGraphLaunch(void*, void*) { std::fprintf(out(), "graph\n"); return 0; }
int hipGraphExecDestroy(void*) { return 0; }
int hipGraphDestroy(void*) { return 0; }
int hipStreamDestroy(void*) { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipEventDestroy(void*) { return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int) { return "fake"; }
}
