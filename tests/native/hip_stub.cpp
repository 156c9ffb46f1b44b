// A stand-in for the HIP runtime, for tests of libvk_gemm.so's host code
// without a GPU: one device of 256 CUs, memory from malloc that holds garbage
// (hipMalloc's contents are undefined), and launches that are logged instead of
// run.  Of what kernels do to memory it carries out what the workspace counters
// depend on: the zero fill clears its words, and the padded copies overwrite
// the start of theirs.  Built as a shared library and loaded with RTLD_GLOBAL
// before libvk_gemm.so, whose references then resolve here.
//
// The log has a line per launch: the kernel's name, its grid and block, and
// "counters=clean", "counters=dirty" (words not all zero as the launch begins)
// or "counters=none" (it does not count).
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

struct Dim3 {
  uint32_t x, y, z;
};
struct CallConfig {
  Dim3 grid, block;
  size_t shmem;
  void* stream;
};

std::map<const void*, std::string> g_names;  // host handle -> mangled kernel name
CallConfig g_config;
std::string g_log;
constexpr size_t kCounterBytes = 8192;  // of every counting kernel below, at the workspace's start

template <typename T>
T arg(void** args, int i) {
  T v;
  std::memcpy(&v, args[i], sizeof v);
  return v;
}

bool all_zero(const unsigned char* p, size_t n) {
  for (size_t i = 0; i < n; i++)
    if (p[i]) return false;
  return true;
}

// Where a launch of this kernel finds its counters (null: it does not count):
// argument `split` says how often K is split, argument `counters` where.
const unsigned char* counters_of(const std::string& name, void** args) {
  struct {
    const char* part;
    int split, least, counters;
  } const kinds[] = {{"f16_stream_kernel", 6, 2, 9},
                     {"f32_stream_kernel", 6, 2, 8},
                     {"f32_mfma4_kernel", 7, 1, 12},
                     {"f16_pp16_sk_kernel", 7, 1, 12}};
  for (const auto& k : kinds)
    if (name.find(k.part) != std::string::npos)
      return arg<int>(args, k.split) >= k.least ? arg<const unsigned char*>(args, k.counters) : nullptr;
  return nullptr;
}

}  // namespace

extern "C" {

const char* stub_log() { return g_log.c_str(); }

void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
  g_names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shmem, void* stream) {
  g_config = {grid, block, shmem, stream};
  return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shmem, void** stream) {
  *grid = g_config.grid;
  *block = g_config.block;
  *shmem = g_config.shmem;
  *stream = g_config.stream;
  return 0;
}

int hipGetDevice(int* d) {
  *d = 0;
  return 0;
}
int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int* v, int, int) {
  *v = 256;
  return 0;
}
int hipStreamIsCapturing(void*, int* s) {
  *s = 0;
  return 0;
}
int hipMalloc(void** p, size_t n) {
  *p = std::malloc(n);
  if (!*p) return 2;
  std::memset(*p, 0xab, n < 65536 ? n : 65536);
  return 0;
}
int hipFree(void* p) {
  std::free(p);
  return 0;
}
int hipGetLastError() { return 0; }
int hipGetSymbolAddress(void**, const void*) { return 1; }
int hipFuncSetAttribute(const void*, int, int) { return 0; }

int hipLaunchKernel(const void* host, Dim3 grid, Dim3 block, void** args, size_t, void*) {
  const std::string& name = g_names[host];
  const unsigned char* counters = counters_of(name, args);
  char line[512];
  std::snprintf(line, sizeof line, "%.300s grid=%u,%u,%u block=%u counters=%s\n", name.c_str(), grid.x, grid.y, grid.z,
                block.x, !counters ? "none" : all_zero(counters, kCounterBytes) ? "clean" : "dirty");
  g_log += line;
  if (name.find("zero_fill_kernel") != std::string::npos) {
    std::memset(arg<void*>(args, 0), 0, arg<size_t>(args, 1) * 4);
  } else if (name.find("repitch_kernel") != std::string::npos) {
    const size_t bytes = (size_t)arg<int>(args, 4) * (size_t)arg<int>(args, 5) * 2;
    std::memset(arg<void*>(args, 1), 0xcd, bytes < 65536 ? bytes : 65536);
  }
  return 0;
}

}  // extern "C"
