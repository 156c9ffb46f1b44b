// vk_gemm.hip -- the C ABI of libvk_gemm.so: version registry, argument
// validation, library-managed workspaces and dispatch.
//
// Stands in for the compile-time dispatch of the reference
// (results/naive_cycle4/include/playground/matmul.hpp:11-23, one template
// specialisation per (dtype, version), picked by -DMATMUL_VERSION in
// results/naive_fable_cycle2/src/CMakeLists.txt:29-50 and :66-70).  Here all
// versions live in one library and are picked at run time by id; an unknown
// id is an error code instead of a configure-time FATAL_ERROR
// (CMakeLists.txt:35-40).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <algorithm>
#include <cstring>
#include <mutex>

#include "vk_device.hpp"
#include "vk_gemm.h"
#include "vk_internal.hpp"

// Workspace of vk_gemm_noalloc: split-K / split-tail partials and their
// arrival counters.  Each device that loads this library holds its own copy
// until the process ends.  In host code this name is only a stand-in for the
// symbol: the device address of a device's copy comes from
// hipGetSymbolAddress (scratch_of below), and only that address is handed to
// kernels.
static __device__ __align__(256) unsigned char scratch[VK_GEMM_SCRATCH_BYTES];

namespace vk {
namespace {

// The registered versions, in a fixed array: a lookup never allocates.
constexpr int kMaxEntries = 48;
struct Registry {
  KernelEntry e[kMaxEntries];
  int n = 0;
  const KernelEntry* begin() const { return e; }
  const KernelEntry* end() const { return e + n; }
};
Registry& registry() {
  static Registry r;
  return r;
}

std::once_flag g_init_once;

void init_registry() {
  std::call_once(g_init_once, [] {
    register_f16_any();
    register_f16_dma();
    register_f16_skinny();
    register_f16_pingpong();
    register_f16_pp128();
    register_f16_skinny_sk();
    register_f16_skinny_wk();
    register_f16_padded();
    register_f32_valu();
    register_f32_mfma();
  });
}

const KernelEntry* find(int version, vk_dtype in) {
  init_registry();
  for (const auto& e : registry())
    if (e.version == version && e.in_dtype == in) return &e;
  return nullptr;
}

size_t dtype_size(vk_dtype d) { return d == VK_DTYPE_F16 ? 2 : 4; }

}  // namespace

const KernelEntry* find_registered(int version, vk_dtype in) { return find(version, in); }

namespace {

struct DeviceState {
  void* ws = nullptr;
  size_t ws_bytes = 0;
  const KernelEntry* ws_entry = nullptr;  // whose launch used the library workspace last (none: unknown)
  int ws_kind = 0;                        // and in which of its layouts
  int num_cus = 0;
  void* scratch = nullptr;  // this device's copy of `scratch` (vk_gemm_noalloc)
};
// One entry per device id, fixed in size: looking a device up never
// allocates (host or device memory).
constexpr int kMaxDevices = 64;
std::mutex g_dev_mutex;
DeviceState g_dev[kMaxDevices];

hipError_t device_state(int dev, DeviceState** out) {
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(g_dev_mutex);
  DeviceState& s = g_dev[dev];
  if (s.num_cus == 0) {
    int cus = 0;
    hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    s.num_cus = cus;
  }
  *out = &s;
  return hipSuccess;
}

// Compute units of the current device (plans depend on them); with no device
// to ask, an MI355X's 256 are assumed.
int cus_or_default() {
  int dev = 0;
  DeviceState* ds = nullptr;
  return hipGetDevice(&dev) == hipSuccess && device_state(dev, &ds) == hipSuccess ? ds->num_cus : 256;
}

// Device address of this device's copy of `scratch`, looked up once per
// device with that device current.
hipError_t scratch_of(int dev, void** out) {
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(g_dev_mutex);
  DeviceState& s = g_dev[dev];
  if (!s.scratch) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    s.scratch = p;
  }
  *out = s.scratch;
  return hipSuccess;
}

// C := 0 for k == 0 (beta = 0 and an empty sum).  A kernel, not
// hipMemsetAsync, so the call stays safe inside stream capture.
__global__ void zero_fill_kernel(uint32_t* __restrict__ p, size_t words) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < words; i += stride) p[i] = 0u;
}
__global__ void zero_fill_u16_kernel(uint16_t* __restrict__ p, size_t count) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < count; i += stride) p[i] = 0u;
}

hipError_t zero_output(void* C, size_t count, vk_dtype out, hipStream_t s) {
  const unsigned blocks = 1024;
  if (out == VK_DTYPE_F32 || (count % 2 == 0 && ((uintptr_t)C & 3u) == 0)) {
    const size_t words = out == VK_DTYPE_F32 ? count : count / 2;
    hipLaunchKernelGGL(zero_fill_kernel, dim3(blocks), dim3(256), 0, s, (uint32_t*)C, words);
  } else {
    hipLaunchKernelGGL(zero_fill_u16_kernel, dim3(blocks), dim3(256), 0, s, (uint16_t*)C, count);
  }
  return hipGetLastError();
}

}  // namespace

hipError_t zero_words(void* p, size_t words, hipStream_t s) {
  const unsigned blocks = (unsigned)std::min<size_t>(1024, (words + 255) / 256);
  hipLaunchKernelGGL(zero_fill_kernel, dim3(blocks ? blocks : 1), dim3(256), 0, s, (uint32_t*)p, words);
  return hipGetLastError();
}

namespace {

int validate(const KernelEntry* e, vk_dtype out, size_t m, size_t n, size_t k, const void* A,
             const void* B, const void* C) {
  if (!e) return VK_ERR_VERSION;
  if (out != VK_DTYPE_F16 && out != VK_DTYPE_F32) return VK_ERR_DTYPE;
  if (!(e->caps.out_dtype_mask & (1 << out))) return VK_ERR_DTYPE;
  const size_t lim = 0x7fffffffu;
  if (m > lim || n > lim || k > lim) return VK_ERR_RANGE;
  if (m == 0 || n == 0) return VK_OK;  // nothing to write
  if (!C) return VK_ERR_NULL;
  if (k == 0) return VK_OK;            // C := 0, A and B unused
  if (!A || !B) return VK_ERR_NULL;
  const vk_caps& c = e->caps;
  if (m % c.div_m || n % c.div_n || k % c.div_k) return VK_ERR_SHAPE;
  if (m > c.max_m) return VK_ERR_SHAPE;
  if (e->shape_ok && !e->shape_ok(m, n, k)) return VK_ERR_SHAPE;
  const uintptr_t al = c.align_bytes ? c.align_bytes : 1;
  if (((uintptr_t)A % al) || ((uintptr_t)B % al) || ((uintptr_t)C % al)) return VK_ERR_ALIGN;
  return VK_OK;
}

int run(int version, vk_dtype in, vk_dtype out, size_t m, size_t n, size_t k, const void* A,
        const void* B, void* C, void* ws, size_t ws_bytes, bool library_ws, void* stream) {
  const KernelEntry* e = find(version, in);
  int st = validate(e, out, m, n, k, A, B, C);
  if (st != VK_OK) return st;
  if (m == 0 || n == 0) return VK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (k == 0) return zero_output(C, m * n, out, s) == hipSuccess ? VK_OK : VK_ERR_HIP;

  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return VK_ERR_HIP;
  DeviceState* ds = nullptr;
  if (device_state(dev, &ds) != hipSuccess) return VK_ERR_HIP;

  const size_t need = e->workspace ? e->workspace(m, n, k, ds->num_cus) : 0;
  bool ws_clean = false;
  int kind = 0;
  bool owns_ws = false;  // this call reads or writes the library workspace
  if (need > 0) {
    if (library_ws) {
      // A graph captured now would keep this workspace's address, which a
      // later call may free and reallocate, and would replay the counter
      // state decided here: under capture the library workspace is refused,
      // and vk_gemm_ws (caller workspace) is the capture-safe form.
      hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing(s, &cs) != hipSuccess) return VK_ERR_HIP;
      if (cs != hipStreamCaptureStatusNone) return VK_ERR_WORKSPACE;
      std::lock_guard<std::mutex> lk(g_dev_mutex);
      if (ds->ws_bytes < need) {
        if (ds->ws) {
          if (hipFree(ds->ws) != hipSuccess) return VK_ERR_HIP;  // synchronises the device
          ds->ws = nullptr;
          ds->ws_bytes = 0;
        }
        ds->ws_entry = nullptr;
        if (hipMalloc(&ds->ws, need) != hipSuccess) return VK_ERR_HIP;
        ds->ws_bytes = need;
      }
      ws = ds->ws;
      ws_bytes = ds->ws_bytes;
      kind = e->workspace_kind ? e->workspace_kind(m, n, k, ds->num_cus) : 0;
      if (kind != kWorkspaceUntouched) {
        ws_clean = ds->ws_entry == e && ds->ws_kind == kind;
        // Until this launch is known to have been enqueued, the counters count
        // as unknown: a failed launch must not leave the next call skipping the
        // clear.
        ds->ws_entry = nullptr;
        owns_ws = true;
      }
    } else if (!ws || ws_bytes < need) {
      return VK_ERR_WORKSPACE;
    }
  }

  GemmArgs a;
  a.m = m;
  a.n = n;
  a.k = k;
  a.A = A;
  a.B = B;
  a.C = C;
  a.out_dtype = out;
  a.workspace = ws;
  a.workspace_bytes = ws_bytes;
  a.workspace_clean = ws_clean;
  a.stream = s;
  a.device = dev;
  a.num_cus = ds->num_cus;
  a.ldc = 0;
  if (e->launch(a) != hipSuccess) return VK_ERR_HIP;
  if (owns_ws) {
    // The kernels of a version leave the counters they use at zero, so the
    // next call of the same version may skip clearing them.
    std::lock_guard<std::mutex> lk(g_dev_mutex);
    if (ds->ws == ws) {
      ds->ws_entry = e;
      ds->ws_kind = kind;
    }
  }
  return VK_OK;
}

// ---- the version for a shape ----
// The fastest version that accepts this shape (checked with vk_gemm_check
// on 4 KiB-aligned placeholder addresses; nothing is launched): for fp16
// the skinny kernels up to M = 128 (version 14 where it suits, else version
// 8; version 4 up to 64) and version 8 from 129 to 255 rows where version 11
// does not suit, then the
// 128 x 128 tiles of version 11 where they suit the grid, then the 256x256 kernels
// (fastest first; version 10 takes shapes off the 256 x 256 x 64 grid
// whose N and K are multiples of 8), then version 15 (N or K off the multiples
// of 8, from M N K = 2^24 on), then the any-shape kernel.  Version 11
// is taken, with T its 128 x 128 tiles on C compute units:
//   * on the 256 x 256 x 64 grid, where T <= C (one wave; with 2 T <= C it
//   splits K over the idle CUs itself).  Measured on MI355X, us per
//   launch against version 9's split tail: 1024 x 4096 x 4096 33.6
//   against 46.2 (version 7: 64.5), 1024 x 1024 x 8192 29.1 against
//   43.9, 512 x 512 x 8192 19.7 against 41.7, 512 x 4096 x 4096 24.7
//   against 35.1; beyond one wave 1536 x 4096 x 4096 (T = 384) took 58.7
//   against 50.6;
//   * off it, where T <= 3 C / 2 (version 10, whose split pieces do not stay
//   on one XCD there and whose edge tiles are twice as wide, measured
//   slower on every such shape: 1000 x 1000 x 1000 23.0 us against 9.8,
//   2000 x 3000 x 1000 (T = 384) 25.2 against 21.2, 1000 x 1000 x 4000
//   (T = 64) 36.6 against 23.0).
// From M = 129 version 11 also beats the skinny split-K version 8 wherever
// it is taken (us per launch, one box: 192 x 4096 x 4096 22.5 against
// 30.2, 192 x 8192 x 8192 39.8 against 46.0, 192 x 14336 x 4096 32.9
// against 42.4, 256 x 8192 x 8192 39.8 against 55.6; another box, v11
// against v8 at N x K = 4096 x 4096 / 4096 x 8192 / 8192 x 4096 / 8192 x
// 8192 / 14336 x 4096 / 4096 x 14336: M = 136 21.1 / 27.1 / 24.1 / 37.1 /
// 28.9 / 37.9 against 25.9 / 31.5 / 27.0 / 37.4 / 32.8 / 39.4; M = 160
// 21.1 / 27.8 / 24.5 / 39.0 / 31.1 / 39.5 against 26.2 / 31.9 / 27.6 /
// 38.5 / 33.8 / 39.8; M = 184 21.9 / 28.3 / 24.8 / 39.8 / 32.6 / 38.9
// against 30.3 / 38.7 / 32.5 / 45.6 / 41.1 / 46.9).
// Version 14 (K split over the waves of a workgroup, 64-column blocks) is
// taken up to M = 64 where 2048 < N <= 4096 (but not up to M = 32 with
// K > 12288) and up to M = 8 where 1024 < N <= 2048 and K <= 8192, and
// from M = 65 to 128 where N <= 4096 and K <= 8192.  Against version 8
// (us per launch, one box): M = 72 / 96 / 128 at N x K = 4096 x 6144
// 16.8 / 19.3 / 22.9 against 20.2 / 22.6 / 25.0, at 4096 x 8192 19.2 /
// 22.2 / 26.6 against 22.7 / 24.3 / 27.7, at 2048 x 8192 16.5 / 18.2 /
// 21.5 against 18.9 / 20.5 / 24.1, at 3072 x 6144 17.4 / 19.5 / 23.1
// against 18.3 / 20.0 / 22.9; at K = 11264 mixed (4096 columns: 23.7 /
// 27.9 / 34.2 against 26.7 / 28.3 / 31.3); M = 1 / 4 / 8 at N x K = 1536 x
// 8192 8.6 / 9.0 / 9.2 against 10.0 / 10.2 / 10.3, 2048 x 8192 9.6 / 10.1
// / 10.6 against 10.4 / 10.7 / 10.7, 2048 x 4096 8.7 / 9.0 / 9.2 against
// 8.9 / 9.1 / 9.2, but 2048 x 14336 16.0 / 16.5 / 16.4 against 15.7 /
// 15.9 / 16.0 and M = 16 at N = 2048 (K = 4096 / 8192 / 14336: 9.3 / 11.1
// / 16.4 against 9.1 / 10.8 / 16.0).  At K = 14336, N = 4096 version 8 is faster up
// to M = 32 (us per launch against version 14, 2 rounds on one box: M = 1
// 22.3 against 22.6, 16 22.5 against 23.6, 32 23.8 against 24.1; N =
// 3072, M = 16 19.1 against 20.1; N = 2560, M = 16 17.8 against 18.0) and
// version 14 from M = 48 (26.1 against 25.4; M = 64 28.4 against 27.2);
// at K = 11264 they are within 2 % (M = 16 19.4 / 19.8, M = 1 19.1 /
// 18.9) and at K = 8192 version 14 wins (M = 1 16.4 / 15.5, 16 16.9 /
// 16.0, 32 18.4 / 16.5).  Measured on MI355X
// against version 8 (us per launch, one box, M = 1 / 16 / 64 / 128):
// N = 4096, K = 4096 8.1 / 9.1 / 14.4 / 18.4 against 9.5 / 9.9 / 16.2 /
// 21.8; N = 3072, K = 2048 7.2 / 7.6 / 11.6 / 14.4 against 8.1 / 8.3 /
// 13.5 / 20.3; N = 4096, K = 14336 22.1 / 22.9 / 27.1 / 39.0 against
// 22.2 / 22.5 / 28.5 / 35.3; N = 2048, K = 8192 at M = 128 21.0 against
// 23.4, at M = 16 10.2 against 10.5; N = 1024, K = 2048 8.3 / 8.6 / 12.4 /
// 15.9 against 6.7 / 7.0 / 10.9 / 17.6.  Every 64 columns re-read all of
// A (at M = 128 twice B's bytes), which costs it at large M and K; from
// N = 5120 its power-of-two K split also leaves CUs idle (80 column blocks
// x 2): 128 x 8192 x 8192 41.8 against 32.9.
// The split-tail version 9 comes first among the 256x256 kernels only where
// its schedule splits tiles on this device (it then needs a workspace);
// elsewhere it would run version 7's whole tiles.  The reference picks
// versions at build time only (CMakeLists.txt MATMUL_VERSION); this is a
// convenience.
int pick(vk_dtype in, vk_dtype out, size_t m, size_t n, size_t k) {
  static constexpr int kOrderF16[] = {14, 8, 4, 11, 9, 7, 10, 6, 5, 3, 2, 15, 1};
  static constexpr int kOrderF32[] = {2, 3, 1};
  const void* at = reinterpret_cast<const void*>(uintptr_t{4096});
  auto takes = [&](int v) { return validate(find(v, in), out, m, n, k, at, at, at) == VK_OK; };
  if (in != VK_DTYPE_F16) {
    for (int v : kOrderF32)
      if (takes(v)) return v;
    return VK_ERR_SHAPE;
  }
  const size_t lim = 0x7fffffffu;  // no version takes more (and the counts below stay within 64 bits)
  if (m > lim || n > lim || k > lim) return VK_ERR_SHAPE;

  const int cus = cus_or_default();
  const size_t tiles = (m + 127) / 128 * ((n + 127) / 128);
  const bool v11_suits =
      m % 256 == 0 && n % 256 == 0 && k % 64 == 0 ? tiles <= (size_t)cus : 2 * tiles <= 3 * (size_t)cus;
  bool v14_suits = m <= 128 && n <= 4096 && !(m <= 32 && k > 12288);
  if (v14_suits) v14_suits = m <= 64 ? n > 2048 || (m <= 8 && n > 1024 && k <= 8192) : k <= 8192;
  const bool v15_suits = (unsigned __int128)m * n * k >= (1u << 24);  // below: version 1

  for (int v : kOrderF16) {
    if (v == 14 && !v14_suits) continue;
    if (v == 8 && m > 128 && v11_suits && takes(11)) continue;
    if (v == 11 && !v11_suits) continue;
    if (v == 15 && !v15_suits) continue;
    if (!takes(v)) continue;
    if (v == 9 && find(9, in)->workspace(m, n, k, cus) == 0) continue;
    return v;
  }
  return VK_ERR_SHAPE;
}

}  // namespace

void register_kernel(const KernelEntry& e) {
  Registry& r = registry();
  if (r.n < kMaxEntries) r.e[r.n++] = e;
}

}  // namespace vk

extern "C" {

int vk_gemm(int version, vk_dtype in_dtype, vk_dtype out_dtype, size_t m, size_t n, size_t k,
            const void* A, const void* B, void* C, void* stream) {
  return vk::run(version, in_dtype, out_dtype, m, n, k, A, B, C, nullptr, 0, true, stream);
}

int vk_gemm_ws(int version, vk_dtype in_dtype, vk_dtype out_dtype, size_t m, size_t n, size_t k,
               const void* A, const void* B, void* C, void* workspace, size_t workspace_bytes,
               void* stream) {
  return vk::run(version, in_dtype, out_dtype, m, n, k, A, B, C, workspace, workspace_bytes, false,
                 stream);
}

int vk_gemm_noalloc(int version, vk_dtype in_dtype, vk_dtype out_dtype, size_t m, size_t n, size_t k,
                    const void* A, const void* B, void* C, void* stream) {
  const int st = vk::validate(vk::find(version, in_dtype), out_dtype, m, n, k, A, B, C);
  if (st != VK_OK || m == 0 || n == 0 || k == 0)
    return st != VK_OK ? st : vk::run(version, in_dtype, out_dtype, m, n, k, A, B, C, nullptr, 0, false, stream);
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return VK_ERR_HIP;
  void* sp = nullptr;
  if (vk::scratch_of(dev, &sp) != hipSuccess) return VK_ERR_HIP;
  // A caller workspace of VK_GEMM_SCRATCH_BYTES: a plan that needs more is
  // refused with VK_ERR_WORKSPACE, and the counters are cleared by a kernel
  // in every call (the scratch keeps whatever the last call left).
  return vk::run(version, in_dtype, out_dtype, m, n, k, A, B, C, sp, VK_GEMM_SCRATCH_BYTES, false, stream);
}

size_t vk_gemm_workspace_bytes(int version, vk_dtype in_dtype, size_t m, size_t n, size_t k) {
  const vk::KernelEntry* e = vk::find(version, in_dtype);
  if (!e || !e->workspace) return 0;
  return e->workspace(m, n, k, vk::cus_or_default());
}

int vk_gemm_pick(vk_dtype in_dtype, vk_dtype out_dtype, size_t m, size_t n, size_t k) {
  return vk::pick(in_dtype, out_dtype, m, n, k);
}

const char* vk_gemm_name(int version, vk_dtype in_dtype) {
  const vk::KernelEntry* e = vk::find(version, in_dtype);
  return e ? e->name : nullptr;
}

int vk_gemm_query(int version, vk_dtype in_dtype, vk_caps* caps) {
  const vk::KernelEntry* e = vk::find(version, in_dtype);
  if (!e) return VK_ERR_VERSION;
  if (caps) *caps = e->caps;
  return VK_OK;
}

int vk_gemm_list(vk_dtype in_dtype, int* out, int max_count) {
  vk::init_registry();
  int n = 0;
  for (const auto& e : vk::registry()) {
    if (e.in_dtype != in_dtype) continue;
    if (out && n < max_count) out[n] = e.version;
    n++;
  }
  return n;
}

int vk_gemm_check(int version, vk_dtype in_dtype, vk_dtype out_dtype, size_t m, size_t n, size_t k,
                  const void* A, const void* B, const void* C) {
  return vk::validate(vk::find(version, in_dtype), out_dtype, m, n, k, A, B, C);
}

int vk_gemm_release(void) {
  std::lock_guard<std::mutex> lk(vk::g_dev_mutex);
  int st = VK_OK;
  int cur = 0;
  if (hipGetDevice(&cur) != hipSuccess) return VK_ERR_HIP;
  for (int d = 0; d < vk::kMaxDevices; d++) {
    if (!vk::g_dev[d].ws) continue;
    if (hipSetDevice(d) != hipSuccess || hipFree(vk::g_dev[d].ws) != hipSuccess) st = VK_ERR_HIP;
    vk::g_dev[d].ws = nullptr;
    vk::g_dev[d].ws_bytes = 0;
    vk::g_dev[d].ws_entry = nullptr;
  }
  if (hipSetDevice(cur) != hipSuccess) st = VK_ERR_HIP;
  return st;
}

const char* vk_status_string(int status) {
  switch (status) {
    case VK_OK: return "ok";
    case VK_ERR_VERSION: return "unknown version for this input dtype";
    case VK_ERR_DTYPE: return "unsupported input/output dtype pair";
    case VK_ERR_SHAPE: return "shape not supported by this version";
    case VK_ERR_ALIGN: return "operand pointer misaligned for this version";
    case VK_ERR_NULL: return "null operand with a non-empty shape";
    case VK_ERR_WORKSPACE: return "workspace too small";
    case VK_ERR_HIP: return "HIP runtime error";
    case VK_ERR_RANGE: return "dimension out of range";
    default: return "unknown status";
  }
}

int vk_gemm_abi_version(void) { return VK_GEMM_ABI_VERSION; }

}  // extern "C"
