// f16_padded.hip -- fp16 GEMM, version 15: any M, N and K at version 10's
// speed, for shapes whose rows are not multiples of 8 halves.
//
// Versions 7-11 load 16-byte chunks of A and B rows straight into LDS, so
// every row must start on a 16-byte boundary: N and K multiples of 8.  Other
// shapes (a vocabulary of 50,257 columns, K = 4095) take one of three ways:
//  * up to 128 rows with K >= 1024: f16_stream.hip reads B once;
//  * up to 2^33 multiply-adds: f16_any.hip loads any alignment through
//    registers (no_copies below);
//  * larger ones run version 10 (any M; N and K multiples of 8) on row-padded
//    copies in the workspace: A (M x K) with row pitch K8 = K rounded up to 8
//    when K % 8 != 0, B (K x N) with pitch N8 and K8 rows when N % 8 or K % 8
//    != 0, the pads zero (A's pad columns meet B's pad rows: zero times zero).
//    C is stored to the caller's rows at whatever alignment they have.
// Through the copies each element's sum runs over the same k as version 10's
// on the padded operands (the pad adds exact zeros), so the results are
// version 10's on explicitly padded inputs, bit for bit; so they are through
// f16_any.hip where version 10 does not split K.
// Measured (us per launch): the copy of a 4096 x 50257 B 152 (5.4 TB/s read
// and written; element by element 220), 4096 x 50257 x 4096 in all 1527 (1784
// with those copies and C through a padded buffer too), 4096 x 4095 x 4096 124
// (153), 2000 x 4095 x 8192 148 (174), 700 x 8191 x 2048 61 (75).
// Workspace: version 10's own (its split tails and counters, first), then
// A' and B' at 256-byte boundaries.
#include "vk_device.hpp"
#include "vk_internal.hpp"

#include <algorithm>

namespace vk {
namespace {

constexpr size_t kWsAlign = 256;
constexpr int kInnerVersion = 10;

size_t round_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

struct PadLayout {
  size_t k8, n8;
  bool pad_a, pad_b;
  size_t inner;                 // version 10's workspace bytes (at offset 0)
  size_t a_off, b_off;          // byte offsets of A', B' (when used)
  size_t total;
};

PadLayout layout_of(size_t m, size_t n, size_t k, int num_cus) {
  PadLayout L{};
  L.k8 = round_up(k, 8);
  L.n8 = round_up(n, 8);
  L.pad_a = L.k8 != k;
  L.pad_b = L.k8 != k || L.n8 != n;
  const KernelEntry* inner = find_registered(kInnerVersion, VK_DTYPE_F16);
  L.inner = inner && inner->workspace ? inner->workspace(m, L.n8, L.k8, num_cus) : 0;
  size_t off = round_up(L.inner, kWsAlign);
  L.a_off = off;
  if (L.pad_a) off = round_up(off + m * L.k8 * 2, kWsAlign);
  L.b_off = off;
  if (L.pad_b) off = round_up(off + L.k8 * L.n8 * 2, kWsAlign);
  if (L.n8 != n) off = round_up(off + m * L.n8 * 4, kWsAlign);
  L.total = off;
  return L;
}

// dst (drows rows of dpitch elements, a multiple of 8) <- src (rows rows of
// width elements), the elements past width or rows zero.  Each thread copies
// one 16-byte chunk of kRows consecutive destination rows, its loads out
// together; adjacent threads take adjacent chunks.  A chunk inside its source
// row is one 16-byte load at any 2-byte address, one at the row's end single
// elements.
constexpr int kRows = 4;
typedef uint32_t uint4u __attribute__((ext_vector_type(4), aligned(2)));
__global__ __launch_bounds__(256) void repitch_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst,
                                                      int rows, int width, int drows, int dpitch) {
  const int col = 8 * (int)(blockIdx.x * 256 + threadIdx.x);
  if (col >= dpitch) return;
  for (int r0 = (int)blockIdx.y * kRows; r0 < drows; r0 += (int)gridDim.y * kRows) {
    uint4v v[kRows];
#pragma unroll
    for (int i = 0; i < kRows; i++) {
      const uint16_t* p = src + (size_t)(r0 + i) * width + col;
      v[i] = uint4v{0u, 0u, 0u, 0u};
      if (r0 + i >= rows) continue;
      if (col + 8 <= width) {
        v[i] = *reinterpret_cast<const uint4u*>(p);
      } else {
        uint16_t x[8];
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = col + e < width ? p[e] : (uint16_t)0;
        __builtin_memcpy(&v[i], x, 16);
      }
    }
#pragma unroll
    for (int i = 0; i < kRows; i++)
      if (r0 + i < drows) *reinterpret_cast<uint4v*>(dst + (size_t)(r0 + i) * dpitch + col) = v[i];
  }
}

hipError_t repitch(const void* src, void* dst, size_t rows, size_t width, size_t drows, size_t dpitch,
                   hipStream_t s) {
  const unsigned gx = (unsigned)((dpitch / 8 + 255) / 256);
  const unsigned gy = (unsigned)std::min<size_t>((drows + kRows - 1) / kRows, 65535);
  hipLaunchKernelGGL(repitch_kernel, dim3(gx, gy), dim3(256), 0, s, static_cast<const uint16_t*>(src),
                     static_cast<uint16_t*>(dst), (int)rows, (int)width, (int)drows, (int)dpitch);
  return hipGetLastError();
}

// Few rows need no copies: f16_stream.hip reads B once at any row alignment.
bool few_rows(size_t m, size_t n, size_t k) { return (n % 8 || k % 8) && f16_stream_takes(m, n, k); }

// Neither do products too small to earn the copies back (f16_any.hip).  us per
// launch against the copies and version 10: 1000 x 1001 x 999 13.5 / 33, 300 x
// 4095 x 4096 44 / 58, 2000 x 2001 x 2002 (2^33) 51 / 56, but 700 x 8191 x 2048
// 64 / 61, 300 x 11007 x 4096 92 / 98 and 4096 x 4095 x 4096 260 / 124.  A few
// tiles of a deep K keep version 10's split sum (300 x 200 x 4095: 28.7 / 49).
bool no_copies(size_t m, size_t n, size_t k, int num_cus) {
  const size_t tiles = (m + 63) / 64 * ((n + 63) / 64);
  if ((m + 127) / 128 > 65535) return false;  // rows of its tiles are grid.y
  return (n % 8 || k % 8) && m * n * k <= ((size_t)1 << 33) && (8 * tiles >= (size_t)num_cus || k <= 1024);
}

hipError_t launch_padded(const GemmArgs& a) {
  if (few_rows(a.m, a.n, a.k)) return f16_stream_launch(a, layout_of(a.m, a.n, a.k, a.num_cus).total);
  if (no_copies(a.m, a.n, a.k, a.num_cus)) return f16_any_launch(a);
  const KernelEntry* inner = find_registered(kInnerVersion, VK_DTYPE_F16);
  if (!inner) return hipErrorInvalidValue;
  const PadLayout L = layout_of(a.m, a.n, a.k, a.num_cus);
  char* ws = static_cast<char*>(a.workspace);
  GemmArgs b = a;
  b.n = L.n8;
  b.k = L.k8;
  b.ldc = a.n;
  hipError_t e = hipSuccess;
  if (L.pad_a) {
    b.A = ws + L.a_off;
    e = repitch(a.A, ws + L.a_off, a.m, a.k, a.m, L.k8, a.stream);
    if (e != hipSuccess) return e;
  }
  if (L.pad_b) {
    b.B = ws + L.b_off;
    // rows that only follow each other (N a multiple of 8) are one long row
    e = L.n8 == a.n ? repitch(a.B, ws + L.b_off, 1, a.k * a.n, 1, L.k8 * L.n8, a.stream)
                    : repitch(a.B, ws + L.b_off, a.k, a.n, L.k8, L.n8, a.stream);
    if (e != hipSuccess) return e;
  }
  b.workspace = L.inner ? ws : nullptr;
  b.workspace_bytes = L.inner;
  // The region where version 10 keeps its counters may have held A' or B' in
  // an earlier call of this version (whose padded problem needed no
  // counters), so they are always cleared first.
  b.workspace_clean = false;
  return inner->launch(b);
}

// Every call of a shape with padded rows asks for the copies' workspace and an
// fp32 C of n8 columns, also those that use less of it or none, so the sizes
// that callers hold workspaces for stay what they have been.
size_t workspace_padded(size_t m, size_t n, size_t k, int num_cus) {
  return layout_of(m, n, k, num_cus).total;
}

// Calls of few rows that split K leave their own counters clean at the
// workspace's start; those that do not, and calls without copies, leave it as
// it was, whatever it holds; the copies overwrite it.
int workspace_kind(size_t m, size_t n, size_t k, int num_cus) {
  if (few_rows(m, n, k))
    return f16_stream_pieces(m, n, k, layout_of(m, n, k, num_cus).total, num_cus) > 1 ? 1 : kWorkspaceUntouched;
  return no_copies(m, n, k, num_cus) ? kWorkspaceUntouched : 0;
}

// Version 10's limits on the padded problem.
bool shape_ok_padded(size_t m, size_t n, size_t k) {
  const KernelEntry* inner = find_registered(kInnerVersion, VK_DTYPE_F16);
  const size_t n8 = round_up(n, 8), k8 = round_up(k, 8);
  return inner && m >= 1 && n >= 1 && k >= 1 && (!inner->shape_ok || inner->shape_ok(m, n8, k8));
}

}  // namespace

void register_f16_padded() {
  KernelEntry e{};
  e.version = 15;
  e.in_dtype = VK_DTYPE_F16;
  e.name = "f16_v15_padded_v10";
  // 16-byte aligned operands, as version 10's: an operand whose rows need no
  // padding goes to version 10 as it is
  e.caps = make_caps(15, VK_DTYPE_F16, kOutF16 | kOutF32, 1, 1, 1, 16, 256, 256, 64, 512, 160 * 1024, 0, 1);
  e.launch = launch_padded;
  e.workspace = workspace_padded;
  e.shape_ok = shape_ok_padded;
  e.workspace_kind = workspace_kind;
  register_kernel(e);
}

}  // namespace vk
