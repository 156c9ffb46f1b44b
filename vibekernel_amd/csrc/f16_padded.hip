// f16_padded.hip -- fp16 GEMM, version 15: any M, N and K at version 10's
// speed, for shapes whose rows are not multiples of 8 halves.
//
// Versions 7-11 load 16-byte chunks of A and B rows straight into LDS, so
// every row must start on a 16-byte boundary: N and K multiples of 8.  Other
// shapes (a vocabulary of 50,257 columns, K = 4095) take one of three ways:
//  * up to 128 rows with K >= 1024: f16_stream.hip reads B once;
//  * products that cannot earn copies back: f16_any.hip loads any alignment
//    through registers (no_copies below);
//  * the others run version 10 (any M; N and K multiples of 8) on row-padded
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
// together; adjacent threads take adjacent chunks, and a workgroup as many
// threads per row as the row has chunks to give them (a power of two).  A chunk
// inside its source row is one 16-byte load at any 2-byte address, one at the
// row's end single elements.
typedef uint32_t uint4u __attribute__((ext_vector_type(4), aligned(2)));
template <int kRows>
__global__ __launch_bounds__(256) void repitch_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst,
                                                      int rows, int width, int drows, int dpitch) {
  const int col = 8 * (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (col >= dpitch) return;
  for (int r0 = (int)(blockIdx.y * blockDim.y + threadIdx.y) * kRows; r0 < drows;
       r0 += (int)(gridDim.y * blockDim.y) * kRows) {
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

template <int kRows>
hipError_t repitch_rows(const void* src, void* dst, size_t rows, size_t width, size_t drows, size_t dpitch,
                        hipStream_t s) {
  unsigned tx = 256;  // threads per row
  while (tx > 1 && tx / 2 >= dpitch / 8) tx /= 2;
  const unsigned ty = 256 / tx;
  const unsigned gx = (unsigned)((dpitch / 8 + tx - 1) / tx);
  const unsigned gy = (unsigned)std::min<size_t>((drows + kRows * ty - 1) / (kRows * ty), 65535);
  hipLaunchKernelGGL(repitch_kernel<kRows>, dim3(gx, gy), dim3(tx, ty), 0, s, static_cast<const uint16_t*>(src),
                     static_cast<uint16_t*>(dst), (int)rows, (int)width, (int)drows, (int)dpitch);
  return hipGetLastError();
}
// 4 rows per thread where that leaves 4 workgroups per CU or more (a 4000 x 33 A:
// 3.2 us with 4, 2.0 with 1).
hipError_t repitch(const void* src, void* dst, size_t rows, size_t width, size_t drows, size_t dpitch,
                   hipStream_t s) {
  const bool many = drows >= 4 && drows * (dpitch / 8) >= ((size_t)1 << 20);
  return many ? repitch_rows<4>(src, dst, rows, width, drows, dpitch, s)
              : repitch_rows<1>(src, dst, rows, width, drows, dpitch, s);
}

// Few rows need no copies: f16_stream.hip reads B once at any row alignment.
bool few_rows(size_t m, size_t n, size_t k) { return (n % 8 || k % 8) && f16_stream_takes(m, n, k); }

// Neither do products that cannot earn the copies back (f16_any.hip), up to 2^33
// multiply-adds.  Where K is a multiple of 8 only B is copied, and the copies earn
// more.  us per launch, f16_any.hip / copies and version 10:
//  * N below 8, whose B is loaded element by element: 100000 x 7 x 258 51 / 57, x 1025
//    182 / 140, x 96 16.5 / 22, 300000 x 2 x 128 59 / 48, 46840 x 1 x 688 60 / 26; 20000 x
//    3 x 256 9.8 / 13.8, 2000 x 1 x 688 16.8 / 20.7, x 1024 26.4 / 25.9;
//  * while 64 x 64 tiles are at most 4 per CU (f16_any_launch's rule for them): 1000
//    x 1001 x 1023 13.0 / 34.3, 2000 x 2001 x 2001 48 / 55.  But a workgroup's k-loop
//    is one chain there, and version 10 splits the sum of few 256 x 256 tiles 10 to 32
//    ways or more: the copies win a deep enough K, unless most of those tiles is empty
//    or copying a wide B is most of the work: up to a tile per CU, B alone copied, 779 x 148 x 13032
//    61 / 65, 2845 x 67 x 14536 85 / 75, 218 x 2606 x 12448 68 / 90, 14946 x 29 x 14024
//    97 / 131; odd K, whose rows of A straddle dwords, 361 x 418 x 11377 66 / 68, 245 x
//    1272 x 14363 92 / 78, 5825 x 33 x 14805 102 / 154; even K 238 x 1456 x 14678 83 / 80,
//    141 x 852 x 14366 66 / 74, 1085 x 178 x 19398 120 / 94, 1987 x 32 x 17674 84 / 97,
//    13398 x 30 x 17198 100 / 314.  With more tiles, B alone copied, 2463 x 419 x 7744
//    68 / 55, 2332 x 409 x 5776 52 / 52, 2764 x 365 x 8104 76 / 63, 413 x 2535 x 5584
//    54 / 62, 763 x 3761 x 2696 43 / 56; with A too 22016 x 16 x 18286 188 / 547.  Fewer
//    tiles than an eighth of the CUs keep version 10's split sum (and its bits) from
//    K = 1025 on, though 300 x 200 x 4095 takes 28.7 / 49;
//  * where half of each 256 x 256 tile is empty: 128 x 50001 x 1023 53 / 67, 100000
//    x 65 x 513 63 / 79, but 100000 x 65 x 512 56 / 42, x 256 35 / 31;
//  * while 128 x 128 tiles are at most 2 per CU, even K and narrow products: 1000 x
//    8001 x 129 18.4 / 20.4, 3000 x 1500 x 1023 35 / 40, x 1500 43 / 46, 26144 x 138 x
//    1910 67 / 80, 3056 x 1576 x 1690 47 / 48, 7627 x 516 x 2126 60 / 67, 19652 x 262 x
//    1461 56 / 62, but 4326 x 1473 x 1281 51 / 43; B alone copied 16000 x 401 x 512
//    24.7 / 20.2, 226 x 21777 x 488 26 / 28, 221 x 30095 x 832 38 / 44;
//  * small K while 128 x 128 tiles are one residency there (4 per CU) and 256 x 256
//    tiles more than one: 11118 x 1328 x 21 16.9 / 19.9, 281 x 41448 x 46 17.8 / 21.9;
//  * past that few columns up to K = 256, whose copy of A is most of the work:
//    50000 x 304 x 193 32 / 36, x 257 47 / 43, 50000 x 200 x 193 24 / 29, x 385 45 /
//    39, 30000 x 600 x 129 28.0 / 29.6; 50000 x 400 x 65 28.7 / 26.3; and few rows whose
//    A or B starts on dwords: 300 x 50000 x 193 32 / 35, x 257 47 / 40; 300 x 50001 x 65
//    30.3 / 29.5, x 130 28.6 / 31.8; 400 x 50000 x 65 31.5 / 26.3, 129 x 100000 x 129
//    38.7 / 34.0; 220 x 42640 x 155 20.6 / 22.9, 239 x 74678 x 144 29.8 / 33.7, 161 x
//    55546 x 16 15.7 / 12.5;
//  * the rest take the copies: 4000 x 4000 x 33 18.6 / 15.3, 4096 x 8192 x 255 55 /
//    40, 8192 x 8193 x 65 111 / 59.
bool no_copies(size_t m, size_t n, size_t k, int num_cus) {
  if (n % 8 == 0 && k % 8 == 0) return false;           // no copies to make
  if ((m + 127) / 128 > 65535) return false;            // rows of its tiles are grid.y
  if (m * n * k > (size_t)1 << 33) return false;
  const size_t c = num_cus;
  const bool copy_a = k % 8 != 0;
  auto tiles = [&](size_t t) { return (m + t - 1) / t * ((n + t - 1) / t); };
  const size_t small = tiles(64), tiles256 = tiles(256);
  if (n < 8) return k <= (copy_a ? 384 : 120) || (k <= 768 && m * k < (size_t)1 << 23);
  if (small <= 4 * c) {
    if (k <= 1024) return true;
    if (8 * small < c) return false;
    bool copies;
    if (copy_a)
      copies = small <= c && 32 * tiles256 <= c && (k % 2 ? k > 12288 : k > 16384 && std::min(m, n) > 128);
    else if (small <= c)
      copies = k > 13312 && n <= m && 20 * tiles256 <= c;
    else if (12 * tiles256 <= c)
      copies = k > (n % 2 ? 4608 : 6144) && n <= 2 * m;  // even N: B's rows start on dwords
    else
      copies = k > 6144 && n <= m && 10 * tiles256 <= c;
    return !copies;
  }
  if (m <= 128) return true;
  if (n <= 128) return copy_a || k < 256;
  const size_t tiles128 = tiles(128);
  if (tiles128 <= 2 * c) {
    if (copy_a) return k % 2 == 0 || k <= 1280 || std::min(m, n) <= 384;
    return m <= 400 || k <= (n % 2 ? 256 : 1536);
  }
  if (tiles128 <= 4 * c && tiles256 > c && k <= 128) return true;
  const bool few = tiles128 <= 5 * c;
  if (few && m <= 256 && n % 2 == 0 && k > 40 && k <= 256) return true;
  if (!copy_a || k > 256) return false;
  const size_t filled = 100 * m * n / (tiles256 * 65536);  // per cent of the 256 x 256 tiles
  return m > n ? n <= 256 || filled <= (few ? 80 : 60) : (n % 8 == 0 || k % 2 == 0) && k > 64 && filled <= 60 && few;
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
