// f16_stream.hip -- fp16 GEMM for up to 128 rows, N >= 8 and K >= 1024: B
// streamed once from memory straight into registers, whatever its row
// alignment (version 15's path for few rows).
//
// Versions 8 and 14 load 16-byte chunks of B rows straight into LDS, so a row
// has to start on a 16-byte boundary.  Other widths (a vocabulary of 50,257
// columns) went through a row-padded copy of B, which moves B three times
// and then runs 256-row tiles on a few rows.  What bounds this job is reading
// B once.  Global loads take any 2-byte address on MI355X at nearly the
// aligned rate (a read of a 4096 x 50257 B, 16 bytes per lane: 5.18 TB/s
// against 5.47 at 50256 columns), so no copy is needed:
//  * a workgroup owns 128 columns (256-byte row pieces) and 1/ks of K; its 4
//    waves each take a contiguous share of that k range on their own: no
//    barrier, no LDS in the k-loop;
//  * per 32-deep k-step lane l loads rows 8(l/16) .. +7, columns 8(l%16) ..
//    +7 (8 loads of 16 bytes, 8 KB per wave), for which the MFMA's B operand
//    (8 k of one column per lane) is one byte permute per pair of halves:
//    fragment c holds columns 8(l%16) + c, so a lane's 8 accumulators of a
//    row are 8 consecutive columns of C and leave as one 16-byte store;
//  * A comes from the caches into registers as MFMA fragments (16 rows x 64
//    bytes per load); kD k-steps of both are in flight per wave.  Where K is
//    odd, every other row starts between two dwords, and such loads from 16
//    rows take half as long again as B's: A is then loaded by whole dwords,
//    one more per fragment, and shifted (up to 9 rows as it is);
//  * the lanes of a last column block that N cuts short take the last 8
//    columns of the matrix instead (N >= 8): every load stays inside B, and
//    columns computed twice are the same sum stored twice;
//  * the k past the last whole step are one more step of the wave that holds
//    the end of K: its loads are moved back into the matrices and both
//    operands' values past K replaced by zeros (an infinity there must not
//    meet a zero);
//  * the 4 waves' sums meet in LDS, wave q adding the rows 4i + q in wave
//    order; the ks workgroups' in memory as version 14's pieces do (a counter
//    per column block and wave, the last arrival sums the pieces in k order),
//    so C does not depend on the arrival order.
// Each output is the sum, in k order, of 4 ks chains over consecutive ranges
// of K.
// Measured (us per launch, fresh operands each, against the padded copies and
// version 10): 4096 x 50257 weights at M = 1 / 32 (fp32 out) / 64 / 128 79.8 /
// 92.2 / 110 / 191 against 311 / 318 / 316 / 326 (the streaming read alone is
// 79.4); 16 x 8191 x 8192 29.5 against 127; 128 x 8191 x 8192 55.6 against 131;
// 16 x 4095 x 4096 13.8 against 59; 64 x 1001 x 1025 15.5 against 33.5; 16 x
// 301 x 16000 14.5 against 74.  Odd K, with A shifted in registers and as loaded
// before: 16 / 64 / 128 x 16391 x 4095 40.5 / 59.7 / 92.6 and 43.2 / 78.0 / 141
// (copies: 127); 128 x 50256 x 1025 62.9 and 82.3 (65.5); 15 x 4816 x 9409 27.7 and
// 28.5, but 9 x 3920 x 5637 15.6 and 15.2, 3 x 3584 x 1183 7.5 and 7.2.
#include "vk_device.hpp"
#include "vk_internal.hpp"
#include "vk_stream.hpp"
#include "vk_tile.hpp"

namespace vk {
namespace {

constexpr int W = kStreamWaves;          // waves per workgroup
constexpr int kThreads = 64 * W;
constexpr int kKStep = 32;
constexpr int kNC = 128;                 // columns per workgroup
constexpr int kMaxRows = 128;

typedef uint32_t uint4u __attribute__((ext_vector_type(4), aligned(2)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));

// MB 16-row blocks, kOdd: K odd.  k-steps in flight per wave, and the workgroups
// per CU the registers are cut for (256 registers per lane at 2).
template <int MB, bool kOdd>
struct StCfg {
  static constexpr int kD = MB == 1 ? 3 : MB == 2 ? 2 : MB == 4 && kOdd ? 3 : 4;
  static constexpr int kOcc = MB <= 2 ? 2 : 1;
};

__device__ __forceinline__ uint4v load16(const char* base, uint32_t off) {
  return *reinterpret_cast<const uint4u*>(base + off);
}

__device__ __forceinline__ uint4v load16_dwords(const char* base, uint32_t off) {
  typedef uint32_t uint4d __attribute__((ext_vector_type(4), aligned(4)));
  return *reinterpret_cast<const uint4d*>(base + off);
}

// The low (kHi = false) or high halves of two dwords: {lo, hi} of the result.
template <bool kHi>
__device__ __forceinline__ uint32_t pack_halves(uint32_t first, uint32_t second) {
  return __builtin_amdgcn_perm(second, first, kHi ? 0x07060302u : 0x05040100u);
}

__device__ __forceinline__ void store_row8(half_t* p, const float4v (&x)[2]) {
  half8 h;
#pragma unroll
  for (int c = 0; c < 8; c++) h[c] = convert_out<half_t>(x[c / 4][c % 4]);
  *reinterpret_cast<uint4u*>(p) = __builtin_bit_cast(uint4v, h);
}
__device__ __forceinline__ void store_row8(float* p, const float4v (&x)[2]) {
  *reinterpret_cast<float4u*>(p) = x[0];
  *reinterpret_cast<float4u*>(p + 4) = x[1];
}

template <int MB, typename OutT, bool kOdd>
__global__ __launch_bounds__(kThreads, (StCfg<MB, kOdd>::kOcc)) void f16_stream_kernel(
    const half_t* __restrict__ A, const half_t* __restrict__ B, OutT* __restrict__ C, int M, int N, int K, int ks,
    int halves, float* __restrict__ part, unsigned* __restrict__ counters) {
  constexpr int D = StCfg<MB, kOdd>::kD;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, i16 = lane & 15;

  const int ncb = (N + kNC - 1) / kNC;
  // the row halves of a column block, which read the same B, and a piece's
  // neighbouring column blocks, which share the cache lines at their edge, on
  // one XCD, a column block's pieces on different ones
  const int id = xcd_remap(blockIdx.x, ncb * ks * halves);
  const int piece = id / halves, m0 = (id - piece * halves) * (16 * MB);
  const int kp = piece / ncb, cb = piece - kp * ncb;
  const int slot0 = (cb * halves + (m0 ? 1 : 0)) * ks;  // this block's first partial slot
  const int n0 = cb * kNC;
  const int parts = ks * W, p = kp * W + wave;
  const int tsteps = K / kKStep;
  const int sbeg = (int)((long long)p * tsteps / parts);
  const int ns = (int)((long long)(p + 1) * tsteps / parts) - sbeg;

  const int col = min(n0 + 8 * i16, N - 8);
  uint32_t offB[8];
#pragma unroll
  for (int j = 0; j < 8; j++) offB[j] = ((uint32_t)(8 * g + j) * (uint32_t)N + (uint32_t)col) * 2u;
  uint32_t offA[MB];
#pragma unroll
  for (int r = 0; r < MB; r++)
    offA[r] = ((uint32_t)min(m0 + 16 * r + i16, M - 1) * (uint32_t)K + (uint32_t)(8 * g)) * 2u;
  const char* gB = reinterpret_cast<const char*>(B) + (size_t)sbeg * kKStep * N * 2;
  const char* gA = reinterpret_cast<const char*>(A) + (size_t)sbeg * kKStep * 2;
  const size_t bstep = (size_t)kKStep * N * 2;

  float4v acc[MB][8];
#pragma unroll
  for (int r = 0; r < MB; r++)
#pragma unroll
    for (int c = 0; c < 8; c++) acc[r][c] = float4v{0.f, 0.f, 0.f, 0.f};

  struct Step {
    uint4v b[8], a[MB];
    uint32_t next[kOdd ? MB : 1];  // kOdd: the dword that an odd row's fragment ends in
  };
  Step buf[D];
  auto load = [&](Step& s, int j) {
    const char* pb = gB + (size_t)j * bstep;
    const char* pa = gA + (size_t)j * (kKStep * 2);
#pragma unroll
    for (int i = 0; i < 8; i++) s.b[i] = load16(pb, offB[i]);
#pragma unroll
    for (int r = 0; r < MB; r++) {
      if constexpr (kOdd) {
        // the last dword once more for an even row, whose fragment may be the
        // end of A
        s.a[r] = load16_dwords(pa, offA[r] & ~3u);
        s.next[r] = *reinterpret_cast<const uint32_t*>(pa + ((offA[r] + 14) & ~3u));
      } else {
        s.a[r] = load16(pa, offA[r]);
      }
    }
  };
  // The fragments of A in a loaded step.
  auto shift_a = [&](Step& s) {
    if constexpr (kOdd)
#pragma unroll
      for (int r = 0; r < MB; r++) {
        const uint32_t sh = (offA[r] & 2u) * 8u;
#pragma unroll
        for (int d = 0; d < 4; d++)
          s.a[r][d] = __builtin_amdgcn_alignbit(d < 3 ? s.a[r][d + 1] : s.next[r], s.a[r][d], sh);
      }
  };
  auto multiply = [&](const Step& s) {
#pragma unroll
    for (int d = 0; d < 4; d++) {
      uint4v lo, hi;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        lo[q] = pack_halves<false>(s.b[2 * q][d], s.b[2 * q + 1][d]);
        hi[q] = pack_halves<true>(s.b[2 * q][d], s.b[2 * q + 1][d]);
      }
#pragma unroll
      for (int r = 0; r < MB; r++) {
        const half8 a = __builtin_bit_cast(half8, s.a[r]);
        acc[r][2 * d] = mfma16x16x32(a, __builtin_bit_cast(half8, lo), acc[r][2 * d]);
        acc[r][2 * d + 1] = mfma16x16x32(a, __builtin_bit_cast(half8, hi), acc[r][2 * d + 1]);
      }
    }
  };

#pragma unroll
  for (int u = 0; u < D; u++) load(buf[u], min(u, ns - 1));
  int s0 = 0;
  // the loads of step s + D go out behind the products of step s
  for (; s0 + 2 * D <= ns; s0 += D) {
#pragma unroll
    for (int u = 0; u < D; u++) {
      __builtin_amdgcn_sched_barrier(0);
      shift_a(buf[u]);
      multiply(buf[u]);
      __builtin_amdgcn_sched_barrier(0);
      load(buf[u], s0 + u + D);
    }
  }
  // fewer than 2 D steps left (the loop above asks no step whether it exists)
#pragma unroll
  for (int u = 0; u < D; u++) {
    if (s0 + u < ns) {
      shift_a(buf[u]);
      multiply(buf[u]);
    }
    if (s0 + u + D < ns) load(buf[u], s0 + u + D);
  }
#pragma unroll
  for (int u = 0; u < D; u++)
    if (s0 + u + D < ns) {
      shift_a(buf[u]);
      multiply(buf[u]);
    }
  if (p == parts - 1 && tsteps * kKStep < K) {
    const int kt = tsteps * kKStep + 8 * g;
    const int past = max(kt + 8 - K, 0);  // of the lane's 8 k, how many lie past K
    Step& s = buf[0];
#pragma unroll
    for (int j = 0; j < 8; j++)
      s.b[j] = load16(reinterpret_cast<const char*>(B + (size_t)min(kt + j, K - 1) * N), (uint32_t)col * 2u);
#pragma unroll
    for (int r = 0; r < MB; r++)
      s.a[r] = load16(reinterpret_cast<const char*>(A + (size_t)min(m0 + 16 * r + i16, M - 1) * K),
                      (uint32_t)min(kt, K - 8) * 2u);
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (kt + j >= K) s.b[j] = uint4v{0u, 0u, 0u, 0u};
#pragma unroll
    for (int r = 0; r < MB; r++) {
      const unsigned __int128 v = __builtin_bit_cast(unsigned __int128, s.a[r]);
      s.a[r] = __builtin_bit_cast(uint4v, past < 8 ? v >> (16 * past) : (unsigned __int128)0);
    }
    multiply(s);
  }

  stream_finish<MB, 2>(acc, lane, wave, ks, kp, slot0, ncb * halves * ks, part, counters,
                       [&](int r, const float4v (&x)[2]) {
                         const int row = m0 + 16 * r + 4 * g + wave;
                         if (row < M) store_row8(C + (size_t)row * N + col, x);
                       });
}

// Up to 64 rows a workgroup takes them all; more are cut in two halves of
// whole 16-row blocks, whose workgroups read the same B next to each other.
// (One workgroup for 128 rows leaves no registers for loads in flight: 128 x
// 50257 x 4096 took 265.7 us.)
int halves_of(size_t m) { return m > 64 ? 2 : 1; }
int blocks_of(size_t m) { return (int)(((m + 15) / 16 + halves_of(m) - 1) / halves_of(m)); }

template <int MB, typename OutT, bool kOdd>
hipError_t launch_t(const GemmArgs& a, size_t ws_limit) {
  const int halves = halves_of(a.m);
  const int ks = f16_stream_pieces(a.m, a.n, a.k, ws_limit, a.num_cus);
  unsigned* counters = nullptr;
  float* part = nullptr;
  const hipError_t e = stream_buffers(a, ks, counters, part);
  if (e != hipSuccess) return e;
  const unsigned grid = (unsigned)((a.n + kNC - 1) / kNC * ks * halves);
  hipLaunchKernelGGL((f16_stream_kernel<MB, OutT, kOdd>), dim3(grid), dim3(kThreads), 0, a.stream,
                     static_cast<const half_t*>(a.A), static_cast<const half_t*>(a.B), static_cast<OutT*>(a.C),
                     (int)a.m, (int)a.n, (int)a.k, ks, halves, part, counters);
  return hipGetLastError();
}

template <int MB, bool kOdd>
hipError_t launch_out(const GemmArgs& a, size_t ws_limit) {
  return a.out_dtype == VK_DTYPE_F16 ? launch_t<MB, half_t, kOdd>(a, ws_limit) : launch_t<MB, float, kOdd>(a, ws_limit);
}
template <int MB>
hipError_t launch_mb(const GemmArgs& a, size_t ws_limit) {
  return a.k % 2 && a.m > 9 ? launch_out<MB, true>(a, ws_limit) : launch_out<MB, false>(a, ws_limit);
}

}  // namespace

// At least 8 columns (a lane's load) and 8 k-steps per wave; lane offsets of
// 32 k-rows of B and 128 rows of A below 2^32 bytes.
bool f16_stream_takes(size_t m, size_t n, size_t k) {
  return m >= 1 && m <= kMaxRows && n >= 8 && n < (1u << 25) && k >= 8 * W * kKStep && k < (1u << 23);
}

int f16_stream_pieces(size_t m, size_t n, size_t k, size_t ws_limit, int num_cus) {
  return stream_pieces((n + kNC - 1) / kNC * halves_of(m), k / kKStep, blocks_of(m), 2, ws_limit, num_cus);
}

hipError_t f16_stream_launch(const GemmArgs& a, size_t ws_limit) {
  switch (blocks_of(a.m)) {
    case 1: return launch_mb<1>(a, ws_limit);
    case 2: return launch_mb<2>(a, ws_limit);
    case 3: return launch_mb<3>(a, ws_limit);
    default: return launch_mb<4>(a, ws_limit);
  }
}

}  // namespace vk
