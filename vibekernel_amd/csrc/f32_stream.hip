// f32_stream.hip -- fp32 GEMM for up to 64 rows, N and K multiples of 4: B
// streamed once from memory straight into registers (version 3's path for few
// rows).
//
// Version 3's tiles are 64 rows high and wait for every k-tile at a barrier;
// a few rows are bound by reading B once instead.  As f16_stream.hip: a
// workgroup owns 64 columns (256-byte row pieces) and 1/ks of K, its 4 waves a
// contiguous share of that each, with no barrier and no LDS in the k-loop.
//  * Per 16-deep k-step lane l loads rows 4(l/16) .. +3, columns 4(l%16) ..
//    +3 of B (4 loads of 16 bytes, 4 KB per wave) and, per 16-row block of A,
//    row l%16, k 4(l/16) .. +3: as they are, value j of A and row j of B are
//    the operands of v_mfma_f32_16x16x4_f32 j of the step (its lane group g
//    holding k = 4g + j), column c of the B row those of accumulator c, so a
//    lane's 4 accumulators of a row are 4 consecutive columns of C;
//  * kD k-steps are in flight per wave;
//  * lanes past N take the matrix's last 4 columns (computed twice, the same
//    sum stored twice); k past K in the last step are moved back into the
//    matrices and replaced by zeros in both operands.
// fp32 products, fp32 sums; each output is the sum, in k order, of 4 ks chains
// over consecutive ranges of K (within a step in the order j, then g).
#include "vk_device.hpp"
#include "vk_internal.hpp"
#include "vk_stream.hpp"
#include "vk_tile.hpp"

namespace vk {
namespace {

constexpr int W = kStreamWaves;
constexpr int kThreads = 64 * W;
constexpr int kKStep = 16;
constexpr int kNC = 64;
constexpr int kMaxRows = 64;

// MB 16-row blocks: k-steps in flight (4 + MB loads of 16 bytes each), and the
// workgroups per CU that the registers are cut for.
template <int MB>
struct StCfg {
  static constexpr int kD = MB <= 2 ? 6 : 4;
  static constexpr int kOcc = 2;
};

template <int MB>
__global__ __launch_bounds__(kThreads, StCfg<MB>::kOcc) void f32_stream_kernel(const float* __restrict__ A,
                                                                               const float* __restrict__ B,
                                                                               float* __restrict__ C, int M, int N,
                                                                               int K, int ks, float* __restrict__ part,
                                                                               unsigned* __restrict__ counters) {
  constexpr int D = StCfg<MB>::kD;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, i16 = lane & 15;

  const int ncb = (N + kNC - 1) / kNC;
  // a piece's column blocks on one XCD, a column block's pieces on different
  // ones
  const int id = xcd_remap(blockIdx.x, ncb * ks);
  const int kp = id / ncb, cb = id - kp * ncb;
  const int parts = ks * W, p = kp * W + wave;
  const int tsteps = (K + kKStep - 1) / kKStep;
  const int sbeg = (int)((long long)p * tsteps / parts);
  const int ns = (int)((long long)(p + 1) * tsteps / parts) - sbeg;

  const int col = min(cb * kNC + 4 * i16, N - 4);
  uint32_t offB[4], offA[MB];
#pragma unroll
  for (int j = 0; j < 4; j++) offB[j] = ((uint32_t)(4 * g + j) * (uint32_t)N + (uint32_t)col) * 4u;
#pragma unroll
  for (int r = 0; r < MB; r++)
    offA[r] = ((uint32_t)min(16 * r + i16, M - 1) * (uint32_t)K + (uint32_t)(4 * g)) * 4u;
  const char* gB = reinterpret_cast<const char*>(B) + (size_t)sbeg * kKStep * N * 4;
  const char* gA = reinterpret_cast<const char*>(A) + (size_t)sbeg * kKStep * 4;
  const size_t bstep = (size_t)kKStep * N * 4;
  // K a multiple of 4: a lane group's 4 k of the last step are all below K or
  // all past it
  const bool cut = p == parts - 1 && K % kKStep != 0;  // this wave's last step reaches past K
  const uint32_t back = 4 * g >= K % kKStep ? (uint32_t)(4 * g) : 0u;  // then: k to move back

  float4v acc[MB][4];
#pragma unroll
  for (int r = 0; r < MB; r++)
#pragma unroll
    for (int c = 0; c < 4; c++) acc[r][c] = float4v{0.f, 0.f, 0.f, 0.f};

  struct Step {
    float4v b[4], a[MB];
  };
  Step buf[D];
  auto load_at = [&](Step& s, int j, uint32_t back_k) {
    const char* pb = gB + (size_t)j * bstep;
    const char* pa = gA + (size_t)j * (kKStep * 4);
#pragma unroll
    for (int i = 0; i < 4; i++)
      s.b[i] = *reinterpret_cast<const float4v*>(pb + (offB[i] - back_k * (uint32_t)N * 4u));
#pragma unroll
    for (int r = 0; r < MB; r++) s.a[r] = *reinterpret_cast<const float4v*>(pa + (offA[r] - back_k * 4u));
  };
  auto load = [&](Step& s, int j) { load_at(s, j, 0u); };
  auto multiply = [&](const Step& s) {
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int r = 0; r < MB; r++)
#pragma unroll
        for (int c = 0; c < 4; c++)
          acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(s.a[r][j], s.b[j][c], acc[r][c], 0, 0, 0);
  };

  const int nw = ns - (cut ? 1 : 0);  // whole steps
  if (nw > 0) {
#pragma unroll
    for (int u = 0; u < D; u++) load(buf[u], min(u, nw - 1));
    int s0 = 0;
    // the loads of step s + D go out behind the products of step s
    for (; s0 + 2 * D <= nw; s0 += D) {
#pragma unroll
      for (int u = 0; u < D; u++) {
        __builtin_amdgcn_sched_barrier(0);
        multiply(buf[u]);
        __builtin_amdgcn_sched_barrier(0);
        load(buf[u], s0 + u + D);
      }
    }
    // fewer than 2 D steps left (the loop above asks no step whether it exists)
#pragma unroll
    for (int u = 0; u < D; u++) {
      if (s0 + u < nw) multiply(buf[u]);
      if (s0 + u + D < nw) load(buf[u], s0 + u + D);
    }
#pragma unroll
    for (int u = 0; u < D; u++)
      if (s0 + u + D < nw) multiply(buf[u]);
  }
  if (cut) {
    Step& s = buf[0];
    load_at(s, nw, back);
    if (back) {
#pragma unroll
      for (int i = 0; i < 4; i++) s.b[i] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < MB; r++) s.a[r] = float4v{0.f, 0.f, 0.f, 0.f};
    }
    multiply(s);
  }

  stream_finish<MB, 1>(acc, lane, wave, ks, kp, cb * ks, ncb * ks, part, counters,
                       [&](int r, const float4v (&x)[1]) {
                         const int row = 16 * r + 4 * g + wave;
                         if (row < M) *reinterpret_cast<float4v*>(C + (size_t)row * N + col) = x[0];
                       });
}

int blocks_of(size_t m) { return (int)((m + 15) / 16); }

template <int MB>
hipError_t launch_mb(const GemmArgs& a, size_t ws_limit) {
  const int ks = f32_stream_pieces(a.m, a.n, a.k, ws_limit, a.num_cus);
  unsigned* counters = nullptr;
  float* part = nullptr;
  const hipError_t e = stream_buffers(a, ks, counters, part);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(f32_stream_kernel<MB>, dim3((unsigned)((a.n + kNC - 1) / kNC * ks)), dim3(kThreads), 0, a.stream,
                     static_cast<const float*>(a.A), static_cast<const float*>(a.B), static_cast<float*>(a.C),
                     (int)a.m, (int)a.n, (int)a.k, ks, part, counters);
  return hipGetLastError();
}

}  // namespace

// N, K multiples of 4; lane offsets of 16 k-rows of B and 64 rows of A below
// 2^32 bytes.  Up to 32 rows everywhere, above where B is large (us per launch,
// fresh operands, against the 64 x 64 tiles): M = 16 at N x K = 64 x 64 / 256 x
// 256 / 512 x 512 / 4096 x 4096 / 8192 x 8192 3.2 / 4.4 / 6.8 / 18.8 / 53.3
// against 3.3 / 7.2 / 8.8 / 30.5 / 97.6, M = 32 at 256 x 256 / 512 x 512 5.5 /
// 8.1 against 7.2 / 8.8; M = 48 at 512 x 512 / 1024 x 1024 / 1024 x 8192 8.4 /
// 11.6 / 20.6 against 8.9 / 10.4 / 24.8; M = 64 at 1024 x 1024 / 1024 x 4096 /
// 4096 x 4096 / 8192 x 8192 13.4 / 21.1 / 28.5 / 79 against 10.8 / 17.6 / 31.7 /
// 98.8.  What bounds the large ones is the read of B (16 x 8192 x 8192: 5.0
// TB/s), the small ones the launch and the pieces' hand-off.
// More than 32 rows are bound by the matrix cores, where a second column block on
// some of the CUs takes as long as one on all of them.  The 64 x 64 tiles (fewer
// 128 x 128 ones than CUs) do better there, and keep it: 56 x 18000 x 4096 205 us
// against 105, 64 x 21776 x 1572 83.6 / 49.3, 64 x 28000 x 512 28.0 / 20.7, 48 x
// 32000 x 2048 81 / 71; from the 128 x 128 tiles on they do not (48 x 32704 x 2048
// 82 / 128, 56 x 34000 x 512 36 / 64, 64 x 40000 x 4096 302 / 314).
// Where K is one to three of the tiles' whole 32-deep k-tiles, the waves have a
// step or two each and their sum is most of the time, so the tiles keep a grid of
// up to one column block per CU (two from 17 rows) and, for 64 rows, the largest
// ones: 32 x 16384 x 64 / 96 4.8 / 5.5 us against 4.4 / 4.9, 32 x 20000 x 64 6.8 /
// 5.5, 64 x 262144 x 64 56.3 / 51.6; but 16 x 20000 x 96 6.2 / 6.4, 32 x 32768 x 64
// 7.3 / 9.0, 64 x 262144 x 128 72 / 79.
bool f32_stream_takes(size_t m, size_t n, size_t k, int num_cus) {
  const size_t c = num_cus > 0 ? num_cus : 1, blocks = (n + kNC - 1) / kNC;
  if (m > 32 && (n * k < ((size_t)1 << 23) || (blocks > c && (n + 127) / 128 < c))) return false;
  if (k % 32 == 0 && m <= 32 && k <= 96 && (blocks <= c || (m > 16 && blocks < 2 * c))) return false;
  if (k % 32 == 0 && m > 56 && k <= 64) return false;
  return m >= 1 && m <= kMaxRows && n >= 4 && n % 4 == 0 && n < (1u << 25) && k >= 4 && k % 4 == 0 && k < (1u << 23);
}

int f32_stream_pieces(size_t m, size_t n, size_t k, size_t ws_limit, int num_cus) {
  return stream_pieces((n + kNC - 1) / kNC, (k + kKStep - 1) / kKStep, blocks_of(m), 1, ws_limit, num_cus);
}

hipError_t f32_stream_launch(const GemmArgs& a, size_t ws_limit) {
  switch (blocks_of(a.m)) {
    case 1: return launch_mb<1>(a, ws_limit);
    case 2: return launch_mb<2>(a, ws_limit);
    case 3: return launch_mb<3>(a, ws_limit);
    default: return launch_mb<4>(a, ws_limit);
  }
}

}  // namespace vk
