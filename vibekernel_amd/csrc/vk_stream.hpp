// vk_stream.hpp -- what the few-row streaming kernels (f16_stream.hip,
// f32_stream.hip) share: the waves' and workgroups' sums of a column block and
// the plan of the K split.
//
// A wave holds 16 MB rows x (16 lanes x 4 H columns): acc[r][c], element e of
// lane l is row 16 r + 4 (l / 16) + e, column 4 H (l % 16) + c.  The 4 waves of
// a workgroup have summed consecutive ranges of K, and so have the ks
// workgroups of a column block.
#pragma once

#include "vk_device.hpp"
#include "vk_internal.hpp"

namespace vk {

constexpr int kStreamWaves = 4;
constexpr int kStreamMaxPieces = 32;
constexpr size_t kStreamCounterBytes = 8192;  // a counter per (block, wave)

// Workgroups per block: doubled while the grid stays within one per CU and
// every wave keeps at least 4 k-steps.  (Two per CU: 16 x 4096 x 4096
// fp32 27.0 us instead of 24.1, 16 x 4095 x 4096 fp16 25.9 instead of 16.8.)
// The pieces of a block belong on different XCDs: dealt next to each other
// these two took 24.1 and 16.8 us, spread 19.1 and 13.7.
// The counters and a slot of 4 waves x mb h KB per piece (mb row blocks, h
// groups of 4 columns per lane) stay within ws_limit bytes.
inline int stream_pieces(size_t blocks, size_t steps, int mb, int h, size_t ws_limit, int num_cus) {
  const size_t slot = (size_t)kStreamWaves * mb * h * 1024;
  int ks = 1;
  if (blocks * kStreamWaves * sizeof(unsigned) > kStreamCounterBytes) return 1;
  while (ks < kStreamMaxPieces && blocks * ks * 2 <= (size_t)num_cus && steps / (ks * 2) >= 4 * kStreamWaves &&
         kStreamCounterBytes + blocks * ks * 2 * slot <= ws_limit)
    ks *= 2;
  return ks;
}

// The workspace of ks pieces: the counters, cleared unless they are known to be
// zero, then the partial slots.  One piece touches nothing there
// (kWorkspaceUntouched), so its call is no word on the counters either.
inline hipError_t stream_buffers(const GemmArgs& a, int ks, unsigned*& counters, float*& part) {
  if (ks == 1) return hipSuccess;
  counters = static_cast<unsigned*>(a.workspace);
  part = reinterpret_cast<float*>(static_cast<char*>(a.workspace) + kStreamCounterBytes);
  return a.workspace_clean ? hipSuccess : zero_words(counters, kStreamCounterBytes / 4, a.stream);
}

// Adds the waves' sums and then the pieces', both in k order, and calls
// store_c(r, x) for each row block: x is row 16 r + 4 (lane / 16) + wave, the
// lane's 4 H columns.  slot0: this block's first slot of `slots`, ks each.
template <int MB, int H, typename Store>
__device__ __forceinline__ void stream_finish(const float4v (&acc)[MB][4 * H], int lane, int wave, int ks, int kp,
                                              int slot0, int slots, float* part, unsigned* counters,
                                              const Store& store_c) {
  constexpr int W = kStreamWaves;
  // Two row blocks at a time through LDS: per wave 8 H pieces of 1 KB
  // (2 blocks x 4 rows x H groups of 4 columns, 16 bytes per lane); wave q
  // keeps row 4g + q of each block.
  constexpr int kPair = 2;
  __shared__ float4v lds[W][kPair * 4 * H][64];
  float4v red[MB][H];
#pragma unroll
  for (int r0 = 0; r0 < MB; r0 += kPair) {
    if (r0) __syncthreads();
#pragma unroll
    for (int i = 0; i < kPair; i++)
      if (r0 + i < MB)
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int h = 0; h < H; h++)
            lds[wave][(i * 4 + e) * H + h][lane] = float4v{acc[r0 + i][4 * h][e], acc[r0 + i][4 * h + 1][e],
                                                           acc[r0 + i][4 * h + 2][e], acc[r0 + i][4 * h + 3][e]};
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPair; i++)
      if (r0 + i < MB)
#pragma unroll
        for (int h = 0; h < H; h++) {
          float4v t = lds[0][(i * 4 + wave) * H + h][lane];
#pragma unroll
          for (int w = 1; w < W; w++) t += lds[w][(i * 4 + wave) * H + h][lane];
          red[r0 + i][h] = t;
        }
  }
  if (ks == 1) {
#pragma unroll
    for (int r = 0; r < MB; r++) store_c(r, red[r]);
    return;
  }
  // K split over workgroups, as in f16_skinny_wk.hip: slot (block, piece)
  // holds 4 wave regions of MB H KB; a wave that finds every other piece in
  // memory is the last and sums them in k order, its own from registers.
  constexpr uint32_t kWaveRegion = MB * H * 1024;
  constexpr uint32_t kSlotBytes = W * kWaveRegion;
  const __amdgpu_buffer_rsrc_t prs =
      __builtin_amdgcn_make_buffer_rsrc(part, 0, (int)((uint32_t)slots * kSlotBytes), kBufferWord3);
  auto soff = [&](int q) { return (uint32_t)(slot0 + q) * kSlotBytes + (uint32_t)wave * kWaveRegion; };
  const uint32_t vlane = (uint32_t)lane * 16;
  unsigned* cnt = counters + slot0 / ks * W + wave;
  const unsigned seen =
      __builtin_amdgcn_readfirstlane(__hip_atomic_load(cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  if (seen != (unsigned)(ks - 1)) {
#pragma unroll
    for (int r = 0; r < MB; r++)
#pragma unroll
      for (int h = 0; h < H; h++) store_partial(prs, vlane + (H * r + h) * 1024, soff(kp), red[r][h]);
    wait_vmcnt0_ordered();  // the partial is in memory before the counter moves
    unsigned old = 0;
    if (lane == 0) old = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(old) != (unsigned)(ks - 1)) return;
  }
  asm volatile("" ::: "memory");  // the other pieces are read after the counter
  // P pieces of RB row blocks at a time (up to 32 loads in flight); a piece
  // past ks reads the last one's slot and is not added.
  auto fold = [&](auto pieces) {
    constexpr int P = decltype(pieces)::value;
    constexpr int RB = 16 / P < MB ? 16 / P : MB;
#pragma unroll
    for (int r0 = 0; r0 < MB; r0 += RB) {
      float4v t[RB][H];
      for (int q0 = 0; q0 < ks; q0 += P) {
        float4v x[P][RB][H];
#pragma unroll
        for (int q = 0; q < P; q++)
#pragma unroll
          for (int i = 0; i < RB; i++)
#pragma unroll
            for (int h = 0; h < H; h++)
              if (r0 + i < MB)
                x[q][i][h] = load_partial(prs, vlane + (H * (r0 + i) + h) * 1024, soff(min(q0 + q, ks - 1)));
#pragma unroll
        for (int q = 0; q < P; q++)
          if (q0 + q < ks)
#pragma unroll
            for (int i = 0; i < RB; i++)
#pragma unroll
              for (int h = 0; h < H; h++)
                if (r0 + i < MB) {
                  const float4v v = q0 + q == kp ? red[r0 + i][h] : x[q][i][h];
                  t[i][h] = q0 + q == 0 ? v : t[i][h] + v;
                }
      }
#pragma unroll
      for (int i = 0; i < RB; i++)
        if (r0 + i < MB) store_c(r0 + i, t[i]);
    }
  };
  if (ks == 2)
    fold(std::integral_constant<int, 2>{});
  else if (ks == 4)
    fold(std::integral_constant<int, 4>{});
  else
    fold(std::integral_constant<int, 8>{});
  if (lane == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace vk
