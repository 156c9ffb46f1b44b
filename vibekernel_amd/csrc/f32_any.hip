// f32_any.hip -- fp32 GEMM on the matrix cores for any shape and any 4-byte
// alignment, with version 1's sum: one fused multiply-add per term, k
// ascending (version 1's path off its asm kernel's grid).
//
// v_mfma_f32_16x16x4_f32 adds its four products to each accumulator one after
// the other, each with one rounding (measured on MI355X against fmaf chains,
// subnormal products included: equal bits, the lowest k first), so giving
// lane group g the k = 4s + g gives every element the bits of a vector-ALU
// loop at the matrix cores' rate.
//  * 8 waves on a 64 x 64 tile (each 32 x 16, 64-deep k-tiles) or, where
//    those need more rounds of the CUs, a 128 x 128 tile (64 x 32, 32-deep);
//    two waves per SIMD, since one alone waits out its LDS reads after each
//    barrier (4 waves of 32 x 32: 29.0 us instead of 26.4 at 1000 x 1001 x
//    999);
//  * rows of A and B start on any 4-byte boundary when K or N is odd, which
//    direct-to-LDS loads of 16 bytes do not take: each thread loads chunks of
//    16 bytes into registers two k-tiles ahead, which land in one of two LDS
//    buffers under the products of the k-tile before theirs, one barrier per
//    k-tile;
//  * LDS: A as four matrices, one per k % 4, so a lane's A values of 4 steps
//    are one 16-byte read (the rows and lane groups of a pass on distinct
//    16-byte slots); B rows as they are, column ^ 16 (k % 4), so the four lane
//    groups read distinct quarters of the banks;
//  * a chunk past M or N is moved to row M - 1 or column 0 (its products are
//    not stored); one that N cuts short reads on into the next row, which
//    exists except at the end of B: the last k-tile (or every one where N or
//    K is below 4) is loaded element by element where K or N cuts it, zeros
//    past K in both operands.
// Measured (us per launch, fresh operands, against the bounds-checked VALU
// kernels this replaced): 1000 x 1001 x 999 26.4 / 75.2, 500 x 510 x 512 14.8 /
// 35.7, 64 x 62 x 65 4.9 / 8.5, 16 x 4095 x 4096 79.6 / 269, 300 x 4095 x 4095
// 158 / 323, 2000 x 2001 x 2002 149 / 289, 4096 x 4095 x 4096 1100 / 1738 (125
// TFLOP/s).  What is left is the wait at each barrier: a k-tile of the 64 x 64
// tile takes 1.24 us where its products take 0.85.
#include "vk_device.hpp"
#include "vk_internal.hpp"
#include "vk_tile.hpp"

#include <algorithm>

namespace vk {
namespace {

constexpr int kThreads = 512;

template <int NB>  // 64 NB x 64 NB tile
struct AnyCfg {
  static constexpr int kT = 64 * NB;             // tile rows and columns
  static constexpr int kBK = NB == 1 ? 64 : 32;  // k-tile depth
  static constexpr int kPitchA = kBK / 4 + 4;    // floats per row of a quarter of A
  static constexpr int kQuarterA = kT * kPitchA;
  static constexpr int kLd = kT * kBK / 4 / kThreads;  // 16-byte chunks per thread and operand
  static constexpr int kChunksA = kBK / 4, kChunksB = kT / 4;
  static constexpr int kRB = 2 * NB, kCB = NB;   // 16 x 16 blocks of a wave: rows, columns
  static_assert(kLd * 4 * kThreads == kT * kBK, "whole chunks per thread");
  static_assert(kQuarterA % 64 == 0 && kPitchA % 8 == 4, "bank layout");
};

typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));

template <int NB>
__global__ __launch_bounds__(kThreads, NB == 1 ? 4 : 2) void f32_any_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                              float* __restrict__ C, int64_t M, int64_t N, int64_t K,
                                                              int tiles_m, int tiles_n) {
  using G = AnyCfg<NB>;
  constexpr int T = G::kT, BK = G::kBK, P = G::kPitchA, L = G::kLd, RB = G::kRB, CB = G::kCB;
  __shared__ __attribute__((aligned(16))) float As[2][4 * G::kQuarterA];
  __shared__ __attribute__((aligned(16))) float Bs[2][BK * T];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, l16 = lane & 15;
  const int id = (int)(blockIdx.y * gridDim.x + blockIdx.x);
  if (id >= tiles_m * tiles_n) return;  // the last row of a folded grid
  int tm, tn;
  tile_of(id, tiles_m, tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * T, n0 = (int64_t)tn * T;

  // Chunk i of this thread: 4 k of a row of A, 4 columns of a k-row of B.
  const float* pa[L];
  const float* pb[L];
  int ak[L], bk[L];         // first k of the A chunk, k-row of the B chunk
  int64_t bc[L];            // first column of the B chunk
  uint32_t wa[L], wb[L];    // LDS offsets (floats)
#pragma unroll
  for (int i = 0; i < L; i++) {
    const int ia = tid + kThreads * i;
    const int row = ia / G::kChunksA, kc = ia % G::kChunksA;
    ak[i] = 4 * kc;
    pa[i] = A + (m0 + row < M ? m0 + row : M - 1) * K + ak[i];
    wa[i] = row * P + kc;
    const int krow = ia / G::kChunksB, c = ia % G::kChunksB;
    bk[i] = krow;
    bc[i] = n0 + 4 * c;
    pb[i] = B + (int64_t)krow * N + (bc[i] < N ? bc[i] : 0);
    wb[i] = krow * T + ((4 * c) ^ (16 * (krow & 3)));
  }
  struct Chunks {
    float4v a[L], b[L];
  };
  Chunks set[2];
  const int64_t nk = (K + BK - 1) / BK;
  const bool narrow = N < 4 || K < 4;
  auto load_whole = [&](Chunks& r, int64_t t) {
#pragma unroll
    for (int i = 0; i < L; i++) r.a[i] = *reinterpret_cast<const float4u*>(pa[i] + t * BK);
#pragma unroll
    for (int i = 0; i < L; i++) r.b[i] = *reinterpret_cast<const float4u*>(pb[i] + t * BK * N);
  };
  auto load = [&](Chunks& r, int64_t t) {
    if (narrow || (t == nk - 1 && (K % BK != 0 || N % 4 != 0))) {
      const int64_t left = K - t * BK;  // k of this k-tile
#pragma unroll
      for (int i = 0; i < L; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const bool in_a = ak[i] + q < left, in_b = bk[i] < left && bc[i] + q < N;
          const float va = (in_a ? pa[i] + t * BK + q : A)[0], vb = (in_b ? pb[i] + t * BK * N + q : B)[0];
          r.a[i][q] = in_a ? va : 0.0f;
          r.b[i][q] = in_b ? vb : 0.0f;
        }
    } else {
      load_whole(r, t);
    }
  };
  auto store = [&](int buf, const Chunks& r) {
#pragma unroll
    for (int i = 0; i < L; i++) {
#pragma unroll
      for (int q = 0; q < 4; q++) As[buf][q * G::kQuarterA + wa[i]] = r.a[i][q];
      *reinterpret_cast<float4v*>(&Bs[buf][wb[i]]) = r.b[i];
    }
  };

  const int wr = (wave >> 2) * 16 * RB, wc = (wave & 3) * 16 * CB;  // this wave's block
  float4v acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; i++)
#pragma unroll
    for (int j = 0; j < CB; j++) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};

  // Fragments of 4 steps (16 k) of a k-tile; the reads of the next ones go out
  // ahead of the products of these.
  struct Frags {
    float4v a[RB];
    float b[CB][4];
  };
  auto read = [&](Frags& f, int buf, int q) {
#pragma unroll
    for (int i = 0; i < RB; i++)
      f.a[i] = *reinterpret_cast<const float4v*>(&As[buf][g * G::kQuarterA + (wr + 16 * i + l16) * P + 4 * q]);
#pragma unroll
    for (int j = 0; j < CB; j++)
#pragma unroll
      for (int s = 0; s < 4; s++) f.b[j][s] = Bs[buf][(16 * q + 4 * s + g) * T + ((wc + 16 * j + l16) ^ (16 * g))];
  };
  // `between` runs behind the first products, under the rest of them.
  auto multiply = [&](int buf, auto between) {
    Frags f[2];
    read(f[0], buf, 0);
#pragma unroll
    for (int q = 0; q < BK / 16; q++) {
      if (q + 1 < BK / 16) read(f[(q + 1) & 1], buf, q + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 4; s++) {
#pragma unroll
        for (int i = 0; i < RB; i++)
#pragma unroll
          for (int j = 0; j < CB; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[q & 1].a[i][s], f[q & 1].b[j][s], acc[i][j], 0, 0, 0);
        if (q == 0 && s == 1) {
          __builtin_amdgcn_sched_barrier(0);
          between();
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // K-tile t is multiplied from LDS buffer t % 2 while tile t + 1 waits in
  // registers and t + 2 is loaded.
  load(set[0], 0);
  if (nk > 1) load(set[1], 1);
  store(0, set[0]);
  __syncthreads();
  int64_t t = 0;
  auto phase = [&](auto odd, int64_t t) {
    constexpr int p = decltype(odd)::value;
    load_whole(set[p], t + 2);
    __builtin_amdgcn_sched_barrier(0);  // the loads go out before the products
    multiply(p, [&] { store(p ^ 1, set[p ^ 1]); });
    __syncthreads();
  };
  if (!narrow)
    for (; t + 4 < nk; t += 2) {  // tiles t + 2 and t + 3 are not the last
      phase(std::integral_constant<int, 0>{}, t);
      phase(std::integral_constant<int, 1>{}, t + 1);
    }
  for (; t < nk; t += 2) {
    if (t + 2 < nk) load(set[0], t + 2);
    multiply(0, [&] {
      if (t + 1 < nk) store(1, set[1]);
    });
    if (t + 1 < nk) {
      __syncthreads();
      if (t + 3 < nk) load(set[1], t + 3);
      multiply(1, [&] {
        if (t + 2 < nk) store(0, set[0]);
      });
      __syncthreads();
    }
  }

  // Block (i, j), register r, lane l: row 4 (l / 16) + r, column l % 16.
#pragma unroll
  for (int i = 0; i < RB; i++)
#pragma unroll
    for (int j = 0; j < CB; j++) {
      const int64_t col = n0 + wc + 16 * j + l16;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int64_t row = m0 + wr + 16 * i + 4 * g + r;
        if (row < M && col < N) C[row * N + col] = acc[i][j][r];
      }
    }
}

template <int NB>
hipError_t launch_any(const GemmArgs& a) {
  const size_t tm = (a.m + AnyCfg<NB>::kT - 1) / AnyCfg<NB>::kT, tn = (a.n + AnyCfg<NB>::kT - 1) / AnyCfg<NB>::kT;
  // A row of tiles per grid.y, or, where that is too wide, the tiles in rows as
  // wide as a grid may be (fewer than 2^32 threads).
  const size_t gx = std::min(tn, (((size_t)1 << 32) - 1) / kThreads), gy = gx == tn ? tm : (tm * tn + gx - 1) / gx;
  hipLaunchKernelGGL(f32_any_kernel<NB>, dim3((unsigned)gx, (unsigned)gy), dim3(kThreads), 0, a.stream,
                     static_cast<const float*>(a.A), static_cast<const float*>(a.B), static_cast<float*>(a.C),
                     (int64_t)a.m, (int64_t)a.n, (int64_t)a.k, (int)tm, (int)tn);
  return hipGetLastError();
}

}  // namespace

// The 128 x 128 tiles, four times the work each, where they need no more
// rounds of the CUs for it.
hipError_t f32_any_launch(const GemmArgs& a) {
  const size_t c = a.num_cus > 0 ? a.num_cus : 1;
  const size_t big = (a.m + 127) / 128 * ((a.n + 127) / 128), small = (a.m + 63) / 64 * ((a.n + 63) / 64);
  // grid.y holds up to 65535 rows of tiles
  const bool use_small = 4 * ((big + c - 1) / c) > (small + c - 1) / c && (a.m + 63) / 64 <= 65535;
  return use_small ? launch_any<1>(a) : launch_any<2>(a);
}

}  // namespace vk
