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
//    exists except at the end of B: in the last k-tile (or every one where N is
//    below 4) what K or N cuts is loaded element by element, zeros past K in both
//    operands;
//  * small K on the 64 x 64 tile, where the loop's two k-tiles of preparation and
//    its 73 KB of LDS are most of the time, has instances of its own: K up to 32
//    and up to 64 in one LDS buffer (8 and 4 workgroups per CU), up to 128 in two
//    k-tiles, each chunk one load, and only the products that are of use; so has
//    any K with N below 4.
// Measured (us per launch, fresh operands, against the bounds-checked VALU
// kernels this replaced): 1000 x 1001 x 999 26.4 / 75.2, 500 x 510 x 512 14.8 /
// 35.7, 64 x 62 x 65 4.9 / 8.5, 16 x 4095 x 4096 79.6 / 269, 300 x 4095 x 4095
// 158 / 323, 2000 x 2001 x 2002 149 / 289, 4096 x 4095 x 4096 1100 / 1738 (125
// TFLOP/s).  What is left is the wait at each barrier: a k-tile of the 64 x 64
// tile takes 1.24 us where its products take 0.85.  Small K, also against the loop
// of any K: 1 x 4194304 x 16 190 / 235 / 583, x 65 552 / 657 / 800, 262143 x 64 x 16
// 21 / 35 / 44, x 65 52 / 61 / 64, 4095 x 4097 x 33 35 / 51 / 45, 262144 x 3 x 256
// 106 / 126 / 140, 262144 x 1 x 1000 344 / 499 / 513.
#include "vk_device.hpp"
#include "vk_internal.hpp"
#include "vk_tile.hpp"

#include <algorithm>

namespace vk {
namespace {

constexpr int kThreads = 512;

// 64 NB x 64 NB tile, kDeep-deep k-tiles; kTiles: K is 1 or 2 of them at most (1
// in one LDS buffer); 0: any number; kTall: any number, N below 4.
constexpr int kTall = 3;
template <int NB, int kDeep, int kTiles>
struct AnyCfg {
  static constexpr int kT = 64 * NB;             // tile rows and columns
  static constexpr int kBK = kDeep;              // k-tile depth
  static constexpr int kBufs = kTiles == 1 ? 1 : 2;
  static constexpr int kPitchA = kBK / 4 + 4;    // floats per row of a quarter of A
  static constexpr int kQuarterA = kT * kPitchA;
  static constexpr int kLd = kT * kBK / 4 / kThreads;  // 16-byte chunks per thread and operand
  static constexpr int kChunksA = kBK / 4, kChunksB = kT / 4;
  static constexpr int kRB = 2 * NB, kCB = NB;   // 16 x 16 blocks of a wave: rows, columns
  static_assert(kLd * 4 * kThreads == kT * kBK, "whole chunks per thread");
  static_assert(kQuarterA % 64 == 0 && kPitchA % 8 == 4, "bank layout");
};

typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));

// A chunk of 4 elements of which its row has `valid` from p on: cut_load loads
// it, moved back to end with the row, or from `safe` where the row has none of
// it (kShort: a row of fewer than 4, element by element), and cut_fix moves the
// values into place, zeros from the row's end on.
template <bool kShort>
__device__ __forceinline__ float4v cut_load(const float* p, int64_t valid, const float* safe) {
  float4v v;
  if constexpr (kShort) {
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = (q < valid ? p + q : safe)[0];
  } else {
    v = *reinterpret_cast<const float4u*>(valid >= 4 ? p : valid <= 0 ? safe : p - (4 - valid));
  }
  return v;
}
template <bool kShort>
__device__ __forceinline__ float4v cut_fix(const float4v& v, int64_t valid) {
  float4v r;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    r[q] = q < valid ? v[q] : 0.0f;
    if constexpr (!kShort)
#pragma unroll
      for (int b = 1; q + b < 4; b++) r[q] = valid == 4 - b ? v[q + b] : r[q];
  }
  return r;
}

template <int NB, int kDeep, int kTiles>
__global__ __launch_bounds__(kThreads, NB == 1 ? 4 : 2) void f32_any_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                              float* __restrict__ C, int64_t M, int64_t N, int64_t K,
                                                              int tiles_m, int tiles_n, int grid_x) {
  using G = AnyCfg<NB, kDeep, kTiles>;
  constexpr int T = G::kT, BK = G::kBK, P = G::kPitchA, L = G::kLd, RB = G::kRB, CB = G::kCB;
  __shared__ __attribute__((aligned(16))) float As[G::kBufs][4 * G::kQuarterA];
  __shared__ __attribute__((aligned(16))) float Bs[G::kBufs][BK * T];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, l16 = lane & 15;
  const int id = (int)(blockIdx.y * (unsigned)grid_x + blockIdx.x);
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
  // K-tile t holds chunks of A or B that K or N cuts.
  const bool short_a = kTiles == 1 && K < 4, short_b = kTiles == kTall || (kTiles != 0 && N < 4);
  auto cut_a = [&](int64_t t) { return short_a || (t == nk - 1 && K % BK != 0); };
  auto cut_b = [&](int64_t t) { return short_b || (t == nk - 1 && (K % BK != 0 || N % 4 != 0)); };
  auto valid_a = [&](int i, int64_t t) { return K - t * BK - ak[i]; };
  auto valid_b = [&](int i, int64_t t) { return bk[i] < K - t * BK ? N - bc[i] : 0; };
  auto load = [&](Chunks& r, int64_t t) {
    if constexpr (kTiles == 0) {
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
      return;
    }
    const bool ca = cut_a(t), cb = cut_b(t);
#pragma unroll
    for (int i = 0; i < L; i++) {
      const float* p = pa[i] + t * BK;
      if (!ca)
        r.a[i] = *reinterpret_cast<const float4u*>(p);
      else
        r.a[i] = short_a ? cut_load<true>(p, valid_a(i, t), A) : cut_load<false>(p, valid_a(i, t), A);
    }
#pragma unroll
    for (int i = 0; i < L; i++) {
      const float* p = pb[i] + t * BK * N;
      if (!cb)
        r.b[i] = *reinterpret_cast<const float4u*>(p);
      else
        r.b[i] = short_b ? cut_load<true>(p, valid_b(i, t), B) : cut_load<false>(p, valid_b(i, t), B);
    }
  };
  // Before a cut k-tile is stored (not when it is loaded: that would wait for
  // the loads).
  auto fix = [&](Chunks& r, int64_t t) {
    if constexpr (kTiles == 0) return;
    if (cut_a(t))
#pragma unroll
      for (int i = 0; i < L; i++)
        r.a[i] = short_a ? cut_fix<true>(r.a[i], valid_a(i, t)) : cut_fix<false>(r.a[i], valid_a(i, t));
    if (cut_b(t))
#pragma unroll
      for (int i = 0; i < L; i++)
        r.b[i] = short_b ? cut_fix<true>(r.b[i], valid_b(i, t)) : cut_fix<false>(r.b[i], valid_b(i, t));
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
  // `between` runs behind the first products, under the rest of them.  kTiles:
  // products of no use are left out: 16-deep groups past the `left` k of a k-tile,
  // blocks past M or N (the branches cost a long k-loop 4 per cent).
  const bool idle = m0 + wr >= M || n0 + wc >= N;
  const int blocks = m0 + wr + 16 >= M ? 1 : RB;  // (RB = 2 with kTiles)
  auto multiply = [&](int buf, int64_t left, auto between) {
    if (kTiles != 0 && idle) {
      between();
      return;
    }
    Frags f[2];
    read(f[0], buf, 0);
#pragma unroll
    for (int q = 0; q < BK / 16; q++) {
      if (kTiles != 0 && q > 0 && 16 * q >= left) break;
      if (q + 1 < BK / 16) read(f[(q + 1) & 1], buf, q + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 4; s++) {
#pragma unroll
        for (int i = 0; i < RB; i++)
#pragma unroll
          for (int j = 0; j < CB; j++)
            if (kTiles == 0 || i < blocks)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[q & 1].a[i][s], f[q & 1].b[j][s], acc[i][j], 0, 0, 0);
        if (q == 0 && s == 1) {
          __builtin_amdgcn_sched_barrier(0);
          between();
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  load(set[0], 0);
  if (kTiles != 1 && nk > 1) load(set[1], 1);
  fix(set[0], 0);
  store(0, set[0]);
  __syncthreads();
  if constexpr (kTiles == 1) {
    multiply(0, K, [] {});
  } else if constexpr (kTiles == 2) {
    multiply(0, BK, [&] {
      fix(set[1], 1);
      store(1, set[1]);
    });
    __syncthreads();
    multiply(1, K - BK, [] {});
  } else {
    // K-tile t is multiplied from LDS buffer t % 2 while tile t + 1 waits in
    // registers and t + 2 is loaded.
    int64_t t = 0;
    auto phase = [&](auto odd, int64_t t) {
      constexpr int p = decltype(odd)::value;
      load_whole(set[p], t + 2);
      __builtin_amdgcn_sched_barrier(0);  // the loads go out before the products
      multiply(p, BK, [&] { store(p ^ 1, set[p ^ 1]); });
      __syncthreads();
    };
    if (!narrow)
      for (; t + 4 < nk; t += 2) {  // tiles t + 2 and t + 3 are not the last
        phase(std::integral_constant<int, 0>{}, t);
        phase(std::integral_constant<int, 1>{}, t + 1);
      }
    for (; t < nk; t += 2) {
      if (t + 2 < nk) load(set[0], t + 2);
      multiply(0, BK, [&] {
        if (t + 1 < nk) {
          fix(set[1], t + 1);
          store(1, set[1]);
        }
      });
      if (t + 1 < nk) {
        __syncthreads();
        if (t + 3 < nk) load(set[1], t + 3);
        multiply(1, BK, [&] {
          if (t + 2 < nk) {
            fix(set[0], t + 2);
            store(0, set[0]);
          }
        });
        __syncthreads();
      }
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

template <int NB, int kDeep, int kTiles>
hipError_t launch_any(const GemmArgs& a) {
  constexpr int T = AnyCfg<NB, kDeep, kTiles>::kT;
  const size_t tm = (a.m + T - 1) / T, tn = (a.n + T - 1) / T;
  // A row of tiles per grid.y, or, where that is too wide, the tiles in rows as
  // wide as a grid may be (fewer than 2^32 threads).
  const size_t gx = std::min(tn, (((size_t)1 << 32) - 1) / kThreads), gy = gx == tn ? tm : (tm * tn + gx - 1) / gx;
  hipLaunchKernelGGL((f32_any_kernel<NB, kDeep, kTiles>), dim3((unsigned)gx, (unsigned)gy), dim3(kThreads), 0, a.stream,
                     static_cast<const float*>(a.A), static_cast<const float*>(a.B), static_cast<float*>(a.C),
                     (int64_t)a.m, (int64_t)a.n, (int64_t)a.k, (int)tm, (int)tn, (int)gx);
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
  if (!use_small) return launch_any<2, 32, 0>(a);
  if (a.k <= 32) return launch_any<1, 32, 1>(a);
  if (a.k <= 64) return launch_any<1, 64, 1>(a);
  if (a.k <= 128) return launch_any<1, 64, 2>(a);
  return a.n < 4 ? launch_any<1, 64, kTall>(a) : launch_any<1, 64, 0>(a);
}

}  // namespace vk
