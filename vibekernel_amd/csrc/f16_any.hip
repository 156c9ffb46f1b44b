// f16_any.hip -- fp16 GEMM for any shape and any 2-byte alignment (version 1,
// and version 15's smaller products).
//
// Direct-to-LDS loads of 16 bytes need rows on 16-byte boundaries, N and K
// multiples of 8.  Global loads into registers take any address at nearly the
// aligned rate, so no padded copy of the operands is needed:
//  * 4 waves on a 64 x 64 tile (each 32 x 32, 128-deep k-tiles) or a 128 x 128
//    tile (64 x 64, 64-deep) of v_mfma_f32_16x16x32_f16;
//  * each thread loads 4 + 4 chunks of 16 bytes into registers two k-tiles
//    ahead; they land in one of two LDS buffers under the products of the
//    k-tile before theirs, one barrier per k-tile;
//  * LDS: chunk ^ f(row) so that the A fragment reads and the transposed B
//    reads of a pass are on distinct 16-byte slots, as in the kernels whose
//    tiles these are (f16_pp128.hip, f16_skinny_wk.hip, f16_pingpong.hip);
//  * a chunk past M or N is moved to row M - 1 or column 0 (its products are
//    not stored); one that N cuts short reads on into the next row, which
//    exists except at the end of B: in the last k-tile the chunks that K or N
//    cuts are loaded from 8 elements further back at most and shifted, zeros
//    past the edge in both operands (an operand whose rows are shorter than 8:
//    element by element);
//  * C goes straight from the registers, 32 bytes of a row at a time, or through
//    LDS in whole rows of a wave's block (launch_nb's rule).
// Measured (us per launch, fresh operands): version 1 before, whose 128 x 128
// tiles loaded element by element, 64 x 62 x 65 12.2, now 4.5; 100 x 300 x 70
// 15.9 / 5.5; 300 x 200 x 4095 950 / 28.7; 700 x 8191 x 2048 474 / 64.  A k-tile
// of the 64 x 64 tile takes 0.85 us where its products take 0.1: what bounds
// it is the wait for loads and barriers with one workgroup per CU, and large
// grids the LDS reads of its small wave blocks (4096 x 4095 x 4096 260 us).
// Every element is summed as version 10 does: k-tiles of 64 ascending, in
// each the 16 x 16 block (i, j) taking the 32-deep step (i ^ j) & 1 first, so
// the results are version 10's on zero-padded operands wherever that does not
// split K.
#include "vk_device.hpp"
#include "vk_internal.hpp"
#include "vk_tile.hpp"

#include <type_traits>

namespace vk {
namespace {

constexpr int kThreads = 256;

template <int NB>  // 64 NB x 64 NB tile, NB = 1 or 2
struct AnyCfg {
  static constexpr int kT = 64 * NB;              // tile rows and columns
  static constexpr int kBK = NB == 1 ? 128 : 64;  // k-tile depth
  static constexpr int kABytes = kT * kBK * 2;    // 16 KB, as B
  static constexpr int kChunksA = kBK / 8, kChunksB = kT / 8;  // 16-byte chunks per row
  static constexpr int kLd = kT * kBK / 8 / kThreads;          // chunks per thread and operand
  static constexpr int kBlocks = 2 * NB;          // 16 x 16 blocks of a wave, each way
  static_assert(kLd == 4, "whole chunks per thread");
  __device__ static constexpr int swz_a(int row) { return NB == 1 ? row & 15 : (row >> 1) & 7; }
  __device__ static constexpr int swz_b(int k) {
    return NB == 1 ? (((k >> 1) & 1) << 1) ^ (((k >> 3) & 1) << 2) : (2 * (k & 3)) ^ (((k >> 3) & 1) << 3);
  }
};

typedef uint32_t uint4u __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t uint2u __attribute__((ext_vector_type(2), aligned(2)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));

// 8 or 4 consecutive columns of C, `valid` of them inside the matrix.
__device__ __forceinline__ void store8(half_t* p, const uint4v& v, int64_t valid) {
  if (valid >= 8) {
    *reinterpret_cast<uint4u*>(p) = v;
  } else {
    const half8 h = __builtin_bit_cast(half8, v);
#pragma unroll
    for (int c = 0; c < 7; c++)
      if (c < valid) p[c] = h[c];
  }
}
__device__ __forceinline__ void store4(half_t* p, const float4v& v, int64_t valid) {
  const half4 h = {(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
  if (valid >= 4) {
    typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
    *reinterpret_cast<uint2u*>(p) = __builtin_bit_cast(uint2v, h);
  } else {
#pragma unroll
    for (int c = 0; c < 3; c++)
      if (c < valid) p[c] = h[c];
  }
}
__device__ __forceinline__ void store4(float* p, const float4v& v, int64_t valid) {
  if (valid >= 4) {
    *reinterpret_cast<float4u*>(p) = v;
  } else {
#pragma unroll
    for (int c = 0; c < 3; c++)
      if (c < valid) p[c] = v[c];
  }
}

// kNarrow: N or K below 8.  kRows: C in whole rows of the wave's block (fp16).
template <int NB, typename OutT, bool kNarrow, bool kRows>
__global__ __launch_bounds__(kThreads, 2) void f16_any_kernel(const half_t* __restrict__ A,
                                                              const half_t* __restrict__ B, OutT* __restrict__ C,
                                                              int64_t M, int64_t N, int64_t K, int tiles_m,
                                                              int tiles_n) {
  using G = AnyCfg<NB>;
  constexpr int T = G::kT, BK = G::kBK, L = G::kLd, NBk = G::kBlocks;
  __shared__ __attribute__((aligned(1024))) char lds[4 * G::kABytes];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int tm, tn;
  tile_of((int)(blockIdx.y * (unsigned)tiles_n + blockIdx.x), tiles_m, tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * T, n0 = (int64_t)tn * T;
  const uint32_t lbase = lds_addr32(lds);  // A of buffers 0, 1, then B of buffers 0, 1

  // Chunk i of this thread: 8 k of a row of A, 8 columns of a k-row of B.
  const half_t* pa[L];
  const half_t* pb[L];
  int ak[L], bk[L];       // first k of the A chunk, k-row of the B chunk
  int64_t bc[L];          // first column of the B chunk
  uint32_t wa[L], wb[L];  // LDS addresses in buffer 0
#pragma unroll
  for (int i = 0; i < L; i++) {
    const int id = tid + kThreads * i;
    const int row = id / G::kChunksA, ca = id % G::kChunksA;
    ak[i] = 8 * ca;
    pa[i] = A + (m0 + row < M ? m0 + row : M - 1) * K + ak[i];
    wa[i] = lbase + row * BK * 2 + 16 * (ca ^ G::swz_a(row));
    const int krow = id / G::kChunksB, cb = id % G::kChunksB;
    bk[i] = krow;
    bc[i] = n0 + 8 * cb;
    pb[i] = B + (int64_t)krow * N + (bc[i] < N ? bc[i] : 0);
    wb[i] = lbase + 2 * G::kABytes + krow * T * 2 + 16 * (cb ^ G::swz_b(krow));
  }
  struct Chunks {
    uint4v a[L], b[L];
  };
  Chunks set[2];
  const int64_t nk = (K + BK - 1) / BK;
  auto load_whole = [&](Chunks& r, int64_t t) {
#pragma unroll
    for (int i = 0; i < L; i++) r.a[i] = *reinterpret_cast<const uint4u*>(pa[i] + t * BK);
#pragma unroll
    for (int i = 0; i < L; i++) r.b[i] = *reinterpret_cast<const uint4u*>(pb[i] + t * BK * N);
  };
  // The 8 elements from p on, zeros from element `valid` on; the load is moved
  // back by what is missing, which the caller has checked to exist.
  auto load_cut = [&](const half_t* p, int64_t valid, const half_t* safe) {
    const int back = valid >= 8 ? 0 : valid <= 0 ? 8 : (int)(8 - valid);
    const uint4v v = *reinterpret_cast<const uint4u*>(back == 8 ? safe : p - back);
    const unsigned __int128 x = __builtin_bit_cast(unsigned __int128, v);
    return __builtin_bit_cast(uint4v, back == 8 ? (unsigned __int128)0 : x >> (16 * back));
  };
  auto load_elements = [&](const half_t* p, int64_t valid, const half_t* safe) {
    half8 h = {};
    if (valid <= 0) return __builtin_bit_cast(uint4v, h);  // most chunks, K or N below 8
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const half_t x = (e < valid ? p + e : safe)[0];
      h[e] = e < valid ? x : (half_t)0.0f;
    }
    return __builtin_bit_cast(uint4v, h);
  };
  auto load = [&](Chunks& r, int64_t t) {
    if (!kNarrow && (t < nk - 1 || (K % BK == 0 && N % 8 == 0))) {
      load_whole(r, t);
      return;
    }
    const int64_t left = K - t * BK;  // k of this k-tile
#pragma unroll
    for (int i = 0; i < L; i++) {
      const int64_t va = left - ak[i], vb = bk[i] < left ? N - bc[i] : 0;
      if constexpr (kNarrow) {
        const half_t *a = pa[i] + t * BK, *b = pb[i] + t * BK * N;
        r.a[i] = K < 8 ? load_elements(a, va, A) : load_cut(a, va, A);
        r.b[i] = N < 8 ? load_elements(b, vb, B) : load_cut(b, vb, B);
      } else {
        r.a[i] = load_cut(pa[i] + t * BK, va, A);
        r.b[i] = load_cut(pb[i] + t * BK * N, vb, B);
      }
    }
  };
  auto lds_put = [](uint32_t at, const uint4v& v) {
    *reinterpret_cast<__attribute__((address_space(3))) uint4v*>(at) = v;
  };
  auto store = [&](int buf, const Chunks& r) {
#pragma unroll
    for (int i = 0; i < L; i++) lds_put(wa[i] + buf * G::kABytes, r.a[i]);
#pragma unroll
    for (int i = 0; i < L; i++) lds_put(wb[i] + buf * G::kABytes, r.b[i]);
  };

  // Fragments (f16_skinny_sk.hip's layouts): A row l % 16, chunk 4 s + l / 16
  // of step s; B by transpose reads, lane 16g + 4jj + q naming k-row 8g + jj
  // (and + 4) of the step, columns 16j + 4q .. +3.
  const int wr = (wave >> 1) * 32 * NB, wc = (wave & 1) * 32 * NB;  // this wave's block
  const int g = lane >> 4, l16 = lane & 15;
  const int krow0 = 8 * g + ((lane >> 2) & 3), q4 = lane & 3;
  uint32_t ra[NBk], rb[NBk];  // rows of A; k-row krow0 of B with the block's chunk
#pragma unroll
  for (int i = 0; i < NBk; i++) ra[i] = lbase + (wr + 16 * i + l16) * BK * 2;
#pragma unroll
  for (int j = 0; j < NBk; j++)
    rb[j] = lbase + 2 * G::kABytes + krow0 * T * 2 + 16 * (((wc + 16 * j) / 8 + (q4 >> 1)) ^ G::swz_b(krow0)) +
            8 * (q4 & 1);
  float4v acc[NBk][NBk];
#pragma unroll
  for (int i = 0; i < NBk; i++)
#pragma unroll
    for (int j = 0; j < NBk; j++) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};

  struct Frags {
    half8 a[2][NBk], b[2][NBk];  // the 2 steps of 64 k
  };
  auto read = [&](Frags& f, int buf, int k64) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int ks = 2 * k64 + s;
#pragma unroll
      for (int i = 0; i < NBk; i++)
        f.a[s][i] = lds_read_h8(ra[i] + buf * G::kABytes + 16 * ((4 * ks + g) ^ G::swz_a(l16)));
#pragma unroll
      for (int j = 0; j < NBk; j++) {
        const uint32_t at = rb[j] + buf * G::kABytes + ks * 32 * T * 2;
        const half4 lo = lds_read_tr16_at(at), hi = lds_read_tr16_at(at + 4 * T * 2);
        f.b[s][j] = half8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    }
  };
  // `between` runs behind the first products, under the rest of them.
  auto multiply = [&](int buf, auto between) {
    Frags f[2];
    read(f[0], buf, 0);
#pragma unroll
    for (int h = 0; h < BK / 64; h++) {
      if (kNarrow && h > 0 && K <= 64 * h) break;
      if (h + 1 < BK / 64) read(f[(h + 1) & 1], buf, h + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 2; s++) {
#pragma unroll
        for (int i = 0; i < NBk; i++)
#pragma unroll
          for (int j = 0; j < NBk; j++) {
            const int k = s ^ ((i ^ j) & 1);
            acc[i][j] = mfma16x16x32(f[h & 1].b[k][j], f[h & 1].a[k][i], acc[i][j]);
          }
        if (h == 0 && s == 0) {
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
  if constexpr (!kNarrow)
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

  // Block (i, j), register r, lane l: row 16 i + l % 16, column 16 j + 4 (l / 16) + r.
  if constexpr (kRows) {
    // Through LDS, in units of 4 columns, unit ^ row.
    constexpr int kUnits = 8 * NB, kRow = 8 * kUnits;  // units and bytes per row of the block
    __syncthreads();  // every wave is done with the k-tiles
    const uint32_t base = lbase + wave * (32 * NB * kRow);
#pragma unroll
    for (int i = 0; i < NBk; i++)
#pragma unroll
      for (int j = 0; j < NBk; j++) {
        const int row = 16 * i + l16;
        const half4 h = {(half_t)acc[i][j][0], (half_t)acc[i][j][1], (half_t)acc[i][j][2], (half_t)acc[i][j][3]};
        lds_write8(base + row * kRow + 8 * ((4 * j + g) ^ (row & (kUnits - 1))), h);
      }
    constexpr int kLanes = kUnits / 2;  // per row, 8 columns each
#pragma unroll
    for (int q = 0; q < 32 * NB * kLanes / 64; q++) {
      const int row = q * (64 / kLanes) + lane / kLanes, c = lane % kLanes;
      const uint4v x = lds_read16(base + row * kRow + 16 * (c ^ ((row & (kUnits - 1)) >> 1)));
      const uint4v v = row & 1 ? uint4v{x[2], x[3], x[0], x[1]} : x;
      const int64_t r = m0 + wr + row, col = n0 + wc + 8 * c;
      if (r < M) store8(reinterpret_cast<half_t*>(C) + r * N + col, v, N - col);
    }
  } else {
#pragma unroll
    for (int i = 0; i < NBk; i++) {
      const int64_t row = m0 + wr + 16 * i + l16;
#pragma unroll
      for (int j = 0; j < NBk; j++) {
        const int64_t col = n0 + wc + 16 * j + 4 * g;
        if (row < M && col < N) store4(C + row * N + col, acc[i][j], N - col);
      }
    }
  }
}

template <int NB, typename OutT, bool kRows>
hipError_t launch_t(const GemmArgs& a) {
  const size_t tm = (a.m + AnyCfg<NB>::kT - 1) / AnyCfg<NB>::kT, tn = (a.n + AnyCfg<NB>::kT - 1) / AnyCfg<NB>::kT;
  auto kfn = a.n < 8 || a.k < 8 ? f16_any_kernel<NB, OutT, true, kRows> : f16_any_kernel<NB, OutT, false, kRows>;
  hipLaunchKernelGGL(kfn, dim3((unsigned)tn, (unsigned)tm), dim3(kThreads), 0, a.stream,
                     static_cast<const half_t*>(a.A), static_cast<const half_t*>(a.B), static_cast<OutT*>(a.C),
                     (int64_t)a.m, (int64_t)a.n, (int64_t)a.k, (int)tm, (int)tn);
  return hipGetLastError();
}

// An fp16 C with an odd number of columns leaves in whole rows of a wave's block
// where at least half of a tile's rows and more than half of its
// columns are there; straight from the registers a row gets 32 bytes at a time.  us
// per launch, rows / straight: 8192 x 8191 x 16 53.7 / 91.7, 4000 x 4001 x 1 15.2 /
// 21.2, 128 x 50001 x 65 11.6 / 14.0; 1 x 1048577 x 65 129.7 / 121.6; an even
// number 8192 x 8190 x 1 46 / 53, 50000 x 130 x 65 18.3 / 17.2, 3000 x 1500 x 193 14.3 /
// 13.5.  (Both in one kernel spill more: 1 x 1048577 x 65 131.3.)
template <int NB>
hipError_t launch_nb(const GemmArgs& a) {
  if (a.out_dtype != VK_DTYPE_F16) return launch_t<NB, float, false>(a);
  const bool rows = a.n % 2 != 0 && 2 * a.m >= (size_t)AnyCfg<NB>::kT && 2 * a.n > (size_t)AnyCfg<NB>::kT;
  return rows ? launch_t<NB, half_t, true>(a) : launch_t<NB, half_t, false>(a);
}

// grid.y, rows of 128-row tiles at least, holds up to 65535.
bool any_shape_ok(size_t m, size_t n, size_t k) {
  (void)n;
  (void)k;
  return (m + 127) / 128 <= 65535;
}

}  // namespace

// 64 x 64 tiles up to 4 per CU (us per launch, against 128 x 128): 1000 x 1001
// x 999 (256 tiles) 13.6 / 27.8, 300 x 11007 x 4096 (860) 92 / 113, 1000 x 4001
// x 1000 (1008) 30.4 / 29.8; 4096 x 4095 x 4096 (4096) 345 / 260.
hipError_t f16_any_launch(const GemmArgs& a) {
  const size_t c = a.num_cus > 0 ? a.num_cus : 1;
  const size_t small = (a.m + 63) / 64 * ((a.n + 63) / 64);
  // grid.y holds up to 65535 rows of tiles
  const bool use_small = small <= 4 * c && (a.m + 63) / 64 <= 65535;
  return use_small ? launch_nb<1>(a) : launch_nb<2>(a);
}

void register_f16_any() {
  KernelEntry e{};
  e.version = 1;
  e.in_dtype = VK_DTYPE_F16;
  e.name = "f16_v1_simple";
  e.caps = make_caps(1, VK_DTYPE_F16, kOutF16 | kOutF32, 1, 1, 1, 2, AnyCfg<2>::kT, AnyCfg<2>::kT, AnyCfg<2>::kBK,
                     kThreads, 4 * AnyCfg<2>::kABytes, 0, 0);
  e.launch = f16_any_launch;
  e.workspace = nullptr;
  e.shape_ok = any_shape_ok;
  register_kernel(e);
}

}  // namespace vk
