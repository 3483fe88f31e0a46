// mm_f32.hip -- fp32 out[M,N] = lhsT[K,M]^T . rhs[K,N] (benchmark config C1).
//
// This is the fp32 semantics the reference checks every kernel against
// (simulate_fp32 rewrites all dtypes to fp32;
// reference nkigym/src/nkigym/synthesis/simulate_nki.py:24-48).  Variant 0
// is a parity path, not a throughput path: an LDS-tiled FMA kernel with the
// K sum in plain sequential order.  lhsT rows are M-contiguous, so a K slice
// of both operands is an outer product of two contiguous vectors and needs
// no transpose.  Variants 1 and 3 below run on the fp32 MFMA; variant 3 is
// the default wherever its 32-bit offsets reach.
#include "mi_registry.hpp"

namespace mi {

template <int BM, int BN, int BK>
__global__ __launch_bounds__(256) void mm_f32_kernel(const float* __restrict__ lhsT, const float* __restrict__ rhs,
                                                     float* __restrict__ out, int M, int N, int K) {
  static_assert(BM == 64 && BN == 64, "16x16 threads, 4x4 outputs each");
  __shared__ float As[BK][BM + 1];
  __shared__ float Bs[BK][BN + 1];
  const int tid = (int)threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  const int tiles_n = (N + BN - 1) / BN;
  const int m0 = ((int)blockIdx.x / tiles_n) * BM;
  const int n0 = ((int)blockIdx.x % tiles_n) * BN;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.0f;

  for (int k0 = 0; k0 < K; k0 += BK) {
    for (int i = tid; i < BK * BM; i += 256) {
      const int kk = i / BM, mm = i % BM;
      const int k = k0 + kk, m = m0 + mm;
      As[kk][mm] = (k < K && m < M) ? lhsT[(size_t)k * M + m] : 0.0f;
    }
    for (int i = tid; i < BK * BN; i += 256) {
      const int kk = i / BN, nn = i % BN;
      const int k = k0 + kk, n = n0 + nn;
      Bs[kk][nn] = (k < K && n < N) ? rhs[(size_t)k * N + n] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < BK; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][ty + 16 * i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx + 16 * j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty + 16 * i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx + 16 * j;
      if (n < N) out[(size_t)m * N + n] = acc[i][j];
    }
  }
}

// Variant 1: the same product on the fp32 MFMA (v_mfma_f32_32x32x2_f32).
// Four waves in a 2 x 2 grid, each a (BM/2) x (BN/2) block of 32x32 MFMA
// tiles.  An fp32 MFMA takes 2 K values per lane (lane l: K row l/32 of the
// step, column l%32), so its operands are read straight from the K-major
// inputs, each lane one 4-byte element and each half-wave one 128-byte row
// segment, with no LDS and no transpose: lhsT[k][m] is the second MFMA
// operand (output column m = lane%32), rhs[k][n] the first (output rows n),
// so a lane ends with 4 consecutive n of one output row per dword quad.
// Each loop step loads U K pairs for every fragment first, then runs their
// MFMAs.  The MFMA adds its two products and the accumulator in one step,
// so the K sum is in a different order from variant 0's sequential one
// (fp32 rounding differences only).  Any M, N, K: loads past an edge read
// 0, stores past an edge are skipped.
template <int BM, int BN>
__global__ __launch_bounds__(256) void mm_f32_mfma_kernel(const float* __restrict__ lhsT,
                                                          const float* __restrict__ rhs, float* __restrict__ out,
                                                          int M, int N, int K) {
  constexpr int TM = BM / 64, TN = BN / 64, U = 8;
  static_assert(BM % 64 == 0 && BN % 64 == 0, "2 x 2 waves of 32x32 MFMA tiles");
  const int tid = (int)threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int tiles_n = (N + BN - 1) / BN;
  const int m0 = ((int)blockIdx.x / tiles_n) * BM + (wave >> 1) * (BM / 2);
  const int n0 = ((int)blockIdx.x % tiles_n) * BN + (wave & 1) * (BN / 2);
  const int kr = lane >> 5, c = lane & 31;
  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x16_t{};
  for (int k0 = 0; k0 < K; k0 += 2 * U) {
    float a[U][TM], b[U][TN];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 2 * u + kr;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int m = m0 + 32 * i + c;
        a[u][i] = (k < K && m < M) ? lhsT[(size_t)k * M + m] : 0.0f;
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + 32 * j + c;
        b[u][j] = (k < K && n < N) ? rhs[(size_t)k * N + n] : 0.0f;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[u][j], a[u][i], acc[i][j], 0, 0, 0);
  }
  // Lane l holds output row m = m0 + 32i + l%32 and, for quad q, columns
  // n0 + 32j + 8q + 4*(l/32) + 0..3 in acc[i][j][4q .. 4q+3].
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + 32 * i + c;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = n0 + 32 * j + 8 * q + 4 * kr + r;
          if (n < N) out[(size_t)m * N + n] = acc[i][j][4 * q + r];
        }
  }
}

// Variant 3: the fp32 MFMA with K split over the waves of a workgroup.
// Every wave computes the whole BM x BN block over its own K chunks of BK
// rows (chunk c goes to wave c % WAVES), straight from global memory into
// registers, one chunk's loads in flight while the MFMAs run on
// the chunk before; the waves' blocks are then added in wave order through
// LDS and stored as whole rows.
//
// Bound: the fp32 MFMA rate (157 TFLOP/s at 2.4 GHz) where tiles fill the
// chip, the latency of the loads where they do not.  An MFMA runs 64 cycles
// on 512 bytes of operands (half as many where a wave's 2x2 fragments share
// them), 4 to 8 bytes a cycle and SIMD, so neither LDS nor L1 is near its
// limit and the operands need no LDS.  Variant 1 waits for every chunk it
// loads and gives a tile one chain of K / 2 MFMAs; here the loads run a
// chunk ahead, and the chain of a tile is spread over WAVES waves of the CU
// that holds it, so a small block, of which there are enough for every CU,
// is not a long chain.
// Measured in graphs of back-to-back calls, variant 1 -> 3: 256x512x512
// (M, N, K) 27.0 -> 4.7 us, 1000x1501x777 60.9 -> 25.3 us (90 TFLOP/s),
// 128x4072x4015 225 -> 39 us, 64x64x4096 224 -> 8.2 us, 2048^3 240 -> 130 us
// (132 TFLOP/s), 4096^3 1921 -> 998 us (138 TFLOP/s, 88 % of the peak).
// The shorter chains also halve the error against float64: 1.14e-6 ->
// 0.57e-6 (2-norm, N(0,1) operands) at K = 4096, 4.0e-7 -> 2.1e-7 at 512.
//
// VA / VB: the loads' width in columns.  With 2, lane c takes the columns
// 2c and 2c+1 of its 64-column operand row in one 8-byte load, and fragment
// i of the operand is its element i (any assignment of columns to lanes
// serves, as long as the store uses the same); it needs an even M (N) and an
// 8-byte aligned operand.  Any M, N, K: a load past the end of an operand
// reads 0 through its descriptor (every K row past K lies there), and a
// column past M (N) that is not past the end reads the next row, whose
// products land in rows and columns that are not stored.
template <int BM, int BN, int BK, int WAVES, int VA, int VB>
__global__ __launch_bounds__(WAVES * 64) void mm_f32_kw_kernel(const float* __restrict__ lhsT,
                                                           const float* __restrict__ rhs, float* __restrict__ out,
                                                           int M, int N, int K, int group_m) {
  static_assert(legal_f32_kw(BM, BN, BK, WAVES, 2).code == MI_OK, "illegal tile config (mi_legal.hpp)");
  // FR x FR fragments, KP K rows per MFMA, NQ accumulator quads per lane.
  constexpr int FR = BM == 16 ? 16 : 32, KP = 64 / FR, NQ = FR * FR / 256;
  constexpr int TM = BM / FR, TN = BN / FR, U = BK / KP, W = WAVES, RS = BN + 4, SLOT = BM * RS;
  using acc_t = std::conditional_t<FR == 32, f32x16_t, f32x4_t>;
  static_assert((VA == 1 || VA == TM) && (VB == 1 || VB == TN), "a vector load covers every fragment or one");
  static_assert(W * SLOT * 4 == lds_f32_kw(BM, BN, WAVES), "host LDS budget out of step");
  __shared__ __attribute__((aligned(16))) float part[W * SLOT];
  const int tid = (int)threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kr = lane / FR, c = lane % FR;
  int tm, tn;
  tile_coords((M + BM - 1) / BM, (N + BN - 1) / BN, group_m, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const uint32_t a_bytes = (uint32_t)K * (uint32_t)M * 4u, b_bytes = (uint32_t)K * (uint32_t)N * 4u;
  // Byte offsets of this lane's K rows inside a chunk (the chunk's own offset
  // rides in its descriptor).
  uint32_t va[U], vb[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    va[u] = ((uint32_t)(KP * u + kr) * (uint32_t)M + (uint32_t)(m0 + VA * c)) * 4u;
    vb[u] = ((uint32_t)(KP * u + kr) * (uint32_t)N + (uint32_t)(n0 + VB * c)) * 4u;
  }
  acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = acc_t{};
  float a[2][U][TM], b[2][U][TN];
  const int chunks = (K + BK - 1) / BK;
  auto load = [&](auto buf_c, int chunk) __attribute__((always_inline)) {
    constexpr int buf = decltype(buf_c)::value;
    // A chunk past the last reads zeros (descriptors of no bytes).
    const bool in = chunk < chunks;
    const uint32_t row = (uint32_t)chunk * (uint32_t)(BK * 4);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc_from(lhsT, a_bytes, in ? row * (uint32_t)M : a_bytes);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc_from(rhs, b_bytes, in ? row * (uint32_t)N : b_bytes);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // Opaque here, so that the second fragment's offset stays an immediate
      // of its load instead of another register hoisted out of the loop.
      if constexpr (VA < TM) asm("" : "+v"(va[u]));
      if constexpr (VB < TN) asm("" : "+v"(vb[u]));
      if constexpr (VA == 2) {
        const f32x2_t v = __builtin_bit_cast(f32x2_t, __builtin_amdgcn_raw_buffer_load_b64(ra, va[u], 0, 0));
        a[buf][u][0] = v.x;
        a[buf][u][TM - 1] = v.y;
      } else {
#pragma unroll
        for (int i = 0; i < TM; ++i)
          a[buf][u][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra, va[u] + (uint32_t)(FR * 4 * i), 0, 0));
      }
      if constexpr (VB == 2) {
        const f32x2_t v = __builtin_bit_cast(f32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rb, vb[u], 0, 0));
        b[buf][u][0] = v.x;
        b[buf][u][TN - 1] = v.y;
      } else {
#pragma unroll
        for (int j = 0; j < TN; ++j)
          b[buf][u][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, vb[u] + (uint32_t)(FR * 4 * j), 0, 0));
      }
    }
    // The loads stay here, ahead of the MFMAs of the chunk before.
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mfmas = [&](auto buf_c) __attribute__((always_inline)) {
    constexpr int buf = decltype(buf_c)::value;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          if constexpr (FR == 32)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[buf][u][j], a[buf][u][i], acc[i][j], 0, 0, 0);
          else
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[buf][u][j], a[buf][u][i], acc[i][j], 0, 0, 0);
        }
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr std::integral_constant<int, 0> b0{};
  constexpr std::integral_constant<int, 1> b1{};
  const int mine = chunks > wave ? (chunks - wave + W - 1) / W : 0;
  load(b0, wave);
  for (int t = 0; t + 1 < mine; t += 2) {
    load(b1, wave + (t + 1) * W);
    mfmas(b0);
    load(b0, wave + (t + 2) * W);
    mfmas(b1);
  }
  if (mine & 1) mfmas(b0);
  // This wave's block to its LDS slot, row-major: lane l holds row VA*c + i
  // (or FR*i + c) and, for quad q, fragment columns 8q + 4*kr + 0..3 (4*kr
  // + 0..3 of a 16-wide fragment).
  float* slot = part + wave * SLOT;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    float* row = slot + (VA == 2 ? 2 * c + i : FR * i + c) * RS;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int f = 8 * q + 4 * kr;
      if constexpr (VB == 2) {
        const acc_t &e = acc[i][0], &o = acc[i][TN - 1];
        *(f32x4_t*)(row + 2 * f) = f32x4_t{e[4 * q], o[4 * q], e[4 * q + 1], o[4 * q + 1]};
        *(f32x4_t*)(row + 2 * f + 4) = f32x4_t{e[4 * q + 2], o[4 * q + 2], e[4 * q + 3], o[4 * q + 3]};
      } else {
#pragma unroll
        for (int j = 0; j < TN; ++j)
          *(f32x4_t*)(row + FR * j + f) =
              f32x4_t{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
      }
    }
  }
  __syncthreads();
  const bool wide = N % 4 == 0 && ((uintptr_t)out & 15) == 0;
  for (int it = tid; it < BM * (BN / 4); it += W * 64) {
    const int r = it / (BN / 4), n4 = it % (BN / 4) * 4;
    f32x4_t s = *(const f32x4_t*)(part + r * RS + n4);
#pragma unroll
    for (int w = 1; w < W; ++w) s += *(const f32x4_t*)(part + w * SLOT + r * RS + n4);
    const int m = m0 + r, n = n0 + n4;
    if (m >= M) continue;
    float* o = out + (size_t)m * (size_t)N + n;
    if (wide) {
      if (n < N) *(f32x4_t*)o = s;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) o[e] = s[e];
    }
  }
}

template <int BM, int BN, int BK, int W>
hipError_t launch_mm_f32_kw(const MiArgs& a, hipStream_t s) {
  constexpr int TM = BM == 64 ? 2 : 1, TN = BN == 64 ? 2 : 1;
  const bool a2 = TM == 2 && a.M % 2 == 0 && ((uintptr_t)a.a & 7) == 0;
  const bool b2 = TN == 2 && a.N % 2 == 0 && ((uintptr_t)a.b & 7) == 0;
  const dim3 grid(grid_tiles(a.M, a.N, BM, BN)), block(W * 64);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, s, (const float*)a.a, (const float*)a.b, (float*)a.out, a.M, a.N, a.K,
                       a.group_m);
  };
  if (a2 && b2) go(mm_f32_kw_kernel<BM, BN, BK, W, TM, TN>);
  else if (a2) go(mm_f32_kw_kernel<BM, BN, BK, W, TM, 1>);
  else if (b2) go(mm_f32_kw_kernel<BM, BN, BK, W, 1, TN>);
  else go(mm_f32_kw_kernel<BM, BN, BK, W, 1, 1>);
  return hipGetLastError();
}

template <int BM, int BN>
hipError_t launch_mm_f32_mfma(const MiArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((mm_f32_mfma_kernel<BM, BN>), dim3(grid_tiles(a.M, a.N, BM, BN)), dim3(256), 0, s,
                     (const float*)a.a, (const float*)a.b, (float*)a.out, a.M, a.N, a.K);
  return hipGetLastError();
}

template <int BM, int BN, int BK>
hipError_t launch_mm_f32(const MiArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((mm_f32_kernel<BM, BN, BK>), dim3(grid_tiles(a.M, a.N, BM, BN)), dim3(256), 0, s,
                     (const float*)a.a, (const float*)a.b, (float*)a.out, a.M, a.N, a.K);
  return hipGetLastError();
}

#define MI_F32_KW_CONFIGS(X)  \
  X(16, 16, 32, 4)            \
  X(16, 16, 32, 8)            \
  X(16, 16, 32, 16)           \
  X(32, 32, 16, 8)            \
  X(32, 32, 16, 16)           \
  X(32, 64, 16, 4)            \
  X(32, 64, 16, 8)            \
  X(64, 32, 16, 4)            \
  X(64, 32, 16, 8)            \
  X(64, 64, 16, 4)
#define MI_F32_KW_ROW(BM, BN, BK, W)                                                               \
  {MI_KERNEL_MATMUL_LHST_RHS_F32, {BM, BN, BK, W, 2, 1, 0, 3}, lds_f32_kw(BM, BN, W), \
   &launch_mm_f32_kw<BM, BN, BK, W>},

const MiEntry* table_f32(int* n) {
  static const MiEntry t[] = {
      {MI_KERNEL_MATMUL_LHST_RHS_F32, {64, 64, 16, 4, 1, 1, 0, 0}, (int)(16 * 65 * 4 * 2), &launch_mm_f32<64, 64, 16>},
      {MI_KERNEL_MATMUL_LHST_RHS_F32, {64, 64, 32, 4, 1, 1, 0, 0}, (int)(32 * 65 * 4 * 2), &launch_mm_f32<64, 64, 32>},
      {MI_KERNEL_MATMUL_LHST_RHS_F32, {64, 64, 16, 4, 1, 1, 0, 1}, 0, &launch_mm_f32_mfma<64, 64>},
      {MI_KERNEL_MATMUL_LHST_RHS_F32, {128, 128, 16, 4, 1, 1, 0, 1}, 0, &launch_mm_f32_mfma<128, 128>},
      MI_F32_KW_CONFIGS(MI_F32_KW_ROW)
  };
  *n = (int)(sizeof(t) / sizeof(t[0]));
  return t;
}

}  // namespace mi
