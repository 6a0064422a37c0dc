// Matrix products in fp32:  C[m][n] = sum_k A[m][k] W[n][k] + b[n],  K and N multiples of 64 (v_mfma_f32_16x16x4_f32).
//
//   gemm_f32_kernel        64 x 64 tiles (64 x 32 up to 128 of those), K halved between two sets of four waves, K in steps of 32 through two LDS
//                          buffers each: the next step's loads are in registers under this step's products, one barrier per step.  Bound by
//                          the matrix cores (153 TFLOP/s in a large library product) once every CU has tiles.  380 rows, 2048 columns, K 2048
//                          and 5440 on average: 81 us, 192 tiles; with four waves, one buffer and K in steps of 16: 157 us.  10880 columns
//                          of K 2048: 165 us, 103 TFLOP/s (171 us).
//   gemm_f32_rows_kernel   up to 32 rows, where the weights are a memory stream: a workgroup owns 16 columns, its eight waves share K, operands
//                          go from memory to registers.  8 rows, the same 2048 columns: 20 us; a whole pass of 24 layers 14.2 -> 3.3 ms (32 rows:
//                          4.5 ms).  From 33 rows on the tiles are ahead: 64 rows 5.9 ms, 6.7 ms this way.
//   Sums run over at most SLAB of K in one chain and are then added up: a third of the rounding error of one chain over K (a pass of 24 layers
//   against 64 bits: 2.4e-6 -> 0.8e-6).
//   grouped: a tile's rows are slots of one group, gathered through row_of (gemm_internal.hpp)
#include "gemm_internal.hpp"
#include "lm_internal.hpp"

namespace {

constexpr int BK = 32, LS = BK + 4;  // K per step; LDS row stride: 16-byte aligned, no bank conflicts

struct F32Args {
  const float* a;
  int64_t lda;
  const float* w;
  const float* bias;
  float* c;
  int64_t ldc;
  int m, k, n_pad;
  const int32_t *row_of, *offsets;
  int groups;
};

// BN: columns
constexpr int SLAB = 256;
template <bool GRP, int BN>
__global__ __launch_bounds__(512) void gemm_f32_kernel(const F32Args p) {
  constexpr int NJ = BN / 32;  // 16-column blocks per wave, f32x4 of the weight tile per thread
  __shared__ __attribute__((aligned(16))) float As[2][2][64 * LS], Ws[2][2][BN * LS];
  const int half = threadIdx.x >> 8, tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
  int m0 = blockIdx.y * 64, m_end = p.m, group = 0;
  if constexpr (GRP)
    if (!grouped_tile(p.offsets, p.groups, 64, blockIdx.y, group, m0, m_end)) return;
  const int n0 = blockIdx.x * BN, wm = (wave & 1) * 32, wn = (wave >> 1) * (BN / 2);
  const int lr = tid >> 3, lc = (tid & 7) * 4;  // f32x4 of the operand tiles: rows lr and lr + 32
  const int kn = p.k >> 1;                      // of this half (a multiple of BK)
  const float *ap[2], *wp[NJ];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    int64_t row = min(m0 + lr + 32 * j, m_end - 1);
    if constexpr (GRP)
      if (p.row_of) row = p.row_of[row];
    ap[j] = p.a + row * p.lda + half * kn + lc;
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) wp[j] = p.w + ((int64_t)group * p.n_pad + n0 + lr + 32 * j) * p.k + half * kn + lc;
  f32x4 av[2], wv[NJ], acc[2][NJ], sum[2][NJ];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int r = lane & 15, kq = lane >> 4;
  auto load = [&](int k0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) av[j] = *(const f32x4*)(ap[j] + k0);
#pragma unroll
    for (int j = 0; j < NJ; ++j) wv[j] = *(const f32x4*)(wp[j] + k0);
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int j = 0; j < 2; ++j) *(f32x4*)(As[half][buf] + (lr + 32 * j) * LS + lc) = av[j];
#pragma unroll
    for (int j = 0; j < NJ; ++j) *(f32x4*)(Ws[half][buf] + (lr + 32 * j) * LS + lc) = wv[j];
  };
  load(0);
  store(0);
  __syncthreads();
  for (int k0 = 0, buf = 0; k0 < kn; k0 += BK, buf ^= 1) {
    const bool more = k0 + BK < kn;  // (uniform)
    if (more) load(k0 + BK);
    const float *as = As[half][buf] + (wm + r) * LS + kq, *ws = Ws[half][buf] + (wn + r) * LS + kq;
    float a[BK / 4][2], w[BK / 4][NJ];
#pragma unroll
    for (int s = 0; s < BK / 4; ++s) {
#pragma unroll
      for (int i = 0; i < 2; ++i) a[s][i] = as[16 * i * LS + 4 * s];
#pragma unroll
      for (int j = 0; j < NJ; ++j) w[s][j] = ws[16 * j * LS + 4 * s];
    }
#pragma unroll
    for (int s = 0; s < BK / 4; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][i], w[s][j], acc[i][j], 0, 0, 0);
    if ((k0 & (SLAB - 1)) == SLAB - BK || !more) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (more) store(buf ^ 1);  // (read last before the previous barrier)
    __syncthreads();
  }
  // the second half's sums to the first, through the operand tiles: [block][thread]
  f32x4* red = (f32x4*)&As[0][0][0];
  static_assert(2 * 2 * 256 * sizeof(f32x4) <= sizeof(As));
  if (half == 1) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) red[(i * NJ + j) * 256 + tid] = sum[i][j];
  }
  __syncthreads();
  if (half == 1) return;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int n = n0 + wn + 16 * j + r;
      const float b = p.bias ? p.bias[n] : 0.f;
      const f32x4 v = sum[i][j] + red[(i * NJ + j) * 256 + tid];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm + 16 * i + 4 * kq + e;
        if (m < m_end) p.c[(int64_t)m * p.ldc + n] = v[e] + b;
      }
    }
}

// MT 16-row tiles.  A unit is 64 of K: 16 products of 4, lane row g takes columns 16 i + 4 g .. + 3 of it
constexpr int RW = 8;  // waves
template <int MT>
__global__ __launch_bounds__(64 * RW) void gemm_f32_rows_kernel(const F32Args p) {
  __shared__ f32x4 red[RW][MT][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const float* wp = p.w + (int64_t)(n0 + r) * p.k + 4 * g;
  const float* ap[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) ap[i] = p.a + (int64_t)min(16 * i + r, p.m - 1) * p.lda + 4 * g;
  const int units = p.k >> 6, lo = units * wave / RW, hi = units * (wave + 1) / RW;
  f32x4 acc[MT], sum[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = sum[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 wf[2][4], af[2][4][MT];
  auto load = [&](auto buf, int u) {
    constexpr int B = decltype(buf)::value;
    const int k = min(u, hi - 1) * 64;  // (past the end: the last unit again, not used)
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      wf[B][h] = __builtin_nontemporal_load((const f32x4*)(wp + k + 16 * h));
#pragma unroll
      for (int i = 0; i < MT; ++i) af[B][h][i] = *(const f32x4*)(ap[i] + k + 16 * h);
    }
  };
  auto multiply = [&](auto buf) {
    constexpr int B = decltype(buf)::value;
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[B][h][e], af[B][h][i][e], acc[i], 0, 0, 0);
  };
  auto add = [&] {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      sum[i] += acc[i];
      acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  constexpr auto B0 = std::integral_constant<int, 0>{};
  constexpr auto B1 = std::integral_constant<int, 1>{};
  if (lo < hi) {
    load(B0, lo);
    for (int u = lo;; u += 2) {
      load(B1, u + 1);
      multiply(B0);
      if (u + 1 >= hi) break;
      load(B0, u + 2);
      multiply(B1);
      if (u + 2 >= hi) break;
      if ((u - lo) % (SLAB / 64) == SLAB / 64 - 2) add();
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) red[wave][i][lane] = sum[i] + acc[i];
  __syncthreads();
  if (wave >= MT) return;
  const int m = 16 * wave + r, n = n0 + 4 * g;  // a lane: four columns of one row
  if (m >= p.m) return;
  f32x4 v = red[0][wave][lane];
#pragma unroll
  for (int w = 1; w < RW; ++w) v += red[w][wave][lane];
  if (p.bias) v += *(const f32x4*)(p.bias + n);
  *(f32x4*)(p.c + (int64_t)m * p.ldc + n) = v;
}

}  // namespace

extern "C" md_status md_gemm_f32(const void* a, int64_t lda, const md_linear* lin, void* c, int64_t ldc, int32_t m, void* stream) {
  MD_CHECK_ARG(a && lin && lin->w && c && m > 0 && lin->n_pad > 0 && lin->n_pad % 64 == 0 && lin->k_pad > 0 && lin->k_pad % 64 == 0);
  MD_CHECK_ARG(lda >= lin->k_pad && lda % 4 == 0 && ldc >= lin->n_pad && ((uintptr_t)a & 15) == 0 && ((uintptr_t)lin->w & 15) == 0);
  const F32Args p = {(const float*)a, lda, (const float*)lin->w, (const float*)lin->b, (float*)c, ldc, m, lin->k_pad, lin->n_pad, nullptr, nullptr, 0};
  const hipStream_t s = (hipStream_t)stream;
  // (16-byte stores of whole column quads need aligned rows)
  if (m <= 32 && ldc % 4 == 0 && ((uintptr_t)c & 15) == 0 && ((uintptr_t)lin->b & 15) == 0) {
    const dim3 grid(lin->n_pad / 16), block(64 * RW);
    if (m <= 16) hipLaunchKernelGGL(gemm_f32_rows_kernel<1>, grid, block, 0, s, p);
    else hipLaunchKernelGGL(gemm_f32_rows_kernel<2>, grid, block, 0, s, p);
  } else {
    const int rows = (m + 63) / 64;
    if (rows * (lin->n_pad / 64) <= 128) hipLaunchKernelGGL((gemm_f32_kernel<false, 32>), dim3(lin->n_pad / 32, rows), dim3(512), 0, s, p);
    else hipLaunchKernelGGL((gemm_f32_kernel<false, 64>), dim3(lin->n_pad / 64, rows), dim3(512), 0, s, p);
  }
  return md_launch_status();
}

md_status lm_grouped_gemm_f32(const void* a, int64_t lda, const int32_t* row_of, const md_linear& lin, int experts, const int32_t* offsets, void* c,
                              int64_t ldc, int slots, hipStream_t s) {
  const F32Args p = {(const float*)a, lda, (const float*)lin.w, nullptr, (float*)c, ldc, slots, lin.k_pad, lin.n_pad, row_of, offsets, experts};
  hipLaunchKernelGGL((gemm_f32_kernel<true, 64>), dim3(lin.n_pad / 64, grouped_tiles(slots, experts, 64)), dim3(512), 0, s, p);
  return md_launch_status();
}
