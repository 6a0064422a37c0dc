// Matrix products in fp32:  C[m][n] = sum_k A[m][k] W[n][k] + b[n],  K and N multiples of 64 (v_mfma_f32_16x16x4_f32).
//
//   gemm_f32_kernel        64 x 64 tiles (64 x 32 up to 128 of those), eight waves, K in steps of 64 through two LDS buffers: the next step's loads
//                          are in registers under this step's products, one barrier per step.  Bound by the matrix cores (153 TFLOP/s in a large
//                          library product) once every CU has tiles.  380 rows, 2048 columns, K 2048 and 5440 on average: 81 us, 192 tiles; with
//                          four waves, one buffer and K in steps of 16: 157 us.  10880 columns of K 2048: 161 us, 105 TFLOP/s (171 us).
//   gemm_f32_rows_kernel   up to 32 rows, where the weights are a memory stream: a workgroup owns 16 columns and all of K, its eight waves load (three
//                          stages ahead), one wave per 16 rows multiplies.  8 rows: a pass of 24 layers 3.2 ms, 14.1 through four-wave tiles; 30
//                          rows: 3.8 ms.  64 rows through the tiles above: 5.6 ms.
//   An element's sum has the same order in both, so a row's result does not depend on the rows beside it.  The order is the caller's:
//     slabs: at most SLAB of K in one chain, the slabs added up.  A third of the rounding error of one chain (a pass of 24 layers against 64
//            bits: 1.5e-6 -> 0.43e-6).
//     chain: all of K in one chain.  For models with retention layers: the output of a sequence's first token is its value times q . k, normed,
//            so that an error in q . k is multiplied by up to 1 / sqrt(eps) where q . k is small.  Such rows have no result that another order
//            would give as well (two prompts of 380 tokens: 1.8e-5 between the two orders, 1e-6 where q . k is not small); they keep the one
//            that results on record were made with.
//   grouped: a tile's rows are slots of one group, gathered through row_of (gemm_internal.hpp)
#include "gemm_internal.hpp"
#include "lm_internal.hpp"

namespace {

constexpr int BK = 64, LS = BK + 4;  // K per step; LDS row stride: 16-byte aligned, no bank conflicts
constexpr int SLAB = 128;

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
  int chain;
};

// BN: columns.  A wave has 32 x 16 of a 64 x 64 tile, 16 x 16 of a 64 x 32 tile
template <bool GRP, int BN>
__global__ __launch_bounds__(512) void gemm_f32_kernel(const F32Args p) {
  constexpr int NI = BN / 32;  // 16-row blocks per wave, f32x4 of the weight tile per thread
  __shared__ __attribute__((aligned(16))) float As[2][64 * LS], Ws[2][BN * LS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int m0 = blockIdx.y * 64, m_end = p.m, group = 0;
  if constexpr (GRP)
    if (!grouped_tile(p.offsets, p.groups, 64, blockIdx.y, group, m0, m_end)) return;
  constexpr int WM = 4 / NI;  // waves along the rows
  const int n0 = blockIdx.x * BN, wm = (wave & (WM - 1)) * 16 * NI, wn = wave / WM * 16;
  const int lr = tid >> 4, lc = (tid & 15) * 4;  // f32x4 of the operand tiles: rows lr and lr + 32
  const float *ap[2], *wp[NI];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    int64_t row = min(m0 + lr + 32 * j, m_end - 1);
    if constexpr (GRP)
      if (p.row_of) row = p.row_of[row];
    ap[j] = p.a + row * p.lda + lc;
  }
#pragma unroll
  for (int j = 0; j < NI; ++j) wp[j] = p.w + ((int64_t)group * p.n_pad + n0 + lr + 32 * j) * p.k + lc;
  f32x4 av[2], wv[NI], acc[NI], sum[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) acc[i] = sum[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int r = lane & 15, kq = lane >> 4;
  auto load = [&](int k0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) av[j] = *(const f32x4*)(ap[j] + k0);
#pragma unroll
    for (int j = 0; j < NI; ++j) wv[j] = *(const f32x4*)(wp[j] + k0);
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int j = 0; j < 2; ++j) *(f32x4*)(As[buf] + (lr + 32 * j) * LS + lc) = av[j];
#pragma unroll
    for (int j = 0; j < NI; ++j) *(f32x4*)(Ws[buf] + (lr + 32 * j) * LS + lc) = wv[j];
  };
  load(0);
  store(0);
  __syncthreads();
  for (int k0 = 0, buf = 0; k0 < p.k; k0 += BK, buf ^= 1) {
    const bool more = k0 + BK < p.k;  // (uniform)
    if (more) load(k0 + BK);
    const float *as = As[buf] + (wm + r) * LS + kq, *ws = Ws[buf] + (wn + r) * LS + kq;
    float a[BK / 4][NI], w[BK / 4];
#pragma unroll
    for (int s = 0; s < BK / 4; ++s) {
#pragma unroll
      for (int i = 0; i < NI; ++i) a[s][i] = as[16 * i * LS + 4 * s];
      w[s] = ws[4 * s];
    }
#pragma unroll
    for (int s = 0; s < BK / 4; ++s)
#pragma unroll
      for (int i = 0; i < NI; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][i], w[s], acc[i], 0, 0, 0);
    if (!more || (!p.chain && (k0 & (SLAB - 1)) == SLAB - BK)) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        sum[i] += acc[i];
        acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
    if (more) store(buf ^ 1);  // (read last before the previous barrier)
    __syncthreads();
  }
  const int n = n0 + wn + r;
  const float b = p.bias ? p.bias[n] : 0.f;
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = m0 + wm + 16 * i + 4 * kq + e;
      if (m < m_end) p.c[(int64_t)m * p.ldc + n] = sum[i][e] + b;
    }
}

// MT 16-row tiles; RK of K per stage, two of them in LDS, AHEAD more in registers.  What bounds a workgroup is the chain of dependent products (22 ns
// each): their operands are read one batch ahead (8 rows, 2048 columns of K 2048, 5440, and 10880 columns: 13.8, 32.2 and 22.3 us; without, 16.8,
// 39.4 and 21.7; eight waves that share K: 11.5, 28.5 and 27.6).
constexpr int RK = SLAB, RS = RK + 4, AHEAD = 3, NB = 4;
template <int MT>
__global__ __launch_bounds__(512) void gemm_f32_rows_kernel(const F32Args p) {
  __shared__ __attribute__((aligned(16))) float Ws[2][16 * RS], As[2][MT][16 * RS];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16, lr = tid >> 5, lc = (tid & 31) * 4;  // f32x4 of a stage's tiles
  const float* wp = p.w + (int64_t)(n0 + lr) * p.k;
  const float* ap[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) ap[i] = p.a + (int64_t)min(16 * i + lr, p.m - 1) * p.lda;
  f32x4 wv[AHEAD], av[AHEAD][MT];
  auto load = [&](int set, int k0) {
    const int k = min(k0 + lc, p.k - 4);
    wv[set] = __builtin_nontemporal_load((const f32x4*)(wp + k));
#pragma unroll
    for (int i = 0; i < MT; ++i) av[set][i] = *(const f32x4*)(ap[i] + k);
  };
  auto store = [&](int set, int buf, int k0) {
    if (k0 + lc >= p.k) {  // past the end: zeros, which add nothing
      wv[set] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < MT; ++i) av[set][i] = wv[set];
    }
    *(f32x4*)(Ws[buf] + lr * RS + lc) = wv[set];
#pragma unroll
    for (int i = 0; i < MT; ++i) *(f32x4*)(As[buf][i] + lr * RS + lc) = av[set][i];
  };
  float a[2][NB], w[2][NB];
  const float *as = As[0][wave < MT ? wave : 0] + r * RS + g, *ws = Ws[0] + r * RS + g;
  auto read = [&](int set, int buf, int batch) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      a[set][i] = as[buf * (MT * 16 * RS) + 4 * (NB * batch + i)];
      w[set][i] = ws[buf * (16 * RS) + 4 * (NB * batch + i)];
    }
  };
  f32x4 acc = {0.f, 0.f, 0.f, 0.f}, sum = acc;
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) load(j, j * RK);
  store(0, 0, 0);
  const int stages = (p.k + RK - 1) / RK;
  for (int s0 = 0; s0 < stages; s0 += 2 * AHEAD) {
#pragma unroll
    for (int j = 0; j < 2 * AHEAD; ++j) {
      const int s = s0 + j, buf = j & 1;
      if (s >= stages) break;  // (uniform)
      __syncthreads();
      load(j % AHEAD, (s + AHEAD) * RK);
      store((j + 1) % AHEAD, buf ^ 1, (s + 1) * RK);  // (that buffer was read before this barrier)
      if (wave < MT) {
        read(0, buf, 0);
#pragma unroll
        for (int b = 0; b < RK / 4 / NB; ++b) {
          if (b + 1 < RK / 4 / NB) read((b + 1) & 1, buf, b + 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < NB; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[b & 1][i], a[b & 1][i], acc, 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (!p.chain) {
          sum += acc;
          acc = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
    }
  }
  if (wave >= MT) return;
  const int m = 16 * wave + r, n = n0 + 4 * g;  // a lane: four columns of one row
  if (m >= p.m) return;
  f32x4 v = sum + acc;
  if (p.bias) v += *(const f32x4*)(p.bias + n);
  *(f32x4*)(p.c + (int64_t)m * p.ldc + n) = v;
}

}  // namespace

md_status lm_gemm_f32(const void* a, int64_t lda, const md_linear& lin, void* c, int64_t ldc, int m, bool chain, hipStream_t s) {
  MD_CHECK_ARG(a && lin.w && c && m > 0 && lin.n_pad > 0 && lin.n_pad % 64 == 0 && lin.k_pad > 0 && lin.k_pad % 64 == 0);
  MD_CHECK_ARG(lda >= lin.k_pad && lda % 4 == 0 && ldc >= lin.n_pad && ((uintptr_t)a & 15) == 0 && ((uintptr_t)lin.w & 15) == 0);
  const F32Args p = {(const float*)a, lda, (const float*)lin.w, (const float*)lin.b, (float*)c, ldc, m, lin.k_pad, lin.n_pad, nullptr, nullptr, 0, chain};
  // (16-byte stores of whole column quads need aligned rows)
  if (m <= 32 && ldc % 4 == 0 && ((uintptr_t)c & 15) == 0 && ((uintptr_t)lin.b & 15) == 0) {
    const dim3 grid(lin.n_pad / 16), block(512);
    if (m <= 16) hipLaunchKernelGGL(gemm_f32_rows_kernel<1>, grid, block, 0, s, p);
    else hipLaunchKernelGGL(gemm_f32_rows_kernel<2>, grid, block, 0, s, p);
  } else {
    const int rows = (m + 63) / 64;
    if (rows * (lin.n_pad / 64) <= 128) hipLaunchKernelGGL((gemm_f32_kernel<false, 32>), dim3(lin.n_pad / 32, rows), dim3(512), 0, s, p);
    else hipLaunchKernelGGL((gemm_f32_kernel<false, 64>), dim3(lin.n_pad / 64, rows), dim3(512), 0, s, p);
  }
  return md_launch_status();
}

extern "C" md_status md_gemm_f32(const void* a, int64_t lda, const md_linear* lin, void* c, int64_t ldc, int32_t m, void* stream) {
  MD_CHECK_ARG(lin);
  return lm_gemm_f32(a, lda, *lin, c, ldc, m, false, (hipStream_t)stream);
}

md_status lm_grouped_gemm_f32(const void* a, int64_t lda, const int32_t* row_of, const md_linear& lin, int experts, const int32_t* offsets, void* c,
                              int64_t ldc, int slots, bool chain, hipStream_t s) {
  const F32Args p = {(const float*)a, lda, (const float*)lin.w, nullptr, (float*)c, ldc, slots, lin.k_pad, lin.n_pad, row_of, offsets, experts, chain};
  hipLaunchKernelGGL((gemm_f32_kernel<true, 64>), dim3(lin.n_pad / 64, grouped_tiles(slots, experts, 64)), dim3(512), 0, s, p);
  return md_launch_status();
}
