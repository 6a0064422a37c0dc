// Matrix products in fp32:  C[m][n] = sum_k A[m][k] W[n][k] + b[n],  K and N multiples of 64 (v_mfma_f32_16x16x4_f32).
//
//   gemm_f32_kernel        tiles of 64 x 64 or 48 x 64, 64 x 32 up to 128 of those; one barrier per step of 64.  Bound by the matrix cores (153 TFLOP/s in a
//                          large library product) once every CU has tiles.
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

#include <type_traits>

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

// WM x WN waves, each MI x NI blocks of 16 x 16: tiles of 16 MI WM x 16 NI WN.  K in steps of 64 through two LDS buffers, the step after the next in
// registers.  What bounds it beside the products is the LDS port (reads of 4 bytes, two lanes to a bank: 58 % busy with 32 x 16 per wave), so a wave has 32 x 32 or 48 x 16,
// and reads its operands NB products ahead, not all at once behind the barrier.  380 rows, K 2048: 10880 columns 188 -> 167 us (32 x 16 per wave, four
// products ahead -> two); two k side by side for one read of 8 bytes: 171 and 167.  48 rows where they even out the CUs: 2048 columns 46 -> 39, K 5440 118 -> 99.
template <bool GRP, int WM, int MI, int WN, int NI, int NB>
__global__ __launch_bounds__(64 * WM * WN) void gemm_f32_kernel(const F32Args p) {
  constexpr int BM = 16 * MI * WM, BN = 16 * WN * NI, NT = 64 * WM * WN, NA = (BM * 16 + NT - 1) / NT, NW = BN * 16 / NT + (BN * 16 % NT != 0);
  __shared__ __attribute__((aligned(16))) float As[2][BM * LS], Ws[2][BN * LS];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int m0 = blockIdx.y * BM, m_end = p.m, group = 0;
  if constexpr (GRP)
    if (!grouped_tile(p.offsets, p.groups, BM, blockIdx.y, group, m0, m_end)) return;
  const int n0 = blockIdx.x * BN, wm = wave % WM * 16 * MI, wn = wave / WM * 16 * NI;
  // f32x4 tid + NT j of the operand tiles, 16 to a row: bytes within the tile (32 bits beside a uniform base), or of gathered rows
  typedef typename std::conditional<GRP, uint64_t, uint32_t>::type Offset;
  Offset ao[NA];
  uint32_t wo[NW];
  auto row_of = [&](int j) { return (tid + NT * j) >> 4; };
  const int lc = (tid & 15) * 4;
  const float *ab = p.a + (GRP ? 0 : (int64_t)m0 * p.lda), *wb = p.w + ((int64_t)group * p.n_pad + n0) * p.k;
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    int64_t row = min(m0 + row_of(j), m_end - 1);
    if constexpr (GRP)
      if (p.row_of) row = p.row_of[row];
    ao[j] = (Offset)(((row - (GRP ? 0 : m0)) * p.lda + lc) * 4);
  }
#pragma unroll
  for (int j = 0; j < NW; ++j) wo[j] = ((uint32_t)min(row_of(j), BN - 1) * (uint32_t)p.k + lc) * 4;
  f32x4 av[2][NA], wv[2][NW], acc[MI][NI], sum[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int r = lane & 15, kq = lane >> 4;
  auto load = [&](auto set_c, int k0) {  // past the end: the last step again, not used
    constexpr int S = decltype(set_c)::value;
    const int k = min(k0, p.k - BK);
#pragma unroll
    for (int j = 0; j < NA; ++j) av[S][j] = *(const f32x4*)((const char*)(ab + k) + ao[j]);
#pragma unroll
    for (int j = 0; j < NW; ++j) wv[S][j] = *(const f32x4*)((const char*)(wb + k) + wo[j]);
  };
  auto store = [&](auto set_c, int buf) {
    constexpr int S = decltype(set_c)::value;
#pragma unroll
    for (int j = 0; j < NA; ++j)
      if (NA * NT == BM * 16 || row_of(j) < BM) *(f32x4*)(As[buf] + row_of(j) * LS + lc) = av[S][j];
#pragma unroll
    for (int j = 0; j < NW; ++j)
      if (NW * NT == BN * 16 || row_of(j) < BN) *(f32x4*)(Ws[buf] + row_of(j) * LS + lc) = wv[S][j];
  };
  float a[2][NB][MI], w[2][NB][NI];
  auto read = [&](int set, int buf, int batch) {
    const float *as = As[buf] + (wm + r) * LS + kq + 4 * NB * batch, *ws = Ws[buf] + (wn + r) * LS + kq + 4 * NB * batch;
#pragma unroll
    for (int s = 0; s < NB; ++s) {
#pragma unroll
      for (int i = 0; i < MI; ++i) a[set][s][i] = as[16 * i * LS + 4 * s];
#pragma unroll
      for (int j = 0; j < NI; ++j) w[set][s][j] = ws[16 * j * LS + 4 * s];
    }
  };
  constexpr auto S0 = std::integral_constant<int, 0>{};
  constexpr auto S1 = std::integral_constant<int, 1>{};
  load(S0, 0);
  load(S1, BK);
  store(S0, 0);
  __syncthreads();
  // buffer B holds step k0; the registers of the other set the next one
  auto step = [&](auto buf_c, int k0) {
    constexpr int B = decltype(buf_c)::value;
    constexpr auto OTHER = std::integral_constant<int, 1 - B>{};
    const bool more = k0 + BK < p.k;  // (uniform)
    read(0, B, 0);
    __builtin_amdgcn_sched_barrier(0);
    load(buf_c, k0 + 2 * BK);
#pragma unroll
    for (int b = 0; b < BK / 4 / NB; ++b) {
      if (b + 1 < BK / 4 / NB) read((b + 1) & 1, B, b + 1);
      if (b == 1 && more) store(OTHER, 1 - B);  // (read last before the previous barrier)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < NB; ++s)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[b & 1][s][i], w[b & 1][s][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!more || (!p.chain && (k0 & (SLAB - 1)) == SLAB - BK)) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    __syncthreads();
  };
  for (int k0 = 0; k0 < p.k; k0 += 2 * BK) {
    step(S0, k0);
    if (k0 + BK < p.k) step(S1, k0 + BK);
  }
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int n = n0 + wn + 16 * j + r;
    const float b = p.bias ? p.bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm + 16 * i + 4 * kq + e;
        if (m < m_end) p.c[(int64_t)m * p.ldc + n] = sum[i][j][e] + b;
      }
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
    // rows that the fullest of the 256 CUs gets: tiles of 48 rows where they even that out (a row of theirs takes 5 % longer; 380 rows, 6144 columns 100 us against 120, 51200: 25
    // tiles of 48 or 19 of 64 on the fullest CU, 1042 and 930)
    const int cols = lin.n_pad / 64, by64 = (rows * cols + 255) / 256 * 64, by48 = ((m + 47) / 48 * cols + 255) / 256 * 48;
    if (rows * cols <= 128) hipLaunchKernelGGL((gemm_f32_kernel<false, 4, 1, 2, 1, 4>), dim3(lin.n_pad / 32, rows), dim3(512), 0, s, p);
    else if (by48 * 22 < by64 * 21) hipLaunchKernelGGL((gemm_f32_kernel<false, 1, 3, 4, 1, 4>), dim3(cols, (m + 47) / 48), dim3(256), 0, s, p);
    else hipLaunchKernelGGL((gemm_f32_kernel<false, 2, 2, 2, 2, 2>), dim3(cols, rows), dim3(256), 0, s, p);
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
  hipLaunchKernelGGL((gemm_f32_kernel<true, 2, 2, 2, 2, 2>), dim3(lin.n_pad / 64, grouped_tiles(slots, experts, 64)), dim3(256), 0, s, p);
  return md_launch_status();
}
