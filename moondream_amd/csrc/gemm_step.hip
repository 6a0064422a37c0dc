// Matrix products of a step of few rows, with the row-wise step behind them in the same launch.
//
// A step of a few tokens reads every weight once (2.4 GB of the 24-layer, 2048-wide models) and does next to nothing with it; what is
// left over the memory time is launches, each of which waits for the one before it.  So a launch here owns COMPLETE output columns --
// the waves of a workgroup share K, their sums meet in LDS -- and goes on with them: bias and store, SiLU gate, or the residual streams'
// mixture and the next norm.  The norm is split: the producer of a row stores  u * w  (bf16) and, per 8 columns, the sum of u^2; the
// consumer multiplies its finished sums by  1 / sqrt(mean u^2 + eps), which is the same product with the row's factor taken out.
//
// Weights go from memory to the matrix operand directly (16 rows x 32 of K per wave and load, used once), and so do the activations: with
// few rows they are a fraction of the weights' bytes per tile.  What one of these products makes for the next lies in the operand's order,
// [column / 8][row][8], so that a load takes consecutive memory.  Two register buffers per wave keep two batches of loads in flight.
//
// Measured, 2048 wide, 5440 feed-forward, one row (16 rows): 8192 columns 9.4 us (11.8), 33 MB; gates 11.8 us (15.6), 44 MB, 3.8 TB/s; the two
// residual products 6.2 us (7.4) on average, 8 and 22 MB.  The tile products with K slices and their row-wise second launches took 12.8, 17.5
// and 12.8 us.  A whole step of the 24-layer models: 1830 -> 1320 us (32 heads of 64), 1610 -> 1140 us (state space and latent attention).  About 4 us
// of every launch are its start, the first loads and the sum over the waves.
#include "lm_internal.hpp"

namespace {

constexpr int EPI_ROWS = 0, EPI_SILU = 1, EPI_RESID = 2;

// W waves, MT 16-row tiles.  A workgroup's columns: TN = 16, the matrix operand's rows; SiLU 8 gates and the 8 inputs beside them; or
// TN = 8, for layers of so few columns that the tiles would not fill the chip evenly (2048 columns: 256 workgroups): the operand's upper 8
// rows then hold the other 32 of a unit's 64 of K, so that one load is still 1 KB of weights.  It is multiplied with either half of the
// activations, and the useful half of either product is kept.  MT = 0: up to 8 rows, whose two halves of K fit one operand as well.
// S: streams of the residual epilogue (0: any count); otherwise 1: rows in order, 2: through rows_idx
template <int MT, int TN, int W, int EPI, int S>
__global__ __launch_bounds__(64 * W) void step_gemm_kernel(const LmStepGemm a) {
  constexpr bool SPLIT = EPI != EPI_SILU && TN == 8, DIAG = MT == 0;
  static_assert(SPLIT || !DIAG, "");
  constexpr int M16 = DIAG ? 1 : MT, U = 2;  // (U: units, 64 of K, per load batch)
  constexpr int PW = SPLIT ? 1 : 2, PA = DIAG ? 1 : 2;  // operands per unit
  constexpr int C = SPLIT && !DIAG ? 2 : 1;             // accumulators per row tile
  auto row_of = [&](int m) { return EPI != EPI_RESID && S == 2 ? a.rows_idx[m] : m; };
  __shared__ f32x4 red[W][M16][64];
  __shared__ float row_scale[16 * M16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * TN;

  // sums of squares of the rows, 16 lanes per row: loaded first, added up behind the products
  constexpr int RR = (16 * M16 + 4 * W - 1) / (4 * W);  // rounds of 4 W rows
  f32x4 sq[RR][4];
  if (EPI != EPI_RESID) {
#pragma unroll
    for (int i = 0; i < RR; ++i)
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const int m = min(i * 4 * W + (tid >> 4), a.rows - 1), c = h * 64 + r * 4;
        sq[i][h] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (a.sumsq && i * 4 * W + (tid >> 4) < a.rows && c < a.sumsq_n) sq[i][h] = *(const f32x4*)(a.sumsq + (int64_t)row_of(m) * a.sumsq_n + c);
      }
  }

  const int64_t n = EPI == EPI_SILU ? (int64_t)(r >> 3) * a.ff_pad + n0 + (r & 7) : n0 + (TN == 8 ? r & 7 : r);
  const int kw = SPLIT ? 4 * (r >> 3) + g : g, ka = DIAG ? kw : g;  // 8-column piece of a unit that this lane takes
  const bf16_t* wp = a.w + n * a.k + 8 * kw;
  const bf16_t* ap[M16];
#pragma unroll
  for (int i = 0; i < M16; ++i) ap[i] = a.a + (int64_t)row_of(min(16 * i + (DIAG ? r & 7 : r), a.rows - 1)) * a.lda + ka * a.chunk;
  const int units = a.k >> 6, lo = units * wave / W, hi = units * (wave + 1) / W;
  f32x4 acc[C][M16];
#pragma unroll
  for (int h = 0; h < C; ++h)
#pragma unroll
    for (int i = 0; i < M16; ++i) acc[h][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // what the residual epilogue reads besides, under way before the weights
  constexpr int SM = EPI != EPI_RESID ? 1 : S > 0 ? S : MD_LM_MAX_STREAMS;
  const int m = 16 * wave + r, c = n0 + 4 * g;
  const bool live = wave < M16 && m < a.rows && 4 * g < TN;
  const int ns = S > 0 ? S : a.streams;
  float* xr = EPI == EPI_RESID ? a.x + (int64_t)m * a.width_pad + c : nullptr;
  f32x4 old[SM], norm_w = {0.f, 0.f, 0.f, 0.f};
  if (EPI == EPI_RESID && live) {
#pragma unroll
    for (int s = 0; s < SM; ++s)
      if (s < ns) old[s] = *(const f32x4*)(xr + s * a.stride);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e < a.width) norm_w[e] = a.norm.w[(int64_t)(c + e) * a.norm.stride];
  }

  u32x4 wf[2][PW * U], af[2][PA * U][M16];
  auto load = [&](auto buf, int u) {  // units u .. u + U - 1; past the end: the last one again, not used
    constexpr int B = decltype(buf)::value;
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int k = min(u + q, hi - 1) * 64, kc = k / 8 * a.chunk;
#pragma unroll
      for (int h = 0; h < PW; ++h) wf[B][PW * q + h] = __builtin_nontemporal_load((const u32x4*)(wp + k + 32 * h));
#pragma unroll
      for (int h = 0; h < PA; ++h)
#pragma unroll
        for (int i = 0; i < M16; ++i) af[B][PA * q + h][i] = *(const u32x4*)(ap[i] + kc + 4 * h * a.chunk);
    }
  };
  auto multiply = [&](auto buf, int u) {
    constexpr int B = decltype(buf)::value;
#pragma unroll
    for (int q = 0; q < U; ++q)
      if (u + q < hi) {
#pragma unroll
        for (int h = 0; h < PA; ++h)
#pragma unroll
          for (int i = 0; i < M16; ++i)
            acc[h % C][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(md_bf16x8v, wf[B][PW * q + h % PW]),
                                                                    __builtin_bit_cast(md_bf16x8v, af[B][PA * q + h][i]), acc[h % C][i], 0, 0, 0);
      }
  };
  constexpr auto B0 = std::integral_constant<int, 0>{};
  constexpr auto B1 = std::integral_constant<int, 1>{};
  if (lo < hi) {
    load(B0, lo);
    for (int u = lo;;) {
      if (u + U >= hi) {
        multiply(B0, u);
        break;
      }
      load(B1, u + U);
      multiply(B0, u);
      u += U;
      if (u + U >= hi) {
        multiply(B1, u);
        break;
      }
      load(B0, u + U);
      multiply(B1, u);
      u += U;
    }
  }
  if (EPI != EPI_RESID) {
#pragma unroll
    for (int i = 0; i < RR; ++i) {
      const int m = i * 4 * W + (tid >> 4);
      f32x4 q = (sq[i][0] + sq[i][1]) + (sq[i][2] + sq[i][3]);
      if (a.sumsq)
        for (int c = 256 + r * 4; c < a.sumsq_n; c += 64)  // (widths above 2048)
          q += *(const f32x4*)(a.sumsq + (int64_t)row_of(min(m, a.rows - 1)) * a.sumsq_n + c);
      float v = (q[0] + q[1]) + (q[2] + q[3]);
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
      if (r == 0 && m < 16 * M16) row_scale[m] = a.sumsq ? 1.0f / sqrtf(v / (float)a.width + a.eps) : 1.0f;
    }
  }
#pragma unroll
  for (int i = 0; i < M16; ++i) {
    f32x4 v = acc[0][i];
    if (SPLIT) {  // columns 0 .. 7: lanes 0 .. 31 of the first half's product, 32 .. 63 of the other's; DIAG: rows 0 .. 7, and 8 .. 15
      const int from = DIAG ? lane ^ 40 : lane ^ 32;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += __shfl(acc[C - 1][i][e], from, 64);
    }
    red[wave][i][lane] = v;
  }
  __syncthreads();

  // a lane holds four columns of one row: m = 16 wave + (lane & 15), columns 4 (lane >> 4) ..
  if (wave >= M16) return;
  auto total = [&](int l) {
    f32x4 v = red[0][wave][l];
#pragma unroll
    for (int w = 1; w < W; ++w) v += red[w][wave][l];
    return v;
  };
  if (EPI == EPI_ROWS) {
    if (!live) return;
    f32x4 v = total(lane) * row_scale[m];
    if (a.bias) v += ld4(a.bias + c);
    st4(a.out + (int64_t)m * a.ldo + c, v);
  } else if (EPI == EPI_SILU) {
    if (!live) return;
    const float s = row_scale[m];
    const f32x4 z = total(lane) * s, u = total(lane + 32) * s;
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = silu_fast(z[e]) * u[e];
    st4(a.out + (c >> 3) * a.out_chunk + m * 8 + (c & 7), y);
  } else {
    const float *in_w = a.next, *out_w = a.prev ? a.prev + ns : nullptr, *mix = a.prev ? a.prev + 2 * ns : nullptr;
    const f32x4 y = total(lane);
    f32x4 u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < SM; ++t) {
      if (t >= ns) continue;
      f32x4 v;
      if (mix) {
        v = out_w[t] * y;
#pragma unroll
        for (int s = 0; s < SM; ++s)
          if (s < ns) v += mix[s * ns + t] * old[s];
      } else {
        v = old[t] + y;
      }
      if (live) *(f32x4*)(xr + t * a.stride) = v;
      u += (in_w ? in_w[t] : 1.0f) * v;
    }
    float q = (u[0] * u[0] + u[1] * u[1]) + (u[2] * u[2] + u[3] * u[3]);
    q += __shfl_xor(q, 16, 64);  // (the two quarters of the 8 columns)
    if (live) {
      st4(a.out + (c >> 3) * a.out_chunk + m * 8 + (c & 7), u * norm_w);
      if (g == 0) a.sumsq_out[(int64_t)m * (a.width_pad / 8) + blockIdx.x] = q;
    }
  }
}

template <int TN, int W, int EPI, int S>
md_status launch(const LmStepGemm& a, int n, hipStream_t s) {
  const dim3 grid(n / TN), block(64 * W);
  if constexpr (EPI != EPI_SILU && TN == 8)
    if (a.rows <= 8) {
      hipLaunchKernelGGL((step_gemm_kernel<0, TN, W, EPI, S>), grid, block, 0, s, a);
      return md_launch_status();
    }
  if (a.rows <= 16) hipLaunchKernelGGL((step_gemm_kernel<1, TN, W, EPI, S>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((step_gemm_kernel<2, TN, W, EPI, S>), grid, block, 0, s, a);
  return md_launch_status();
}

// 8 columns instead of 16 where that evens out few tiles and a unit is one load of either operand (6144 columns, 1 row: 8.5 us against
// 9.7; 16 rows: 13.3 against 11.8; 51200 columns, 1 row: 50 against 41)
template <int S>
md_status rows(const LmStepGemm& a, int n, hipStream_t s) {
  auto most = [&](int tn) { return (n / tn + 255) / 256 * tn; };  // columns that the fullest of the 256 CUs gets
  return a.rows <= 8 && n <= 256 * 32 && most(8) < most(16) ? launch<8, 8, EPI_ROWS, S>(a, n, s) : launch<16, 8, EPI_ROWS, S>(a, n, s);
}

static_assert(LM_STEP_ROWS <= 32, "two row tiles");
inline bool takes(const LmStepGemm& a) {
  return a.rows >= 1 && a.rows <= LM_STEP_ROWS && a.k >= 64 && a.k % 64 == 0 && a.lda % 8 == 0 && a.chunk % 8 == 0 &&
         (((uintptr_t)a.a | (uintptr_t)a.w | (uintptr_t)a.out) & 15) == 0;
}

}  // namespace

md_status lm_step_rows(const LmStepGemm& a, int n, hipStream_t s) {
  MD_CHECK_ARG(takes(a) && n % 64 == 0 && a.ldo % 4 == 0);
  return a.rows_idx ? rows<2>(a, n, s) : rows<1>(a, n, s);
}

md_status lm_step_silu(const LmStepGemm& a, hipStream_t s) {
  MD_CHECK_ARG(takes(a) && a.ff_pad % 64 == 0);
  return launch<8, 4, EPI_SILU, 1>(a, a.ff_pad, s);
}

md_status lm_step_resid(const LmStepGemm& a, hipStream_t s) {
  MD_CHECK_ARG(takes(a) && a.width_pad % 64 == 0 && a.streams >= 1 && a.streams <= MD_LM_MAX_STREAMS);
  switch (a.streams) {
    case 1: return launch<8, 8, EPI_RESID, 1>(a, a.width_pad, s);
    case 2: return launch<8, 8, EPI_RESID, 2>(a, a.width_pad, s);
    case 4: return launch<8, 8, EPI_RESID, 4>(a, a.width_pad, s);
    default: return launch<8, 8, EPI_RESID, 0>(a, a.width_pad, s);
  }
}
