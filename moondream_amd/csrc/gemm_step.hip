// Matrix products of a step of few rows, with the row-wise step behind them in the same launch.
//
// A step of a few tokens reads every weight once (2.4 GB of the 24-layer, 2048-wide models) and does next to nothing with it; what is
// left over the memory time is launches, each of which waits for the one before it.  So a launch here owns COMPLETE output columns --
// the waves of a workgroup share K, their sums meet in LDS -- and goes on with them: bias and store, SiLU gate, or the residual streams'
// mixture and the next norm.  The norm is split: the producer of a row stores  u * w  (bf16) and, per 8 columns, the sum of u^2; the
// consumer multiplies its finished sums by  1 / sqrt(mean u^2 + eps), which is the same product with the row's factor taken out.
//
// Weights go from memory to the matrix operand directly, used once, in whole cache lines (8 rows x 128 bytes per wave and load) with the
// non-temporal policy: loads of 16 rows x 64 bytes, the operand's own shape, fetch half lines that are dropped before the other half is asked
// for (4.9 TB/s of the 6.9 that a plain read reaches).  Activations are read directly too: with few rows they are a fraction of the weights'
// bytes.  What one of these products makes for the next lies in the operand's order, [column / 8][row][8], so that a load takes consecutive memory.
// Two register buffers per wave keep two batches of loads in flight.
//
// Measured, 2048 wide, 5440 feed-forward, one row (16 rows, 28 rows): 8192 columns 9.0 us (9.5, 10.9), 33 MB; gates 10.9 us (11.5, 14.3), 44 MB; the two
// residual products 4.4 and 7.0 us (5.0 and 8.3; 6.0 and 11.0), 8 and 22 MB; the head, 51200 columns, 36 us (40, 57), 210 MB.  With half lines: gates 12.2 us
// (15.9), head 47 us.  The tile products with K slices and their row-wise second launches took 12.8, 17.5 and 12.8 us.  About 4 us of every launch
// are its start, the first loads and the sum over the waves.
#include "lm_internal.hpp"

namespace {

constexpr int EPI_ROWS = 0, EPI_SILU = 1, EPI_RESID = 2;

// W waves, MT 16-row tiles (0: up to 8 rows), U units of 64 of K per load batch.  A workgroup's columns are NX operands of 8; SiLU: 8 gates and the 8
// inputs beside them.  A load is 8 rows x 128 bytes of weights, whole cache lines: the operand's upper 8 rows hold the other 32 of a unit's 64
// of K.  It is multiplied with either half of the activations, and the useful half of either product is kept; up to 8 rows the two halves of
// K of the activations fit one operand as well.  NX = 1: layers of so few columns that more would not fill the chip evenly.
// S: streams of the residual epilogue (0: any count); otherwise 1: rows in order, 2: through rows_idx
template <int MT, int NX, int W, int U, int EPI, int S>
__global__ __launch_bounds__(64 * W) void step_gemm_kernel(const LmStepGemm a) {
  static_assert(EPI != EPI_SILU || NX == 2, "gates and inputs");
  constexpr bool DIAG = MT == 0;
  constexpr int M16 = DIAG ? 1 : MT, TN = EPI == EPI_SILU ? 8 : 8 * NX;
  constexpr int PA = DIAG ? 1 : 2;  // operands of activations per unit, and accumulators per operand of weights
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

  const int kw = 4 * (r >> 3) + g, ka = DIAG ? kw : g;  // 8-column piece of a unit that this lane takes
  const bf16_t* wp[NX];
#pragma unroll
  for (int x = 0; x < NX; ++x) wp[x] = a.w + ((int64_t)x * (EPI == EPI_SILU ? a.ff_pad : 8) + n0 + (r & 7)) * a.k + 8 * kw;
  const bf16_t* ap[M16];
#pragma unroll
  for (int i = 0; i < M16; ++i) ap[i] = a.a + (int64_t)row_of(min(16 * i + (DIAG ? r & 7 : r), a.rows - 1)) * a.lda + ka * a.chunk;
  const int units = a.k >> 6, lo = units * wave / W, hi = units * (wave + 1) / W;
  f32x4 acc[NX][PA][M16];
#pragma unroll
  for (int x = 0; x < NX; ++x)
#pragma unroll
    for (int h = 0; h < PA; ++h)
#pragma unroll
      for (int i = 0; i < M16; ++i) acc[x][h][i] = f32x4{0.f, 0.f, 0.f, 0.f};

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

  u32x4 wf[2][U][NX], af[2][U][PA][M16];
  auto load = [&](auto buf, int u) {  // units u .. u + U - 1; past the end: the last one again, not used
    constexpr int B = decltype(buf)::value;
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int k = min(u + q, hi - 1) * 64, kc = k / 8 * a.chunk;
#pragma unroll
      for (int x = 0; x < NX; ++x) wf[B][q][x] = __builtin_nontemporal_load((const u32x4*)(wp[x] + k));
#pragma unroll
      for (int h = 0; h < PA; ++h)
#pragma unroll
        for (int i = 0; i < M16; ++i) af[B][q][h][i] = *(const u32x4*)(ap[i] + kc + 4 * h * a.chunk);
    }
  };
  auto multiply = [&](auto buf, int u) {
    constexpr int B = decltype(buf)::value;
#pragma unroll
    for (int q = 0; q < U; ++q)
      if (u + q < hi) {
#pragma unroll
        for (int x = 0; x < NX; ++x)
#pragma unroll
          for (int h = 0; h < PA; ++h)
#pragma unroll
            for (int i = 0; i < M16; ++i)
              acc[x][h][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(md_bf16x8v, wf[B][q][x]), __builtin_bit_cast(md_bf16x8v, af[B][q][h][i]),
                                                                     acc[x][h][i], 0, 0, 0);
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
    // an operand's 8 columns: lanes 0 .. 31 of the first half's product, 32 .. 63 of the other's; DIAG: rows 0 .. 7, and 8 .. 15.  The second
    // operand's go to lanes 32 .. 63
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (NX == 1) {
        v[e] = acc[0][0][i][e] + __shfl(acc[0][PA - 1][i][e], DIAG ? lane ^ 40 : lane ^ 32, 64);
      } else if (DIAG) {
        const float x = acc[0][0][i][e] + __shfl(acc[0][0][i][e], lane ^ 40, 64);
        const float y = __shfl(acc[NX - 1][0][i][e], lane ^ 32, 64) + __shfl(acc[NX - 1][0][i][e], lane ^ 8, 64);
        v[e] = g < 2 ? x : y;
      } else {
        v[e] = (g < 2 ? acc[0][0][i][e] : acc[NX - 1][PA - 1][i][e]) + __shfl(g < 2 ? acc[NX - 1][0][i][e] : acc[0][PA - 1][i][e], lane ^ 32, 64);
      }
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

template <int MT, int NX, int W, int U, int EPI, int S>
md_status launch(const LmStepGemm& a, int n, hipStream_t s) {
  hipLaunchKernelGGL((step_gemm_kernel<MT, NX, W, U, EPI, S>), dim3(n / (EPI == EPI_SILU ? 8 : 8 * NX)), dim3(64 * W), 0, s, a);
  return md_launch_status();
}
template <int NX, int W, int U, int EPI, int S>
md_status by_rows(const LmStepGemm& a, int n, hipStream_t s) {
  return a.rows <= 8 ? launch<0, NX, W, U, EPI, S>(a, n, s) : a.rows <= 16 ? launch<1, NX, W, U, EPI, S>(a, n, s) : launch<2, NX, W, U, EPI, S>(a, n, s);
}

// Columns and waves of a workgroup.  More than four workgroups of 16 columns per CU: two waves (51200 columns, 1 / 12 / 28 rows: 36 / 40 / 57 us; four waves
// 36 / 41 / 58, eight 39 / 48 / 76).  Up to 8 rows, where a unit's activations are one load: 8 columns where that evens out few workgroups (6144
// columns, 8 rows: 7.5 us against 8.0; 8192: 9.5 against 8.7), eight waves to share K otherwise.
template <int S>
md_status rows(const LmStepGemm& a, int n, hipStream_t s) {
  auto most = [&](int tn) { return (n / tn + 255) / 256 * tn; };  // columns that the fullest of the 256 CUs gets
  if (n > 256 * 64) return by_rows<2, 2, 1, EPI_ROWS, S>(a, n, s);
  if (a.rows > 8) return by_rows<2, 4, 2, EPI_ROWS, S>(a, n, s);
  return n <= 256 * 32 && most(8) < most(16) ? launch<0, 1, 4, 2, EPI_ROWS, S>(a, n, s) : launch<0, 2, 8, 1, EPI_ROWS, S>(a, n, s);
}

// Up to 8 rows four units per batch where K is long (5440: 6.8 us against 7.7; 2048: 4.4 either way)
template <int S>
md_status resid(const LmStepGemm& a, hipStream_t s) {
  return a.rows <= 8 && a.k > 4096 ? launch<0, 1, 8, 4, EPI_RESID, S>(a, a.width_pad, s) : by_rows<1, 8, 2, EPI_RESID, S>(a, a.width_pad, s);
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
  return by_rows<2, 2, 1, EPI_SILU, 1>(a, a.ff_pad, s);
}

md_status lm_step_resid(const LmStepGemm& a, hipStream_t s) {
  MD_CHECK_ARG(takes(a) && a.width_pad % 64 == 0 && a.streams >= 1 && a.streams <= MD_LM_MAX_STREAMS);
  switch (a.streams) {
    case 1: return resid<1>(a, s);
    case 2: return resid<2>(a, s);
    case 4: return resid<4>(a, s);
    default: return resid<0>(a, s);
  }
}
