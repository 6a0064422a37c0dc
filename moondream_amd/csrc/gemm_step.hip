// Matrix products of a step of few rows, with the row-wise step behind them in the same launch.
//
// A step of a few tokens reads every weight once (2.4 GB of the 24-layer, 2048-wide models) and does next to nothing with it; what is
// left over the memory time is launches, each of which waits for the one before it.  So a launch here owns COMPLETE output columns --
// the waves of a workgroup share K, their sums meet in LDS -- and goes on with them: bias and store, SiLU gate, or the residual streams'
// mixture and the next norm.  The norm is split: the producer of a row stores  u * w  (bf16) and, per 8 columns, the sum of u^2; the
// consumer multiplies its finished sums by  1 / sqrt(mean u^2 + eps), which is the same product with the row's factor taken out.
//
// Weights are used once and come in whole cache lines (8 rows x 128 bytes per wave and load) with the
// non-temporal policy: loads of 16 rows x 64 bytes, the operand's own shape, fetch half lines that are dropped before the other half is asked
// for (4.9 TB/s of the 6.9 that a plain read reaches).  They go through LDS, a ring of each wave's own without a barrier (see load_weights), but for layers
// of up to 8 rows and few columns, where what counts is the way from the first load to the sum (2048 wide, 2048 columns 5.2 us, through LDS 5.3; 4096 wide 7.0 and
// 7.3).  Activations are read directly: with few rows they are a fraction of the weights' bytes.  What a product or a mixer makes for the next one lies in the operand's order, [column / 8][row][8], so that a load takes consecutive memory
// (rows 4 KB apart meet on few channels: output projection of 40 rows 9.9 us against 7.6).
//
// Units of K are under way without a gap in between (stream_units): while the weights' loads into LDS were global ones, every use of loaded activations waited for
// all loads, once in a ring's length.  In a model's decode steps, before and since, in turn: gates of up to 8 / 16 / 32 / 40 rows 11.3 -> 10.7, 10.9 -> 10.5, 12.2 -> 11.3, 13.1 -> 12.7 us; 8192
// columns 9.5 -> 9.2, 8.2 either way, 9.4 -> 9.1, 10.7 -> 10.2; 6144 columns of up to 8 and 16 rows 8.2 and 7.5 either way, 32 / 40 rows 9.4 -> 9.0, 10.6 -> 10.1.  The residual products are bound by
// the activations and did not change.
//
// Measured, 2048 wide, 5440 feed-forward, one stream, one row (16 rows, 28, 40): 8192 columns 8.6 us (8.0, 8.8, 10.1), 33 MB; gates 9.7 us (10.0, 10.9, 12.2), 44 MB;
// the two residual products 4.5 and 6.7 us (4.9 and 8.2; 5.7 and 10.0; 6.5 and 11.9), 8 and 22 MB; the head, 51200 columns, 35 us (36, 41, 45),
// 210 MB.  With the weights loaded in the operand's shape: 8.5 us (8.3, 9.8, 11.2), 10.1 (10.8, 12.2, 13.9), 6.6 (8.5, 10.4, 12.3), 36 (39, 48, 57).  The tile products
// at 40 rows: gates 16.2 us, the residual products and their row-wise launches 13.3 us each, 4352 columns in K slices 12.5 us (9.0).
// About 4 us of every launch are its start, the first loads and the sum over the waves; at 40 rows the activations, which every workgroup reads, are as many bytes
// as the weights.
#include "lm_internal.hpp"
#include "step_weights.hpp"

#include <algorithm>

namespace {

constexpr int EPI_ROWS = 0, EPI_SILU = 1, EPI_RESID = 2;

// W waves, MT 16-row tiles (0: up to 8 rows; others: the residual product), U units of 64 of K under way (in registers: two batches of U).  A workgroup's columns are NX operands of 8;
// SiLU: 8 gates and the 8 inputs beside them.  A load is 8 rows x 128 bytes of weights, whole cache lines: the operand's upper 8 rows hold the other 32 of a unit's 64
// of K.  It is multiplied with either half of the activations, and the useful half of either product is kept; up to 8 rows the two halves of
// K of the activations fit one operand as well.  NX = 1: layers of so few columns that more would not fill the chip evenly.
// S: streams of the residual epilogue (0: any count); otherwise 1: rows in order, 2: through rows_idx
template <int MT, int NX, int W, int U, int EPI, int S>
__global__ __launch_bounds__(64 * W) void step_gemm_kernel(const LmStepGemm a) {
  static_assert(EPI != EPI_SILU || NX == 2, "gates and inputs");
  static_assert(EPI == EPI_RESID || MT == 0, "step_gemm_tall_kernel's");
  constexpr bool DIAG = MT == 0;
  constexpr int M16 = DIAG ? 1 : MT, TN = EPI == EPI_SILU ? 8 : 8 * NX;
  constexpr int PA = DIAG ? 1 : 2;  // operands of activations per unit, and accumulators per operand of weights
  auto row_of = [&](int m) { return EPI != EPI_RESID && S == 2 ? a.rows_idx[m] : m; };
  constexpr bool LDS = NX > 1 || !DIAG;  // weights through LDS
  __shared__ f32x4 red[W][M16][64];
  __shared__ __attribute__((aligned(128))) char ring[W][LDS ? U * NX * 1024 : 16];
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
  auto w_row = [&](int x) { return (int64_t)x * (EPI == EPI_SILU ? a.ff_pad : 8) + n0; };
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
  constexpr int HEADS = 8;  // sums of squares per lane under way with them
  float head_sq[HEADS];
  if (EPI == EPI_RESID && live) {
#pragma unroll
    for (int s = 0; s < SM; ++s)
      if (s < ns) old[s] = *(const f32x4*)(xr + s * a.stride);
#pragma unroll
    for (int e = 0; e < 4; ++e) norm_w[e] = a.norm.w[(int64_t)min(c + e, a.width - 1) * a.norm.stride];  // (columns beyond hold zeros)
  }
  const float* sq_row = EPI == EPI_RESID ? a.head_sumsq + (int64_t)min(m, a.rows - 1) * a.heads : nullptr;
  if (EPI == EPI_RESID && a.head_sumsq && a.groups == 1 && wave < M16)
#pragma unroll
    for (int j = 0; j < HEADS; ++j) head_sq[j] = sq_row[min(4 * j + g, a.heads - 1)];

  if constexpr (LDS) {
    char* mine = ring[wave];
    const uint32_t rd = lds_address(mine) + (r & 7) * 128 + (kw ^ (r & 7)) * 16, at = weight_at(lane, a.k);
    __amdgpu_buffer_rsrc_t w_rows[NX];
#pragma unroll
    for (int x = 0; x < NX; ++x) w_rows[x] = weight_rows(a.w + w_row(x) * a.k);
    u32x4 af[U][PA][M16];
    constexpr int P = NX + PA * M16;
    auto load = [&](int b, int u) {
      const int k = u * 64, kc = k / 8 * a.chunk;
#pragma unroll
      for (int x = 0; x < NX; ++x) load_weights(w_rows[x], at, 2u * k, mine + (b * NX + x) * 1024);
#pragma unroll
      for (int h = 0; h < PA; ++h)
#pragma unroll
        for (int i = 0; i < M16; ++i) af[b][h][i] = *(const u32x4*)(ap[i] + kc + 4 * h * a.chunk);
      asm volatile("" ::: "memory");  // (the waits count: a unit's loads stay together)
    };
    auto multiply = [&](int b) {
      u32x4 w[NX];
      read_weights<NX>(rd + b * NX * 1024, w);
#pragma unroll
      for (int x = 0; x < NX; ++x)
#pragma unroll
        for (int h = 0; h < PA; ++h)
#pragma unroll
          for (int i = 0; i < M16; ++i)
            acc[x][h][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(md_bf16x8v, w[x]), __builtin_bit_cast(md_bf16x8v, af[b][h][i]), acc[x][h][i], 0, 0, 0);
    };
    stream_units<U, P, !(W == 2 && EPI == EPI_ROWS)>(lo, hi, load, multiply, [] {});
  } else {
    const bf16_t* wp[NX];
#pragma unroll
    for (int x = 0; x < NX; ++x) wp[x] = a.w + (w_row(x) + (r & 7)) * a.k + 8 * kw;
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
  // norm groups: a wave's eighth of K lies in one of them.  Lane row g adds up the eighths 2 g and 2 g + 1 of the heads
  float eighth[2] = {0.f, 0.f};
  if (EPI == EPI_RESID && a.head_sumsq && a.groups > 1 && wave < M16) {
    const int per = a.heads / 8;
    float q[2][HEADS];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < HEADS; ++j) q[i][j] = sq_row[(2 * g + i) * per + min(j, per - 1)];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int j = 0; j < HEADS; ++j)
        if (j < per) eighth[i] += q[i][j];
      for (int j = HEADS; j < per; ++j) eighth[i] += sq_row[(2 * g + i) * per + j];
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
      } else {
        const float x = acc[0][0][i][e] + __shfl(acc[0][0][i][e], lane ^ 40, 64);
        const float y = __shfl(acc[NX - 1][0][i][e], lane ^ 32, 64) + __shfl(acc[NX - 1][0][i][e], lane ^ 8, 64);
        v[e] = g < 2 ? x : y;
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
    st4(a.out + m * a.ldo + in_chunks(c, a.out_chunk), y);
  } else {
    const float *in_w = a.next, *out_w = a.prev ? a.prev + ns : nullptr, *mix = a.prev ? a.prev + 2 * ns : nullptr;
    static_assert(EPI != EPI_RESID || W == 8, "norm groups: eighths of K");
    f32x4 y;
    if (a.head_sumsq && a.groups > 1) {
      float q[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) q[k] = __shfl(eighth[k & 1], (k >> 1) * 16 + r, 64);
      if (a.groups <= 4)
#pragma unroll
        for (int k = 0; k < 8; k += 2) q[k] = q[k + 1] = q[k] + q[k + 1];
      if (a.groups <= 2)
#pragma unroll
        for (int k = 0; k < 8; k += 4) q[k] = q[k + 1] = q[k + 2] = q[k + 3] = q[k] + q[k + 2];
      y = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < W; ++w) y += red[w][wave][lane] * (1.0f / sqrtf(q[w & 7] / (float)a.normed + a.eps));
    } else {
      y = total(lane);
    }
    if (a.head_sumsq && a.groups == 1) {
      float q = 0.f;
#pragma unroll
      for (int j = 0; j < HEADS; ++j)
        if (4 * j + g < a.heads) q += head_sq[j];
      for (int j = 4 * HEADS + g; j < a.heads; j += 4) q += sq_row[j];
      q += __shfl_xor(q, 16, 64);
      q += __shfl_xor(q, 32, 64);
      y *= 1.0f / sqrtf(q / (float)a.normed + a.eps);
    }
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
      st4(a.out + m * a.ldo + in_chunks(c, a.out_chunk), u * norm_w);
      if (g == 0) a.sumsq_out[(int64_t)m * (a.width_pad / 8) + blockIdx.x] = q;
    }
  }
}

// Rows and gates of more than 8 rows, operands of 16 columns (SiLU: an odd NX of operands with 8 gates and the 8 inputs beside them, or pairs of 16 gates
// and 16 inputs).  Two loads of 8 rows x 128 bytes make the operands of both halves of a unit's 64 of K.
// Half the matrix instructions of the kernel above, and more columns per
// workgroup: what bounds it beside the weights is that every workgroup reads all activations (28 rows, gates: 680 workgroups of 8 columns 14.7 us, 227
// of 24 13.0).  The waves' parts of K are dealt in turn: with the same part first on every CU, loads meet on the same channels (227 of 24: 12.3 us; through LDS
// 11.2).  D units under way: three and four changed nothing but for NX = 3 (28 rows, 10304 columns 11.0 and 10.8 us).
template <int MT, int NX, int W, int D, int EPI, int S>
__global__ __launch_bounds__(64 * W) void step_gemm_tall_kernel(const LmStepGemm a) {
  constexpr int TN = EPI == EPI_SILU ? 8 * NX : 16 * NX;  // columns of the result
  auto row_of = [&](int m) { return S == 2 ? a.rows_idx[m] : m; };
  constexpr int STAGE = NX * 2048, RING = D * STAGE > NX * MT * 1024 ? D * STAGE : NX * MT * 1024;
  __shared__ __attribute__((aligned(128))) char ring[W][RING];
  __shared__ float row_scale[16 * MT];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4, upper = r >> 3;
  const int n0 = blockIdx.x * TN;

  constexpr int RR = (16 * MT + 4 * W - 1) / (4 * W);  // sums of squares: 16 lanes per row, rounds of 4 W rows, under way before the products
  f32x4 sq[RR][4];
#pragma unroll
  for (int i = 0; i < RR; ++i)
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const int m = min(i * 4 * W + (tid >> 4), a.rows - 1), c = h * 64 + r * 4;
      const float* p = a.sumsq ? a.sumsq + (int64_t)row_of(m) * a.sumsq_n + min(c, a.sumsq_n - 4) : (const float*)a.w;
      sq[i][h] = *(const f32x4*)p;
    }

  // load h of an operand: its rows 8 h .., the piece of a unit that this lane takes
  __amdgpu_buffer_rsrc_t w_rows[NX][2];
#pragma unroll
  for (int x = 0; x < NX; ++x)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // (the last workgroup's columns may go beyond the last one)
      const int64_t first = EPI != EPI_SILU ? min(n0 + 16 * x + 8 * h, a.n - 8)
                            : NX & 1      ? (int64_t)h * a.ff_pad + min(n0 + 8 * x, a.n - 8)
                                          : (int64_t)(x & 1) * a.ff_pad + min(n0 + 16 * (x >> 1) + 8 * h, a.n - 8);
      w_rows[x][h] = weight_rows(a.w + first * a.k);
    }
  char* mine = ring[wave];
  const uint32_t at = weight_at(lane, a.k);
  const uint32_t rd = lds_address(mine) + upper * 1024 + (r & 7) * 128 + (g ^ (r & 7)) * 16;
  const bf16_t* ap[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) ap[i] = a.a + (int64_t)row_of(min(16 * i + r, a.rows - 1)) * a.lda + g * a.chunk;
  const int units = a.k >> 6, part = (wave + (int)(blockIdx.x >> 3)) % W, lo = units * part / W, hi = units * (part + 1) / W;
  f32x4 acc[NX][2][MT];
#pragma unroll
  for (int x = 0; x < NX; ++x)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[x][h][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  u32x4 af[D][2][MT];
  constexpr int P = 2 * NX + 2 * MT;
  auto load = [&](int b, int u) {
    const int k = u * 64, kc = k / 8 * a.chunk;
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
      for (int h = 0; h < 2; ++h) load_weights(w_rows[x][h], at, 2u * k, mine + b * STAGE + x * 2048 + h * 1024);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < MT; ++i) af[b][h][i] = *(const u32x4*)(ap[i] + kc + 4 * h * a.chunk);
    asm volatile("" ::: "memory");  // (the waits count: a unit's loads stay together)
  };
  auto multiply = [&](int b) {
    u32x4 w[NX][2];
    read_weights<NX>(rd + b * STAGE, w);
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          acc[x][h][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(md_bf16x8v, w[x][h]), __builtin_bit_cast(md_bf16x8v, af[b][h][i]), acc[x][h][i], 0, 0, 0);
  };
  float factor[RR];
  stream_units<D, P, !(NX == 4 && MT == 3)>(lo, hi, load, multiply, [&] {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < RR; ++i) {
      f32x4 q = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < 4; ++h)
        if (h * 64 + r * 4 < a.sumsq_n) q += sq[i][h];
      factor[i] = (q[0] + q[1]) + (q[2] + q[3]);
    }
    __builtin_amdgcn_sched_barrier(0);
  });
#pragma unroll
  for (int i = 0; i < RR; ++i) {
    const int m = i * 4 * W + (tid >> 4);
    if (a.sumsq)
      for (int c = 256 + r * 4; c < a.sumsq_n; c += 64) {  // (widths above 2048)
        const f32x4 q = *(const f32x4*)(a.sumsq + (int64_t)row_of(min(m, a.rows - 1)) * a.sumsq_n + c);
        factor[i] += (q[0] + q[1]) + (q[2] + q[3]);
      }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) factor[i] += __shfl_xor(factor[i], o, 64);
    if (r == 0 && m < 16 * MT) row_scale[m] = a.sumsq ? 1.0f / sqrtf(factor[i] / (float)a.width + a.eps) : 1.0f;
  }
#pragma unroll
  for (int x = 0; x < NX; ++x)
#pragma unroll
    for (int i = 0; i < MT; ++i) ((f32x4*)mine)[(x * MT + i) * 64 + lane] = acc[x][0][i] + acc[x][1][i];  // (its own ring, read to the end)
  __syncthreads();

  // a lane holds four columns of one row: m = 16 i + (lane & 15), columns 4 (lane >> 4) .. of the operand's
  auto total = [&](int t, int l) {
    auto of = [&](int p) { return ((const f32x4*)ring[(p + 8 * W - (int)(blockIdx.x >> 3) % W) % W])[t * 64 + l]; };  // part p's wave
    f32x4 v = of(0);
#pragma unroll
    for (int w = 1; w < W; ++w) v += of(w);
    return v;
  };
  if (EPI == EPI_ROWS) {
    for (int t = wave; t < NX * MT; t += W) {
      const int m = 16 * (t % MT) + r, c = n0 + 16 * (t / MT) + 4 * g;
      if (m >= a.rows || c >= a.n) continue;
      f32x4 v = total(t, lane) * row_scale[m];
      if (a.bias) v += ld4(a.bias + c);
      st4(a.out + (int64_t)m * a.ldo + c, v);
    }
  } else {
    constexpr int PAIRS = NX & 1 ? NX : NX / 2;
    for (int t = wave; t < PAIRS * MT; t += W) {
      const int x = t / MT, i = t % MT, m = 16 * i + r, c = n0 + (NX & 1 ? 8 : 16) * x + 4 * g;
      if (m >= a.rows || c >= a.n || (NX & 1 && g >= 2)) continue;
      const float s = row_scale[m];
      const f32x4 z = total(NX & 1 ? t : 2 * x * MT + i, lane) * s, u = (NX & 1 ? total(t, lane + 32) : total((2 * x + 1) * MT + i, lane)) * s;
      f32x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = silu_fast(z[e]) * u[e];
      st4(a.out + m * a.ldo + in_chunks(c, a.out_chunk), y);
    }
  }
}

template <int MT, int NX, int W, int U, int EPI, int S>
md_status launch(const LmStepGemm& a, hipStream_t s) {
  hipLaunchKernelGGL((step_gemm_kernel<MT, NX, W, U, EPI, S>), dim3(a.n / (EPI == EPI_SILU ? 8 : 8 * NX)), dim3(64 * W), 0, s, a);
  return md_launch_status();
}
template <int MT, int NX, int W, int EPI, int S>
md_status tall_rows(const LmStepGemm& a, hipStream_t s) {
  constexpr int TN = EPI == EPI_SILU ? 8 * NX : 16 * NX;
  hipLaunchKernelGGL((step_gemm_tall_kernel<MT, NX, W, NX == 3 ? 3 : 2, EPI, S>), dim3((a.n + TN - 1) / TN), dim3(64 * W), 0, s, a);
  return md_launch_status();
}
template <int NX, int W, int EPI, int S>
md_status tall(const LmStepGemm& a, hipStream_t s) {
  return a.rows <= 16 ? tall_rows<1, NX, W, EPI, S>(a, s) : a.rows <= 32 ? tall_rows<2, NX, W, EPI, S>(a, s) : tall_rows<3, NX, W, EPI, S>(a, s);
}
// As many operands per workgroup as leave the fullest of the 256 CUs with the fewest columns, the larger number where that is the same (40 rows,
// 10304 columns: 1, 2, 3 operands 21.5, 17.8, 12.0 us; 8192: 15.4, 10.4, 11.5; 4352: 14.2, 9.5, 10.8)
template <int EPI, int S>
md_status tall_by_columns(const LmStepGemm& a, hipStream_t s) {
  auto most = [&](int nx) {
    const int tn = (EPI == EPI_SILU ? 8 : 16) * nx;
    return ((a.n + tn - 1) / tn + 255) / 256 * nx;
  };
  if (most(3) <= std::min(most(1), most(2))) return tall<3, 8, EPI, S>(a, s);
  return most(2) <= most(1) ? tall<2, 8, EPI, S>(a, s) : tall<1, 8, EPI, S>(a, s);
}

// Columns and waves of a workgroup.  Up to 8 rows, where a unit's activations are one load: 8 columns where that evens out few workgroups (6144
// columns, 8 rows: 7.4 us against 7.9; 8192: 9.4 against 8.5), eight waves to share K otherwise.  More than four workgroups of 16 columns per CU: fewer
// waves (51200 columns, 1 row: two waves 34.6 us, eight 37.0), and from 17 rows on more columns, whose activations are read less often (16 / 28 / 40 rows: 32 columns to
// four waves 36.6 / 43 / 50 us, 64 columns 38.4 / 41 / 46, 64 to eight waves 43 / 47 / 51).
template <int S>
md_status rows(const LmStepGemm& a, hipStream_t s) {
  auto most = [&](int tn) { return (a.n / tn + 255) / 256 * tn; };  // columns that the fullest of the 256 CUs gets
  const bool many = a.n > 256 * 64;
  if (a.rows > 8) return !many ? tall_by_columns<EPI_ROWS, S>(a, s) : a.rows <= 16 ? tall<2, 4, EPI_ROWS, S>(a, s) : tall<4, 4, EPI_ROWS, S>(a, s);
  if (many) return launch<0, 2, 2, 2, EPI_ROWS, S>(a, s);
  return a.n <= 256 * 32 && most(8) < most(16) ? launch<0, 1, 4, 2, EPI_ROWS, S>(a, s) : launch<0, 2, 8, 2, EPI_ROWS, S>(a, s);
}

// Waves that share K, up to 8 rows.  Up to one workgroup of 8 columns per CU the chain of loads bounds it: eight (2048 wide, 256 / 2048 columns, 1 row: 5.2 /
// 6.0 us, four 6.2 / 6.8, two 8.2 / 8.5; 4096 wide 6.9 / 8.7, two 13.9 / 15.6).  More: four (4096 wide, 10944 columns: 31 us, two 40, eight 32; 1024 wide, 5440
// columns: 6.3, 6.9, 6.5), but two where the workgroups are many and a wave's half of K is of 8 to 16 units (2048 wide, 5440 / 8192 columns: 10.2 / 12.7
// us, four 10.1 / 13.6; 2816 columns: 9.1 and 7.3).  Four units under way: nothing but for two waves (5440 columns 10.1, 8192 13.0).
md_status gates(const LmStepGemm& a, hipStream_t s) {
  if (a.n <= 256 * 8) return launch<0, 2, 8, 2, EPI_SILU, 1>(a, s);
  return a.n > 2 * 256 * 8 && a.k > 1024 && a.k <= 2048 ? launch<0, 2, 2, 2, EPI_SILU, 1>(a, s) : launch<0, 2, 4, 2, EPI_SILU, 1>(a, s);
}

// Up to 8 rows four units per batch where K is long (5440: 6.8 us against 7.7; 2048: 4.4 either way)
template <int S>
md_status resid(const LmStepGemm& a, hipStream_t s) {
  // (more rows: two units under way, three row tiles have the registers for one: 5440 wide, 40 rows 11.9 us, two 12.2, three 12.1; 16 rows 9.6 and 8.2)
  if (a.rows <= 8) return a.k > 4096 ? launch<0, 1, 8, 4, EPI_RESID, S>(a, s) : launch<0, 1, 8, 2, EPI_RESID, S>(a, s);
  return a.rows <= 16 ? launch<1, 1, 8, 2, EPI_RESID, S>(a, s) : a.rows <= 32 ? launch<2, 1, 8, 2, EPI_RESID, S>(a, s) : launch<3, 1, 8, 1, EPI_RESID, S>(a, s);
}

static_assert(LM_STEP_ROWS <= 48, "three row tiles");
inline bool takes(const LmStepGemm& a) {
  return a.rows >= 1 && a.rows <= LM_STEP_ROWS && a.k >= 64 && a.k % 64 == 0 && a.lda % 8 == 0 && a.chunk % 8 == 0 &&
         (((uintptr_t)a.a | (uintptr_t)a.w | (uintptr_t)a.out) & 15) == 0;
}

}  // namespace

md_status lm_step_rows(const LmStepGemm& g, int n, hipStream_t s) {
  MD_CHECK_ARG(takes(g) && n % 64 == 0 && g.ldo % 4 == 0);
  LmStepGemm a = g;
  a.n = n;
  return a.rows_idx ? rows<2>(a, s) : rows<1>(a, s);
}

md_status lm_step_silu(const LmStepGemm& g, hipStream_t s) {
  MD_CHECK_ARG(takes(g) && g.ff_pad % 64 == 0);
  LmStepGemm a = g;
  a.n = a.ff_pad;
  return a.rows <= 8 ? gates(a, s) : tall_by_columns<EPI_SILU, 1>(a, s);
}

md_status lm_step_resid(const LmStepGemm& g, hipStream_t s) {
  MD_CHECK_ARG(takes(g) && g.width_pad % 64 == 0 && g.streams >= 1 && g.streams <= MD_LM_MAX_STREAMS);
  // (norm groups: a wave's part of K is an eighth, and lies in one of them)
  MD_CHECK_ARG(!g.head_sumsq || (g.heads >= 1 && g.normed > 0 && (g.groups == 1 || ((g.groups == 2 || g.groups == 4 || g.groups == 8) && g.heads % 8 == 0 && g.k % 512 == 0))));
  LmStepGemm a = g;
  a.n = a.width_pad;
  switch (a.streams) {
    case 1: return resid<1>(a, s);
    case 2: return resid<2>(a, s);
    case 4: return resid<4>(a, s);
    default: return resid<0>(a, s);
  }
}
