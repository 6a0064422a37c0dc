// Products of a step's rows with the matrices of the experts that they chose, few rows per expert.
//
// A decode step reads every chosen expert's weights once and uses them for a handful of rows, so the weights' bytes bound it.  A workgroup owns
// complete output columns of ONE expert: its waves share K and their sums meet in LDS, so there are no partial products in memory.  It finds
// the expert's rows itself, by ballots over the step's choices, so the choices need no sorting and no launch for it; results stay in the
// order of the choices.
//
// A weight load is 8 rows x 128 bytes, whole cache lines, non-temporal, through LDS: the operand's upper 8 rows
// hold the other 32 of a unit's 64 of K.  It is multiplied with either half of the activations and the useful half of either
// product kept; up to 8 rows of activations, the two halves of K fit one operand as well.  16 rows x 64 bytes per load, the operand's
// own shape, fetches half lines: 4.95 TB/s with the non-temporal policy, which drops a line before its other half is asked for, 5.66 without,
// against 6.4 (a plain read of the same bytes: 6.9).  Activations of rows that do not exist are not fetched (a buffer load out of range gives zeros).
//
// Measured, 32 experts, 4 per row, 2 x 1360 and 1360 columns of 2048, against tiles of 64 rows and the launch that sorts the choices (4.6 us):
// 23 rows 77 -> 53.7 us (358 MB) and 42 -> 29.4 us (179 MB), 6.7 and 6.1 TB/s; weights loaded in the operand's shape, two units on their way, 54.7 and 30.4.  Three units
// on their way: one 57.0 and 31.3, two 53.5 and 30.1, four 53.8 and 30.3.  Twice the columns per workgroup: 56.8 and 30.2.
#include "step_weights.hpp"

namespace {

constexpr int EPI_ROWS = 0, EPI_SILU = 1;
constexpr int W = 2;  // waves
constexpr int D = 3;  // units of 64 of K under way

// A workgroup's 16 columns, two operands of 8: columns 0 .. 7 and 8 .. 15; SiLU: 8 gates and the 8 inputs beside them
template <int EPI>
__global__ __launch_bounds__(64 * W) void expert_gemm_kernel(const LmExpertGemm a) {
  __shared__ f32x4 red[W][2][64];
  __shared__ __attribute__((aligned(128))) char ring[W][D * 2048];
  __shared__ uint16_t lists[W][LM_EXPERT_CHOICES];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const bool by_choice = a.n < a.experts;  // one workgroup per choice, or per expert: whatever there are fewer of
  const int expert = by_choice ? a.chosen[blockIdx.y] : blockIdx.y;
  const int n0 = blockIdx.x * (EPI == EPI_SILU ? 8 : 16);

  // the choices that fell on this expert, in order (every wave for itself: no barrier)
  uint16_t* list = lists[wave];
  const unsigned long long before = (1ull << lane) - 1;
  int count = 0;
  for (int b = 0; b < a.n; b += 64) {
    const int i = b + lane;
    const bool mine = i < a.n && a.chosen[min(i, a.n - 1)] == expert;
    const unsigned long long who = __ballot(mine);
    if (mine) list[count + __popcll(who & before)] = (uint16_t)i;
    count += __popcll(who);
  }
  __builtin_amdgcn_wave_barrier();
  if (count == 0 || (by_choice && list[0] != blockIdx.y)) return;  // (the same in every wave) nobody's, or an earlier choice's

  const int kw = 4 * (r >> 3) + g;  // 8-column piece of a unit, 64 of K, that this lane takes
  const bf16_t* w0 = a.w + expert * a.expert_stride + (int64_t)n0 * a.k;
  const __amdgpu_buffer_rsrc_t w_rows[2] = {weight_rows(w0), weight_rows(w0 + (int64_t)(EPI == EPI_SILU ? a.ff_pad : 8) * a.k)};
  const uint32_t w_at = weight_at(lane, a.k);
  char* mine = ring[wave];
  const uint32_t rd = lds_address(mine) + (r & 7) * 128 + (kw ^ (r & 7)) * 16;
  const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc((void*)a.a, 0, (int)(a.a_rows * a.lda * 2), 0x00020000);
  const int units = a.k >> 6, lo = units * wave / W, hi = units * (wave + 1) / W;

  auto run = [&](auto few) {  // up to 8 choices, or 16 at a time
    constexpr bool FEW = decltype(few)::value;
    constexpr int ROWS = FEW ? 8 : 16, PA = FEW ? 1 : 2;
    for (int r0 = 0; r0 < count; r0 += ROWS) {
      const int row = r0 + (FEW ? r & 7 : r);
      const uint32_t at = row < count ? (uint32_t)(list[min(row, count - 1)] / a.per) * (uint32_t)(a.lda * 2) + 16u * (FEW ? kw : g) : 0x80000000u;
      f32x4 acc[2][PA];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int h = 0; h < PA; ++h) acc[i][h] = f32x4{0.f, 0.f, 0.f, 0.f};
      u32x4 af[D][PA];
      auto load = [&](int b, int u) {
        load_weights(w_rows[0], w_at, 128u * u, mine + b * 2048);
        load_weights(w_rows[1], w_at, 128u * u, mine + b * 2048 + 1024);
#pragma unroll
        for (int h = 0; h < PA; ++h) af[b][h] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rows, at + 128u * u + 64u * h, 0, 0));
        asm volatile("" ::: "memory");  // (the waits count: a unit's loads stay together)
      };
      auto multiply = [&](int b) {
        u32x4 w[2];
        read_weights<2>(rd + b * 2048, w);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int h = 0; h < PA; ++h)
            acc[i][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(md_bf16x8v, w[i]), __builtin_bit_cast(md_bf16x8v, af[b][h]), acc[i][h], 0, 0, 0);
      };
      stream_units<D, 2 + PA>(lo, hi, load, multiply, [] {});
      if (r0 > 0) __syncthreads();  // (the sums before these were read)
      // 8 columns: lanes 0 .. 31 of the first half's product, 32 .. 63 of the other's; up to 8 choices: rows 0 .. 7, and 8 .. 15
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        f32x4 v = acc[i][0];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += __shfl(acc[i][PA - 1][e], FEW ? lane ^ 40 : lane ^ 32, 64);
        red[wave][i][lane] = v;
      }
      __syncthreads();

      // a lane holds columns 4 g .. of operand `wave` (SiLU: of both) of one choice
      const int m = r0 + r;
      if ((FEW && r >= 8) || m >= count || g >= 2) continue;
      auto total = [&](int i) {
        f32x4 v = red[0][i][lane];
#pragma unroll
        for (int w = 1; w < W; ++w) v += red[w][i][lane];
        return v;
      };
      const int64_t out = (int64_t)list[m] * a.ldo + n0 + 4 * g;
      if (EPI == EPI_SILU) {
        if (wave) continue;
        const float s = a.factor ? a.factor[list[m] / a.per] : 1.0f;
        const f32x4 z = total(0) * s, u = total(1) * s;
        f32x4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = silu_fast(z[e]) * u[e];
        st4((bf16_t*)a.out + out, y);
      } else {
        st4((float*)a.out + out + 8 * wave, total(wave));
      }
    }
  };
  if (count <= 8) run(std::true_type{});
  else run(std::false_type{});
}
static_assert(W == 2, "the epilogue: a wave per operand");

template <int EPI>
md_status launch(const LmExpertGemm& a, int n, hipStream_t s) {
  hipLaunchKernelGGL(expert_gemm_kernel<EPI>, dim3(n / (EPI == EPI_SILU ? 8 : 16), a.n < a.experts ? a.n : a.experts), dim3(64 * W), 0, s, a);
  return md_launch_status();
}

inline bool takes(const LmExpertGemm& a) {
  return a.n >= 1 && a.n <= LM_EXPERT_CHOICES && a.per >= 1 && a.k >= 64 && a.k % 64 == 0 && a.lda >= a.k && a.lda % 8 == 0 && a.ldo % 4 == 0 &&
         a.a_rows >= 1 && (int64_t)a.a_rows * a.lda * 2 < (1ll << 31) && ((a.n - 1) / a.per) < a.a_rows && a.experts >= 1 && a.experts <= 65535 &&
         (((uintptr_t)a.a | (uintptr_t)a.w | (uintptr_t)a.out) & 15) == 0;
}

}  // namespace

// Up to ten choices per expert (the sums of more than 16 read the weights again): 24 layers of 32 experts, both products and what sorts the
// choices, 80 rows 2.92 ms against 3.18 of 64-row tiles, 100 rows 3.48 against 3.21.  The line is drawn for choices that spread.  Where all rows choose the same
// experts (copies of one text) it would lie at 32 rows: a step of two layers, 32 experts of 1360, 32 / 48 / 80 rows 197 / 263 / 391 us against 221 / 228 /
// 300 of tiles (spread: 80 rows 363 against 403).  Two tiles of 16 rows per pass cost registers, 2 to 7 % of spread choices; the workgroups of experts without
// choices as helpers 4 to 11 % of 20 to 32 alike rows.
bool lm_expert_step_takes(int rows, int top, int experts) {
  const int64_t n = (int64_t)rows * top;
  return n <= LM_EXPERT_CHOICES && n <= (int64_t)10 * experts && experts <= 65535;
}

md_status lm_expert_silu(const LmExpertGemm& a, hipStream_t s) {
  MD_CHECK_ARG(takes(a) && a.ff_pad > 0 && a.ff_pad % 64 == 0);
  return launch<EPI_SILU>(a, a.ff_pad, s);
}

md_status lm_expert_rows(const LmExpertGemm& a, int n, hipStream_t s) {
  MD_CHECK_ARG(takes(a) && n > 0 && n % 64 == 0 && a.ldo >= n);
  return launch<EPI_ROWS>(a, n, s);
}
