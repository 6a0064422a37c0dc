// Mixture of experts: router, choice, and the grouping of a step's rows by expert.
//
//   route_row_kernel    one workgroup per row: logits on the vector ALUs (any dtype), choice and weights; a decode step, fp32 models
//   route_tile_kernel   sixteen rows per workgroup: logits on the matrix cores (bf16 operands, fp32 sums), choice and weights
//   group_kernel        one workgroup per expert: its slots in row order, deterministic, no atomics
// The products over the slots are gemm_bf16.hip's and gemm_f32.hip's; those of few rows per expert are gemm_experts.hip's and need no group_kernel.
//
// Logits, softmax and weights are fp32.  A slot is one (row, chosen expert) pair; slots are numbered expert by expert.
#include "gemm_internal.hpp"
#include "lm_internal.hpp"

namespace {

// floats in a total order (NaN included): a larger key, a larger float
__device__ __forceinline__ unsigned order_key(float z) {
  const unsigned u = __builtin_bit_cast(unsigned, z);
  return u & 0x80000000u ? ~u : u | 0x80000000u;
}

// one wave: the `top` largest of z[0 .. n) (LDS; ties: the lower index), largest first, and the softmax over them.  An expert's place is the
// number of experts before it.
__device__ __forceinline__ void choose(const float* z, int n, int top, int32_t* chosen, float* weight) {
  const int lane = threadIdx.x & 63;
  auto place = [&](int e, unsigned key) {
    int before = 0;
#pragma unroll 8
    for (int k = 0; k < n; ++k) {
      const unsigned other = order_key(z[k]);
      before += other > key || (other == key && k < e);
    }
    return before;
  };
  float best = -INFINITY;
  for (int e = lane; e < n; e += 64) best = fmaxf(best, z[e]);
  best = wave_max(best);
  if (n <= 64) {  // (uniform) one expert per lane
    const float mine = lane < n ? z[lane] : -INFINITY;
    const int at = lane < n ? place(lane, order_key(mine)) : n;
    const float w = at < top ? expf(mine - best) : 0.f, sum = wave_sum(w);
    if (at < top) {
      chosen[at] = lane;
      weight[at] = w / sum;
    }
    return;
  }
  float sum = 0.f;
  for (int e = lane; e < n; e += 64)
    if (place(e, order_key(z[e])) < top) sum += expf(z[e] - best);
  sum = wave_sum(sum);
  for (int e = lane; e < n; e += 64) {
    const int at = place(e, order_key(z[e]));
    if (at < top) {
      chosen[at] = e;
      weight[at] = expf(z[e] - best) / sum;
    }
  }
}

// sixteen waves, each every sixteenth expert, two at a time
template <typename T>
__global__ __launch_bounds__(1024) void route_row_kernel(const LmRoute a) {
  extern __shared__ float z[];
  constexpr int BATCH = 4;  // loads of a row in flight
  const int row = blockIdx.x, lane = threadIdx.x & 63;
  const T* h = (const T*)a.h + (int64_t)row * a.k_pad;
  // (requested first and used last, without a branch)
  const float* sumsq = a.sumsq + (int64_t)row * a.sumsq_n;
  f32x4 sq = *(const f32x4*)(a.sumsq ? sumsq + min(lane * 4, a.sumsq_n - 4) : (const float*)a.router);
  for (int e = threadIdx.x >> 6; e < a.experts; e += 32) {
    const int e2 = min(e + 16, a.experts - 1);
    const T *w = (const T*)a.router + (int64_t)e * a.k_pad, *w2 = (const T*)a.router + (int64_t)e2 * a.k_pad;
    const float bias = a.bias[e], bias2 = a.bias[e2];
    f32x4 s = {0.f, 0.f, 0.f, 0.f}, s2 = s;
    for (int k0 = lane * 8; k0 < a.k_pad; k0 += 512 * BATCH) {
      decltype(ld8(h)) x[BATCH], y[BATCH], y2[BATCH];
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        const int k = min(k0 + 512 * i, a.k_pad - 8);
        x[i] = ld8(h + k);
        y[i] = ld8(w + k);
        y2[i] = ld8(w2 + k);
      }
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        const float in = k0 + 512 * i < a.k_pad ? 1.f : 0.f;  // (what was read again past the end)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const f32x4 xv = half8(x[i], p) * in;
          s += xv * half8(y[i], p);
          s2 += xv * half8(y2[i], p);
        }
      }
    }
    const float t = wave_sum(s[0] + s[1] + s[2] + s[3]), t2 = wave_sum(s2[0] + s2[1] + s2[2] + s2[3]);
    float factor = 1.0f;
    if (a.sumsq) {
      f32x4 q = lane * 4 < a.sumsq_n ? sq : f32x4{0.f, 0.f, 0.f, 0.f};
      for (int c = 256 + lane * 4; c < a.sumsq_n; c += 256) q += *(const f32x4*)(sumsq + c);  // (widths above 2048)
      factor = 1.0f / sqrtf(wave_sum((q[0] + q[1]) + (q[2] + q[3])) / (float)a.width + a.eps);
    }
    if (lane == 0) {
      z[e] = t * factor + bias;
      if (e + 16 < a.experts) z[e2] = t2 * factor + bias2;
      if (e == 0 && a.sumsq) a.factor[row] = factor;
    }
  }
  __syncthreads();
  if (threadIdx.x < 64) choose(z, a.experts, a.top, a.chosen + (int64_t)row * a.top, a.weight + (int64_t)row * a.top);
}

// ET: tiles of 16 experts.  The waves share K, their sums meet in LDS.
template <int ET>
__global__ __launch_bounds__(256) void route_tile_kernel(const LmRoute a) {
  __shared__ float part[4][16][16 * ET + 1], z[4][16 * ET];
  constexpr int BATCH = ET <= 2 ? 8 : ET == 4 ? 4 : 2;  // K steps in flight
  const int r0 = blockIdx.x * 16, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const bf16_t* h = (const bf16_t*)a.h + (int64_t)min(r0 + r, a.rows - 1) * a.k_pad + 8 * q;
  const bf16_t* w[ET];
  f32x4 acc[ET];
#pragma unroll
  for (int t = 0; t < ET; ++t) {
    w[t] = (const bf16_t*)a.router + (int64_t)min(16 * t + r, a.experts - 1) * a.k_pad + 8 * q;
    acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (int k0 = 32 * wave; k0 < a.k_pad; k0 += 128 * BATCH) {
    u32x4 x[BATCH], y[BATCH][ET];
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const int k = min(k0 + 128 * i, a.k_pad - 32);
      x[i] = *(const u32x4*)(h + k);
#pragma unroll
      for (int t = 0; t < ET; ++t) y[i][t] = *(const u32x4*)(w[t] + k);
    }
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      if (k0 + 128 * i >= a.k_pad) x[i] = u32x4{0u, 0u, 0u, 0u};  // (what was read again past the end)
#pragma unroll
      for (int t = 0; t < ET; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(md_bf16x8v, x[i]), __builtin_bit_cast(md_bf16x8v, y[i][t]), acc[t], 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < ET; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) part[wave][4 * q + e][16 * t + r] = acc[t][e];
  __syncthreads();
  for (int i = wave; i < 16 && r0 + i < a.rows; i += 4) {
    for (int e = lane; e < a.experts; e += 64) z[wave][e] = part[0][i][e] + part[1][i][e] + part[2][i][e] + part[3][i][e] + a.bias[e];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    choose(z[wave], a.experts, a.top, a.chosen + (int64_t)(r0 + i) * a.top, a.weight + (int64_t)(r0 + i) * a.top);
  }
}

// grid (experts), sixteen waves, each with a run of consecutive choices, 64 at a time: how many fall on lower experts and on this one, then
// this expert's slots in the order of the rows
__global__ __launch_bounds__(1024) void group_kernel(const LmRoute a) {
  __shared__ int lows[16], mines[16];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = a.rows * a.top;
  const int per = (n + 1023) / 1024 * 64, i0 = wave * per, i1 = min(i0 + per, n);
  const unsigned long long before = (1ull << lane) - 1;
  auto each = [&](auto f) {
    constexpr int BATCH = 16;
    for (int b = i0; b < i1; b += 64 * BATCH) {
      int c[BATCH];
#pragma unroll
      for (int k = 0; k < BATCH; ++k) {
        const int i = b + 64 * k + lane;
        c[k] = a.chosen[min(i, n - 1)];
        if (i >= i1) c[k] = a.experts;  // (nobody's)
      }
#pragma unroll
      for (int k = 0; k < BATCH; ++k) f(b + 64 * k + lane, c[k]);
    }
  };
  int lower = 0, mine = 0;  // (wave-uniform)
  each([&](int, int c) {
    lower += __popcll(__ballot(c < e));
    mine += __popcll(__ballot(c == e));
  });
  if (lane == 0) {
    lows[wave] = lower;
    mines[wave] = mine;
  }
  __syncthreads();
  int base = 0, at = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    base += lows[w];
    if (w < wave) at += mines[w];
  }
  at += base;
  if (tid == 0) {
    a.offsets[e] = base;
    if (e == a.experts - 1) a.offsets[a.experts] = n;
  }
  if (mine == 0) return;
  each([&](int i, int c) {
    const unsigned long long who = __ballot(c == e);
    if (c == e) {
      const int slot = at + __popcll(who & before);
      a.row_of[slot] = i / a.top;
      a.slot_of[i] = slot;
    }
    at += __popcll(who);
  });
}

}  // namespace

md_status lm_route(int dtype, const LmRoute& a, hipStream_t s) {
  if (a.experts > 8192) return MD_ERR_UNSUPPORTED;
  const int lds = a.experts * 4;
  if (dtype == MD_DTYPE_F32) hipLaunchKernelGGL(route_row_kernel<float>, dim3(a.rows), dim3(1024), lds, s, a);
  else if (a.rows <= 128 || a.experts > 128) hipLaunchKernelGGL(route_row_kernel<bf16_t>, dim3(a.rows), dim3(1024), lds, s, a);
  else {
    auto fn = a.experts <= 16 ? route_tile_kernel<1> : a.experts <= 32 ? route_tile_kernel<2> : a.experts <= 64 ? route_tile_kernel<4> : route_tile_kernel<8>;
    hipLaunchKernelGGL(fn, dim3((a.rows + 15) / 16), dim3(256), 0, s, a);
  }
  MD_TRY(md_launch_status());
  if (!a.offsets) return MD_OK;
  hipLaunchKernelGGL(group_kernel, dim3(a.experts), dim3(1024), 0, s, a);
  return md_launch_status();
}
