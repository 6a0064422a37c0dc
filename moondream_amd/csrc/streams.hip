// Row-wise steps of models with several residual streams, learned positions or expert feed-forwards.
//
// The streams are fp32 [S][rows][width_pad] whatever the model's dtype, columns width .. width_pad - 1 zero.  Between two sublayers ONE
// launch per step: the old streams are read once, mixed and written with the sublayer's result added, the next sublayer's input is their
// weighted sum, normed.  A thread owns four columns of every stream (NV such pieces), so the S x S mixture stays in its registers.
#include "lm_internal.hpp"

namespace {

template <typename T, int NV>
__global__ __launch_bounds__(256) void embed_streams_kernel(const T* __restrict__ table, const T* __restrict__ pos, int positions, md_rms_weight w,
                                                            float eps, int width, int width_pad, const int32_t* __restrict__ tokens,
                                                            const int32_t* __restrict__ row_pos, float* __restrict__ x, int64_t stride, int streams,
                                                            int vocab) {
  __shared__ float red[4];
  const int row = blockIdx.x;
  const T* src = table + (int64_t)min(max(tokens[row], 0), vocab - 1) * width_pad;
  const T* ps = pos ? pos + (int64_t)min(max(row_pos[row], 0), positions - 1) * width_pad : nullptr;
  f32x4 v[NV];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (threadIdx.x + i * 256) * 4;
    if (c >= width_pad) continue;
    v[i] = ld4(src + c);
    if (ps) v[i] += ld4(ps + c);
    ss += v[i][0] * v[i][0] + v[i][1] * v[i][1] + v[i][2] * v[i][2] + v[i][3] * v[i][3];
  }
  float r = 1.0f;
  if (w.w) r = 1.0f / sqrtf(block_sum_256(ss, red) / (float)width + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (threadIdx.x + i * 256) * 4;
    if (c >= width_pad) continue;
    if (w.w) {
      f32x4 g;
#pragma unroll
      for (int e = 0; e < 4; ++e) g[e] = c + e < width ? w.w[(int64_t)(c + e) * w.stride] : 0.f;
      v[i] = v[i] * r * g;
    }
    for (int s = 0; s < streams; ++s) *(f32x4*)(x + s * stride + (int64_t)row * width_pad + c) = v[i];
  }
}

// sum of the K-slice partial products of four columns; the usual counts with all loads in flight
__device__ __forceinline__ f32x4 slice_sum(const float* p, int slices, int64_t stride) {
  auto n = [&](auto count) {
    constexpr int N = decltype(count)::value;
    f32x4 v[N], y;
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = *(const f32x4*)(p + k * stride);
    y = v[0];
#pragma unroll
    for (int k = 1; k < N; ++k) y += v[k];
    return y;
  };
  switch (slices) {  // (uniform)
    case 1: return *(const f32x4*)p;
    case 2: return n(std::integral_constant<int, 2>{});
    case 4: return n(std::integral_constant<int, 4>{});
    case 8: return n(std::integral_constant<int, 8>{});
    default: break;
  }
  f32x4 y = *(const f32x4*)p;
  for (int k = 1; k < slices; ++k) y += *(const f32x4*)(p + k * stride);
  return y;
}

// the pending sublayer result of four columns of a row
template <typename T>
__device__ __forceinline__ f32x4 addend(const LmAddend& a, int row, int c) {
  if (a.top == 0) return a.slices == 0 ? ld4((const T*)a.src + (int64_t)row * a.ld + c) : slice_sum((const float*)a.src + (int64_t)row * a.ld + c, a.slices, a.slice_stride);
  f32x4 y = {0.f, 0.f, 0.f, 0.f};
  const float* w = a.weight + (int64_t)row * a.top;
  if (!a.slot_of) {
    const float* src = (const float*)a.src + (int64_t)row * a.top * a.ld + c;
#pragma unroll 4
    for (int k = 0; k < a.top; ++k) y += w[k] * *(const f32x4*)(src + k * a.ld);
    return y;
  }
  const int32_t* slot = a.slot_of + (int64_t)row * a.top;
  if (a.slices == 0) {
#pragma unroll 4
    for (int k = 0; k < a.top; ++k) y += w[k] * ld4((const T*)a.src + (int64_t)slot[k] * a.ld + c);
  } else if (a.slices == 1) {
#pragma unroll 4
    for (int k = 0; k < a.top; ++k) y += w[k] * *(const f32x4*)((const float*)a.src + (int64_t)slot[k] * a.ld + c);
  } else {
    for (int k = 0; k < a.top; ++k) y += w[k] * slice_sum((const float*)a.src + (int64_t)slot[k] * a.ld + c, a.slices, a.slice_stride);
  }
  return y;
}

// S > 0: exactly that many streams; 0: up to MD_LM_MAX_STREAMS
template <typename T, int S, int NV>
__global__ __launch_bounds__(256) void stream_step_kernel(const LmStreams a) {
  __shared__ float red[4];
  constexpr int SM = S > 0 ? S : MD_LM_MAX_STREAMS;
  const int n = S > 0 ? S : a.streams;
  const int row = a.rows_idx ? a.rows_idx[blockIdx.x] : blockIdx.x;
  float* xr = a.x + (int64_t)row * a.width_pad;
  const float *in_w = a.next, *out_w = a.prev ? a.prev + n : nullptr, *mix = a.prev ? a.prev + 2 * n : nullptr;
  f32x4 u[NV];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (threadIdx.x + i * 256) * 4;
    if (c >= a.width_pad) continue;
    f32x4 old[SM];
#pragma unroll
    for (int s = 0; s < SM; ++s)
      if (s < n) old[s] = *(const f32x4*)(xr + s * a.stride + c);
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    if (a.add.src) {
      const f32x4 y = addend<T>(a.add, row, c);
#pragma unroll
      for (int t = 0; t < SM; ++t) {
        if (t >= n) continue;
        f32x4 acc;
        if (mix) {
          acc = out_w[t] * y;
#pragma unroll
          for (int s = 0; s < SM; ++s)
            if (s < n) acc += mix[s * n + t] * old[s];
        } else {
          acc = old[t] + y;  // (a plain residual sum)
        }
        if (a.write_x) *(f32x4*)(xr + t * a.stride + c) = acc;
        sum += (in_w ? in_w[t] : 1.0f) * acc;
      }
    } else {
#pragma unroll
      for (int t = 0; t < SM; ++t)
        if (t < n) sum += (in_w ? in_w[t] : 1.0f) * old[t];
    }
    u[i] = sum;
    ss += sum[0] * sum[0] + sum[1] * sum[1] + sum[2] * sum[2] + sum[3] * sum[3];
    if (a.sum_out) *(f32x4*)(a.sum_out + (int64_t)row * a.width_pad + c) = sum;
  }
  if (a.y == nullptr) return;  // (uniform)
  const float r = 1.0f / sqrtf(block_sum_256(ss, red) / (float)a.width + a.eps);
  T* yr = (T*)a.y + (int64_t)blockIdx.x * a.width_pad;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (threadIdx.x + i * 256) * 4;
    if (c >= a.width_pad) continue;
    f32x4 g;
    if (a.w.stride == 1 && c + 3 < a.width) g = *(const f32x4*)(a.w.w + c);
    else
#pragma unroll
      for (int e = 0; e < 4; ++e) g[e] = c + e < a.width ? a.w.w[(int64_t)(c + e) * a.w.stride] : 0.f;
    st4(yr + c, u[i] * r * g);
  }
}

// The same for few rows whose reader norms them: no sum over a row to wait for, so a row's columns go to several workgroups (23 rows of four streams, 2048
// wide: 6.8 us -> 4.9, and the reader's operand order)
template <int S>
__global__ __launch_bounds__(64) void stream_split_kernel(const LmStreams a) {
  constexpr int SM = S > 0 ? S : MD_LM_MAX_STREAMS;
  const int n = S > 0 ? S : a.streams;
  const int row = blockIdx.x, c = (blockIdx.y * 64 + threadIdx.x) * 4;
  if (c >= a.width_pad) return;
  float* xr = a.x + (int64_t)row * a.width_pad + c;
  const float *in_w = a.next, *out_w = a.prev ? a.prev + n : nullptr, *mix = a.prev ? a.prev + 2 * n : nullptr;
  f32x4 old[SM], norm_w, sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < SM; ++s)
    if (s < n) old[s] = *(const f32x4*)(xr + s * a.stride);
#pragma unroll
  for (int e = 0; e < 4; ++e) norm_w[e] = a.w.w[(int64_t)min(c + e, a.width - 1) * a.w.stride];  // (columns beyond hold zeros)
  const f32x4 y = a.add.src ? addend<bf16_t>(a.add, row, c) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < SM; ++t) {
    if (t >= n) continue;
    f32x4 v = old[t];
    if (a.add.src) {
      if (mix) {
        v = out_w[t] * y;
#pragma unroll
        for (int s = 0; s < SM; ++s)
          if (s < n) v += mix[s * n + t] * old[s];
      } else {
        v += y;
      }
      *(f32x4*)(xr + t * a.stride) = v;
    }
    sum += (in_w ? in_w[t] : 1.0f) * v;
  }
  float q = (sum[0] * sum[0] + sum[1] * sum[1]) + (sum[2] * sum[2] + sum[3] * sum[3]);
  q += __shfl_xor(q, 1, 64);
  st4((bf16_t*)a.y + row * 8 + in_chunks(c, a.out_chunk), sum * norm_w);
  if (!(threadIdx.x & 1)) a.sumsq_out[(int64_t)row * (a.width_pad / 8) + c / 8] = q;
}

template <typename T, int S>
md_status step_by_width(const LmStreams& a, int rows, hipStream_t s) {
  if (a.width_pad <= 1024) hipLaunchKernelGGL((stream_step_kernel<T, S, 1>), dim3(rows), dim3(256), 0, s, a);
  else if (a.width_pad <= 2048) hipLaunchKernelGGL((stream_step_kernel<T, S, 2>), dim3(rows), dim3(256), 0, s, a);
  else if (a.width_pad <= 4096) hipLaunchKernelGGL((stream_step_kernel<T, S, 4>), dim3(rows), dim3(256), 0, s, a);
  else if (a.width_pad <= 16384) hipLaunchKernelGGL((stream_step_kernel<T, S, 16>), dim3(rows), dim3(256), 0, s, a);
  else return MD_ERR_UNSUPPORTED;
  return md_launch_status();
}
template <typename T>
md_status step_by_streams(const LmStreams& a, int rows, hipStream_t s) {
  switch (a.streams) {
    case 1: return step_by_width<T, 1>(a, rows, s);
    case 2: return step_by_width<T, 2>(a, rows, s);
    case 3: return step_by_width<T, 3>(a, rows, s);
    case 4: return step_by_width<T, 4>(a, rows, s);
    default: return a.streams <= MD_LM_MAX_STREAMS ? step_by_width<T, 0>(a, rows, s) : MD_ERR_UNSUPPORTED;
  }
}

template <typename T>
md_status embed(const md_lm_model* m, const int32_t* tokens, const int32_t* row_pos, float* x, int64_t stride, int rows, hipStream_t s) {
  auto go = [&](auto nv) {
    hipLaunchKernelGGL((embed_streams_kernel<T, decltype(nv)::value>), dim3(rows), dim3(256), 0, s, (const T*)m->embed, (const T*)m->pos, m->positions,
                       m->embed_norm, m->eps, m->width, m->width_pad, tokens, row_pos, x, stride, m->streams > 0 ? m->streams : 1, m->vocab);
    return md_launch_status();
  };
  if (m->width_pad <= 1024) return go(std::integral_constant<int, 1>{});
  if (m->width_pad <= 4096) return go(std::integral_constant<int, 4>{});
  if (m->width_pad <= 16384) return go(std::integral_constant<int, 16>{});
  return MD_ERR_UNSUPPORTED;
}

}  // namespace

md_status lm_embed_streams(const md_lm_model* m, const int32_t* tokens, const int32_t* row_pos, float* x, int64_t stride, int rows, hipStream_t s) {
  return m->dtype == MD_DTYPE_F32 ? embed<float>(m, tokens, row_pos, x, stride, rows, s) : embed<bf16_t>(m, tokens, row_pos, x, stride, rows, s);
}

md_status lm_stream_step(int dtype, const LmStreams& a, int rows, hipStream_t s) {
  if (rows == 0) return MD_OK;
  return dtype == MD_DTYPE_F32 ? step_by_streams<float>(a, rows, s) : step_by_streams<bf16_t>(a, rows, s);
}

md_status lm_stream_split(const LmStreams& a, int rows, hipStream_t s) {
  if (rows == 0) return MD_OK;
  if (a.streams < 1 || a.streams > MD_LM_MAX_STREAMS) return MD_ERR_UNSUPPORTED;
  auto fn = a.streams == 1 ? stream_split_kernel<1> : a.streams == 2 ? stream_split_kernel<2> : a.streams == 4 ? stream_split_kernel<4> : stream_split_kernel<0>;
  hipLaunchKernelGGL(fn, dim3(rows, (a.width_pad + 255) / 256), dim3(64), 0, s, a);
  return md_launch_status();
}
