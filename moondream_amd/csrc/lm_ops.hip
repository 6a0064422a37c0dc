// Row-wise steps of the layered language models.
//
// The residual stream is fp32 [rows][width_pad] whatever the model's dtype; columns width .. width_pad - 1 stay zero (the linears'
// padded rows are zero), and the normed rows carry zeros there, so they feed a GEMM whose K is padded.
#include "lm_internal.hpp"

namespace {

template <typename T>
__global__ __launch_bounds__(256) void lm_embed_kernel(const T* __restrict__ table, int64_t ld, const int32_t* __restrict__ tokens,
                                                       float* __restrict__ x, int vocab) {
  const int row = blockIdx.x;
  const int id = min(max(tokens[row], 0), vocab - 1);
  const T* src = table + (int64_t)id * ld;
  float* dst = x + (int64_t)row * ld;
  for (int c = threadIdx.x * 4; c < ld; c += 1024) st4(dst + c, ld4(src + c));
}

struct ResidArgs {
  float* x;
  int64_t ldx;
  const void* src;     // rows of T, or fp32 partial products
  int64_t lds, slice_stride;
  int slices;
  md_rms_weight w;
  float eps;
  int width, width_pad;
  void* y;
  int64_t ldy;
  const int32_t* rows_idx;
  int write_x;
};

// SRC 0: nothing to add, 1: rows of T, 2: K-slice partial products.  NV: f32x4 per thread (256 threads cover width_pad).
template <typename T, int SRC, int NV>
__global__ __launch_bounds__(256) void resid_norm_kernel(const ResidArgs a) {
  __shared__ float red[4];
  const int row = a.rows_idx ? a.rows_idx[blockIdx.x] : blockIdx.x;
  float* xr = a.x + (int64_t)row * a.ldx;
  f32x4 v[NV];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (threadIdx.x + i * 256) * 4;
    if (c >= a.width_pad) continue;
    v[i] = *(const f32x4*)(xr + c);
    if (SRC == 1) v[i] += ld4((const T*)a.src + (int64_t)row * a.lds + c);
    if (SRC == 2) {
      const float* p = (const float*)a.src + (int64_t)row * a.lds + c;
      f32x4 sum = *(const f32x4*)p;
      for (int k = 1; k < a.slices; ++k) sum += *(const f32x4*)(p + k * a.slice_stride);
      v[i] += sum;
    }
    if (SRC != 0 && a.write_x) *(f32x4*)(xr + c) = v[i];
    ss += v[i][0] * v[i][0] + v[i][1] * v[i][1] + v[i][2] * v[i][2] + v[i][3] * v[i][3];
  }
  if (a.y == nullptr) return;  // (uniform: the last sum of a forward whose logits are not wanted)
  ss = block_sum_256(ss, red);
  const float r = 1.0f / sqrtf(ss / (float)a.width + a.eps);
  T* yr = (T*)a.y + (int64_t)blockIdx.x * a.ldy;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (threadIdx.x + i * 256) * 4;
    if (c >= a.width_pad) continue;
    f32x4 g;
    if (a.w.stride == 0) g = f32x4{a.w.w[0], a.w.w[0], a.w.w[0], a.w.w[0]};
    else
#pragma unroll
      for (int e = 0; e < 4; ++e) g[e] = c + e < a.width ? a.w.w[(int64_t)(c + e) * a.w.stride] : 0.f;
    st4(yr + c, v[i] * r * g);
  }
}

template <typename T, int SRC>
md_status launch_resid(const ResidArgs& a, int rows, hipStream_t s) {
  if (rows == 0) return MD_OK;
  if (a.width_pad <= 1024) hipLaunchKernelGGL((resid_norm_kernel<T, SRC, 1>), dim3(rows), dim3(256), 0, s, a);
  else if (a.width_pad <= 2048) hipLaunchKernelGGL((resid_norm_kernel<T, SRC, 2>), dim3(rows), dim3(256), 0, s, a);
  else if (a.width_pad <= 4096) hipLaunchKernelGGL((resid_norm_kernel<T, SRC, 4>), dim3(rows), dim3(256), 0, s, a);
  else if (a.width_pad <= 8192) hipLaunchKernelGGL((resid_norm_kernel<T, SRC, 8>), dim3(rows), dim3(256), 0, s, a);
  else if (a.width_pad <= 16384) hipLaunchKernelGGL((resid_norm_kernel<T, SRC, 16>), dim3(rows), dim3(256), 0, s, a);
  else return MD_ERR_UNSUPPORTED;
  return md_launch_status();
}

template <typename T>
__global__ __launch_bounds__(256) void silu_mul_kernel(const T* __restrict__ gu, int64_t ldg, T* __restrict__ act, int64_t lda, int rows, int ff_pad) {
  const int per_row = ff_pad / 4;
  const int64_t n = (int64_t)rows * per_row;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int64_t row = i / per_row;
    const int c = (int)(i - row * per_row) * 4;
    const T* g = gu + row * ldg + c;
    const f32x4 z = ld4(g), u = ld4(g + ff_pad);
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = silu_for<T>(z[e]) * u[e];
    st4(act + row * lda + c, o);
  }
}

__global__ __launch_bounds__(256) void reduce_silu_mul_kernel(const float* __restrict__ part, int slices, int64_t ldp, int64_t stride,
                                                              bf16_t* __restrict__ act, int64_t lda, int rows, int ff_pad) {
  const int per_row = ff_pad / 4;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= rows * per_row) return;
  const int row = i / per_row, c = (i - row * per_row) * 4;
  const float* p = part + (int64_t)row * ldp + c;
  f32x4 z = *(const f32x4*)p, u = *(const f32x4*)(p + ff_pad);
  for (int k = 1; k < slices; ++k) {
    z += *(const f32x4*)(p + k * stride);
    u += *(const f32x4*)(p + k * stride + ff_pad);
  }
  f32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = silu_fast(z[e]) * u[e];
  st4(act + (int64_t)row * lda + c, o);
}

__global__ __launch_bounds__(256) void reduce_rows_kernel(const float* __restrict__ part, int slices, int64_t ldp, int64_t stride,
                                                          const bf16_t* __restrict__ bias, bf16_t* __restrict__ out, int64_t ldo, int rows, int n) {
  const int per_row = n / 4, i = blockIdx.x * 256 + threadIdx.x;
  if (i >= rows * per_row) return;
  const int row = i / per_row, c = (i - row * per_row) * 4;
  const float* p = part + (int64_t)row * ldp + c;
  f32x4 y = bias ? ld4(bias + c) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < slices; ++k) y += *(const f32x4*)(p + k * stride);
  st4(out + (int64_t)row * ldo + c, y);
}

}  // namespace

md_status lm_embed(int dtype, const void* table, int64_t ld, const int32_t* tokens, float* x, int rows, int vocab, hipStream_t s) {
  if (dtype == MD_DTYPE_F32)
    hipLaunchKernelGGL(lm_embed_kernel<float>, dim3(rows), dim3(256), 0, s, (const float*)table, ld, tokens, x, vocab);
  else
    hipLaunchKernelGGL(lm_embed_kernel<bf16_t>, dim3(rows), dim3(256), 0, s, (const bf16_t*)table, ld, tokens, x, vocab);
  return md_launch_status();
}

md_status lm_resid_norm(int dtype, float* x, int64_t ldx, const void* src, int64_t lds, const md_rms_weight& w, float eps, int width,
                        int width_pad, void* y, int64_t ldy, const int32_t* rows_idx, bool write_x, int rows, hipStream_t s) {
  const ResidArgs a{x, ldx, src, lds, 0, 1, w, eps, width, width_pad, y, ldy, rows_idx, write_x ? 1 : 0};
  if (dtype == MD_DTYPE_F32) return src ? launch_resid<float, 1>(a, rows, s) : launch_resid<float, 0>(a, rows, s);
  return src ? launch_resid<bf16_t, 1>(a, rows, s) : launch_resid<bf16_t, 0>(a, rows, s);
}

md_status lm_reduce_resid_norm(float* x, int64_t ldx, const float* part, int slices, int64_t ldp, int64_t slice_stride,
                               const md_rms_weight& w, float eps, int width, int width_pad, void* y, int64_t ldy, const int32_t* rows_idx,
                               bool write_x, int rows, hipStream_t s) {
  const ResidArgs a{x, ldx, part, ldp, slice_stride, slices, w, eps, width, width_pad, y, ldy, rows_idx, write_x ? 1 : 0};
  return launch_resid<bf16_t, 2>(a, rows, s);
}

md_status lm_silu_mul(int dtype, const void* gu, int64_t ldg, void* act, int64_t lda, int rows, int ff_pad, hipStream_t s) {
  const int64_t n = (int64_t)rows * (ff_pad / 4);
  const unsigned grid = (unsigned)((n + 255) / 256 < 8192 ? (n + 255) / 256 : 8192);
  if (dtype == MD_DTYPE_F32)
    hipLaunchKernelGGL(silu_mul_kernel<float>, dim3(grid), dim3(256), 0, s, (const float*)gu, ldg, (float*)act, lda, rows, ff_pad);
  else
    hipLaunchKernelGGL(silu_mul_kernel<bf16_t>, dim3(grid), dim3(256), 0, s, (const bf16_t*)gu, ldg, (bf16_t*)act, lda, rows, ff_pad);
  return md_launch_status();
}

md_status lm_reduce_silu_mul(const float* part, int slices, int64_t ldp, int64_t slice_stride, void* act, int64_t lda, int rows, int ff_pad,
                             hipStream_t s) {
  const int n = rows * (ff_pad / 4);
  hipLaunchKernelGGL(reduce_silu_mul_kernel, dim3((n + 255) / 256), dim3(256), 0, s, part, slices, ldp, slice_stride, (bf16_t*)act, lda, rows,
                     ff_pad);
  return md_launch_status();
}

md_status lm_reduce_rows(const float* part, int slices, int64_t ldp, int64_t slice_stride, const void* bias, void* out, int64_t ldo, int rows, int n,
                         hipStream_t s) {
  hipLaunchKernelGGL(reduce_rows_kernel, dim3((rows * (n / 4) + 255) / 256), dim3(256), 0, s, part, slices, ldp, slice_stride, (const bf16_t*)bias,
                     (bf16_t*)out, ldo, rows, n);
  return md_launch_status();
}
