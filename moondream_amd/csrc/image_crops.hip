// Crops of images, cut on the device: per image the whole picture at crop x crop and tiles_y x tiles_x windows at `stride` of the picture
// resized to (tiles * stride + crop - stride) (reference: image_crops.py:58-167).  The resize is the separable convolution with the Lanczos
// window of three lobes, and gives the bytes that the host's PIL branch gives: weights in fp64, normalised and rounded to 22 bits behind the
// point, whole-number sums, columns first, bytes between the two passes.
//
// On the host this is 60 to 70 passes over the picture's bytes in one thread per image (768 x 1024: 21 ms, with the device waiting); here the
// source goes over the bus once (2.4 MB, the 13 crops are 5.6 MB) and four such images take 130 us.  Bound by the byte loads of the taps.
#include "md_common.hpp"

namespace {

constexpr int BITS = 22, LOBES = 3, ROWS = 4;

struct Image {
  int32_t height, width, tiles_y, tiles_x;
};
inline Image image(const int32_t* im, int i) { return {im[4 * i], im[4 * i + 1], im[4 * i + 2], im[4 * i + 3]}; }

struct Axis {  // table: first source index [out], taps [out], weights [tap][out]
  int64_t table;
  int32_t in, out, taps, pad;
};
struct Plane {  // a picture resized along its rows
  int64_t src, dst;
  int32_t h, w, ld, axis;
};
struct Crop {
  int64_t src;
  int32_t ld, axis, y0, x0;  // x0: bytes
};

inline int taps_of(int in, int out) { return in == out ? 1 : 2 * (int)((int64_t)LOBES * (in > out ? in : out) / out + 1) + 1; }
inline int64_t up16(int64_t n) { return (n + 15) & ~(int64_t)15; }

struct Sizes {
  int64_t plan, staged, work;
  int32_t crops, max_out, max_h, max_w;
};

// Where everything lies; written to plan (axes, planes and crops of all images, one after the other) if there is one.  False: out of range.
bool lay_out(const int32_t* im, int n, int crop, int stride, Sizes& z, void* plan, int64_t* offsets) {
  if (!im || n <= 0 || n > 8192 || crop <= 0 || (crop & 1) || stride <= 0 || (stride & 1) || crop <= stride || crop > 4096) return false;
  int64_t crops = 0;
  for (int i = 0; i < n; ++i) {
    const Image m = image(im, i);
    if (m.height <= 0 || m.width <= 0 || m.height > (1 << 18) || m.width > (1 << 18) || m.tiles_y <= 0 || m.tiles_x <= 0) return false;
    if (m.tiles_y > 256 || m.tiles_x > 256) return false;
    crops += 1 + (int64_t)m.tiles_y * m.tiles_x;
  }
  if (crops > 65535) return false;
  Axis* axes = (Axis*)plan;
  Plane* planes = (Plane*)(axes + 4 * (int64_t)n);
  Crop* cut = (Crop*)(planes + 2 * (int64_t)n);
  z = Sizes{up16((int64_t)n * (4 * sizeof(Axis) + 2 * sizeof(Plane)) + crops * (int64_t)sizeof(Crop)), 0, 0, (int32_t)crops, 0, 0, 0};
  z.staged = z.plan;
  int64_t at = 0;
  for (int i = 0; i < n; ++i) {
    const Image m = image(im, i);
    const int64_t src = z.staged;
    if (offsets) offsets[i] = src;
    z.staged += up16((int64_t)m.height * m.width * 3);
    const bool one = m.tiles_y == 1 && m.tiles_x == 1;  // both pictures are the same
    Plane p[2];
    for (int k = 0; k < 2; ++k) {
      const int oh = k ? crop : m.tiles_y * stride + crop - stride, ow = k ? crop : m.tiles_x * stride + crop - stride;
      const int32_t in[2] = {m.width, m.height}, out[2] = {ow, oh};
      for (int d = 0; d < 2; ++d) {
        const Axis a = {z.work, in[d], k && one ? 0 : out[d], taps_of(in[d], out[d]), 0};
        z.work += up16((int64_t)a.out * (a.taps + 2) * 4);
        if (plan) axes[4 * i + 2 * k + d] = a;
        if (z.max_out < out[d]) z.max_out = out[d];
      }
      p[k] = Plane{src, z.work, k && one ? 0 : m.height, m.width, (ow * 3 + 3) & ~3, 4 * i + 2 * k};
      z.work += up16((int64_t)p[k].h * p[k].ld);
      if (plan) planes[2 * i + k] = p[k];
      if (z.max_w < ow) z.max_w = ow;
    }
    if (z.max_h < m.height) z.max_h = m.height;
    if (plan) {
      const int g = one ? 0 : 1;
      cut[at] = Crop{p[g].dst, p[g].ld, p[g].axis + 1, 0, 0};
      for (int y = 0; y < m.tiles_y; ++y)
        for (int x = 0; x < m.tiles_x; ++x) cut[at + 1 + y * m.tiles_x + x] = Crop{p[0].dst, p[0].ld, p[0].axis + 1, y * stride, x * stride * 3};
    }
    at += 1 + m.tiles_y * m.tiles_x;
  }
  return true;
}

__device__ double lanczos(double x) {
  if (x == 0.0) return 1.0;
  if (!(x > -LOBES && x < LOBES)) return 0.0;
  const double a = M_PI * x, b = a / LOBES;
  return sin(a) / a * (sin(b) / b);
}

// grid (outputs / 4, axes): a wave per output.  (What an ulp of the sine or a fused product moves lies 2^-27 of a weight's last bit away.)
__global__ __launch_bounds__(256) void crop_weights_kernel(const Axis* axes, char* work) {
  const Axis a = axes[blockIdx.y];
  const int o = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (o >= a.out) return;
  int32_t* tab = (int32_t*)(work + a.table);
  if (a.in == a.out) {
    if (lane == 0) {
      tab[o] = o;
      tab[a.out + o] = 1;
      tab[2 * a.out + o] = 1 << BITS;
    }
    return;
  }
  const double scale = (double)a.in / a.out, wide = scale > 1.0 ? scale : 1.0, reach = LOBES * wide, centre = (o + 0.5) * scale;
  const int lo = max((int)(centre - reach + 0.5), 0), n = min(min((int)(centre + reach + 0.5), a.in) - lo, a.taps);
  double sum = 0.0;
  for (int t = lane; t < n; t += 64) sum += lanczos((t + lo - centre + 0.5) / wide);
#pragma unroll
  for (int m = 32; m; m >>= 1) sum += __shfl_xor(sum, m);
  for (int t = lane; t < n; t += 64) {
    const double w = lanczos((t + lo - centre + 0.5) / wide) / sum * (double)(1 << BITS);
    tab[(2 + t) * (int64_t)a.out + o] = (int32_t)(w < 0.0 ? w - 0.5 : w + 0.5);
  }
  if (lane == 0) {
    tab[o] = lo;
    tab[a.out + o] = n;
  }
}

__device__ __forceinline__ uint32_t to_byte(int v) { return (uint32_t)min(max(v >> BITS, 0), 255); }

// grid (columns / 256, rows / ROWS, planes): a thread has one column of ROWS rows, so that a weight serves 12 products
__global__ __launch_bounds__(256) void crop_rows_kernel(const Axis* axes, const Plane* planes, const uint8_t* staged, char* work) {
  const Plane p = planes[blockIdx.z];
  const Axis a = axes[p.axis];
  const int o = blockIdx.x * 256 + threadIdx.x;
  if (o >= a.out) return;
  const int32_t* tab = (const int32_t*)(work + a.table);
  const int lo = tab[o], n = tab[a.out + o];
  for (int y0 = blockIdx.y * ROWS; y0 < p.h; y0 += gridDim.y * ROWS) {
    const uint8_t* s[ROWS];
    int acc[ROWS][3];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      s[r] = staged + p.src + ((int64_t)min(y0 + r, p.h - 1) * p.w + lo) * 3;
#pragma unroll
      for (int c = 0; c < 3; ++c) acc[r][c] = 1 << (BITS - 1);
    }
    for (int t = 0; t < n; ++t) {
      const int k = tab[(2 + t) * (int64_t)a.out + o];
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) acc[r][c] += s[r][3 * t + c] * k;
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
      if (y0 + r < p.h)
#pragma unroll
        for (int c = 0; c < 3; ++c) work[p.dst + (int64_t)(y0 + r) * p.ld + 3 * o + c] = (char)to_byte(acc[r][c]);
  }
}

// grid (byte pairs of a crop's row / 256, rows, crops)
__global__ __launch_bounds__(256) void crop_columns_kernel(const Axis* axes, const Crop* crops, const char* work, uint8_t* out, int crop) {
  const int i = blockIdx.x * 256 + threadIdx.x, y = blockIdx.y, bytes = crop * 3;
  if (2 * i >= bytes) return;
  const Crop c = crops[blockIdx.z];
  const Axis a = axes[c.axis];
  const int32_t* tab = (const int32_t*)(work + a.table) + c.y0 + y;
  const int lo = tab[0], n = tab[a.out];
  const char* s = work + c.src + (int64_t)lo * c.ld + c.x0 + 2 * i;
  int a0 = 1 << (BITS - 1), a1 = a0;
#pragma unroll 4
  for (int t = 0; t < n; ++t) {
    const uint32_t v = *(const uint16_t*)(s + (int64_t)t * c.ld);
    const int k = tab[(2 + t) * (int64_t)a.out];
    a0 += (int)(v & 255) * k;
    a1 += (int)(v >> 8) * k;
  }
  *(uint16_t*)(out + ((int64_t)blockIdx.z * crop + y) * bytes + 2 * i) = (uint16_t)(to_byte(a0) | to_byte(a1) << 8);
}

}  // namespace

extern "C" size_t md_crops_staged_bytes(const int32_t* images, int32_t n, int32_t crop, int32_t stride, int64_t* offsets) {
  Sizes z;
  return lay_out(images, n, crop, stride, z, nullptr, offsets) ? (size_t)z.staged : 0;
}

extern "C" size_t md_crops_workspace_bytes(const int32_t* images, int32_t n, int32_t crop, int32_t stride) {
  Sizes z;
  return lay_out(images, n, crop, stride, z, nullptr, nullptr) ? (size_t)z.work : 0;
}

extern "C" md_status md_crops_plan(const int32_t* images, int32_t n, int32_t crop, int32_t stride, void* staged, size_t staged_bytes) {
  Sizes z;
  MD_CHECK_ARG(staged && ((uintptr_t)staged & 15) == 0 && lay_out(images, n, crop, stride, z, nullptr, nullptr) && staged_bytes >= (size_t)z.staged);
  lay_out(images, n, crop, stride, z, staged, nullptr);
  return MD_OK;
}

extern "C" md_status md_cut_crops(const int32_t* images, int32_t n, int32_t crop, int32_t stride, const void* staged, void* workspace,
                                  size_t workspace_bytes, void* out, void* stream) {
  Sizes z;
  MD_CHECK_ARG(staged && workspace && out && lay_out(images, n, crop, stride, z, nullptr, nullptr));
  MD_CHECK_ARG((((uintptr_t)staged | (uintptr_t)workspace) & 15) == 0 && ((uintptr_t)out & 1) == 0);
  if (workspace_bytes < (size_t)z.work) return MD_ERR_WORKSPACE;
  const hipStream_t s = (hipStream_t)stream;
  const Axis* axes = (const Axis*)staged;
  const Plane* planes = (const Plane*)(axes + 4 * (int64_t)n);
  const Crop* crops = (const Crop*)(planes + 2 * (int64_t)n);
  hipLaunchKernelGGL(crop_weights_kernel, dim3((z.max_out + 3) / 4, 4 * n), dim3(256), 0, s, axes, (char*)workspace);
  MD_TRY(md_launch_status());
  const int rows = min((z.max_h + ROWS - 1) / ROWS, 65535);
  hipLaunchKernelGGL(crop_rows_kernel, dim3((z.max_w + 255) / 256, rows, 2 * n), dim3(256), 0, s, axes, planes, (const uint8_t*)staged, (char*)workspace);
  MD_TRY(md_launch_status());
  hipLaunchKernelGGL(crop_columns_kernel, dim3((crop * 3 / 2 + 255) / 256, crop, z.crops), dim3(256), 0, s, axes, crops, (const char*)workspace,
                     (uint8_t*)out, crop);
  return md_launch_status();
}
