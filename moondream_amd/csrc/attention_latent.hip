// Attention over a cached latent row per position: keys and values of every head are linear in it (k = U_k c, v = U_v c), so the cache
// holds c alone.
//
//   latent_rows_kernel     RMS norm of the step's latent rows -> cache (and, for a prefill, the packed rows of the whole context)
//   latent_gather_kernel   cached rows of earlier steps -> packed rows
//   latent_plain_kernel    one workgroup per (query row, head), in the latent space, fp32 on the vector ALUs: any dtype, any size
//   latent_prefill_kernel  bf16 prefill on the matrix cores over expanded keys and values (one GEMM makes them from the packed rows)
//   decode (bf16), in the latent space: a head's query goes through U_k^T once and meets the cached rows themselves, whatever the number of
//   heads each row is read once:
//     latent_absorb_kernel   queries -> latent space; norm and cache row of the new position
//     latent_decode_kernel   split-key attention; scores and weighted sum from one LDS copy of 32 rows
//     latent_out_kernel      sum over the splits, U_v, output gate
//
// Scores, softmax and sums are fp32; q, c, the expanded keys / values, softmax weights and queries in the latent space enter matrix products as bf16.
#include "lm_internal.hpp"

#include <algorithm>

namespace {

constexpr float LOG2E = 1.4426950408889634f;

__device__ __forceinline__ float sigmoid_f32(float z) { return 1.0f / (1.0f + expf(-z)); }

// one wave: row of the step -> normed latent row in the cache and, with `packed`, there
template <typename T>
__device__ __forceinline__ void latent_row(const LmLatent& a, int row, int seq, T* packed) {
  const int lane = threadIdx.x & 63, pos = a.r.row_pos[row];
  const T* src = (const T*)a.proj + (int64_t)row * a.ldp + a.col_c;
  T* dst = (T*)a.cache + ((int64_t)a.r.seq_slot[seq] * a.ctx + pos) * a.rp;
  float ss = 0.f;
  for (int c = lane * 4; c < a.rp; c += 256) {
    const f32x4 v = ld4(src + c);
    ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
  }
  const float r = 1.0f / sqrtf(wave_sum(ss) / (float)a.rank + a.eps);
  for (int c = lane * 4; c < a.rp; c += 256) {
    const f32x4 v = ld4(src + c) * r * *(const f32x4*)(a.norm + c);
    st4(dst + c, v);
    if (packed) st4(packed + c, v);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void latent_rows_kernel(const LmLatent a, int pack) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.r.n_rows) return;
  const int seq = a.r.row_seq[row];
  latent_row<T>(a, row, seq, pack ? (T*)a.c_rows + ((int64_t)a.seq_ctx0[seq] + a.r.row_pos[row]) * a.rp : nullptr);
}

// grid (., sequences)
template <typename T>
__global__ __launch_bounds__(256) void latent_gather_kernel(const LmLatent a) {
  const int seq = blockIdx.y;
  const int64_t n = (int64_t)a.r.seq_pos0[seq] * a.rp;
  const T* src = (const T*)a.cache + (int64_t)a.r.seq_slot[seq] * a.ctx * a.rp;
  T* dst = (T*)a.c_rows + (int64_t)a.seq_ctx0[seq] * a.rp;
  for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4; i < n; i += (int64_t)gridDim.x * 1024) st4(dst + i, ld4(src + i));
}

// grid (heads, rows)
template <typename T>
__global__ __launch_bounds__(256) void latent_plain_kernel(const LmLatent a) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  __shared__ float red[4], ps[256];
  const int h = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, R = a.rp;
  float *qs = sm, *ql = qs + a.dp, *z = ql + R;
  const int seq = a.r.row_seq[row], i = a.r.row_pos[row];
  const T* c = (const T*)a.cache + (int64_t)a.r.seq_slot[seq] * a.ctx * R;
  const T* proj = (const T*)a.proj + (int64_t)row * a.ldp;
  for (int d = tid; d < a.dp; d += 256) qs[d] = ldf(proj + a.col_q + h * a.dp + d);
  __syncthreads();
  for (int r = tid; r < R; r += 256) {
    const T* w = (const T*)a.up_k_t + ((int64_t)h * R + r) * a.dp;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int d = 0; d < a.dp; d += 4) s += *(const f32x4*)(qs + d) * ld4(w + d);  // (columns behind the head's are zeros)
    ql[r] = (s[0] + s[1]) + (s[2] + s[3]);
    z[r] = 0.f;
  }
  float m = -INFINITY, l = 0.f;
  for (int j0 = 0; j0 <= i; j0 += 256) {
    const int n = min(256, i + 1 - j0);
    __syncthreads();
    float s = -INFINITY;
    if (tid < n) {
      f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
      for (int r = 0; r < R; r += 4) d += ld4(c + (int64_t)(j0 + tid) * R + r) * *(const f32x4*)(ql + r);
      s = ((d[0] + d[1]) + (d[2] + d[3])) * a.scale;
    }
    const float wm = wave_max(s);
    if (lane == 0) red[wave] = wm;
    __syncthreads();
    const float mn = fmaxf(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])), m), f = expf(m - mn), p = expf(s - mn);
    ps[tid] = p;
    l = l * f + block_sum_256(p, red);  // (its barriers also publish ps)
    m = mn;
    for (int r = tid; r < R; r += 256) {
      float o = z[r] * f;
#pragma unroll 16
      for (int j = 0; j < n; ++j) o += ps[j] * ldf(c + (int64_t)(j0 + j) * R + r);
      z[r] = o;
    }
  }
  __syncthreads();
  for (int e = tid; e < a.vp; e += 256) {
    const T* w = (const T*)a.up_kv.w + ((int64_t)a.heads * a.dp + h * a.vp + e) * R;
    f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int r = 0; r < R; r += 4) y += *(const f32x4*)(z + r) * ld4(w + r);
    float o = ((y[0] + y[1]) + (y[2] + y[3])) / l;
    if (a.col_g >= 0) o *= sigmoid_f32(ldf(proj + a.col_g + h * a.vp + e));
    stf((T*)a.out + (int64_t)row * a.ldo + in_chunks(h * a.vp + e, a.out_chunk), o);
  }
}

// ---------------------------------------------------------------------------------------------------------------------------
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 read_tr(const bf16_t* p) {  // lane i of a 16-lane group: four rows of column i % 16 (see read_columns)
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p));
}

// Four waves of 32 queries of one (sequence, head); keys and values stream through LDS in tiles of 64, two buffers, the next tile's loads in
// registers meanwhile.  S^T = K Q^T (32x32x16), so a lane holds one query and 16 of every 32 keys: maximum and sum stay in the lane but for
// one exchange, and the weights go from the accumulators straight into the second operand of O^T += V^T P^T; the order of the keys that this
// implies is the one in which the transposing LDS reads fetch V.  D: dp / 32, C: vp / 32
// KG: groups of four waves that take the tiles of keys in turn; the second's sums go to the first through LDS.  What bounds a workgroup is the chain through its tiles
// (2 us each with one wave on a SIMD, where LDS and the address unit are half idle; 2.6 for two tiles with two), so two groups where each CU has one workgroup.
// Whole passes of 8 layers, one group and two: 16 heads of 128, one prompt of 700 tokens 771 and 757 us (28 and 24 a launch), 1000 890 : 837, 2000 1293 : 1179; 4 heads
// of 64, 1000 757 : 702, 3 x 2000 1512 : 1407.  Not for up to three tiles (7 x 100, 16 heads 684 : 690, 4 heads 556 : 590) and not past a workgroup per CU (32 heads,
// 2000 1222 : 1266).  Two groups of two waves and blocks of 64 queries: as one group or slower, each tile's loads and LDS writes serve half as many queries.
// The rule counts the workgroups and keys of the step, so a prompt's rounding hangs on the prompts beside it.  Against 64 bits, one group and two: 16 heads of 128, 700 tokens 2.03e-3
// and 2.00e-3 (sharp scores 1.89e-3, 1.80e-3), 4 of 64, 2000 tokens 2.08e-3 and 2.05e-3 (1.97e-3, 1.88e-3): weights are bf16, either way.
constexpr int value_stride(int vp) { return vp == 32 ? 32 : vp == 128 ? 160 : 96; }  // four rows of 64 bytes fall on different banks
template <int D, int C, int KG>
struct PrefillLds {
  static constexpr int KS = 32 * D + 8, VS = value_stride(32 * C), buffer = 64 * (KS + VS), OS = 32 * C + 8;
  static constexpr int tiles = 2 * KG * buffer, outputs = 4 * 32 * OS, sums = KG > 1 ? 2 * 256 * (16 * C + 2) : 0;  // (fp32: two elements)
  static constexpr int bytes = 2 * (tiles > outputs + sums ? tiles : outputs + sums);
};
template <int D, int C, int KG>
__global__ __launch_bounds__(256 * KG, 2 / KG) void latent_prefill_kernel(const LmLatent a, int n_qblk) {
  using M = PrefillLds<D, C, KG>;
  constexpr int dp = 32 * D, vp = 32 * C, KS = M::KS, VS = M::VS;
  extern __shared__ __attribute__((aligned(16))) bf16_t psm[];
  // all query blocks of a (sequence, head) on one XCD, whose L2 then holds its keys and values; the longest first
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, bh = (slot / n_qblk) * 8 + xcd;
  if (bh >= a.r.n_seq * a.heads) return;
  const int seq = bh / a.heads, h = bh - seq * a.heads, tid = threadIdx.x & 255, lane = tid & 63, hi = lane >> 5, l31 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, pos0 = a.r.seq_pos0[seq];
  const int q0 = (n_qblk - 1 - slot % n_qblk) * 128;
  if (q0 >= len) return;
  const int kv_end = pos0 + min(q0 + 128, len);
  const int w0 = q0 + 32 * wave, t = min(w0 + l31, len - 1), qpos = pos0 + t;
  const int w_lo = pos0 + min(w0, len - 1), w_hi = pos0 + min(w0 + 31, len - 1);
  const int64_t ldkv = a.up_kv.n_pad;
  const bf16_t* Kg = (const bf16_t*)a.kv + (int64_t)a.seq_ctx0[seq] * ldkv + h * dp;
  const bf16_t* Vg = (const bf16_t*)a.kv + (int64_t)a.seq_ctx0[seq] * ldkv + a.heads * dp + h * vp;
  const bf16_t* qrow = (const bf16_t*)a.proj + (int64_t)(row0 + t) * a.ldp + a.col_q + h * dp;
  u32x4 qf[2 * D];
#pragma unroll
  for (int s = 0; s < 2 * D; ++s) qf[s] = *(const u32x4*)(qrow + 16 * s + 8 * hi);
  f32x16 o[C];
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[c][e] = 0.f;
  float m = -INFINITY, l = 0.f;
  const float sc = a.scale * LOG2E;

  u32x4 kr[D], vr[C];
  auto load = [&](int j0) {
#pragma unroll
    for (int i = 0; i < D; ++i) {
      const int piece = tid + 256 * i, j = piece / (dp / 8), d = (piece - j * (dp / 8)) * 8;
      kr[i] = *(const u32x4*)(Kg + (int64_t)min(j0 + j, kv_end - 1) * ldkv + d);  // rows past the end replay the last one; masked
    }
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int piece = tid + 256 * i, j = piece / (vp / 8), d = (piece - j * (vp / 8)) * 8;
      vr[i] = *(const u32x4*)(Vg + (int64_t)min(j0 + j, kv_end - 1) * ldkv + d);
    }
  };
  auto store = [&](bf16_t* K) {
    bf16_t* V = K + 64 * KS;
#pragma unroll
    for (int i = 0; i < D; ++i) {
      const int piece = tid + 256 * i, j = piece / (dp / 8), d = (piece - j * (dp / 8)) * 8;
      *(u32x4*)(K + j * KS + d) = kr[i];
    }
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int piece = tid + 256 * i, j = piece / (vp / 8), d = (piece - j * (vp / 8)) * 8;
      *(u32x4*)(V + j * VS + d) = vr[i];
    }
  };
  constexpr int STEP = 64 * KG;
  const int first = 64 * kg;  // (tiles past the end replay its last row, and are not used)
  bf16_t* tiles = psm + 2 * kg * M::buffer;
  load(first);
  store(tiles);
  if (first + STEP < kv_end) load(first + STEP);
  const int i16 = lane & 15, v_lane = (4 * hi + (i16 >> 2)) * VS + 16 * ((lane >> 4) & 1) + 4 * (i16 & 3);
  int buf = 0;
  for (int j0 = first; j0 - first < kv_end; j0 += STEP, buf ^= 1) {
    __syncthreads();  // this tile is in LDS, and nobody reads the other buffer any more
    const bf16_t *K = tiles + buf * M::buffer, *V = K + 64 * KS;
    if (j0 + STEP < kv_end) {
      store(tiles + (buf ^ 1) * M::buffer);
      if (j0 + 2 * STEP < kv_end) load(j0 + 2 * STEP);
    }
    if (j0 > w_hi || w0 >= len) continue;  // (wave-uniform) no key of this tile is visible to the wave
    f32x16 s[2];
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
#pragma unroll
      for (int e = 0; e < 16; ++e) s[sub][e] = 0.f;
#pragma unroll
      for (int k = 0; k < 2 * D; ++k)
        s[sub] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(*(const u32x4*)(K + (32 * sub + l31) * KS + 16 * k + 8 * hi)), op(qf[k]), s[sub], 0, 0, 0);
    }
    if (j0 + 63 > w_lo) {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (j0 + 32 * sub + 8 * (e >> 2) + 4 * hi + (e & 3) > qpos) s[sub][e] = -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[sub][e]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * sc;  // (a negative scale turns the order round: the bound below still holds for sc > 0 only)
    if (__any(mx - m > 6.0f)) {  // rescale only when a weight could exceed 2^6; the first tile always holds key 0, visible to all
      const float mn = fmaxf(m, mx), f = KG > 1 && mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= f;
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[c][e] *= f;
    }
    const float ref = KG > 1 && m == -INFINITY ? 0.f : m;  // (a second group's query may have seen no key yet)
    u32x4 p[2][2];
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float p0 = __builtin_amdgcn_exp2f(fmaf(s[sub][8 * u + 2 * e], sc, -ref)), p1 = __builtin_amdgcn_exp2f(fmaf(s[sub][8 * u + 2 * e + 1], sc, -ref));
          l += p0 + p1;
          p[sub][u][e] = pack_bf16x2(p0, p1);
        }
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const bf16_t* vp_ = V + v_lane + (32 * sub + 16 * u) * VS + 32 * c;
          const u32x2 v0 = read_tr(vp_), v1 = read_tr(vp_ + 8 * VS);
          o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op(u32x4{v0[0], v0[1], v1[0], v1[1]}), op(p[sub][u]), o[c], 0, 0, 0);
        }
  }
  __syncthreads();
  if constexpr (KG > 1) {
    float* sums = (float*)(psm + M::outputs) + tid;
    constexpr int N = 16 * C;
    if (kg) {
#pragma unroll
      for (int i = 0; i < N; ++i) sums[256 * i] = o[i >> 4][i & 15];
      sums[256 * N] = m;
      sums[256 * (N + 1)] = l;
    }
    __syncthreads();
    if (kg) return;
    const float m1 = sums[256 * N], mn = fmaxf(m, m1), f0 = __builtin_amdgcn_exp2f(m - mn), f1 = __builtin_amdgcn_exp2f(m1 - mn);  // (m: key 0's group)
    l = l * f0 + sums[256 * (N + 1)] * f1;
#pragma unroll
    for (int i = 0; i < N; ++i) o[i >> 4][i & 15] = o[i >> 4][i & 15] * f0 + sums[256 * i] * f1;
  }
  if (w0 >= len) return;
  const float inv = 1.0f / (l + __shfl_xor(l, 32, 64));
  const bf16_t* grow = (const bf16_t*)a.proj + (int64_t)(row0 + t) * a.ldp + a.col_g + h * vp;
  bf16_t* ot = psm + wave * 32 * M::OS;
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int e0 = 32 * c + 8 * g + 4 * hi;
      f32x4 v = f32x4{o[c][4 * g], o[c][4 * g + 1], o[c][4 * g + 2], o[c][4 * g + 3]} * inv;
      if (a.col_g >= 0) {
        const f32x4 gv = ld4(grow + e0);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= sigmoid_f32(gv[e]);
      }
      st4(ot + l31 * M::OS + e0, v);
    }
  bf16_t* out = (bf16_t*)a.out + (int64_t)row0 * a.ldo;
  for (int i = lane; i < 32 * (vp / 8); i += 64) {  // (the wave's own tile: its LDS operations are in order)
    const int rr = i / (vp / 8), e = (i - rr * (vp / 8)) * 8;
    if (w0 + rr < len) *(u32x4*)(out + (int64_t)(w0 + rr) * a.ldo + in_chunks(h * vp + e, a.out_chunk)) = *(const u32x4*)(ot + rr * M::OS + e);
  }
}

typedef void (*PrefillKernel)(const LmLatent, int);
struct PrefillPick {
  PrefillKernel fn[2];  // one and two groups
  int lds[2];
};
template <int D, int C>
PrefillPick prefill_of() {
  return {{latent_prefill_kernel<D, C, 1>, latent_prefill_kernel<D, C, 2>}, {PrefillLds<D, C, 1>::bytes, PrefillLds<D, C, 2>::bytes}};
}
template <int D>
PrefillPick prefill_by_width(int c) {
  switch (c) {
    case 1: return prefill_of<D, 1>();
    case 2: return prefill_of<D, 2>();
    case 3: return prefill_of<D, 3>();
    case 4: return prefill_of<D, 4>();
    default: return {};
  }
}
PrefillPick prefill_pick(const LmLatent& a) {
  if (!(a.scale > 0.f)) return {};
  switch (a.dp / 32) {
    case 1: return prefill_by_width<1>(a.vp / 32);
    case 2: return prefill_by_width<2>(a.vp / 32);
    case 3: return prefill_by_width<3>(a.vp / 32);
    case 4: return prefill_by_width<4>(a.vp / 32);
    default: return {};
  }
}

// ---------------------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ f32x4 mfma16(const u32x4& a, const u32x4& b, const f32x4& c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(op(a), op(b), c, 0, 0, 0); }

// grid (heads, rp / 64 + 1): the last block column norms and stores the new latent rows
template <int D>
__global__ __launch_bounds__(256) void latent_absorb_kernel(const LmLatent a) {
  constexpr int dp = 32 * D;
  const int h = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, q = lane >> 4;
  if ((int)blockIdx.y * 64 == a.rp) {
    for (int seq = h * 4 + wave; seq < a.r.n_seq; seq += a.heads * 4) latent_row<bf16_t>(a, a.r.seq_row0[seq], seq, nullptr);
    return;
  }
  const int r0 = blockIdx.y * 64 + 16 * wave;
  u32x4 w[D];
#pragma unroll
  for (int s = 0; s < D; ++s) w[s] = *(const u32x4*)((const bf16_t*)a.up_k_t + ((int64_t)h * a.rp + r0 + c16) * dp + 32 * s + 8 * q);
  for (int s0 = 0; s0 < a.r.n_seq; s0 += 16) {
    const int seq = min(s0 + c16, a.r.n_seq - 1);
    const bf16_t* qr = (const bf16_t*)a.proj + (int64_t)a.r.seq_row0[seq] * a.ldp + a.col_q + h * dp;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < D; ++s) v = mfma16(w[s], *(const u32x4*)(qr + 32 * s + 8 * q), v);
    if (s0 + c16 < a.r.n_seq) st4((bf16_t*)a.q_lat + ((int64_t)seq * a.heads + h) * a.rp + r0 + 4 * q, v);
  }
}

// grid (splits, sequences, groups of 16 WH heads).  A workgroup's waves: WK groups of 32 keys x WH tiles of 16 heads x WR parts of the
// latent's columns.  The 32 rows of a key group lie in one LDS tile that its WH * WR waves load and share; S^T = c q^T (16x16x32) leaves 8 of
// the 32 keys of a head per lane, which are the operand of z^T += c^T P^T (with WR > 1 the waves of a part repeat the scores and share the
// sums).  At the end the key groups' sums meet in LDS.  RT: rp / 64
template <int RT, int WK, int WH, int WR>
struct DecodeShape {
  static constexpr int R = 64 * RT, waves = WK * WH * WR, CS = R + 8, ZS = R + 4;
  static constexpr int tiles = WK * 32 * CS * 2, sums = 16 * WH * ZS * 4, lds = tiles > sums ? tiles : sums;
};
template <int RT, int WK, int WH, int WR>
__global__ __launch_bounds__(64 * WK * WH * WR, 2) void latent_decode_kernel(const LmLatent a) {
  using M = DecodeShape<RT, WK, WH, WR>;
  constexpr int R = M::R, CS = M::CS, ZS = M::ZS, SHARE = WH * WR, PIECES = R / 16 / SHARE, ZT = 4 * RT / WR, NT = 64 * M::waves;
  static_assert(R / 16 % SHARE == 0 && 4 * RT % WR == 0, "whole pieces and tiles per wave");
  extern __shared__ __attribute__((aligned(16))) char dsm[];
  __shared__ float mw[WK][16 * WH], lw[WK][16 * WH];
  const int split = blockIdx.x, seq = blockIdx.y, g0 = blockIdx.z * 16 * WH, tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wk = wave / SHARE, part = wave % SHARE, wh = part % WH, wr = part / WH;
  // a sequence's keys in equal splits, whatever its length: every workgroup has work
  constexpr int step = 32 * WK;
  const int pos = a.r.row_pos[a.r.seq_row0[seq]], per = ((pos + a.n_split) / a.n_split + step - 1) / step * step;
  const int k0 = split * per, k1 = min(k0 + per, pos + 1);
  const int64_t heads_splits = (int64_t)a.heads * a.n_split;
  float* pm = a.part + (int64_t)a.r.n_seq * heads_splits * R;  // (m, l) pairs behind the sums
  if (k0 >= k1) {
    for (int h = tid; h < 16 * WH; h += NT)
      if (g0 + h < a.heads) {
        float* p = pm + ((int64_t)seq * heads_splits + (int64_t)(g0 + h) * a.n_split + split) * 2;
        p[0] = -INFINITY;
        p[1] = 0.f;
      }
    return;
  }
  const bf16_t* c = (const bf16_t*)a.cache + (int64_t)a.r.seq_slot[seq] * a.ctx * R;
  bf16_t* tile = (bf16_t*)dsm + wk * 32 * CS;
  u32x4 cr[PIECES];
  auto load = [&](int j0) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int piece = lane + 64 * (i * SHARE + part), j = piece / (R / 8), d = (piece - j * (R / 8)) * 8;
      cr[i] = *(const u32x4*)(c + (int64_t)min(j0 + j, pos) * R + d);  // rows past the end replay the last one; masked
    }
  };
  load(k0 + 32 * wk);
  u32x4 qf[2 * RT];
#pragma unroll
  for (int s = 0; s < 2 * RT; ++s)
    qf[s] = *(const u32x4*)((const bf16_t*)a.q_lat + ((int64_t)seq * a.heads + min(g0 + 16 * wh + c16, a.heads - 1)) * R + 32 * s + 8 * q);
  f32x4 z[ZT];
#pragma unroll
  for (int i = 0; i < ZT; ++i) z[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const float sc = a.scale * LOG2E;
  for (int b0 = k0; b0 < k1; b0 += step) {  // (uniform: every wave takes part in the barriers)
    const int j0 = b0 + 32 * wk;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int piece = lane + 64 * (i * SHARE + part), j = piece / (R / 8), d = (piece - j * (R / 8)) * 8;
      *(u32x4*)(tile + j * CS + d) = cr[i];
    }
    __syncthreads();
    if (b0 + step < k1) load(j0 + step);
    if (j0 >= k1) continue;
    f32x4 s[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      s[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 2 * RT; ++k) s[b] = mfma16(*(const u32x4*)(tile + (16 * b + c16) * CS + 32 * k + 8 * q), qf[k], s[b]);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[b][e] = j0 + 16 * b + 4 * q + e < k1 ? s[b][e] * sc : -INFINITY;
        mx = fmaxf(mx, s[b][e]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx), f = __builtin_amdgcn_exp2f(m - mn);
    m = mn;
    float p[8], sum = 0.f;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p[4 * b + e] = __builtin_amdgcn_exp2f(s[b][e] - mn);
        sum += p[4 * b + e];
      }
    l = l * f + sum;
    const u32x4 pb = {pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3]), pack_bf16x2(p[4], p[5]), pack_bf16x2(p[6], p[7])};
#pragma unroll
    for (int i = 0; i < ZT; ++i) {
      const bf16_t* cp = tile + (4 * q + (c16 >> 2)) * CS + 16 * (wr * ZT + i) + 4 * (c16 & 3);
      const u32x2 v0 = read_tr(cp), v1 = read_tr(cp + 16 * CS);
      z[i] = mfma16(u32x4{v0[0], v0[1], v1[0], v1[1]}, pb, z[i] * f);
    }
  }
  // the key groups' sums: maximum of all, then group by group into LDS
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  const int h = 16 * wh + c16;
  if (q == 0 && wr == 0) {
    mw[wk][h] = m;
    lw[wk][h] = l;
  }
  float* zs = (float*)dsm;
#pragma unroll
  for (int w = 0; w < WK; ++w) {
    __syncthreads();  // (the first: every wave has left its tile, and mw is complete)
    if (w != wk) continue;
    float mb = mw[0][h];
#pragma unroll
    for (int k = 1; k < WK; ++k) mb = fmaxf(mb, mw[k][h]);
    const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mb);
#pragma unroll
    for (int i = 0; i < ZT; ++i) {
      f32x4* p = (f32x4*)(zs + h * ZS + 16 * (wr * ZT + i) + 4 * q);
      *p = w == 0 ? z[i] * f : *p + z[i] * f;
    }
  }
  __syncthreads();
  const int nh = min(16 * WH, a.heads - g0);
  for (int i = tid * 4; i < nh * R; i += 4 * NT) {
    const int hh = i / R, r = i - hh * R;
    *(f32x4*)(a.part + ((int64_t)seq * heads_splits + (int64_t)(g0 + hh) * a.n_split + split) * R + r) = *(const f32x4*)(zs + hh * ZS + r);
  }
  if (tid < nh) {
    float mb = mw[0][tid], lb = 0.f;
#pragma unroll
    for (int k = 1; k < WK; ++k) mb = fmaxf(mb, mw[k][tid]);
#pragma unroll
    for (int k = 0; k < WK; ++k) lb += mw[k][tid] == -INFINITY ? 0.f : lw[k][tid] * __builtin_amdgcn_exp2f(mw[k][tid] - mb);
    float* p = pm + ((int64_t)seq * heads_splits + (int64_t)(g0 + tid) * a.n_split + split) * 2;
    p[0] = mb;
    p[1] = lb;
  }
}

// grid (heads, sequences / SEQ, parts of the columns): sum over the splits, then eight threads per output column share the latent's columns, 32 columns
// after the other.  SEQ 1: the waves share the splits of one sequence; 4: a wave per sequence, and every weight that is read serves four.  What bounds it is
// the chain of loads (weights of a head are 64 to 128 KB, sums as much): the weights are under way before the sums are looked up, and a head's columns go to
// several workgroups, which add up the splits each for itself.  20 sequences, 16 heads of 128, rank 512: 17.6 us with all columns of a head in a workgroup and
// its weights behind the sums, 10.0 with 32 columns per workgroup; 23 of 32 x 64: 10.0 and 8.2, one 9.7 and 7.1; 40 of 32 x 64, rank 256: 7.7 and 7.0.
constexpr int MAX_SPLITS = 64, OUT_COLS = 32, MAX_RANK = 512;
template <int SEQ>
__global__ __launch_bounds__(256) void latent_out_kernel(const LmLatent a) {
  static_assert(SEQ == 1 || SEQ == 4, "");
  extern __shared__ __attribute__((aligned(16))) float zsm[];  // [4][rp]
  __shared__ float fs[4][MAX_SPLITS];
  const int h = blockIdx.x, s0 = blockIdx.y * SEQ, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, R = a.rp, n = a.n_split;
  const int s = tid & 7;
  u32x4 wv[MAX_RANK / 64];
  auto load = [&](int e) {
    const bf16_t* w = (const bf16_t*)a.up_kv.w + ((int64_t)a.heads * a.dp + h * a.vp + e) * R + 8 * s;
#pragma unroll
    for (int i = 0; i < MAX_RANK / 64; ++i) wv[i] = *(const u32x4*)(w + (64 * i < R ? 64 * i : 0));
  };
  load(blockIdx.z * OUT_COLS + (tid >> 3));
  const int mine = SEQ == 1 ? s0 : min(s0 + wave, a.r.n_seq - 1);
  const int64_t base = ((int64_t)mine * a.heads + h) * n;
  const float* pm = a.part + (int64_t)a.r.n_seq * a.heads * n * R + base * 2;
  const float mk = lane < n ? pm[2 * lane] : -INFINITY, lk = lane < n ? pm[2 * lane + 1] : 0.f;
  const float m = wave_max(mk), f0 = lk == 0.f ? 0.f : __builtin_amdgcn_exp2f(mk - m), sum = wave_sum(f0 * lk);
  const int live = 64 - __clzll((long long)__ballot(lk != 0.f));  // (an empty split wrote no sums; those behind the sequence's end are)
  fs[wave][lane] = f0 / sum;
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the wave's own row)
  for (int r = 4 * lane; r < R; r += 256) {
    f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int k = SEQ == 1 ? wave : 0; k < live; k += SEQ == 1 ? 4 : 1) {
      const f32x4 v = *(const f32x4*)(a.part + (base + k) * R + r);
      const float f = fs[wave][k];
      z += f != 0.f ? f * v : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    *(f32x4*)(zsm + wave * R + r) = z;
  }
  __syncthreads();
  for (int e0 = blockIdx.z * OUT_COLS; e0 < a.vp; e0 += gridDim.z * OUT_COLS) {
    const int e = e0 + (tid >> 3);
    float o[SEQ];
#pragma unroll
    for (int i = 0; i < SEQ; ++i) o[i] = 0.f;
#pragma unroll
    for (int i = 0; i < MAX_RANK / 64; ++i) {
      if (64 * i >= R) break;
      const f32x4 w0 = half8(wv[i], 0), w1 = half8(wv[i], 1);
      const float* z = zsm + 64 * i + 8 * s;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const f32x4 t = w0 * *(const f32x4*)(z + k * R) + w1 * *(const f32x4*)(z + k * R + 4);
        o[SEQ == 1 ? 0 : k] += (t[0] + t[1]) + (t[2] + t[3]);
      }
    }
    if (e0 + (int)gridDim.z * OUT_COLS < a.vp) load(e + gridDim.z * OUT_COLS);
#pragma unroll
    for (int i = 0; i < SEQ; ++i)
#pragma unroll
      for (int d = 1; d < 8; d <<= 1) o[i] += __shfl_xor(o[i], d, 64);
    float v = o[0];
#pragma unroll
    for (int i = 1; i < SEQ; ++i) v = s == i ? o[i] : v;  // thread s writes sequence s
    if (s >= SEQ || s0 + s >= a.r.n_seq) continue;
    const int64_t row = a.r.seq_row0[s0 + s];
    if (a.col_g >= 0) v *= sigmoid_f32(bf2f(((const bf16_t*)a.proj)[row * a.ldp + a.col_g + h * a.vp + e]));
    ((bf16_t*)a.out)[row * a.ldo + in_chunks(h * a.vp + e, a.out_chunk)] = f2bf(v);
  }
}

// Parts of a head's columns: as many as give four workgroups per CU.  Beyond that adding up the splits again costs more than it hides.  A step of four layers of
// this attention and little else, rank 512: 128 sequences, 128 heads of 128 (4096 workgroups) 659 us in one part, 698 in two, 778 in four; 16 of 128 (512) 294,
// 281, 293; 64 sequences (256) 252, 235, 229.
inline int out_parts(int workgroups, int tiles) {
  const int most = std::max(1, std::min(tiles, 1024 / workgroups));
  return (tiles + (tiles + most - 1) / most - 1) / ((tiles + most - 1) / most);
}

typedef void (*LatentKernel)(const LmLatent);
struct DecodePick {
  LatentKernel absorb, attend;
  int lds, threads, head_tiles;
};
template <int RT, int WK, int WH, int WR>
DecodePick decode_of() {
  using M = DecodeShape<RT, WK, WH, WR>;
  return {nullptr, latent_decode_kernel<RT, WK, WH, WR>, M::lds, 64 * M::waves, WH};
}
template <int RT>
DecodePick decode_by_heads(int heads) {
  if constexpr (RT <= 4) return heads > 16 ? decode_of<RT, 2, 2, 1>() : decode_of<RT, 4, 1, 1>();
  else return heads > 16 ? decode_of<RT, 2, 2, 2>() : decode_of<RT, 2, 1, 2>();
}
DecodePick decode_pick(int heads, int dp, int rp) {
  DecodePick k = {nullptr, nullptr, 0, 0, 1};
  switch (rp / 64) {
    case 1: k = decode_by_heads<1>(heads); break;
    case 2: k = decode_by_heads<2>(heads); break;
    case 3: k = decode_by_heads<3>(heads); break;
    case 4: k = decode_by_heads<4>(heads); break;
    case 5: k = decode_by_heads<5>(heads); break;
    case 6: k = decode_by_heads<6>(heads); break;
    case 7: k = decode_by_heads<7>(heads); break;
    case 8: k = decode_by_heads<8>(heads); break;
    default: return k;
  }
  switch (dp / 32) {
    case 1: k.absorb = latent_absorb_kernel<1>; break;
    case 2: k.absorb = latent_absorb_kernel<2>; break;
    case 3: k.absorb = latent_absorb_kernel<3>; break;
    case 4: k.absorb = latent_absorb_kernel<4>; break;
    default: break;
  }
  return k;
}

}  // namespace

md_status lm_latent_rows(int dtype, const LmLatent& a, bool pack, hipStream_t s) {
  const dim3 grid((a.r.n_rows + 3) / 4);
  if (dtype == MD_DTYPE_F32) hipLaunchKernelGGL(latent_rows_kernel<float>, grid, dim3(256), 0, s, a, pack ? 1 : 0);
  else hipLaunchKernelGGL(latent_rows_kernel<bf16_t>, grid, dim3(256), 0, s, a, pack ? 1 : 0);
  MD_TRY(md_launch_status());
  if (!pack || a.ctx_rows == a.r.n_rows) return MD_OK;
  const int blocks = (a.r.max_ctx * (a.rp / 4) + 1023) / 1024;
  const dim3 ggrid(blocks < 256 ? blocks : 256, a.r.n_seq);
  if (dtype == MD_DTYPE_F32) hipLaunchKernelGGL(latent_gather_kernel<float>, ggrid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(latent_gather_kernel<bf16_t>, ggrid, dim3(256), 0, s, a);
  return md_launch_status();
}

md_status lm_latent_plain(int dtype, const LmLatent& a, hipStream_t s) {
  const int lds = (a.dp + 2 * a.rp) * 4;
  if (lds > 60 * 1024) return MD_ERR_UNSUPPORTED;
  MD_TRY(lm_latent_rows(dtype, a, false, s));
  const dim3 grid(a.heads, a.r.n_rows);
  if (dtype == MD_DTYPE_F32) hipLaunchKernelGGL(latent_plain_kernel<float>, grid, dim3(256), lds, s, a);
  else hipLaunchKernelGGL(latent_plain_kernel<bf16_t>, grid, dim3(256), lds, s, a);
  return md_launch_status();
}

bool lm_latent_mfma_takes(const LmLatent& a) { return prefill_pick(a).fn[0] != nullptr; }
md_status lm_latent_mfma(const LmLatent& a, hipStream_t s) {
  const PrefillPick k = prefill_pick(a);
  if (!k.fn[0]) return MD_ERR_UNSUPPORTED;
  const int n_qblk = (a.r.max_len + 127) / 128, n_bh = a.r.n_seq * a.heads;
  const int two = a.r.max_ctx > 192 && n_bh * n_qblk <= 256;  // a workgroup per CU, and tiles for both groups
  MD_TRY(md_ensure_dynamic_lds((const void*)k.fn[two], k.lds[two]));
  hipLaunchKernelGGL(k.fn[two], dim3((n_bh + 7) / 8 * 8 * n_qblk), dim3(two ? 512 : 256), k.lds[two], s, a, n_qblk);
  return md_launch_status();
}

int lm_latent_decode_splits(int n_seq, int heads, int max_keys) {
  const int groups = (heads + 31) / 32, blocks = (max_keys + 63) / 64;
  int splits = 256 / (n_seq * groups);  // a workgroup per CU: more of them re-load queries and write sums, and gain nothing
  splits = splits > MAX_SPLITS ? MAX_SPLITS : splits;
  splits = splits > blocks ? blocks : splits;
  return splits < 1 ? 1 : splits;
}
size_t lm_latent_decode_part_floats(int n_seq, int n_split, int heads, int rp) { return (size_t)n_seq * n_split * heads * (rp + 2); }
bool lm_latent_decode_takes(const LmLatent& a) {
  const DecodePick k = decode_pick(a.heads, a.dp, a.rp);
  return k.attend && k.absorb && a.scale > 0.f;
}
md_status lm_latent_decode(const LmLatent& a, hipStream_t s) {
  const DecodePick k = decode_pick(a.heads, a.dp, a.rp);
  MD_TRY(md_ensure_dynamic_lds((const void*)k.attend, k.lds));
  hipLaunchKernelGGL(k.absorb, dim3(a.heads, a.rp / 64 + 1), dim3(256), 0, s, a);
  MD_TRY(md_launch_status());
  hipLaunchKernelGGL(k.attend, dim3(a.n_split, a.r.n_seq, (a.heads + 16 * k.head_tiles - 1) / (16 * k.head_tiles)), dim3(k.threads), k.lds, s, a);
  MD_TRY(md_launch_status());
  const int seqs = a.r.n_seq >= 16 ? (a.r.n_seq + 3) / 4 : a.r.n_seq, z = out_parts(a.heads * seqs, a.vp / OUT_COLS);
  if (a.r.n_seq >= 16) hipLaunchKernelGGL(latent_out_kernel<4>, dim3(a.heads, seqs, z), dim3(256), 4 * a.rp * 4, s, a);
  else hipLaunchKernelGGL(latent_out_kernel<1>, dim3(a.heads, seqs, z), dim3(256), 4 * a.rp * 4, s, a);
  return md_launch_status();
}
