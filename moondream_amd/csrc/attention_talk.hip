// Attention whose heads' scores are mixed before the softmax, over the keys of the query's own chunk:
//   score_h(i, j) = sum_g mix[h][g] (q_g(i) . k_g'(j) * scale - slope[g] (i - j)),   j <= i, j / chunk == i / chunk
// with keys and queries that went through a short causal convolution over time and an RMS norm over the whole projection.
//
//   attn_prep_kernel     one workgroup per (row, q | k | v): convolution from the step's rows and the slot's last projections, norm,
//                        query row / cache row written
//   attn_prep_step_kernel   the same for a decode step (one row per sequence), up to 8192 columns, in registers
//   attn_prep_block_kernel  the same for 8 positions per workgroup (prefill, up to 4096 columns)
//   conv_state_kernel    the last projections of every sequence of the step -> its slot (row p % taps of the slot's ring)
//   attn_plain_kernel    one workgroup per query row or two, fp32 on the vector ALUs: any dtype, any head size
//   attn_mfma_kernel     bf16 prefill on the matrix cores: 16 queries x all heads per workgroup
//   attn_heads_*         bf16 decode step with one key head per query head: see there
//   attn_decode_kernel   any other bf16 decode step: split-key attention behind attn_prep_kernel (made in every split, the convolution and norms
//                        would be its longest chain of dependent loads)
//   attn_combine_kernel  ... and the sum over the splits
//
// attn_mfma_kernel.  The heads' mixture couples all heads of a (query, key) pair before the softmax, so a workgroup owns 16 queries
// with ALL heads.  Per key tile of 16 * NW keys:
//   1. wave w computes S_g^T = K_g Q_g^T of its 16 keys for every head (v_mfma 16x16x32): a lane holds 4 keys of one query for every
//      head.  K comes straight from the cache (each element is used by one wave only), Q from LDS.
//   2. the mixture is a matrix product over heads, [H x H] . [H x pairs], on the matrix cores too.  Its B operand wants 4 (8) heads of
//      one pair per 16-lane row where step 1 left 4 keys of one head: a 4 x 4 transpose between lane rows and registers, done with
//      v_permlane32_swap / v_permlane16_swap, no LDS.  The fp32 scores are split into two bf16 (16 mantissa bits), the mixing matrix
//      is exact in bf16.  The distance bias is linear, so its mixture is one slope per head, applied after the product in fp32.
//   3. a lane then holds all 16 keys of the wave for its (query, head): the maximum and the sum over keys need no lane exchange, the
//      maximum over the waves goes through LDS.
//   4. P goes to LDS as the A operand of P V; wave w owns the outputs of H / NW heads.
// The cache holds keys and values in operand order, so every load of either is 1 KiB of consecutive memory per wave.
#include "lm_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace {

// ---------------------------------------------------------------------------------------------------------------------------
// the convolution of one row's q (part 0), k (1) or v (2) columns -> conv_out (LDS, fp32); returns the thread's share of the sum of
// squares.  store_state: the row's own projection also goes to the ring (a decode step)
template <typename T>
__device__ __forceinline__ float conv_row(const LmAttn& a, int row, int seq, int pos, int part, float* conv_out, bool store_state) {
  const int row0 = a.r.seq_row0[seq], pos0 = a.r.seq_pos0[seq], slot = a.r.seq_slot[seq];
  const int col0 = part == 0 ? a.col_q : part == 1 ? a.col_k : a.col_v;
  const int ncol = part == 0 ? a.heads * a.dp : a.kv_heads * (part == 1 ? a.dp : a.vp);
  const T* proj = (const T*)a.proj + col0;
  T* ring = (T*)a.conv_state + (int64_t)slot * a.taps * a.conv_ld + col0;
  const float* cw = a.conv + col0;
  float ss = 0.f;
  auto input = [&](int p, int c) { return p >= pos0 ? ld4(proj + (int64_t)(row0 + p - pos0) * a.ldp + c) : ld4(ring + (int64_t)(p % a.taps) * a.conv_ld + c); };
#pragma unroll 2
  for (int c = threadIdx.x * 4; c < ncol; c += 1024) {
    constexpr int AT_ONCE = 4;  // the newest taps: all their loads are requested before the first is used
    f32x4 u[AT_ONCE], w[AT_ONCE], y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < AT_ONCE; ++k) {
      u[k] = w[k] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (k < a.taps && pos - k >= 0) {
        u[k] = input(pos - k, c);
        w[k] = *(const f32x4*)(cw + (int64_t)(a.taps - 1 - k) * a.conv_ld + c);
      }
    }
    for (int k = AT_ONCE; k < a.taps && pos - k >= 0; ++k) y += *(const f32x4*)(cw + (int64_t)(a.taps - 1 - k) * a.conv_ld + c) * input(pos - k, c);
#pragma unroll
    for (int k = AT_ONCE - 1; k >= 0; --k) y += w[k] * u[k];
    if (store_state && a.taps > 1) st4(ring + (int64_t)(pos % a.taps) * a.conv_ld + c, u[0]);
    *(f32x4*)(conv_out + c) = y;
    ss += y[0] * y[0] + y[1] * y[1] + y[2] * y[2] + y[3] * y[3];
  }
  return ss;
}

// RMS norm over all of conv_out (whole q or k projection): element c goes to put(c, four normed values)
template <typename F>
__device__ __forceinline__ void norm_row(const LmAttn& a, int nh, float ss, const float* w, const float* conv_out, float* red, F put) {
  ss = block_sum_256(ss, red);
  const float r = 1.0f / sqrtf(ss / (float)(nh * a.dim) + a.eps);
  for (int c = threadIdx.x * 4; c < nh * a.dp; c += 1024) put(c, *(const f32x4*)(conv_out + c) * r * *(const f32x4*)(w + c));
}

// the row's values in conv_out (complete and visible), normed per head -> cache; NW waves
template <typename T, int NW = 4>
__device__ __forceinline__ void store_values(const LmAttn& a, int slot, int pos, const float* conv_out) {
  const int lane = threadIdx.x & 63, nh = a.kv_heads, hp = a.vp;
  for (int g = threadIdx.x >> 6; g < nh; g += NW) {
    float r = 1.0f;
    if (a.value_norm) {
      float s = 0.f;
      for (int d = lane; d < hp; d += 64) s += conv_out[g * hp + d] * conv_out[g * hp + d];
      r = 1.0f / sqrtf(wave_sum(s) / (float)a.vdim + a.eps);
    }
    T* dst = (T*)a.v + (int64_t)slot * a.ctx * nh * hp;
    for (int d = lane; d < hp; d += 64) stf(dst + value_index(pos, g, d, nh, hp), conv_out[g * hp + d] * r);
  }
}

template <typename T>
__device__ __forceinline__ void store_key4(const LmAttn& a, int slot, int pos, int c, const f32x4& v) {
  const int g = c / a.dp, d = c - g * a.dp;
  st4((T*)a.k + (int64_t)slot * a.ctx * a.kv_heads * a.dp + key_index(pos, g, d, a.kv_heads, a.dp), v);
}

template <typename T, bool STEP>  // STEP: a decode step (one row per sequence), which also writes the convolution state
__global__ __launch_bounds__(256) void attn_prep_kernel(const LmAttn a) {
  extern __shared__ __attribute__((aligned(16))) float conv_out[];
  __shared__ float red[4];
  const int row = blockIdx.x, part = blockIdx.y;  // 0 q, 1 k, 2 v
  const int seq = a.r.row_seq[row], pos = a.r.row_pos[row], slot = a.r.seq_slot[seq];
  const float ss = conv_row<T>(a, row, seq, pos, part, conv_out, STEP);
  if (part == 0) {
    norm_row(a, a.heads, ss, a.q_norm, conv_out, red, [&](int c, const f32x4& v) { st4((T*)a.q + (int64_t)row * a.heads * a.dp + c, v); });
  } else if (part == 1) {
    norm_row(a, a.kv_heads, ss, a.k_norm, conv_out, red, [&](int c, const f32x4& v) { store_key4<T>(a, slot, pos, c, v); });
  } else {
    __syncthreads();
    store_values<T>(a, slot, pos, conv_out);
  }
}

// A decode step: grid (sequences, q | k | v), 4 NI columns per thread.  What bounds it is the chain of dependent loads, so the row is its
// sequence, everything the row needs is requested at once, and the convolved columns stay in registers (2048 columns, one row: 5.5 us
// against 8.9; 16 rows: 7.5 against 11.4).
template <int NI>
__global__ __launch_bounds__(512) void attn_prep_step_kernel(const LmAttn a) {
  extern __shared__ __attribute__((aligned(16))) float conv_out[];
  __shared__ float red[8];
  const int row = blockIdx.x, part = blockIdx.y, tid = threadIdx.x;  // 0 q, 1 k, 2 v
  const int pos = a.r.row_pos[row], slot = a.r.seq_slot[row];
  const int col0 = part == 0 ? a.col_q : part == 1 ? a.col_k : a.col_v;
  const int ncol = part == 0 ? a.heads * a.dp : a.kv_heads * (part == 1 ? a.dp : a.vp);
  const bf16_t* proj = (const bf16_t*)a.proj + (int64_t)row * a.ldp + col0;
  bf16_t* ring = (bf16_t*)a.conv_state + (int64_t)slot * a.taps * a.conv_ld + col0;
  const float *cw = a.conv + col0, *norm = part == 0 ? a.q_norm : a.k_norm;
  f32x4 y[NI], nw[NI];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int c = (tid + 512 * i) * 4;
    y[i] = nw[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (c >= ncol) continue;
    constexpr int AT_ONCE = 4;  // the newest taps
    // (a branch for each would wait for each: rows before the sequence's first are read from somewhere else and not used)
    u32x2 raw[AT_ONCE];
    f32x4 u[AT_ONCE], w[AT_ONCE];
#pragma unroll
    for (int k = 0; k < AT_ONCE; ++k) {
      const bool in = k < a.taps && pos - k >= 0;
      raw[k] = *(const u32x2*)(k > 0 && in ? ring + (int64_t)((pos - k) % a.taps) * a.conv_ld + c : proj + c);
      w[k] = *(const f32x4*)(cw + (int64_t)(in ? a.taps - 1 - k : 0) * a.conv_ld + c);
    }
    nw[i] = *(const f32x4*)(part < 2 ? norm + c : cw + c);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < AT_ONCE; ++k)
      u[k] = k < a.taps && pos - k >= 0 ? f32x4{lo_bf(raw[k][0]), hi_bf(raw[k][0]), lo_bf(raw[k][1]), hi_bf(raw[k][1])} : f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k = AT_ONCE; k < a.taps && pos - k >= 0; ++k)
      y[i] += *(const f32x4*)(cw + (int64_t)(a.taps - 1 - k) * a.conv_ld + c) * ld4(ring + (int64_t)((pos - k) % a.taps) * a.conv_ld + c);
#pragma unroll
    for (int k = AT_ONCE - 1; k >= 0; --k) y[i] += w[k] * u[k];
    if (a.taps > 1) st4(ring + (int64_t)(pos % a.taps) * a.conv_ld + c, u[0]);
    ss += y[i][0] * y[i][0] + y[i][1] * y[i][1] + y[i][2] * y[i][2] + y[i][3] * y[i][3];
    if (part == 2) *(f32x4*)(conv_out + c) = y[i];
  }
  if (part == 2) {
    __syncthreads();
    store_values<bf16_t, 8>(a, slot, pos, conv_out);
    return;
  }
  ss = block_sum<8>(ss, red);
  const float r = 1.0f / sqrtf(ss / (float)((part == 0 ? a.heads : a.kv_heads) * a.dim) + a.eps);
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int c = (tid + 512 * i) * 4;
    if (c >= ncol) continue;
    const f32x4 v = y[i] * r * nw[i];
    if (part == 0) st4((bf16_t*)a.q + (int64_t)row * a.heads * a.dp + c, v);
    else store_key4<bf16_t>(a, slot, pos, c, v);
  }
}

__device__ __forceinline__ void store8(bf16_t* p, const float (&v)[8]) {
  *(u32x4*)p = u32x4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
}
__device__ __forceinline__ void store8(float* p, const float (&v)[8]) {
  *(f32x4*)p = f32x4{v[0], v[1], v[2], v[3]};
  *(f32x4*)(p + 4) = f32x4{v[4], v[5], v[6], v[7]};
}

// grid (blocks of 8 positions, sequences, q | k | v); a block starts at a multiple of 8, so its values fill whole operand rows of the
// cache.  A thread owns columns 4 tid .., all 8 rows in registers (as many threads as that takes: 2048 columns, 40 / 900 / 14000 tokens 8.4 / 12.3 / 85 us, 256 threads with
// eight columns each 10.1 / 13.4 / 96; 4096 columns 10.2 / 24.5 / 225, with sixteen each 16.1 / 31.3 / 315).  The norms' sums run in one order whatever the threads.  TAPS: taps of the convolution when they are
// few (every projected row is then read once), 0: any number.
template <typename T, int TAPS, int NT>
__global__ __launch_bounds__(NT) void attn_prep_block_kernel(const LmAttn a) {
  extern __shared__ __attribute__((aligned(16))) float hs[];  // [8][NT] sums of squares of four columns; values: then [8][kv_heads];
                                                              // bf16: then the finished cache rows, in the cache's order
  __shared__ float red[8][4];
  const int seq = blockIdx.y, part = blockIdx.z, tid = threadIdx.x;
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, pos0 = a.r.seq_pos0[seq], slot = a.r.seq_slot[seq];
  const int t0 = (pos0 / 8 + blockIdx.x) * 8, lo = max(t0, pos0), hi = min(t0 + 7, pos0 + len - 1);
  if (lo > hi) return;
  const int nh = part == 0 ? a.heads : a.kv_heads, hp = part == 2 ? a.vp : a.dp, ncol = nh * hp;
  const bool all = lo == t0 && hi == t0 + 7;
  constexpr bool STAGE = sizeof(T) == 2;  // whole blocks of 8 positions leave through LDS: 16-byte pieces in the order of the cache
  bf16_t* stage = (bf16_t*)(hs + 8 * NT + 8 * a.kv_heads);
  const int col0 = part == 0 ? a.col_q : part == 1 ? a.col_k : a.col_v;
  const T* proj = (const T*)a.proj + (int64_t)(row0 - pos0) * a.ldp + col0;  // + position * ldp
  const T* ring = (const T*)a.conv_state + (int64_t)slot * a.taps * a.conv_ld + col0;
  f32x4 y[8];
  const int c = 4 * tid;
#pragma unroll
  for (int r = 0; r < 8; ++r) y[r] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (c < ncol) {
    auto input = [&](int p) { return p >= pos0 ? ld4(proj + (int64_t)p * a.ldp + c) : ld4(ring + (int64_t)(p % a.taps) * a.conv_ld + c); };
    if constexpr (TAPS > 0) {
      f32x4 w[TAPS];
#pragma unroll
      for (int j = 0; j < TAPS; ++j) w[j] = *(const f32x4*)(a.conv + col0 + (int64_t)j * a.conv_ld + c);
      f32x4 u[7 + TAPS];  // no branch around the loads: they are all requested before the first is used
#pragma unroll
      for (int k = 0; k < 7 + TAPS; ++k) {
        const int p = min(max(t0 - TAPS + 1 + k, max(lo - TAPS + 1, 0)), hi);
        u[k] = ld4(p >= pos0 ? proj + (int64_t)p * a.ldp + c : ring + (int64_t)(p % TAPS) * a.conv_ld + c);
      }
#pragma unroll
      for (int k = 0; k < 7 + TAPS; ++k) {
        if (t0 - TAPS + 1 + k < 0) u[k] = f32x4{0.f, 0.f, 0.f, 0.f};  // before the sequence
#pragma unroll
        for (int r = 0; r < 8; ++r)
          if (k - r >= 0 && k - r < TAPS) y[r] += w[k - r] * u[k];
      }
    } else
    for (int j = 0; j < a.taps; ++j) {
      const f32x4 w = *(const f32x4*)(a.conv + col0 + (int64_t)j * a.conv_ld + c);
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int p = t0 + r - a.taps + 1 + j;
        if (t0 + r < lo || t0 + r > hi || p < 0) continue;
        y[r] += w * input(p);
      }
    }
  }
  float ss[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) ss[r] = y[r][0] * y[r][0] + y[r][1] * y[r][1] + y[r][2] * y[r][2] + y[r][3] * y[r][3];
  if (NT > 256 || part == 2) {
#pragma unroll
    for (int r = 0; r < 8; ++r) hs[r * NT + tid] = ss[r];
    __syncthreads();
  }
  if (part < 2) {
    // a row's sum in norm_row's order, whatever NT: 256 lanes take every 256th column group, then a butterfly per 64 lanes, then the four.  (256 threads: what they hold.  Through LDS as
    // the others, 512 columns, 2400 / 7500 tokens 9.5 / 16.6 us take 10.9 / 18.9.)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if constexpr (NT == 256) {
#pragma unroll
      for (int r = 0; r < 8; ++r) ss[r] = wave_sum(ss[r]);
      if ((tid & 63) == 0)
#pragma unroll
        for (int r = 0; r < 8; ++r) red[r][wave] = ss[r];
    } else {
#pragma unroll
      for (int k = wave; k < 32; k += NT / 64) {
        const float* from = hs + (k >> 2) * NT + (k & 3) * 64 + (tid & 63);
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < NT / 256; ++i) s += from[256 * i];
        s = wave_sum(s);
        if ((tid & 63) == 0) red[k >> 2][k & 3] = s;
      }
    }
    __syncthreads();
    const float* w = part == 0 ? a.q_norm : a.k_norm;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      if (t0 + r < lo || t0 + r > hi) continue;
      const float f = 1.0f / sqrtf((red[r][0] + red[r][1] + red[r][2] + red[r][3]) / (float)(nh * a.dim) + a.eps);
      if (c >= ncol) continue;
      const f32x4 o = y[r] * f * *(const f32x4*)(w + c);
      if (part == 0) st4((T*)a.q + (int64_t)(row0 + t0 + r - pos0) * ncol + c, o);
      else if (STAGE && all) st4(stage + (c >> 3) * 64 + r * 8 + (c & 7), o);
      else store_key4<T>(a, slot, t0 + r, c, o);
    }
    if (STAGE && all && part == 1) {
      __syncthreads();
      bf16_t* dst = (bf16_t*)a.k + (int64_t)slot * a.ctx * nh * hp;
      for (int k = tid; k < ncol; k += NT) {  // piece k: eight coordinates of position t0 + k % 8
        const int c = (k >> 3) * 8, g = c / hp;
        *(u32x4*)(dst + key_index(t0 + (k & 7), g, c - g * hp, nh, hp)) = *(const u32x4*)(stage + k * 8);
      }
    }
    return;
  }
  float* rn = hs + 8 * NT;
  for (int k = tid; k < 8 * nh; k += NT) {
    const int r = k / nh, g = k - r * nh, m = hp / 4;
    float s = 0.f;
    for (int e = 0; e < m; ++e) s += hs[r * NT + g * m + e];
    rn[k] = a.value_norm ? 1.0f / sqrtf(s / (float)a.vdim + a.eps) : 1.0f;
  }
  __syncthreads();
  if (c < ncol) {
    const int g = c / hp, e0 = c - g * hp;
    T* dst = (T*)a.v + (int64_t)slot * a.ctx * nh * hp;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) v[r] = y[r][e] * rn[r * nh + g];
      if (STAGE && all) {
        store8(stage + (c + e) * 8, v);
      } else if (all) {
        store8(dst + value_index(t0, g, e0 + e, nh, hp), v);
      } else {
#pragma unroll
        for (int r = 0; r < 8; ++r)
          if (t0 + r >= lo && t0 + r <= hi) stf(dst + value_index(t0 + r, g, e0 + e, nh, hp), v[r]);
      }
    }
  }
  if (STAGE && all) {
    __syncthreads();
    bf16_t* dst = (bf16_t*)a.v + (int64_t)slot * a.ctx * nh * hp;
    for (int c = tid; c < ncol; c += NT) {
      const int g = c / hp;
      *(u32x4*)(dst + value_index(t0, g, c - g * hp, nh, hp)) = *(const u32x4*)(stage + c * 8);
    }
  }
}

// the projections of a sequence's last taps - 1 positions of this step -> ring rows p % taps (the rest of the ring stays)
template <typename T>
__global__ __launch_bounds__(256) void conv_state_kernel(const LmAttn a, int ncol) {
  const int seq = blockIdx.x;
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, pos0 = a.r.seq_pos0[seq], slot = a.r.seq_slot[seq];
  T* ring = (T*)a.conv_state + (int64_t)slot * a.taps * a.conv_ld;
  const int keep = min(len, a.taps - 1);
  for (int t = len - keep; t < len; ++t)
    for (int c = threadIdx.x * 4; c < ncol; c += 1024)
      st4(ring + (int64_t)((pos0 + t) % a.taps) * a.conv_ld + c, ld4((const T*)a.proj + (int64_t)(row0 + t) * a.ldp + c));
}

// ---------------------------------------------------------------------------------------------------------------------------
constexpr int PLAIN_TK = 64;

// A row's tiles are a chain of loads, mixture, softmax and loads again, which waves shorten (380 rows of 190 keys, 16 heads of 128, fp32: four waves 93 us, 560 us with one element per load; eight or
// sixteen 65).  NR rows that follow one another in a sequence (and, with chunks, begin at the same key): a key or value is read once for all of them.  Sums run over coordinates and keys in order, one
// chain each: the same bits whatever NR and NT.
inline int plain_lds(const LmAttn& a, int nr) { return nr * (a.heads * (a.dp + a.vp) + 2 * a.heads * PLAIN_TK + 3 * a.heads) * 4; }
template <typename T, int NT, int NR>
__device__ __forceinline__ void attn_plain_rows(const LmAttn& a, int row, float* sm) {
  const int H = a.heads, G = a.kv_heads, dp = a.dp, vp = a.vp, rep = H / G;
  float* qs = sm;                           // [NR][H][dp]
  float* acc = qs + NR * H * dp;            // [NR][H][vp]
  float* raw = acc + NR * H * vp;           // [NR][H][TK]
  float* mixed = raw + NR * H * PLAIN_TK;   // [NR][H][TK]
  float* ms = mixed + NR * H * PLAIN_TK;    // [NR][H] running maximum
  float* ls = ms + NR * H;                  // [NR][H] running sum
  float* al = ls + NR * H;                  // [NR][H] rescale of this tile
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int seq = a.r.row_seq[row], i = a.r.row_pos[row], slot = a.r.seq_slot[seq];
  const T* kb = (const T*)a.k + (int64_t)slot * G * a.ctx * dp;
  const T* vb = (const T*)a.v + (int64_t)slot * G * a.ctx * vp;
  for (int c = tid; c < NR * H * dp; c += NT) qs[c] = ldf((const T*)a.q + (int64_t)row * H * dp + c);
  for (int c = tid; c < NR * H * vp; c += NT) acc[c] = 0.f;
  for (int h = tid; h < NR * H; h += NT) {
    ms[h] = -INFINITY;
    ls[h] = 0.f;
  }
  __syncthreads();
  const int first = a.chunk > 0 ? i / a.chunk * a.chunk : 0;
  for (int j0 = first; j0 < i + NR; j0 += PLAIN_TK) {
    int n[NR];  // keys of this tile that a row sees
#pragma unroll
    for (int r = 0; r < NR; ++r) n[r] = max(0, min(PLAIN_TK, i + r + 1 - j0));
    for (int e = tid; e < H * PLAIN_TK; e += NT) {
      const int g = e / PLAIN_TK, jj = e - g * PLAIN_TK;
      if (jj >= n[NR - 1]) continue;
      float s[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r) s[r] = 0.f;
#pragma unroll 4
      for (int d = 0; d < dp; d += 8) {  // (coordinates behind the head's are zeros)
        const auto k = ld8(kb + key_index(j0 + jj, g / rep, d, G, dp));
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          const f32x4 kv = half8(k, hf);
#pragma unroll
          for (int r = 0; r < NR; ++r) {
            const f32x4 qv = *(const f32x4*)(qs + (r * H + g) * dp + d + 4 * hf);
#pragma unroll
            for (int t = 0; t < 4; ++t) s[r] = __builtin_fmaf(qv[t], kv[t], s[r]);
          }
        }
      }
#pragma unroll
      for (int r = 0; r < NR; ++r) raw[r * H * PLAIN_TK + e] = __builtin_fmaf(a.scale, s[r], -(a.slope[g] * (float)(i + r - (j0 + jj))));
    }
    __syncthreads();
    for (int e = tid; e < NR * H * PLAIN_TK; e += NT) {
      const int r = NR == 1 ? 0 : e / (H * PLAIN_TK), h = e / PLAIN_TK - r * H, jj = e % PLAIN_TK;
      float s = -INFINITY;
      if (jj < min(PLAIN_TK, i + r + 1 - j0)) {
        s = 0.f;
#pragma unroll 4
        for (int g = 0; g < H; ++g) s += a.mix[h * H + g] * raw[(r * H + g) * PLAIN_TK + jj];
      }
      mixed[e] = s;
    }
    __syncthreads();
    for (int h = wave; h < NR * H; h += NT / 64) {
      if (NR > 1 && j0 > i + h / H) {  // (uniform) no key of this tile
        if (lane == 0) al[h] = 1.f;
        continue;
      }
      const float s = mixed[h * PLAIN_TK + lane];
      const float mo = ms[h], mn = fmaxf(mo, wave_max(s));
      const float p = expf(s - mn), f = expf(mo - mn);
      const float sum = wave_sum(p);
      mixed[h * PLAIN_TK + lane] = p;
      if (lane == 0) {
        ms[h] = mn;
        ls[h] = ls[h] * f + sum;
        al[h] = f;
      }
    }
    __syncthreads();
    for (int c = tid; c < H * vp; c += NT) {
      const int h = c / vp, d = c - h * vp;
      const float* p = mixed + h * PLAIN_TK;
      float o[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r) o[r] = acc[r * H * vp + c] * al[r * H + h];
      auto one = [&](int jj) {
        const float v = ldf(vb + value_index(j0 + jj, h / rep, d, G, vp));
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if (jj < n[r]) o[r] = __builtin_fmaf(p[r * H * PLAIN_TK + jj], v, o[r]);
      };
      const int lo = min(-j0 & 7, n[0]), hi = lo + ((n[0] - lo) & ~7);  // the values of a row of eight keys lie together
      for (int jj = 0; jj < lo; ++jj) one(jj);
#pragma unroll 4
      for (int jj = lo; jj < hi; jj += 8) {
        const auto v = ld8(vb + value_index(j0 + jj, h / rep, d, G, vp));
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
          for (int r = 0; r < NR; ++r) o[r] = __builtin_fmaf(p[r * H * PLAIN_TK + jj + t], half8(v, t / 4)[t & 3], o[r]);
      }
      for (int jj = hi; jj < n[NR - 1]; ++jj) one(jj);
#pragma unroll
      for (int r = 0; r < NR; ++r) acc[r * H * vp + c] = o[r];
    }
    __syncthreads();
  }
  for (int c = tid; c < NR * H * vp; c += NT) {
    const int r = NR == 1 ? 0 : c / (H * vp), cc = c - r * H * vp;
    stf((T*)a.out + (int64_t)(row + r) * a.ldo + in_chunks(cc, a.out_chunk), acc[c] / ls[r * H + cc / vp]);
  }
}
template <typename T, int NT, int NR>
__global__ __launch_bounds__(NT) void attn_plain_kernel(const LmAttn a) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  if constexpr (NR == 1) {
    attn_plain_rows<T, NT, 1>(a, blockIdx.x, sm);
  } else {
    const int row = blockIdx.x * NR, end = min(row + NR, a.r.n_rows), last = end - 1, i = a.r.row_pos[row];
    if (end - row == NR && a.r.row_seq[row] == a.r.row_seq[last] && (a.chunk <= 0 || i / a.chunk == (i + NR - 1) / a.chunk)) {  // all of one sequence, from the same key on
      attn_plain_rows<T, NT, NR>(a, row, sm);
      return;
    }
    for (int r = row; r < end; ++r) {
      attn_plain_rows<T, NT, 1>(a, r, sm);
      __syncthreads();
    }
  }
}

template <typename T, int NT>
void (*prep_block_pick(int taps))(const LmAttn) {
  switch (taps) {
    case 1: return attn_prep_block_kernel<T, 1, NT>;
    case 2: return attn_prep_block_kernel<T, 2, NT>;
    case 3: return attn_prep_block_kernel<T, 3, NT>;
    case 4: return attn_prep_block_kernel<T, 4, NT>;
    default: return attn_prep_block_kernel<T, 0, NT>;
  }
}

template <typename T>
md_status prep(const LmAttn& a, bool state, hipStream_t s) {
  const int mx = a.heads * a.dp > a.kv_heads * a.vp ? a.heads * a.dp : a.kv_heads * a.vp;
  const int lds = mx * 4;
  const bool step = a.r.max_len == 1;
  auto fn = step ? attn_prep_kernel<T, true> : attn_prep_kernel<T, false>;
  const int mc = mx > a.kv_heads * a.dp ? mx : a.kv_heads * a.dp;
  if (step && sizeof(T) == 2 && mc <= 8192) {
    auto sf = mc <= 2048 ? attn_prep_step_kernel<1> : mc <= 4096 ? attn_prep_step_kernel<2> : attn_prep_step_kernel<4>;
    hipLaunchKernelGGL(sf, dim3(a.r.n_rows, a.own_kv ? 3 : 1), dim3(512), a.own_kv ? a.kv_heads * a.vp * 4 : 0, s, a);
  } else if (!step && mc <= 4096) {
    auto bf = mc <= 1024 ? prep_block_pick<T, 256>(a.taps) : mc <= 2048 ? prep_block_pick<T, 512>(a.taps) : prep_block_pick<T, 1024>(a.taps);
    const int nt = mc <= 1024 ? 256 : mc <= 2048 ? 512 : 1024;
    const int kvc = a.kv_heads * (a.dp > a.vp ? a.dp : a.vp);
    const int block_lds = (8 * nt + 8 * a.kv_heads) * 4 + (sizeof(T) == 2 && a.own_kv ? kvc * 16 : 0);
    MD_TRY(md_ensure_dynamic_lds((const void*)bf, 150 * 1024));
    hipLaunchKernelGGL(bf, dim3((a.r.max_len + 14) / 8, a.r.n_seq, a.own_kv ? 3 : 1), dim3(nt), block_lds, s, a);
  } else {
    if (lds > 150 * 1024) return MD_ERR_UNSUPPORTED;
    MD_TRY(md_ensure_dynamic_lds((const void*)fn, 150 * 1024));
    hipLaunchKernelGGL(fn, dim3(a.r.n_rows, a.own_kv ? 3 : 1), dim3(256), lds, s, a);
  }
  MD_TRY(md_launch_status());
  if (step || a.taps == 1 || !state) return MD_OK;
  hipLaunchKernelGGL(conv_state_kernel<T>, dim3(a.r.n_seq), dim3(256), 0, s, a, a.conv_ld);
  return md_launch_status();
}

// Eight waves where rows are so few that their chains bound it, four where CUs hold more rows than the keys' way needs, pairs of rows where that way does (ms of 12 layers, four waves / eight / pairs).
// 16 heads of 128, fp32: one prompt of 300 / 700 / 900 tokens 2.32 / 1.79 / 2.35, 4.26 / 4.13 / 4.40, 5.70 / 6.47 / 5.40, 8 x 1000 61.8 / 50.9 / 34.4; 30 x 20, whose chains are short, 1.69 / 1.66 / 1.63.
// 8 of 64: 300 / 1000 tokens 0.99 / 0.86 / 1.02, 2.21 / 2.19 / 2.30, 8 x 1000 11.1 / 12.0 / 10.0; 12 of 64: 800 tokens 2.38 / 2.43 / 2.81, 8 x 1000 16.1 / 17.7 / 15.1; 9 of 32: 5 x 500 2.61 / 2.71 / 2.74.  Up
// to four heads leave half of eight waves idle: 4 of 32, 900 tokens 1.05 / 1.35 / 1.61; 2 of 64, 8 x 1000 5.04 / 7.12 / 6.57.  Where two workgroups with pairs do not fit a CU's LDS, pairs pay only if keys and
// values outweigh the mixture: 40 of 128, 900 tokens / 3 x 900 19.6 / 17.6 / 19.5, 53.3 / 59.8 / 46.2; 64 of 64 21.4 / 16.0 / 20.9, 49.9 / 41.1 / 47.5; 48 of 64, 3 x 900 31.6 / 27.9 / 33.9.  bf16 halves
// that way: 40 of 64, 3 x 900 18.1 / 15.8 / 19.2, 64 of 64 42.2 / 27.9 / 34.4.
struct PlainShape {
  int threads, rows;  // of a workgroup
};
PlainShape plain_shape(const LmAttn& a, bool f32) {
  const int H = a.heads, rows = a.r.n_rows, cols = H * (a.dp + a.vp);
  if (H <= 4) return {256, 1};
  if (!f32 || rows < 8 * a.r.n_seq || plain_lds(a, 2) > 160 * 1024) return {512, 1};
  const bool many = rows >= 2048;
  if (plain_lds(a, 2) > 80 * 1024) return {512, many && a.kv_heads * (a.dp + a.vp) >= 5 * H * H ? 2 : 1};
  if (rows <= 512 || (rows <= 768 && a.r.max_ctx > PLAIN_TK)) return {512, 1};
  const bool pairs = many ? cols >= 1536 || (cols >= 1024 && H % 8 == 0) : cols >= 4096;
  return pairs ? PlainShape{512, 2} : PlainShape{256, 1};
}

template <typename T>
md_status plain(const LmAttn& a, hipStream_t s) {
  if (plain_lds(a, 1) > 160 * 1024) return MD_ERR_UNSUPPORTED;
  const PlainShape shape = plain_shape(a, sizeof(T) == 4);
  auto fn = shape.threads == 256 ? attn_plain_kernel<T, 256, 1> : attn_plain_kernel<T, 512, 1>;
  if constexpr (sizeof(T) == 4)
    if (shape.rows == 2) fn = attn_plain_kernel<T, 512, 2>;
  MD_TRY(md_ensure_dynamic_lds((const void*)fn, 160 * 1024));
  hipLaunchKernelGGL(fn, dim3((a.r.n_rows + shape.rows - 1) / shape.rows), dim3(shape.threads), plain_lds(a, shape.rows), s, a);
  return md_launch_status();
}

}  // namespace

md_status lm_attn_prep(int dtype, const LmAttn& a, hipStream_t s) { return dtype == MD_DTYPE_F32 ? prep<float>(a, true, s) : prep<bf16_t>(a, true, s); }
md_status lm_attn_plain(int dtype, const LmAttn& a, hipStream_t s) { return dtype == MD_DTYPE_F32 ? plain<float>(a, s) : plain<bf16_t>(a, s); }

// ---------------------------------------------------------------------------------------------------------------------------
namespace {

constexpr float kLog2e = 1.4426950408889634f;

typedef __attribute__((ext_vector_type(2))) unsigned int u32pair;

// lane rows of 16: x0 .. x3 at lane row q become column q of the 4 x 4 (register, lane row) block
__device__ __forceinline__ void transpose_rows4(uint32_t& x0, uint32_t& x1, uint32_t& x2, uint32_t& x3) {
  u32pair r = __builtin_bit_cast(u32pair, __builtin_amdgcn_permlane32_swap(x0, x2, false, false));
  x0 = r[0];
  x2 = r[1];
  r = __builtin_bit_cast(u32pair, __builtin_amdgcn_permlane32_swap(x1, x3, false, false));
  x1 = r[0];
  x3 = r[1];
  r = __builtin_bit_cast(u32pair, __builtin_amdgcn_permlane16_swap(x0, x1, false, false));
  x0 = r[0];
  x1 = r[1];
  r = __builtin_bit_cast(u32pair, __builtin_amdgcn_permlane16_swap(x2, x3, false, false));
  x2 = r[0];
  x3 = r[1];
}

struct TalkLds {
  int q, p, mx, al, ms, total;  // byte offsets
};
__host__ __device__ constexpr TalkLds talk_lds(int hpad, int dp, int nw) {
  TalkLds l = {};
  l.q = 0;
  l.p = l.q + hpad * 16 * (dp + 8) * 2;
  l.mx = l.p + hpad * 16 * (16 * nw + 8) * 2;
  l.al = l.mx + nw * hpad * 16 * 4;
  l.ms = l.al + hpad * 16 * 4;
  l.total = l.ms + hpad * 4;
  return l;
}

// Order of a step's tiles, as workgroups go to XCDs and their engines in turn (so neighbours have to be alike) and an XCD's CUs share keys and values in L2:
//   ROUNDS  every eighth tile of a sequence to an XCD, in eight rounds over the sequences, so that the last tiles are short
//   WHOLE   whole sequences to an XCD, tile by tile
//   ACROSS  the last tile of every sequence, then the ones before it, so turned that any sequence's go evenly to the 32 engines
// Longest first in each.  32 heads of 64: 11 ragged prompts, 13250 tokens, 699 us with a run of tiles per XCD, shortest first, 513 in ROUNDS; 3 x 2048 tokens 544 and
// 330; 8 x 2048 817, 785 and 691 WHOLE (launches of one after the other; in a whole pass 915 with a run per XCD, 798 WHOLE).  Persistent workgroups with a
// queue per XCD: 697, 460 and 1064, the loop around the tile costs registers.
enum { TALK_ROUNDS, TALK_WHOLE, TALK_ACROSS };

// Parts of a tile's keys: a tile's place among all tiles of a step (a sequence has at most len / 16 + 2), and what one part leaves.  Their room is the most that any
// step up to the workspace's size can want, since a workspace of the largest serves all: at most 208 MB with 32 heads of 64 (1536 times 135 KB).
constexpr int TALK_TURNS = 8, TALK_PARTS = 1536, TALK_LEAST = 3;  // parts of a step at most; 64 keys of a part at least
__host__ __device__ inline int talk_turns(int tiles8, int parts) { return parts > 1 ? 1 : tiles8 < TALK_TURNS ? tiles8 : TALK_TURNS; }
inline int talk_longest(int span) { return (span + 31 + 63) / 64; }  // of 64 keys each; the first may begin before the chunk
__device__ __forceinline__ int talk_slot(int row0, int seq, int tile) { return row0 / 16 + 2 * seq + tile; }
__host__ __device__ inline int64_t talk_part_floats(int heads, int vp) { return (int64_t)heads * (16 * vp + 32); }

// keeps the compiler from overlapping the phases of a tile: their register peaks would add up
#define PHASE() __builtin_amdgcn_sched_barrier(0)

// HB: blocks of 16 heads, NW: waves, HPW: output heads per wave, D: dp / 32 (0: at run time), C: vp / 32.
// The loads of a tile run ahead of their use: K in groups of heads (the first group of the next tile is requested before this tile's
// P V), V two steps of 32 keys ahead (the first before the softmax).  Heads beyond H run on zero queries and the last head's keys; the
// mixing matrix is zero there and nothing of theirs is stored, so no per-head branch cuts the schedule.  Rows past the last live key
// are read (up to TK of them: the slabs have as many spare rows at their end) and masked.
template <int HB, int NW, int HPW, int D, int C>
__global__ __launch_bounds__(NW * 64, NW / 4) void attn_mfma_kernel(const LmAttn a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int HP = HB * 16, TK = 16 * NW, PS = TK + 8;
  constexpr int KF = D == 0 ? 1 : D;                        // operand pieces per head held in registers at once
  constexpr int KG = D == 0 ? 1 : 16 / (D == 3 ? 4 : D);  // heads per K group: divides 16
  constexpr int NG = HP / KG;
  static_assert(NG * KG == HP, "every head belongs to a group");
  constexpr int NS = HPW * (TK / 32), PD = 2;  // V steps of a tile, and how many are requested ahead
  const int H = a.heads, G = a.kv_heads, rep = H / G, dp = D ? 32 * D : a.dp, vp = 32 * C;
  const TalkLds L = talk_lds(HP, dp, NW);
  bf16_t* Qs = (bf16_t*)(smem + L.q);
  bf16_t* Ps = (bf16_t*)(smem + L.p);
  float* mxs = (float*)(smem + L.mx);
  float* als = (float*)(smem + L.al);
  float* mss = (float*)(smem + L.ms);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, q = lane >> 4;

  // which tile, counted from the sequence's last, and which part of its keys
  const int tiles = (a.r.max_len + 30) / 16, N = a.r.n_seq, xcd = blockIdx.x & 7, item = blockIdx.x >> 3;
  int seq, nth, part = 0;
  if (a.order == TALK_ACROSS) {
    const int rank = blockIdx.x / N;
    part = rank / tiles;
    nth = rank - part * tiles;
    seq = (blockIdx.x + (N - nth * min(N & -N, 32) / 32 % N)) % N;  // (a step of N workgroups meets 32 / gcd(N, 32) engines)
  } else if (a.order == TALK_WHOLE) {
    const int each = (N + 7) >> 3;
    nth = item / each;
    seq = 8 * (item - nth * each) + xcd;
    if (seq >= N) return;
  } else {
    const int tiles8 = (tiles + 7) >> 3, turns = talk_turns(tiles8, a.n_split), per = (tiles8 + turns - 1) / turns;
    part = a.n_split > 1 ? item / (per * N) : 0;
    const int at = item - part * per * N;
    seq = at / per % N;
    nth = (at / (per * N) * per + (at + (N == 1 ? part : 0)) % per) * 8 + ((xcd + seq) & 7);  // (a single sequence's parts begin at another engine each)
  }
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, pos0 = a.r.seq_pos0[seq], slot = a.r.seq_slot[seq];
  const int tile = (pos0 + len - 1) / 16 - pos0 / 16 - nth;
  if (tile < 0) return;
  const int t0 = (pos0 / 16 + tile) * 16;
  const int lo = max(t0, pos0), hi = min(t0 + 15, pos0 + len - 1);  // positions of the tile's live queries
  // its keys, and this part of them
  const int kfirst = (a.chunk > 0 ? lo / a.chunk * a.chunk : 0) & ~31;
  const int kstart = kfirst + part * a.split_keys, klast = min(hi, kstart + a.split_keys - 1);
  if (kstart > hi) return;
  const bool whole = kfirst + a.split_keys > hi;
  const bf16_t* Kb = (const bf16_t*)a.k + (int64_t)slot * G * a.ctx * dp;
  const bf16_t* Vb = (const bf16_t*)a.v + (int64_t)slot * G * a.ctx * vp;

  {  // queries of the tile (rows outside it replay a live one)
    const int dc = dp >> 3;
    for (int i = tid; i < HP * 16 * dc; i += NW * 64) {
      const int ch = i % dc, hn = i / dc, qn = hn & 15, h = hn >> 4;
      const int64_t row = row0 + min(max(t0 + qn, lo), hi) - pos0;
      u32x4 v = {0u, 0u, 0u, 0u};
      if (h < H) v = *(const u32x4*)((const bf16_t*)a.q + (row * H + h) * dp + ch * 8);
      *(u32x4*)(Qs + hn * (dp + 8) + ch * 8) = v;
    }
    constexpr int LH = NW * 64 / HP;  // lanes per head
    float s = 0.f;
    for (int h = tid / LH, g = tid % LH; g < H; g += LH) s += h < H ? a.mix[h * H + g] * a.slope[g] : 0.f;
#pragma unroll
    for (int o = LH / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (tid % LH == 0) mss[tid / LH] = s * kLog2e;
  }
  // A operand of the mixture: row h = 16 mt + n, heads 8 q .. 8 q + 7 (HB 2) or 4 q .. 4 q + 3 (HB 1)
  bf16x8 tf[HB];
#pragma unroll
  for (int mt = 0; mt < HB; ++mt)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int h = 16 * mt + n, g = HB == 2 ? 8 * q + j : 4 * q + j;
      tf[mt][j] = (h < H && g < H && (HB == 2 || j < 4)) ? (short)f2bf(a.mix[h * H + g]) : (short)0;
    }
  __syncthreads();

  float m_run[HB * 4], l_run[HB * 4], ms[HB * 4];
#pragma unroll
  for (int i = 0; i < HB * 4; ++i) {
    m_run[i] = -INFINITY;
    l_run[i] = 0.f;
    ms[i] = mss[16 * (i >> 2) + 4 * q + (i & 3)];
  }
  f32x4 oacc[HPW][2 * C];
#pragma unroll
  for (int i = 0; i < HPW; ++i)
#pragma unroll
    for (int t = 0; t < 2 * C; ++t) oacc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  const float scale = a.scale * kLog2e;
  const int qpos = t0 + n, qfirst = a.chunk > 0 ? qpos / a.chunk * a.chunk : 0;
  const int hfirst = a.chunk > 0 ? hi / a.chunk * a.chunk : 0;

  // Byte strides of a block of 32 keys / values and the reciprocal of the group size, made opaque once per tile: the heads' base addresses are
  // then computed where they are used (scalar) instead of being kept in registers across the whole loop.
  const uint32_t lane16 = 16 * lane;
  uint32_t kbs = (uint32_t)G * dp * 64, vbs = (uint32_t)G * vp * 64, inv_rep = (65535u + rep) / rep;
  auto kv_head = [&](int h) { return ((uint32_t)min(h, H - 1) * inv_rep) >> 16; };
  bf16x8 kf[2][KG][KF];
  auto load_k = [&](int buf, int grp, int jw) {
    if constexpr (D > 0) {
      const char* blk = (const char*)Kb + (uint64_t)(jw >> 5) * kbs + ((jw >> 4) & 1) * (D * 1024);
#pragma unroll
      for (int k = 0; k < KG; ++k) {
        const char* kb = blk + kv_head(grp * KG + k) * (2048 * D);
#pragma unroll
        for (int d = 0; d < KF; ++d) kf[buf][k][d] = *(const bf16x8*)(kb + 1024 * d + lane16);
      }
    }
  };
  u32x4 vr[PD + 1][2 * C];
  auto load_v = [&](int step, int j0) {  // step = output head of this wave * (TK / 32) + block of 32 keys
    const char* vb = (const char*)Vb + (uint64_t)((j0 >> 5) + step % (TK / 32)) * vbs + kv_head(wave * HPW + step / (TK / 32)) * (2048 * C);
#pragma unroll
    for (int t = 0; t < 2 * C; ++t) vr[step % (PD + 1)][t] = *(const u32x4*)(vb + 1024 * t + lane16);
  };

  load_k(0, 0, kstart + 16 * wave);
  for (int j0 = kstart; j0 <= klast; j0 += TK) {
    asm volatile("" : "+s"(kbs), "+s"(vbs), "+s"(inv_rep));
    const int jw = j0 + 16 * wave;
    const bool live = jw <= hi;
    f32x4 st[4][4][HB];  // [r'][q'][block of 16 heads]: key 4 q' + r', heads 16 mt + 4 q + r
    float mx[HB * 4];
#pragma unroll
    for (int i = 0; i < HB * 4; ++i) mx[i] = -INFINITY;
    if (live) {
      f32x4 acc[HP];
      if constexpr (D > 0) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          if (g + 1 < NG) load_k((g + 1) & 1, g + 1, jw);
          PHASE();
#pragma unroll
          for (int k = 0; k < KG; ++k) acc[g * KG + k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int d = 0; d < KF; ++d)
#pragma unroll
            for (int k = 0; k < KG; ++k) {
              const int h = g * KG + k;
              const bf16x8 qf = *(const bf16x8*)(Qs + (h * 16 + n) * (dp + 8) + 8 * q + 32 * d);
              acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(md_bf16x8v, kf[g & 1][k][d]), __builtin_bit_cast(md_bf16x8v, qf),
                                                               acc[h], 0, 0, 0);
            }
        }
      } else {
#pragma unroll
        for (int h = 0; h < HP; ++h) {
          acc[h] = f32x4{0.f, 0.f, 0.f, 0.f};
          const bf16_t* kp = Kb + key_block(jw, kv_head(h), G, dp) + ((jw >> 4) & 1) * (dp >> 5) * 512 + 8 * lane;
          const bf16_t* qp = Qs + (h * 16 + n) * (dp + 8) + 8 * q;
          for (int d = 0; d < dp; d += 32)
            acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(md_bf16x8v, *(const bf16x8*)(kp + 16 * d)),
                                                             __builtin_bit_cast(md_bf16x8v, *(const bf16x8*)(qp + d)), acc[h], 0, 0, 0);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        PHASE();
        uint32_t ph[HP / 2], pl[HP / 2];
#pragma unroll
        for (int i = 0; i < HP / 2; ++i) {
          const float x = acc[2 * i][r], y = acc[2 * i + 1][r];
          ph[i] = pack_bf16x2(x, y);
          pl[i] = pack_bf16x2(x - lo_bf(ph[i]), y - hi_bf(ph[i]));
        }
        constexpr int W = HB == 2 ? 4 : 2;  // dwords of an operand
#pragma unroll
        for (int i = 0; i < W; ++i) {
          transpose_rows4(ph[i], ph[W + i], ph[2 * W + i], ph[3 * W + i]);
          transpose_rows4(pl[i], pl[W + i], pl[2 * W + i], pl[3 * W + i]);
        }
#pragma unroll
        for (int part = 0; part < 2; ++part)  // low parts, then high parts on top
#pragma unroll
          for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int mt = 0; mt < HB; ++mt) {
              const uint32_t* p = part == 0 ? pl : ph;
              const f32x4 z = part == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : st[r][k][mt];
              if constexpr (HB == 2) {
                const u32x4 b = {p[4 * k], p[4 * k + 1], p[4 * k + 2], p[4 * k + 3]};
                st[r][k][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(md_bf16x8v, tf[mt]), __builtin_bit_cast(md_bf16x8v, b), z, 0, 0, 0);
              } else {
                const u32x2 b = {p[2 * k], p[2 * k + 1]};
                const bf16x4 t = {tf[mt][0], tf[mt][1], tf[mt][2], tf[mt][3]};
                st[r][k][mt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(t, __builtin_bit_cast(bf16x4, b), z, 0, 0, 0);
              }
            }
      }
      PHASE();
      // scaled and biased scores (in powers of two), the wave's maximum per (head, query)
      const float dist0 = (float)(qpos - jw);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float dist = dist0 - (float)(4 * k + r);
#pragma unroll
          for (int i = 0; i < HB * 4; ++i) st[r][k][i >> 2][i & 3] = st[r][k][i >> 2][i & 3] * scale - ms[i] * dist;
        }
      if (!(jw >= hfirst && jw + 15 <= lo)) {  // some pair of the block is not visible
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int j = jw + 4 * k + r;
            if (j > qpos || j < qfirst) {
#pragma unroll
              for (int i = 0; i < HB * 4; ++i) st[r][k][i >> 2][i & 3] = -INFINITY;
            }
          }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int i = 0; i < HB * 4; ++i) mx[i] = fmaxf(mx[i], st[r][k][i >> 2][i & 3]);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int mt = 0; mt < HB; ++mt) st[r][k][mt] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    }
#pragma unroll
    for (int p = 0; p < PD; ++p)
      if (p < NS) load_v(p, j0);
#pragma unroll
    for (int i = 0; i < HB * 4; ++i) mxs[(wave * HP + 16 * (i >> 2) + 4 * q + (i & 3)) * 16 + n] = mx[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < HB * 4; ++i) {
      PHASE();
      const int h = 16 * (i >> 2) + 4 * q + (i & 3);
      float m = m_run[i];
#pragma unroll
      for (int w = 0; w < NW; ++w) m = fmaxf(m, mxs[(w * HP + h) * 16 + n]);
      const float ref = m == -INFINITY ? 0.f : m;
      const float f = __builtin_amdgcn_exp2f(m_run[i] - ref);
      if (wave == 0) als[h * 16 + n] = f;
      float sum = 0.f;
      uint32_t pk[8];
#pragma unroll
      for (int k2 = 0; k2 < 8; ++k2) {  // keys 2 k2, 2 k2 + 1
        const float p0 = __builtin_amdgcn_exp2f(st[(2 * k2) & 3][(2 * k2) >> 2][i >> 2][i & 3] - ref);
        const float p1 = __builtin_amdgcn_exp2f(st[(2 * k2 + 1) & 3][(2 * k2 + 1) >> 2][i >> 2][i & 3] - ref);
        sum += p0 + p1;
        pk[k2] = pack_bf16x2(p0, p1);
      }
      l_run[i] = l_run[i] * f + sum;
      m_run[i] = m;
      bf16_t* dst = Ps + (h * 16 + n) * PS + 16 * wave;
      *(u32x4*)dst = u32x4{pk[0], pk[1], pk[2], pk[3]};
      *(u32x4*)(dst + 8) = u32x4{pk[4], pk[5], pk[6], pk[7]};
    }
    __syncthreads();
    if (j0 + TK <= klast) load_k(0, 0, jw + TK);
#pragma unroll
    for (int step = 0; step < NS; ++step) {
      if (step + PD < NS) load_v(step + PD, j0);
      PHASE();
      const int hh = step / (TK / 32), s = step % (TK / 32), h = wave * HPW + hh;
      if (s == 0) {
        const f32x4 al = *(const f32x4*)(als + h * 16 + 4 * q);
        if (__any(al[0] != 1.f || al[1] != 1.f || al[2] != 1.f || al[3] != 1.f)) {
#pragma unroll
          for (int t = 0; t < 2 * C; ++t) oacc[hh][t] *= al;
        }
      }
      const bf16x8 pf = *(const bf16x8*)(Ps + (h * 16 + n) * PS + 32 * s + 8 * q);
#pragma unroll
      for (int t = 0; t < 2 * C; ++t)
        oacc[hh][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(md_bf16x8v, pf), __builtin_bit_cast(md_bf16x8v, vr[step % (PD + 1)][t]),
                                                              oacc[hh][t], 0, 0, 0);
    }
  }
  // the waves' sums over their own keys (they shared every maximum)
#pragma unroll
  for (int i = 0; i < HB * 4; ++i) mxs[(wave * HP + 16 * (i >> 2) + 4 * q + (i & 3)) * 16 + n] = l_run[i];
  __syncthreads();
  // one of several parts: its sums as the lanes hold them, its maxima and weights
  float* part_o = a.part + ((int64_t)talk_slot(row0, seq, tile) * a.n_split + part) * talk_part_floats(H, vp);
  float* part_ml = part_o + H * 16 * vp;
  if (!whole && wave == 0)
#pragma unroll
    for (int i = 0; i < HB * 4; ++i) {
      const int h = 16 * (i >> 2) + 4 * q + (i & 3);
      if (h < H) part_ml[h * 32 + n] = m_run[i];
    }
#pragma unroll
  for (int hh = 0; hh < HPW; ++hh) {
    const int h = wave * HPW + hh;
    if (h >= H) continue;
    f32x4 l = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) l += *(const f32x4*)(mxs + (w * HP + h) * 16 + 4 * q);
    if (!whole) {
      if (n == 0) *(f32x4*)(part_ml + h * 32 + 16 + 4 * q) = l;
#pragma unroll
      for (int t = 0; t < 2 * C; ++t) *(f32x4*)(part_o + ((h * 2 * C + t) * 64 + lane) * 4) = oacc[hh][t];
      continue;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int pos = t0 + 4 * q + r;
      if (pos < lo || pos > hi) continue;
      const float inv = 1.0f / l[r];
      bf16_t* dst = (bf16_t*)a.out + (int64_t)(row0 + pos - pos0) * a.ldo + in_chunks(h * vp + n, a.out_chunk);
#pragma unroll
      for (int t = 0; t < 2 * C; ++t) dst[2 * t * a.out_chunk] = f2bf(oacc[hh][t][r] * inv);
    }
  }
}

// sums the parts of a tile: grid (tiles, sequences, groups of 4 heads), a wave per head
__global__ __launch_bounds__(256) void attn_parts_kernel(const LmAttn a) {
  const int seq = blockIdx.y, h = blockIdx.z * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, n = lane & 15, q = lane >> 4;
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, pos0 = a.r.seq_pos0[seq];
  const int tile = blockIdx.x, t0 = (pos0 / 16 + tile) * 16, lo = max(t0, pos0), hi = min(t0 + 15, pos0 + len - 1);
  const int kfirst = (a.chunk > 0 ? lo / a.chunk * a.chunk : 0) & ~31;
  if (lo > hi || h >= a.heads || kfirst + a.split_keys > hi) return;
  const int parts = (hi - kfirst) / a.split_keys + 1, pieces = a.vp / 16;
  const int64_t stride = talk_part_floats(a.heads, a.vp);
  const float* p = a.part + (int64_t)talk_slot(row0, seq, tile) * a.n_split * stride;
  const float* ml = p + a.heads * 16 * a.vp + h * 32 + 4 * q;
  f32x4 m = {-INFINITY, -INFINITY, -INFINITY, -INFINITY}, l = {0.f, 0.f, 0.f, 0.f}, o[8];
  for (int k = 0; k < parts; ++k) {
    const f32x4 mk = *(const f32x4*)(ml + k * stride);
#pragma unroll
    for (int r = 0; r < 4; ++r) m[r] = fmaxf(m[r], mk[r]);
  }
#pragma unroll
  for (int t = 0; t < 8; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < parts; ++k) {
    const f32x4 mk = *(const f32x4*)(ml + k * stride), lk = *(const f32x4*)(ml + k * stride + 16);
    f32x4 w;
#pragma unroll
    for (int r = 0; r < 4; ++r) w[r] = __builtin_amdgcn_exp2f(mk[r] - m[r]);
    l += w * lk;
#pragma unroll
    for (int t = 0; t < 8; ++t)
      if (t < pieces) o[t] += w * *(const f32x4*)(p + k * stride + ((h * pieces + t) * 64 + lane) * 4);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int pos = t0 + 4 * q + r;
    if (pos < lo || pos > hi) continue;
    const float inv = 1.0f / l[r];
    bf16_t* dst = (bf16_t*)a.out + (int64_t)(row0 + pos - pos0) * a.ldo + in_chunks(h * a.vp + n, a.out_chunk);
#pragma unroll
    for (int t = 0; t < 8; ++t)
      if (t < pieces) dst[2 * t * a.out_chunk] = f2bf(o[t][r] * inv);
  }
}

typedef void (*TalkKernel)(const LmAttn);
struct TalkPick {
  TalkKernel fn;
  int waves, lds;
};

template <int HB, int NW, int HPW, int C>
TalkKernel talk_by_dim(int dp) {
  if (dp == 32 * C) return attn_mfma_kernel<HB, NW, HPW, C, C>;  // keys as wide as values: operand loads run ahead
  return attn_mfma_kernel<HB, NW, HPW, 0, C>;
}
template <int HB, int NW, int HPW>
TalkKernel talk_by_width(int dp, int vp) {
  switch (vp / 32) {
    case 1: return talk_by_dim<HB, NW, HPW, 1>(dp);
    case 2: return talk_by_dim<HB, NW, HPW, 2>(dp);
    case 3: return talk_by_dim<HB, NW, HPW, 3>(dp);
    case 4: return talk_by_dim<HB, NW, HPW, 4>(dp);
    default: return nullptr;
  }
}

TalkPick talk_pick(const LmAttn& a) {
  constexpr int LDS = 160 * 1024;
  const int H = a.heads, dp = a.dp, vp = a.vp;
  TalkPick t{nullptr, 0, 0};
  auto fits = [&](int hpad, int nw) { return (t.lds = talk_lds(hpad, dp, nw).total) <= LDS; };
  if (H <= 16 && fits(16, 4)) {
    t.waves = 4;
    t.fn = H <= 4 ? talk_by_width<1, 4, 1>(dp, vp) : H <= 8 ? talk_by_width<1, 4, 2>(dp, vp) : talk_by_width<1, 4, 4>(dp, vp);
  } else if (H > 16 && H <= 32 && vp <= 64 && fits(32, 4)) {
    t.waves = 4;
    t.fn = vp == 32 ? talk_by_dim<2, 4, 8, 1>(dp) : talk_by_dim<2, 4, 8, 2>(dp);
  }
  return t;
}

}  // namespace

bool lm_attn_mfma_takes(const LmAttn& a) { return talk_pick(a).fn != nullptr; }
// How many parts a tile's keys are cut into, and their length.  A tile of 64 keys takes 9.7 us and a workgroup 12 us besides, so a step of
// fewer tiles than CUs lasts as long as its longest: 32 heads of 64, one prompt of 1000 tokens (63 tiles) 163 us, in six parts 63; 700 tokens 117 and 57, 350
// 67 and 48, 200 as before; two prompts of 1500 tokens 246 and 162, five ragged ones (3900 tokens, 244 tiles) 227 and 200.  Up to 128 tiles the parts fill the
// CUs once, up to 256 twice.  With more tiles the sums of the parts (132 KB each, written and read) cost more than they even out: 3 x 2048 tokens
// 341 us whole, 368 in three parts.  So they do where nearly every CU has a tile and all are alike short, so the expected times are compared: two layers,
// 12 x 300 tokens 594 us whole and 597 in parts, 6 x 600 677 and 692, 16 x 240 564 and 596, 10 x 400 674 (not cut).
int lm_attn_mfma_parts(const LmRows& r, int ctx_rows, int span, int heads, int vp, int* split_keys) {
  const int tiles = r.n_rows / 16 + r.n_seq, longest = talk_longest(span);
  int keys = longest;
  if (tiles <= 256) {
    const double mean = longest - std::min<double>(r.n_rows / r.n_seq, span) / 128;
    keys = std::max(TALK_LEAST, (int)(1.4 * tiles * mean / (tiles <= 128 ? 256 : 512)));
    const int most = TALK_PARTS / (r.n_rows / 16 + 2 * r.n_seq);
    if (most < 2) keys = longest;
    else keys = std::max(keys, (longest + most - 1) / most);
  }
  if (keys + 1 < longest) {
    double mean = (ctx_rows - 0.5 * r.n_rows) / r.n_seq;  // keys of a tile
    if (span < r.max_ctx) mean = std::min(mean, 0.5 * span);
    mean /= 64;
    const double most = 12 + 9.7 * keys, parts = tiles * (mean / keys + 0.5);
    const double compute = parts <= 256 ? most : std::max(most, (12 * parts + 9.7 * tiles * mean) / 256 + most / 2);
    if (compute + 5 + parts * talk_part_floats(heads, vp) * 4 / 2e6 >= 12 + 9.7 * longest) keys = longest;  // (sums: 1 MB in 0.5 us)
  } else {
    keys = longest;
  }
  *split_keys = 64 * keys;
  return (longest + keys - 1) / keys;
}
size_t lm_attn_mfma_part_floats_most(int n_rows, int n_seq, int span, int heads, int vp) {
  const int64_t parts = (talk_longest(span) + TALK_LEAST - 1) / TALK_LEAST, slots = n_rows / 16 + 2 * n_seq;
  return parts > 1 ? (size_t)std::min<int64_t>(TALK_PARTS, slots * parts) * talk_part_floats(heads, vp) : 0;
}
// WHOLE where the fullest XCD has at most a tenth more than the mean: two layers, 15 x 1000 tokens 2336 us in ROUNDS and 2117, 7 x 2000 + 1999 2978 and
// 2834, 32 x 100 520 and 505.  Otherwise ACROSS for fewer than 16 tiles, which leave most XCDs or engines idle in ROUNDS, and for parts of several sequences: 63
// single tokens beside a prompt of 40, 1900 keys, 1117 and 619 us, 39 beside 1500 tokens, 1000 keys, 937 and 713, 20 x 200 648 and 606 (one sequence after
// the other).
static int talk_order(const LmRows& r, int n_split) {
  const int64_t fullest = (int64_t)((r.n_seq + 7) / 8) * 8 * r.max_len;
  if (n_split == 1 && 10 * fullest <= 11 * (int64_t)r.n_rows) return TALK_WHOLE;
  return (r.max_len + 30) / 16 < 16 || (n_split > 1 && r.n_seq > 1) ? TALK_ACROSS : TALK_ROUNDS;
}
md_status lm_attn_mfma(const LmAttn& args, hipStream_t s) {
  const TalkPick t = talk_pick(args);
  if (!t.fn) return MD_ERR_UNSUPPORTED;
  MD_TRY(md_ensure_dynamic_lds((const void*)t.fn, 160 * 1024));
  LmAttn a = args;
  a.order = talk_order(a.r, a.n_split);
  const int tiles = (a.r.max_len + 30) / 16, tiles8 = (tiles + 7) / 8, turns = talk_turns(tiles8, a.n_split);
  const int items = a.order == TALK_ACROSS  ? tiles * a.r.n_seq * a.n_split
                    : a.order == TALK_WHOLE ? 8 * ((a.r.n_seq + 7) / 8) * tiles
                                            : 8 * turns * ((tiles8 + turns - 1) / turns) * a.r.n_seq * a.n_split;
  hipLaunchKernelGGL(t.fn, dim3(items), dim3(t.waves * 64), t.lds, s, a);
  MD_TRY(md_launch_status());
  if (a.n_split == 1) return MD_OK;
  hipLaunchKernelGGL(attn_parts_kernel, dim3(tiles, a.r.n_seq, (a.heads + 3) / 4), dim3(256), 0, s, a);
  return md_launch_status();
}

// ---------------------------------------------------------------------------------------------------------------------------
// Prompts of up to 978 keys (PAIRS_MOST blocks of 32; see lm_attn_pairs_takes) and 40 million scores: attn_mfma_kernel has few tiles then, and each is a long chain.  The mixed scores of all pairs fit the caches (4 bytes of a head
// and pair), so they go through memory:
//   attn_pairs_scores_kernel  (32 keys, 16 queries): a wave's share of the heads, their scores to LDS in the order of the mixture's operand (two bf16 for
//                             a float), mixture, scale, distance and mask; the scores leave in the order of the other kernel's operand.  One workgroup row
//                             more keeps the convolution's state
//   attn_pairs_out_kernel     (head, 16 queries): softmax over all keys, weighted values; a wave has every NW-th block of 32 keys, whose scores are loaded
//                             before the first is used, and the waves' sums meet in LDS
// 32 heads of 64, one prompt of 40 / 250 tokens: 10 and 4 / 5 us a layer, against 28 / 53 us (parts of keys and their sum) and 6 for the state.  Whole prompts through
// 24 layers (12 of attention), before and now, with attn_prep_block_kernel's share: 40 / 250 / 550 / 900 tokens 2.06 / 3.15 / 3.75 / 4.82 -> 1.78 / 2.58 / 3.33 / 4.53 ms; 4 x 50 / 200 / 500
// 2.72 / 4.60 / 7.97 -> 2.44 / 4.15 / 7.83.  Scores of 48 million floats (12 x 300 tokens) took 11.64 for 11.51 ms: hence PAIRS_FLOATS.
namespace {

typedef void (*TalkKernelBlocks)(const LmAttn, int);
constexpr int PAIRS_BLOCKS = 4, PAIRS_MOST = 8 * PAIRS_BLOCKS;  // blocks of 32 keys: of a wave, and of a tile

// (a tile's first block may begin before the chunk, and its last query may be one of the next chunk)
__host__ __device__ inline int pairs_blocks(int span) { return (span - 1 + 15 + 31) / 32 + 1; }
__host__ __device__ inline int64_t pairs_at(int64_t slot, int h, int kb, int H, int blocks) { return ((slot * H + h) * blocks + kb) * 512; }

// The sequence whose tile has this slot (talk_slot), and which of its tiles that is.  Workgroups are launched for slots, of which a sequence of one token has two, and not for
// as many tiles as the longest of the sequences has: steps of ten layers, 4 heads of 64, 60 running sequences of 850 keys beside a prompt of 900 1.40 -> 0.94 ms (58 empty tiles
// a running sequence, each in 30 blocks of keys; attn_mfma_kernel 1.13), 8 heads 1.57 -> 1.12 (1.30); even batches as before
__device__ __forceinline__ int pairs_seq(const LmRows& r, int slot, int& tile) {
  int seq = 0;
  if (r.n_seq > 1) {
    const int lane = threadIdx.x & 63;
    seq = -1;
    for (int s0 = 0; s0 < r.n_seq; s0 += 64) {
      const int n = __popcll(__ballot(s0 + lane < r.n_seq && talk_slot(r.seq_row0[min(s0 + lane, r.n_seq - 1)], s0 + lane, 0) <= slot));
      seq += n;
      if (n < 64) break;
    }
  }
  tile = slot - talk_slot(r.seq_row0[seq], seq, 0);
  return seq;
}
inline int pairs_slots(const LmRows& r) { return r.n_rows / 16 + 2 * r.n_seq; }

template <int HB, int D>
__global__ __launch_bounds__(256) void attn_pairs_scores_kernel(const LmAttn a, int blocks) {
  constexpr int HP = 16 * HB, HW = HP / 4, dp = 32 * D, W = HW / 2;  // heads of a wave, dwords of them in an operand
  typedef typename std::conditional<HB == 2, u32x4, u32x2>::type Op;
  __shared__ Op b_lds[32][2][4][16];  // [key][high | low part][wave][query]
  __shared__ float mss[HP];
  const int H = a.heads, G = a.kv_heads, rep = H / G, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, q = lane >> 4;
  const int kb = blockIdx.x, keeps = (int)blockIdx.y - ((int)gridDim.y - a.r.n_seq);  // >= 0: the sequence whose state is kept
  int tile = 0;
  const int seq = keeps >= 0 ? keeps : pairs_seq(a.r, blockIdx.y, tile);
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, pos0 = a.r.seq_pos0[seq], slot = a.r.seq_slot[seq];
  if (keeps >= 0) {  // conv_state_kernel's work
    bf16_t* ring = (bf16_t*)a.conv_state + (int64_t)slot * a.taps * a.conv_ld;
    const int keep = min(len, a.taps - 1), pieces = a.conv_ld / 4, n_pieces = keep * pieces, step = gridDim.x * 256;
    constexpr int AT_ONCE = 8;
    for (int p0 = kb * 256 + tid; p0 < n_pieces; p0 += AT_ONCE * step) {
      u32x2 v[AT_ONCE];
#pragma unroll
      for (int k = 0; k < AT_ONCE; ++k) {
        const int p = min(p0 + k * step, n_pieces - 1), t = len - keep + p / pieces;
        v[k] = *(const u32x2*)((const bf16_t*)a.proj + (int64_t)(row0 + t) * a.ldp + p % pieces * 4);
      }
#pragma unroll
      for (int k = 0; k < AT_ONCE; ++k) {
        const int p = p0 + k * step, t = len - keep + p / pieces;
        if (p < n_pieces) *(u32x2*)(ring + (int64_t)((pos0 + t) % a.taps) * a.conv_ld + p % pieces * 4) = v[k];
      }
    }
    return;
  }
  const int t0 = (pos0 / 16 + tile) * 16, lo = max(t0, pos0), hi = min(t0 + 15, pos0 + len - 1);  // positions of the live queries
  const int j0 = ((a.chunk > 0 ? lo / a.chunk * a.chunk : 0) & ~31) + 32 * kb;
  if (lo > hi || j0 > hi) return;
  const bf16_t* qrow = (const bf16_t*)a.q + (int64_t)(row0 + min(max(t0 + n, lo), hi) - pos0) * H * dp + 8 * q;  // (rows outside replay a live one)
  const bf16_t* Kb = (const bf16_t*)a.k + (int64_t)slot * G * a.ctx * dp + 8 * lane;
  // everything that the wave reads is requested before the first product (the second 16 keys where the first ones' registers get free)
  constexpr int LH = 256 / HP;  // lanes per head of the slopes' mixture
  float tm[HB][8], slope_in = 0.f;  // A operand of the mixture, as in attn_mfma_kernel
#pragma unroll
  for (int mt = 0; mt < HB; ++mt)
#pragma unroll
    for (int j = 0; j < (HB == 2 ? 8 : 4); ++j) tm[mt][j] = a.mix[min(16 * mt + n, H - 1) * H + min(HB == 2 ? 8 * q + j : 4 * q + j, H - 1)];
  u32x4 qf[HW][D], kf[HW][D];
  auto keys = [&](int x, int mt) {  // (heads beyond the last: their mixture's weights are zero)
    const bf16_t* kh = Kb + key_block(j0, min(HW * wave + x, H - 1) / rep, G, dp);
#pragma unroll
    for (int d = 0; d < D; ++d) kf[x][d] = *(const u32x4*)(kh + (mt * D + d) * 512);
  };
#pragma unroll
  for (int x = 0; x < HW; ++x) {
#pragma unroll
    for (int d = 0; d < D; ++d) qf[x][d] = *(const u32x4*)(qrow + min(HW * wave + x, H - 1) * dp + 32 * d);
    keys(x, 0);
  }
#pragma unroll
  for (int k = 0; k < HP / LH; ++k) {
    const int h = tid / LH, g = tid % LH + LH * k;
    const float w = a.mix[min(h, H - 1) * H + min(g, H - 1)] * a.slope[min(g, H - 1)];
    slope_in += h < H && g < H ? w : 0.f;
  }
  PHASE();
  f32x4 acc[HW][2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int x = 0; x < HW; ++x) {
      acc[x][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < D; ++d) acc[x][mt] = mfma(kf[x][d], qf[x][d], acc[x][mt]);
      if (mt == 0) keys(x, 1);
      PHASE();
    }
#pragma unroll
  for (int o = LH / 2; o > 0; o >>= 1) slope_in += __shfl_xor(slope_in, o, 64);
  if (tid % LH == 0) mss[tid / LH] = slope_in * kLog2e;
  bf16x8 tf[HB];
#pragma unroll
  for (int mt = 0; mt < HB; ++mt)
#pragma unroll
    for (int j = 0; j < 8; ++j) tf[mt][j] = (16 * mt + n < H && (HB == 2 ? 8 * q + j : 4 * q + j) < H && (HB == 2 || j < 4)) ? (short)f2bf(tm[mt][j]) : (short)0;
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      Op high, low;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const float x = acc[2 * w][mt][e], y = acc[2 * w + 1][mt][e];
        high[w] = pack_bf16x2(x, y);
        low[w] = pack_bf16x2(x - lo_bf(high[w]), y - hi_bf(high[w]));
      }
      const int key = 16 * mt + 4 * q + e;
      b_lds[key][0][wave][n] = high;
      b_lds[key][1][wave][n] = low;
    }
  __syncthreads();
  // keys 8 wave ..: heads 16 mt + 4 q + r of query n
  const float scale = a.scale * kLog2e;
  const int qpos = t0 + n, qfirst = a.chunk > 0 ? qpos / a.chunk * a.chunk : 0;
  float ms[HB][4];
#pragma unroll
  for (int mt = 0; mt < HB; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) ms[mt][r] = mss[16 * mt + 4 * q + r];
  float* out = a.part + pairs_at(talk_slot(row0, seq, tile), 0, kb, H, blocks) + (wave * 16 + n) * 4;
#pragma unroll
  for (int kg = 0; kg < 2; ++kg) {
    f32x4 st[4][HB];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int part = 1; part >= 0; --part) {  // low parts, then high parts on top
        const Op b = b_lds[8 * wave + 4 * kg + k][part][q][n];
#pragma unroll
        for (int mt = 0; mt < HB; ++mt) {
          const f32x4 z = part ? f32x4{0.f, 0.f, 0.f, 0.f} : st[k][mt];
          if constexpr (HB == 2) {
            st[k][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(md_bf16x8v, tf[mt]), __builtin_bit_cast(md_bf16x8v, b), z, 0, 0, 0);
          } else {
            const bf16x4 t = {tf[mt][0], tf[mt][1], tf[mt][2], tf[mt][3]};
            st[k][mt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(t, __builtin_bit_cast(bf16x4, b), z, 0, 0, 0);
          }
        }
      }
#pragma unroll
    for (int mt = 0; mt < HB; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int h = 16 * mt + 4 * q + r;
        f32x4 o;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int j = j0 + 8 * wave + 4 * kg + k;
          o[k] = j > qpos || j < qfirst ? -INFINITY : st[k][mt][r] * scale - ms[mt][r] * (float)(qpos - j);
        }
        if (h < H) *(f32x4*)(out + (int64_t)h * blocks * 512 + kg * 256) = o;
      }
  }
}

template <int NW, int C>
__global__ __launch_bounds__(64 * NW) void attn_pairs_out_kernel(const LmAttn a, int blocks) {
  constexpr int vp = 32 * C, NB = PAIRS_BLOCKS;
  __shared__ __attribute__((aligned(16))) float o_lds[NW][16][vp + 4], m_lds[NW][16], l_lds[NW][16];
  const int H = a.heads, G = a.kv_heads, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, q = lane >> 4;
  const int h = blockIdx.x;
  int tile;
  const int seq = pairs_seq(a.r, blockIdx.y, tile);
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, pos0 = a.r.seq_pos0[seq], slot = a.r.seq_slot[seq];
  const int t0 = (pos0 / 16 + tile) * 16, lo = max(t0, pos0), hi = min(t0 + 15, pos0 + len - 1);
  if (lo > hi) return;
  const int kfirst = (a.chunk > 0 ? lo / a.chunk * a.chunk : 0) & ~31, nkb = (hi - kfirst) / 32 + 1;
  const float* in = a.part + pairs_at(talk_slot(row0, seq, tile), h, 0, H, blocks) + 4 * lane;
  const bf16_t* Vb = (const bf16_t*)a.v + (int64_t)slot * G * a.ctx * vp + key_block(kfirst, h / (H / G), G, vp) + 8 * lane;
  const int64_t vstep = (int64_t)G * 32 * vp;
  f32x4 s[NB][2];  // keys 8 q + 4 i .. of query n
  u32x4 vf[NB][2 * C];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int kb = wave + NW * b;
    s[b][0] = s[b][1] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if (kb >= nkb) continue;
#pragma unroll
    for (int i = 0; i < 2; ++i) s[b][i] = *(const f32x4*)(in + (int64_t)kb * 512 + i * 256);
#pragma unroll
    for (int t = 0; t < 2 * C; ++t) vf[b][t] = *(const u32x4*)(Vb + kb * vstep + t * 512);
  }
  float m = -INFINITY;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) m = fmaxf(m, fmaxf(s[b][0][e], s[b][1][e]));
  m = fmaxf(m, __shfl_xor(m, 16, 64));
  m = fmaxf(m, __shfl_xor(m, 32, 64));
  const float ref = m == -INFINITY ? 0.f : m;
  f32x4 o[2 * C];
#pragma unroll
  for (int t = 0; t < 2 * C; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float l = 0.f;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (wave + NW * b >= nkb) continue;
    u32x4 p;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float p0 = __builtin_amdgcn_exp2f(s[b][i][2 * e] - ref), p1 = __builtin_amdgcn_exp2f(s[b][i][2 * e + 1] - ref);
        l += p0 + p1;
        p[2 * i + e] = pack_bf16x2(p0, p1);
      }
#pragma unroll
    for (int t = 0; t < 2 * C; ++t) o[t] = mfma(p, vf[b][t], o[t]);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (q == 0) {
    m_lds[wave][n] = m;
    l_lds[wave][n] = l;
  }
#pragma unroll
  for (int t = 0; t < 2 * C; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) o_lds[wave][4 * q + r][16 * t + n] = o[t][r];
  __syncthreads();
  for (int at = tid; at < 16 * vp / 8; at += 64 * NW) {  // eight coordinates of a query
    const int row = at / (vp / 8), e0 = at % (vp / 8) * 8, pos = t0 + row;
    if (pos < lo || pos > hi) continue;
    float M = -INFINITY, L = 0.f, v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, m_lds[w][row]);
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = __builtin_amdgcn_exp2f(m_lds[w][row] - M);
      L += f * l_lds[w][row];
      const f32x4 x = *(const f32x4*)(&o_lds[w][row][e0]), y = *(const f32x4*)(&o_lds[w][row][e0 + 4]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] += f * x[e];
        v[4 + e] += f * y[e];
      }
    }
    const float inv = 1.0f / L;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] *= inv;
    store8((bf16_t*)a.out + (int64_t)(row0 + pos - pos0) * a.ldo + in_chunks(h * vp + e0, a.out_chunk), v);
  }
}

constexpr int64_t PAIRS_FLOATS = 40 << 20;  // most scores of a step
// Slots, and half as many sequences at most, are a grid's height.  A slot has two blocks of a head's scores at least (pairs_blocks), which bounds them
static_assert(PAIRS_FLOATS / (2 * 512) * 3 / 2 <= 65535, "grid height");
int64_t pairs_floats(int n_rows, int n_seq, int span, int H) { return (int64_t)(n_rows / 16 + 2 * n_seq) * H * std::min(pairs_blocks(span), PAIRS_MOST) * 512; }
bool pairs_form(int H, int dp, int vp) { return H <= 32 && dp <= 128 && vp <= 128 && (H <= 16 || dp <= 64); }

template <int HB>
TalkKernelBlocks pairs_scores_pick(int dp) {
  if (dp == 32) return attn_pairs_scores_kernel<HB, 1>;
  if constexpr (HB == 1)  // (pairs_form: more than 16 heads up to 64 wide)
    if (dp > 64) return dp == 96 ? attn_pairs_scores_kernel<1, 3> : attn_pairs_scores_kernel<1, 4>;
  return attn_pairs_scores_kernel<HB, 2>;
}
template <int NW>
TalkKernelBlocks pairs_out_pick(int vp) {
  switch (vp / 32) {
    case 1: return attn_pairs_out_kernel<NW, 1>;
    case 2: return attn_pairs_out_kernel<NW, 2>;
    case 3: return attn_pairs_out_kernel<NW, 3>;
    default: return attn_pairs_out_kernel<NW, 4>;
  }
}

}  // namespace

size_t lm_attn_pairs_floats_most(int n_rows, int n_seq, int span, int H, int dp, int vp) {
  return pairs_form(H, dp, vp) ? (size_t)std::min(PAIRS_FLOATS, pairs_floats(n_rows, n_seq, span, H)) : 0;
}
// ... and of 60 million scores (keys wider than 64: 40) with the heads that fill up the products' 16 or 32, which cost as much: 12 layers, 8 x 940 tokens, 4 heads of 64 2.42 -> 2.58 ms against
// attn_mfma_kernel, of 128 2.76 -> 3.35, one head of 128 2.56 -> 2.90; 24 x 300, 4 of 128 2.18 -> 2.27; but 4 x 940, 4 of 64 1.70 -> 1.52.  All heads at 30 blocks at most, 914 keys: one prompt of 800 / 950 tokens, 32
// heads of 64 on 8 of keys 1.33 -> 1.19 / 1.38 -> 1.41, 32 of 32 1.11 -> 1.01 / 1.20 -> 1.28; 20 of 64 still 1.29 -> 1.22.
bool lm_attn_pairs_takes(const LmAttn& a, int span) {
  if (!pairs_form(a.heads, a.dp, a.vp) || pairs_blocks(span) > (a.heads > 24 ? 30 : PAIRS_MOST)) return false;
  auto floats = [&](int heads) { return pairs_floats(a.r.n_rows, a.r.n_seq, span, heads); };
  return floats(a.heads) <= PAIRS_FLOATS && floats(a.heads <= 16 ? 16 : 32) <= (a.dp > 64 ? 40 << 20 : 60 << 20);
}
md_status lm_attn_pairs(const LmAttn& a, int span, hipStream_t s) {
  if (!lm_attn_pairs_takes(a, span)) return MD_ERR_UNSUPPORTED;
  MD_TRY(prep<bf16_t>(a, false, s));
  const int blocks = pairs_blocks(span), slots = pairs_slots(a.r);
  const auto scores = a.heads <= 16 ? pairs_scores_pick<1>(a.dp) : pairs_scores_pick<2>(a.dp);
  const auto out = blocks <= 2 * PAIRS_BLOCKS ? pairs_out_pick<2>(a.vp) : blocks <= 4 * PAIRS_BLOCKS ? pairs_out_pick<4>(a.vp) : pairs_out_pick<8>(a.vp);
  const int waves = blocks <= 2 * PAIRS_BLOCKS ? 2 : blocks <= 4 * PAIRS_BLOCKS ? 4 : 8;
  hipLaunchKernelGGL(scores, dim3(blocks, slots + a.r.n_seq), dim3(256), 0, s, a, blocks);
  MD_TRY(md_launch_status());
  hipLaunchKernelGGL(out, dim3(a.heads, slots), dim3(64 * waves), 0, s, a, blocks);
  return md_launch_status();
}

// ---------------------------------------------------------------------------------------------------------------------------
namespace {

constexpr int NWD = 8;  // waves of a decode workgroup

struct DecodeLds {
  int q, raw, p, mix, stat, total;
};
__host__ __device__ inline DecodeLds decode_lds(int H, int dp, int tk) {
  const int hs = (H + 3) / 4 * 4;
  DecodeLds l;
  l.q = 0;
  l.raw = l.q + H * dp * 2;
  l.p = l.raw + H * tk * 4;
  l.mix = l.p + hs * tk * 4;
  l.stat = l.mix + H * hs * 4;
  l.total = l.stat + 4 * hs * 4;
  return l;
}

// grid (splits, sequences).  Split s covers the keys base + s * split_keys ..., base = the chunk's first key rounded down to a block;
// queries and the row's own key and value are attn_prep_kernel's.  HPW: output heads per wave, D: dp / 32, C: vp / 32, TK: keys per tile.
// Waves read many blocks before they use the first (no branch between loads): keys of a whole tile row by groups of heads, values of one
// head at a time; blocks past the last key are read (finite spare positions) and masked.
// Few keys: what counts is the chain of dependent loads.  Splits of one block of 32 keys (up to 63 sequences in a graph) have tiles of their own: TK = 32 deals
// the key heads to four pairs of waves and requests everything a wave reads, keys and values, before the queries are staged; the mixture's sum
// over heads is shared by the halves of a wave.  32 heads of 64 (which attn_heads_* take since), one sequence at 100 keys: 11.8 us against 13.9 in tiles of 64, which read a block of
// values beyond the split, one key head batch after the other, and waited for each of what is staged (with the waits 13.0: a step of the 24-layer model 1104 us against 1120, with 16 heads of 128 1093
// against 1119, 24 sequences at 1500 keys 2454 against 2529).
template <int HPW, int D, int C, int TK>
__global__ __launch_bounds__(64 * NWD, 2) void attn_decode_kernel(const LmAttn a) {
  extern __shared__ __attribute__((aligned(16))) char dsm[];
  const int H = a.heads, G = a.kv_heads, rep = H / G, dp = 32 * D, vp = 32 * C, hs = (H + 3) / 4 * 4;
  const DecodeLds L = decode_lds(H, dp, TK);
  bf16_t* qs = (bf16_t*)(dsm + L.q);
  float *raw = (float*)(dsm + L.raw), *ps = (float*)(dsm + L.p), *mixT = (float*)(dsm + L.mix);
  float *ms = (float*)(dsm + L.stat), *ls = ms + hs, *al = ls + hs, *sl = al + hs;
  const int split = blockIdx.x, seq = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n16 = lane & 15, q4 = lane >> 4;
  const int row = a.r.seq_row0[seq], i = a.r.seq_pos0[seq], slot = a.r.seq_slot[seq];
  const int first = a.chunk > 0 ? i / a.chunk * a.chunk : 0;
  const int k0 = (first & ~31) + split * a.split_keys, k1 = min(k0 + a.split_keys - 1, i);
  float* part = a.part + ((int64_t)seq * a.n_split + split) * (H * vp + 2 * H);
  if (k0 > i) {  // nothing to see for this split
    for (int h = tid; h < H; h += 64 * NWD) {
      part[H * vp + 2 * h] = -INFINITY;
      part[H * vp + 2 * h + 1] = 0.f;
    }
    return;
  }
  const bf16_t* Kb = (const bf16_t*)a.k + (int64_t)slot * G * a.ctx * dp;
  const bf16_t* Vb = (const bf16_t*)a.v + (int64_t)slot * G * a.ctx * vp;
  float acc[HPW][2 * C];  // heads wave, wave + NWD, ..: coordinate 16 t + n16, the keys of this lane row
#pragma unroll
  for (int u = 0; u < HPW; ++u)
#pragma unroll
    for (int t = 0; t < 2 * C; ++t) acc[u][t] = 0.f;

  constexpr int KW = TK / 16, PARTS = NWD / KW;  // waves of a tile's keys, and of its key heads
  const int kwave = wave % KW, heads_each = (G + PARTS - 1) / PARTS, g_lo = wave / KW * heads_each, g_hi = min(G, g_lo + heads_each);
  constexpr bool AHEAD = TK == 32;  // values of all heads of the wave requested behind the first keys
  constexpr int UG = D >= 3 ? 2 : 4, NB = TK / 32, VB = AHEAD && HPW * C <= 8 ? HPW : 2;
  // queries, the mixture (transposed, heads padded to a multiple of four) and slopes: the first round's loads go out before the keys', without a wait between
  constexpr int MIX = 2, T = 64 * NWD;
  auto mix_at = [&](int e) { return min(e % hs, H - 1) * H + min(e / hs, H - 1); };
  const u32x4 q_in = *(const u32x4*)((const bf16_t*)a.q + (int64_t)row * H * dp + min(tid * 8, H * dp - 8));
  float mix_in[MIX], slope_in = a.slope[min(tid, H - 1)];
#pragma unroll
  for (int k = 0; k < MIX; ++k) mix_in[k] = a.mix[mix_at(tid + T * k)];
  __builtin_amdgcn_sched_barrier(0);
  auto stage = [&] {
    if (tid * 8 < H * dp) *(u32x4*)(qs + tid * 8) = q_in;
    for (int c = (tid + T) * 8; c < H * dp; c += T * 8) *(u32x4*)(qs + c) = *(const u32x4*)((const bf16_t*)a.q + (int64_t)row * H * dp + c);
#pragma unroll
    for (int k = 0; k < MIX; ++k)
      if (tid + T * k < H * hs) mixT[tid + T * k] = (tid + T * k) % hs < H ? mix_in[k] : 0.f;
    for (int e = tid + T * MIX; e < H * hs; e += T) mixT[e] = e % hs < H ? a.mix[mix_at(e)] : 0.f;
    if (tid < hs) {  // (at most 64 heads)
      ms[tid] = -INFINITY;
      ls[tid] = 0.f;
      sl[tid] = tid < H ? slope_in : 0.f;
    }
    __syncthreads();
  };
  if (!AHEAD) stage();
  for (int j0 = k0; j0 <= k1; j0 += TK) {  // (AHEAD: once)
    const int n = min(TK, k1 + 1 - j0);
    // scores of keys 16 kwave .. 16 kwave + 15, this wave's key heads, 16 query heads of one key head per matrix product
    const bf16_t* kw = Kb + key_block(j0 + 16 * kwave, 0, G, dp) + (kwave & 1) * (D * 512) + 8 * lane;
    const float dist = (float)(i - (j0 + 16 * kwave + 4 * q4));
    bf16x8 kf[2][UG][D];
    auto load = [&](int buf, int g0) {
#pragma unroll
      for (int u = 0; u < UG; ++u)
#pragma unroll
        for (int d = 0; d < D; ++d) kf[buf][u][d] = *(const bf16x8*)(kw + min(g0 + u, G - 1) * (32 * dp) + 512 * d);
    };
    auto scores = [&](int buf, int g0) {
#pragma unroll
      for (int u = 0; u < UG; ++u) {
        if (g0 + u >= g_hi) continue;
        const int g = g0 + u;
        for (int r0 = 0; r0 < rep; r0 += 16) {
          const int h = g * rep + min(r0 + n16, rep - 1);
          f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int d = 0; d < D; ++d)
            s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(md_bf16x8v, kf[buf][u][d]),
                                                        __builtin_bit_cast(md_bf16x8v, *(const bf16x8*)(qs + h * dp + 32 * d + 8 * q4)), s, 0, 0, 0);
          if (r0 + n16 < rep) {
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = s[e] * a.scale - sl[h] * (dist - (float)e);
            *(f32x4*)(raw + h * TK + 16 * kwave + 4 * q4) = o;
          }
        }
      }
    };
    u32x4 vf[VB][NB][2 * C];
    auto load_v = [&](int u) {
      const bf16_t* vh = Vb + key_block(j0, min(wave + NWD * u, H - 1) / rep, G, vp) + 8 * lane;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int t = 0; t < 2 * C; ++t) vf[u % VB][b][t] = *(const u32x4*)(vh + (int64_t)b * G * (32 * vp) + t * 512);
    };
    if (AHEAD) {
      load(0, g_lo);
      if (g_lo + UG < g_hi) load(1, g_lo + UG);
#pragma unroll
      for (int u = 0; u < VB; ++u) load_v(u);
      __builtin_amdgcn_sched_barrier(0);
      stage();
      for (int g0 = g_lo; g0 < g_hi; g0 += 2 * UG) {
        scores(0, g0);
        if (g0 + 2 * UG < g_hi) load(0, g0 + 2 * UG);
        scores(1, g0 + UG);
        if (g0 + 3 * UG < g_hi) load(1, g0 + 3 * UG);
      }
    } else {
      if (16 * kwave < n && g_lo < g_hi) {
        load(0, g_lo);
        for (int g0 = g_lo; g0 < g_hi; g0 += 2 * UG) {
          load(1, g0 + UG);
          scores(0, g0);
          load(0, g0 + 2 * UG);  // (past the last head: clamped, unused)
          scores(1, g0 + UG);
        }
      }
      load_v(0);  // under the mixture and the softmax
    }
    __syncthreads();
    for (int h0 = 4 * wave; h0 < H; h0 += 4 * NWD) {
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
      const int key = lane % TK, half = (H + 1) / 2, m_lo = TK == 32 ? (lane >> 5) * half : 0, m_n = TK == 32 ? half : H;
#pragma unroll 8
      for (int k = 0; k < m_n; ++k) {
        const int g = m_lo + k;
        if (TK == 64 || g < H) s += *(const f32x4*)(mixT + g * hs + h0) * raw[g * TK + key];
      }
      if (TK == 32)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += __shfl_xor(s[e], 32, 64);
      if (key >= n || j0 + key < first) s = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      const f32x4 mo = *(const f32x4*)(ms + h0);
      f32x4 mn = s, p, sum;
#pragma unroll
      for (int o = TK / 2; o > 0; o >>= 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) mn[e] = fmaxf(mn[e], __shfl_xor(mn[e], o, 64));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        mn[e] = fmaxf(mn[e], mo[e]);
        p[e] = sum[e] = expf(s[e] - mn[e]);
        ps[(h0 + e) * TK + key] = p[e];
      }
#pragma unroll
      for (int o = TK / 2; o > 0; o >>= 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] += __shfl_xor(sum[e], o, 64);
      if (lane == 0) {
        f32x4 f;
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = expf(mo[e] - mn[e]);
        *(f32x4*)(ls + h0) = *(const f32x4*)(ls + h0) * f + sum;
        *(f32x4*)(al + h0) = f;
        *(f32x4*)(ms + h0) = mn;
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < HPW; ++u) {
      if (VB == 2 ? u + 1 < HPW && (u > 0 || !AHEAD) : false) load_v(u + 1);
      const int h = min(wave + NWD * u, H - 1);
      const float f = al[h];
#pragma unroll
      for (int t = 0; t < 2 * C; ++t) acc[u][t] *= f;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const f32x4 p0 = *(const f32x4*)(ps + h * TK + 32 * b + 8 * q4), p1 = *(const f32x4*)(ps + h * TK + 32 * b + 8 * q4 + 4);
#pragma unroll
        for (int t = 0; t < 2 * C; ++t) {
          const u32x4 v = vf[u % VB][b][t];
          acc[u][t] += p0[0] * lo_bf(v[0]) + p0[1] * hi_bf(v[0]) + p0[2] * lo_bf(v[1]) + p0[3] * hi_bf(v[1]) + p1[0] * lo_bf(v[2]) +
                       p1[1] * hi_bf(v[2]) + p1[2] * lo_bf(v[3]) + p1[3] * hi_bf(v[3]);
        }
      }
    }
    if (AHEAD) break;
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < HPW; ++u) {
    const int h = wave + NWD * u;
    if (h >= H) continue;
    const float inv = 1.0f / ls[h];
#pragma unroll
    for (int t = 0; t < 2 * C; ++t) {
      float o = acc[u][t];
      o += __shfl_xor(o, 16, 64);
      o += __shfl_xor(o, 32, 64);
      if (q4 != 0) continue;
      if (a.n_split == 1) ((bf16_t*)a.out)[(int64_t)row * a.ldo + in_chunks(h * vp + 16 * t + n16, a.out_chunk)] = f2bf(o * inv);
      else part[h * vp + 16 * t + n16] = o;
    }
  }
  if (a.n_split > 1)
    for (int h = tid; h < H; h += 64 * NWD) {
      part[H * vp + 2 * h] = ms[h];
      part[H * vp + 2 * h + 1] = ls[h];
    }
}

// grid (heads, sequences).  Few sequences: a chain of loads again, so a split's maximum and sum are read once and together, and the sums four splits
// at a time up to the last that saw a key (n_split is what the longest sequence would need; up to 1024).
__global__ __launch_bounds__(256) void attn_combine_kernel(const LmAttn a) {
  __shared__ float ws[1024], sums[256], red[4], red_last[4];
  const int h = blockIdx.x, seq = blockIdx.y, tid = threadIdx.x, w = a.heads * a.vp, n = a.n_split;
  const int64_t stride = w + 2 * a.heads;
  const float* p = a.part + (int64_t)seq * n * stride;
  constexpr int R = 4;
  md_f32x2 ml[R];
#pragma unroll
  for (int j = 0; j < R; ++j) ml[j] = *(const md_f32x2*)(p + min(tid + 256 * j, n - 1) * stride + w + 2 * h);
  float m = -INFINITY, last = -1.f;
#pragma unroll
  for (int j = 0; j < R; ++j)
    if (tid + 256 * j < n) {
      m = fmaxf(m, ml[j][0]);
      if (ml[j][1] != 0.f) last = (float)(tid + 256 * j);
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    m = fmaxf(m, __shfl_xor(m, o, 64));
    last = fmaxf(last, __shfl_xor(last, o, 64));
  }
  if ((tid & 63) == 0) {
    red[tid >> 6] = m;
    red_last[tid >> 6] = last;
  }
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const int live = 1 + (int)fmaxf(fmaxf(red_last[0], red_last[1]), fmaxf(red_last[2], red_last[3]));
  float l = 0.f;
#pragma unroll
  for (int j = 0; j < R; ++j)
    if (tid + 256 * j < n) {
      const float ls = ml[j][1], f = ls == 0.f ? 0.f : expf(ml[j][0] - m);
      ws[tid + 256 * j] = f;
      l += ls * f;
    }
  __syncthreads();  // (red is read above and written below)
  l = block_sum_256(l, red);
  const int groups = 256 / a.vp, e = tid % a.vp, g = tid / a.vp;
  float o = 0.f;
  if (g < groups)
    for (int s0 = g; s0 < live; s0 += groups * R) {
      float v[R];
#pragma unroll
      for (int j = 0; j < R; ++j) v[j] = p[min(s0 + groups * j, live - 1) * stride + h * a.vp + e];
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int s = s0 + groups * j;
        if (s < live && ws[s] != 0.f) o += ws[s] * v[j];  // an empty split wrote no sums
      }
    }
  sums[tid] = o;
  __syncthreads();
  if (tid >= a.vp) return;
  for (int k = 1; k < groups; ++k) o += sums[k * a.vp + e];
  ((bf16_t*)a.out)[(int64_t)a.r.seq_row0[seq] * a.ldo + in_chunks(h * a.vp + e, a.out_chunk)] = f2bf(o / l);
}

}  // namespace

int lm_attn_decode_splits(int n_seq, int span, int* split_keys) {
  const int blocks = (span + 31 + 31) / 32;  // of 32 keys; the first may begin before the chunk
  int splits = (4096 + n_seq - 1) / n_seq;   // many rounds of workgroups: how many of them see keys depends on the positions
  splits = splits > 1024 ? 1024 : splits;
  splits = splits > blocks ? blocks : splits;
  const int per = (blocks + splits - 1) / splits;
  *split_keys = per * 32;
  return (blocks + per - 1) / per;
}
size_t lm_attn_decode_part_floats(int n_seq, int n_split, int heads, int vp) { return n_split > 1 ? (size_t)n_seq * n_split * (heads * vp + 2 * heads) : 0; }

namespace {
template <int TK, int D, int C>
TalkKernel decode_by_heads(int heads) {
  return heads <= 8 ? attn_decode_kernel<1, D, C, TK> : heads <= 16 ? attn_decode_kernel<2, D, C, TK> : heads <= 32 ? attn_decode_kernel<4, D, C, TK>
         : heads <= 64 && D * C <= 4 ? attn_decode_kernel<8, D, C, TK> : nullptr;
}
template <int TK, int D>
TalkKernel decode_by_width(const LmAttn& a) {
  switch (a.vp / 32) {
    case 1: return decode_by_heads<TK, D, 1>(a.heads);
    case 2: return decode_by_heads<TK, D, 2>(a.heads);
    case 3: return decode_by_heads<TK, D, 3>(a.heads);
    case 4: return decode_by_heads<TK, D, 4>(a.heads);
    default: return nullptr;
  }
}
template <int TK>
TalkKernel decode_by_dim(const LmAttn& a) {
  switch (a.dp / 32) {
    case 1: return decode_by_width<TK, 1>(a);
    case 2: return decode_by_width<TK, 2>(a);
    case 3: return decode_by_width<TK, 3>(a);
    case 4: return decode_by_width<TK, 4>(a);
    default: return nullptr;
  }
}
TalkKernel decode_pick(const LmAttn& a, int tk) {
  if (decode_lds(a.heads, a.dp, 64).total > 160 * 1024) return nullptr;
  return tk == 32 ? decode_by_dim<32>(a) : decode_by_dim<64>(a);
}
}  // namespace

bool lm_attn_decode_takes(const LmAttn& a) { return decode_pick(a, 64) != nullptr; }
md_status lm_attn_decode(const LmAttn& a, hipStream_t s) {
  const int tk = a.split_keys == 32 ? 32 : 64;
  const TalkKernel fn = decode_pick(a, tk);
  if (!fn) return MD_ERR_UNSUPPORTED;
  MD_TRY(md_ensure_dynamic_lds((const void*)fn, 160 * 1024));
  MD_TRY(lm_attn_prep(MD_DTYPE_BF16, a, s));
  hipLaunchKernelGGL(fn, dim3(a.n_split, a.r.n_seq), dim3(64 * NWD), decode_lds(a.heads, a.dp, tk).total, s, a);
  MD_TRY(md_launch_status());
  if (a.n_split == 1) return MD_OK;
  hipLaunchKernelGGL(attn_combine_kernel, dim3(a.heads, a.r.n_seq), dim3(256), 0, s, a);
  return md_launch_status();
}

// ---------------------------------------------------------------------------------------------------------------------------
// A decode step in two launches instead of three, where a layer's own keys and values have one head per query head.  Few sequences are bound by chains of dependent
// loads in a few workgroups, so all that can be is done beside another chain, and heads as well as keys go to different workgroups.
//   attn_heads_scores_kernel  (256 columns of heads, 128 keys, sequence): convolution of its queries, their scores with the cached keys, heads unmixed; the
//                             workgroup of the new position also makes its key, its value (-> cache) and the convolution state.  The norms' factors are taken out of
//                             the products: every workgroup leaves the sums of squares of its columns
//   attn_heads_mix_kernel     (head, 256 keys, sequence): mixture, softmax, weighted values; the last of a head's workgroups adds up their parts
// The score of a head and key is one float, so the mixture's all-to-all costs 4 bytes, read by every head, beside the 4 dim of keys and values, read
// once.  How many keys there are is known on the device only (a captured step sees any number): workgroups beyond the last key leave at once.
// 32 heads of 64, one sequence at 100 keys: 6.6 and 5.8 us a layer against 5.1, 11.9 and 4.7; a step of two such layers and two of retention, before and now: 1 / 8
// sequences at 100 keys 217 / 232 -> 200 / 217 us, 8 at 1500 269 -> 250, 32 at 100 / 500 / 1500 286 / 367 / 508 -> 274 / 314 / 420, 64 at 500 / 1500 642 / 706 -> 494 / 696, 128
// at 20 / 1500 528 / 1131 -> 523 / 1090; 16 heads of 128 within 1 % of the same.
namespace {

constexpr int HEADS_COLS = 256, HEADS_KEYS = 128, HEADS_SPAN = 256;

struct HeadsPart {  // places in a.part, in floats
  int keys;       // room for the keys of a sequence
  int64_t raw, khat, sq, part, ticket, total;
};
__host__ __device__ inline HeadsPart heads_part(int n_seq, int span, int H, int dp, int vp) {
  HeadsPart f;
  const int splits = (span + 31 + HEADS_SPAN - 1) / HEADS_SPAN, groups = H * dp / HEADS_COLS;
  f.keys = splits * HEADS_SPAN;
  f.raw = 0;
  f.khat = f.raw + (int64_t)n_seq * H * f.keys;
  f.sq = f.khat + (int64_t)n_seq * H * dp;
  f.part = f.sq + (int64_t)n_seq * 2 * groups;
  f.ticket = f.part + (int64_t)n_seq * H * splits * (vp + 2);
  f.total = f.ticket + (int64_t)n_seq * H;
  return f;
}

template <int D>
__global__ __launch_bounds__(256) void attn_heads_scores_kernel(const LmAttn a, const HeadsPart f) {
  constexpr int dp = 32 * D, HG = HEADS_COLS / dp, TILES = HEADS_KEYS / 16 / 4;  // heads of a workgroup, key tiles of a wave
  __shared__ __attribute__((aligned(16))) bf16_t qs[HEADS_COLS];
  __shared__ float ks[HEADS_COLS], red[4];
  const int H = a.heads, groups = H / HG, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n16 = lane & 15, q4 = lane >> 4;
  const int seq = blockIdx.y, group = blockIdx.x % groups, split = blockIdx.x / groups;
  const int row = a.r.seq_row0[seq], i = a.r.seq_pos0[seq], slot = a.r.seq_slot[seq];
  const int base = (a.chunk > 0 ? i / a.chunk * a.chunk : 0) & ~31, k0 = base + split * HEADS_KEYS;
  if (k0 > i) return;
  const bool own = i < k0 + HEADS_KEYS;  // the new position's workgroup

  // column c of a projection, convolved: the newest taps are requested together (rows before the sequence's first are read from somewhere else and not used)
  const int c = group * HEADS_COLS + tid;
  constexpr int TAPS = 4;
  struct Column {
    bf16_t u[TAPS];
    float w[TAPS], norm;
  };
  const bf16_t* ring = (const bf16_t*)a.conv_state + (int64_t)slot * a.taps * a.conv_ld;
  auto request = [&](int col0, const float* norm) {
    Column x;
    const int col = col0 + c;
    const bf16_t* proj = (const bf16_t*)a.proj + (int64_t)row * a.ldp + col;
#pragma unroll
    for (int k = 0; k < TAPS; ++k) {
      const bool in = k < a.taps && i - k >= 0;
      x.u[k] = *(k > 0 && in ? ring + (int64_t)((i - k) % a.taps) * a.conv_ld + col : proj);
      x.w[k] = a.conv[(int64_t)(in ? a.taps - 1 - k : 0) * a.conv_ld + col];
    }
    x.norm = norm ? norm[c] : 1.f;
    return x;
  };
  auto convolve = [&](const Column& x) {
    float y = 0.f;
#pragma unroll
    for (int k = TAPS - 1; k >= 0; --k)
      if (k < a.taps && i - k >= 0) y += x.w[k] * bf2f(x.u[k]);
    return y;
  };
  Column q = request(a.col_q, a.q_norm), kx, vx;
  if (own) {
    kx = request(a.col_k, a.k_norm);
    vx = request(a.col_v, nullptr);
  }
  const bf16_t* Kb = (const bf16_t*)a.k + (int64_t)slot * H * a.ctx * dp;
  u32x4 kf[TILES][HG][D];
#pragma unroll
  for (int t = 0; t < TILES; ++t) {
    const int j = k0 + 16 * (wave + 4 * t);
    if (j > i) continue;
    const bf16_t* kw = Kb + key_block(j, group * HG, H, dp) + ((j >> 4) & 1) * (D * 512) + 8 * lane;
#pragma unroll
    for (int h = 0; h < HG; ++h)
#pragma unroll
      for (int d = 0; d < D; ++d) kf[t][h][d] = *(const u32x4*)(kw + h * (32 * dp) + 512 * d);
  }
  __builtin_amdgcn_sched_barrier(0);

  const float y = convolve(q);
  qs[tid] = f2bf(y * q.norm);
  float* sq = a.part + f.sq + (int64_t)seq * 2 * groups + group;
  if (own) {
    const float k = convolve(kx), v = convolve(vx);
    const float qq = block_sum_256(y * y, red), kk = block_sum_256(k * k, red);
    if (tid == 0) {
      sq[0] = qq;
      sq[groups] = kk;
    }
    ks[tid] = k * kx.norm;
    a.part[f.khat + (int64_t)seq * H * dp + c] = k * kx.norm;
    float r = 1.0f;
    if (a.value_norm) {
      float s = v * v;
#pragma unroll
      for (int o = (dp < 64 ? dp : 64) / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
      if (dp == 128) {
        __syncthreads();
        if (lane == 0) red[wave] = s;
        __syncthreads();
        s = red[wave] + red[wave ^ 1];
      }
      r = 1.0f / sqrtf(s / (float)a.vdim + a.eps);
    }
    const int g = c / dp, e = c % dp;
    ((bf16_t*)a.v)[(int64_t)slot * a.ctx * H * dp + value_index(i, g, e, H, dp)] = f2bf(v * r);
    if (a.taps > 1) {
      bf16_t* to = (bf16_t*)a.conv_state + ((int64_t)slot * a.taps + i % a.taps) * a.conv_ld + c;
      to[a.col_q] = q.u[0];
      to[a.col_k] = kx.u[0];
      to[a.col_v] = vx.u[0];
    }
    if (tid < HG) ((unsigned*)(a.part + f.ticket))[seq * H + group * HG + tid] = 0u;
  }
  __syncthreads();
  float* raw = a.part + f.raw + ((int64_t)seq * H + group * HG) * f.keys + (k0 - base);  // [head][key]
#pragma unroll
  for (int t = 0; t < TILES; ++t) {
    const int at = 16 * (wave + 4 * t);
    if (k0 + at > i) continue;
    f32x4 mine = {0.f, 0.f, 0.f, 0.f};  // lane n16 keeps head n16's (the product's columns are all the same query)
#pragma unroll
    for (int h = 0; h < HG; ++h) {
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < D; ++d) s = mfma(kf[t][h][d], *(const u32x4*)(qs + h * dp + 32 * d + 8 * q4), s);
      if (n16 == h) mine = s;
    }
    if (n16 >= HG) continue;
    float* to = raw + (int64_t)n16 * f.keys + at + 4 * q4;
    const int left = i - (k0 + at + 4 * q4);  // keys of these four before the new one
    if (left >= 4) {
      *(f32x4*)to = mine * a.scale;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e < left) to[e] = mine[e] * a.scale;
    }
  }
  if (!own) return;
  for (int h = wave; h < HG; h += 4) {  // the new key's scores
    float s = 0.f;
    for (int d = lane; d < dp; d += 64) s += bf2f(qs[h * dp + d]) * ks[h * dp + d];
    s = wave_sum(s);
    if (lane == 0) raw[(int64_t)h * f.keys + i - k0] = s * a.scale;
  }
}

template <int C>
__global__ __launch_bounds__(256) void attn_heads_mix_kernel(const LmAttn a, const HeadsPart f) {
  constexpr int vp = 32 * C, BLOCKS = HEADS_SPAN / 32 / 4;  // blocks of 32 keys of a wave
  __shared__ __attribute__((aligned(16))) float ps[HEADS_SPAN], sums[4][vp], red[4];
  __shared__ unsigned order;
  const int H = a.heads, dp = vp, groups = H * dp / HEADS_COLS, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n16 = lane & 15,
            q4 = lane >> 4;
  const int seq = blockIdx.y, h = blockIdx.x % H, split = blockIdx.x / H;
  const int row = a.r.seq_row0[seq], i = a.r.seq_pos0[seq], slot = a.r.seq_slot[seq];
  const int first = a.chunk > 0 ? i / a.chunk * a.chunk : 0, base = first & ~31, k0 = base + split * HEADS_SPAN;
  if (k0 > i) return;
  const int live = (i - base) / HEADS_SPAN + 1;
  const bf16_t* Vb = (const bf16_t*)a.v + (int64_t)slot * H * a.ctx * vp;
  const float* sq = a.part + f.sq + (int64_t)seq * 2 * groups;
  const float qq_in = lane < groups ? sq[lane] : 0.f, kk_in = lane < groups ? sq[groups + lane] : 0.f;
  const float slope_in = lane < H ? a.mix[h * H + lane] * a.slope[lane] : 0.f;
  const float* raw = a.part + f.raw + (int64_t)seq * H * f.keys + split * HEADS_SPAN + tid;
  const float* mix = a.mix + h * H;
  float s = 0.f;
  u32x4 vf[BLOCKS][2 * C];
  constexpr int AT_ONCE = 32;
  float x[AT_ONCE];
#pragma unroll
  for (int g = 0; g < AT_ONCE; ++g) x[g] = raw[(int64_t)min(g, H - 1) * f.keys];  // (keys beyond the last: whatever is there, masked)
#pragma unroll
  for (int b = 0; b < BLOCKS; ++b) {
    const int j = k0 + 32 * (wave + 4 * b);
    const bf16_t* vh = Vb + key_block(min(j, i), h, H, vp) + 8 * lane;
#pragma unroll
    for (int t = 0; t < 2 * C; ++t) vf[b][t] = *(const u32x4*)(vh + t * 512);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int g = 0; g < AT_ONCE; ++g)
    if (g < H) s += mix[g] * x[g];
  for (int g = AT_ONCE; g < H; ++g) s += mix[g] * raw[(int64_t)g * f.keys];
  const float qq = wave_sum(qq_in), kk = wave_sum(kk_in), slope = wave_sum(slope_in);
  const float rq = 1.0f / sqrtf(qq / (float)(H * a.dim) + a.eps), rk = 1.0f / sqrtf(kk / (float)(H * a.dim) + a.eps);
  const int j = k0 + tid;
  s = s * (j == i ? rq * rk : rq) - slope * (float)(i - j);
  if (j > i || j < first) s = -INFINITY;
  float m = wave_max(s);
  if (lane == 0) red[wave] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float p = expf(s - m);
  ps[tid] = p;
  const float l = block_sum_256(p, red);  // (its barriers also publish ps)
  float acc[2 * C];
#pragma unroll
  for (int t = 0; t < 2 * C; ++t) acc[t] = 0.f;
#pragma unroll
  for (int b = 0; b < BLOCKS; ++b) {
    const int at = 32 * (wave + 4 * b);
    if (k0 + at > i) continue;
    const f32x4 p0 = *(const f32x4*)(ps + at + 8 * q4), p1 = *(const f32x4*)(ps + at + 8 * q4 + 4);
#pragma unroll
    for (int t = 0; t < 2 * C; ++t) {
      const u32x4 v = vf[b][t];
      acc[t] += p0[0] * lo_bf(v[0]) + p0[1] * hi_bf(v[0]) + p0[2] * lo_bf(v[1]) + p0[3] * hi_bf(v[1]) + p1[0] * lo_bf(v[2]) + p1[1] * hi_bf(v[2]) +
                p1[2] * lo_bf(v[3]) + p1[3] * hi_bf(v[3]);
    }
  }
#pragma unroll
  for (int t = 0; t < 2 * C; ++t) {
    acc[t] += __shfl_xor(acc[t], 16, 64);
    acc[t] += __shfl_xor(acc[t], 32, 64);
    if (q4 == 0) sums[wave][16 * t + n16] = acc[t];
  }
  __syncthreads();
  if (i < k0 + HEADS_SPAN && tid < dp)  // the new key, with its norm's factor
    ((bf16_t*)a.k)[(int64_t)slot * a.ctx * H * dp + key_index(i, h, tid, H, dp)] = f2bf(a.part[f.khat + (int64_t)seq * H * dp + h * dp + tid] * rk);
  float o = 0.f;
  if (tid < vp) o = (sums[0][tid] + sums[1][tid]) + (sums[2][tid] + sums[3][tid]);
  bf16_t* out = (bf16_t*)a.out + (int64_t)row * a.ldo;
  if (live == 1) {
    if (tid < vp) out[in_chunks(h * vp + tid, a.out_chunk)] = f2bf(o / l);
    return;
  }
  // several parts: stores and loads past the private L2s, the last to arrive adds up
  auto leave = [](float* to, float v) { __hip_atomic_store(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  auto fetch = [](const float* from) { return __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  const int splits = f.keys / HEADS_SPAN;
  float* part = a.part + f.part + ((int64_t)seq * H + h) * splits * (vp + 2);
  if (tid < vp) leave(part + split * (vp + 2) + tid, o);
  if (tid == 0) {
    leave(part + split * (vp + 2) + vp, m);
    leave(part + split * (vp + 2) + vp + 1, l);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) order = __hip_atomic_fetch_add((unsigned*)(a.part + f.ticket) + seq * H + h, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (order != (unsigned)live - 1 || tid >= vp) return;
  float M = -INFINITY, L = 0.f, O = 0.f;
  for (int k = 0; k < live; ++k) M = fmaxf(M, fetch(part + k * (vp + 2) + vp));
#pragma unroll 4
  for (int k = 0; k < live; ++k) {
    const float w = expf(fetch(part + k * (vp + 2) + vp) - M);
    L += w * fetch(part + k * (vp + 2) + vp + 1);
    O += w * fetch(part + k * (vp + 2) + tid);
  }
  out[in_chunks(h * vp + tid, a.out_chunk)] = f2bf(O / L);
}

// (heads that divide 256 columns)
bool heads_takes(int H, int G, int dp, int vp, int taps, bool own_kv) {
  return own_kv && H == G && dp == vp && (dp == 32 || dp == 64 || dp == 128) && H * dp % HEADS_COLS == 0 && H <= 64 && taps <= 4;
}

}  // namespace

size_t lm_attn_heads_floats(int n_seq, int span, int H, int G, int dp, int vp, int taps, bool own_kv) {
  return heads_takes(H, G, dp, vp, taps, own_kv) ? (size_t)heads_part(n_seq, span, H, dp, vp).total : 0;
}
// Where the three launches of attn_decode_kernel are the better ones (steps of attention layers alone, ms, three launches / two).  Its workgroups read a head's scores from LDS, these from memory, H times for
// every key, which counts against the 4 dim of keys and values from H = dim on: 64 heads of 64, 40 sequences at 200 / 500 / 1000 keys 0.90 / 0.73, 1.20 / 1.19, 1.79 / 1.97, 24 at 500 / 1000
// 0.86 / 0.80, 1.18 / 1.25; 64 of 32, where the others are slower, 40 at 1500 1.91 / 1.79, 64 2.78 / 2.90; 32 of 32, 24 / 64 at 1000 0.477 / 0.477, 0.87 / 0.89.  The fewest keys of more than
// 40 sequences: 64 of 64 at 30 0.72 / 0.79, 48 of 64 0.635 / 0.587.  One or two groups of columns, from where parts of a head are added up: 24 layers of 4 of 64, one sequence at 200 / 500 /
// 1500 0.501 / 0.503, 0.508 / 0.546, 0.54 / 0.60, 40 at 500 0.78 / 0.75; 16 of 32, 24 / 40 at 1500 0.96 / 1.04, 1.23 / 1.32; but 4 of 128, 8 at 1000 0.69 / 0.66.  Twelve layers: 16 of 32, 64 / 128 at
// 1800 1.03 / 1.10, 1.66 / 1.85, where 4 of 64 take 0.93 / 0.75, 1.30 / 1.10; 48 of 64, 128 at 800 / 1000 / 1800 4.96 / 4.73, 4.73 / 5.29, 7.73 / 9.05, 64 at 1800 5.13 / 4.80; 40 of 64, 128 at 1800
// 6.90 / 6.96.  A second workgroup for a few keys of each of many heads: 64 of 32, 20 at 220 / 300 / 420 0.67 / 0.59, 0.69 / 0.75, 0.96 / 0.78; 64 of 64, 40 at 300 1.36 / 1.44.
bool lm_attn_heads_takes(const LmAttn& a, int span) {
  if (!heads_takes(a.heads, a.kv_heads, a.dp, a.vp, a.taps, a.own_kv)) return false;
  const int64_t H = a.heads, dp = a.dp, n_seq = a.r.n_seq;
  const bool scores = (H >= dp && n_seq * span * dp * dp > 20480 * H * H) || (4 * H >= 3 * dp && n_seq * span > 120000);
  const bool many = H > 48 && (n_seq > 40 || (n_seq >= 16 && span > HEADS_SPAN && 2 * span <= 3 * HEADS_SPAN));
  const bool few = H * dp <= 512 && span > HEADS_SPAN && (dp == 32 || (dp == 64 && n_seq <= 20));
  return !(scores || many || few) || !lm_attn_decode_takes(a);
}
md_status lm_attn_heads(const LmAttn& a, int span, hipStream_t s) {
  if (!heads_takes(a.heads, a.kv_heads, a.dp, a.vp, a.taps, a.own_kv)) return MD_ERR_UNSUPPORTED;
  const HeadsPart f = heads_part(a.r.n_seq, span, a.heads, a.dp, a.vp);
  const int groups = a.heads * a.dp / HEADS_COLS;
  auto scores = a.dp == 32 ? attn_heads_scores_kernel<1> : a.dp == 64 ? attn_heads_scores_kernel<2> : attn_heads_scores_kernel<4>;
  auto mix = a.dp == 32 ? attn_heads_mix_kernel<1> : a.dp == 64 ? attn_heads_mix_kernel<2> : attn_heads_mix_kernel<4>;
  hipLaunchKernelGGL(scores, dim3(groups * ((span + 31 + HEADS_KEYS - 1) / HEADS_KEYS), a.r.n_seq), dim3(256), 0, s, a, f);
  MD_TRY(md_launch_status());
  hipLaunchKernelGGL(mix, dim3(a.heads * (f.keys / HEADS_SPAN), a.r.n_seq), dim3(256), 0, s, a, f);
  return md_launch_status();
}
