// Retention: linear attention with a fixed decay per head, S <- decay S + k v^T, o = S^T q, with rotated q and k.
//
// The state of a head is kept transposed, fp32 [vdim][dim].
//
// Plain kernels (any dtype, fp32 on the vector ALUs): rotation, token-by-token recurrence, output norm and gate.
//
// bf16 prefill on the matrix cores, in chunks of 64 tokens:
//   ret_increment_kernel  per (sequence, head, chunk): what the chunk adds to the state, sum_t decay^(n-1-t) v_t k_t^T
//   ret_states_kernel     running over the chunks: the state at the start of each, and the slot's state at the end
//   ret_chunk_kernel      per (sequence, head, chunk): decay^(t+1) S^T q_t + sum_{s<=t} decay^(t-s) (q_t . k_s) v_s, output norm, gate
// Everything behind the projections counts as fp32: rotated q and k, decay-weighted products and states enter a product as the sum of
// two bf16 (16 mantissa bits; hi hi + hi lo + lo hi), the values are the projection's own bf16.
//
// bf16 decode step: ret_decode_kernel, one workgroup per (sequence, head): rotation, state update, output, norm and gate in one launch.
#include "lm_internal.hpp"

namespace {

// element d of a head's rotated row: the first rot_dims coordinates turn in pairs (d, d + rot_dims / 2)
template <typename T>
__device__ __forceinline__ float rotated(const T* h, int d, int rot_dims, const float* cs) {
  const int half = rot_dims >> 1;
  if (d >= rot_dims) return ldf(h + d);
  const int i = d < half ? d : d - half;
  const float c = cs[2 * i], sn = cs[2 * i + 1];
  return d < half ? ldf(h + d) * c - ldf(h + d + half) * sn : ldf(h + d) * c + ldf(h + d - half) * sn;
}

template <typename T>
__global__ __launch_bounds__(256) void ret_rotate_kernel(const LmRet a) {
  const int row = blockIdx.x, n = a.heads * a.dp;
  const float* cs = a.rope + (int64_t)a.r.row_pos[row] * a.rot_dims;  // [rot_dims / 2][2]
  const T* q = (const T*)a.proj + (int64_t)row * a.ldp + a.col_q;
  const T* k = (const T*)a.proj + (int64_t)row * a.ldp + a.col_k;
  for (int c = threadIdx.x; c < n; c += 256) {
    const int h = c / a.dp, d = c - h * a.dp;
    a.qf[(int64_t)row * n + c] = rotated(q + h * a.dp, d, a.rot_dims, cs);
    a.kf[(int64_t)row * n + c] = rotated(k + h * a.dp, d, a.rot_dims, cs) * a.scale;
  }
}

// grid (n_seq, heads, vp / 16): 16 columns of the state, 16 neighbouring lanes per column, each owning every 16th row of it.  Tokens are
// staged 16 at a time and then run without a barrier: the recurrence is a chain, what counts is what lies on it (two sequences of 190 tokens,
// 16 heads of 128: 35 us; 235 us with three barriers per token).  An output is summed down a lane's rows, then over the lanes in turn: a first
// token's result hangs on the order where q . k is small (gemm_f32.hip).
// Q: quads of state rows per lane, dp <= 64 Q
constexpr int PLAIN_TOKENS = 16;
template <typename T, int Q>
__global__ __launch_bounds__(256) void ret_scan_kernel(const LmRet a) {
  constexpr int R = 4 * Q, LD = R + 4;  // rows per lane, their stride: [token][lane][row]
  __shared__ __attribute__((aligned(16))) float qs[PLAIN_TOKENS][16 * LD], ks[PLAIN_TOKENS][16 * LD];
  __shared__ float vs[PLAIN_TOKENS][16], os[PLAIN_TOKENS][16][17];
  const int seq = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, l = tid & 15, col = tid >> 4, e0 = blockIdx.z * 16, e = e0 + col;
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, pos0 = a.r.seq_pos0[seq];
  const int dp = a.dp, vp = a.vp, H = a.heads;
  float* st = a.state + (((int64_t)a.r.seq_slot[seq] * H + h) * vp + e) * dp;
  const float decay = a.decay[h];
  float S[R];
#pragma unroll
  for (int i = 0; i < R; ++i) S[i] = (pos0 > 0 && 16 * i < dp) ? st[16 * i + l] : 0.f;
  if (dp < 64 * Q)  // rows behind the head's: zeros, which add nothing
    for (int i = tid; i < PLAIN_TOKENS * 16 * LD; i += 256) (&qs[0][0])[i] = (&ks[0][0])[i] = 0.f;
  f32x4 qn[Q], kn[Q];  // the next tokens', under way during these
  float vn = 0.f;
  const int quads = dp / 4;
  auto load = [&](int t0) {
    const int n = min(PLAIN_TOKENS, len - t0);
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      const int i = tid + 256 * j, t = i / quads;
      if (t >= n) continue;
      const int64_t at = ((int64_t)(row0 + t0 + t) * H + h) * dp + (i - t * quads) * 4;
      qn[j] = *(const f32x4*)(a.qf + at);
      kn[j] = *(const f32x4*)(a.kf + at);
    }
    if (col < n) vn = ldf((const T*)a.proj + (int64_t)(row0 + t0 + col) * a.ldp + a.col_v + h * vp + e0 + l);
  };
  load(0);
  for (int t0 = 0; t0 < len; t0 += PLAIN_TOKENS) {
    const int n = min(PLAIN_TOKENS, len - t0);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      const int i = tid + 256 * j, t = i / quads, d = (i - t * quads) * 4;
      if (t >= n) continue;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        qs[t][((d & 15) + k) * LD + (d >> 4)] = qn[j][k];
        ks[t][((d & 15) + k) * LD + (d >> 4)] = kn[j][k];
      }
    }
    if (col < n) vs[col][l] = vn;
    __syncthreads();
    if (t0 + PLAIN_TOKENS < len) load(t0 + PLAIN_TOKENS);
#pragma unroll 4
    for (int t = 0; t < n; ++t) {
      const float v = vs[t][col];
      float o = 0.f;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const f32x4 kq = *(const f32x4*)(ks[t] + l * LD + 4 * q), qq = *(const f32x4*)(qs[t] + l * LD + 4 * q);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          S[4 * q + k] = __builtin_fmaf(decay, S[4 * q + k], kq[k] * v);
          o = __builtin_fmaf(S[4 * q + k], qq[k], o);
        }
      }
      os[t][col][l] = o;
    }
    __syncthreads();
    if (col < n) {  // this thread's token col, column l
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) sum += os[col][l][i];
      a.of[((int64_t)(row0 + t0 + col) * H + h) * vp + e0 + l] = sum;
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i)
    if (16 * i < dp) st[16 * i + l] = S[i];
}

template <typename T>
__global__ __launch_bounds__(256) void ret_out_kernel(const LmRet a) {
  const int row = blockIdx.x, lane = threadIdx.x & 63;
  for (int h = threadIdx.x >> 6; h < a.heads; h += 4) {
    const float* o = a.of + ((int64_t)row * a.heads + h) * a.vp;
    float ss = 0.f;
    for (int d = lane; d < a.vp; d += 64) ss += o[d] * o[d];
    const float r = 1.0f / sqrtf(wave_sum(ss) / (float)a.vdim + a.eps);
    const T* g = (const T*)a.proj + (int64_t)row * a.ldp + a.col_g + h * a.vp;
    T* dst = (T*)a.out + (int64_t)row * a.ldo;
    for (int d = lane; d < a.vp; d += 64) stf(dst + in_chunks(h * a.vp + d, a.out_chunk), o[d] * r * silu_f32(ldf(g + d)));
  }
}

template <typename T>
md_status plain(const LmRet& a, hipStream_t s) {
  if (a.dp > 256) return MD_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(ret_rotate_kernel<T>, dim3(a.r.n_rows), dim3(256), 0, s, a);
  MD_TRY(md_launch_status());
  auto scan = a.dp <= 64 ? ret_scan_kernel<T, 1> : a.dp <= 128 ? ret_scan_kernel<T, 2> : a.dp <= 192 ? ret_scan_kernel<T, 3> : ret_scan_kernel<T, 4>;
  hipLaunchKernelGGL(scan, dim3(a.r.n_seq, a.heads, a.vp / 16), dim3(256), 0, s, a);
  MD_TRY(md_launch_status());
  hipLaunchKernelGGL(ret_out_kernel<T>, dim3(a.r.n_rows), dim3(256), 0, s, a);
  return md_launch_status();
}

}  // namespace

md_status lm_ret_plain(int dtype, const LmRet& a, hipStream_t s) { return dtype == MD_DTYPE_F32 ? plain<float>(a, s) : plain<bf16_t>(a, s); }

namespace {

// eight consecutive elements (d0 a multiple of 8) of a head's rotated row
__device__ __forceinline__ void rotated8(const bf16_t* h, int d0, int rot_dims, const float* cs, float (&o)[8]) {
  const u32x4 own = *(const u32x4*)(h + d0);
  const int half = rot_dims >> 1;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = (e & 1) ? hi_bf(own[e >> 1]) : lo_bf(own[e >> 1]);
  if (d0 >= rot_dims) return;
  if ((half & 7) == 0) {
    const bool low = d0 < half;
    const u32x4 other = *(const u32x4*)(h + (low ? d0 + half : d0 - half));
    const float* c = cs + 2 * (low ? d0 : d0 - half);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float p = (e & 1) ? hi_bf(other[e >> 1]) : lo_bf(other[e >> 1]);
      const float sn = c[2 * e + 1];
      o[e] = o[e] * c[2 * e] + (low ? -p : p) * sn;
    }
  } else {
    for (int e = 0; e < 8; ++e) o[e] = rotated(h, d0 + e, rot_dims, cs);
  }
}

__device__ __forceinline__ float pow_int(float log2_decay, int n) { return n == 0 ? 1.0f : __builtin_amdgcn_exp2f(log2_decay * (float)n); }

__device__ __forceinline__ void split8(const float (&v)[8], u32x4& hi, u32x4& lo) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    hi[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
    lo[i] = pack_bf16x2(v[2 * i] - lo_bf(hi[i]), v[2 * i + 1] - hi_bf(hi[i]));
  }
}
__device__ __forceinline__ md_bf16x8v as_op(const u32x4& v) { return __builtin_bit_cast(md_bf16x8v, v); }
__device__ __forceinline__ f32x4 mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_op(a), as_op(b), c, 0, 0, 0);
}

constexpr int RC = LM_RET_CHUNK;

// grid (chunks, heads, sequences)
__global__ __launch_bounds__(256) void ret_increment_kernel(const LmRet a) {
  extern __shared__ __attribute__((aligned(16))) bf16_t rsm[];
  constexpr int TS = RC + 8;
  const int c = blockIdx.x, h = blockIdx.y, seq = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, dp = a.dp, vp = a.vp;
  const int n = min(RC, len - c * RC);
  if (n <= 0) return;
  bf16_t *Kh = rsm, *Kl = Kh + dp * TS, *Vt = Kl + dp * TS;  // [d][t], [d][t], [e][t]
  const float ld = log2f(a.decay[h]);
  const bf16_t* base = (const bf16_t*)a.proj + (int64_t)(row0 + c * RC) * a.ldp;
  for (int i = tid; i < RC * (dp >> 3); i += 256) {
    const int t = i & (RC - 1), d0 = (i / RC) * 8;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (t < n) {
      const int pos = a.r.seq_pos0[seq] + c * RC + t;
      rotated8(base + (int64_t)t * a.ldp + a.col_k + h * dp, d0, a.rot_dims, a.rope + (int64_t)pos * a.rot_dims, v);
      const float w = a.scale * pow_int(ld, n - 1 - t);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] *= w;
    }
    u32x4 hi, lo;
    split8(v, hi, lo);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      Kh[(d0 + e) * TS + t] = (bf16_t)(hi[e >> 1] >> (16 * (e & 1)));
      Kl[(d0 + e) * TS + t] = (bf16_t)(lo[e >> 1] >> (16 * (e & 1)));
    }
  }
  for (int i = tid; i < RC * (vp >> 3); i += 256) {
    const int t = i & (RC - 1), e0 = (i / RC) * 8;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (t < n) v = *(const u32x4*)(base + (int64_t)t * a.ldp + a.col_v + h * vp + e0);
#pragma unroll
    for (int e = 0; e < 8; ++e) Vt[(e0 + e) * TS + t] = (bf16_t)(v[e >> 1] >> (16 * (e & 1)));
  }
  __syncthreads();
  float* dst = a.chunk_state + (((int64_t)seq * a.n_chunk_max + c) * a.heads + h) * vp * dp;
  const int r = lane & 15, q = lane >> 4, nd = dp >> 4, tiles = (vp >> 4) * nd;
  for (int tile = wave; tile < tiles; tile += 4) {
    const int te = tile / nd, td = tile - te * nd;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < RC; s += 32) {
      const u32x4 v = *(const u32x4*)(Vt + (16 * te + r) * TS + s + 8 * q);
      acc = mfma(v, *(const u32x4*)(Kh + (16 * td + r) * TS + s + 8 * q), acc);
      acc = mfma(v, *(const u32x4*)(Kl + (16 * td + r) * TS + s + 8 * q), acc);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) dst[(int64_t)(16 * te + 4 * q + e) * dp + 16 * td + r] = acc[e];
  }
}

// grid (heads * vp * dp / 2048, sequences): a thread owns eight consecutive state elements.  In: the chunks' increments; out, in their
// place: the state at the start of each chunk as [8 bf16 high parts | 8 bf16 low parts].
__global__ __launch_bounds__(256) void ret_states_kernel(const LmRet a) {
  const int seq = blockIdx.y, per_head = a.vp * a.dp;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8, n_el = (int64_t)a.heads * per_head;
  if (i >= n_el) return;
  const int h = (int)(i / per_head), len = a.r.seq_row0[seq + 1] - a.r.seq_row0[seq], nc = (len + RC - 1) / RC;
  const float ld = log2f(a.decay[h]), full = pow_int(ld, RC);
  float* st = a.state + (int64_t)a.r.seq_slot[seq] * n_el + i;
  float* p = a.chunk_state + (int64_t)seq * a.n_chunk_max * n_el + i;
  float S[8];
  const bool cont = a.r.seq_pos0[seq] > 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) S[e] = cont ? st[e] : 0.f;
  constexpr int U = 4;  // chunks in flight
  for (int c0 = 0; c0 < nc; c0 += U) {
    f32x4 inc[U][2];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c0 + u < nc) {
        inc[u][0] = *(const f32x4*)(p + (c0 + u) * n_el);
        inc[u][1] = *(const f32x4*)(p + (c0 + u) * n_el + 4);
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c0 + u < nc) {
        u32x4 hi, lo;
        split8(S, hi, lo);
        *(u32x4*)(p + (c0 + u) * n_el) = hi;
        *(u32x4*)(p + (c0 + u) * n_el + 4) = lo;
        const int n = min(RC, len - (c0 + u) * RC);
        const float f = n == RC ? full : pow_int(ld, n);
#pragma unroll
        for (int e = 0; e < 8; ++e) S[e] = f * S[e] + inc[u][e >> 2][e & 3];
      }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) st[e] = S[e];
}

// grid (chunks, heads, sequences), four waves of 16 tokens.  D: dp / 32, C: vp / 32; column n of output tile t is coordinate 2 C n + t.
template <int D, int C>
__global__ __launch_bounds__(256) void ret_chunk_kernel(const LmRet a) {
  constexpr int dp = 32 * D, vp = 32 * C, KS = dp + 8, VS = RC + 4;
  __shared__ __attribute__((aligned(16))) bf16_t Kh[RC * KS], Kl[RC * KS], Vt[vp * VS];
  const int c = blockIdx.x, h = blockIdx.y, seq = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, q = lane >> 4;
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0;
  const int n = min(RC, len - c * RC);
  if (n <= 0) return;
  const int p0 = a.r.seq_pos0[seq] + c * RC;
  const float ld = log2f(a.decay[h]);
  const bf16_t* base = (const bf16_t*)a.proj + (int64_t)(row0 + c * RC) * a.ldp;
  for (int i = tid; i < RC * (dp >> 3); i += 256) {
    const int t = i / (dp >> 3), d0 = (i - t * (dp >> 3)) * 8;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (t < n) {
      rotated8(base + (int64_t)t * a.ldp + a.col_k + h * dp, d0, a.rot_dims, a.rope + (int64_t)(p0 + t) * a.rot_dims, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] *= a.scale;
    }
    u32x4 hi, lo;
    split8(v, hi, lo);
    *(u32x4*)(Kh + t * KS + d0) = hi;
    *(u32x4*)(Kl + t * KS + d0) = lo;
  }
  for (int i = tid; i < RC * (vp >> 3); i += 256) {
    const int t = i & (RC - 1), e0 = (i / RC) * 8;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (t < n) v = *(const u32x4*)(base + (int64_t)t * a.ldp + a.col_v + h * vp + e0);
#pragma unroll
    for (int e = 0; e < 8; ++e) Vt[(e0 + e) * VS + t] = (bf16_t)(v[e >> 1] >> (16 * (e & 1)));
  }
  const int t = 16 * wave + r, tq = min(t, n - 1);  // this lane's query (rows past the chunk's end replay its last one)
  u32x4 qh[D], ql[D];
#pragma unroll
  for (int s = 0; s < D; ++s) {
    float v[8];
    rotated8(base + (int64_t)tq * a.ldp + a.col_q + h * dp, 32 * s + 8 * q, a.rot_dims, a.rope + (int64_t)(p0 + tq) * a.rot_dims, v);
    split8(v, qh[s], ql[s]);
  }
  __syncthreads();
  if (16 * wave >= n) return;
  f32x4 o[2 * C];
#pragma unroll
  for (int i = 0; i < 2 * C; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (p0 > 0) {
    const float* S = a.chunk_state + (((int64_t)seq * a.n_chunk_max + c) * a.heads + h) * vp * dp;
#pragma unroll
    for (int s = 0; s < D; ++s)
#pragma unroll
      for (int i = 0; i < 2 * C; ++i) {
        const float* sp = S + (2 * C * r + i) * dp + 32 * s + 8 * q;
        const u32x4 sh = *(const u32x4*)sp, sl = *(const u32x4*)(sp + 4);
        o[i] = mfma(qh[s], sh, o[i]);
        o[i] = mfma(qh[s], sl, o[i]);
        o[i] = mfma(ql[s], sh, o[i]);
      }
    f32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = pow_int(ld, 16 * wave + 4 * q + e + 1);
#pragma unroll
    for (int i = 0; i < 2 * C; ++i) o[i] *= w;
  }
#pragma unroll
  for (int b = 0; b < RC / 32; ++b) {
    if (2 * b > wave) continue;
    float p[8];  // token slots (block 2 b, 4 q + j) and (block 2 b + 1, 4 q + j) of the products' contraction
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int sb = 2 * b + half;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      if (sb <= wave) {
#pragma unroll
        for (int s = 0; s < D; ++s) {
          const u32x4 kh = *(const u32x4*)(Kh + (16 * sb + r) * KS + 32 * s + 8 * q), kl = *(const u32x4*)(Kl + (16 * sb + r) * KS + 32 * s + 8 * q);
          acc = mfma(kh, qh[s], acc);
          acc = mfma(kh, ql[s], acc);
          acc = mfma(kl, qh[s], acc);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = t - (16 * sb + 4 * q + e);
        p[4 * half + e] = (sb <= wave && d >= 0) ? acc[e] * pow_int(ld, d) : 0.f;
      }
    }
    u32x4 ph, pl;
    split8(p, ph, pl);
#pragma unroll
    for (int i = 0; i < 2 * C; ++i) {
      const bf16_t* vr = Vt + (2 * C * r + i) * VS + 32 * b + 4 * q;
      const u32x2 v0 = *(const u32x2*)vr, v1 = *(const u32x2*)(vr + 16);
      const u32x4 v = {v0[0], v0[1], v1[0], v1[1]};
      o[i] = mfma(ph, v, o[i]);
      o[i] = mfma(pl, v, o[i]);
    }
  }
  f32x4 ss = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 2 * C; ++i) ss += o[i] * o[i];
#pragma unroll
  for (int m = 1; m < 16; m <<= 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) ss[e] += __shfl_xor(ss[e], m, 64);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int tt = 16 * wave + 4 * q + e;
    if (tt >= n) continue;
    const float rn = 1.0f / sqrtf(ss[e] / (float)a.vdim + a.eps);
    const bf16_t* g = base + (int64_t)tt * a.ldp + a.col_g + h * vp + 2 * C * r;
    bf16_t* dst = (bf16_t*)a.out + (int64_t)(row0 + c * RC + tt) * a.ldo;
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const uint32_t gg = *(const uint32_t*)(g + 2 * i);
      *(uint32_t*)(dst + in_chunks(h * vp + 2 * C * r + 2 * i, a.out_chunk)) = pack_bf16x2(o[2 * i][e] * rn * silu_f32(lo_bf(gg)), o[2 * i + 1][e] * rn * silu_f32(hi_bf(gg)));
    }
  }
}

typedef void (*RetKernel)(const LmRet);
template <int D>
RetKernel ret_chunk_by_width(int c) {
  switch (c) {
    case 1: return ret_chunk_kernel<D, 1>;
    case 2: return ret_chunk_kernel<D, 2>;
    case 3: return ret_chunk_kernel<D, 3>;
    case 4: return ret_chunk_kernel<D, 4>;
    default: return nullptr;
  }
}
RetKernel ret_chunk_pick(const LmRet& a) {
  switch (a.dp / 32) {
    case 1: return ret_chunk_by_width<1>(a.vp / 32);
    case 2: return ret_chunk_by_width<2>(a.vp / 32);
    case 3: return ret_chunk_by_width<3>(a.vp / 32);
    case 4: return ret_chunk_by_width<4>(a.vp / 32);
    default: return nullptr;
  }
}

// grid (heads, sequences).  Sixteen lanes per state row, sixteen rows at a time, R rows of up to 64 E columns per thread.  Few sequences: the chain of loads
// bounds it, and all of a head's rows are under way before the first use (ALL).  8 sequences, 16 heads of 128: 17.1 us with a row loaded after the other,
// 9.6 this way; 1 sequence, 32 heads of 64: 6.7 and 5.7; 64 of 32 x 64: 16.7 and 14.9.  Many: the state's bytes, and more workgroups per CU hide more than
// registers full of rows (128 sequences, 8 heads of 256: 122 us with all, 104 with a row after the other; 16 of 192: 141 and 114).
template <int R, int E, bool ALL>
__global__ __launch_bounds__(256) void ret_decode_kernel(const LmRet a) {
  __shared__ __attribute__((aligned(16))) float qs[256], ks[256], os[256];
  __shared__ float red[4];
  const int h = blockIdx.x, seq = blockIdx.y, tid = threadIdx.x, l = tid & 15, e0 = tid >> 4;
  const int row = a.r.seq_row0[seq], pos = a.r.seq_pos0[seq], dp = a.dp, vp = a.vp;
  float* st = a.state + ((int64_t)a.r.seq_slot[seq] * a.heads + h) * vp * dp;
  const bf16_t* p = (const bf16_t*)a.proj + (int64_t)row * a.ldp;
  f32x4 S[R][E];
  float v[R];
  auto load = [&](int e1) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int e = e1 + e0 + 16 * i;
#pragma unroll
      for (int j = 0; j < E; ++j) {
        S[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (pos > 0 && e < vp && 4 * l + 64 * j < dp) S[i][j] = *(const f32x4*)(st + (int64_t)e * dp + 4 * l + 64 * j);
      }
      v[i] = bf2f(p[a.col_v + h * vp + min(e, vp - 1)]);
    }
  };
  load(0);
  const float gate = bf2f(p[a.col_g + h * vp + min(tid, vp - 1)]), decay = a.decay[h];
  const float* cs = a.rope + (int64_t)pos * a.rot_dims;
  for (int d = tid; d < dp; d += 256) {
    qs[d] = rotated(p + a.col_q + h * dp, d, a.rot_dims, cs);
    ks[d] = rotated(p + a.col_k + h * dp, d, a.rot_dims, cs) * a.scale;
  }
  __syncthreads();
  for (int e1 = 0; e1 < vp; e1 += 16 * R) {
    if (e1 > 0) load(e1);  // (ALL: once)
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int e = e1 + e0 + 16 * i;
      if (e >= vp) break;
      float o = 0.f;
#pragma unroll
      for (int j = 0; j < E; ++j) {
        const int d = 4 * l + 64 * j;
        if (d >= dp) continue;
        const f32x4 k = *(const f32x4*)(ks + d), qv = *(const f32x4*)(qs + d);
        const f32x4 s = decay * S[i][j] + k * v[i];
        *(f32x4*)(st + (int64_t)e * dp + d) = s;
        o += s[0] * qv[0] + s[1] * qv[1] + s[2] * qv[2] + s[3] * qv[3];
      }
#pragma unroll
      for (int m = 1; m < 16; m <<= 1) o += __shfl_xor(o, m, 64);
      if (l == 0) os[e] = o;
    }
    if (ALL) break;
  }
  __syncthreads();
  const float o = tid < vp ? os[tid] : 0.f;
  const float ss = block_sum_256(o * o, red);
  if (tid < vp) ((bf16_t*)a.out)[(int64_t)row * a.ldo + in_chunks(h * vp + tid, a.out_chunk)] = f2bf(o / sqrtf(ss / (float)a.vdim + a.eps) * silu_f32(gate));
}
template <int R, bool ALL>
RetKernel ret_decode_by_width(int dp) {
  return dp <= 64 ? ret_decode_kernel<R, 1, ALL> : dp <= 128 ? ret_decode_kernel<R, 2, ALL> : ret_decode_kernel<R, 4, ALL>;
}
// All rows at once as long as every workgroup's registers are on the chip at the same time, two rows after the other beyond.  A step of four layers of retention and
// little else, all / two: 8 heads of 256, 32 sequences 187 / 220 us, 64 400 / 377; 16 of 128, 64 sequences 241 / 252, 96 354 / 338; 32 of 64, 64
// sequences 188 / 188, 128 297 / 283; 16 of 192, 32 sequences 242 / 223.
RetKernel ret_decode_pick(const LmRet& a) {
  const int rows = a.vp <= 32 ? 2 : a.vp <= 64 ? 4 : a.vp <= 128 ? 8 : 16, columns = a.dp <= 64 ? 1 : a.dp <= 128 ? 2 : 4, workgroups = a.heads * a.r.n_seq;
  if (workgroups > 2048 || workgroups * rows * columns > 256 * 64) return ret_decode_by_width<2, false>(a.dp);
  return rows == 2 ? ret_decode_by_width<2, true>(a.dp) : rows == 4 ? ret_decode_by_width<4, true>(a.dp) : rows == 8 ? ret_decode_by_width<8, true>(a.dp) : ret_decode_by_width<16, true>(a.dp);
}

}  // namespace

bool lm_ret_mfma_takes(const LmRet& a) { return ret_chunk_pick(a) != nullptr; }
md_status lm_ret_mfma(const LmRet& a, hipStream_t s) {
  const RetKernel fn = ret_chunk_pick(a);
  if (!fn) return MD_ERR_UNSUPPORTED;
  const dim3 grid(a.n_chunk_max, a.heads, a.r.n_seq);
  const int lds = (2 * a.dp + a.vp) * (RC + 8) * 2;
  hipLaunchKernelGGL(ret_increment_kernel, grid, dim3(256), lds, s, a);
  MD_TRY(md_launch_status());
  hipLaunchKernelGGL(ret_states_kernel, dim3((a.heads * a.vp * a.dp + 2047) / 2048, a.r.n_seq), dim3(256), 0, s, a);
  MD_TRY(md_launch_status());
  hipLaunchKernelGGL(fn, grid, dim3(256), 0, s, a);
  return md_launch_status();
}

bool lm_ret_decode_takes(const LmRet& a) { return a.dp <= 256 && a.vp <= 256; }
md_status lm_ret_decode(const LmRet& a, hipStream_t s) {
  hipLaunchKernelGGL(ret_decode_pick(a), dim3(a.heads, a.r.n_seq), dim3(256), 0, s, a);
  return md_launch_status();
}
