// Retention: linear attention with a fixed decay per head, S <- decay S + k v^T, o = S^T q, with rotated q and k.
//
// The state of a head is kept transposed, fp32 [vdim][dim].
//
// Plain kernels (any dtype, fp32 on the vector ALUs): rotation, token-by-token recurrence, output norm and gate.
//
// bf16 prefill on the matrix cores, in chunks of 64 tokens, the chunks of a segment one after the other with the state in registers:
//   ret_run_kernel        per (sequence, head, segment): decay^(t+1) S^T q_t + sum_{s<=t} decay^(t-s) (q_t . k_s) v_s, output norm, gate, and the chunk's
//                         sum_t decay^(n-1-t) v_t k_t^T onto the state
//   ret_increment_kernel, ret_segments_kernel  where more segments than one fill the chip: what the chunks add to the state, and the states that segments start from
// Everything behind the projections counts as fp32: rotated q and k, decay-weighted products and states enter a product as the sum of
// two bf16 (16 mantissa bits; hi hi + hi lo + lo hi), the values are the projection's own bf16.
//
// bf16 decode step: ret_decode_kernel, one workgroup per (sequence, head): rotation, state update, output, norm and gate in one launch.
#include "lm_internal.hpp"

#include <algorithm>

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

__device__ __forceinline__ float pow_int(float log2_decay, int n) { return n == 0 ? 1.0f : __builtin_amdgcn_exp2f(log2_decay * (float)n); }

constexpr int RC = LM_RET_CHUNK;

// chunks of a sequence before its last segment
__device__ __forceinline__ int ret_chunks_ahead(const LmRet& a, int len) {
  const int per = a.seg_chunks * RC;
  return ((len + per - 1) / per - 1) * a.seg_chunks;
}
// Memory of a step in more segments than one, per sequence: the state that it starts from, then what each chunk before the last segment adds to it.  The
// last chunk's place before a segment becomes the state which that segment starts from: place k * seg_chunks of segment k.
__device__ __forceinline__ float* ret_seg_state(const LmRet& a, int seq, int place, int h) {
  return a.seg + (((int64_t)seq * ((a.n_seg - 1) * a.seg_chunks + 1) + place) * a.heads + h) * a.vp * a.dp;
}

// Two pieces of eight coordinates of a head's row: unit j < rot_dims / 16 the pieces j and j + rot_dims / 16, which turn into each other, with one load
// of the angles; units behind them two pieces that do not turn.  rot_dims not a multiple of 16: pieces 2 j and 2 j + 1, element by element.
struct RetUnit {
  int d[2];
  bool turns, whole;
};
__device__ __forceinline__ RetUnit ret_unit(int j, int rot_dims) {
  const bool whole = (rot_dims & 15) == 0;
  const int hp = whole ? rot_dims >> 4 : 0;
  const bool turns = whole && j < hp;
  return RetUnit{{8 * (turns ? j : 2 * j), 8 * (turns ? j + hp : 2 * j + 1)}, turns, whole};
}
// the angles of a unit of row t
__device__ __forceinline__ void ret_angles(const RetUnit& u, const float* angles, int t, int rot_dims, f32x4 (&cs)[4]) {
  if (rot_dims <= 0) return;
  const uint32_t from = (uint32_t)t * (uint32_t)rot_dims + (u.turns ? 2 * u.d[0] : 0);
#pragma unroll
  for (int k = 0; k < 4; ++k) cs[k] = u.whole ? *(const f32x4*)(angles + (from + 4 * k)) : f32x4{0.f, 0.f, 0.f, 0.f};
}
// own * c + other * s.  Which of the two products is rounded by itself is written out, so that a prompt's bits do not hang on the compiler's choice: the first, but
// for the first of eight coordinates, as recorded results have it.
__device__ __forceinline__ float turned(int e, float own, float other, float c, float s) { return e == 0 ? fmaf(own, c, other * s) : fmaf(other, s, own * c); }
// row: the head's row in memory (only read where pieces turn element by element).  ALL: all of a row turns
template <bool ALL>
__device__ __forceinline__ void ret_turn(const RetUnit& u, const u32x4& a, const u32x4& b, const f32x4 (&cs)[4], const bf16_t* row, int rot_dims, const float* angles,
                                         float (&x)[8], float (&y)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float p = (e & 1) ? hi_bf(a[e >> 1]) : lo_bf(a[e >> 1]), q = (e & 1) ? hi_bf(b[e >> 1]) : lo_bf(b[e >> 1]);
    const float c = cs[e >> 1][2 * (e & 1)], s = cs[e >> 1][2 * (e & 1) + 1];
    x[e] = ALL || u.turns ? turned(e, p, -q, c, s) : p;
    y[e] = ALL || u.turns ? turned(e, q, p, c, s) : q;
  }
  if (!ALL && !u.whole)
    for (int e = 0; e < 8; ++e) {
      x[e] = rotated(row, u.d[0] + e, rot_dims, angles);
      y[e] = rotated(row, u.d[1] + e, rot_dims, angles);
    }
}

// y = x * w, rounded: what is left of it behind the high parts is not taken from the product itself, so that a key has the same bits in every kernel
__device__ __forceinline__ void scaled8(const float (&x)[8], float w, float (&y)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    y[e] = x[e] * w;
    asm("" : "+v"(y[e]));
  }
}

// The LDS of a workgroup, in elements: keys and values by token, queries [high | low], the state, and the keys with their weights, high and low parts each but for the
// values.  The weighted keys take the place of the keys, two barriers more per chunk, where a workgroup of their own size would not fit a CU, or not twice.
template <int D, int C>
struct RetLds {
  static constexpr int dp = 32 * D, vp = 32 * C, KS = dp + 8, VS = vp + 8, QS = (2 * dp > vp ? 2 * dp : vp) + 8;
  static constexpr int joint = 2 * (RC * (2 * KS + VS + QS) + 2 * vp * KS), own = joint + 4 * RC * KS;
  static constexpr bool apart = own <= 81920 || (joint > 81920 && own <= 163840);
  static constexpr int bytes = apart ? own : joint, increment = 2 * RC * (2 * KS + VS);
  static constexpr int resident = C * D == 1 ? 3 : bytes <= 81920 ? 2 : 1;  // workgroups on a CU: by LDS, and the registers of the smallest heads
};
// Tile p of 16 columns of v: row or column n of it in a product is column v_column(p, n).  A lane of the outputs then has 8 C columns in a row.
template <int C>
__device__ __forceinline__ int v_column(int p, int n) { return 8 * C * (n >> 2) + 4 * p + (n & 3); }
// ... in LDS tile after tile: a piece of 8 columns lies in two
template <int C>
__device__ __forceinline__ void put_values(bf16_t* row, int piece, const u32x4& v) {
  bf16_t* at = row + 32 * (piece % C) + 4 * (piece / C);
  *(u32x2*)at = u32x2{v[0], v[1]};
  *(u32x2*)(at + 16) = u32x2{v[2], v[3]};
}
// as read_columns, lane row q with tokens t0 + 8 q .. + 7
__device__ __forceinline__ u32x4 read_tokens(const bf16_t* tile, int stride, int t0, int c0, int lane) {
  const bf16_t* p = tile + (t0 + 8 * (lane >> 4) + ((lane & 15) >> 2)) * stride + c0 + 4 * (lane & 3);
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p + 4 * stride));
  const u32x2 lo = __builtin_bit_cast(u32x2, a), hi = __builtin_bit_cast(u32x2, b);
  return u32x4{lo[0], lo[1], hi[0], hi[1]};
}
// sum_t w_t v_t k_t^T of a chunk for each of a wave's C * D tiles of the state: use(tile, sums)
template <int D, int C, class F>
__device__ __forceinline__ void ret_increments(const bf16_t* V, const bf16_t* Wh, const bf16_t* Wl, int wave, int lane, F&& use) {
  using M = RetLds<D, C>;
  constexpr int PT = 2 * C, PER = C == 3 ? 3 : C == 4 ? 2 : 1;  // a wave's tiles i and i + PER have the same 16 columns of v
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    u32x4 v[RC / 32];
#pragma unroll
    for (int k = 0; k < RC / 32; ++k) v[k] = read_tokens(V, M::VS, 32 * k, 16 * ((wave + 4 * j) % PT), lane);
#pragma unroll
    for (int i = j; i < C * D; i += PER) {
      const int nt = (wave + 4 * i) / PT;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < RC / 32; ++k) {
        acc = mfma(read_tokens(Wh, M::KS, 32 * k, 16 * nt, lane), v[k], acc);
        acc = mfma(read_tokens(Wl, M::KS, 32 * k, 16 * nt, lane), v[k], acc);
      }
      use(i, acc);
    }
  }
}

// Prefill.  grid (heads, segments, sequences), four waves; a workgroup walks the chunks of a segment with the head's state in registers, a wave owns 16
// tokens of the outputs and C * D 16 x 16 tiles of the state.  The next chunk's rows are under way while one is worked on.  All memory is read and
// written by pieces of 16 bytes that follow one another, four lanes to 64 bytes at least, and reordered in LDS: a load whose lanes each take another row costs
// four times that (what bounded the form before this, a workgroup per chunk with the state at its start from memory).  A wave's gates lie over its own queries, which it
// has in registers by then, and its outputs over its gates.
// The state goes from chunk to chunk as decay^n S + increment, the increment summed by itself, whatever the segments: a sequence has the same bits alone and beside others.
// The keys take the weights in fp32, before they become two parts; the values' own bits enter.  (Weights on the values, rounded as two parts again: states 4.4e-6 from 64 bits,
// 2.5e-6 this way; 1500 tokens.)
// 8 x 2048 tokens, all launches: 32 heads of 64 169 us, 16 of 128 279; a workgroup per chunk with states in memory 318 and 504; bytes 65.  One prompt of 700: 24 and 35, 33 and 51.  What
// bounds a chunk is vector instructions (about 1000 per wave; 16 gates per lane in full precision are 300 of them) and LDS.
// D: dp / 32, C: vp / 32
template <int D, int C>
__global__ __launch_bounds__(256, (RetLds<D, C>::resident)) void ret_run_kernel(const LmRet a) {
  using M = RetLds<D, C>;
  constexpr int dp = M::dp, vp = M::vp, QS = M::QS, KS = M::KS, VS = M::VS, NT = C * D, PT = 2 * C;
  constexpr int UNITS = dp / 16, NU = (RC * UNITS + 255) / 256;
  extern __shared__ __attribute__((aligned(16))) bf16_t rsm[];
  bf16_t *Kh = rsm, *Kl = Kh + RC * KS, *V = Kl + RC * KS, *Q = V + RC * VS, *Sh = Q + RC * QS, *Sl = Sh + vp * KS;
  bf16_t *Wh = M::apart ? Sl + vp * KS : Kh, *Wl = Wh + RC * KS;
  const int h = blockIdx.x, sg = blockIdx.y, seq = blockIdx.z, tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, first = sg * a.seg_chunks * RC, last = min(first + a.seg_chunks * RC, len);
  if (first >= last) return;
  const bool final = last == len;
  const int pos0 = a.r.seq_pos0[seq];
  const float ld = log2f(a.decay[h]);
  const bf16_t* proj = (const bf16_t*)a.proj + (int64_t)row0 * a.ldp;
  const int cq = a.col_q + h * dp, ck = a.col_k + h * dp, cv = a.col_v + h * vp, cg = a.col_g + h * vp;
  const bool all_turns = a.rot_dims == dp;

  f32x4 S[NT];
  float* slot = a.state + ((int64_t)a.r.seq_slot[seq] * a.heads + h) * vp * dp;
  const float* from = pos0 + first == 0 ? nullptr : a.n_seg > 1 ? ret_seg_state(a, seq, sg * a.seg_chunks, h) : slot;
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int tile = wave + 4 * i, pt = tile % PT, nt = tile / PT;
    S[i] = from ? *(const f32x4*)(from + v_column<C>(pt, r) * dp + 16 * nt + 4 * q) : f32x4{0.f, 0.f, 0.f, 0.f};
  }

  u32x4 qr[NU][2], kr[NU][2], vr[C], gr[C];
  f32x4 cs[NU][4];
  constexpr u32x4 none = {0u, 0u, 0u, 0u};
  auto load = [&](int t0) {  // rows past the end: the last one again
    const int n = min(RC, last - t0);
    const bf16_t* rows = proj + (int64_t)t0 * a.ldp;
    const float* angles = a.rope + (int64_t)(pos0 + t0) * a.rot_dims;
    auto piece = [&](int t, int c) { return *(const u32x4*)(rows + ((uint32_t)min(t, n - 1) * (uint32_t)a.ldp + (uint32_t)c)); };
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + 256 * i, t = u / UNITS;
      const RetUnit at = ret_unit(u % UNITS, a.rot_dims);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        qr[i][k] = piece(t, cq + at.d[k]);
        kr[i][k] = piece(t, ck + at.d[k]);
      }
      ret_angles(at, angles, min(t, n - 1), a.rot_dims, cs[i]);
    }
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int p = tid + 256 * i;
      vr[i] = piece(p / (vp / 8), cv + p % (vp / 8) * 8);
    }
#pragma unroll
    for (int i = 0; i < C; ++i) {  // the wave's own tokens
      const int p = lane + 64 * i;
      gr[i] = piece(16 * wave + p / (vp / 8), cg + p % (vp / 8) * 8);
    }
  };
  load(first);
  const int t = 16 * wave + r;  // this lane's query
  const float et = pow_int(ld, t + 1);

  for (int t0 = first; t0 < last; t0 += RC) {
    const int n = min(RC, last - t0);
    const bool stated = from || t0 > first, on = final || t0 + RC < last;  // on: somebody needs the state behind this chunk
    u32x4 wh[NU][2], wl[NU][2];
    __syncthreads();  // the previous chunk's tiles have been read
    auto stage = [&](auto all) {
      constexpr bool ALL = decltype(all)::value;
#pragma unroll
      for (int i = 0; i < NU; ++i) {
        const int u = tid + 256 * i, tu = u / UNITS;
        if (RC * UNITS % 256 != 0 && u >= RC * UNITS) break;
        const RetUnit at = ret_unit(u % UNITS, a.rot_dims);
        const int tl = min(tu, n - 1);
        const bf16_t* row = proj + (int64_t)(t0 + tl) * a.ldp;
        const float* angles = a.rope + (int64_t)(pos0 + t0 + tl) * a.rot_dims;
        float x[2][8];
        u32x4 hi, lo;
        ret_turn<ALL>(at, qr[i][0], qr[i][1], cs[i], row + cq, a.rot_dims, angles, x[0], x[1]);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          split8(x[k], hi, lo);
          *(u32x4*)(Q + tu * QS + at.d[k]) = hi;
          *(u32x4*)(Q + tu * QS + dp + at.d[k]) = lo;
        }
        ret_turn<ALL>(at, kr[i][0], kr[i][1], cs[i], row + ck, a.rot_dims, angles, x[0], x[1]);
        const float w = a.scale * pow_int(ld, n - 1 - tl);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          float y[8];
          scaled8(x[k], a.scale, y);
          split8(y, hi, lo);
          const bool dead = n < RC && tu >= n;
          *(u32x4*)(Kh + tu * KS + at.d[k]) = dead ? none : hi;
          *(u32x4*)(Kl + tu * KS + at.d[k]) = dead ? none : lo;
          if (!on) continue;
          scaled8(x[k], w, y);
          split8(y, wh[i][k], wl[i][k]);
          if (dead) wh[i][k] = wl[i][k] = none;
          if (M::apart) {
            *(u32x4*)(Wh + tu * KS + at.d[k]) = wh[i][k];
            *(u32x4*)(Wl + tu * KS + at.d[k]) = wl[i][k];
          }
        }
      }
    };
    if (all_turns) stage(std::true_type{});
    else stage(std::false_type{});
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int p = tid + 256 * i, tv = p / (vp / 8);
      put_values<C>(V + tv * VS, p % (vp / 8), n < RC && tv >= n ? none : vr[i]);
    }
    if (stated)
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int tile = wave + 4 * i, pt = tile % PT, nt = tile / PT, at = (16 * pt + r) * KS + 16 * nt + 4 * q;
        const u32x2 hi = {pack_bf16x2(S[i][0], S[i][1]), pack_bf16x2(S[i][2], S[i][3])};
        *(u32x2*)(Sh + at) = hi;
        *(u32x2*)(Sl + at) = u32x2{pack_bf16x2(S[i][0] - lo_bf(hi[0]), S[i][1] - hi_bf(hi[0])), pack_bf16x2(S[i][2] - lo_bf(hi[1]), S[i][3] - hi_bf(hi[1]))};
      }
    u32x4 gc[C];
#pragma unroll
    for (int i = 0; i < C; ++i) gc[i] = gr[i];
    __syncthreads();
    if (t0 + RC < last) load(t0 + RC);

    if (16 * wave < n) {
      bf16_t* G = Q + 16 * wave * QS;  // the wave's own rows
      u32x4 qh[D], ql[D];
#pragma unroll
      for (int s = 0; s < D; ++s) {
        qh[s] = *(const u32x4*)(G + r * QS + 32 * s + 8 * q);
        ql[s] = *(const u32x4*)(G + r * QS + dp + 32 * s + 8 * q);
      }
      wave_lds_order();
#pragma unroll
      for (int i = 0; i < C; ++i) {
        const int p = lane + 64 * i;
        *(u32x4*)(G + p / (vp / 8) * QS + p % (vp / 8) * 8) = gc[i];
      }
      wave_lds_order();
      f32x4 o[PT];
#pragma unroll
      for (int i = 0; i < PT; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (stated) {
#pragma unroll
        for (int s = 0; s < D; ++s)
#pragma unroll
          for (int i = 0; i < PT; ++i) {
            const u32x4 sh = *(const u32x4*)(Sh + (16 * i + r) * KS + 32 * s + 8 * q), sl = *(const u32x4*)(Sl + (16 * i + r) * KS + 32 * s + 8 * q);
            o[i] = mfma(sh, qh[s], o[i]);
            o[i] = mfma(sl, qh[s], o[i]);
            o[i] = mfma(sh, ql[s], o[i]);
          }
#pragma unroll
        for (int i = 0; i < PT; ++i) o[i] *= et;
      }
      int age0 = t - 4 * q;
      asm volatile("" : "+v"(age0));  // (powers made here: 16 registers less than in front of the loop)
#pragma unroll
      for (int b = 0; b < RC / 32; ++b) {
        if (2 * b > wave) continue;
        float p[8];  // tokens 32 b + 4 q + j and 32 b + 16 + 4 q + j: the order of read_columns
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
            const int age = age0 - 16 * sb - e;
            p[4 * half + e] = sb <= wave && age >= 0 ? acc[e] * pow_int(ld, age) : 0.f;
          }
        }
        u32x4 ph, pl;
        split8(p, ph, pl);
#pragma unroll
        for (int i = 0; i < PT; ++i) {
          const u32x4 v = read_columns(V, VS, 32 * b, 16 * i, lane);
          o[i] = mfma(v, ph, o[i]);
          o[i] = mfma(v, pl, o[i]);
        }
      }
      // the lane's columns 8 C q ..: four sums of 2 C in a row, then over the quarters (written out, as the rotation)
      float sq[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        auto at = [&](int d) { return o[(PT * k + d) >> 2][(PT * k + d) & 3]; };
        sq[k] = fmaf(at(0), at(0), at(1) * at(1));
#pragma unroll
        for (int d = 2; d < PT; ++d) sq[k] = fmaf(at(d), at(d), sq[k]);
      }
      float ss = (sq[0] + sq[1]) + (sq[2] + sq[3]);
      ss += __shfl_xor(ss, 16, 64);
      ss += __shfl_xor(ss, 32, 64);
      const float rn = 1.0f / sqrtf(ss / (float)a.vdim + a.eps);
#pragma unroll
      for (int i = 0; i < C; ++i) {
        bf16_t* at = G + r * QS + 8 * C * q + 8 * i;
        const u32x4 g = *(const u32x4*)at;
        u32x4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f32x4& x = o[2 * i + (e >> 1)];
          const int c = 2 * (e & 1);
          y[e] = pack_bf16x2(x[c] * rn * silu_f32(lo_bf(g[e])), x[c + 1] * rn * silu_f32(hi_bf(g[e])));
        }
        *(u32x4*)at = y;
      }
      wave_lds_order();
#pragma unroll
      for (int i = 0; i < C; ++i) {
        const int p = lane + 64 * i, tg = p / (vp / 8), d = p % (vp / 8) * 8;
        if (16 * wave + tg < n)
          *(u32x4*)((bf16_t*)a.out + (int64_t)(row0 + t0 + 16 * wave + tg) * a.ldo + in_chunks(h * vp + d, a.out_chunk)) = *(const u32x4*)(G + tg * QS + d);
      }
    }
    if (!on) break;
    if (!M::apart) {
      __syncthreads();  // the keys have been read
#pragma unroll
      for (int i = 0; i < NU; ++i) {
        const int u = tid + 256 * i, tu = u / UNITS;
        if (RC * UNITS % 256 != 0 && u >= RC * UNITS) break;
        const RetUnit at = ret_unit(u % UNITS, a.rot_dims);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          *(u32x4*)(Wh + tu * KS + at.d[k]) = wh[i][k];
          *(u32x4*)(Wl + tu * KS + at.d[k]) = wl[i][k];
        }
      }
      __syncthreads();
    }
    const float keep = pow_int(ld, n);
    ret_increments<D, C>(V, Wh, Wl, wave, lane, [&](int i, const f32x4& inc) { S[i] = S[i] * keep + inc; });
  }
  if (final)
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int tile = wave + 4 * i, pt = tile % PT, nt = tile / PT;
      *(f32x4*)(slot + v_column<C>(pt, r) * dp + 16 * nt + 4 * q) = S[i];
    }
}

// grid (heads, chunks, sequences): what each chunk before the last segment adds to the state
template <int D, int C>
__global__ __launch_bounds__(256) void ret_increment_kernel(const LmRet a) {
  using M = RetLds<D, C>;
  constexpr int dp = M::dp, vp = M::vp, KS = M::KS, VS = M::VS, PT = 2 * C, UNITS = dp / 16, NU = (RC * UNITS + 255) / 256;
  extern __shared__ __attribute__((aligned(16))) bf16_t rsm[];
  bf16_t *Wh = rsm, *Wl = Wh + RC * KS, *V = Wl + RC * KS;
  const int h = blockIdx.x, c = blockIdx.y, seq = blockIdx.z, tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0;
  if (c >= ret_chunks_ahead(a, len)) return;  // (all of them whole)
  const float ld = log2f(a.decay[h]);
  const bf16_t* rows = (const bf16_t*)a.proj + (int64_t)(row0 + c * RC) * a.ldp;
  const float* angles = a.rope + (int64_t)(a.r.seq_pos0[seq] + c * RC) * a.rot_dims;
  const int ck = a.col_k + h * dp, cv = a.col_v + h * vp;
  auto piece = [&](int t, int col) { return *(const u32x4*)(rows + ((uint32_t)t * (uint32_t)a.ldp + (uint32_t)col)); };
  u32x4 vr[C];
#pragma unroll
  for (int i = 0; i < C; ++i) {
    const int p = tid + 256 * i;
    vr[i] = piece(p / (vp / 8), cv + p % (vp / 8) * 8);
  }
#pragma unroll
  for (int i = 0; i < NU; ++i) {
    const int u = tid + 256 * i, t = u / UNITS;
    if (RC * UNITS % 256 != 0 && u >= RC * UNITS) break;
    const RetUnit at = ret_unit(u % UNITS, a.rot_dims);
    f32x4 cs[4];
    ret_angles(at, angles, t, a.rot_dims, cs);
    float x[2][8];
    ret_turn<false>(at, piece(t, ck + at.d[0]), piece(t, ck + at.d[1]), cs, rows + (int64_t)t * a.ldp + ck, a.rot_dims, angles + (int64_t)t * a.rot_dims, x[0], x[1]);
    const float w = a.scale * pow_int(ld, RC - 1 - t);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      float y[8];
      u32x4 hi, lo;
      scaled8(x[k], w, y);
      split8(y, hi, lo);
      *(u32x4*)(Wh + t * KS + at.d[k]) = hi;
      *(u32x4*)(Wl + t * KS + at.d[k]) = lo;
    }
  }
#pragma unroll
  for (int i = 0; i < C; ++i) {
    const int p = tid + 256 * i;
    put_values<C>(V + p / (vp / 8) * VS, p % (vp / 8), vr[i]);
  }
  __syncthreads();
  float* to = ret_seg_state(a, seq, c + 1, h);
  ret_increments<D, C>(V, Wh, Wl, wave, lane, [&](int i, const f32x4& inc) {
    const int tile = wave + 4 * i, pt = tile % PT, nt = tile / PT;
    *(f32x4*)(to + v_column<C>(pt, r) * dp + 16 * nt + 4 * q) = inc;
  });
}

// grid (heads * vp * dp / 1024, sequences): the states that the segments start from, chunk by chunk as within a segment
__global__ __launch_bounds__(256) void ret_segments_kernel(const LmRet a) {
  const int seq = blockIdx.y, per_head = a.vp * a.dp;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4, n_el = (int64_t)a.heads * per_head;
  if (i >= n_el) return;
  const int h = (int)(i / per_head), n = ret_chunks_ahead(a, a.r.seq_row0[seq + 1] - a.r.seq_row0[seq]);
  const float keep = pow_int(log2f(a.decay[h]), RC);
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  if (a.r.seq_pos0[seq] > 0) S = *(const f32x4*)(a.state + (int64_t)a.r.seq_slot[seq] * n_el + i);
  float* p = ret_seg_state(a, seq, 0, 0) + i;
  *(f32x4*)p = S;
  constexpr int U = 4;  // chunks in flight
  for (int c0 = 0; c0 < n; c0 += U) {
    f32x4 inc[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c0 + u < n) inc[u] = *(const f32x4*)(p + (c0 + u + 1) * n_el);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c0 + u < n) {
        S = S * keep + inc[u];
        if ((c0 + u + 1) % a.seg_chunks == 0) *(f32x4*)(p + (c0 + u + 1) * n_el) = S;  // in the place of what is in it now
      }
  }
}

typedef void (*RetKernel)(const LmRet);
struct RetPick {
  RetKernel run, inc;
  int lds, inc_lds, resident;
};
template <int D, int C>
RetPick ret_run_of() {
  using M = RetLds<D, C>;
  static_assert(M::bytes <= 163840, "LDS");
  return RetPick{ret_run_kernel<D, C>, ret_increment_kernel<D, C>, M::bytes, M::increment, M::resident};
}
template <int D>
RetPick ret_run_by_width(int c) {
  switch (c) {
    case 1: return ret_run_of<D, 1>();
    case 2: return ret_run_of<D, 2>();
    case 3: return ret_run_of<D, 3>();
    case 4: return ret_run_of<D, 4>();
    default: return RetPick{};
  }
}
RetPick ret_run_by_widths(int dp, int vp) {
  switch (dp / 32) {
    case 1: return ret_run_by_width<1>(vp / 32);
    case 2: return ret_run_by_width<2>(vp / 32);
    case 3: return ret_run_by_width<3>(vp / 32);
    case 4: return ret_run_by_width<4>(vp / 32);
    default: return RetPick{};
  }
}
RetPick ret_run_pick(const LmRet& a) {
  if ((a.col_q | a.col_k | a.col_v | a.col_g | a.ldp | a.ldo | a.out_chunk) % 8 != 0) return RetPick{};  // pieces of eight
  return ret_run_by_widths(a.dp, a.vp);
}

// grid (heads, sequences).  Sixteen lanes per state row, sixteen rows at a time, R rows of up to 64 E columns per thread.  Few sequences: the chain of loads
// bounds it, and all of a head's rows are under way before the first use (ALL).  8 sequences, 16 heads of 128: 17.1 us with a row loaded after the other,
// 9.6 this way; 1 sequence, 32 heads of 64: 6.7 and 5.7; 64 of 32 x 64: 16.7 and 14.9.  Many: the state's bytes, and more workgroups per CU hide more than
// registers full of rows (128 sequences, 8 heads of 256: 122 us with all, 104 with a row after the other; 16 of 192: 141 and 114).
// The state is read and written once a step, past the caches (non-temporal): 32 heads of 64, 16 / 32 / 64 sequences 6.8 / 9.5 / 16.3 -> 6.2 / 8.0 / 14.1 us, 16 of 128
// 9.8 / 17.4 / 28.6 -> 8.9 / 13.4 / 24.2, 96 23.1 -> 22.1 and 40.2 -> 39.8; one sequence 5.1 and 5.2.
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
        if (pos > 0 && e < vp && 4 * l + 64 * j < dp) S[i][j] = __builtin_nontemporal_load((const f32x4*)(st + (int64_t)e * dp + 4 * l + 64 * j));
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
        __builtin_nontemporal_store(s, (f32x4*)(st + (int64_t)e * dp + d));
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

// Segments: as many as keep to the workgroups that the CUs hold by their LDS (64 x 64: two, larger heads mostly one).  The increments cost about half of the outputs, and
// they and the states two launches, about two chunks.  us with 1, 2, .. segments: 32 heads of 64 x 64, one prompt of 130 tokens 17.4, 19.1, 14.9; 700 11 segments 23.8, 6 24.9;
// 3 x 2048 5 79.0, 8 80.7; 8 x 2048 184, 168, 200 (3).  16 of 64 x 128, 16 segments of 2000 38.8 and 32 41.1; 3 x 700 4 41.6, 6 49.3; 8 x 500 66.8, 52.7, 58.9 (4); 8 x 2048 259,
// 175, 191 (4).  16 of 96 x 96, 8 x 2048 286, 202, 224 (4).
inline int ret_room(int dp, int vp) { return 256 * ret_run_by_widths(dp, vp).resident; }
int lm_ret_segments(int n_seq, int heads, int dp, int vp, int max_len, int* chunks) {
  const int n = (max_len + RC - 1) / RC, segs = ret_room(dp, vp) / (n_seq * heads), per = segs > 1 ? (n + segs - 1) / segs : n;
  *chunks = 3 * per + 3 <= 2 * n ? per : n;
  return (n + *chunks - 1) / *chunks;
}
int lm_ret_most_states(int n_seq, int heads, int dp, int vp, int max_len) {
  const int n = (max_len + RC - 1) / RC;
  return n > 1 ? std::min(n_seq, ret_room(dp, vp) / (2 * heads)) * n : 0;  // (more sequences: no segments)
}
bool lm_ret_mfma_takes(const LmRet& a) { return ret_run_pick(a).run != nullptr; }
md_status lm_ret_mfma(const LmRet& a, hipStream_t s) {
  const RetPick k = ret_run_pick(a);
  if (!k.run) return MD_ERR_UNSUPPORTED;
  const dim3 grid(a.heads, a.n_seg, a.r.n_seq);
  MD_TRY(md_ensure_dynamic_lds((const void*)k.run, k.lds));
  if (a.n_seg > 1) {
    MD_TRY(md_ensure_dynamic_lds((const void*)k.inc, k.inc_lds));
    hipLaunchKernelGGL(k.inc, dim3(a.heads, (a.n_seg - 1) * a.seg_chunks, a.r.n_seq), dim3(256), k.inc_lds, s, a);
    MD_TRY(md_launch_status());
    hipLaunchKernelGGL(ret_segments_kernel, dim3((a.heads * a.vp * a.dp + 1023) / 1024, a.r.n_seq), dim3(256), 0, s, a);
    MD_TRY(md_launch_status());
  }
  hipLaunchKernelGGL(k.run, grid, dim3(256), k.lds, s, a);
  return md_launch_status();
}

bool lm_ret_decode_takes(const LmRet& a) { return a.dp <= 256 && a.vp <= 256; }
md_status lm_ret_decode(const LmRet& a, hipStream_t s) {
  hipLaunchKernelGGL(ret_decode_pick(a), dim3(a.heads, a.r.n_seq), dim3(256), 0, s, a);
  return md_launch_status();
}
