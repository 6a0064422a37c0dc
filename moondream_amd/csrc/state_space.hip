// Selective state spaces (Mamba-2): S <- exp(-decay dt) S + dt B x^T, y = S^T C + skip x, behind a causal convolution, with a gate and a
// grouped RMS norm behind it.
//
// The state of a head is kept transposed, fp32 [vdim][dim].
//
//   ssm_conv_kernel        convolution + bias + silu of x | B | C, softplus of dt: whole rows, inputs before the step from the slot's ring
//   ssm_scan_kernel        plain recurrence, token by token, any dtype, fp32 on the vector ALUs
//   ssm_chunk_kernel       bf16 prefill on the matrix cores, 64 tokens at a time (below)
//   ssm_segments_kernel    states at the start of every segment
//   ssm_decode_kernel      bf16 decode step, one workgroup per (sequence, head): convolution, state update, output and gate in one launch
//   ssm_norm_kernel        grouped RMS norm of the gated outputs, in place; and the last projections of every sequence of the step -> its slot
//                          (row p % taps of the ring)
//
// ssm_chunk_kernel.  A workgroup walks the chunks of a segment of a sequence for one head with the state in registers:
//   y_t = exp(c_t) S^T C_t + sum_{s<=t} exp(c_t - c_s) dt_s (C_t . B_s) x_s + skip x_t,   c: running sum of -decay dt in the chunk
//   S  <- exp(c_end) S + sum_s exp(c_end - c_s) dt_s B_s x_s^T
// B, C and x are bf16 behind their convolution; what the recurrence makes of them counts as fp32: weighted scores, weighted inputs and the
// state enter a product as the sum of two bf16 (16 mantissa bits).  Operands that need consecutive tokens per lane come from row-major LDS
// tiles through the transposing LDS read.  When sequences x heads do not fill the chip, a sequence is cut into segments: a first launch of
// the same kernel makes what every segment adds to the state (INC), ssm_segments_kernel the states they start from.
// What bounds a chunk is the chain through it (load, LDS, products, LDS; 4.2 us of 64 x 64 x 128).  C, the gates and the outputs go through LDS too, so that
// memory is read and written by whole pieces in a row, not by a piece of another row per lane: 5 ragged sequences, 4900 tokens, 64 heads of 64 x 128, 106 -> 102 us, 700
// tokens of 16 x 128 x 128 in segments 17.7 -> 16.0 and 8.8 -> 8.1.
#include "lm_internal.hpp"

namespace {

__device__ __forceinline__ float softplus_f32(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

// a thread: 8 columns of x | B | C of ROWS consecutive rows; behind those blocks, 8 heads' dt of one row.
// TAPS > 0: inputs slide through registers; 0: any number
template <typename T, int TAPS, int ROWS>
__global__ __launch_bounds__(256) void ssm_conv_kernel(const LmSsm a, unsigned conv_blocks) {
  const int cw = a.cw();
  if (blockIdx.x >= conv_blocks) {
    const unsigned i = (blockIdx.x - conv_blocks) * 256 + threadIdx.x, units = (a.heads + 7) / 8, row = i / units;
    if (row >= (unsigned)a.r.n_rows) return;
    const int h0 = (i - row * units) * 8;
    const auto raw = ld8((const T*)a.proj + (int64_t)row * a.ldp + a.col_dt + h0);
    float* dt = a.dt + (int64_t)row * a.heads + h0;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (h0 + e < a.heads) dt[e] = softplus_f32(half8(raw, e / 4)[e % 4] + a.dt_bias[h0 + e]);
    return;
  }
  const unsigned idx = blockIdx.x * 256 + threadIdx.x, units = cw / 8, rb = idx / units;
  const int unit = idx - rb * units, r0 = rb * ROWS, r1 = min(r0 + ROWS, a.r.n_rows);
  if (r0 >= r1) return;
  const int c = unit * 8;
  const T* proj = (const T*)a.proj + a.col_x + c;
  constexpr int W = TAPS > 0 ? TAPS : 1;
  f32x4 w[W][2], win[W][2], bias[2];  // w[k], win[k]: k steps back
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    bias[h] = *(const f32x4*)(a.conv_bias + c + 4 * h);
#pragma unroll
    for (int k = 0; k < W; ++k) w[k][h] = TAPS > 0 ? *(const f32x4*)(a.conv + (int64_t)(TAPS - 1 - k) * cw + c + 4 * h) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  int seq = -1, pos0 = 0, slot = 0;
  auto input = [&](int row, int pos, int k, int h) {  // the projection k steps before `pos`
    const int p = pos - k;
    if (p < 0) return f32x4{0.f, 0.f, 0.f, 0.f};
    if (p >= pos0) return ld4(proj + (int64_t)(row - k) * a.ldp + 4 * h);
    return ld4((const T*)a.conv_state + ((int64_t)slot * a.taps + p % a.taps) * cw + c + 4 * h);
  };
  auto start = [&](int row) {  // a sequence's rows begin, or go on from another thread's
    seq = a.r.row_seq[row];
    pos0 = a.r.seq_pos0[seq];
    slot = a.r.seq_slot[seq];
    const int pos = a.r.row_pos[row];
#pragma unroll
    for (int k = 1; k < W; ++k)
#pragma unroll
      for (int h = 0; h < 2; ++h) win[k - 1][h] = input(row, pos, k, h);  // (moves to k when the row itself comes)
  };
  auto store = [&](int row, f32x4 (&y)[2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) y[h][e] = silu_for<T>(y[h][e]);
    st8((T*)a.u + (int64_t)row * cw + c, y[0], y[1]);
  };
  if constexpr (TAPS > 0) {
    auto walk = [&](auto whole) {  // whole: ROWS rows of one sequence
      constexpr int BATCH = ROWS < 8 ? ROWS : 8;  // rows whose loads are in flight together
      start(r0);
#pragma unroll
      for (int b = 0; b < ROWS; b += BATCH) {
        const int b0 = r0 + b;
        if (!whole && b0 >= r1) break;
        decltype(ld8(proj)) in[BATCH];
#pragma unroll
        for (int i = 0; i < BATCH; ++i) in[i] = ld8(proj + (int64_t)(whole ? b0 + i : min(b0 + i, r1 - 1)) * a.ldp);
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
          if (!whole && b0 + i >= r1) break;
          if (!whole && b0 + i > r0 && a.r.row_seq[b0 + i] != seq) start(b0 + i);
          f32x4 y[2] = {bias[0], bias[1]};
#pragma unroll
          for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int k = W - 1; k > 0; --k) {
              win[k][h] = win[k - 1][h];
              y[h] += w[k][h] * win[k][h];
            }
            win[0][h] = half8(in[i], h);
            y[h] += w[0][h] * win[0][h];
          }
          store(b0 + i, y);
        }
      }
    };
    if (r1 - r0 == ROWS && a.r.row_seq[r0] == a.r.row_seq[r1 - 1]) walk(std::true_type{});
    else walk(std::false_type{});
  } else {
    for (int row = r0; row < r1; ++row) {
      if (a.r.row_seq[row] != seq) start(row);
      const int pos = a.r.row_pos[row];
      f32x4 y[2] = {bias[0], bias[1]};
      for (int k = a.taps - 1; k >= 0; --k)
#pragma unroll
        for (int h = 0; h < 2; ++h) y[h] += *(const f32x4*)(a.conv + (int64_t)(a.taps - 1 - k) * cw + c + 4 * h) * input(row, pos, k, h);
      store(row, y);
    }
  }
}

// block of 1024 columns of a sequence's last projections -> its slot's ring (behind the convolution, which reads what was there)
template <typename T>
__device__ __forceinline__ void ssm_ring(const LmSsm& a, int seq, int block) {
  const int cw = a.cw(), c = (block * 256 + threadIdx.x) * 4;
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, pos0 = a.r.seq_pos0[seq], slot = a.r.seq_slot[seq];
  T* ring = (T*)a.conv_state + (int64_t)slot * a.taps * cw;
  const int keep = min(len, a.taps - 1);
  if (c >= cw) return;
  for (int t = len - keep; t < len; ++t) st4(ring + (int64_t)((pos0 + t) % a.taps) * cw + c, ld4((const T*)a.proj + (int64_t)(row0 + t) * a.ldp + a.col_x + c));
}

// 16 rows per thread, or 4 where that leaves most of the chip without a workgroup (700 rows, 2304 columns: 6.3 us, 16.6 with 16 rows;
// 17 rows of 2176: 5.0 us, 8.3)
template <typename T>
md_status conv(const LmSsm& a, hipStream_t s) {
  const int64_t units = a.cw() / 8, n_dt = (int64_t)a.r.n_rows * ((a.heads + 7) / 8);
  if ((a.r.n_rows + 15) / 16 * units >= 1 << 30 || n_dt >= 1 << 30) return MD_ERR_UNSUPPORTED;
  const bool few = a.taps <= 4 && (a.r.n_rows + 15) / 16 * units <= 256 * 256;
  const int64_t n = (a.r.n_rows + (few ? 3 : 15)) / (few ? 4 : 16) * units;
  const unsigned conv_blocks = (unsigned)((n + 255) / 256), dt_blocks = (unsigned)((n_dt + 255) / 256);
  auto pick = [&](auto rows) {
    constexpr int R = decltype(rows)::value;
    return a.taps == 1 ? ssm_conv_kernel<T, 1, R> : a.taps == 2 ? ssm_conv_kernel<T, 2, R> : a.taps == 3 ? ssm_conv_kernel<T, 3, R> : ssm_conv_kernel<T, 4, R>;
  };
  auto fn = a.taps > 4 ? ssm_conv_kernel<T, 0, 16> : few ? pick(std::integral_constant<int, 4>{}) : pick(std::integral_constant<int, 16>{});
  hipLaunchKernelGGL(fn, dim3(conv_blocks + dt_blocks), dim3(256), 0, s, a, conv_blocks);
  return md_launch_status();
}

// grid (n_seq, heads, vp / 16): 16 columns of the state, 16 neighbouring lanes per column, each owning rows 4 l .. + 3 of every 64.  Tokens are
// staged 16 at a time (8 for states above 256) and then run without a barrier: the recurrence is a chain, what counts is what lies on it (one
// sequence of 300 tokens, 32 heads of 64 x 64, fp32: 67 us, 342 us token by token).
// Q: quads of state rows per thread, dp <= 64 Q (and for Q = 2 more than 64)
template <typename T, int Q>
__global__ __launch_bounds__(256) void ssm_scan_kernel(const LmSsm a) {
  constexpr int SCAN_TOKENS = Q <= 4 ? 16 : 8;
  __shared__ __attribute__((aligned(16))) float bs[SCAN_TOKENS][64 * Q], cs[SCAN_TOKENS][64 * Q];
  __shared__ float xs[SCAN_TOKENS][16], zs[SCAN_TOKENS][16], os[SCAN_TOKENS][16], dts[SCAN_TOKENS], keeps[SCAN_TOKENS];
  const int seq = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, l = tid & 15, col = tid >> 4, e0 = blockIdx.z * 16, e = e0 + col;
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, pos0 = a.r.seq_pos0[seq];
  const int dp = a.dp, vp = a.vp, H = a.heads, cw = a.cw(), g = h / (H / a.groups);
  float* st = a.state + (((int64_t)a.r.seq_slot[seq] * H + h) * vp + e) * dp;
  const float decay = a.decay[h], skip = a.skip[h];
  f32x4 S[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int d = 64 * i + 4 * l;
    S[i] = (pos0 > 0 && d < dp) ? *(const f32x4*)(st + d) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  constexpr int QT = SCAN_TOKENS * 16 * Q / 256;  // quads of B (and C) per thread
  f32x4 bn[QT], cn[QT];  // the next tokens', under way during these
  float xn = 0.f, zn = 0.f, dtn = 0.f;
  const int quads = dp / 4;
  auto load = [&](int t0) {
    const int n = min(SCAN_TOKENS, len - t0);
#pragma unroll
    for (int j = 0; j < QT; ++j) {
      const int i = tid + 256 * j, t = i / quads;
      if (t >= n) continue;
      const T* u = (const T*)a.u + (int64_t)(row0 + t0 + t) * cw + H * vp + (i - t * quads) * 4;
      bn[j] = ld4(u + g * dp);
      cn[j] = ld4(u + (a.groups + g) * dp);
    }
    if (col < n) {
      const int64_t row = row0 + t0 + col;
      xn = ldf((const T*)a.u + row * cw + h * vp + e0 + l);
      zn = ldf((const T*)a.proj + row * a.ldp + a.col_z + h * vp + e0 + l);
    }
    if (tid < n) dtn = a.dt[(int64_t)(row0 + t0 + tid) * H + h];
  };
  load(0);
  for (int t0 = 0; t0 < len; t0 += SCAN_TOKENS) {
    const int n = min(SCAN_TOKENS, len - t0);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < QT; ++j) {
      const int i = tid + 256 * j, t = i / quads, d = (i - t * quads) * 4;
      if (t >= n) continue;
      *(f32x4*)(bs[t] + d) = bn[j];
      *(f32x4*)(cs[t] + d) = cn[j];
    }
    if (col < n) {
      xs[col][l] = xn;
      zs[col][l] = zn;
    }
    if (tid < n) {
      dts[tid] = dtn;
      keeps[tid] = expf(-decay * dtn);
    }
    __syncthreads();
    if (t0 + SCAN_TOKENS < len) load(t0 + SCAN_TOKENS);
#pragma unroll 4
    for (int t = 0; t < n; ++t) {
      const float keep = keeps[t], x = xs[t][col], in = dts[t] * x;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const int d = 64 * i + 4 * l;
        if ((Q <= 2 && i + 1 < Q) || d < dp) {
          S[i] = keep * S[i] + *(const f32x4*)(bs[t] + d) * in;
          o += S[i] * *(const f32x4*)(cs[t] + d);
        }
      }
      const float sum = row_sum_16((o[0] + o[1]) + (o[2] + o[3]));
      if (l == 0) os[t][col] = sum + skip * x;
    }
    __syncthreads();
    if (col < n) stf((T*)a.out + (int64_t)(row0 + t0 + col) * a.ldo + in_chunks(h * vp + e0 + l, a.out_chunk), os[col][l] * silu_f32(zs[col][l]));
  }
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int d = 64 * i + 4 * l;
    if (d < dp) *(f32x4*)(st + d) = S[i];
  }
}

// one row per workgroup.  Norm group k: elements k * gs .. of the heads' outputs without their padding; element f lies at column
// f / vdim * vp + f % vdim.  BLOCK: all waves take the groups one after the other, else a wave takes every fourth group.
// V: consecutive elements at a time (groups and heads are multiples of it).  Workgroups behind the rows': the rings of the sequences.
template <typename T, bool BLOCK, int V>
__global__ __launch_bounds__(256) void ssm_norm_kernel(const LmSsm a) {
  __shared__ float red[4];
  if ((int)blockIdx.x >= a.r.n_rows) {
    const int i = blockIdx.x - a.r.n_rows, blocks = (a.cw() + 1023) / 1024;
    return ssm_ring<T>(a, i / blocks, i % blocks);
  }
  T* row = (T*)a.out + (int64_t)blockIdx.x * a.ldo;
  const int gs = a.heads * a.vdim / a.norm_groups, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int k = BLOCK ? 0 : wave; k < a.norm_groups; k += BLOCK ? 1 : 4) {
    auto column = [&](int i) {
      const int f = k * gs + i, h = f / a.vdim;
      return h * a.vp + f - h * a.vdim;
    };
    auto at = [&](int c) { return row + in_chunks(c, a.out_chunk); };
    const int first = (BLOCK ? threadIdx.x : lane) * V, step = (BLOCK ? 256 : 64) * V;
    float ss = 0.f;
    for (int i = first; i < gs; i += step) {
      const T* p = at(column(i));
      if (V == 4) {
        const f32x4 v = ld4(p);
        ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
      } else {
        ss += ldf(p) * ldf(p);
      }
    }
    ss = BLOCK ? block_sum_256(ss, red) : wave_sum(ss);
    const float r = 1.0f / sqrtf(ss / (float)gs + a.eps);
    for (int i = first; i < gs; i += step) {
      const int c = column(i);
      if (V == 4) st4(at(c), ld4(at(c)) * r * *(const f32x4*)(a.out_norm + c));
      else stf(at(c), ldf(at(c)) * r * a.out_norm[c]);
    }
  }
}

// ring: behind conv(), whose inputs the next step's go on from
template <typename T>
md_status norm(const LmSsm& a, bool ring, hipStream_t s) {
  const int gs = a.heads * a.vdim / a.norm_groups;
  const bool v4 = a.vdim % 4 == 0 && gs % 4 == 0, block = a.norm_groups < 4;
  auto fn = v4 ? (block ? ssm_norm_kernel<T, true, 4> : ssm_norm_kernel<T, false, 4>) : (block ? ssm_norm_kernel<T, true, 1> : ssm_norm_kernel<T, false, 1>);
  hipLaunchKernelGGL(fn, dim3(a.r.n_rows + (ring && a.taps > 1 ? a.r.n_seq * ((a.cw() + 1023) / 1024) : 0)), dim3(256), 0, s, a);
  return md_launch_status();
}

template <typename T>
md_status plain(const LmSsm& a, hipStream_t s) {
  if (a.dp > 512) return MD_ERR_UNSUPPORTED;
  MD_TRY(conv<T>(a, s));
  auto scan = a.dp <= 64 ? ssm_scan_kernel<T, 1> : a.dp <= 128 ? ssm_scan_kernel<T, 2> : a.dp <= 256 ? ssm_scan_kernel<T, 4> : ssm_scan_kernel<T, 8>;
  hipLaunchKernelGGL(scan, dim3(a.r.n_seq, a.heads, a.vp / 16), dim3(256), 0, s, a);
  MD_TRY(md_launch_status());
  return norm<T>(a, true, s);
}

// ---------------------------------------------------------------------------------------------------------------------------
constexpr float LOG2E = 1.4426950408889634f;

constexpr int L = LM_SSM_CHUNK;

// grid (heads, segments, sequences), four waves; a wave owns 16 tokens of the outputs and C * D 16 x 16 tiles of the state.
// D: dp / 32, C: vp / 32
template <int D, int C, bool INC>
__global__ __launch_bounds__(256, C * D > 9 ? 1 : 2) void ssm_chunk_kernel(const LmSsm a) {
  constexpr int dp = 32 * D, vp = 32 * C, XS = vp + 8, BS = dp + 8, QS = (dp > vp ? dp : vp) + 8, NT = C * D, PT = 2 * C;
  constexpr int PER = C == 3 ? 3 : C == 4 ? 2 : 1;  // a wave's state tiles i and i + PER have the same 16 columns of x
  extern __shared__ __attribute__((aligned(16))) bf16_t sm[];
  bf16_t *X = sm, *B = X + L * XS, *Sh = B + L * BS, *Sl = Sh + vp * BS, *Q = Sl + vp * BS;  // Q: C of the chunk, then a wave's gates and outputs over its own rows
  __shared__ float cum[L], dts[L], ws[L];
  const int h = blockIdx.x, sg = blockIdx.y, seq = blockIdx.z, tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = a.heads, cw = a.cw(), g = h / (H / a.groups);
  const int row0 = a.r.seq_row0[seq], len = a.r.seq_row0[seq + 1] - row0, first = sg * a.seg_chunks * L, last = min(first + a.seg_chunks * L, len);
  if (first >= last) return;
  const bool final = last == len;
  if (INC && final) return;  // nobody starts behind the last segment
  const float rate = -a.decay[h] * LOG2E, skip = a.skip[h];
  const bf16_t* u = (const bf16_t*)a.u + (int64_t)row0 * cw;
  const int cx = h * vp, cb = H * vp + g * dp, cc = H * vp + (a.groups + g) * dp;

  f32x4 S[NT];
  float* slot = a.state + ((int64_t)a.r.seq_slot[seq] * H + h) * vp * dp;
  float* seg = a.seg + (((int64_t)seq * a.n_seg + sg) * H + h) * vp * dp;
  const float* from = INC ? nullptr : a.n_seg > 1 ? seg : a.r.seq_pos0[seq] > 0 ? slot : nullptr;
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int tile = wave + 4 * i, pt = tile % PT, nt = tile / PT;
    S[i] = from ? *(const f32x4*)(from + (16 * pt + r) * dp + 16 * nt + 4 * q) : f32x4{0.f, 0.f, 0.f, 0.f};
  }

  u32x4 xr[C], br[D], qr[D], zr[C];
  float dt_r = 0.f;
  auto load = [&](int t0) {
    const int n = min(L, last - t0);
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int piece = tid + 256 * i, t = piece / (vp / 8), d = (piece - t * (vp / 8)) * 8;
      xr[i] = t < n ? *(const u32x4*)(u + (int64_t)(t0 + t) * cw + cx + d) : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < D; ++i) {
      const int piece = tid + 256 * i, t = piece / (dp / 8), d = (piece - t * (dp / 8)) * 8;
      br[i] = t < n ? *(const u32x4*)(u + (int64_t)(t0 + t) * cw + cb + d) : u32x4{0u, 0u, 0u, 0u};
    }
    if (!INC) {
#pragma unroll
      for (int i = 0; i < D; ++i) {
        const int piece = tid + 256 * i, t = piece / (dp / 8), d = (piece - t * (dp / 8)) * 8;
        qr[i] = t < n ? *(const u32x4*)(u + (int64_t)(t0 + t) * cw + cc + d) : u32x4{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int i = 0; i < C; ++i) {  // gates: the wave's own tokens
        const int piece = lane + 64 * i, t = 16 * wave + piece / (vp / 8), d = piece % (vp / 8) * 8;
        zr[i] = t < n ? *(const u32x4*)((const bf16_t*)a.proj + (int64_t)(row0 + t0 + t) * a.ldp + a.col_z + h * vp + d) : u32x4{0u, 0u, 0u, 0u};
      }
    }
    if (tid < L) dt_r = tid < n ? a.dt[(int64_t)(row0 + t0 + tid) * H + h] : 0.f;
  };
  load(first);
  float total_log = 0.f;

  for (int t0 = first; t0 < last; t0 += L) {
    const int n = min(L, last - t0);
    __syncthreads();  // the previous chunk's tiles have been read
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int piece = tid + 256 * i, t = piece / (vp / 8), d = (piece - t * (vp / 8)) * 8;
      *(u32x4*)(X + t * XS + d) = xr[i];
    }
#pragma unroll
    for (int i = 0; i < D; ++i) {
      const int piece = tid + 256 * i, t = piece / (dp / 8), d = (piece - t * (dp / 8)) * 8;
      *(u32x4*)(B + t * BS + d) = br[i];
    }
    if (!INC) {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int tile = wave + 4 * i, pt = tile % PT, nt = tile / PT, at = (16 * pt + r) * BS + 16 * nt + 4 * q;
        const u32x2 hi = {pack_bf16x2(S[i][0], S[i][1]), pack_bf16x2(S[i][2], S[i][3])};
        *(u32x2*)(Sh + at) = hi;
        *(u32x2*)(Sl + at) = u32x2{pack_bf16x2(S[i][0] - lo_bf(hi[0]), S[i][1] - hi_bf(hi[0])), pack_bf16x2(S[i][2] - lo_bf(hi[1]), S[i][3] - hi_bf(hi[1]))};
      }
#pragma unroll
      for (int i = 0; i < D; ++i) {
        const int piece = tid + 256 * i, t = piece / (dp / 8), d = (piece - t * (dp / 8)) * 8;
        *(u32x4*)(Q + t * QS + d) = qr[i];
      }
    }
    u32x4 zc[C];
    if (!INC)
#pragma unroll
      for (int i = 0; i < C; ++i) zc[i] = zr[i];
    if (tid < L) {
      float c = rate * dt_r;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const float up = __shfl_up(c, o, 64);
        if (lane >= o) c += up;
      }
      cum[tid] = c;
      dts[tid] = dt_r;
      ws[tid] = __builtin_amdgcn_exp2f(__shfl(c, 63, 64) - c) * dt_r;
    }
    __syncthreads();
    if (t0 + L < last) load(t0 + L);
    const float total = cum[L - 1];

    if (!INC && 16 * wave < n) {
      const int t = 16 * wave + r;
      const float ct = cum[t];
      bf16_t* G = Q + 16 * wave * QS;
      u32x4 qc[D];
#pragma unroll
      for (int s = 0; s < D; ++s) qc[s] = *(const u32x4*)(G + r * QS + 32 * s + 8 * q);
      wave_lds_order();
#pragma unroll
      for (int i = 0; i < C; ++i) {
        const int piece = lane + 64 * i;
        *(u32x4*)(G + piece / (vp / 8) * QS + piece % (vp / 8) * 8) = zc[i];
      }
      wave_lds_order();
      f32x4 o[PT];
#pragma unroll
      for (int i = 0; i < PT; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < D; ++s)
#pragma unroll
        for (int i = 0; i < PT; ++i) {
          o[i] = mfma(*(const u32x4*)(Sh + (16 * i + r) * BS + 32 * s + 8 * q), qc[s], o[i]);
          o[i] = mfma(*(const u32x4*)(Sl + (16 * i + r) * BS + 32 * s + 8 * q), qc[s], o[i]);
        }
      const float et = __builtin_amdgcn_exp2f(ct);
#pragma unroll
      for (int i = 0; i < PT; ++i) o[i] *= et;
#pragma unroll
      for (int b = 0; b < L / 32; ++b) {
        if (2 * b > wave) continue;
        float p[8];  // tokens 32 b + 4 q + j and 32 b + 16 + 4 q + j: the order of read_columns
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          const int sb = 2 * b + half;
          f32x4 acc = {0.f, 0.f, 0.f, 0.f};
          if (sb <= wave) {
#pragma unroll
            for (int s = 0; s < D; ++s) acc = mfma(*(const u32x4*)(B + (16 * sb + r) * BS + 32 * s + 8 * q), qc[s], acc);
          }
          const f32x4 cs = *(const f32x4*)(cum + 16 * sb + 4 * q), ds = *(const f32x4*)(dts + 16 * sb + 4 * q);
#pragma unroll
          for (int e = 0; e < 4; ++e) p[4 * half + e] = (sb <= wave && 16 * sb + 4 * q + e <= t) ? acc[e] * __builtin_amdgcn_exp2f(ct - cs[e]) * ds[e] : 0.f;
        }
        u32x4 ph, pl;
        split8(p, ph, pl);
#pragma unroll
        for (int i = 0; i < PT; ++i) {
          const u32x4 x = read_columns(X, XS, 32 * b, 16 * i, lane);
          o[i] = mfma(x, ph, o[i]);
          o[i] = mfma(x, pl, o[i]);
        }
      }
#pragma unroll
      for (int i = 0; i < PT; ++i) {
        bf16_t* at = G + r * QS + 16 * i + 4 * q;
        const f32x4 x = ld4(X + t * XS + 16 * i + 4 * q), zz = ld4(at);
        f32x4 y = o[i] + skip * x;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] *= silu_fast(zz[e]);
        st4(at, y);
      }
      wave_lds_order();
#pragma unroll
      for (int i = 0; i < C; ++i) {
        const int piece = lane + 64 * i, tz = piece / (vp / 8), d = piece % (vp / 8) * 8;
        if (16 * wave + tz < n)
          *(u32x4*)((bf16_t*)a.out + (int64_t)(row0 + t0 + 16 * wave + tz) * a.ldo + in_chunks(h * vp + d, a.out_chunk)) = *(const u32x4*)(G + tz * QS + d);
      }
    }

    const float keep = __builtin_amdgcn_exp2f(total);
    if (INC) total_log += total;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int pt = (wave + 4 * j) % PT;
      u32x4 xh[L / 32], xl[L / 32];
#pragma unroll
      for (int k = 0; k < L / 32; ++k) {
        const u32x4 x = read_columns(X, XS, 32 * k, 16 * pt, lane);
        const f32x4 w0 = *(const f32x4*)(ws + 32 * k + 4 * q), w1 = *(const f32x4*)(ws + 32 * k + 16 + 4 * q);
        const float v[8] = {lo_bf(x[0]) * w0[0], hi_bf(x[0]) * w0[1], lo_bf(x[1]) * w0[2], hi_bf(x[1]) * w0[3],
                            lo_bf(x[2]) * w1[0], hi_bf(x[2]) * w1[1], lo_bf(x[3]) * w1[2], hi_bf(x[3]) * w1[3]};
        split8(v, xh[k], xl[k]);
      }
#pragma unroll
      for (int i = j; i < NT; i += PER) {
        const int nt = (wave + 4 * i) / PT;
        S[i] *= keep;
#pragma unroll
        for (int k = 0; k < L / 32; ++k) {
          const u32x4 bb = read_columns(B, BS, 32 * k, 16 * nt, lane);
          S[i] = mfma(bb, xh[k], S[i]);
          S[i] = mfma(bb, xl[k], S[i]);
        }
      }
    }
  }
  float* to = INC ? seg : final ? slot : nullptr;
  if (to)
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int tile = wave + 4 * i, pt = tile % PT, nt = tile / PT;
      *(f32x4*)(to + (16 * pt + r) * dp + 16 * nt + 4 * q) = S[i];
    }
  if (INC && tid == 0) a.seg_decay[((int64_t)seq * a.n_seg + sg) * H + h] = total_log;
}

// grid (heads * vp * dp / 1024, sequences): what the segments add -> the states they start from
__global__ __launch_bounds__(256) void ssm_segments_kernel(const LmSsm a) {
  const int seq = blockIdx.y, per_head = a.vp * a.dp;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4, n_el = (int64_t)a.heads * per_head;
  if (i >= n_el) return;
  const int h = (int)(i / per_head), len = a.r.seq_row0[seq + 1] - a.r.seq_row0[seq], n = (len + a.seg_chunks * L - 1) / (a.seg_chunks * L);
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  if (a.r.seq_pos0[seq] > 0) S = *(const f32x4*)(a.state + (int64_t)a.r.seq_slot[seq] * n_el + i);
  for (int sg = 0; sg < n; ++sg) {
    float* p = a.seg + ((int64_t)seq * a.n_seg + sg) * n_el + i;
    f32x4 inc = {0.f, 0.f, 0.f, 0.f};
    float keep = 0.f;
    if (sg + 1 < n) {
      inc = *(const f32x4*)p;
      keep = __builtin_amdgcn_exp2f(a.seg_decay[((int64_t)seq * a.n_seg + sg) * a.heads + h]);
    }
    *(f32x4*)p = S;
    S = keep * S + inc;
  }
}

typedef void (*SsmKernel)(const LmSsm);
struct ChunkPick {
  SsmKernel run, inc;
  int lds;
};
template <int D, int C>
ChunkPick chunk_of() {
  return ChunkPick{ssm_chunk_kernel<D, C, false>, ssm_chunk_kernel<D, C, true>, (L * (32 * C + 8) + (L + 64 * C) * (32 * D + 8) + L * (32 * (D > C ? D : C) + 8)) * 2};
}
template <int D>
ChunkPick chunk_by_width(int c) {
  switch (c) {
    case 1: return chunk_of<D, 1>();
    case 2: return chunk_of<D, 2>();
    case 3: return chunk_of<D, 3>();
    case 4: return chunk_of<D, 4>();
    default: return ChunkPick{nullptr, nullptr, 0};
  }
}
ChunkPick chunk_pick(const LmSsm& a) {
  switch (a.dp / 32) {
    case 1: return chunk_by_width<1>(a.vp / 32);
    case 2: return chunk_by_width<2>(a.vp / 32);
    case 3: return chunk_by_width<3>(a.vp / 32);
    case 4: return chunk_by_width<4>(a.vp / 32);
    default: return ChunkPick{nullptr, nullptr, 0};
  }
}

// grid (heads, sequences).  Sixteen lanes per state row, sixteen rows at a time; the state is requested before anything else.
// The state's bytes bound it from about eight sequences on.  It is read and written once a step, past the caches (non-temporal, both): 40 sequences, 32 heads of 64 x 64,
// 12.2 -> 9.9 us (42 MB); 23, 64 of 64 x 128, 25.0 -> 20.2 us (96 MB, 4.8 TB/s); 8 of these 10.8 -> 8.9; one 6.3 and 6.4; 32 of 64 x 64, one 5.7 and 5.8.
// Either alone: stores 12.1 and 24.2 us, loads 11.8 and 23.0.
// C: vp / 32, E: passes of 64 state columns.  a.sumsq: rows are left before their norm, times its weights, with every head's sum of squares: the
// product behind takes the rows' factors, and there is no launch of one workgroup per row (4.8 us) between them.
template <int C, int E>
__global__ __launch_bounds__(256) void ssm_decode_kernel(const LmSsm a) {
  __shared__ __attribute__((aligned(16))) float us[32 * C + 2 * 64 * E];
  __shared__ float red[4];
  const int h = blockIdx.x, seq = blockIdx.y, tid = threadIdx.x, l = tid & 15, dp = a.dp, vp = 32 * C, H = a.heads, cw = a.cw(), g = h / (H / a.groups);
  const int row = a.r.seq_row0[seq], pos = a.r.seq_pos0[seq], slot = a.r.seq_slot[seq];
  float* st = a.state + ((int64_t)slot * H + h) * vp * dp;
  f32x4 S[2 * C][E];
#pragma unroll
  for (int i = 0; i < 2 * C; ++i)
#pragma unroll
    for (int k = 0; k < E; ++k) {
      const int d = 64 * k + 4 * l;
      S[i][k] = __builtin_nontemporal_load((const f32x4*)(st + (int64_t)((tid >> 4) + 16 * i) * dp + min(d, dp - 4)));
    }
  const bf16_t* p = (const bf16_t*)a.proj + (int64_t)row * a.ldp;
  const int mine = h * vp + min(tid, vp - 1);  // the output that this thread writes in the end
  const bf16_t z = p[a.col_z + mine];
  const float norm_w = a.sumsq ? a.out_norm[mine] : 1.0f;
  const bf16_t dt_in = p[a.col_dt + h];
  const float dt_bias = a.dt_bias[h], decay = a.decay[h], skip = a.skip[h];
  const bool shared_cols = h % (H / a.groups) == 0;  // the head of its group that also writes the ring's B and C columns
  bf16_t* ring = (bf16_t*)a.conv_state + (int64_t)slot * a.taps * cw;
  for (int i = tid * 4; i < vp + 2 * dp; i += 1024) {
    const int c = i < vp ? h * vp + i : i < vp + dp ? H * vp + g * dp + i - vp : H * vp + (a.groups + g) * dp + i - vp - dp;
    constexpr int AT_ONCE = 4;  // the newest taps: all their loads are requested before the first is used
    // (a branch for each would wait for each: rows before the sequence's first are read from somewhere else and not used)
    u32x2 raw[AT_ONCE];
    f32x4 x[AT_ONCE], w[AT_ONCE], y = *(const f32x4*)(a.conv_bias + c);
#pragma unroll
    for (int k = 0; k < AT_ONCE; ++k) {
      const bool in = k < a.taps && pos - k >= 0;
      raw[k] = *(const u32x2*)(k > 0 && in ? ring + (int64_t)((pos - k) % a.taps) * cw + c : p + a.col_x + c);
      w[k] = *(const f32x4*)(a.conv + (int64_t)(in ? a.taps - 1 - k : 0) * cw + c);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < AT_ONCE; ++k)
      x[k] = k < a.taps && pos - k >= 0 ? f32x4{lo_bf(raw[k][0]), hi_bf(raw[k][0]), lo_bf(raw[k][1]), hi_bf(raw[k][1])} : f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k = AT_ONCE; k < a.taps && pos - k >= 0; ++k) y += *(const f32x4*)(a.conv + (int64_t)(a.taps - 1 - k) * cw + c) * ld4(ring + (int64_t)((pos - k) % a.taps) * cw + c);
#pragma unroll
    for (int k = AT_ONCE - 1; k >= 0; --k) y += w[k] * x[k];
    // row pos % taps is read by no head of this step
    if (a.taps > 1 && (i < vp || shared_cols)) st4(ring + (int64_t)(pos % a.taps) * cw + c, x[0]);
#pragma unroll
    for (int e = 0; e < 4; ++e) us[i + e] = bf2f(f2bf(silu_f32(y[e])));  // as a prefill stores it
  }
  const float dt = softplus_f32(bf2f(dt_in) + dt_bias), keep = expf(-decay * dt);
#pragma unroll
  for (int i = 0; i < 2 * C; ++i)
#pragma unroll
    for (int k = 0; k < E; ++k)
      if (pos == 0 || 64 * k + 4 * l >= dp) S[i][k] = f32x4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();
  float* out = us;  // (only the x part: every row's x is read by its own sixteen lanes before they write)
#pragma unroll
  for (int i = 0; i < 2 * C; ++i) {
    const int e = (tid >> 4) + 16 * i;
    const float x = us[e], in = dt * x;
    float o = 0.f;
#pragma unroll
    for (int k = 0; k < E; ++k) {
      const int d = 64 * k + 4 * l;
      if (d < dp) {
        const f32x4 b = *(const f32x4*)(us + vp + d), c = *(const f32x4*)(us + vp + dp + d);
        const f32x4 s = keep * S[i][k] + b * in;
        __builtin_nontemporal_store(s, (f32x4*)(st + (int64_t)e * dp + d));
        o += s[0] * c[0] + s[1] * c[1] + s[2] * c[2] + s[3] * c[3];
      }
    }
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) o += __shfl_xor(o, m, 64);
    if (l == 0) out[e] = o + skip * x;
  }
  __syncthreads();
  const float v = tid < vp ? out[tid] * silu_f32(bf2f(z)) : 0.f;
  if (tid < vp) ((bf16_t*)a.out)[(int64_t)row * a.ldo + in_chunks(mine, a.out_chunk)] = f2bf(v * norm_w);
  if (!a.sumsq) return;
  const float ss = block_sum_256(v * v, red);
  if (tid == 0) a.sumsq[(int64_t)row * H + h] = ss;
}

template <int C>
SsmKernel decode_by_state(int dp) {
  return dp <= 64 ? ssm_decode_kernel<C, 1> : dp <= 128 ? ssm_decode_kernel<C, 2> : dp <= 256 ? ssm_decode_kernel<C, 4> : nullptr;
}
SsmKernel decode_pick(const LmSsm& a) {
  switch (a.vp / 32) {
    case 1: return decode_by_state<1>(a.dp);
    case 2: return decode_by_state<2>(a.dp);
    case 3: return decode_by_state<3>(a.dp);
    case 4: return decode_by_state<4>(a.dp);
    default: return nullptr;
  }
}

}  // namespace

md_status lm_ssm_plain(int dtype, const LmSsm& a, hipStream_t s) { return dtype == MD_DTYPE_F32 ? plain<float>(a, s) : plain<bf16_t>(a, s); }

// Segments: as many as keep to two workgroups per CU.  The increments cost half of the outputs, and they and the states two launches, about
// two chunks: one sequence of 700 tokens, 16 heads of 128 x 128: 11 segments of one chunk 30 us, 2 of six 76 us.
int lm_ssm_segments(int n_seq, int heads, int max_len, int* chunks) {
  const int n = (max_len + L - 1) / L, segs = 512 / (n_seq * heads), per = segs > 1 ? (n + segs - 1) / segs : n;
  *chunks = 3 * per + 4 < 2 * n ? per : n;
  return (n + *chunks - 1) / *chunks;
}
int lm_ssm_most_segments(int n_seq, int heads, int max_len) {
  const int64_t n = (max_len + L - 1) / L;
  return n > 1 ? (int)std::min(n_seq * n, (int64_t)(512 / heads)) : 0;
}
bool lm_ssm_mfma_takes(const LmSsm& a) { return chunk_pick(a).run != nullptr; }
md_status lm_ssm_mfma(const LmSsm& a, hipStream_t s) {
  const ChunkPick k = chunk_pick(a);
  if (!k.run) return MD_ERR_UNSUPPORTED;
  MD_TRY(conv<bf16_t>(a, s));
  const dim3 grid(a.heads, a.n_seg, a.r.n_seq);
  MD_TRY(md_ensure_dynamic_lds((const void*)k.run, k.lds));
  if (a.n_seg > 1) {
    MD_TRY(md_ensure_dynamic_lds((const void*)k.inc, k.lds));
    hipLaunchKernelGGL(k.inc, grid, dim3(256), k.lds, s, a);
    MD_TRY(md_launch_status());
    hipLaunchKernelGGL(ssm_segments_kernel, dim3((a.heads * a.vp * a.dp + 1023) / 1024, a.r.n_seq), dim3(256), 0, s, a);
    MD_TRY(md_launch_status());
  }
  hipLaunchKernelGGL(k.run, grid, dim3(256), k.lds, s, a);
  MD_TRY(md_launch_status());
  return norm<bf16_t>(a, true, s);
}

bool lm_ssm_decode_takes(const LmSsm& a) { return decode_pick(a) != nullptr; }
md_status lm_ssm_decode(const LmSsm& a, hipStream_t s) {
  hipLaunchKernelGGL(decode_pick(a), dim3(a.heads, a.r.n_seq), dim3(256), 0, s, a);
  MD_TRY(md_launch_status());
  return a.sumsq ? MD_OK : norm<bf16_t>(a, false, s);
}
