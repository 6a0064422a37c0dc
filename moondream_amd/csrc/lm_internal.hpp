// Internal interface between the translation units of the layered language models (not part of the C ABI).
#pragma once
#include "md_common.hpp"

#include <type_traits>

// ---- element access: the model's dtype in memory, fp32 in registers ---------------------------------------------------
__device__ __forceinline__ float ldf(const bf16_t* p) { return bf2f(*p); }
__device__ __forceinline__ float ldf(const float* p) { return *p; }
__device__ __forceinline__ void stf(bf16_t* p, float v) { *p = f2bf(v); }
__device__ __forceinline__ void stf(float* p, float v) { *p = v; }

// four consecutive elements (offset a multiple of 4)
__device__ __forceinline__ f32x4 ld4(const bf16_t* p) {
  const u32x2 q = *(const u32x2*)p;
  return f32x4{lo_bf(q[0]), hi_bf(q[0]), lo_bf(q[1]), hi_bf(q[1])};
}
__device__ __forceinline__ f32x4 ld4(const float* p) { return *(const f32x4*)p; }
// eight elements as they lie in memory (offset a multiple of 8), and their halves
struct Raw8f {
  f32x4 v[2];
};
__device__ __forceinline__ u32x4 ld8(const bf16_t* p) { return *(const u32x4*)p; }
__device__ __forceinline__ Raw8f ld8(const float* p) { return Raw8f{{ld4(p), ld4(p + 4)}}; }
__device__ __forceinline__ f32x4 half8(const u32x4& q, int h) { return f32x4{lo_bf(q[2 * h]), hi_bf(q[2 * h]), lo_bf(q[2 * h + 1]), hi_bf(q[2 * h + 1])}; }
__device__ __forceinline__ f32x4 half8(const Raw8f& q, int h) { return q.v[h]; }
__device__ __forceinline__ void st4(bf16_t* p, f32x4 v) { *(u32x2*)p = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])}; }
__device__ __forceinline__ void st4(float* p, f32x4 v) { *(f32x4*)p = v; }
__device__ __forceinline__ void st8(bf16_t* p, f32x4 a, f32x4 b) {
  *(u32x4*)p = u32x4{pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(b[0], b[1]), pack_bf16x2(b[2], b[3])};
}
__device__ __forceinline__ void st8(float* p, f32x4 a, f32x4 b) {
  st4(p, a);
  st4(p + 4, b);
}

// where column c lies in a row whose groups of 8 columns are `chunk` elements apart: 8 in plain rows, 8 * rows in the order of the matrix operand
// that the products of few rows read (gemm_step.hip)
__device__ __forceinline__ int in_chunks(int c, int chunk) { return (c >> 3) * chunk + (c & 7); }

typedef short s16x4 __attribute__((ext_vector_type(4)));
// Eight tokens of one column per lane from a row-major LDS tile: lane row q (lane / 16) gets tokens t0 + 4 q .. + 3 and t0 + 16 + 4 q .. + 3 of
// column c0 + lane % 16 (in a 16-lane group, lane i points at four columns of token i / 4 and receives four tokens of column i % 16).
__device__ __forceinline__ u32x4 read_columns(const bf16_t* tile, int stride, int t0, int c0, int lane) {
  const bf16_t* p = tile + (t0 + 4 * (lane >> 4) + ((lane & 15) >> 2)) * stride + c0 + 4 * (lane & 3);
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p + 16 * stride));
  const u32x2 lo = __builtin_bit_cast(u32x2, a), hi = __builtin_bit_cast(u32x2, b);
  return u32x4{lo[0], lo[1], hi[0], hi[1]};
}
// orders a wave's LDS accesses before against those behind, also between its lanes (they are carried out in order)
__device__ __forceinline__ void wave_lds_order() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float silu_f32(float z) { return z / (1.0f + expf(-z)); }
template <typename T>
__device__ __forceinline__ float silu_for(float z) {
  return std::is_same<T, float>::value ? silu_f32(z) : silu_fast(z);
}

// sum over the 16 lanes of a row; every lane gets it (vector instructions only)
__device__ __forceinline__ float row_sum_16(float v) {
  auto turned = [](float x, auto by) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + decltype(by)::value, 0xf, 0xf, false)); };
  v += turned(v, std::integral_constant<int, 8>{});
  v += turned(v, std::integral_constant<int, 4>{});
  v += turned(v, std::integral_constant<int, 2>{});
  v += turned(v, std::integral_constant<int, 1>{});
  return v;
}

// sum over a workgroup of N waves; every thread gets it.  red: N floats of LDS.
template <int N>
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  __syncthreads();  // red may still be read from the previous call
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = red[0];
#pragma unroll
  for (int i = 1; i < N; ++i) v += red[i];
  return v;
}
__device__ __forceinline__ float block_sum_256(float v, float* red) { return block_sum<4>(v, red); }

typedef __bf16 md_bf16x8v __attribute__((ext_vector_type(8)));  // what the gfx950 MFMA builtins take
__device__ __forceinline__ md_bf16x8v op(const u32x4& v) { return __builtin_bit_cast(md_bf16x8v, v); }
__device__ __forceinline__ f32x4 mfma(const u32x4& a, const u32x4& b, const f32x4& c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(op(a), op(b), c, 0, 0, 0); }
// fp32 as the sum of two bf16 (16 mantissa bits)
__device__ __forceinline__ void split8(const float (&v)[8], u32x4& hi, u32x4& lo) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    hi[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
    lo[i] = pack_bf16x2(v[2 * i] - lo_bf(hi[i]), v[2 * i + 1] - hi_bf(hi[i]));
  }
}

// ---- cache layout: keys and values in the order the matrix instructions take them -------------------------------------------
// A slot is a run of blocks of 32 positions, each holding all heads one after the other (a workgroup that reads all heads of a tile
// reads consecutive memory).  A head's keys of a block: pieces of 16 keys x 32 coordinates, 512 elements each, laid out
// [coordinate / 8][key][8 coordinates]: lane l of a 16x16x32 product reads elements 8 l .. 8 l + 7.  Its values: pieces of 32 keys x 16
// coordinates, [key / 8][coordinate][8 keys], read the same way.
__device__ __forceinline__ int64_t key_block(int j, int g, int G, int dp) { return ((int64_t)(j >> 5) * G + g) * (32 * dp); }
__device__ __forceinline__ int64_t key_index(int j, int g, int d, int G, int dp) {
  return key_block(j, g, G, dp) + (((j >> 4) & 1) * (dp >> 5) + (d >> 5)) * 512 + ((d >> 3) & 3) * 128 + (j & 15) * 8 + (d & 7);
}
__device__ __forceinline__ int64_t value_index(int j, int g, int e, int G, int vp) {
  return key_block(j, g, G, vp) + (e >> 4) * 512 + ((j >> 3) & 3) * 128 + (e & 15) * 8 + (j & 7);
}

// ---- a mixer's launch description ---------------------------------------------------------------------------------------
struct LmRows {
  int n_seq, n_rows, max_len, max_ctx;
  const int32_t *row_seq, *row_pos, *seq_row0, *seq_pos0, *seq_slot;
};

struct LmAttn {
  LmRows r;
  const void* proj;  // [n_rows][ldp]: the projection (bias added), before the convolution
  int64_t ldp;
  int col_q, col_k, col_v;
  int heads, kv_heads, dim, vdim, dp, vp;  // dp, vp: padded head sizes
  int taps;
  const float *conv, *q_norm, *k_norm;
  int conv_ld;  // = in.n_pad
  int value_norm;
  float eps, scale;
  const float *slope, *mix;
  int chunk;
  int own_kv;      // this layer writes its keys and values
  void *k, *v;     // slabs read (and, with own_kv, written)
  void* conv_state;
  int ctx;
  void* q;         // [n_rows][heads * dp]: normed queries
  void* out;       // in_chunks(column, out_chunk) of rows ldo apart
  int64_t ldo;
  int out_chunk;
  float* part;     // split keys: partial (m, l) and accumulators
  int n_split, split_keys;
  int order;       // of the tiles of a matrix-core prefill (attention_talk.hip)
};

struct LmRet {
  LmRows r;
  const void* proj;
  int64_t ldp;
  int col_q, col_k, col_v, col_g;
  int heads, dim, vdim, dp, vp;
  float eps, scale;
  const float *decay, *rope;
  int rot_dims;
  float* state;    // [slots][heads][vp][dp]
  void* out;
  int64_t ldo;
  int out_chunk;
  float *qf, *kf;  // plain kernels: rotated q and k, [n_rows][heads * dp]
  float* of;       // plain kernels: unnormed outputs, [n_rows][heads * vp]
  float* seg;      // matrix-core prefill in more segments than one: increments of chunks, states that segments start from (retention.hip)
  int n_seg, seg_chunks;  // segments per sequence, their length in chunks
};

struct LmLatent {
  LmRows r;
  const void* proj;      // [n_rows][ldp]
  int64_t ldp;
  int col_q, col_c, col_g;  // col_g < 0: no output gate
  int heads, dim, vdim, dp, vp, rank, rp;
  float eps, scale;
  const float* norm;     // [rp]
  const void* up_k_t;    // [heads][rp][dp]
  md_linear up_kv;       // rows: keys of every head | values of every head
  void* cache;           // [slots][ctx][rp]
  int ctx;
  void* out;
  int64_t ldo;
  int out_chunk;
  // prefill on the matrix cores: latent rows of every position of the step's sequences, packed by seq_ctx0, and what they expand to
  int ctx_rows;
  const int32_t* seq_ctx0;
  void *c_rows, *kv;     // [ctx_rows][rp], [ctx_rows][up_kv.n_pad]
  // decode: queries in the latent space, and the splits' partial sums
  void* q_lat;           // [n_seq][heads][rp]
  float* part;
  int n_split;
};

struct LmSsm {
  LmRows r;
  const void* proj;      // [n_rows][ldp]
  int64_t ldp;
  int col_z, col_x, col_b, col_c, col_dt;  // x | B | C are adjacent
  int heads, groups, dim, vdim, dp, vp, taps, norm_groups;
  const float *conv, *conv_bias, *dt_bias, *decay, *skip, *out_norm;
  float eps;
  void* conv_state;      // [slots][taps][cw]
  float* state;          // [slots][heads][vp][dp]
  void* out;
  int64_t ldo;
  int out_chunk;
  float* sumsq;          // decode: [n_rows][heads], rows before their norm; nullptr: normed rows
  void* u;               // [n_rows][cw]: x | B | C behind the convolution and silu
  float* dt;             // [n_rows][heads], behind softplus
  float *seg, *seg_decay;  // matrix-core prefill in segments: [n_seq][n_seg][heads][vp][dp], [n_seq][n_seg][heads]
  int n_seg, seg_chunks;
  __host__ __device__ int cw() const { return heads * vp + 2 * groups * dp; }
};

// a sublayer result that the next row-wise step adds to the residual stream(s): rows of the model's dtype, or K-slice partial products
// (slices > 0); top > 0: per row the weighted sum of `top` of the rows
struct LmAddend {
  const void* src;       // nullptr: nothing pending
  int64_t ld, slice_stride;
  int slices, top;
  const int32_t* slot_of;  // [rows][top]; nullptr: src is in the order of the choices
  const float* weight;     // [rows][top]
};

struct LmStreams {
  float* x;              // [streams][rows][width_pad], `stride` floats apart
  int64_t stride;
  int streams;
  LmAddend add;
  const float* prev;     // in | out | mix weights around the sublayer that made `add`; nullptr: plain residual sum
  const float* next;     // in weights of the sublayer that reads y; nullptr: all ones
  md_rms_weight w;
  float eps;
  int width, width_pad;
  void* y;               // [.][width_pad] normed rows, or nullptr
  float* sum_out;        // optional: the weighted sum before the norm, fp32
  const int32_t* rows_idx;
  int write_x;
  // lm_stream_split: y = the weighted sum times its norm weight, in chunks of columns; the rows' factors are left to who reads it, with these sums
  int out_chunk;
  float* sumsq_out;      // [rows][width_pad / 8]
};

struct LmRoute {
  const void* h;         // [rows][k_pad]
  int rows, k_pad, experts, top;
  const void* router;    // [.][k_pad]
  const float* bias;
  int32_t* chosen;       // [rows][top]
  float* weight;         // [rows][top]
  // rows before their norm: sums of squares (LmStepGemm), and where to leave the rows' factors; nullptr: normed rows
  const float* sumsq;
  int sumsq_n, width;
  float eps;
  float* factor;         // [rows]
  // rows sorted by expert: slots offsets[e] .. offsets[e + 1] - 1 belong to expert e
  int32_t *offsets, *row_of, *slot_of;  // [experts + 1], [rows * top], [rows][top]; nullptr: not wanted
};

// A product of a step of few rows and what follows it (gemm_step.hip).  Rows that a residual epilogue wrote carry no norm factor: it
// comes from their sums of squares (sumsq; nullptr: the rows are complete).
// Up to how many rows they are ahead of the tile products and row-wise launches.  24 layers, 2048 wide, 20 / 28 / 32 / 40 / 48 rows: 0.81 / 0.81 / 0.84 / 0.90 /
// 0.94 of a step's time with state space and latent attention (1301, 1409, 1469, 1614, 1729 us with 32 heads of 64; 0.81 to 0.92 with 16 of 128), 0.84 /
// 0.83 / 0.81 / 0.86 / 0.89 with attention and retention (1431, 1531, 1593, 1734, 1857 us); at 64 rows gates would take 18.2 us against 16.3.  Every
// workgroup reads all rows, so their share grows with the width, and from 2048 columns on there is more than one workgroup of the residual product per CU.
// Four layers, 24 / 32 / 33 / 48 rows: 2560 wide 0.80 / 0.97 / 1.05 / 1.10, 3072 wide 0.80 / 0.96 / 1.01 / 1.10, 3584 wide 0.83 / 1.01 / 1.15 / 1.24, 4096
// wide 0.75 / 0.92 / 1.00 / 1.08, 5120 wide 0.80 / 1.12 / 1.28 / 1.38.
constexpr int LM_STEP_ROWS = 48;
inline int lm_step_most_rows(int width_pad) { return width_pad <= 2048 ? LM_STEP_ROWS : width_pad <= 4096 ? 32 : 28; }
struct LmStepGemm {
  const bf16_t* a;       // row m's columns 8 c .. 8 c + 7 at m * lda + c * chunk (plain rows: chunk 8)
  int64_t lda;
  int chunk;
  const bf16_t* w;       // [.][k]
  int k, rows;
  const int32_t* rows_idx;  // which rows of a (nullptr: 0, 1, ..); not for the residual epilogue
  const float* sumsq;    // [.][sumsq_n] partial sums of squares of the rows of a before their norm
  int sumsq_n;
  float eps;
  int width;             // that the mean of squares is over
  bf16_t* out;           // rows: [rows][ldo]; otherwise in_chunks(column, out_chunk) of rows ldo apart; residual: the next sublayer's input times its norm weight
  int64_t ldo;
  int out_chunk;
  const bf16_t* bias;
  int n, ff_pad;         // columns of the result; SiLU gate: rows 0 .. of w are the gates, ff_pad .. the inputs
  // residual epilogue: streams, weights around this sublayer and of the next one (nullptr: plain sum), as in LmStreams
  float* x;
  int64_t stride;
  int streams, width_pad;
  const float *prev, *next;
  md_rms_weight norm;
  float* sumsq_out;      // [rows][width_pad / 8]
  // ... of rows of a before a norm over `normed` elements: [rows][heads] sums of squares; nullptr: complete rows
  // groups (2, 4, 8) of as many heads each: heads % 8 == 0, k / 64 a multiple of 8 and all of it theirs
  const float* head_sumsq;
  int heads, groups, normed;
};
md_status lm_step_rows(const LmStepGemm& a, int n, hipStream_t s);   // out = a w^T + bias
md_status lm_step_silu(const LmStepGemm& a, hipStream_t s);          // out = silu(gate) * input
md_status lm_step_resid(const LmStepGemm& a, hipStream_t s);         // streams += a w^T; out and sumsq_out for the next product

// A product of the rows of a step with the matrices of the experts that they chose (gemm_experts.hip): choice i = k-th expert of row i / top
constexpr int LM_EXPERT_CHOICES = 1024;
struct LmExpertGemm {
  const bf16_t* a;       // choice i reads row i / per
  int64_t lda;
  int a_rows, per;
  const bf16_t* w;       // [expert][.][k]
  int64_t expert_stride;
  int k, experts;
  const int32_t* chosen;  // [n]
  int n;                 // choices
  int ff_pad;            // SiLU gate: rows 0 .. of a matrix are the gates, ff_pad .. the inputs
  const float* factor;   // SiLU gate: of the rows of a, nullptr: ones
  void* out;             // [n][ldo], in the order of the choices
  int64_t ldo;
};
bool lm_expert_step_takes(int rows, int top, int experts);
md_status lm_expert_silu(const LmExpertGemm& a, hipStream_t s);          // out (bf16) = silu(gate) * input
md_status lm_expert_rows(const LmExpertGemm& a, int n, hipStream_t s);   // out (fp32) = a w^T, n columns

// dtype: MD_DTYPE_*
md_status lm_embed_streams(const md_lm_model* m, const int32_t* tokens, const int32_t* row_pos, float* x, int64_t stride, int rows, hipStream_t s);
md_status lm_stream_step(int dtype, const LmStreams& a, int rows, hipStream_t s);
md_status lm_stream_split(const LmStreams& a, int rows, hipStream_t s);  // bf16

md_status lm_latent_plain(int dtype, const LmLatent& a, hipStream_t s);  // any dtype and sizes
bool lm_latent_mfma_takes(const LmLatent& a);
md_status lm_latent_mfma(const LmLatent& a, hipStream_t s);              // bf16 prefill (the caller's GEMM expands the latent rows in between)
md_status lm_latent_rows(int dtype, const LmLatent& a, bool pack, hipStream_t s);  // norm, cache rows; pack: c_rows of the whole context
bool lm_latent_decode_takes(const LmLatent& a);
int lm_latent_decode_splits(int n_seq, int heads, int max_keys);
size_t lm_latent_decode_part_floats(int n_seq, int n_split, int heads, int rp);
md_status lm_latent_decode(const LmLatent& a, hipStream_t s);            // bf16 decode step in the latent space

md_status lm_ssm_plain(int dtype, const LmSsm& a, hipStream_t s);
bool lm_ssm_mfma_takes(const LmSsm& a);
constexpr int LM_SSM_CHUNK = 64;
int lm_ssm_segments(int n_seq, int heads, int max_len, int* chunks);     // segments per sequence that fill the chip, chunks of each
int lm_ssm_most_segments(int n_seq, int heads, int max_len);  // segments that need memory, of all sequences, of steps up to that length
md_status lm_ssm_mfma(const LmSsm& a, hipStream_t s);                    // bf16 prefill, chunked on the matrix cores
bool lm_ssm_decode_takes(const LmSsm& a);
md_status lm_ssm_decode(const LmSsm& a, hipStream_t s);                  // bf16 decode step

md_status lm_route(int dtype, const LmRoute& a, hipStream_t s);          // router, choice, weights, rows by expert
// C[slot] = A[row of slot] W_e^T for the slots of every expert e; lin: one expert's matrix, all follow one another
md_status lm_grouped_gemm_f32(const void* a, int64_t lda, const int32_t* row_of, const md_linear& lin, int experts, const int32_t* offsets, void* c,
                              int64_t ldc, int slots, bool chain, hipStream_t s);
// md_gemm_f32, the order of sums chosen (gemm_f32.hip)
md_status lm_gemm_f32(const void* a, int64_t lda, const md_linear& lin, void* c, int64_t ldc, int rows, bool chain, hipStream_t s);

// dtype: MD_DTYPE_*
md_status lm_embed(int dtype, const void* table, int64_t ld, const int32_t* tokens, float* x, int rows, int vocab, hipStream_t s);
// x[row] += src (rows of the model's dtype, or nullptr); y = rms_norm(x) * w.  rows_idx: optional gather for y-only use (x is then
// not written back).
md_status lm_resid_norm(int dtype, float* x, int64_t ldx, const void* src, int64_t lds, const md_rms_weight& w, float eps, int width,
                        int width_pad, void* y, int64_t ldy, const int32_t* rows_idx, bool write_x, int rows, hipStream_t s);
// the same with src = K-slice partial products (fp32 [slices][rows][ldp])
md_status lm_reduce_resid_norm(float* x, int64_t ldx, const float* part, int slices, int64_t ldp, int64_t slice_stride,
                               const md_rms_weight& w, float eps, int width, int width_pad, void* y, int64_t ldy, const int32_t* rows_idx,
                               bool write_x, int rows, hipStream_t s);
// act = silu(gate) * up over [gate | up] rows: fp32 products, and those with a bias
md_status lm_silu_mul(int dtype, const void* gu, int64_t ldg, void* act, int64_t lda, int rows, int ff_pad, hipStream_t s);
md_status lm_reduce_silu_mul(const float* part, int slices, int64_t ldp, int64_t slice_stride, void* act, int64_t lda, int rows, int ff_pad,
                             hipStream_t s);

// out = sum of K-slice partial products + bias (bf16 rows)
md_status lm_reduce_rows(const float* part, int slices, int64_t ldp, int64_t slice_stride, const void* bias, void* out, int64_t ldo, int rows, int n,
                         hipStream_t s);

md_status lm_attn_prep(int dtype, const LmAttn& a, hipStream_t s);      // convolution, norms, cache rows, convolution state
md_status lm_attn_plain(int dtype, const LmAttn& a, hipStream_t s);     // one workgroup per query row, any dtype
// bf16 prompts of up to 978 keys and 40 million scores, scores through memory: lm_attn_prep and the rest (span: most keys of a query)
bool lm_attn_pairs_takes(const LmAttn& a, int span);
size_t lm_attn_pairs_floats_most(int n_rows, int n_seq, int span, int heads, int dp, int vp);  // of steps up to that size
md_status lm_attn_pairs(const LmAttn& a, int span, hipStream_t s);
bool lm_attn_mfma_takes(const LmAttn& a);
int lm_attn_mfma_parts(const LmRows& r, int ctx_rows, int span, int heads, int vp, int* split_keys);
size_t lm_attn_mfma_part_floats_most(int n_rows, int n_seq, int span, int heads, int vp);  // floats that the parts of steps up to that size take at most
md_status lm_attn_mfma(const LmAttn& a, hipStream_t s);                 // bf16 prefill on the matrix cores
int lm_attn_decode_splits(int n_seq, int max_keys, int* split_keys);
size_t lm_attn_decode_part_floats(int n_seq, int n_split, int heads, int vp);
bool lm_attn_decode_takes(const LmAttn& a);
md_status lm_attn_decode(const LmAttn& a, hipStream_t s);               // bf16 decode step: prep + split-key attention + combine
// ... of heads with keys of their own, in two launches (span: most keys of a query)
bool lm_attn_heads_takes(const LmAttn& a, int span);
size_t lm_attn_heads_floats(int n_seq, int span, int heads, int kv_heads, int dp, int vp, int taps, bool own_kv);
md_status lm_attn_heads(const LmAttn& a, int span, hipStream_t s);

md_status lm_ret_plain(int dtype, const LmRet& a, hipStream_t s);
constexpr int LM_RET_CHUNK = 64;
int lm_ret_segments(int n_seq, int heads, int dp, int vp, int max_len, int* chunks);  // as lm_ssm_segments
int lm_ret_most_states(int n_seq, int heads, int dp, int vp, int max_len);  // that any step of up to so many sequences and tokens keeps in memory
bool lm_ret_mfma_takes(const LmRet& a);
md_status lm_ret_mfma(const LmRet& a, hipStream_t s);                   // bf16 prefill, chunked on the matrix cores
bool lm_ret_decode_takes(const LmRet& a);
md_status lm_ret_decode(const LmRet& a, hipStream_t s);                 // bf16 decode step

md_status md_argmax_advance(const void* logits, int64_t ld, int32_t batch, int32_t vocab, int32_t suppress_id, int32_t* next, int32_t* pos,
                            hipStream_t stream);
md_status md_argmax_advance_f32(const void* logits, int64_t ld, int32_t batch, int32_t vocab, int32_t suppress_id, int32_t* next,
                                int32_t* pos, hipStream_t stream);
