// Internal interface between the GEMM translation units (not part of the C ABI).
#pragma once
#include "md_common.hpp"

// One launch of  C = epilogue(A . W^T + b)  as the kernels see it.
struct GemmK {
  const bf16_t* A;
  const bf16_t* W;
  const bf16_t* bias;
  const bf16_t* R;
  bf16_t* C;
  int64_t lda, ldw, ldc, ldr;
  int M, n_store, n_pad, K;
  int tiles_m, tiles_n;
  int res_row_mod;
  int group_m;    // tile-order grouping (row panels per group)
  int gelu_from;  // EPI_GELU: columns >= gelu_from get the GELU
  int nt;         // decode regime: stream the weights with the non-temporal policy
  // launch-boundary split-K: every K slice stores its fp32 partial tile [slice][m][ldp] and exits;
  // the consumer kernel sums the slices (md_reduce_residual_layernorm)
  float* partial;
  int64_t partial_ld, partial_slice_stride;
  // split-K (decode regime only): K slices per output tile, fp32 slabs, arrival tickets
  int slices;
  float* slabs;
  unsigned* tickets;
  // MD_EPI_QKV_ROPE (four-wave kernel only): the decoder prefill's fused [q | k | v | gelu(fc1)] layer with the partial RoPE
  // (rope.py:20-48) and the KV-cache update (text.py:45-46, moondream.py:74-78) applied in the epilogue
  const float* rope_cs = nullptr;      // fp32 [M][32]: (cos, sin) of the row's position for the 16 rotated pairs
  const uint32_t* rope_kv = nullptr;   // [M]: byte offset of (slot, position) in a layer's K / V slab
  bf16_t* kslab = nullptr;
  bf16_t* vslab = nullptr;
  uint32_t slab_bytes = 0;             // bytes of one layer's K (= V) slab
  int rope_d = 0;                      // n_heads * 64: width of each of the q, k, v sections
  int rope_ctx = 0;                    // cache positions per head
  // grouped products (md_gemm_grouped_bf16): rows of A / C are slots, offsets[g] .. offsets[g + 1] - 1 belong to group g, whose matrix
  // begins at W + g * group_stride; slot s reads row row_of[s] of A (nullptr: row s)
  const int32_t* offsets = nullptr;
  const int32_t* row_of = nullptr;
  int groups = 0;
  int64_t group_stride = 0;
  int round_first = 0;  // MD_EPI_SILU: gate and input are rounded to bf16 before they are multiplied (more than 128 rows), or not
};

// Row tiles of a grouped product: every group has its own ceil(rows / bm) tiles.  How many a launch needs at most, and which group and rows
// tile `index` is (false: there are fewer tiles).  One wave-wide prefix sum per 64 groups; uniform per workgroup.
inline int grouped_tiles(int slots, int groups, int bm) {
  const int n = slots / bm + groups;
  return n < slots ? n : slots;
}
__device__ __forceinline__ bool grouped_tile(const int32_t* offsets, int groups, int bm, int index, int& group, int& first, int& end) {
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int g0 = 0; g0 < groups; g0 += 64) {
    const int g = g0 + lane, lo = g < groups ? offsets[g] : 0, hi = g < groups ? offsets[g + 1] : 0, tiles = (hi - lo + bm - 1) / bm;
    int run = tiles;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(run, o, 64);
      if (lane >= o) run += up;
    }
    const int mine = index - before - (run - tiles);  // index of the tile within this lane's group
    const unsigned long long b = __ballot(mine >= 0 && mine < tiles);
    if (b) {
      const int l = __ffsll((unsigned long long)b) - 1;
      group = __builtin_amdgcn_readfirstlane(g0 + l);
      first = __builtin_amdgcn_readfirstlane(__shfl(lo + mine * bm, l, 64));
      end = __builtin_amdgcn_readfirstlane(__shfl(hi, l, 64));
      return true;
    }
    before += __shfl(run, 63, 64);
  }
  return false;
}

// row tiles that the groups have
__device__ __forceinline__ int grouped_total(const int32_t* offsets, int groups, int bm) {
  const int lane = threadIdx.x & 63;
  int n = 0;
  for (int g = lane; g < groups; g += 64) n += (offsets[g + 1] - offsets[g] + bm - 1) / bm;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
  return __builtin_amdgcn_readfirstlane(n);
}

// C[s] = A[row_of[s]] . W_g^T for the slots s of every group g (bf16; lin: one group's matrix, n == n_pad, all follow one another).
// silu: the matrix is [gate | input], C[s] = silu(gate) * input
md_status md_gemm_grouped_bf16(const void* a, int64_t lda, const int32_t* row_of, const md_linear& lin, int groups, const int32_t* offsets, void* c,
                               int64_t ldc, int slots, bool silu, bool round_first, hipStream_t stream);
// C = silu(gate) * input of A . [gate | input]^T in one launch (bf16; n == n_pad, no bias)
md_status md_gemm_silu_bf16(const void* a, int64_t lda, const md_linear& lin, void* c, int64_t ldc, int rows, hipStream_t stream);
// the same as fp32 K-slice partial products [slice][slot][ld] (few rows per group)
int md_gemm_grouped_slices(const md_linear& lin, int groups, int slots);
size_t md_gemm_grouped_most(const md_linear& lin, int groups, int slots);  // floats that those of up to that many slots take at most
md_status md_gemm_grouped_partial(const void* a, int64_t lda, const int32_t* row_of, const md_linear& lin, int groups, const int32_t* offsets, float* partial,
                                  int64_t ld, int64_t slice_stride, int slots, hipStream_t stream);
// K-slice partial products of any number of rows: how many slices pay (0: a whole product is faster), and the launch
int md_gemm_partial_count(const md_linear& lin, int rows);
size_t md_gemm_partial_most(const md_linear& lin, int rows);  // floats that the partial products of up to that many rows take at most
md_status md_gemm_partial_rows(const void* a, int64_t lda, const md_linear& lin, int rows, int slices, float* partial, int64_t ld_partial,
                               int64_t slice_stride, hipStream_t stream);
constexpr int MD_EPI_QKV_ROPE = 3;     // internal to the library (md_gemm_qkv_rope)
constexpr int MD_EPI_SILU = 4;         // internal: columns are [gate | input], C = silu(gate) * input, half as wide

// The fused layer of a decoder block at prefill with RoPE + KV write in its epilogue, when the four-wave kernel takes the
// shape (MD_ERR_UNSUPPORTED otherwise: the caller runs md_gemm_bf16 + md_rope_kv_write).  MHA, head_dim 64, rot_dim 32.
struct md_rope_fuse {
  const float* row_cs;
  const uint32_t* row_kv;
  void* kslab;
  void* vslab;
  uint64_t slab_bytes;
  int n_heads, ctx;
};
md_status md_gemm_qkv_rope(const md_gemm_args* a, const md_rope_fuse* rf, hipStream_t stream);
// the same for the opt-in FP8 mode's tile GEMM (gemm_f8.hip); rf8 (or its slabs) may be null: no e4m3 copy of the cache
struct md_rope_fuse_f8 {
  void* k8slab;
  void* v8slab;
  float k_scale, v_scale;
};
int md_gemm_auto_group_m(int n_store);  // tile-order grouping by shape (gemm_bf16.hip): round 3's rule (eight-wave kernels, fp8 kernel)
int md_gemm_auto_group_m_w4(int n_store, int k);  // the four-wave kernel's, re-swept in round 4
bool md_gemm_knob_rope_fuse();  // MD_ROPE_FUSE / md_gemm_set_tuning("rope_fuse"): A/B and tests
md_status md_gemm_f8_qkv_rope(const md_gemm_f8_args* a, const md_rope_fuse* rf, const md_rope_fuse_f8* rf8, hipStream_t stream);

// gemm_w4.hip: the 256x256 tile kernel with one wave per SIMD (4 waves x 128x128), persistent.
// epi = MD_EPI_*.  Fills tiles_m / tiles_n itself.
md_status md_gemm_w4_launch(const GemmK& k, int epi, hipStream_t stream);
md_status md_gemm_w4_launch_grouped(const GemmK& k, int epi, hipStream_t stream);  // k.offsets: bias-free rows or MD_EPI_SILU
bool md_gemm_w4_takes(const GemmK& k, int epi);  // shape limits of the four-wave kernel for this launch
// gemm_mid.hip: tiles of bm (256 or 128) x 128, and fp32 sums of k.slices slices of K by 128 x 128 (k.partial); the bits of the four-wave kernel
md_status md_gemm_mid_launch(const GemmK& k, int epi, int bm, hipStream_t stream);
md_status md_gemm_mid_launch_grouped(const GemmK& k, int epi, int bm, hipStream_t stream);  // k.offsets: bias-free rows or MD_EPI_SILU
md_status md_gemm_mid_partial(const GemmK& k, hipStream_t stream);
void md_gemm_w4_set_grid(int v);     // persistent workgroups per launch of the four-wave kernel (0 = one per CU)
void md_gemm_w4_set_debug(int half, uint32_t v);  // measurement builds: device buffer for in-kernel stamps
void md_gemm_w4_set_variant(int v);  // measurement hook: schedule / ablation variant of the bias-epilogue kernel
__attribute__((weak)) void md_attention_set_skip_dead(int v);  // absent from the language-model build of the library; attention.hip: exact work skipping of the prefill kernel (bit 0: dead half of the last key tile, bit 1: waves without a live query row)
