// bf16 products of a few hundred to a few thousand rows:  C = epilogue(A . W^T + b)  where 256 x 256 tiles leave CUs without work.
//
// A workgroup owns one BM x BN tile, or a slice of its K.  K is walked in slices of 64, copied to an LDS ring of S stages by LDS-DMA (rows of 128
// bytes, 16-byte piece c of row r at piece c ^ (r >> 1 & 7), so that the 16 rows of an operand read meet 16 different banks).  A wave holds the
// operands of TWO slices in registers: those of slice t + 1 are read while slice t is multiplied, so no product waits for LDS, the barrier of
// a slice only says that the next one has landed, and a stage is free for the DMA one slice earlier than where operands are read just ahead of their use.
// What bounds it is the LDS port: DMA writes (64 bytes a clock) and operand reads (about 225) do not overlap; products of 64 x 64 per wave need 1.3
// times the clocks of their matrix instructions.
//
// 16x16x32 products, K in order: the bits are those of the 256 x 256 kernel (gemm_w4.hip), whatever the tile.
//
// Measured, weights from memory, against 256 x 128 tiles with operands read just ahead of their use: 700 rows, 10880 columns, K 2048: 40 -> 35 us; 2322 rows, 2048
// columns, K 5440 70 -> 63; 1458 x 3456, K 1152 18.8 -> 17.6.  Against 256 x 256: 2940 rows, 2048 columns, K 2048 / 8192 43 / 169 -> 29 / 102 us.  128 x 128 in two slices of K, 700
// rows, 2048 columns, K 5440: 31 -> 27 (half of that the order of the tiles: an XCD read three quarters of the weights).  One more wave that asks for the
// weights' lines ahead of the ring: K 8192 38.5 -> 36.9, K 2048 20.0 -> 21.3; four waves of 128 x 64: registers are copied.
#include "gemm_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int BK = 64;

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// not tracked by the compiler: wait_lds() before use
template <int OFF>
__device__ __forceinline__ void lds_read(bf16x8& dst, uint32_t addr) {
  static_assert(OFF >= 0 && OFF < 65536, "offset field");
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "i"(OFF));
}

// PART: fp32 sums of a slice of K -> p.partial.  EPI as in gemm_bf16.hip; SiLU: a wave's 64 columns are 32 gates and their inputs
// GRP: a grouped product (GemmK.offsets): a tile's rows are slots of one group, gathered through row_of, its matrix is that group's
template <int BM, int BN, int WM, int WN, int S, int EPI, bool PART, bool GRP>
__global__ __launch_bounds__(WM * WN * 64, 1) void gemm_mid_kernel(const GemmK p) {
  constexpr int NT = WM * WN * 64, TM = BM / WM, TN = BN / WN, MI = TM / 16, NI = TN / 16;
  constexpr int A_BYTES = BM * 128, STAGE = (BM + BN) * 128;
  constexpr int NA = BM * 8 / NT, NB = BN * 8 / NT, P = NA + NB;  // DMA pieces per thread and slice
  static_assert(BM * 8 % NT == 0 && BN * 8 % NT == 0 && TN == 64 && TM % 32 == 0 && S >= 3 && (S - 1) * P < 64, "tile");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WN, wn = wave % WN;

  // slices of K apart, then a run of tiles per XCD, group_m row panels of a column panel after the other
  const int tiles = (GRP ? grouped_total(p.offsets, p.groups, BM) : p.tiles_m) * p.tiles_n;
  if (GRP && (int)blockIdx.x >= tiles) return;  // (a grouped launch knows an upper bound)
  const int L0 = xcd_remap(blockIdx.x, tiles * p.slices);
  const int slice = PART ? L0 / tiles : 0, L = PART ? L0 - slice * tiles : L0;
  int m0, n0, m_end = p.M, group = 0;  // m_end: rows from there on belong to another group, or to nobody
  if constexpr (GRP) {
    // a row panel's columns after one another: few panels share weights, all of a panel's tiles its rows
    if (!grouped_tile(p.offsets, p.groups, BM, L / p.tiles_n, group, m0, m_end)) return;
    n0 = L % p.tiles_n * BN;
  } else {
    const int per_group = p.group_m * p.tiles_n, first_m = L / per_group * p.group_m, gsz = min(p.tiles_m - first_m, p.group_m);
    m0 = (first_m + L % per_group % gsz) * BM;
    n0 = L % per_group / gsz * BN;
  }

  int nk = p.K / BK, k0 = 0;
  if constexpr (PART) {
    const int per = (nk + p.slices - 1) / p.slices;
    k0 = min(slice * per, nk);
    nk = min(k0 + per, nk) - k0;
  }
  const char *a_src[NA], *b_src[NB];
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    const int at = j * NT + tid, row = at >> 3, c = (at & 7) ^ ((row >> 1) & 7);
    int a_row = min(m0 + row, m_end - 1);
    if (GRP && p.row_of) a_row = p.row_of[a_row];
    a_src[j] = (const char*)(p.A + (int64_t)a_row * p.lda + k0 * BK + c * 8);
  }
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int at = j * NT + tid, row = at >> 3, c = (at & 7) ^ ((row >> 1) & 7);
    int n = min(n0 + row, p.n_pad - 1);
    if constexpr (EPI == MD_EPI_SILU) {
      const int v = n0 + row, half = p.n_pad >> 1;
      n = min((v >> 6) * 32 + (v & 31), half - 1) + ((v & 32) ? half : 0);
    }
    b_src[j] = (const char*)(p.W + (GRP ? group * p.group_stride : 0) + (int64_t)n * p.ldw + k0 * BK + c * 8);
  }
  auto issue = [&](auto piece_c, int stage) {
    constexpr int X = decltype(piece_c)::value;
    char* base = smem + stage * STAGE + wave * 1024;
    if constexpr (X < NA) {
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)a_src[X],
                                       (__attribute__((address_space(3))) void*)(base + X * NT * 16), 16, 0, 0);
      a_src[X] += 128;
    } else {
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)b_src[X - NA],
                                       (__attribute__((address_space(3))) void*)(base + A_BYTES + (X - NA) * NT * 16), 16, 0, 0);
      b_src[X - NA] += 128;
    }
  };

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const uint32_t piece[2] = {(uint32_t)((g ^ (r >> 1)) * 16), (uint32_t)(((4 + g) ^ (r >> 1)) * 16)};
  const uint32_t a_at = lds0 + (wm * TM + r) * 128, b_at = lds0 + A_BYTES + (wn * TN + r) * 128;
  f32x4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  constexpr int PER = MI + NI, READS = 2 * PER, MULS = 2 * MI * NI;
  bf16x8 f[2][2][PER];  // [slice & 1][half of its K][rows of W, rows of A]
  auto read = [&](auto buf_c, auto x_c, uint32_t st) {
    constexpr int B = decltype(buf_c)::value, X = decltype(x_c)::value, H = X / PER, Y = X % PER;
    if constexpr (Y < NI) lds_read<Y * 2048>(f[B][H][Y], st + b_at + piece[H]);
    else lds_read<(Y - NI) * 2048>(f[B][H][Y], st + a_at + piece[H]);
  };
  auto in_flight = [&](int n) {  // waits until at most n slices (of P pieces) are under way
    static_for<0, S>([&](auto c) {
      constexpr int N = decltype(c)::value;
      if (n == N) wait_vm<N * P>();
    });
  };
  auto barrier = [&] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  static_for<0, S>([&](auto c) {
    if (decltype(c)::value < nk) static_for<0, P>([&](auto x) { issue(x, decltype(c)::value); });
  });
  in_flight(max(0, min(S, nk) - 1));
  barrier();
  if (nk > 0) static_for<0, READS>([&](auto x) { read(std::integral_constant<int, 0>{}, x, 0u); });
  wait_lds();
  __builtin_amdgcn_sched_barrier(0);

  const bool live = m0 + wm * TM < m_end;
  // slice t: its operands are in f[t & 1].  STEADY: slice t + S exists
  auto step = [&](int t, auto buf_c, auto steady_c) {
    constexpr int B = decltype(buf_c)::value;
    constexpr bool STEADY = decltype(steady_c)::value;
    if constexpr (STEADY) wait_vm<(S - 2) * P>();  // slice t + 1 has landed, later ones are under way
    else in_flight(max(0, min(S - 2, nk - 2 - t)));
    barrier();  // ... everybody's part of it; and everybody has read slice t
    const bool more = STEADY || t + 1 < nk, refill = STEADY || t + S < nk;
    const int stage = t % S;
    if (GRP && !live) {  // (wave-uniform) only padding: this wave's share of the copies
      if (refill) static_for<0, P>([&](auto y) { issue(y, stage); });
      return;
    }
    const uint32_t st1 = (uint32_t)((t + 1) % S) * STAGE;
    static_for<0, MULS>([&](auto x_c) {
      constexpr int X = decltype(x_c)::value, H = X / (MI * NI), I = X / NI % MI, J = X % NI;
      acc[I][J] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[B][H][J], f[B][H][NI + I], acc[I][J], 0, 0, 0);
      // reads and DMA pieces evenly between the products
      static_for<X * READS / MULS, (X + 1) * READS / MULS>([&](auto y) {
        __builtin_amdgcn_sched_barrier(0);
        if (more) read(std::integral_constant<int, 1 - B>{}, y, st1);
        __builtin_amdgcn_sched_barrier(0);
      });
      static_for<X * P / MULS, (X + 1) * P / MULS>([&](auto y) {
        __builtin_amdgcn_sched_barrier(0);
        if (refill) issue(y, stage);
        __builtin_amdgcn_sched_barrier(0);
      });
    });
    __builtin_amdgcn_sched_barrier(0);
    wait_lds();
    __builtin_amdgcn_sched_barrier(0);
  };
  int t = 0;
  for (; t + 1 + S < nk; t += 2) {
    step(t, std::integral_constant<int, 0>{}, std::true_type{});
    step(t + 1, std::integral_constant<int, 1>{}, std::true_type{});
  }
  for (; t < nk; t += 2) {
    step(t, std::integral_constant<int, 0>{}, std::false_type{});
    if (t + 1 < nk) step(t + 1, std::integral_constant<int, 1>{}, std::false_type{});
  }
  __syncthreads();  // the ring has been read

  // acc[i][j]: row 16 i + r, columns 16 j + 4 g ..
  const int mw = m0 + wm * TM, nw = n0 + wn * TN;
  if constexpr (PART) {
    // 32 rows of 64 fp32 at a time through the wave's own part of LDS, so that rows are stored in runs of 256 bytes
    constexpr int LD = 64 + 4;
    float* own = (float*)smem + wave * 32 * LD;
    float* dst = p.partial + (int64_t)slice * p.partial_slice_stride;
#pragma unroll
    for (int b = 0; b < MI / 2; ++b) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) *(f32x4*)(own + (16 * i + r) * LD + 16 * j + 4 * g) = acc[2 * b + i][j];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int row = 4 * q + g, m = mw + 32 * b + row, n = nw + 4 * r;
        const f32x4 v = *(const f32x4*)(own + row * LD + 4 * r);
        if (m < m_end && n < p.n_store) *(f32x4*)(dst + (int64_t)m * p.partial_ld + n) = v;
      }
    }
    return;
  }
  char* own = smem + wave * 4096;  // 32 rows of 64 columns
  if constexpr (EPI == MD_EPI_SILU) {
#pragma unroll
    for (int b = 0; b < MI / 2; ++b) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int row = 16 * i + r, ch = 2 * j + (g >> 1);
          float y[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float z = acc[2 * b + i][j][e], u = acc[2 * b + i][j + 2][e];
            if (p.round_first) z = bf2f(f2bf(z)), u = bf2f(f2bf(u));  // (uniform)
            y[e] = silu_fast(z) * u;
          }
          *(u32x2*)(own + row * 64 + ((ch ^ ((row >> 1) & 3)) * 16) + (g & 1) * 8) = u32x2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
        }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int idx = q * 64 + lane, row = idx >> 2, ch = idx & 3;
        const u32x4 v = *(const u32x4*)(own + row * 64 + ((ch ^ ((row >> 1) & 3)) * 16));
        const int m = mw + 32 * b + row, n = (nw >> 1) + ch * 8;
        if (m < m_end && n < (p.n_store >> 1)) *(u32x4*)(p.C + (int64_t)m * p.ldc + n) = v;
      }
    }
    return;
  }
  f32x4 bias[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int n = nw + 16 * j + 4 * g;
    u32x2 b = {0u, 0u};
    if (p.bias != nullptr && n < p.n_pad) b = *(const u32x2*)(p.bias + n);
    bias[j] = f32x4{lo_bf(b[0]), hi_bf(b[0]), lo_bf(b[1]), hi_bf(b[1])};
  }
  // residual: requested up front; r may alias c, a piece is read and later written by the same lane
  u32x4 res[EPI == MD_EPI_RESIDUAL ? MI / 2 : 1][4];
  if constexpr (EPI == MD_EPI_RESIDUAL)
#pragma unroll
    for (int b = 0; b < MI / 2; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = mw + 32 * b + 8 * q + (lane >> 3), n = nw + (lane & 7) * 8;
        res[b][q] = u32x4{0u, 0u, 0u, 0u};
        if (m < m_end && n < p.n_store) res[b][q] = *(const u32x4*)(p.R + (int64_t)(p.res_row_mod ? m % p.res_row_mod : m) * p.ldr + n);
      }
#pragma unroll
  for (int b = 0; b < MI / 2; ++b) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int row = 16 * i + r, ch = 2 * j + (g >> 1);
        const f32x4 v = acc[2 * b + i][j] + bias[j];
        *(u32x2*)(own + row * 128 + ((ch ^ (row & 7)) * 16) + (g & 1) * 8) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = 8 * q + (lane >> 3), ch = lane & 7, m = mw + 32 * b + row, n = nw + ch * 8;
      u32x4 v = *(const u32x4*)(own + row * 128 + ((ch ^ (row & 7)) * 16));
      if (m >= m_end || n >= p.n_store) continue;
      if constexpr (EPI == MD_EPI_GELU) {
        if (n >= p.gelu_from)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const md_f32x2 y = gelu_tanh_f32x2(md_f32x2{lo_bf(v[e]), hi_bf(v[e])});
            v[e] = pack_bf16x2(y[0], y[1]);
          }
      } else if constexpr (EPI == MD_EPI_RESIDUAL) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = pack_bf16x2(lo_bf(res[b][q][e]) + lo_bf(v[e]), hi_bf(res[b][q][e]) + hi_bf(v[e]));
      }
      *(u32x4*)(p.C + (int64_t)m * p.ldc + n) = v;
    }
  }
}

// Row panels per group: those with which an XCD's run of tiles reads the fewest rows of both operands
inline int mid_group(int tiles_m, int tiles_n, int slices, int bm, int bn) {
  const int run = std::max(1, (tiles_m * tiles_n * slices + 7) / 8);
  int best = 1;
  long least = -1;
  for (int g = 1; g <= std::min(tiles_m, 32); ++g) {
    const long rows = (long)std::min(g, run) * bm + (long)((run + g - 1) / g) * bn;
    if (least < 0 || rows < least) least = rows, best = g;
  }
  return best;
}

template <int BM, int BN, int WM, int WN, int S, int EPI, bool PART, bool GRP = false>
md_status launch(GemmK k, hipStream_t s) {
  constexpr int lds = S * (BM + BN) * 128;
  static_assert(lds <= 163840 && lds >= WM * WN * 32 * 68 * 4, "LDS");
  const auto fn = gemm_mid_kernel<BM, BN, WM, WN, S, EPI, PART, GRP>;
  MD_TRY(md_ensure_dynamic_lds((const void*)fn, lds));
  k.tiles_m = GRP ? grouped_tiles(k.M, k.groups, BM) : (k.M + BM - 1) / BM;
  k.tiles_n = (k.n_store + BN - 1) / BN;
  if (!PART) k.slices = 1;
  k.group_m = mid_group(k.tiles_m, k.tiles_n, k.slices, BM, BN);
  hipLaunchKernelGGL(fn, dim3(k.tiles_m * k.tiles_n * k.slices), dim3(WM * WN * 64), lds, s, k);
  return md_launch_status();
}

}  // namespace

namespace {
template <int EPI>
md_status by_height(const GemmK& k, int bm, hipStream_t s) {
  return bm == 256 ? launch<256, 128, 4, 2, 3, EPI, false>(k, s) : launch<128, 128, 2, 2, 4, EPI, false>(k, s);
}
}  // namespace

md_status md_gemm_mid_launch(const GemmK& k, int epi, int bm, hipStream_t s) {
  switch (epi) {
    case MD_EPI_BIAS: return by_height<MD_EPI_BIAS>(k, bm, s);
    case MD_EPI_GELU: return by_height<MD_EPI_GELU>(k, bm, s);
    case MD_EPI_RESIDUAL: return by_height<MD_EPI_RESIDUAL>(k, bm, s);
    case MD_EPI_SILU: return by_height<MD_EPI_SILU>(k, bm, s);
    default: return MD_ERR_UNSUPPORTED;
  }
}
md_status md_gemm_mid_launch_grouped(const GemmK& k, int epi, int bm, hipStream_t s) {
  if (epi == MD_EPI_SILU) return bm == 256 ? launch<256, 128, 4, 2, 3, MD_EPI_SILU, false, true>(k, s) : launch<128, 128, 2, 2, 4, MD_EPI_SILU, false, true>(k, s);
  if (epi == MD_EPI_BIAS) return bm == 256 ? launch<256, 128, 4, 2, 3, MD_EPI_BIAS, false, true>(k, s) : launch<128, 128, 2, 2, 4, MD_EPI_BIAS, false, true>(k, s);
  return MD_ERR_UNSUPPORTED;
}
md_status md_gemm_mid_partial(const GemmK& k, hipStream_t s) { return launch<128, 128, 2, 2, 4, MD_EPI_BIAS, true>(k, s); }
