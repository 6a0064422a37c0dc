// How the products of few rows read their weights (gemm_step.hip, gemm_experts.hip).
#pragma once
#include "lm_internal.hpp"

namespace {

// Weights through LDS: a wave's load of 8 rows x 128 bytes puts piece p of row r at 128 r + 16 (p ^ r) of a kilobyte of its own, from which operands are
// read without bank conflicts.  A load into registers in the operand's shape has its neighbouring lanes in different rows, which costs the address unit 80 cycles per
// KB, and 8 lanes to a row 38; into LDS 20.
__device__ __forceinline__ uint32_t lds_address(char* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)p; }
// As buffer loads: beside a flat or global load into LDS, which counts as one of either memory, the compiler lets a use of ANY loaded register wait for all
// loads under way, and every ring ran empty once in its length (see stream_units).  rows: of 8 or more rows of k from here on (base uniform); at: a lane's place in 8 of them
__device__ __forceinline__ __amdgpu_buffer_rsrc_t weight_rows(const bf16_t* base) { return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)0xffffffff, 0x00020000); }
__device__ __forceinline__ uint32_t weight_at(int lane, int k) { return 2u * ((uint32_t)(lane >> 3) * (uint32_t)k + 8u * (uint32_t)((lane & 7) ^ (lane >> 3))); }
__device__ __forceinline__ void load_weights(__amdgpu_buffer_rsrc_t rows, uint32_t at, uint32_t offset, char* dst) {  // (2: non-temporal)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (__attribute__((address_space(3))) void*)dst, 16, at, offset, 0, 2);
}
// One operand, or the two of a unit of 16 columns, for each x: in assembly, as the compiler would wait for all loads into LDS that are under way
template <int NX>
__device__ __forceinline__ void read_weights(uint32_t p, u32x4 (&w)[NX]) {
  static_assert(NX == 1 || NX == 2, "operands");
  if constexpr (NX == 1) asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(w[0]) : "v"(p) : "memory");
  else asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:1024\n\ts_waitcnt lgkmcnt(0)" : "=&v"(w[0]), "=&v"(w[1]) : "v"(p) : "memory");
}
template <int NX>
__device__ __forceinline__ void read_weights(uint32_t p, u32x4 (&w)[NX][2]) {
  const uint32_t q = p ^ 64;  // the other 32 of a unit's 64 of K
  if constexpr (NX == 1) {
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)" : "=&v"(w[0][0]), "=&v"(w[0][1]) : "v"(p), "v"(q) : "memory");
  } else {
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %4 offset:2048\n\tds_read_b128 %3, %5 offset:2048\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(w[1][0]), "=&v"(w[1][1]) : "v"(p), "v"(q) : "memory");
    if constexpr (NX == 3)
      asm volatile("ds_read_b128 %0, %2 offset:4096\n\tds_read_b128 %1, %3 offset:4096\n\ts_waitcnt lgkmcnt(0)" : "=&v"(w[2][0]), "=&v"(w[2][1]) : "v"(p), "v"(q) : "memory");
    if constexpr (NX == 4)
      asm volatile("ds_read_b128 %0, %4 offset:4096\n\tds_read_b128 %1, %5 offset:4096\n\tds_read_b128 %2, %4 offset:6144\n\tds_read_b128 %3, %5 offset:6144\n\ts_waitcnt lgkmcnt(0)"
                   : "=&v"(w[2][0]), "=&v"(w[2][1]), "=&v"(w[3][0]), "=&v"(w[3][1]) : "v"(p), "v"(q) : "memory");
  }
}
// Waits until a unit's P loads have arrived, with those of `left` more, D at most, under way behind it
template <int D, int P>
__device__ __forceinline__ void wait_units(int left) {
  static_assert(D * P < 64, "vmcnt has six bits");
  if constexpr (D == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  else if (left >= D) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(D * P) : "memory");
  else wait_units<D - 1, P>(left);
}

// The units lo .. hi - 1 of a wave, D under way: load(b, u) requests unit u (P loads, always) into buffer b, multiply(b) uses it; between() runs behind the
// first requests.  PEELED: the loads of the loop stand under no condition.  The compiler counts loads into registers by itself; where one may not have been
// issued it waits as if it had not, and the ring runs short once in its length.  It costs registers and instructions: not for the head's products, 51200 columns, where two waves to a
// workgroup lose one of seven workgroups (1 row 36.5 us, peeled 37.2), and 64 columns of 48 rows one of two (232 registers to 254; 40 rows 49 us, peeled 58).
template <int D, int P, bool PEELED = true, class Load, class Multiply, class Between>
__device__ __forceinline__ void stream_units(int lo, int hi, Load load, Multiply multiply, Between between) {
  if constexpr (!PEELED) {
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (lo + d < hi) load(d, lo + d);
    between();
    for (int u = lo; u < hi; u += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int left = hi - 1 - (u + d);
        if (left < 0) break;
        wait_units<D - 1, P>(left);
        multiply(d);
        if (left >= D) load(d, u + d + D);
      }
    }
  } else if (hi - lo >= D) {
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, lo + d);
    between();
    int u = lo;
    for (; u + 2 * D <= hi; u += D)
#pragma unroll
      for (int d = 0; d < D; ++d) {
        wait_units<D - 1, P>(D - 1);
        multiply(d);
        load(d, u + D + d);
      }
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int left = hi - 1 - (u + d);
      wait_units<D - 1, P>(left);
      multiply(d);
      if (left >= D) load(d, u + D + d);
    }
    u += D;
#pragma unroll
    for (int d = 0; d < D - 1; ++d) {
      const int left = hi - 1 - (u + d);
      if (left < 0) break;
      wait_units<D - 1, P>(left);
      multiply(d);
    }
  } else {
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
      if (lo + d < hi) load(d, lo + d);
    between();
#pragma unroll
    for (int d = 0; d < D - 1; ++d) {
      const int left = hi - 1 - (lo + d);
      if (left < 0) break;
      wait_units<D - 1, P>(left);
      multiply(d);
    }
  }
}

}  // namespace
