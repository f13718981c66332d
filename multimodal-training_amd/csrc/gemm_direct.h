// Direct global -> LDS loads, hand-placed waits and the transposing LDS read, as the bf16 GEMM kernels use them.
// The compiler does not see these loads: waits for them are placed by hand (a wave's memory instructions complete in order).
#pragma once
#include "gemm_common.h"

namespace {

template <int N>
__device__ __forceinline__ void pp_wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
__device__ __forceinline__ void pp_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void pp_load(unsigned lds_addr, unsigned voff, const char* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(voff), "s"(base) : "memory");
}
// the same for the lanes with k < limit only; the instruction is issued (and counted by vmcnt) even when no lane takes part
__device__ __forceinline__ void pp_load_below(unsigned lds_addr, unsigned voff, const char* base, int k, int limit) {
  unsigned long long saved;
  asm volatile(
      "s_mov_b32 m0, %1\n\tv_cmp_gt_i32 vcc, %5, %4\n\ts_mov_b64 %0, exec\n\ts_and_b64 exec, exec, vcc\n\ts_nop 0\n\t"
      "global_load_lds_dwordx4 %2, %3\n\ts_mov_b64 exec, %0"
      : "=&s"(saved) : "s"(lds_addr), "v"(voff), "s"(base), "v"(k), "s"(limit) : "memory", "vcc", "scc");
}
// per-lane 64-bit addresses: 16 bytes per lane, and the same for the lanes with k < limit only
__device__ __forceinline__ void pp_load_at(unsigned lds_addr, const char* addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_addr), "v"(addr) : "memory");
}
__device__ __forceinline__ void pp_load_at_below(unsigned lds_addr, const char* addr, int k, int limit) {
  unsigned long long saved;
  asm volatile(
      "s_mov_b32 m0, %1\n\tv_cmp_gt_i32 vcc, %4, %3\n\ts_mov_b64 %0, exec\n\ts_and_b64 exec, exec, vcc\n\ts_nop 0\n\t"
      "global_load_lds_dwordx4 %2, off\n\ts_mov_b64 exec, %0"
      : "=&s"(saved) : "s"(lds_addr), "v"(addr), "v"(k), "s"(limit) : "memory", "vcc", "scc");
}
__device__ __forceinline__ void pp_load_dword_at(unsigned lds_addr, const char* addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(lds_addr), "v"(addr) : "memory");
}
__device__ __forceinline__ bf16x8 pp_read_tr(const unsigned char* p, int second) {
  typedef s16x4 __attribute__((address_space(3))) * lds_ptr_t;
  s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(p));
  s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(p + second));
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  return __builtin_bit_cast(bf16x8, (s16x8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
}

// Columns of a product whose B operand comes through the transposing read.  The read takes 16 consecutive columns per fragment, so
// an accumulator holds columns 4 * (l / 16) .. + 3 of its block of 16.  Trading one value of block 0 (x) with one of block 1 (y)
// between neighbouring groups of 16 lanes leaves each lane with eight consecutive columns of the 32, from tr_first_column(l / 16):
// x of the exchange is the first half, y the second.  (Dealing the columns to the fragments instead, as a row-major B's are, makes the
// read take 8 bytes of every 16: half of the banks, twice the cycles.  us per K tile of 64 with both operands behind the
// transposing read, 64 tiles of 256 x 256, before -> now 1.34 -> 1.31; on all units the clock, and with it the time, stays as it was.)
__device__ __forceinline__ int tr_first_column(int g4) { return (g4 & 1) * 16 + (g4 >> 1) * 8; }
__device__ __forceinline__ void tr_columns(float& x, float& y) {
  const float a = x, b = y;
  const auto t = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  const unsigned t0 = t[0], t1 = t[1];
  x = __builtin_bit_cast(float, t0);
  y = __builtin_bit_cast(float, t1);
}

}  // namespace
