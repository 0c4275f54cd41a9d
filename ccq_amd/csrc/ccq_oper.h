// Building blocks shared by the register walks and their chunk-parallel partners (ccq_gwalk.hip,
// ccq_gla.hip): direct-to-LDS loads, transposing reads, B operands straight from accumulator tiles, and
// row tiles in LDS that serve as plain and as transposed operands.
//
// Operand order of a contraction over 32 indices: lane 16 g + m holds indices 4 g .. +3 and 16 + 4 g .. +3
// of row / column m -- the order in which two stacked 16x16 accumulator tiles hold their rows, so that
// they are a B operand as they stand.
#pragma once

#include "ccq_tile.h"

namespace ccq {

// workgroup barrier after this wave's LDS operations; global memory operations stay in flight
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Direct-to-LDS load of 16 bytes per lane: wave-uniform global base + 32-bit lane byte offset, lane i's
// piece lands at LDS byte m0 + 16 i (m0 wave-uniform).  Inline assembly so that the compiler does not
// drain every load before LDS reads; completion is waited for by wait_loads alone.  M0 is read one wait
// state after it is written (the s_nop).
typedef __attribute__((address_space(3))) char lds_char;
__device__ __forceinline__ unsigned lds_addr(const void* p) {
  return __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_char*)const_cast<void*>(p));
}
__device__ __forceinline__ void lds_load16(const void* base, unsigned off, unsigned m0) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void lds_load4(const void* base, unsigned off, unsigned m0) {  // (lane i: 4 bytes at m0 + 4 i)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(m0), "v"(off), "s"(base) : "memory", "m0");
}
// all but the N youngest vector memory operations of this wave are complete
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0xF70);
  asm volatile("" ::: "memory");
}

typedef __attribute__((address_space(3))) bf16x4_t lds_bf4;
// four consecutive contraction elements of the lane's operand row (ds_read_b64_tr_b16): lane j of a
// 16-lane group names the 8-byte piece holding columns 4 (j & 3) .. +3 of row j >> 2
__device__ __forceinline__ bf16x4_t read_tr(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf4*)p);
}
__device__ __forceinline__ bf16x8 join(const bf16x4_t& a, const bf16x4_t& b) {
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

// four values as packed hi and lo words
__device__ __forceinline__ void split4(const f32x4& a, u32x2& hi, u32x2& lo) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    unsigned x, y;
    split2x2(a[2 * i], a[2 * i + 1], x, y);
    hi[i] = x;
    lo[i] = y;
  }
}
// hi / lo B operand of two stacked accumulator tiles (contraction slots 0-3: tile a, 4-7: tile b)
__device__ __forceinline__ void split_pair(const f32x4& a, const f32x4& b, bf16x8& hi, bf16x8& lo) {
  u32x2 ah, al, bh, bl;
  split4(a, ah, al);
  split4(b, bh, bl);
  hi = __builtin_bit_cast(bf16x8, u32x4{ah[0], ah[1], bh[0], bh[1]});
  lo = __builtin_bit_cast(bf16x8, u32x4{al[0], al[1], bl[0], bl[1]});
}

// k tile of a chunk in LDS: rows of 2 K bytes, 16-byte piece s of row t at piece s ^ swz(t).  The swizzle
// puts the 32 bytes that a transposing read takes of each of four consecutive rows into different banks,
// and spreads the sixteen rows of an A operand over all pieces of 128 bytes.
__device__ __forceinline__ int swz(int t) { return ((t & 3) << 1) | ((t >> 2) & 1); }
// Byte offset of the lane's 16 bytes of the 1 KiB direct load i of a k tile (rows at or past L as row
// L - 1: finite, and every product with them meets a zero gate)
template <int K>
__device__ __forceinline__ unsigned k_tile_off(int i, int rsk, int L, int l) {
  const int t = (512 / K) * i + l / (K / 8), pos = l & (K / 8 - 1);
  return (unsigned)(min(t, L - 1) * rsk * 2 + ((pos ^ swz(t)) << 4));
}
// the same of a [64][W] bf16 tile of rows rs apart (v, dO)
template <int W>
__device__ __forceinline__ unsigned row_tile_off(int i, int rs, int L, int l) {
  const int t = (512 / W) * i + l / (W / 8);
  return (unsigned)(min(t, L - 1) * rs * 2 + 16 * (l & (W / 8 - 1)));
}
// A operand of K S: token rows 16 tt + m, state rows 32 p + 4 g .. +3 and 32 p + 16 + 4 g .. +3
template <int K>
__device__ __forceinline__ bf16x8 k_frag(const char* s, int tt, int p, int g, int m) {
  const int t = 16 * tt + m, pc = 4 * p + (g >> 1);
  const char* r = s + t * (2 * K) + 8 * (g & 1);
  return join(*(const bf16x4_t*)(r + ((pc ^ swz(t)) << 4)), *(const bf16x4_t*)(r + (((pc + 2) ^ swz(t)) << 4)));
}
// A operand of K^T U: state rows 16 rt + m, tokens 32 q + 4 g .. +3 and 32 q + 16 + 4 g .. +3
template <int K>
__device__ __forceinline__ bf16x8 kt_frag(const char* s, int rt, int q, int g, int m) {
  const int t = 32 * q + 4 * g + (m >> 2), pc = 2 * rt + ((m >> 1) & 1);  // (t and t + 16 have one swizzle)
  const char* r = s + t * (2 * K) + ((pc ^ swz(t)) << 4) + 8 * (m & 1);
  return join(read_tr(r), read_tr(r + 16 * 2 * K));
}

// Workgroup -> (unit, value block): the blocks of one unit share k, T and the gates, so they go to one
// XCD (linear ids are handed out round-robin); the grid is padded to whole groups of eight units.
__device__ __forceinline__ bool unit_map(int bid, int nv, int nunits, int& unit, int& vt) {
  const int slot = bid >> 3;
  vt = slot % nv;
  unit = (slot / nv) * 8 + (bid & 7);
  return unit < nunits;
}

}  // namespace ccq
