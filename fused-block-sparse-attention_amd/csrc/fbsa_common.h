// Shared device/host helpers for the gfx950 block-sparse attention kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

#include "fbsa.h"

namespace fbsa {

typedef __bf16 bf16;
typedef _Float16 f16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// ---- host-side error reporting (thread-local message, status code) ----
int fail(int code, const char *fmt, ...);
int hip_check(hipError_t e, const char *what);

// ---- element conversions ----
template <typename T> __device__ __forceinline__ float to_f32(T x) { return (float)x; }
template <typename T> __device__ __forceinline__ T from_f32(float x) { return (T)x; }

// ---- LDS chunk swizzle -----------------------------------------------------
// A tile row of cpr 16-byte chunks stores logical chunk c at position
// c ^ swz(row). LDS has 64 banks of 4 bytes. Measured on gfx950 with the
// bank-conflict counters: a ds_read_b128 is served in 4 passes of 16 lanes,
// lanes l and l' sharing a pass iff they agree in lane bit 5 and in the parity
// of lane bits 2..4; a ds_read_b64_tr_b16 in 2 passes (lanes 0-31, 32-63).
// swz is linear in row bits 0..3 and keeps on distinct banks, for every cpr:
//  (a) an MFMA operand load, lane (g, p) reading row 16m + p, chunk 4ks + g;
//  (b) a transposing load, 8 aligned rows x two adjacent chunks per pass;
//  (c) the fp32 operand loads (16 rows x 4 bytes of one chunk, and 4 rows x
//      4 chunks), for cpr >= 16.
__host__ __device__ constexpr int swz(int row, int cpr) {
  return cpr >= 16 ? (((row & 7) << 1) ^ (13 * ((row >> 3) & 1)))
       : cpr == 8  ? ((((row >> 1) & 3) << 1) ^ (5 * ((row >> 3) & 1)))
       : cpr == 4  ? ((((row >> 2) & 1) << 1) ^ (3 * ((row >> 3) & 1)))
       : 0;
}

// ---- gfx950 primitives ----------------------------------------------------
// Direct-to-LDS global loads (global_load_lds, LDS destination in M0):
// lane l's 4 or 16 bytes land at lds_wave_base + 4*l or + 16*l, the base
// wave-uniform. They are issued by inline asm because the compiler's wait
// insertion cannot tell the LDS they write from any LDS a later ordinary load
// reads: it waits for vmcnt(0) there, which also waits for the ring stages just
// prefetched and so takes away the overlap the ring exists for. Every consumer
// waits for its stage itself (wait_vmcnt / wait_ring, then lds_barrier() or
// __syncthreads()); the "memory" clobber keeps LDS accesses from moving across
// an issue. Waits the compiler inserts for its own loads stay correct (loads
// leave vmcnt in issue order, so uncounted DMA only makes them wait longer).
// M0 is written here without being preserved. Nothing else in the library uses
// M0 (no message, GWS or indexed register move), so no value of the compiler's
// lives in it across the asm.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// The LDS destination is given as a pointer or as its LDS address (the low 32
// bits of the pointer).
__device__ __forceinline__ void g2lds16(const void *gsrc, unsigned lds_wave_base) {
  const unsigned m = __builtin_amdgcn_readfirstlane(lds_wave_base);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(gsrc), "s"(m) : "memory", "m0");
}
__device__ __forceinline__ void g2lds16(const void *gsrc, void *lds_wave_base) {
  g2lds16(gsrc, (unsigned)(uintptr_t)lds_wave_base);
}
// The same load with a wave-uniform 64-bit base in SGPRs and a 32-bit per-lane
// byte offset (the instruction's saddr form): no 64-bit address VALU op per load.
__device__ __forceinline__ void g2lds16_s(const void *sbase, unsigned voff, unsigned lds_wave_base) {
  const unsigned m = __builtin_amdgcn_readfirstlane(lds_wave_base);
  // the base is uniform by contract; readfirstlane puts it in SGPRs (folded away
  // when the compiler already holds it there)
  // (readfirstlane returns int: each half goes through uint32_t so that the
  // low word is zero-extended, never sign-extended, into the 64-bit base)
  const uint64_t bp = (uint64_t)(uintptr_t)sbase;
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((unsigned)(bp >> 32));
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((unsigned)bp);
  const uint64_t sb = ((uint64_t)hi << 32) | (uint64_t)lo;
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(sb), "s"(m)
               : "memory", "m0");
}
__device__ __forceinline__ void g2lds16_s(const void *sbase, unsigned voff, void *lds_wave_base) {
  g2lds16_s(sbase, voff, (unsigned)(uintptr_t)lds_wave_base);
}
__device__ __forceinline__ void g2lds4(const void *gsrc, void *lds_wave_base) {
  const unsigned m = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds_wave_base);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(gsrc), "s"(m) : "memory", "m0");
}
#pragma clang diagnostic pop

// s_waitcnt with only the vector-memory counter constrained (gfx9 encoding:
// vmcnt[3:0] at bits 3:0, vmcnt[5:4] at bits 15:14, expcnt/lgkmcnt left open).
template <int N> __device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x70 | 0xF00);
}

// Wait until at most `pending` ring stages of N direct-to-LDS loads each are
// still in flight (the loads of older stages have landed).
template <int N> __device__ __forceinline__ void wait_ring(int pending) {
  switch (pending) {
    case 0: wait_vmcnt<0>(); break;
    case 1: wait_vmcnt<(N < 64 ? N : 63)>(); break;
    case 2: wait_vmcnt<(2 * N < 64 ? 2 * N : 63)>(); break;
    default: wait_vmcnt<(3 * N < 64 ? 3 * N : 63)>(); break;
  }
}

// Workgroup barrier for LDS-staged pipelines. Unlike __syncthreads() it does
// not wait for outstanding vector-memory ops (which would drain the
// direct-to-LDS prefetch ring); callers wait for their own DMA with
// wait_vmcnt<N>() first. Pending LDS reads are drained (lgkmcnt(0)) and the
// empty asm statements keep the compiler from moving memory ops across it.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Transposing LDS read (ds_read_b64_tr_b16). Within each 16-lane group, lane i
// supplies the address of 4 consecutive 16-bit elements C[i][0..3]; lane j
// receives C[4e + j/4][j%4] for e = 0..3.
// Issued as inline asm: the compiler's builtin form makes it wait for every
// outstanding direct-to-LDS load first, which would drain the prefetch ring.
// The result is NOT ready until lds_wait_all() and must pass through
// lds_ready() before use.
__device__ __forceinline__ s16x4 lds_read_tr16(const void *lds_addr) {
  s16x4 r;
  const unsigned a = (unsigned)(uintptr_t)lds_addr;
  asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(r) : "v"(a));
  return r;
}
__device__ __forceinline__ void lds_wait_all() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// Wait until at most N LDS/scalar-memory operations are outstanding (N <= 15,
// the counter's range). LDS operations complete in issue order, so an
// operation followed by at least N later ones has then completed.
template <int N> __device__ __forceinline__ void lds_wait_le() {
  static_assert(N >= 0 && N <= 15, "lgkmcnt range");
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}
// lgkmcnt wait for a count known after unrolling (values above 15 wait for 15)
__device__ __forceinline__ void lds_wait_upto(int n) {
  switch (n < 15 ? n : 15) {
    case 0: lds_wait_le<0>(); break;
    case 1: lds_wait_le<1>(); break;
    case 2: lds_wait_le<2>(); break;
    case 3: lds_wait_le<3>(); break;
    case 4: lds_wait_le<4>(); break;
    case 5: lds_wait_le<5>(); break;
    case 6: lds_wait_le<6>(); break;
    case 7: lds_wait_le<7>(); break;
    case 8: lds_wait_le<8>(); break;
    case 9: lds_wait_le<9>(); break;
    case 10: lds_wait_le<10>(); break;
    case 11: lds_wait_le<11>(); break;
    case 12: lds_wait_le<12>(); break;
    case 13: lds_wait_le<13>(); break;
    case 14: lds_wait_le<14>(); break;
    default: lds_wait_le<15>(); break;
  }
}

// 16-byte LDS read issued as inline asm (not reordered with the other asm LDS
// reads); like lds_read_tr16 the result needs a wait and lds_ready() before use.
__device__ __forceinline__ s16x8 lds_read_b128(const void *lds_addr) {
  s16x8 r;
  asm volatile("ds_read_b128 %0, %1" : "=v"(r) : "v"((unsigned)(uintptr_t)lds_addr));
  return r;
}
template <typename V> __device__ __forceinline__ void lds_ready(V &x) { asm volatile("" : "+v"(x)); }
// The same reads with a compile-time byte offset in the instruction's offset
// field (vaddr = a per-lane base plus the stage address): no address VALU op
// per read.
template <int OFF> __device__ __forceinline__ s16x8 lds_read_b128_at(unsigned vaddr) {
  static_assert(OFF >= 0 && OFF < 65536, "ds offset field");
  s16x8 r;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(vaddr), "n"(OFF));
  return r;
}
template <int OFF> __device__ __forceinline__ s16x4 lds_read_tr16_at(unsigned vaddr) {
  static_assert(OFF >= 0 && OFF < 65536, "ds offset field");
  s16x4 r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(vaddr), "n"(OFF));
  return r;
}

// static_for<N>(fn): fn(std::integral_constant<int, i>{}) for i = 0 .. N-1
// (the index is a constant expression inside fn)
template <typename Fn, int... Is>
__device__ __forceinline__ void static_for_(Fn &&fn, std::integer_sequence<int, Is...>) {
  (fn(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename Fn> __device__ __forceinline__ void static_for(Fn &&fn) {
  static_for_(fn, std::make_integer_sequence<int, N>{});
}

// Swizzled operand-tile addressing as per-lane bases plus constants. swz
// depends on row bits 0..3 only and is below 16, so for the MFMA operand read
// of row 16m + p, chunk 4ks + g (16-bit types):
//   byte offset = kbase(ks % 4) + (ks / 4) * 256 + m * 256 * CPR
// with kbase(l) = (p * CPR + ((4l + g) ^ swz(p))) * 16; and for the transposing
// read of rows ra = 32 k2 + 4g + p/4 (+16 for the high half), chunk 2t + h,
// h = (p & 3) / 2, half p & 1:
//   byte offset = vbase(t % 8) + (t / 8) * 256 + k2 * 512 * CPR (+ 256 * CPR)
// with vbase(l) = ((4g + p/4) * CPR + ((2l + h) ^ swz(4g + p/4))) * 16 + (p & 1) * 8.
__device__ __forceinline__ unsigned tile_kbase(int l, int g, int p, int cpr) {
  return (unsigned)((p * cpr + ((4 * l + g) ^ swz(p, cpr))) * 16);
}
__device__ __forceinline__ unsigned tile_vbase(int l, int g, int p, int cpr) {
  const int ra = 4 * g + (p >> 2);
  return (unsigned)((ra * cpr + ((2 * l + ((p & 3) >> 1)) ^ swz(ra, cpr))) * 16 + (p & 1) * 8);
}

__device__ __forceinline__ float shfl_xor_f(float x, int m) { return __shfl_xor(x, m, 64); }

// MFMA 16x16x32 (bf16 / f16 inputs, fp32 accumulate). Operand lane layout:
// lane l holds row/col (l % 16) and k = 8*(l/16) + e, e = 0..7 (any k
// permutation works if A and B agree). Result: lane l holds rows 4*(l/16)+r,
// column l % 16, r = 0..3.
template <typename T> struct Mfma16;
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
template <> struct Mfma16<bf16> {
  __device__ static __forceinline__ f32x4 run(s16x8 a, s16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  // k = 16 variant: lane l holds k = 4*(l/16) + e, e = 0..3
  __device__ static __forceinline__ f32x4 run16(s16x4 a, s16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma16<f16> {
  __device__ static __forceinline__ f32x4 run(s16x8 a, s16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  __device__ static __forceinline__ f32x4 run16(s16x4 a, s16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a),
                                                 __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
  }
};

// fp32 MFMA 16x16x4: lane l holds row/col l%16, k = l/16.
__device__ __forceinline__ f32x4 mfma_f32_16x16x4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <typename T> __device__ __forceinline__ short bits16(T x) { return __builtin_bit_cast(short, x); }

// Pack 8 fp32 into 8 16-bit values of type T.
template <typename T> __device__ __forceinline__ s16x8 pack8(const float *x) {
  s16x8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = bits16<T>((T)x[e]);
  return r;
}

// Two-term split of fp32 values into a 16-bit MFMA operand pair: hi = x
// in T (rounded, or for bf16 truncated), lo = (x - hi) rounded to T (x - hi is
// exact in fp32). A product with an exact 16-bit operand then takes two MFMAs
// (hi, then lo into the same accumulator) and carries x to about 2^-16
// relative for bf16 instead of the 2^-9 of one rounding.
// bf16: hi is x truncated to its upper 16 bits (the pair gathered by one
// v_perm_b32), lo = x - hi (exact) rounded once; three VALU ops per value.
template <typename T> __device__ __forceinline__ void pack8_split(const float *x, s16x8 &hi, s16x8 &lo) {
  float r[8];
  if constexpr (__is_same(T, bf16)) {
    u32x4 hw;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t a = __float_as_uint(x[2 * j]), b = __float_as_uint(x[2 * j + 1]);
      hw[j] = __builtin_amdgcn_perm(b, a, 0x07060302u);  // (b >> 16) << 16 | a >> 16
      r[2 * j] = x[2 * j] - __uint_as_float(a & 0xFFFF0000u);
      r[2 * j + 1] = x[2 * j + 1] - __uint_as_float(b & 0xFFFF0000u);
    }
    hi = __builtin_bit_cast(s16x8, hw);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const T h = (T)x[e];
      hi[e] = bits16<T>(h);
      r[e] = x[e] - (float)h;
    }
  }
  lo = pack8<T>(r);
}
template <typename T> __device__ __forceinline__ void pack4_split(const float *x, s16x4 &hi, s16x4 &lo) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const T h = (T)x[e];
    hi[e] = bits16<T>(h);
    lo[e] = bits16<T>((T)(x[e] - (float)h));
  }
}

// XCD-aware work order: launch order bid is dispatched round-robin over the
// 8 XCDs; returning w = (bid % 8) * (n / 8) + bid / 8 gives each XCD a
// contiguous range of the work order (the tail beyond 8*(n/8) maps 1:1).
__device__ __forceinline__ int64_t xcd_remap(int64_t bid, int64_t n) {
  const int64_t per = n / 8;
  if (bid >= per * 8) return bid;
  return (bid % 8) * per + bid / 8;
}

// Launch order of query-major kernels with grouped query heads: work unit u
// (b, KV head, query block) goes to XCD u % 8 (round-robin, like plain launch
// order) and its grp query-head workgroups run back to back on that XCD, so the
// K/V tiles they share are fetched into one L2 once instead of into grp of
// them. Returns the unit of launch order bid and sets the head within the
// group; with grp == 1 it is the identity. Units past the last full round of 8
// map in launch order.
// (launch indices and unit counts are below 2^31, a grid's x limit: 32-bit
// division, a short sequence, instead of the long 64-bit expansion)
__device__ __forceinline__ int64_t gqa_unit(int64_t bid, int64_t nunits, int grp, int *hin) {
  const uint32_t b32 = (uint32_t)bid, g = (uint32_t)grp;
  const uint32_t full = (uint32_t)nunits / 8u * 8u;
  const uint32_t base = full * g;
  if (b32 >= base) {
    const uint32_t r = b32 - base;
    *hin = (int)(r % g);
    return (int64_t)(full + r / g);
  }
  const uint32_t s = b32 / 8u;
  *hin = (int)(s % g);
  return (int64_t)((s / g) * 8u + b32 % 8u);
}

}  // namespace fbsa
