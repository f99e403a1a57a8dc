// Wave-level helpers for the gfx950 paged-attention kernels: MFMA wrappers,
// 16-bit packing, E5M2 dequantisation and cross-lane reductions.
//
// They take the place of the upstream helper header
// (include/paged_attention_utils.hpp: padding_mask :314-363, mat_vec_mul_broadcast
// :734-804, mat_vec_div_broadcast :806-879, group_reduce_t :881-960) but share no
// structure with it: here a "tile" is the register image of a 16x16 MFMA operand in
// one 64-lane wavefront.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace fa {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

struct F16 {};   // query / output element tags
struct BF16 {};

// ---- in-kernel timeline (debug builds with -DFA_TIMELINE only) -------------------------------------
// Wall-clock stamps (the 100 MHz counter of s_memrealtime) that wavefronts of the persistent kernels
// leave in a device array, eight 64-bit slots per wavefront; fa_debug_timeline() copies it to the host.
// Slots: 0 kernel entry, 1 lengths in and items ranked, 2 first K tile in registers, 3 last chunk
// done, 4 last merge stored, 5 chunks this wavefront ran, 6 HW_ID register, 7 XCC_ID register.
// Compiled out of the product library.
#ifdef FA_TIMELINE
constexpr int kTimelineWaves = 8192, kTimelineSlots = 8;
static __device__ unsigned long long timeline_words[kTimelineWaves * kTimelineSlots];
__device__ __forceinline__ void timeline_put(int slot, unsigned long long value) {
  const int wave = (int)blockIdx.x * (int)(blockDim.x >> 6) + (int)(threadIdx.x >> 6);
  if ((threadIdx.x & 63) == 0 && wave < kTimelineWaves) timeline_words[wave * kTimelineSlots + slot] = value;
}
__device__ __forceinline__ void timeline_stamp(int slot) { timeline_put(slot, wall_clock64()); }
__device__ __forceinline__ void timeline_where() {
  timeline_put(6, __builtin_amdgcn_s_getreg((31 << 11) | 4));   // HW_ID
  timeline_put(7, __builtin_amdgcn_s_getreg((31 << 11) | 20));  // XCC_ID
}
#define FA_TIMELINE_STAMP(slot) ::fa::timeline_stamp(slot)
#define FA_TIMELINE_PUT(slot, value) ::fa::timeline_put(slot, (unsigned long long)(value))
#define FA_TIMELINE_WHERE() ::fa::timeline_where()
#else
#define FA_TIMELINE_STAMP(slot) ((void)0)
#define FA_TIMELINE_PUT(slot, value) ((void)0)
#define FA_TIMELINE_WHERE() ((void)0)
#endif

// Which kv head the q-th of a sequence's work items is, in the persistent kernels.  Work-groups are handed to the
// XCCs in turn (work-group g runs on XCC g mod 8) and consecutive positions of the item list are the kv heads of
// one sequence, so with a multiple of eight kv heads XCC k gets positions k, k + 8, ... of every sequence.  In a
// pool whose blocks hold the heads' chunks side by side, head h lies h * (bytes of a head's chunk) into a block.
// The timings below fit a memory that is dealt to its eight stacks in 4 KiB units, by address bits 12 to 14 (an
// inference from the measurements, not a documented fact): position q takes the head for which those bits equal
// q mod 8, so that every XCC reads one stack and every stack is read by one XCC.
// Measured on the FP8 Llama-7B decode batch (32 heads, chunks of 2 KiB, so that heads in plain order put two stacks
// on each pair of neighbouring XCCs): 53.8 -> 52.8 us, and the XCCs' mean finishing times 47.8-51.1 -> within
// 1.5 us of each other; giving every XCC every stack (heads rotated by the sequence's number) 53.1 us.  With chunks
// of 4 KiB (16-bit cache, head size 128, blocks of 16) plain order is that map already.  Heads whose chunks are
// smaller than 1 KiB or larger than 4 KiB (upstream's layout, where a head's share of a block is one token row at
// a time; large blocks) stay in plain order.  The grid forms (one work-group per (sequence, kv head), blockIdx.x
// the head) keep plain order too: there the map measured 2 % slower (512 sequences of the same shape: 838 against
// 820 us).  shift: log2(4 KiB / chunk), or -1 for plain order.
#ifndef FA_ITEM_HEAD_AFFINE
#define FA_ITEM_HEAD_AFFINE 1
#endif
__device__ __forceinline__ int stack_affine_shift(int64_t head_chunk_bytes, int heads) {
  if (!FA_ITEM_HEAD_AFFINE || head_chunk_bytes < 1024 || head_chunk_bytes > 4096 ||
      (head_chunk_bytes & (head_chunk_bytes - 1)) != 0)
    return -1;
  const int shift = head_chunk_bytes == 4096 ? 0 : head_chunk_bytes == 2048 ? 1 : 2;
  return heads % (8 << shift) == 0 ? shift : -1;
}
__device__ __forceinline__ int stack_affine_head(int q, int shift) {
  if (shift < 0) return q;
  const int k = q & 7, a = q >> 3;
  return ((a >> shift) << (shift + 3)) | (k << shift) | (a & ((1 << shift) - 1));
}

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// D[16x16] += A[16x32] * B[32x16] on one wavefront.  Lane l = 16*r + i holds
//   A[row i][k-slots 8r .. 8r+7]   (8 x 16 bit = 4 dwords)
//   B[k-slots 8r .. 8r+7][col i]
//   D[rows 4r .. 4r+3][col i]      (4 x fp32)
// Which head-dim element or token a k-slot stands for is free as long as A and
// B agree, which is what lets every operand be loaded straight from HBM.
template <typename QT>
__device__ __forceinline__ f32x4 mfma_16x16x32(u32x4 a, u32x4 b, f32x4 c);

template <>
__device__ __forceinline__ f32x4 mfma_16x16x32<F16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma_16x16x32<BF16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Two fp32 values -> one dword of two 16-bit floats (lo in bits 0..15), round to nearest even.
template <typename QT>
__device__ __forceinline__ uint32_t pack2(float lo, float hi);
template <>
__device__ __forceinline__ uint32_t pack2<F16>(float lo, float hi) {
  f16x2 v = {(_Float16)lo, (_Float16)hi};
  return __builtin_bit_cast(uint32_t, v);
}
template <>
__device__ __forceinline__ uint32_t pack2<BF16>(float lo, float hi) {
  bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

template <typename QT>
__device__ __forceinline__ float load_scalar16(const void *p);
template <>
__device__ __forceinline__ float load_scalar16<F16>(const void *p) {
  return (float)*reinterpret_cast<const _Float16 *>(p);
}
template <>
__device__ __forceinline__ float load_scalar16<BF16>(const void *p) {
  return (float)*reinterpret_cast<const __bf16 *>(p);
}

// E5M2 is binary16 cut to its top byte: byte b decodes to the fp16 with bits b << 8; into bf16
// it goes through v_cvt_scalef32_pk_bf16_bf8 (exact: 2 mantissa bits, exponent range inside
// bf16's).
// Dword w holds four E5M2 bytes; decode bytes (2*half, 2*half+1) to a 16-bit pair.
template <typename QT>
__device__ __forceinline__ uint32_t e5m2_adjacent_pair(uint32_t w, int half);
template <>
__device__ __forceinline__ uint32_t e5m2_adjacent_pair<F16>(uint32_t w, int half) {
  // one byte permute: result bytes (0, w[2*half], 0, w[2*half + 1]); selector 0x0c yields zero
  return half == 0 ? __builtin_amdgcn_perm(w, w, 0x010c000cu) : __builtin_amdgcn_perm(w, w, 0x030c020cu);
}
template <>
__device__ __forceinline__ uint32_t e5m2_adjacent_pair<BF16>(uint32_t w, int half) {
  bf16x2 v = half == 0 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w, 1.0f, false)
                       : __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w, 1.0f, true);
  return __builtin_bit_cast(uint32_t, v);
}

// FP8 cache formats.  kKvE5M2: 1-5-2, binary16 cut to its top byte.  kKvE4M3: 1-4-3 "fn"
// (bias 7, no infinities, 0x7f / 0xff NaN), decoded by the CDNA4 conversion instructions;
// both decode exactly into fp16 and bf16.
constexpr int kKv16 = 0, kKvE5M2 = 1, kKvE4M3 = 2;

// Decode byte k (0..3) of dword y into the low and byte k of dword x into the high 16-bit
// half: the V transpose takes its two tokens from two registers.  One byte permute does the
// gather -- for E5M2 into fp16 it is the whole decode (bytes land in the top halves), otherwise
// it puts the bytes next to each other for the conversion instruction.
template <int KVF, typename QT>
__device__ __forceinline__ uint32_t fp8_pair_at(uint32_t y, uint32_t x, int k) {
  // v_perm_b32 selectors: 0..3 = bytes of the second operand, 4..7 = bytes of the first, 0x0c = 0
  if constexpr (KVF == kKvE5M2 && std::is_same<QT, F16>::value) {
    return __builtin_amdgcn_perm(x, y, 0x000c000cu | ((uint32_t)k << 8) | ((uint32_t)(4 + k) << 24));
  } else {
    const uint32_t two = __builtin_amdgcn_perm(x, y, 0x0c0c0000u | (uint32_t)k | ((uint32_t)(4 + k) << 8));
    if constexpr (KVF == kKvE4M3) {
      if constexpr (std::is_same<QT, BF16>::value) {
        return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(two, 1.0f, false));
      } else {
        return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(two, 1.0f, false));
      }
    } else {
      return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(two, 1.0f, false));
    }
  }
}
template <int KVF, typename QT>
__device__ __forceinline__ uint32_t fp8_adjacent_pair(uint32_t w, int half) {
  if constexpr (KVF == kKvE4M3) {
    if constexpr (std::is_same<QT, BF16>::value) {
      const bf16x2 v = half == 0 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false)
                                 : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true);
      return __builtin_bit_cast(uint32_t, v);
    } else {
      const f16x2 v = half == 0 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false)
                                : __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true);
      return __builtin_bit_cast(uint32_t, v);
    }
  } else {
    return e5m2_adjacent_pair<QT>(w, half);
  }
}

// Reductions over the four 16-lane rows of a wavefront (lanes i, i+16, i+32, i+48), the result in every lane.  v_permlane16_swap
// exchanges the odd rows of one register with the even rows of another, v_permlane32_swap the upper half with the lower
// half: given the same value twice, they leave a pair's two members in the same lane of the two registers.  Vector
// instructions; the shuffles through LDS that did this before took two LDS latencies, one behind the other, of
// every chunk of keys, between its scores and its exponentials.
template <typename F>
__device__ __forceinline__ float rows_fold(float v, F &&f) {
  const uint32_t a = __builtin_bit_cast(uint32_t, v);
  const auto x = __builtin_amdgcn_permlane16_swap(a, a, false, false);
  const uint32_t b = __builtin_bit_cast(uint32_t, f(__builtin_bit_cast(float, (uint32_t)x[0]), __builtin_bit_cast(float, (uint32_t)x[1])));
  const auto y = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return f(__builtin_bit_cast(float, (uint32_t)y[0]), __builtin_bit_cast(float, (uint32_t)y[1]));
}
__device__ __forceinline__ float rows_max(float v) {
  return rows_fold(v, [](float x, float y) { return fmaxf(x, y); });
}
__device__ __forceinline__ float rows_sum(float v) {
  return rows_fold(v, [](float x, float y) { return x + y; });
}
// The value of the lane N places on within a row of 16 lanes (in a ring).
template <int N>
__device__ __forceinline__ float row_rotated(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + N, 0xF, 0xF, true));
}
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, row_rotated<8>(v));
  v = fmaxf(v, row_rotated<4>(v));
  v = fmaxf(v, row_rotated<2>(v));
  v = fmaxf(v, row_rotated<1>(v));
  return rows_max(v);
}
__device__ __forceinline__ float wave_sum(float v) {
  v += row_rotated<8>(v);
  v += row_rotated<4>(v);
  v += row_rotated<2>(v);
  v += row_rotated<1>(v);
  return rows_sum(v);
}

// Load one int32 of read-only input through the scalar unit.  `p` must be wave-uniform and
// must point at memory the kernel never writes (block tables, context lengths): the
// constant address space tells the compiler exactly that, so the load stays a scalar load
// even when the kernel has stored to other buffers before it.
__device__ __forceinline__ int32_t load_uniform_i32(const int32_t *p) {
  typedef const int32_t __attribute__((address_space(4))) *const_ptr;
  return *(const_ptr)(uintptr_t)p;
}

__device__ __forceinline__ float load_uniform_f32(const float *p) {
  typedef const float __attribute__((address_space(4))) *const_ptr;
  return *(const_ptr)(uintptr_t)p;
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// K/V bytes are read exactly once per launch.  STREAM marks a load non-temporal so that it
// does not displace the few lines that are re-used (queries, block tables, scratch).
template <bool STREAM, typename T>
__device__ __forceinline__ T kv_load(const T *p) {
  if constexpr (STREAM) {
    return __builtin_nontemporal_load(p);
  } else {
    return *p;
  }
}

// Global loads of 4, 8 or 16 bytes per lane.
template <int DWORDS, bool STREAM>
struct VLoad;
template <bool STREAM>
struct VLoad<4, STREAM> {
  static __device__ __forceinline__ void ld(uint32_t (&dst)[4], const char *p) {
    u32x4 t = kv_load<STREAM>(reinterpret_cast<const u32x4 *>(p));
    dst[0] = t[0]; dst[1] = t[1]; dst[2] = t[2]; dst[3] = t[3];
  }
};
template <bool STREAM>
struct VLoad<2, STREAM> {
  static __device__ __forceinline__ void ld(uint32_t (&dst)[2], const char *p) {
    u32x2 t = kv_load<STREAM>(reinterpret_cast<const u32x2 *>(p));
    dst[0] = t[0]; dst[1] = t[1];
  }
};
template <bool STREAM>
struct VLoad<1, STREAM> {
  static __device__ __forceinline__ void ld(uint32_t (&dst)[1], const char *p) {
    dst[0] = kv_load<STREAM>(reinterpret_cast<const uint32_t *>(p));
  }
};

}  // namespace fa
