// Loop path, rows cut into pieces (paged_attn_loop_cut_kernel, walk_segment_items<..., ROW_MERGE = true>): how the
// work-groups that share a (sequence, kv head) row hand their softmax states to whichever of them is
// last, inside one launch.
//
// A wavefront of a work-group owns one slice of the output of every piece its work-group takes (the
// slice it merges out of LDS), and wavefront `tw` owns the same slice in every work-group.  So the
// pieces of a row meet per slice: the wavefront writes its slice of the piece -- un-normalised sums with
// their maximum and total, fp32 -- to the piece's slot of the workspace, sets the flag of that slice of
// the piece, and if it then finds the flags of all the row's pieces set, reads their slices, its own
// among them, and stores the result.  Nobody waits for anybody: there is no spin and no order among
// work-groups that the launch depends on.  Pieces are merged in the order of their keys whoever merges
// them, so the result does not depend on the arrival order.
//
// How the last one is found: a wavefront sets the flag of its slice of its piece and then looks at the flags of
// that slice of all the row's pieces, 64 at a time.  Whoever's flag is last in memory sees them all and merges; so
// may another whose flag went out at the same time, and then both store the same values.  (One counter per row and
// slice was built first: with its increments contended by every piece of the row, 59 pieces that end together
// took 90 us instead of 35.  A claim word that lets one of them merge costs two more trips to memory at the end of
// the launch, more than a second merge.)
// Where the flags lie: those of a slice side by side, the row's pieces in order, so that looking at 64 of them takes four to
// eight requests.  (A line of its own for every piece made that 64, for each of the row's pieces: 8 rows of 32 pieces
// 28.6 us, now 14.7; 24 rows of 900-4096 keys 17.8, now 14.9.)
// The flags lie in workspace that nobody has cleared.  A set flag holds the nonce of the launch, any other contents
// mean "not set", and the merging wavefront clears the row's.  So a launch leaves no nonce of its own behind -- a HIP
// graph that replays the launch, nonce and all, finds none -- and memory that happens to hold the nonce has a chance
// of 2^-64 per word.
#pragma once

#include "paged_attention_items.h"
#include "paged_attention_wave.h"

namespace fa {

// Floats of one wavefront's slice of one piece: `cols` columns of 4 * SL values (four lane rows of SL
// each) and two scalars, rounded up to 16 bytes.
constexpr int merge_slice_floats(int cols, int sl) { return (cols * (4 * sl + 2) + 3) & ~3; }

struct MergeSlot {
  float *at;
  int cols, sl;
  // pair `half` of four values, and the two scalars of a column
  __device__ __forceinline__ uint64_t *pair(int k, int half, int r, int col) const {
    return reinterpret_cast<uint64_t *>(at + ((k * 4 + r) * cols + col) * 4 + 2 * half);
  }
  __device__ __forceinline__ uint64_t *scalars(int col) const {
    return reinterpret_cast<uint64_t *>(at + 4 * sl * cols + 2 * col);
  }
};

// What one work-group writes and another, on any XCD, reads within the launch goes past the L2 caches, which are
// one per XCD: agent-scope atomic stores write through to memory, agent-scope atomic loads come from there.  With
// plain accesses a release and an acquire fence per piece would have to write back and invalidate a whole L2:
// measured, that made every piece cost 0.1-0.2 us of the whole launch (384 rows: 42 -> 157 us).
__device__ __forceinline__ void share_pair(uint64_t *at, float a, float b) {
  __hip_atomic_store(at, (uint64_t)__float_as_uint(b) << 32 | __float_as_uint(a), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void shared_pair(const uint64_t *at, float &a, float &b) {
  const uint64_t w = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  a = __uint_as_float((uint32_t)w);
  b = __uint_as_float((uint32_t)(w >> 32));
}

// Slot of slice tw of a piece; `piece`: number of the piece among all pieces of the launch.
__device__ __forceinline__ MergeSlot merge_slot(const PagedAttnParams &p, int64_t piece, int tw, int slices, int cols, int sl) {
  return {p.merge_pieces + (piece * slices + tw) * merge_slice_floats(cols, sl), cols, sl};
}

// Number, among all pieces of the launch, of piece j of the row of `it`.
__device__ __forceinline__ int64_t merge_piece(const MergeItem &it, int j) {
  return j < it.whole ? it.first_piece + (int64_t)j * it.piece_step : it.last_piece;
}

// Flag of slice tw of piece j of the row of `it`.  The flags of a slice lie side by side, a row's pieces in order
// (it.whole + 1 of them, used or not): every wavefront that finishes a piece looks at all of them.
__device__ __forceinline__ uint64_t *merge_flag(const PagedAttnParams &p, const MergeItem &it, int j, int tw, int slices) {
  return p.merge_flags + (int64_t)it.first_flag * slices + tw * (it.whole + 1) + j;
}

// Says that slice tw of piece it.piece lies in its slot; true if the calling wavefront is to merge that slice of
// the row.  All lanes.
__device__ __forceinline__ bool merge_arrive(const PagedAttnParams &p, const MergeItem &it, int tw, int slices, int lane) {
  // the slice has reached memory (share_pair) before its flag goes out ...
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (lane == 0)
    __hip_atomic_store(merge_flag(p, it, it.part0, tw, slices), p.merge_nonce, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // ... and the flag before the others' are looked at: of two wavefronts at least one sees the other's
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  bool missing = false;
  for (int j = lane; j < it.pieces; j += 64)
    missing |= __hip_atomic_load(merge_flag(p, it, j, tw, slices), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) !=
               p.merge_nonce;
  if (__any(missing)) return false;
  asm volatile("" ::: "memory");  // the others' slices are read behind their flags, not before
  for (int j = lane; j < it.pieces; j += 64)
    __hip_atomic_store(merge_flag(p, it, j, tw, slices), 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// Merges slice tw of all pieces of the row of `it`.  On return lane (r, i), i < cols, holds the row's
// un-normalised values in o, their maximum in M and their total in L, as a lane does after the merge in LDS.
// With fewer than 9 columns the lanes of a 16-lane row work on several pieces at a time.
template <int SL>
__device__ __forceinline__ void merge_pieces(const PagedAttnParams &p, const MergeItem &it, int tw, int slices, int cols, int r,
                                             int i, float &M, float &L, float (&o)[SL]) {
  const int width = cols > 8 ? 16 : cols > 4 ? 8 : cols > 2 ? 4 : cols;  // 1, 2, 4, 8, 16
  const int c = i & (width - 1), sub = i / width, subs = 16 / width;
  constexpr int U = 4;  // pieces in flight per lane
  float m = -INFINITY, l = 0.f;
#pragma unroll
  for (int e = 0; e < SL; ++e) o[e] = 0.f;
  for (int j0 = 0; j0 < it.pieces; j0 += U * subs) {  // wave-uniform
    float pm[U], pl[U], f[U];
    float v[U][SL];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = j0 + u * subs + sub;
      pm[u] = -INFINITY;
      pl[u] = 0.f;
#pragma unroll
      for (int e = 0; e < SL; ++e) v[u][e] = 0.f;
      if (j < it.pieces && c < cols) {
        const MergeSlot slot = merge_slot(p, merge_piece(it, j), tw, slices, cols, SL);
        shared_pair(slot.scalars(c), pm[u], pl[u]);
#pragma unroll
        for (int e = 0; e < SL; e += 2) shared_pair(slot.pair(e >> 2, (e >> 1) & 1, r, c), v[u][e], v[u][e + 1]);
      }
    }
    float mx = m;
#pragma unroll
    for (int u = 0; u < U; ++u) mx = fmaxf(mx, pm[u]);
    const float keep = m == -INFINITY ? 0.f : fast_exp2(m - mx);
#pragma unroll
    for (int u = 0; u < U; ++u) f[u] = pm[u] == -INFINITY ? 0.f : fast_exp2(pm[u] - mx);
    m = mx;
    l *= keep;
#pragma unroll
    for (int u = 0; u < U; ++u) l += f[u] * pl[u];
#pragma unroll
    for (int e = 0; e < SL; ++e) {
      o[e] *= keep;
#pragma unroll
      for (int u = 0; u < U; ++u) o[e] += f[u] * v[u][e];
    }
  }
  M = m;
  for (int d = width; d < 16; d <<= 1) M = fmaxf(M, __shfl_xor(M, d));
  const float f = m == -INFINITY ? 0.f : fast_exp2(m - M);
  L = l * f;
#pragma unroll
  for (int e = 0; e < SL; ++e) o[e] *= f;
  for (int d = width; d < 16; d <<= 1) {
    L += __shfl_xor(L, d);
#pragma unroll
    for (int e = 0; e < SL; ++e) o[e] += __shfl_xor(o[e], d);
  }
}

}  // namespace fa
