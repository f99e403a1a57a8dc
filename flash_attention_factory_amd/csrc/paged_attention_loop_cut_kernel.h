// Loop path given workspace: the persistent loop kernel, or where some rows are long enough the same rows cut into
// pieces that are merged within the launch (paged_attention_row_merge.h).  Which of the two, the device decides from the
// lengths (MergeRows::cut), every wavefront for itself.
//
// A launch of short rows lasts 5 to 10 us, so what comes before its first load of keys counts, and so does everything
// that the compiler puts there for the sake of the other branch.  The parameters of a kernel are loaded where it begins
// and kept from there on; with the parameters of both branches in one body, 120 to 250 of them went into lanes of spare
// vector registers one by one (29 to 76 in the persistent loop kernel), over half a microsecond of every launch.  So each
// branch, and the decision, reads the parameters it needs again through a pointer that the compiler cannot see through
// (kernel_params), and rows that stay whole run the code of the persistent loop kernel.  Table columns for 16384
// keys, back to back (us; persistent loop kernel | whole rows and pieces in one body | this kernel):
//   16-bit cache: 4 sequences of 1-256 keys, 8 heads of 64   5.2 |  5.7 |  5.1   4 of 100-500, 32 heads on 8   9.0 | 10.0 |  8.9
//                 16 of 100-1000                            18.4 | 18.9 | 18.4   48 of 2600, not worth a cut  94.6 | 95.4 | 95.3
//   byte cache:   the same four             5.0 |  5.8 |  5.0,  7.5 |  8.5 |  7.3,  11.0 | 11.5 | 10.9,  45.5 | 46.5 | 45.9
// What is left on long rows that are not cut is the decision itself.
#pragma once

#include "paged_attention_loop_persistent_kernel.h"
#include "paged_attention_segment_kernel.h"

namespace fa {

// The parameters of the running kernel (its only argument), to be loaded anew.
__device__ __forceinline__ const PagedAttnParams &kernel_params() {
  auto *at = (const __attribute__((address_space(4))) PagedAttnParams *)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(at));
  return *(const PagedAttnParams *)at;
}

template <int D, typename QT, int KVF, int NWG, int OCC, int TPC, bool EXT, bool KROW>
__global__ void __launch_bounds__(NWG * 64) __attribute__((amdgpu_waves_per_eu(OCC)))
paged_attn_loop_cut_kernel(const PagedAttnParams p) {
  using W = WaveAttn<D, QT, KVF, TPC, Pipeline<(KVF != 0)>::stream_loads_loop, EXT, KROW>;
  FA_TIMELINE_STAMP(0);
  FA_TIMELINE_WHERE();
  __shared__ ItemStates<NWG, W::NR> sm;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row_count = p.num_seqs * p.num_kv_heads;  // no more than there are work-groups (the launcher sees to it)
  LoopItems<TPC> rows;
  rows.build(p, lane, wave, row_count, W::CT);
  MergeRows merge;
  constexpr int kBytes = KVF == kKv16 ? 2 : 1, kStayWhole = merge_whole_partitions(D, kBytes);
  bool cut = __any(max(rows.len0, rows.len1) > kStayWhole * p.partition_size);
  if (cut) cut = merge.cut<D == 64>(kernel_params(), rows.len0, rows.len1, kStayWhole, merge_extra_cost(D, kBytes));
  if (!cut) {
    if ((int)blockIdx.x >= row_count) return;
    // (the extended instances, given p, get a stack frame that they do not use, and with it scratch memory)
    if constexpr (EXT) walk_loop_items<D, QT, KVF, NWG, TPC, EXT, KROW, 1>(kernel_params(), rows, row_count, sm);
    else walk_loop_items<D, QT, KVF, NWG, TPC, EXT, KROW, 1>(p, rows, row_count, sm);
    return;
  }
  const PagedAttnParams &again = kernel_params();
  SegmentItems<true> pieces;
  pieces.build(again, merge, lane, gridDim.x, W::ROWB);
  walk_segment_items<D, QT, KVF, NWG, TPC, EXT, 1, true, KROW>(again, pieces, sm);
}

}  // namespace fa
