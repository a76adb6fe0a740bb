// Window kernel for calls of several launch classes: one launch for all of them.
// Included by one .hip file per (id type, weight mode).
#pragma once

#include "tbe_lookup_impl.h"

namespace tra {

// As tbe_pooled_cu_kernel, with blocks of all weight types and lane chunks in one grid: a block pools bags of one
// sub-class and picks its body by it.  Lane chunks are at most 16 accumulators wide here: wider bodies would not fit the
// 128 registers that sixteen waves leave each other.  With 32-bit ids they do without weights; up to 4 registers are kept
// in scratch memory with per-sample and 7 with position weights, with 64-bit ids up to 1 without, 9 with per-sample and 15
// with position weights.
template <typename IdxT, int WEIGHTED, bool FROM_LENGTHS>
__global__ __launch_bounds__(kCuThreads) void tbe_pooled_multi_kernel(const void* p_offsets, const FeatureDesc* p_cdescs,
                                                                      int32_t p_B, int32_t p_xcd_blocks,
                                                                      int32_t p_xcd_count, const MultiArgs m) {
  extern __shared__ unsigned char tra_dyn_smem[];  // (room that a tuning override asks for, unused)
  TRA_WINDOW(IdxT, s_window);
  const LookupArgs& a = m.common;
  int blk = blockIdx.x;
  if (p_xcd_blocks > 0) blk = (blk % p_xcd_count) * p_xcd_blocks + blk / p_xcd_count;
  int s = 0;
#pragma unroll
  for (int i = 1; i < kMaxMultiSub; ++i)
    if (blk >= m.tile_start[i]) s = i;  // (INT32_MAX behind the last one)
  const SubClass sc = m.sub[s];
  const int kind = m.kind[s];
  const int nb_all = sc.count * p_B;
  const int q0 = (blk - sc.tile_start) * sc.window;
  if (q0 >= nb_all) return;
  const int nb = min(sc.window, nb_all - q0);
  const int fi_lo = q0 / p_B;
  const auto starts = stage_window<IdxT, FROM_LENGTHS>(s_window, a, p_offsets, p_cdescs, p_B, sc, q0, nb, fi_lo);
  const bool vec = (kind & kMultiVec) != 0;
#define TRA_MULTI(D, CB)                                                                                       \
  case multi_kind(D, CB):                                                                                      \
    pool_window<D, CB, IdxT, WEIGHTED, 4, kBodiesMany>(s_window, a, sc, nb, fi_lo, starts, [&] { return vec; }); \
    break;
  switch (kind & ~kMultiVec) {
    TRA_MULTI(TRA_INT8, 16)
    TRA_MULTI(TRA_INT8, 8)
    TRA_MULTI(TRA_INT8, 4)
    TRA_MULTI(TRA_INT4, 8)
    TRA_MULTI(TRA_INT4, 4)
    TRA_MULTI(TRA_INT2, 4)
    TRA_MULTI(TRA_FP16, 16)
    TRA_MULTI(TRA_FP16, 8)
    TRA_MULTI(TRA_FP16, 4)
    TRA_MULTI(TRA_FP32, 16)
    TRA_MULTI(TRA_FP32, 8)
    TRA_MULTI(TRA_FP32, 4)
  }
#undef TRA_MULTI
}

#define TRA_DEFINE_MULTI(T, W)                                                                                    \
  template <>                                                                                                     \
  void launch_multi<T, W>(const MultiArgs& a, int grid, int lds_bytes, bool from_lengths, hipStream_t stream) {   \
    const LookupArgs& c = a.common;                                                                               \
    if (from_lengths)                                                                                             \
      hipLaunchKernelGGL((tbe_pooled_multi_kernel<T, W, true>), dim3(grid), dim3(kCuThreads), lds_bytes, stream,  \
                         c.offsets, c.cdescs, c.B, c.xcd_blocks, c.xcd_count, a);                                 \
    else                                                                                                          \
      hipLaunchKernelGGL((tbe_pooled_multi_kernel<T, W, false>), dim3(grid), dim3(kCuThreads), lds_bytes, stream, \
                         c.offsets, c.cdescs, c.B, c.xcd_blocks, c.xcd_count, a);                                 \
  }

}  // namespace tra
