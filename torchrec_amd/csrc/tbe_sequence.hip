// Sequence lookup: one dequantized row per id, no reduction.
#include "tbe_lookup_impl.h"

namespace tra {

// Range of ids of class feature `ci` at key position `pos`.  `starts` (kBoundsTotals) holds the keys' first ids.
template <typename IdxT>
__device__ __forceinline__ void sequence_bounds(const LookupArgs& a, int ci, int pos, const int64_t* starts,
                                                int64_t& first, int64_t& n) {
  int64_t last;
  if (a.bounds_kind == kBoundsOffsets) {
    first = load_index<IdxT>(a.offsets, (int64_t)pos * a.B);
    last = load_index<IdxT>(a.offsets, (int64_t)(pos + 1) * a.B);
  } else if (a.bounds_kind == kBoundsTotals) {
    first = starts[pos];
    last = starts[pos + 1];
  } else {
    first = a.pw_off[ci];
    last = first + a.pw_len[ci];
  }
  // (never outside the ids array, whatever the bounds say)
  first = first < 0 ? 0 : first;
  last = last > a.num_indices ? a.num_indices : last;
  n = last > first ? last - first : 0;
}

// Lane c's NE outputs of the row slice at `pos`.  Results are written once and read by a later kernel: as whole
// lines with the non-temporal hint where a lane holds one or two 16-byte vectors (finish_bag exchanges two).
template <int NE>
__device__ __forceinline__ void store_row(float (&acc)[NE], const LookupArgs& a, int64_t pos, int c, int lpr, int lane,
                                          bool active) {
  if constexpr (NE == 8) {
    if (a.vec_store && a.out_fp16) {
      u32x4_t v;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t lo = __half_as_ushort(__float2half_rn(acc[2 * k]));
        const uint32_t hi = __half_as_ushort(__float2half_rn(acc[2 * k + 1]));
        v[k] = lo | (hi << 16);
      }
      if (active)
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4_t*>(reinterpret_cast<__half*>(a.out) + pos + c * NE));
      return;
    }
  }
  finish_bag<NE>(acc, a, 0, pos, c, lpr, lane, active, a.vec_store != 0);
}

// A feature's ids are cut into tiles of sc.window consecutive ids; the tiles of
// the sub-class's features are numbered through, and block t of the sub-class
// takes tiles t, t + blocks, ...: features of very different sizes still fill
// the chip evenly.  Every wave finds the feature of its tile by a scan over the
// features' tile counts.
//
// A tile is walked in steps of kSequenceUnroll rows per lane group: ids, then all row
// chunks, then the arithmetic and the stores, so a wave has 4 rows per lane
// group in flight.  Every lane runs every step (positions past the tile's end
// are clamped and not stored), which is what the matrix instruction of the
// sub-byte conversions needs.
//
// Bound by memory: a 132-byte row costs two 128-byte lines, so 2.1 M int8 rows
// of 128 columns with fp16 results move 1083 MB.  One row per lane group and
// plain stores took 206 us; four in flight, and results that leave as whole
// lines past the caches (store_row), 187 us = 5.8 TB/s, what a gather of random
// lines reaches (rows loaded with the non-temporal hint as well: 208 us).
template <int DTYPE, int CB, typename IdxT>
__global__ __launch_bounds__(kBlockThreads) void tbe_nobag_kernel(const LookupArgs a) {
  constexpr int NE = CB * 8 / Traits<DTYPE>::kBits;
  constexpr int U = kSequenceUnroll;
  __shared__ int64_t s_starts[kMaxTotalKeys + 1];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  if (a.bounds_kind == kBoundsTotals) {
    if (wave == 0) {
      const int64_t* totals = reinterpret_cast<const int64_t*>(a.offsets);
      int64_t before = 0;
      for (int k0 = 0; k0 < a.num_keys; k0 += kWaveSize) {
        const int64_t v = k0 + lane < a.num_keys ? totals[k0 + lane] : 0;
        const int64_t incl = wave_scan_incl(v);
        if (k0 + lane < a.num_keys) s_starts[k0 + lane + 1] = before + incl;
        before += wave_last(incl);
      }
      if (lane == 0) s_starts[0] = 0;
    }
    __syncthreads();
  }
  const int blk = blockIdx.x;
  int s = 0;
#pragma unroll
  for (int i = 1; i < kMaxSub; ++i)
    if (i < a.n_sub && blk >= a.sub[i].tile_start) s = i;
  const SubClass sc = a.sub[s];
  const int tile_ids = sc.window;
  const int lpr = sc.lpr;
  const int gpw = kWaveSize / lpr;
  const int g = lane / lpr;
  const int c = lane - g * lpr;
  for (int64_t t = blk - sc.tile_start;; t += sc.tiles_per_feat) {
    // Tile t of the sub-class: its feature and its place among the feature's tiles.
    int fi = -1;
    int64_t first = 0, n = 0, tile = 0, before = 0;
    for (int i0 = 0; i0 < sc.count; i0 += kWaveSize) {
      const int i = min(i0 + lane, sc.count - 1);
      const int ci = sc.first + i;
      const int pos = sc.key0 >= 0 ? sc.key0 + i : a.cdescs[ci].feature;
      int64_t f1, n1;
      sequence_bounds<IdxT>(a, ci, pos, s_starts, f1, n1);
      // (32-bit arithmetic: tiles of under 128 ids are taken only for calls of a few thousand tiles)
      const int tiles = i0 + lane < sc.count ? (int)((n1 + tile_ids - 1) / tile_ids) : 0;
      const int incl = wave_scan_incl((int32_t)tiles);
      const uint64_t past = __builtin_amdgcn_ballot_w64(before + incl > t);
      if (past != 0) {
        const int hit = __builtin_ctzll(past);
        fi = i0 + hit;
        first = __shfl(f1, hit, kWaveSize);
        n = __shfl(n1, hit, kWaveSize);
        tile = t - before - __shfl(incl - tiles, hit, kWaveSize);
        break;
      }
      before += wave_last(incl);
    }
    if (fi < 0) return;
    const FeatureDesc d = a.cdescs[__builtin_amdgcn_readfirstlane(sc.first + fi)];
    RowWalk w;
    w.chunk_off = Traits<DTYPE>::kHeader + d.payload_off + c * CB;
    w.lane_base = a.weights + d.table_offset + w.chunk_off;
    w.set_rows(d.rows, d.row_bytes);
    w.count_errors = c == 0 && g < gpw && d.payload_off == 0;
    w.hdr_lane = lane - c;
    w.sel0 = mfma_byte_selector(lane, 0);
    w.sel1 = mfma_byte_selector(lane, 1);
    const int64_t col = (int64_t)d.payload_off * 8 / Traits<DTYPE>::kBits;
    const int64_t begin = first + tile * tile_ids;
    const int64_t end = min(begin + tile_ids, first + n);
    // (a step's rows are dealt to the waves before the unroll, so a short tile still keeps all waves busy)
    for (int64_t j0 = begin + wave * gpw + g; j0 - g < end; j0 += kWavesPerBlock * gpw * U) {
      IdxT id[U];
      bool active[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t j = j0 + u * (kWavesPerBlock * gpw);
        active[u] = g < gpw && j < end;
        id[u] = reinterpret_cast<const IdxT*>(a.indices)[active[u] ? j : end - 1];
      }
      RowBuf<CB> r[U];
      int bad[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        bad[u] = fetch_row<DTYPE, CB, kUnweighted, IdxT>(r[u], id[u], (IdxT)0, (IdxT)0, a, w);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (bad[u] != 0 && active[u] && w.count_errors) atomicAdd(a.err_count, 1ull);
        if (bad[u] != 0 && a.bad_to_row0 != 0) r[u].valid = 1;  // the row fetched for it is row 0
        float acc[NE];
#pragma unroll
        for (int k = 0; k < NE; ++k) acc[k] = 0.0f;
        consume_row<DTYPE, CB, false>(acc, r[u], w);
        store_row<NE>(acc, a, (j0 + u * (kWavesPerBlock * gpw)) * (int64_t)d.dim + col, c, lpr, lane, active[u]);
      }
    }
  }
}

template <int DTYPE, int CB>
static void launch_sequence_cb(const LookupArgs& a, bool idx64, int grid, hipStream_t stream) {
  if (idx64)
    hipLaunchKernelGGL((tbe_nobag_kernel<DTYPE, CB, int64_t>), dim3(grid), dim3(kBlockThreads), 0, stream, a);
  else
    hipLaunchKernelGGL((tbe_nobag_kernel<DTYPE, CB, int32_t>), dim3(grid), dim3(kBlockThreads), 0, stream, a);
}

template <int DTYPE>
static bool launch_sequence_type(const LookupArgs& a, int cb, bool idx64, int grid, hipStream_t stream) {
  if (cb == 16) {
    if constexpr (DTYPE < kSplitHeader) launch_sequence_cb<DTYPE, 16>(a, idx64, grid, stream);
    return DTYPE < kSplitHeader;
  }
  if (cb == 8) {
    launch_sequence_cb<DTYPE, 8>(a, idx64, grid, stream);
    return true;
  }
  if (cb == 4) launch_sequence_cb<DTYPE, 4>(a, idx64, grid, stream);
  return cb == 4;
}

int launch_sequence(const LookupArgs& a, int dtype, int cb, bool split, bool idx64, int grid, hipStream_t stream) {
  bool ok = false;
  switch (split ? dtype + kSplitHeader : dtype) {
    case TRA_FP32: ok = launch_sequence_type<TRA_FP32>(a, cb, idx64, grid, stream); break;
    case TRA_FP16: ok = launch_sequence_type<TRA_FP16>(a, cb, idx64, grid, stream); break;
    case TRA_INT8: ok = launch_sequence_type<TRA_INT8>(a, cb, idx64, grid, stream); break;
    case TRA_INT4: ok = launch_sequence_type<TRA_INT4>(a, cb, idx64, grid, stream); break;
    case TRA_INT2: ok = launch_sequence_type<TRA_INT2>(a, cb, idx64, grid, stream); break;
    case TRA_INT8 + kSplitHeader: ok = launch_sequence_type<TRA_INT8 + kSplitHeader>(a, cb, idx64, grid, stream); break;
    case TRA_INT4 + kSplitHeader: ok = launch_sequence_type<TRA_INT4 + kSplitHeader>(a, cb, idx64, grid, stream); break;
    case TRA_INT2 + kSplitHeader: ok = launch_sequence_type<TRA_INT2 + kSplitHeader>(a, cb, idx64, grid, stream); break;
  }
  if (!ok) {
    set_error("bad chunk size %d", cb);
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TRA_OK : hip_fail(e, "sequence lookup launch");
}

}  // namespace tra
