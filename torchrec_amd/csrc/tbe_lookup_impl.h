// Gather + dequantize + pool kernels for packed int-N / fp16 / fp32 embedding
// rows (gfx950, wave64).  Included by one .hip file per weight type so the
// instantiations compile in parallel.
//
// Work mapping.  A row's payload is cut into chunks of CB bytes (16, 8 or 4);
// a lane owns one chunk, i.e. a fixed, contiguous set of output columns, and
// keeps one fp32 accumulator per column in registers.  LPR = payload / CB
// lanes form a lane group that owns one bag and walks its ids in order, so the
// sum is evaluated in exactly the order and with exactly the operations of the
// CPU kernels (acc = fmaf(w*scale, q, acc + w*bias)): no cross-lane reduction
// and no reassociation.  A wave holds 64 / LPR lane groups; rows are loaded
// with one CB-byte vector load per lane, U rows per lane group in flight, with
// the next U rows requested before the current U are consumed.
#pragma once

#include <hip/hip_fp16.h>

#include <type_traits>
#include <vector>

#include "tra_common.h"

namespace tra {

constexpr int kWavesPerBlock = 4;
constexpr int kBlockThreads = kWavesPerBlock * kWaveSize;
constexpr int kMaxSub = 8;
constexpr int kMaxPos = 128;

// Where a sequence lookup finds the range of ids of the feature at key position p.
constexpr int kBoundsOffsets = 0;  // offsets[p * B], offsets[(p + 1) * B]
constexpr int kBoundsTotals = 1;   // a.offsets is int64 totals[num_keys]: ids per key, at most kMaxTotalKeys keys
constexpr int kBoundsHost = 2;     // in the launch arguments: class feature ci starts at pw_off[ci], pw_len[ci] ids
constexpr int kMaxTotalKeys = 256;
// Sequence kernel: rows a lane group has in flight.
constexpr int kSequenceUnroll = 4;

// Features of one launch that share LPR (i.e. share dim).
struct SubClass {
  int32_t first;           // index of the first feature in the class feature list
  int32_t count;           // features in this sub-class
  int32_t lpr;             // lanes per row
  int32_t tiles_per_feat;  // blocks per feature
  int32_t tile_start;      // first block of this sub-class in the grid
  int32_t window;          // window kernel: bags per block; sequence kernel: ids per tile
  int32_t key0;            // key position of the first feature when the sub-class's features sit
                           // at consecutive key positions (feature fi at key0 + fi), else -1
};

struct LookupArgs {
  const uint8_t* weights;
  const FeatureDesc* descs;  // all features of the plan (device)
  const int32_t* feats;      // feature ids of this launch (device)
  const FeatureDesc* cdescs; // the same features' descriptors in launch order: cdescs[i] == descs[feats[i]]
  const void* indices;
  const void* offsets;
  const float* psw;
  void* out;
  int64_t out_stride;  // elements
  unsigned long long* err_count;
  int64_t num_indices;
  int32_t B;
  int32_t n_sub;  // window and sequence kernels
  int32_t mean;
  int32_t vec_store;  // 1: every lane's output slice is 16-byte aligned
  int32_t out_fp16;
  int32_t bad_to_row0;  // 1: an id outside its table (other than -1) reads row 0 instead of being skipped
  int32_t xcd_blocks;   // balanced pooled kernel: blocks per XCD (0: no XCD remap)
  int32_t xcd_count;    // balanced pooled kernel: XCDs the grid is dealt to
  int16_t feat_pos[kMaxPos];  // balanced pooled kernel: key position of the class's first features
  // Position weighting (posw != nullptr): the weight of the id at position k of
  // a bag of class feature ci is posw[pw_off[ci] + min(k, pw_len[ci] - 1)], or
  // 1 when pw_len[ci] is 0.  Takes the place of psw; classes of at most
  // kMaxPos features.
  const float* posw;
  int32_t pw_off[kMaxPos];
  int32_t pw_len[kMaxPos];
  // Sequence lookup: where a feature's ids lie (kBounds*).
  int32_t bounds_kind;
  int32_t num_keys;       // kBoundsTotals: input keys
#ifdef TRA_INSTRUMENT
  unsigned long long* ts;  // [waves][8] wall-clock stamps
#endif
  SubClass sub[kMaxSub];
};

// ---- element helpers ------------------------------------------------------
template <int DTYPE>
struct Traits;
template <>
struct Traits<TRA_INT8> {
  static constexpr int kBits = 8;
  static constexpr int kHeader = 4;
};
template <>
struct Traits<TRA_INT4> {
  static constexpr int kBits = 4;
  static constexpr int kHeader = 4;
};
template <>
struct Traits<TRA_INT2> {
  static constexpr int kBits = 2;
  static constexpr int kHeader = 4;
};
// Kernel-internal type codes for int-N rows too wide for one wave of lanes
// (more than 64 chunks of at most 8 bytes): such a row is cut into column
// slices, and only its first slice has the row header in front of it, so
// these variants load the header on its own (kHeaderWithChunk false).
constexpr int kSplitHeader = 16;
template <>
struct Traits<TRA_INT8 + kSplitHeader> : Traits<TRA_INT8> {};
template <>
struct Traits<TRA_INT4 + kSplitHeader> : Traits<TRA_INT4> {};
template <>
struct Traits<TRA_INT2 + kSplitHeader> : Traits<TRA_INT2> {};
// The weight type proper of a kernel type code.
constexpr int base_type(int dtype) { return dtype >= kSplitHeader ? dtype - kSplitHeader : dtype; }
// Does a lane load the dword in front of its chunk together with the chunk
// (for a row's first lane: the header)?  Rows with a header, 8- or 4-byte
// chunks, whole row in one slice.
template <int DTYPE, int CB>
constexpr bool header_with_chunk() { return Traits<DTYPE>::kHeader != 0 && CB <= 8 && DTYPE < kSplitHeader; }

template <>
struct Traits<TRA_FP16> {
  static constexpr int kBits = 16;
  static constexpr int kHeader = 0;
};
template <>
struct Traits<TRA_FP32> {
  static constexpr int kBits = 32;
  static constexpr int kHeader = 0;
};

template <int CB>
struct Chunk {
  uint32_t v[CB / 4];
};

// CB bytes from a 4-byte aligned address in one vector load.
template <int CB>
__device__ __forceinline__ Chunk<CB> load_chunk(const uint8_t* p) {
  Chunk<CB> c;
  __builtin_memcpy(&c, __builtin_assume_aligned(p, 4), CB);
  return c;
}

// Byte K of x as float: a single v_cvt_f32_ubyteK.  Written as inline asm
// because the compiler otherwise extracts the byte first (v_bfe / SDWA and)
// and then converts, which costs a second VALU op per element.
template <int K>
__device__ __forceinline__ float byte_to_float(uint32_t x) {
  float f;
  if constexpr (K == 0)
    asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(f) : "v"(x));
  else if constexpr (K == 1)
    asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(f) : "v"(x));
  else if constexpr (K == 2)
    asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(f) : "v"(x));
  else
    asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(f) : "v"(x));
  return f;
}

typedef float float2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float half_bits_to_float(uint32_t h) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}

// acc = fmaf(s, q, acc + b): one rounded add, then one fused multiply-add.
__device__ __forceinline__ void fma_step(float& acc, float s, float q, float b) {
  float t = acc + b;
  acc = __builtin_fmaf(s, q, t);
}

// Sub-byte fields to floats on the matrix core.  Eight bytes 0x00 .. 0x0f per
// lane (two payload dwords' worth of masked fields) become eight floats with
// two v_mfma_f32_16x16x32_bf8_fp8: the lane's bytes are one column slice of the
// B operand (FP8 E4M3: a byte 0x0q is exactly q * 2^-9, subnormals and the
// first binade), the A operand holds 2^9 (BF8 0x60) where row m selects byte
// (m & 3) [+ 4] of lane group m >> 2, and C is zero; so output register r of a
// lane is 2^9 * (its own byte r [+ 4]) plus exact zeros: the integer q, with no
// rounding anywhere.  This takes the conversions (one v_cvt_pk_f32_fp8 per two
// elements otherwise) off the vector ALU, which the pooling loop saturates;
// the matrix core runs beside it.
typedef float float4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ long mfma_byte_selector(int lane, int half) {
  const int m = lane & 15, gp = lane >> 4;
  unsigned long long v = 0;
  if (gp == (m >> 2)) v = 0x60ull << (8 * ((m & 3) + 4 * half));
  return (long)v;
}

// Accumulate the elements of one payload dword.  `acc` points at the
// accumulators of this dword's elements.  int4 / int2 fields are converted on
// the matrix core (mfma_byte_selector above; sel0 / sel1 are the lane's two
// selector operands), int8 bytes by v_cvt_f32_ubyteN.
template <int DTYPE_CODE, bool WEIGHTED, bool MATRIX>
__device__ __forceinline__ void accumulate_dword(float* acc, uint32_t x, float s,
                                                 float b, long sel0, long sel1) {
  constexpr int DTYPE = base_type(DTYPE_CODE);
  if constexpr (DTYPE == TRA_INT4 && MATRIX) {
    // Low nibbles in the low dword, high nibbles in the high dword of the
    // matrix instruction's 8-byte operand; element 2k is byte k's low nibble.
    const uint32_t lo = x & 0x0f0f0f0fu;
    const uint32_t hi = (x >> 4) & 0x0f0f0f0fu;
    const long data = (long)(((unsigned long long)hi << 32) | lo);
    const float4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
    const float4_t l = __builtin_amdgcn_mfma_f32_16x16x32_bf8_fp8(sel0, data, z, 0, 0, 0);
    const float4_t h = __builtin_amdgcn_mfma_f32_16x16x32_bf8_fp8(sel1, data, z, 0, 0, 0);
    fma_step(acc[0], s, l[0], b);
    fma_step(acc[1], s, h[0], b);
    fma_step(acc[2], s, l[1], b);
    fma_step(acc[3], s, h[1], b);
    fma_step(acc[4], s, l[2], b);
    fma_step(acc[5], s, h[2], b);
    fma_step(acc[6], s, l[3], b);
    fma_step(acc[7], s, h[3], b);
  } else if constexpr (DTYPE == TRA_INT8) {
    fma_step(acc[0], s, byte_to_float<0>(x), b);
    fma_step(acc[1], s, byte_to_float<1>(x), b);
    fma_step(acc[2], s, byte_to_float<2>(x), b);
    fma_step(acc[3], s, byte_to_float<3>(x), b);
  } else if constexpr (DTYPE == TRA_INT4 && !WEIGHTED) {
    // (16-byte lane chunks: 32 accumulators per lane leave no registers for the
    // matrix instruction's operands and results, so the vector ALU converts.)
    // A byte 0x0q read as an FP8 (E4M3) value is exactly q * 2^-9 for q = 0..15
    // (subnormals, then the first binade), and one instruction converts two
    // bytes.  The scale is multiplied by 2^9 instead (exact: s is at most
    // 65504 here), so every product is the same real number as s * q.
    const uint32_t lo = x & 0x0f0f0f0fu;
    const uint32_t hi = (x >> 4) & 0x0f0f0f0fu;
    const float s9 = s * 512.0f;
    const float2_t l01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, false);
    const float2_t l23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, true);
    const float2_t h01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, false);
    const float2_t h23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, true);
    fma_step(acc[0], s9, l01.x, b);
    fma_step(acc[1], s9, h01.x, b);
    fma_step(acc[2], s9, l01.y, b);
    fma_step(acc[3], s9, h01.y, b);
    fma_step(acc[4], s9, l23.x, b);
    fma_step(acc[5], s9, h23.x, b);
    fma_step(acc[6], s9, l23.y, b);
    fma_step(acc[7], s9, h23.y, b);
  } else if constexpr (DTYPE == TRA_INT4) {
    // With per-sample weights the scale w*scale may be subnormal, where a
    // multiplication by 2^9 is inexact, so the fields are shifted down instead.
    const uint32_t lo = x & 0x0f0f0f0fu;
    const uint32_t hi = (x >> 4) & 0x0f0f0f0fu;
    fma_step(acc[0], s, byte_to_float<0>(lo), b);
    fma_step(acc[1], s, byte_to_float<0>(hi), b);
    fma_step(acc[2], s, byte_to_float<1>(lo), b);
    fma_step(acc[3], s, byte_to_float<1>(hi), b);
    fma_step(acc[4], s, byte_to_float<2>(lo), b);
    fma_step(acc[5], s, byte_to_float<2>(hi), b);
    fma_step(acc[6], s, byte_to_float<3>(lo), b);
    fma_step(acc[7], s, byte_to_float<3>(hi), b);
  } else if constexpr (DTYPE == TRA_INT2 && MATRIX) {
    // The four 2-bit fields of every byte, two field positions per pair of
    // matrix instructions; element 4 * k + e is field e of byte k.
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
      const uint32_t m0 = (x >> (2 * e)) & 0x03030303u;
      const uint32_t m1 = (x >> (2 * e + 2)) & 0x03030303u;
      const long data = (long)(((unsigned long long)m1 << 32) | m0);
      const float4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
      const float4_t l = __builtin_amdgcn_mfma_f32_16x16x32_bf8_fp8(sel0, data, z, 0, 0, 0);
      const float4_t h = __builtin_amdgcn_mfma_f32_16x16x32_bf8_fp8(sel1, data, z, 0, 0, 0);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        fma_step(acc[4 * k + e], s, l[k], b);
        fma_step(acc[4 * k + e + 1], s, h[k], b);
      }
    }
  } else if constexpr (DTYPE == TRA_INT2 && !WEIGHTED) {
    // Same FP8 reading as for int4, on the four 2-bit fields of every byte.
    const float s9 = s * 512.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t m = (x >> (2 * e)) & 0x03030303u;
      const float2_t m01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)m, false);
      const float2_t m23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)m, true);
      fma_step(acc[0 + e], s9, m01.x, b);
      fma_step(acc[4 + e], s9, m01.y, b);
      fma_step(acc[8 + e], s9, m23.x, b);
      fma_step(acc[12 + e], s9, m23.y, b);
    }
  } else if constexpr (DTYPE == TRA_INT2) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t m = (x >> (2 * e)) & 0x03030303u;
      fma_step(acc[0 + e], s, byte_to_float<0>(m), b);
      fma_step(acc[4 + e], s, byte_to_float<1>(m), b);
      fma_step(acc[8 + e], s, byte_to_float<2>(m), b);
      fma_step(acc[12 + e], s, byte_to_float<3>(m), b);
    }
  } else if constexpr (DTYPE == TRA_FP16) {
    // s carries the per-sample weight (1.0f when unweighted).
    acc[0] = __builtin_fmaf(s, half_bits_to_float(x & 0xffffu), acc[0]);
    acc[1] = __builtin_fmaf(s, half_bits_to_float(x >> 16), acc[1]);
  } else {
    acc[0] = __builtin_fmaf(s, __builtin_bit_cast(float, x), acc[0]);
  }
}

template <typename T>
__device__ __forceinline__ int64_t load_index(const void* p, int64_t i) {
  return (int64_t) reinterpret_cast<const T*>(p)[i];
}

// One prefetched row chunk.
template <int CB>
struct RowBuf {
  Chunk<CB> d;
  uint32_t hdr;
  float w;
  int valid;  // 1: accumulate; 0: skip
};

// Everything a lane needs to walk rows of its feature's table.
struct RowWalk {
  const uint8_t* lane_base;  // table + this lane's chunk offset inside a row
  int64_t rows;
  uint32_t rows32;     // min(rows, 2^31): bound for int32 ids
  uint32_t row_bytes;
  int chunk_off;
  bool count_errors;
  // Where a lane loads the dword in front of its chunk together with the chunk
  // (header_with_chunk), the row's header arrives in the row's first lane.
  int hdr_lane;
  // Selector operands of the matrix instruction that converts int4 / int2
  // fields (mfma_byte_selector); they depend on the lane only.
  long sel0, sel1;
  // position weighting: this bag's weight vector (always readable), its last
  // index, whether the feature has one at all, and where the bag starts
  const float* pw;
  uint32_t pw_last;
  bool pw_on;
  int64_t bag_start;
  __device__ __forceinline__ void set_position_weights(const LookupArgs& a, int ci, int64_t start);
  __device__ __forceinline__ void set_rows(int64_t r, int32_t rb) {
    rows = r;
    rows32 = r < (int64_t(1) << 31) ? (uint32_t)r : 0x80000000u;
    row_bytes = (uint32_t)rb;
  }
};

__device__ __forceinline__ void RowWalk::set_position_weights(const LookupArgs& a, int ci,
                                                              int64_t start) {
  pw = a.posw;
  pw_last = 0;
  pw_on = false;
  bag_start = start;
  if (a.posw != nullptr) {
    const int n = ci < kMaxPos ? a.pw_len[ci] : 0;
    pw_on = n > 0;
    pw = a.posw + (n > 0 ? a.pw_off[ci] : 0);
    pw_last = (uint32_t)(n > 0 ? n - 1 : 0);
  }
}

// Id of position j, or -1 (= skip) when the position is outside the bag.  The
// load itself is unconditional (position clamped into the ids array) and the
// result is selected afterwards: a load under a lane predicate would be
// followed by a full wait at the re-convergence point and serialize the ids.
template <typename IdxT>
__device__ __forceinline__ IdxT fetch_id(const LookupArgs& a, bool in_range, IdxT j, IdxT last) {
  // Ids and positions stay in the width of the index type: with int32 ids the
  // whole address computation is 32-bit (plus one 64-bit add to the base).
  using UIdxT = typename std::make_unsigned<IdxT>::type;
  const IdxT jc = (UIdxT)j < (UIdxT)last ? j : last;  // also catches a wrapped position
  const IdxT id = reinterpret_cast<const IdxT*>(a.indices)[jc];
  return in_range ? id : (IdxT)-1;
}

// Values of the kernels' WEIGHTED parameter: how a row's weight is obtained.
constexpr int kUnweighted = 0;
constexpr int kPerSample = 1;   // psw[j]
constexpr int kByPosition = 2;  // position weight of the id's place in its bag

// Issue the loads of one row chunk (header dword, CB payload bytes, weight).
// Branch-free: an id outside [0, rows) (a pruned id -1, a lane past the end of
// its bag, or a bad id) is redirected to row 0 and flagged invalid; consume_row
// then multiplies it away exactly.  Returns 1 for a bad id (out of range and
// not -1).
// GIVEN_W: the caller already holds the row's weight (`given_w`), fetched a
// lane group at a time like the ids; no weight load is issued here.
template <int DTYPE, int CB, int WEIGHTED, typename IdxT, bool GIVEN_W = false>
__device__ __forceinline__ int fetch_row(RowBuf<CB>& r, IdxT id, IdxT j, IdxT last,
                                          const LookupArgs& a, const RowWalk& w, float given_w = 1.0f) {
  const uint8_t* lane_base = w.lane_base;  // table + this lane's chunk offset
  const int chunk_off = w.chunk_off;
  bool valid;
  const uint8_t* chunk;
  if constexpr (sizeof(IdxT) == 4) {
    // One unsigned compare covers negative ids; the row address is a single
    // 32 x 32 + 64 bit multiply-add.
    valid = (uint32_t)id < w.rows32;
    const uint32_t idc = valid ? (uint32_t)id : 0u;
    chunk = lane_base + (uint64_t)idc * (uint64_t)w.row_bytes;
  } else {
    valid = (uint64_t)id < (uint64_t)w.rows;
    const int64_t idc = valid ? (int64_t)id : 0;
    chunk = lane_base + idc * (int64_t)w.row_bytes;
  }
  if constexpr (header_with_chunk<DTYPE, CB>()) {
    // One load: the dword in front of the lane's chunk and the chunk.  For the
    // row's first lane that dword is the header; consume_row hands it round.
    const Chunk<CB + 4> t = load_chunk<CB + 4>(chunk - 4);
    r.hdr = t.v[0];
#pragma unroll
    for (int i = 0; i < CB / 4; ++i) r.d.v[i] = t.v[i + 1];
  } else {
    if constexpr (Traits<DTYPE>::kHeader != 0)
      r.hdr = *reinterpret_cast<const uint32_t*>(chunk - chunk_off);
    else
      r.hdr = 0;
    r.d = load_chunk<CB>(chunk);
  }
  if constexpr (WEIGHTED != 0 && GIVEN_W) {
    r.w = given_w;
  } else if constexpr (WEIGHTED) {
    using UIdxT = typename std::make_unsigned<IdxT>::type;
    if constexpr (WEIGHTED == kByPosition) {
      // The weight of this id's place in its bag, clamped into the feature's
      // weight vector (a slot past the end of its bag reads some valid weight
      // and is dropped later); 1 for a feature without position weights.
      const UIdxT k = (UIdxT)(j - (IdxT)w.bag_start);
      const uint32_t kc = k < (UIdxT)w.pw_last ? (uint32_t)k : w.pw_last;
      const float v = w.pw[kc];
      r.w = w.pw_on ? v : 1.0f;
    } else {
      const IdxT jc = (UIdxT)j < (UIdxT)last ? j : last;
      r.w = a.psw[jc];
    }
  } else {
    r.w = 1.0f;
  }
  r.valid = valid;
  return (!valid && id != (IdxT)-1) ? 1 : 0;
}

// Accumulate one fetched row chunk.  An invalid row contributes fmaf(+0, q,
// acc + (+0)), which leaves acc unchanged bit-for-bit: acc is never -0 (it
// starts at +0 and a round-to-nearest sum is -0 only if both addends are), and
// q is a finite integer.  For fp16 / fp32 rows the payload of an invalid row is
// zeroed as well, so a stored inf / nan in row 0 cannot leak in.
// Every lane of the wave calls this (trip counts are wave-uniform, skipped rows
// and rows past an end are masked, never branched around): the matrix
// instruction reads its operands from all 64 lanes whatever the execution mask.
template <int DTYPE, int CB, bool WEIGHTED>
__device__ __forceinline__ void consume_row(float* acc, const RowBuf<CB>& r0, const RowWalk& w) {
  constexpr int EPD = 32 / Traits<DTYPE>::kBits;  // elements per dword
  RowBuf<CB> r = r0;
  if constexpr (header_with_chunk<DTYPE, CB>())
    r.hdr = (uint32_t)__shfl((int)r0.hdr, w.hdr_lane, kWaveSize);  // the header sits with the row's first lane
  float s, b;
  if constexpr (Traits<DTYPE>::kHeader != 0) {
    if constexpr (WEIGHTED) {
      // The weight of a skipped slot is whatever lies at the clamped
      // position, possibly inf / nan: select after the products.
      s = r.w * half_bits_to_float(r.hdr & 0xffffu);
      b = r.w * half_bits_to_float(r.hdr >> 16);
      s = r.valid ? s : 0.0f;
      b = r.valid ? b : 0.0f;
    } else {
      const uint32_t hdr = r.valid ? r.hdr : 0u;  // scale = bias = +0
      s = half_bits_to_float(hdr & 0xffffu);
      b = half_bits_to_float(hdr >> 16);
    }
    // int4 fields go through the matrix core where a lane holds at most 16
    // accumulators (8-byte chunks), int2 fields always.
    constexpr bool kMatrix = Traits<DTYPE>::kBits == 2 || (Traits<DTYPE>::kBits == 4 && CB <= 8);
    if constexpr (kMatrix)
      asm volatile("" : "+v"(s));  // the converted scale stays in a register: no fp16 operand in the fused multiply-adds
#pragma unroll
    for (int i = 0; i < CB / 4; ++i)
      accumulate_dword<DTYPE, WEIGHTED, kMatrix>(acc + i * EPD, r.d.v[i], s, b, w.sel0, w.sel1);
  } else {
    s = r.valid ? r.w : 0.0f;
#pragma unroll
    for (int i = 0; i < CB / 4; ++i)
      accumulate_dword<DTYPE, WEIGHTED, false>(acc + i * EPD, r.valid ? r.d.v[i] : 0u, s, 0.0f, 0, 0);
  }
}

// Store NE consecutive outputs starting at element `pos`.  `vec`: every lane's
// output slice is 16-byte aligned.
template <int NE>
__device__ __forceinline__ void store_outputs(const LookupArgs& a, int64_t pos,
                                              const float* acc, bool vec) {
  if (a.out_fp16) {
    __half* o = reinterpret_cast<__half*>(a.out) + pos;
    if constexpr (NE >= 8) {
      if (vec) {
#pragma unroll
        for (int i = 0; i < NE; i += 8) {
          uint4 v;
          uint32_t* pv = reinterpret_cast<uint32_t*>(&v);
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint32_t lo = __half_as_ushort(__float2half_rn(acc[i + 2 * k]));
            const uint32_t hi = __half_as_ushort(__float2half_rn(acc[i + 2 * k + 1]));
            pv[k] = lo | (hi << 16);
          }
          *reinterpret_cast<uint4*>(o + i) = v;
        }
        return;
      }
    }
#pragma unroll
    for (int i = 0; i < NE; ++i) o[i] = __float2half_rn(acc[i]);
  } else {
    float* o = reinterpret_cast<float*>(a.out) + pos;
    if constexpr (NE >= 4) {
      if (vec) {
#pragma unroll
        for (int i = 0; i < NE; i += 4)
          *reinterpret_cast<float4*>(o + i) =
              make_float4(acc[i], acc[i + 1], acc[i + 2], acc[i + 3]);
        return;
      }
    }
#pragma unroll
    for (int i = 0; i < NE; ++i) o[i] = acc[i];
  }
}

__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const int o = __shfl_xor(v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}

// Built with -DTRA_INSTRUMENT (never in the shipped library), every wave
// records wall-clock stamps at the phases of the window kernel into a.ts; a
// standalone harness that includes this header reads them back.
#ifdef TRA_INSTRUMENT
#define TRA_STAMP(k)                                                                      \
  do {                                                                                    \
    if ((threadIdx.x & 63) == 0)                                                          \
      a.ts[((size_t)blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64) * 8 + (k)] = wall_clock64(); \
  } while (0)
#else
#define TRA_STAMP(k)
#endif

constexpr int kNarrowLane = 8;  // accumulators per lane up to which one instance serves all widths (see odd_lanes)
constexpr int kFewAccumulators = 16;  // per lane, up to which the compiler keeps the pooling loop's loads in flight by itself

// ---- pooled lookup ----------------------------------------------------------

// Pool one bag per lane group: ids [start, start + len), in order, into acc.
// max_len is the longest bag among the wave's lane groups (wave-uniform trip
// count).  Software pipeline, per lane group: ids are requested two batches of
// U rows ahead, row chunks one batch ahead, so neither an id load nor a row
// load is waited for in the batch that issued it.
template <int DTYPE, int CB, typename IdxT, int WEIGHTED, int U, int NE>
__device__ __forceinline__ int pool_bag(float (&acc)[NE], const LookupArgs& a,
                                         const RowWalk& w, int64_t start64, int len,
                                         int max_len_any_lane) {
  // Wave-uniform by construction; telling the compiler keeps the loop control
  // on the scalar unit and the loads free of lane-mask bookkeeping.
  const int max_len = __builtin_amdgcn_readfirstlane(max_len_any_lane);
  const IdxT start = (IdxT)start64;
  const IdxT last = (IdxT)(a.num_indices - 1);
  IdxT idA[U], idB[U];
  RowBuf<CB> bufA[U], bufB[U];
  int bad = 0;
  // Row slots at or beyond max_len belong to no lane group: the (wave-uniform)
  // tests below skip their loads and their arithmetic altogether.
#pragma unroll
  for (int u = 0; u < U; ++u) idA[u] = fetch_id<IdxT>(a, u < len, start + u, last);
#pragma unroll
  for (int u = 0; u < U; ++u) idB[u] = fetch_id<IdxT>(a, U + u < len, start + U + u, last);
#pragma unroll
  for (int u = 0; u < U; ++u)
    bad += fetch_row<DTYPE, CB, WEIGHTED, IdxT>(bufA[u], idA[u], start + u, last, a, w);
  for (int it = 0; it < max_len; it += 2 * U) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      idA[u] = fetch_id<IdxT>(a, it + 2 * U + u < len, start + it + 2 * U + u, last);
#pragma unroll
    for (int u = 0; u < U; ++u)
      bad += fetch_row<DTYPE, CB, WEIGHTED, IdxT>(bufB[u], idB[u], start + it + U + u, last, a, w);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (it + u < max_len) consume_row<DTYPE, CB, (WEIGHTED != 0)>(acc, bufA[u], w);
    if (it + U >= max_len) break;
#pragma unroll
    for (int u = 0; u < U; ++u)
      idB[u] = fetch_id<IdxT>(a, it + 3 * U + u < len, start + it + 3 * U + u, last);
#pragma unroll
    for (int u = 0; u < U; ++u)
      bad += fetch_row<DTYPE, CB, WEIGHTED, IdxT>(bufA[u], idA[u], start + it + 2 * U + u, last, a, w);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (it + U + u < max_len) consume_row<DTYPE, CB, (WEIGHTED != 0)>(acc, bufB[u], w);
  }
  // Bad ids are counted by the lane that owns column 0.
  if (bad != 0 && w.count_errors) atomicAdd(a.err_count, (unsigned long long)bad);
  return bad;
}

// The same pooling with the ids fetched a block at a time: lane c of the group
// loads id number c of a block, and each row's id is then passed to the group's
// lanes with a cross-lane read, so there is one id load per block instead of
// one per row.  The block after the current one, requested when the current one
// is entered, is at least two batches ahead, like the ids of pool_bag.
//
// P == 0: a block is lpr ids (a power of two, 16 or more).
// P > 0: a block is the 2 * U ids of one loop iteration, in 2 * U / P loads of P
// ids each (the lane group has at least P lanes; those beyond load ids of the
// next blocks and nobody reads them).  The block then changes at a fixed
// place in the loop and its load is unconditional, so the number of loads in
// flight is the same on every path and the compiler can wait for the oldest
// batch alone.  (Behind a conditional load it has to assume the worst and
// drains all loads, which undoes the double buffering once per iteration.)
template <int DTYPE, int CB, typename IdxT, int WEIGHTED, int U, int NE, int P>
__device__ __forceinline__ int pool_bag_bulk(float (&acc)[NE], const LookupArgs& a,
                                              const RowWalk& w, int64_t start64, int len,
                                              int max_len_any_lane, int lpr, int c,
                                              int group_lane0) {
  constexpr bool TWO_BATCHES = P > 0;
  constexpr int LOADS = TWO_BATCHES ? 2 * U / P : 1;  // loads (registers) per block
  const int max_len = __builtin_amdgcn_readfirstlane(max_len_any_lane);
  const int block = TWO_BATCHES ? 2 * U : __builtin_amdgcn_readfirstlane(lpr);
  const IdxT start = (IdxT)start64;
  const IdxT last = (IdxT)(a.num_indices - 1);
  struct IdBlock { IdxT v[LOADS]; };
  struct WeightBlock { float v[LOADS]; };
  auto load_block = [&](int j) -> IdBlock {
    IdBlock x;
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
      const int r = j * block + k * P + c;
      x.v[k] = fetch_id<IdxT>(a, r < len, start + (IdxT)r, last);
    }
    return x;
  };
  // Weights travel the same way: the lane that loads an id loads its weight
  // (per-sample weights: psw at that position; position weights: the table
  // entry of that place in the bag).
  auto load_weights = [&](int j) -> WeightBlock {
    WeightBlock x;
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
      const int r = j * block + k * P + c;
      if constexpr (WEIGHTED == kPerSample) {
        using UIdxT = typename std::make_unsigned<IdxT>::type;
        const IdxT p = start + (IdxT)r;
        x.v[k] = a.psw[(UIdxT)p < (UIdxT)last ? p : last];
      } else if constexpr (WEIGHTED == kByPosition) {
        const float v = w.pw[(uint32_t)r < w.pw_last ? (uint32_t)r : w.pw_last];
        x.v[k] = w.pw_on ? v : 1.0f;
      } else {
        x.v[k] = 1.0f;
      }
    }
    return x;
  };
  IdBlock cur = load_block(0);
  IdBlock nxt = load_block(1);
  WeightBlock wcur = load_weights(0);
  WeightBlock wnxt = load_weights(1);
  int cur_j = 0;
  // Id of row r (wave-uniform), or -1 past the bag's end.  r lies in the
  // current block: a batch of U rows never straddles two blocks and enter() is
  // called before each batch.  Reading `cur` only matters: a select between
  // cur and nxt would wait for the load of nxt that enter() has just issued.
  // `at`: row r's place in its loop iteration (known at compile time).
  auto id_of = [&](int r, int at) -> IdxT {
    if constexpr (TWO_BATCHES)
      return (IdxT)__shfl(cur.v[at / P], group_lane0 + at % P, kWaveSize);
    else
      return (IdxT)__shfl(cur.v[0], group_lane0 + (r - cur_j * block), kWaveSize);
  };
  auto weight_of = [&](int r, int at) -> float {
    if constexpr (WEIGHTED == 0)
      return 1.0f;
    else if constexpr (TWO_BATCHES)
      return __shfl(wcur.v[at / P], group_lane0 + at % P, kWaveSize);
    else
      return __shfl(wcur.v[0], group_lane0 + (r - cur_j * block), kWaveSize);
  };
  // The step to the next block, where it is known to happen (P > 0: at every second batch).
  auto advance = [&]() {
    cur = nxt;
    ++cur_j;
    nxt = load_block(cur_j + 1);
    if constexpr (WEIGHTED != 0) {
      wcur = wnxt;
      wnxt = load_weights(cur_j + 1);
    }
  };
  // Entering the block of row rb: make it the current one and request the next.
  auto enter = [&](int rb) {
    if (rb / block > cur_j) advance();
  };
  RowBuf<CB> bufA[U], bufB[U];
  int bad = 0;
#pragma unroll
  for (int u = 0; u < U; ++u)
    bad += fetch_row<DTYPE, CB, WEIGHTED, IdxT, true>(bufA[u], id_of(u, u), start + u, last, a, w, weight_of(u, u));
  int it = 0;
  if constexpr (TWO_BATCHES) {
    // Whole iterations (2 * U rows, all inside the longest bag) run without the
    // per-row tests: every buffer is consumed on the way round, so the
    // compiler knows at the top of the loop that only the newest batch and
    // the id block are in flight and need not drain them before it reuses a
    // consumed buffer's registers.  The last, partial iteration follows below.
    // (With 32 accumulators a lane a batch's loads are held in front of the batch consumed meanwhile: short of registers,
    // the compiler puts each behind the row before it, and waits for it at once.  41 K bags of 20 ids of 1 M int4 rows of
    // 256 columns 52.0 us, so 42.8.  With 64 it is better left to the compiler: 41 K position-weighted bags of 20 ids of 512
    // cached int2 columns 109 us held, 86 not.)
    for (; it + 2 * U <= max_len; it += 2 * U) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        bad += fetch_row<DTYPE, CB, WEIGHTED, IdxT, true>(bufB[u], id_of(it + U + u, U + u), start + it + U + u, last, a, w, weight_of(it + U + u, U + u));
      if constexpr (NE == 2 * kFewAccumulators) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u) consume_row<DTYPE, CB, (WEIGHTED != 0)>(acc, bufA[u], w);
      advance();
#pragma unroll
      for (int u = 0; u < U; ++u)
        bad += fetch_row<DTYPE, CB, WEIGHTED, IdxT, true>(bufA[u], id_of(it + 2 * U + u, u), start + it + 2 * U + u, last, a, w, weight_of(it + 2 * U + u, u));
      if constexpr (NE == 2 * kFewAccumulators) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u) consume_row<DTYPE, CB, (WEIGHTED != 0)>(acc, bufB[u], w);
    }
  }
  for (; it < max_len; it += 2 * U) {
    if constexpr (!TWO_BATCHES) enter(it + U);
#pragma unroll
    for (int u = 0; u < U; ++u)
      bad += fetch_row<DTYPE, CB, WEIGHTED, IdxT, true>(bufB[u], id_of(it + U + u, U + u), start + it + U + u, last, a, w, weight_of(it + U + u, U + u));
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (it + u < max_len) consume_row<DTYPE, CB, (WEIGHTED != 0)>(acc, bufA[u], w);
    if (it + U >= max_len) break;
    if constexpr (TWO_BATCHES) advance(); else enter(it + 2 * U);
#pragma unroll
    for (int u = 0; u < U; ++u)
      bad += fetch_row<DTYPE, CB, WEIGHTED, IdxT, true>(bufA[u], id_of(it + 2 * U + u, u), start + it + 2 * U + u, last, a, w, weight_of(it + 2 * U + u, u));
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (it + U + u < max_len) consume_row<DTYPE, CB, (WEIGHTED != 0)>(acc, bufB[u], w);
  }
  if (bad != 0 && w.count_errors) atomicAdd(a.err_count, (unsigned long long)bad);
  return bad;
}

// The bags of a wave pooled once more, where the launch wants an id outside
// its table to pool row 0 (what fbgemm's bounds_check_indices makes of such an
// id in its WARNING and IGNORE modes: it rewrites it to 0) and one of the
// wave's bags held such an id.  The pooling loops above skip it; since the
// order of the additions is part of the result, the bag cannot be corrected
// afterwards and is pooled again from zero, one row at a time (rare by
// assumption: bad ids are an input error).  Bad ids are not counted again.
template <int DTYPE, int CB, typename IdxT, int WEIGHTED, int NE>
__device__ __forceinline__ void repool_bad_ids_as_row0(float (&acc)[NE], const LookupArgs& a,
                                                    const RowWalk& w, int64_t start64, int len,
                                                    int max_len_any_lane) {
  const int max_len = __builtin_amdgcn_readfirstlane(max_len_any_lane);
  const IdxT start = (IdxT)start64;
  const IdxT last = (IdxT)(a.num_indices - 1);
#pragma unroll
  for (int k = 0; k < NE; ++k) acc[k] = 0.0f;
  for (int r = 0; r < max_len; ++r) {
    const IdxT id = fetch_id<IdxT>(a, r < len, start + (IdxT)r, last);
    RowBuf<CB> buf;
    fetch_row<DTYPE, CB, WEIGHTED, IdxT>(buf, id, start + (IdxT)r, last, a, w);
    if (id != (IdxT)-1) buf.valid = 1;  // fetch_row has redirected an id outside the table to row 0
    consume_row<DTYPE, CB, (WEIGHTED != 0)>(acc, buf, w);
  }
}

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// Vector v (16 bytes) of a lane's NE outputs.
template <int NE, bool FP16>
__device__ __forceinline__ u32x4_t out_vector(const float (&acc)[NE], int v) {
  u32x4_t x;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (FP16) {
      const uint32_t lo = __half_as_ushort(__float2half_rn(acc[8 * v + 2 * k]));
      const uint32_t hi = __half_as_ushort(__float2half_rn(acc[8 * v + 2 * k + 1]));
      x[k] = lo | (hi << 16);
    } else {
      x[k] = __builtin_bit_cast(uint32_t, acc[4 * v + k]);
    }
  }
  return x;
}

// Results leave a wave through LDS: where a lane holds V 16-byte vectors of a row, storing them as they lie would write
// a part of every line with each store instruction.  Room per lane, in vectors:
constexpr int kStageVectors = 4;
// Where a wave puts vector k of lane's V: lane by lane, the vectors of neighbouring lanes in different banks.
template <int V>
__device__ __forceinline__ int stage_slot(int lane, int k) {
  return lane * V + (k ^ (lane & (V - 1)));
}

// LDS accesses of the lanes of one wave in order: what they have written is visible to its other lanes.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}

// A vector of a row of results.  Results are written once and read by a later kernel: with the non-temporal hint (`past`
// the caches), or, where the rest of a line follows with another store instruction, into them until it has come.
__device__ __forceinline__ void store_vector(u32x4_t x, u32x4_t* to, bool past) {
  if (past) {
    __builtin_nontemporal_store(x, to);
  } else {
    // (fenced: the compiler makes one store of the two otherwise, without the hint)
    asm volatile("" ::: "memory");
    *to = x;
    asm volatile("" ::: "memory");
  }
}

// Lane c of a group holds NE columns of the group's row from `row` on, on 16-byte boundaries.  The lanes of a group change
// their vectors in LDS, kStageVectors of each at a time, so that a store instruction writes whole runs of the row.
// Calls of 213 K bags of two cached ids, us, vectors stored as they lie (two a lane exchanged by cross-lane reads, for
// lane groups of powers of two) / this: fp32 results, int8 256 columns 102 / 55, int8 128 50 / 32, int4 128 49 / 32, 34
// features of int8 128 and 256 90 / 59; fp16 results, int2 128 33 / 27, int8 256 49 / 48; 65 K bags of 20, int8 256 to
// fp16 51 / 48, to fp32 57 / 49.
// OWN: two vectors of a lane that is alone, or in a group of no power of two, are stored as they lie: 213 K bags of two
// ids to fp32, int8 104 39.6 and through LDS 41.5, int4 104 39.8 and 41.4, fp16 104 37.8 and 39.7, 78 K bags of eight, int8
// 72 17.5 and 18.0.  (Not in the several-class kernel, whose bodies it costs 4 to 10 registers in scratch memory: 60 K
// position-weighted bags of two ids 23.0 / 23.6.)
// The hint pays where a store instruction writes whole lines of a row (int8 256 to fp32, without / with, 84 / 55), and below
// that in groups of powers of two with two vectors a lane (two ids a bag, int4 64 to fp16 21.6 / 20.2, int4 32 17.8 / 17.2; eight,
// int8 32 to fp32 12.8 / 11.9) and of four lanes with four fp16 vectors (int2 128, two ids 25.6 / 26.7, eight 18.3 / 16.8, 41 K
// bags of 20 ids of 1 M rows 26.7 / 25.3), but not elsewhere: int2 128 to fp32 33 / 42, int4 64 to fp32 23 / 26, int2 64 to fp16
// 21 / 30, int8 40 - 104 to fp32 36 / 40, int2 48 - 112 to fp16 28 / 34.
template <int NE, bool FP16, bool OWN>
__device__ __forceinline__ void store_group_row(const float (&acc)[NE], u32x4_t* stage, unsigned char* row, int c,
                                                int lpr, int lane, bool active) {
  constexpr int V = NE * (FP16 ? 2 : 4) / 16;
  const bool two_to_n = lpr >= 2 && (lpr & (lpr - 1)) == 0;
  const bool past = (V <= kStageVectors && lpr % 8 == 0) || (V == 2 && two_to_n) || (FP16 && V == 4 && lpr == 4);
  if (V == 1 || (OWN && V == 2 && lpr % 8 != 0 && !two_to_n)) {
    if (active)
#pragma unroll
      for (int v = 0; v < V; ++v) store_vector(out_vector<NE, FP16>(acc, v), reinterpret_cast<u32x4_t*>(row) + c * V + v, past);
  } else {
    // (Places in LDS are computed where they are used: kept through the pooling loop they would push its registers out.)
    asm volatile("" : "+v"(lane), "+v"(c));
    constexpr int P = V < kStageVectors ? V : kStageVectors;
#pragma unroll
    for (int h = 0; h < V; h += P) {
      wave_lds_sync();
#pragma unroll
      for (int k = 0; k < P; ++k) stage[stage_slot<P>(lane, k)] = out_vector<NE, FP16>(acc, h + k);
      wave_lds_sync();
#pragma unroll
      for (int k = 0; k < P; ++k) {
        const int i = k * lpr + c;  // which of the group's vectors this lane stores
        const int from = min(lane - c + i / P, kWaveSize - 1);  // (lanes behind the last whole group)
        const u32x4_t x = stage[stage_slot<P>(from, i % P)];
        if (active) store_vector(x, reinterpret_cast<u32x4_t*>(row) + (i / P * V + h + i % P), past);
      }
    }
  }
}

// Finish one bag per lane group (MEAN scaling, rounding, store).  Lane c of the
// group's lpr lanes holds the NE outputs at columns row_pos + c * NE.  Every
// lane of the wave calls this; `active` says whether its group holds a bag.
// `stage`: the wave's room in LDS, 64 * kStageVectors vectors.
template <int NE, bool OWN>
__device__ __forceinline__ void finish_bag(float (&acc)[NE], const LookupArgs& a, u32x4_t* stage, int len,
                                           int64_t row_pos, int c, int lpr, int lane, bool active, bool vec) {
  if (a.mean && len > 0) {
    const float inv = 1.0f / (float)len;
#pragma unroll
    for (int i = 0; i < NE; ++i) acc[i] *= inv;
  }
  if (vec) {
    unsigned char* row = reinterpret_cast<unsigned char*>(a.out) + row_pos * (a.out_fp16 ? 2 : 4);
    if constexpr (NE >= 8) {
      if (a.out_fp16) {
        store_group_row<NE, true, OWN>(acc, stage, row, c, lpr, lane, active);
        return;
      }
    }
    if constexpr (NE >= 4) {
      if (!a.out_fp16) {
        store_group_row<NE, false, OWN>(acc, stage, row, c, lpr, lane, active);
        return;
      }
    }
  }
  if (active) store_outputs<NE>(a, row_pos + (int64_t)c * NE, acc, vec);
}

// Balanced mapping.  One 1024-thread block per compute unit owns a window of
// consecutive bags (of one sub-class, possibly spanning features).  It ranks
// them by length in LDS, longest first, and cuts the order into rounds of gpw
// bags; a round is pooled by one wave, one bag per lane group, so the lane
// groups that run in lock step hold bags of nearly equal length.  Rounds are
// dealt to the four SIMDs in serpentine order (waves w, w+4, w+8, w+12 share SIMD
// w & 3); a SIMD's waves take its rounds as they become free.  A bag is still pooled whole and in id order by one lane group; there is no
// scratch memory, atomic or pre-pass.
#ifndef TRA_CU_THREADS  // (measurement builds override these two)
#define TRA_CU_THREADS 1024
#endif
#ifndef TRA_MAX_WINDOW
#define TRA_MAX_WINDOW 2048
#endif
constexpr int kCuThreads = TRA_CU_THREADS;
constexpr int kCuWaves = kCuThreads / kWaveSize;
static_assert(kCuWaves >= 2, "the window kernel splits its prologue between the first wave and the others");
constexpr int kMaxWindow = TRA_MAX_WINDOW;
constexpr int kBagBits = 20;  // window entry = (feature index in sub-class << 20) | sample

constexpr int kLenBins = 256;
constexpr int kMaxWinFeat = 32;  // feature descriptors a window keeps in LDS

// Sort key of a bag length: exact below 192, then steps of 64, then one bin.
// (A negative length, which only a malformed input holds, ranks as empty.)
__device__ __forceinline__ int length_bin(int len) {
  return len < 192 ? max(len, 0) : min(kLenBins - 1, 192 + ((len - 192) >> 6));
}

// Accumulator of the from-lengths prologue: as wide as the index type (with
// int32 offsets every partial sum fits 32 bits by definition).
template <typename IdxT>
struct SumOf { using type = int64_t; };
template <>
struct SumOf<int32_t> { using type = int32_t; };

// This thread's share of sum(lengths[0 .. p)).  The block reads the range 16
// bytes per lane per step, kPrefixBatch independent loads at a time (a lane's
// index past the end is clamped and its value dropped, so no load is
// predicated).
// start() adds up every batch but the last and leaves the last one in flight;
// finish() adds it, so the last round trip overlaps whatever the caller does
// between the two calls.
// Every block of the grid reads a prefix of the same array at the same moment;
// starting each block at a different 16 KB step to spread the L2 channels
// measured the same as all starting at the front, so they start at the front.
// `lengths` is 16-byte aligned.
constexpr int kPrefixBatch = 8;

template <typename IdxT>
struct PrefixSum {
  using S = typename SumOf<IdxT>::type;
  static constexpr int V = 16 / (int)sizeof(IdxT);
  struct __align__(16) Vec { IdxT v[V]; };

  const Vec* vin;
  int nvec, nk, last, k_last;
  S part;
  IdxT tail;
  Vec x[kPrefixBatch];

  // Step k of this thread covers vector k * kCuThreads + threadIdx.x; a step
  // past the end reads the last vector again (clamped) and adds nothing.
  __device__ __forceinline__ Vec fetch(int k) const {
    return vin[min(k * kCuThreads + (int)threadIdx.x, last)];
  }
  __device__ __forceinline__ void add(int k, const Vec& v) {
    S sum = 0;
#pragma unroll
    for (int i = 0; i < V; ++i) sum += (S)v.v[i];
    part += k * kCuThreads + (int)threadIdx.x < nvec ? sum : (S)0;
  }
  __device__ __forceinline__ void issue(int k0) {
#pragma unroll
    for (int k = 0; k < kPrefixBatch; ++k) x[k] = fetch(k0 + k);
  }
  __device__ __forceinline__ void consume(int k0) {
#pragma unroll
    for (int k = 0; k < kPrefixBatch; ++k) add(k0 + k, x[k]);
  }
  __device__ __forceinline__ void start(const IdxT* __restrict__ lengths, int64_t p) {
    vin = reinterpret_cast<const Vec*>(lengths);
    nvec = (int)(p / V);
    nk = (nvec + kCuThreads - 1) / kCuThreads;
    last = max(nvec - 1, 0);
    part = 0;
    // the elements after the last whole 16-byte step: one per lane, clamped like the rest
    const int64_t rest = p - (int64_t)nvec * V;
    const int64_t ti = (int64_t)nvec * V + min((int64_t)threadIdx.x, max(rest - 1, (int64_t)0));
    tail = lengths[max(min(ti, p - 1), (int64_t)0)];
    if ((int64_t)threadIdx.x >= rest) tail = 0;
    k_last = nk > 0 ? ((nk - 1) / kPrefixBatch) * kPrefixBatch : 0;
    // kPrefixBatch loads stay in flight: each step adds the oldest (loads
    // return in issue order) and puts the load of the step one batch ahead
    // in its place.  The last batch is left for finish().
    issue(0);
    for (int k0 = 0; k0 < k_last; k0 += kPrefixBatch) {
#pragma unroll
      for (int k = 0; k < kPrefixBatch; ++k) {
        add(k0 + k, x[k]);
        x[k] = fetch(k0 + kPrefixBatch + k);
      }
    }
  }
  __device__ __forceinline__ S finish() {
    consume(k_last);
    return part + (S)tail;
  }
};

// The same sum for waves that have nothing else in flight: the number of loads
// follows the length of the range (in steps of four per thread), and all of
// them are requested before the first is waited for.
template <typename IdxT>
struct PrefixSumAtOnce {
  using S = typename SumOf<IdxT>::type;
  static constexpr int V = 16 / (int)sizeof(IdxT);
  struct __align__(16) Vec { IdxT v[V]; };
  const Vec* vin;
  int tid, nt, nvec, last;

  template <int N, bool TWO>
  __device__ __forceinline__ void steps(int k0, S& part, int nvec2, S& part2) const {
    Vec x[N];
#pragma unroll
    for (int k = 0; k < N; ++k) x[k] = vin[min((k0 + k) * nt + tid, last)];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      S sum = 0;
#pragma unroll
      for (int i = 0; i < V; ++i) sum += (S)x[k].v[i];
      part += (k0 + k) * nt + tid < nvec ? sum : (S)0;
      if constexpr (TWO) part2 += (k0 + k) * nt + tid < nvec2 ? sum : (S)0;
    }
  }
  // The elements of [0, p) after the last whole 16-byte step: one per thread.
  __device__ __forceinline__ S tail(const IdxT* __restrict__ lengths, int64_t p) const {
    const int64_t whole = p / V * V, rest = p - whole;
    const int64_t ti = whole + min((int64_t)tid, max(rest - 1, (int64_t)0));
    const IdxT x = lengths[max(min(ti, p - 1), (int64_t)0)];
    return (int64_t)tid < rest ? (S)x : (S)0;
  }
  // This thread's share of sum(lengths[0 .. p)) and, TWO, of sum(lengths[0 .. p2)), both in one go over the longer of
  // the two; thread tid_ of nt_.
  template <bool TWO>
  __device__ __forceinline__ void run(const IdxT* __restrict__ lengths, int64_t p, int64_t p2, int tid_, int nt_,
                                      S& part, S& part2) {
    tid = tid_;
    nt = nt_;
    vin = reinterpret_cast<const Vec*>(lengths);
    nvec = (int)(p / V);
    const int nvec2 = TWO ? (int)(p2 / V) : 0, most = max(nvec, nvec2);
    last = max(most - 1, 0);
    const int nk = (most + nt - 1) / nt;
    const S tail1 = tail(lengths, p), tail2 = TWO ? tail(lengths, p2) : (S)0;
    part = part2 = 0;
    int k0 = 0;
    for (; nk - k0 > 16; k0 += 16) steps<16, TWO>(k0, part, nvec2, part2);
    const int r = nk - k0;
    if (r > 12)
      steps<16, TWO>(k0, part, nvec2, part2);
    else if (r > 8)
      steps<12, TWO>(k0, part, nvec2, part2);
    else if (r > 4)
      steps<8, TWO>(k0, part, nvec2, part2);
    else if (r > 0)
      steps<4, TWO>(k0, part, nvec2, part2);
    part += tail1;
    part2 += tail2;
  }
  __device__ __forceinline__ S run(const IdxT* __restrict__ lengths, int64_t p, int tid_, int nt_) {
    S part, none;
    run<false>(lengths, p, 0, tid_, nt_, part, none);
    return part;
  }
};

// Inclusive scan over the 64 lanes of a wave.  32-bit sums use the data-parallel
// lane moves of the VALU (shifts inside each row of 16 lanes, then lane 15 and
// lane 31 broadcast into the following rows): six adds, no trip through the LDS
// crossbar.  Lanes without a source receive 0.
__device__ __forceinline__ int32_t wave_scan_incl(int32_t v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}
__device__ __forceinline__ int64_t wave_scan_incl(int64_t v) {
  const int ln = threadIdx.x & (kWaveSize - 1);
#pragma unroll
  for (int off = 1; off < kWaveSize; off <<= 1) {
    const int64_t o = __shfl_up(v, off, kWaveSize);
    if (ln >= off) v += o;
  }
  return v;
}
// A value that is the same in every lane, in scalar registers.
__device__ __forceinline__ int32_t uniform(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uniform(int64_t v) {
  return (int64_t)(((uint64_t)(uint32_t)uniform((int32_t)(v >> 32)) << 32) | (uint32_t)uniform((int32_t)v));
}
// Lane 63's value of v, in every lane.
__device__ __forceinline__ int32_t wave_last(int32_t v) { return __builtin_amdgcn_readlane(v, kWaveSize - 1); }
__device__ __forceinline__ int64_t wave_last(int64_t v) { return __shfl(v, kWaveSize - 1, kWaveSize); }

// Position of feature `fi` of a sub-class among the input keys: from the launch
// arguments when the class is small enough, else from the descriptors.
__device__ __forceinline__ int feat_key_pos(const LookupArgs& a, const SubClass& sc, int fi) {
  if (sc.key0 >= 0) return sc.key0 + fi;  // no load: the bag bounds can be requested at once
  return sc.first + fi < kMaxPos ? (int)a.feat_pos[sc.first + fi]
                                 : a.descs[a.feats[sc.first + fi]].feature;
}

// A window's bags in LDS, in arrays of their own (so that the compiler can tell
// accesses to one from accesses to another).
template <typename IdxT>
struct Window {
  using Sum = typename SumOf<IdxT>::type;
  int64_t* start;
  int* len;
  uint32_t* ent;
  uint16_t* order;
  uint16_t* slot;
  int* hist;
  FeatureDesc* desc;
  Sum* red;
  Sum* wave_tot;
  int* taken;  // [4] rounds that a SIMD's waves have asked for after their first
  u32x4_t* stage;  // 64 * kStageVectors vectors of results per wave
};
#define TRA_WINDOW(IdxT, name)                                                                       \
  __shared__ int64_t s_start[kMaxWindow];                                                            \
  __shared__ __align__(16) int s_len[kMaxWindow];                                                    \
  __shared__ uint32_t s_ent[kMaxWindow];                                                             \
  __shared__ uint16_t s_order[kMaxWindow];                                                           \
  __shared__ uint16_t s_slot[kMaxWindow];                                                            \
  __shared__ int s_hist[kLenBins];                                                                   \
  __shared__ FeatureDesc s_desc[kMaxWinFeat];                                                        \
  __shared__ typename SumOf<IdxT>::type s_red[kCuWaves], s_wave_tot[kCuWaves];                       \
  __shared__ int s_taken[4];                                                                            \
  __shared__ u32x4_t s_stage[kCuWaves * kWaveSize * kStageVectors];                                  \
  const Window<IdxT> name{s_start, s_len, s_ent, s_order, s_slot, s_hist, s_desc, s_red, s_wave_tot, s_taken, s_stage}

// What a staged window's bag starts in LDS still lack: `add`, and from the sub-class's feature `second` on `second_add`.
template <typename Sum>
struct WindowStarts {
  Sum add = 0, second_add = 0;
  int second = INT32_MAX;
};

// The launch arguments that pooling reads, asked for together while the window is staged: fetched one behind the
// other after the staging's barrier, as the compiler places them, they cost every wave a trip to memory each with
// nothing else in flight (graph replays, us, without / with this: 26 int4 tables of 128 columns, 2048 samples
// 19.1 / 18.7; 16 int2 tables of 256 columns, 2048 samples 20.8 / 20.5; 8 fp16 tables, 8192 samples 18.0 / 17.85).
__device__ __forceinline__ void hold_pool_args(const LookupArgs& a) {
  asm volatile("" ::"s"(a.weights), "s"(a.cdescs), "s"(a.indices), "s"(a.out), "s"(a.out_stride), "s"(a.num_indices),
               "s"(a.mean), "s"(a.vec_store), "s"(a.out_fp16), "s"(a.bad_to_row0));
}

// Stages bags [q0, q0 + nb) of a sub-class and ranks them by length.
// FROM_LENGTHS: p_offsets points at the KJT's lengths instead of its offsets
// and the block derives its bags' start positions itself: one block-wide sum
// of everything in front of the window plus a scan of the window in LDS.
template <typename IdxT, bool FROM_LENGTHS>
__device__ __forceinline__ WindowStarts<typename SumOf<IdxT>::type> stage_window(
    const Window<IdxT> w, const LookupArgs& a, const void* p_offsets, const FeatureDesc* p_cdescs, int32_t p_B,
    const SubClass& sc, int q0, int nb, int fi_lo) {
  using Sum = typename SumOf<IdxT>::type;

  // Bag q0 + i of the window: where it sits in the offsets (or lengths) array.
  auto bag_of = [&](int i, int& fi, int& b) -> int64_t {
    const int q = q0 + i;
    fi = q / p_B;
    b = q - fi * p_B;
    return (int64_t)feat_key_pos(a, sc, fi) * p_B + b;
  };
  WindowStarts<Sum> starts;
  if (threadIdx.x < 4) w.taken[threadIdx.x] = 0;
  // A window of at most 4 x 64 bags is staged, scanned and ranked by the
  // block's first wave alone, four consecutive bags per lane, with no block
  // barrier on the way; from lengths, the other fifteen waves meanwhile sum
  // the lengths in front of the window.  One barrier joins the two.
  // The features' keys need not follow one another: a window whose bags lie in
  // two runs has both runs' fronts summed in one go (graph replays, us, the
  // general route for keys out of order / this: 26 int4 tables of 128 columns, 2048
  // samples 31.1 / 29.2; 64 int8 tables of 64 columns, 300 samples 15.4 / 13.9, 40 of
  // them, 1000 samples of 64-bit ids 26.8 / 24.2; a position-weighted call of 20
  // features 22.8 / 21.3).
  bool solo = FROM_LENGTHS && nb <= 4 * kWaveSize;
  int key_lo = 0, key_second = 0;  // key positions of the window's first feature and of the second run's
  if (solo) {
    key_lo = feat_key_pos(a, sc, fi_lo);
    if (sc.key0 < 0) {
      const int fi_hi = (q0 + nb - 1) / p_B;
      int before = key_lo;
      for (int fi = fi_lo + 1; fi <= fi_hi; ++fi) {
        const int key = feat_key_pos(a, sc, fi);
        if (key != before + 1) {
          solo = solo && starts.second == INT32_MAX;
          starts.second = fi;
          key_second = key;
        }
        before = key;
      }
    }
  }
  if (solo) {
    const int wv = threadIdx.x / kWaveSize;
    const int ln = threadIdx.x & (kWaveSize - 1);
    if (wv == 0) {
      IdxT given[4];  // lengths as they stand in the KJT (lanes past the window repeat its last bag)
      int fis[4], bs[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int q = q0 + min(4 * ln + k, nb - 1);
        fis[k] = q / p_B;
        bs[k] = q - fis[k] * p_B;
        const int key = fis[k] < starts.second ? key_lo + (fis[k] - fi_lo) : key_second + (fis[k] - starts.second);
        given[k] = reinterpret_cast<const IdxT*>(p_offsets)[(int64_t)key * p_B + bs[k]];
      }
      {
        const int nfeat = min((q0 + nb - 1) / p_B - fi_lo + 1, kMaxWinFeat);
        if (ln < nfeat) w.desc[ln] = p_cdescs[sc.first + fi_lo + ln];
      }
#pragma unroll
      for (int k = 0; k < kLenBins / kWaveSize; ++k) w.hist[ln + k * kWaveSize] = 0;
      wave_lds_sync();
      TRA_STAMP(6);
      int len[4], slot[4];
      Sum raw[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = 4 * ln + k;
        raw[k] = 0;
        len[k] = 0;
        slot[k] = 0;
        if (i < nb) {
          // Kept as given: bag starts are the running sum of the lengths as
          // they are; a negative length only makes its own bag empty.
          raw[k] = (Sum)given[k];
          len[k] = (int)given[k];
          w.len[i] = len[k];
          w.ent[i] = ((uint32_t)fis[k] << kBagBits) | (uint32_t)bs[k];
          slot[k] = atomicAdd(&w.hist[length_bin(len[k])], 1);
        }
      }
      // Bag starts inside the window: exclusive scan in window order.
      const Sum tot = raw[0] + raw[1] + raw[2] + raw[3];
      Sum run = wave_scan_incl(tot) - tot;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (4 * ln + k < nb) w.start[4 * ln + k] = (int64_t)run;
        run += raw[k];
      }
      if (ln == 0) w.red[0] = 0;
      wave_lds_sync();
      hold_pool_args(a);
      TRA_STAMP(7);
      TRA_STAMP(1);
      {  // counting sort, longest first (as in the general route below)
        int h[kLenBins / kWaveSize];
        int sum = 0;
#pragma unroll
        for (int k = 0; k < kLenBins / kWaveSize; ++k) {
          h[k] = w.hist[kLenBins - 1 - (ln * (kLenBins / kWaveSize) + k)];
          sum += h[k];
        }
        const int incl = wave_scan_incl((int32_t)sum);
        int base = incl - sum;
#pragma unroll
        for (int k = 0; k < kLenBins / kWaveSize; ++k) {
          w.hist[kLenBins - 1 - (ln * (kLenBins / kWaveSize) + k)] = base;
          base += h[k];
        }
      }
      wave_lds_sync();
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (4 * ln + k < nb) w.order[w.hist[length_bin(len[k])] + slot[k]] = (uint16_t)(4 * ln + k);
    } else {
      PrefixSumAtOnce<IdxT> front_sum;
      const IdxT* lengths = reinterpret_cast<const IdxT*>(p_offsets);
      const int64_t p = (int64_t)key_lo * p_B + (q0 - fi_lo * p_B);
      const int tid = (int)threadIdx.x - kWaveSize, nt = kCuThreads - kWaveSize;
      Sum mine, second;
      if (starts.second == INT32_MAX) {
        mine = front_sum.run(lengths, p, tid, nt);
      } else {
        front_sum.template run<true>(lengths, p, (int64_t)key_second * p_B, tid, nt, mine, second);
        second = wave_last(wave_scan_incl(second));
        if (ln == 0) w.wave_tot[wv] = second;
      }
      hold_pool_args(a);
      const Sum front_w = wave_last(wave_scan_incl(mine));
      if (ln == 0) w.red[wv] = front_w;
    }
    lds_barrier();
#pragma unroll
    for (int v = 0; v < kCuWaves; ++v) starts.add += w.red[v];
    if (starts.second != INT32_MAX) {
      // (its bags' starts in LDS go on from the first run's)
      starts.second_add = (Sum)-w.start[starts.second * p_B - q0];
#pragma unroll
      for (int v = 1; v < kCuWaves; ++v) starts.second_add += w.wave_tot[v];
      starts.second_add = uniform(starts.second_add);
    }
    starts.add = uniform(starts.add);
    TRA_STAMP(2);
  } else {
    // The first bag of every thread is requested before anything else: the
    // barrier below waits for outstanding loads, and this way the bag bounds
    // and the descriptors share one memory latency instead of queueing up.
    IdxT first_lo = 0, first_hi = 0;
    if ((int)threadIdx.x < nb) {
      int fi, b;
      const int64_t bag = bag_of(threadIdx.x, fi, b);
      first_lo = reinterpret_cast<const IdxT*>(p_offsets)[bag];
      if (!FROM_LENGTHS) first_hi = reinterpret_cast<const IdxT*>(p_offsets)[bag + 1];
    }
    // Descriptors of the features this window touches, kept in LDS so that a
    // round does not start with two dependent global loads.
    {
      const int nfeat = min((q0 + nb - 1) / p_B - fi_lo + 1, kMaxWinFeat);
      if ((int)threadIdx.x < nfeat) w.desc[threadIdx.x] = p_cdescs[sc.first + fi_lo + threadIdx.x];
    }
    // From lengths: the total of everything in front of the window.  Its loads
    // go out after the window's own (loads return in order: whatever is waited
    // for first has to be issued first) and stay in flight until the scan
    // below needs the sum.
    PrefixSum<IdxT> front_sum;
    if (FROM_LENGTHS)
      front_sum.start(reinterpret_cast<const IdxT*>(p_offsets),
                      (int64_t)feat_key_pos(a, sc, fi_lo) * p_B + (q0 - fi_lo * p_B));
    if (threadIdx.x < kLenBins) w.hist[threadIdx.x] = 0;
    lds_barrier();
    TRA_STAMP(6);
    for (int i = threadIdx.x; i < nb; i += kCuThreads) {
      int fi, b;
      const int64_t bag = bag_of(i, fi, b);
      const bool first = i == (int)threadIdx.x;
      int len;
      if (FROM_LENGTHS) {
        // Kept as given: bag starts are the running sum of the lengths as they
        // are (what a separate cumsum would produce); a negative length only
        // makes its own bag empty.
        len = (int)(first ? (int64_t)first_lo : load_index<IdxT>(p_offsets, bag));
      } else {
        const int64_t st = first ? (int64_t)first_lo : load_index<IdxT>(p_offsets, bag);
        const int64_t en = first ? (int64_t)first_hi : load_index<IdxT>(p_offsets, bag + 1);
        w.start[i] = st;
        len = max(0, (int)(en - st));
      }
      w.len[i] = len;
      w.ent[i] = ((uint32_t)fi << kBagBits) | (uint32_t)b;
      w.slot[i] = (uint16_t)atomicAdd(&w.hist[length_bin(len)], 1);
    }
    lds_barrier();
    TRA_STAMP(7);
    if (FROM_LENGTHS) {
      const int t = threadIdx.x;
      const int wv = t / kWaveSize;
      const int ln = t & (kWaveSize - 1);
      // Exclusive scan of the window's lengths (window order): two bags per
      // thread, wave scan, then the 16 wave totals.  The same barrier carries
      // the block-wide total of everything in front of the window.
      // (Only the waves that hold bags scan; every instruction that all 16 waves
      // of the block execute costs 16 issue cycles per SIMD.)
      const bool holds_bags = 2 * wv * kWaveSize < nb;
      Sum x0 = 0, x1 = 0, inc = 0;
      if (holds_bags) {
        x0 = 2 * t < nb ? w.len[2 * t] : 0;
        x1 = 2 * t + 1 < nb ? w.len[2 * t + 1] : 0;
        inc = wave_scan_incl((Sum)(x0 + x1));
      }
      const Sum front_w = wave_last(wave_scan_incl(front_sum.finish()));
      if (ln == kWaveSize - 1) w.wave_tot[wv] = inc;
      if (ln == 0) w.red[wv] = front_w;
      lds_barrier();
      Sum before = 0, front = 0;
#pragma unroll
      for (int v = 0; v < kCuWaves; ++v) front += w.red[v];
      if (holds_bags) {
#pragma unroll
        for (int v = 0; v < kCuWaves; ++v)
          if (v < wv) before += w.wave_tot[v];
      }
      const Sum excl = before + inc - (x0 + x1);
      // The window covers bags of features fi_lo .. fi_hi of the sub-class.  A
      // feature's bags are contiguous in `lengths`; where the next feature's
      // key position follows directly, the run simply continues.
      const int fi_hi = (q0 + nb - 1) / p_B;
      bool one_run = true;
      if (sc.key0 < 0)
        for (int fi = fi_lo; fi < fi_hi; ++fi) one_run = one_run && feat_key_pos(a, sc, fi + 1) == feat_key_pos(a, sc, fi) + 1;
      if (one_run) {
        if (2 * t < nb) w.start[2 * t] = (int64_t)(front + excl);
        if (2 * t + 1 < nb) w.start[2 * t + 1] = (int64_t)(front + excl + x0);
        lds_barrier();
      } else {
        // General case: keep the bare scan, then add to each run what lies in
        // front of it (summed again for every run that does not continue the
        // previous one).
        if (2 * t < nb) w.start[2 * t] = (int64_t)excl;
        if (2 * t + 1 < nb) w.start[2 * t + 1] = (int64_t)(excl + x0);
        lds_barrier();
        int64_t adj = (int64_t)front;  // start = adj + scan value, for the current run
        int64_t next_pos = -1;
        for (int fi = fi_lo; fi <= fi_hi; ++fi) {
          const int first = max(0, fi * p_B - q0);        // first bag of this feature in the window
          const int last = min(nb, (fi + 1) * p_B - q0);  // one past its last bag
          const int64_t pos = (int64_t)feat_key_pos(a, sc, fi) * p_B + (q0 + first - fi * p_B);
          if (fi != fi_lo && pos != next_pos) {
            PrefixSum<IdxT> again;
            again.start(reinterpret_cast<const IdxT*>(p_offsets), pos);
            const Sum w_ = wave_last(wave_scan_incl(again.finish()));
            if (ln == 0) w.red[wv] = w_;
            lds_barrier();
            Sum total = 0;
#pragma unroll
            for (int v = 0; v < kCuWaves; ++v) total += w.red[v];
            adj = (int64_t)total - w.start[first];
          }
          next_pos = pos + (last - first);
          lds_barrier();  // w.red and w.start[first] have been read by everyone
          for (int i = first + t; i < last; i += kCuThreads) w.start[i] += adj;
          lds_barrier();
        }
      }
    }
    TRA_STAMP(1);
    // Counting sort, longest first: a permutation of 0..nb-1.  hist[] holds the
    // bin sizes and every bag already has its slot within its bin; one wave
    // turns the sizes into start positions (bins in descending order).
    if (threadIdx.x < kWaveSize) {
      const int l = threadIdx.x;
      int h[kLenBins / kWaveSize];
      int sum = 0;
#pragma unroll
      for (int k = 0; k < kLenBins / kWaveSize; ++k) {
        h[k] = w.hist[kLenBins - 1 - (l * (kLenBins / kWaveSize) + k)];
        sum += h[k];
      }
      const int incl = wave_scan_incl((int32_t)sum);
      int base = incl - sum;
#pragma unroll
      for (int k = 0; k < kLenBins / kWaveSize; ++k) {
        w.hist[kLenBins - 1 - (l * (kLenBins / kWaveSize) + k)] = base;
        base += h[k];
      }
    }
    lds_barrier();
    for (int i = threadIdx.x; i < nb; i += kCuThreads)
      w.order[w.hist[length_bin(w.len[i])] + w.slot[i]] = (uint16_t)i;
    lds_barrier();
    TRA_STAMP(2);
  }

  return starts;
}

// Which pooling bodies a kernel instance holds (see odd_lanes).
constexpr int kBodiesOdd = 1;   // id blocks of four for every lane group of four lanes or more
constexpr int kBodiesMany = 2;  // the same, one body of several in a kernel
constexpr int kBodiesEven = 0;  // id blocks for powers of two from eight lanes, for others where the registers allow

// Pools a staged window.  vec(): whether every lane's output slice is 16-byte aligned (asked where a bag is stored).
template <int DTYPE, int CB, typename IdxT, int WEIGHTED, int U, int BODIES, typename Vec>
__device__ __forceinline__ void pool_window(const Window<IdxT> win, const LookupArgs& a, const SubClass& sc, int nb,
                                            int fi_lo, const WindowStarts<typename SumOf<IdxT>::type> starts,
                                            Vec&& vec) {
  constexpr int NE = CB * 8 / Traits<DTYPE>::kBits;
  constexpr bool ODD = BODIES != kBodiesEven, kOwn = BODIES != kBodiesMany;
  // Where a lane holds more than 16 accumulators, what the pooling loop does not need is found anew behind it (the lane's
  // place in the wave, where its bag's results go): kept, it would push the loop's registers out.  Registers in scratch
  // memory, int4 in 16-byte chunks, 32-bit ids from lengths, without, with per-sample and with position weights: 16, 16 and
  // 24 with all of it kept, 4, 5 and 4 so.
  constexpr bool kWide = NE > kFewAccumulators;
  const auto lane_now = [&] {
    if constexpr (!kWide) return (int)(threadIdx.x & (kWaveSize - 1));
    int none = 0;
    asm volatile("" : "+v"(none));
    return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, none));
  };
  const int wave = uniform((int)(threadIdx.x / kWaveSize));
  const int lpr = sc.lpr;
  const int gpw = kWaveSize / lpr;
  const int rounds = (nb + gpw - 1) / gpw;
  // Rounds are ordered longest first and dealt to the four SIMDs (waves w, w + 4, w + 8 and w + 12 share one) in alternating
  // direction.  A wave's first one is fixed; after that it takes the next one of its SIMD that nobody has: waves of equal work
  // end at very different times (64 rounds of the same length, four a wave: the first wave done after 190 us, the last after
  // 340), and a compute unit that a part of its waves has left keeps fewer requests in flight.  One counter for all
  // SIMDs gives rounds to the waves that are free first, and so two of four that are left to one SIMD.  us, fixed
  // throughout / one counter / one a SIMD: bags of 80 cached ids, twenty rounds a block, weighted int4 512 columns
  // 72.8 / 77.2 / 71.9, int8 256 44.8 / 47.9 / 44.4; bags of 20, forty rounds, int8 256 32.1 / 29.9 / 29.6, int2 512
  // 92.5 / 83.7 / 84.1.
  const auto round_of = [](int simd, int k) { return 4 * k + ((k & 1) ? 3 - simd : simd); };
  for (int r = round_of(wave & 3, wave >> 2); r < rounds;) {
    const auto bag_at = [&](int g, bool& active, int& i, int& fi, int& b) {
      const int pos = r * gpw + g;
      active = g < gpw && pos < nb;
      i = win.order[active ? pos : r * gpw];
      const uint32_t ent = win.ent[i];
      fi = (int)(ent >> kBagBits);
      b = (int)(ent & ((1u << kBagBits) - 1));
    };
    bool active;
    int i, fi, b;
    const int lane = lane_now(), g = lane / lpr, c = lane - g * lpr;
    bag_at(g, active, i, fi, b);
    const FeatureDesc d = fi - fi_lo < kMaxWinFeat ? win.desc[fi - fi_lo] : a.cdescs[sc.first + fi];
    const int64_t start = win.start[i] + (int64_t)(fi < starts.second ? starts.add : starts.second_add);
    const int len = active ? max(win.len[i], 0) : 0;
    // The round's trip count.  Lengths below 192 have a sort bin each, so
    // the round's first bag is its longest; from 192 up a bin holds a range of
    // lengths in arrival order, and the longest of the round is found by
    // comparing what the lane groups actually hold.
    int max_len = win.len[win.order[r * gpw]];
    if (max_len >= 192) max_len = wave_max(len);

    RowWalk w;
    w.chunk_off = Traits<DTYPE>::kHeader + d.payload_off + c * CB;
    w.lane_base = a.weights + d.table_offset + w.chunk_off;
    // The lanes behind the last whole group read ids of other groups where pool_bag_bulk's cross-lane
    // read passes lane 63: for them every id lies outside the table, so none of its rows is fetched.
    w.set_rows(g < gpw ? d.rows : 0, d.row_bytes);
    w.count_errors = c == 0 && g < gpw && d.payload_off == 0;
    w.hdr_lane = lane - c;
    w.sel0 = mfma_byte_selector(lane, 0);
    w.sel1 = mfma_byte_selector(lane, 1);
    w.set_position_weights(a, sc.first + fi, start);

    float acc[NE];
#pragma unroll
    for (int k = 0; k < NE; ++k) acc[k] = 0.0f;
    int bad;
    // Which bodies an instance holds: see odd_lanes.
    constexpr bool kAllWidths = NE <= kNarrowLane || (CB == 4 && NE <= 2 * kNarrowLane);
    if constexpr (U == 4 && ODD) {
      if (lpr >= 4)
        bad = pool_bag_bulk<DTYPE, CB, IdxT, WEIGHTED, U, NE, 4>(acc, a, w, start, len, max_len, lpr, c, lane - c);
      else
        bad = pool_bag<DTYPE, CB, IdxT, WEIGHTED, U, NE>(acc, a, w, start, len, max_len);
    } else if constexpr (U == 4) {
      if (lpr >= 16 && (lpr & (lpr - 1)) == 0)
        bad = pool_bag_bulk<DTYPE, CB, IdxT, WEIGHTED, U, NE, 0>(acc, a, w, start, len, max_len, lpr, c, lane - c);
      else if (kAllWidths ? lpr >= 8 : lpr == 8)
        bad = pool_bag_bulk<DTYPE, CB, IdxT, WEIGHTED, U, NE, 8>(acc, a, w, start, len, max_len, lpr, c, lane - c);
      else if (kAllWidths && lpr >= 4)
        bad = pool_bag_bulk<DTYPE, CB, IdxT, WEIGHTED, U, NE, 4>(acc, a, w, start, len, max_len, lpr, c, lane - c);
      else
        bad = pool_bag<DTYPE, CB, IdxT, WEIGHTED, U, NE>(acc, a, w, start, len, max_len);
    } else {
      bad = pool_bag<DTYPE, CB, IdxT, WEIGHTED, U, NE>(acc, a, w, start, len, max_len);
    }
    if (a.bad_to_row0 != 0 && __builtin_amdgcn_ballot_w64(bad != 0 && g < gpw) != 0)
      repool_bad_ids_as_row0<DTYPE, CB, IdxT, WEIGHTED, NE>(acc, a, w, start, len, max_len);
    TRA_STAMP(3);
#ifdef TRA_INSTRUMENT
    if (lane == 0) a.ts[((size_t)blockIdx.x * (blockDim.x / 64) + wave) * 8 + 5] = (unsigned long long)max_len;
#endif
    // (what hangs on the wave's number is computed here: kept through the loop it would push scalar registers out)
    int w0 = wave;
    asm volatile("" : "+s"(w0));
    u32x4_t* stage = win.stage + w0 * (kWaveSize * kStageVectors);
    if constexpr (kWide) {
      const int l = lane_now(), g2 = l / lpr, c2 = l - g2 * lpr;
      bag_at(g2, active, i, fi, b);
      const int out_col = fi - fi_lo < kMaxWinFeat ? win.desc[fi - fi_lo].out_col : a.cdescs[sc.first + fi].out_col;
      finish_bag<NE, kOwn>(acc, a, stage, active ? max(win.len[i], 0) : 0, (int64_t)b * a.out_stride + out_col, c2, lpr, l, active,
                     vec());
    } else {
      finish_bag<NE, kOwn>(acc, a, stage, len, (int64_t)b * a.out_stride + d.out_col, c, lpr, lane, active, vec());
    }
    TRA_STAMP(4);
    if (rounds <= kCuWaves) break;
    const int next = lane_now() == 0 ? atomicAdd(win.taken + (w0 & 3), 1) : 0;
    r = round_of(w0 & 3, kCuWaves / 4 + __builtin_amdgcn_readfirstlane(next));
  }
}

// ODD: the instance for launch classes of mostly odd lane groups (kOddInstance).
template <int DTYPE, int CB, typename IdxT, int WEIGHTED, int U, bool FROM_LENGTHS = false, bool ODD = false>
__global__ __launch_bounds__(kCuThreads) void tbe_pooled_cu_kernel(
    const void* p_offsets, const FeatureDesc* p_cdescs, int32_t p_B, int32_t p_xcd_blocks,
    int32_t p_xcd_count, int32_t p_n_sub, int32_t p_window0, int32_t p_count0, int32_t p_key0,
    const LookupArgs a) {
  extern __shared__ unsigned char tra_dyn_smem[];  // (room that a tuning override asks for, unused)
  TRA_WINDOW(IdxT, s_window);

  TRA_STAMP(0);
  // Block -> (sub-class, window).  Consecutive windows go to the same XCD
  // (blocks are dealt round-robin to the 8 XCDs), so each L2 sees few tables.
  // The leading kernel parameters repeat what the first fetches need (the
  // hardware preloads them into SGPRs): the block's bag bounds can be
  // requested without waiting for the launch arguments to arrive from memory.
  int blk = blockIdx.x;
  if (p_xcd_blocks > 0) blk = (blk % p_xcd_count) * p_xcd_blocks + blk / p_xcd_count;
  SubClass sc;
  if (p_n_sub == 1) {
    sc.first = 0;
    sc.count = p_count0;
    sc.lpr = a.sub[0].lpr;
    sc.tiles_per_feat = 0;
    sc.tile_start = 0;
    sc.window = p_window0;
    sc.key0 = p_key0;
  } else {
    int s = 0;
#pragma unroll
    for (int i = 1; i < kMaxSub; ++i)
      if (i < a.n_sub && blk >= a.sub[i].tile_start) s = i;
    sc = a.sub[s];
  }
  const int nb_all = sc.count * p_B;
  const int q0 = (blk - sc.tile_start) * sc.window;
  if (q0 >= nb_all) return;
  const int nb = min(sc.window, nb_all - q0);

  const int fi_lo = q0 / p_B;
  const auto starts = stage_window<IdxT, FROM_LENGTHS>(s_window, a, p_offsets, p_cdescs, p_B, sc, q0, nb, fi_lo);
  pool_window<DTYPE, CB, IdxT, WEIGHTED, U, ODD ? kBodiesOdd : kBodiesEven>(s_window, a, sc, nb, fi_lo, starts,
                                                                             [&] { return a.vec_store != 0; });
}

// ---- host side of one launch ----------------------------------------------
// Lane groups that fetch their ids in blocks only in some instances of the
// window kernel: 4 to 7 lanes, and more where they are no power of two.  Every
// body that an instance holds costs all of its widths registers, and where a
// lane holds many accumulators they are spilled.  So:
//   up to 8 accumulators a lane, and 16 in 4-byte chunks (whose lane groups are
//   odd by themselves): one instance with the bodies for all widths;
//   16: two instances, and a launch class takes the one for most of its slices;
//   32 and 64: no blocks for these widths.
// Measured on 12 tables, bags of 1 - 40 ids, us with the rows in the L2 / in HBM:
//   int8 dim 72 (9 lanes of 8 accumulators): ids one by one 13.1 / 16.8, in
//   blocks 10.4 / 16.6; weighted 17.2 / 19.7 and 10.2 / 16.5;
//   int8 dim 112 (7 lanes of 16): one by one 15.9 / 18.1, in blocks 13.9 / 17.3;
//   int8 dim 128, int64 ids (8 lanes of 16): 15.4 / 29.3 in an instance that
//   holds what the powers of two need, 16.4 / 33.0 in one with all bodies;
//   int2 dim 320 (5 lanes of 64): one by one 36 / 47, in blocks 84 / 104.
inline bool odd_lanes(int lpr) { return lpr >= 4 && lpr != 8 && !(lpr >= 16 && (lpr & (lpr - 1)) == 0); }
template <int DTYPE, int CB>
constexpr bool kOddInstance = DTYPE < kSplitHeader && CB > 4 && CB * 8 / Traits<DTYPE>::kBits == 2 * kNarrowLane;

struct LaunchClass {
  int dtype;
  int cb;
  bool odd = false;    // more slices of odd_lanes than others
  bool split = false;  // rows cut into several column slices, header loaded on its own (kSplitHeader)
  std::vector<int32_t> feats;  // plan order: sorted by lpr
  std::vector<int32_t> lprs;   // lanes per row of each feature
  int32_t* feats_dev = nullptr;
  // every slice's first output column is 16-byte aligned for fp16 / fp32 outputs
  bool cols_aligned_fp16 = true;
  bool cols_aligned_fp32 = true;
};

struct LaunchParams {
  int grid;
  int lds_bytes;  // window kernel: dynamic LDS beside its own 107 KB, which already leave a compute unit one block
  int unroll;     // rows per pipeline batch: 2, 4 or 8
  bool idx64;
  bool weighted;
  bool from_lengths;  // window kernel reads lengths and derives offsets itself
  bool odd;           // window kernel: the instance for odd lane groups, where there is one
};

template <int DTYPE>
int launch_lookup(const LookupArgs& a, int cb, const LaunchParams& p, hipStream_t stream);

// Consecutive columns of one feature, as the sixteen-lane kernel takes them.
struct GroupSlice {
  int64_t table_offset;
  int64_t rows;
  uint32_t rows32;      // min(rows, 2^31)
  int32_t row_bytes;    // stride
  int32_t cols;
  int32_t out_col;
  int32_t payload;      // byte offset of the slice's columns inside a row
  int32_t kind;         // group_kind(weight type, columns per lane, mode)
  int32_t key;          // key position
  uint8_t even;         // the first output column is
  uint8_t first_slice;  // holds column 0 of its feature
  uint8_t lanes_log2;   // lanes per bag: 16, 32 or 64
  uint8_t part;         // which of the lanes / 16 descriptors of the slice: a block takes that share of its window's bags
};
// How the sixteen-lane kernel addresses a slice's rows.
constexpr int kNear = 0;   // 32-bit offsets, header in front of the columns (or none)
constexpr int kFar = 1;    // a table beyond 4 GiB
constexpr int kSplit = 2;  // a row with a header, in several slices or by more than sixteen lanes
constexpr int group_kind(int dtype, int ne, int mode) { return (dtype * 4 + mode) * 32 + ne; }
// What a launch needs and no more: the launch arguments are written over the bus for every call, and a small call's
// time is its launch (with the window kernel's arguments, 3.0 KB, the entry point takes 4.2 us of the host's time, with
// these 3.5; two boxes, evened out by the time of torch.empty).
struct GroupArgs {
  const uint8_t* weights;
  const GroupSlice* slices;
  const void* indices;
  const void* offsets;
  const float* psw;
  const float* posw;
  void* out;
  int64_t out_stride;  // elements
  unsigned long long* err_count;
  int64_t num_indices;
  int32_t B;
  uint8_t mean;
  uint8_t out_fp16;
  uint8_t pairs;        // two fp16 results of an even column make an aligned dword
  uint8_t bad_to_row0;  // as in LookupArgs
};
// Position weights of the launch's slices, as in LookupArgs.
struct GroupPositions {
  int32_t off[kMaxPos];
  int32_t len[kMaxPos];
};
struct NoPositions {};
struct GroupLaunch {
  int grid;
  int per_group;  // bags per lane group (at most 16)
  int tiles;      // blocks per slice
  int key0;       // slice i sits at key key0 + i; -1: each slice says where
};

// Pooled lookup, all weight types in one launch (tbe_group_impl.h).
template <typename IdxT, int WEIGHTED>
void launch_group(const GroupArgs& a, const GroupPositions* p, const GroupLaunch& l, bool from_lengths,
                  hipStream_t stream);

// Several launch classes in one launch of windows (tbe_multi_impl.h).
constexpr int kMaxMultiSub = 16;
constexpr int kMultiVec = 1;  // in a kind: every lane's output slice is 16-byte aligned
constexpr int multi_kind(int dtype, int cb) { return dtype * 64 + cb * 2; }
struct MultiArgs {
  LookupArgs common;                 // (sub, n_sub and vec_store are not read)
  int32_t tile_start[kMaxMultiSub];  // first block of every entry of sub; INT32_MAX behind the last one
  int32_t kind[kMaxMultiSub];
  SubClass sub[kMaxMultiSub];
};
static_assert(sizeof(MultiArgs) + 48 <= 4096, "launch arguments");
template <typename IdxT, int WEIGHTED>
void launch_multi(const MultiArgs& a, int grid, int lds_bytes, bool from_lengths, hipStream_t stream);

// The sequence lookup of one class (tbe_sequence.hip).
int launch_sequence(const LookupArgs& a, int dtype, int cb, bool split, bool idx64, int grid, hipStream_t stream);

template <int DTYPE, int CB, typename IdxT>
void launch_typed(const LookupArgs& a, const LaunchParams& p, hipStream_t stream) {
  dim3 g(p.grid);
// What the window kernel's first fetches need, repeated as its leading parameters.
#define TRA_CU_LEADING_ARGS                                                                   \
  a.offsets, a.cdescs, a.B, a.xcd_blocks, a.xcd_count, a.n_sub, a.sub[0].window, a.sub[0].count, \
      a.sub[0].key0
#define TRA_POOLED(W, U)                                                                       \
  do {                                                                                         \
    constexpr bool O = kOddInstance<DTYPE, CB>;                                                \
    if (O && p.odd && p.from_lengths)                                                          \
      hipLaunchKernelGGL((tbe_pooled_cu_kernel<DTYPE, CB, IdxT, W, 4, true, O>), g,            \
                         dim3(kCuThreads), p.lds_bytes, stream, TRA_CU_LEADING_ARGS, a);       \
    else if (O && U == 4 && p.odd)                                                             \
      hipLaunchKernelGGL((tbe_pooled_cu_kernel<DTYPE, CB, IdxT, W, U, false, O && U == 4>), g, \
                         dim3(kCuThreads), p.lds_bytes, stream, TRA_CU_LEADING_ARGS, a);       \
    else if (p.from_lengths)                                                                   \
      hipLaunchKernelGGL((tbe_pooled_cu_kernel<DTYPE, CB, IdxT, W, 4, true>), g,               \
                         dim3(kCuThreads), p.lds_bytes, stream, TRA_CU_LEADING_ARGS, a);       \
    else                                                                                       \
      hipLaunchKernelGGL((tbe_pooled_cu_kernel<DTYPE, CB, IdxT, W, U>), g, dim3(kCuThreads),   \
                         p.lds_bytes, stream, TRA_CU_LEADING_ARGS, a);                         \
  } while (0)
  if constexpr (DTYPE >= kSplitHeader) {  // (one unroll depth for the rare split rows)
    if (a.posw != nullptr) TRA_POOLED(kByPosition, 4); else if (p.weighted) TRA_POOLED(kPerSample, 4); else TRA_POOLED(kUnweighted, 4);
  } else if (a.posw != nullptr) {
    TRA_POOLED(kByPosition, 4);  // (one unroll depth: the others are tuning variants)
  } else if (p.weighted) {
    if (p.unroll >= 8) TRA_POOLED(kPerSample, 8); else if (p.unroll >= 4) TRA_POOLED(kPerSample, 4); else TRA_POOLED(kPerSample, 2);
  } else {
    if (p.unroll >= 8) TRA_POOLED(kUnweighted, 8); else if (p.unroll >= 4) TRA_POOLED(kUnweighted, 4); else TRA_POOLED(kUnweighted, 2);
  }
#undef TRA_POOLED
#undef TRA_CU_LEADING_ARGS
}

template <int DTYPE, int CB>
int launch_lookup_cb(const LookupArgs& a, const LaunchParams& p, hipStream_t stream) {
  if (p.idx64)
    launch_typed<DTYPE, CB, int64_t>(a, p, stream);
  else
    launch_typed<DTYPE, CB, int32_t>(a, p, stream);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "tbe lookup launch");
  return TRA_OK;
}

#define TRA_DEFINE_LAUNCH(DTYPE)                                                          \
  template <>                                                                             \
  int launch_lookup<DTYPE>(const LookupArgs& a, int cb, const LaunchParams& p,            \
                           hipStream_t stream) {                                          \
    switch (cb) {                                                                         \
      case 16:                                                                            \
        if constexpr (DTYPE < kSplitHeader) return launch_lookup_cb<DTYPE, 16>(a, p, stream); \
        break;                                                                            \
      case 8: return launch_lookup_cb<DTYPE, 8>(a, p, stream);                            \
      case 4: return launch_lookup_cb<DTYPE, 4>(a, p, stream);                            \
    }                                                                                     \
    set_error("bad chunk size %d", cb);                                                   \
    return TRA_ERR_INVALID_ARGUMENT;                                                      \
  }

}  // namespace tra
