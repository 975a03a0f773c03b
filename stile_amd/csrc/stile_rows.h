// A wave's run over sparse entries, shared by the sparse-row and the streaming
// kernels of libstile_hip.so.
#pragma once

#include "stile_device.h"

namespace stile {

// ---------------------------------------------------------------------------
// One wave runs a stretch of the sparse part's entries (column, value) for
// 64 * VW output columns: every lane gathers VW elements of each entry's B row.
// What an entry needs besides its B row is the same for the whole wave, so the
// columns, values and row ends are scalar loads, an entry's address is one
// scalar base and the lane's constant offset, and a row's end is a scalar
// branch.  The gathers of the next kRowBatch entries are issued before the
// current ones are multiplied, across row ends, and the scalar loads run one
// batch further ahead; a short row then costs its entries, not a chain of
// latencies, and rows of any lengths keep the wave full.
//
// Bound: B-row gathers from L2 / MALL.  R-MAT scale 17, N = 128, FP32: the
// 2.55 M entries of this kernel take 115 us (11.3 TB/s of gathered rows); with
// one row per 16-lane group, four rows of unequal length per wave and each
// row's entries in sequence they took 444 us.  Scale 15, N = 250 (rows that are
// not 16-byte aligned): 932 -> 83 us for the whole product.
// ---------------------------------------------------------------------------
constexpr int kRowBatch = 8;

// VW elements of an entry's B row for this lane, as FP32.  kVec: consecutive
// columns (one aligned load); else columns 64 apart (any alignment; each load is
// still one contiguous run of the wave).  Lanes at or beyond N repeat the last
// columns.  kBuf (B below 4 GiB): buffer loads, whose row offset is one scalar
// product; an address in vector registers per entry would alias the registers
// of loads in flight and wait for them.  Otherwise a scalar 64-bit row address
// (the empty asm keeps it scalar).
template <typename TB, int VW, bool kVec, bool kBuf>
struct RowReader {
  const TB* B;
  int64_t ldb;
  __amdgpu_buffer_rsrc_t rs;
  uint32_t off[kVec ? 1 : VW];  // bytes from the row's start
  __device__ __forceinline__ RowReader(const TB* __restrict__ Bp, int64_t ld, uint32_t bytes, int n0, int N,
                                       int lane)
      : B(Bp), ldb(ld) {
    rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<TB*>(Bp), 0, bytes, 0x00020000);
    if constexpr (kVec) {
      off[0] = (uint32_t)min(n0 + VW * lane, N - VW) * sizeof(TB);  // N % VW == 0
    } else {
#pragma unroll
      for (int c = 0; c < VW; ++c) off[c] = (uint32_t)min(n0 + lane + 64 * c, N - 1) * sizeof(TB);
    }
  }
  template <int kBytes>
  __device__ __forceinline__ auto raw(const unsigned char* row, uint32_t soff, uint32_t o) const {
    if constexpr (kBuf) {
      if constexpr (kBytes == 2)
        return __builtin_amdgcn_raw_buffer_load_b16(rs, o, soff, 0);
      else if constexpr (kBytes == 4)
        return __builtin_amdgcn_raw_buffer_load_b32(rs, o, soff, 0);
      else if constexpr (kBytes == 8)
        return __builtin_amdgcn_raw_buffer_load_b64(rs, o, soff, 0);
      else
        return __builtin_amdgcn_raw_buffer_load_b128(rs, o, soff, 0);
    } else {
      typedef uint32_t u2 __attribute__((ext_vector_type(2)));
      typedef uint32_t u4 __attribute__((ext_vector_type(4)));
      typedef typename std::conditional<
          kBytes == 2, uint16_t,
          typename std::conditional<kBytes == 4, uint32_t,
                                    typename std::conditional<kBytes == 8, u2, u4>::type>::type>::type T;
      return *reinterpret_cast<const T*>(row + o);
    }
  }
  __device__ __forceinline__ void load(int k, float (&b)[VW]) const {
    const unsigned char* row = nullptr;
    uint32_t soff = 0;
    if constexpr (kBuf) {
      soff = (uint32_t)k * ((uint32_t)ldb * (uint32_t)sizeof(TB));
    } else {
      row = reinterpret_cast<const unsigned char*>(B + (int64_t)k * ldb);
      asm volatile("" : "+s"(row));
    }
    if constexpr (kVec && VW > 1) {
      typedef TB vec_t __attribute__((ext_vector_type(VW)));
      const vec_t v = __builtin_bit_cast(vec_t, raw<VW * (int)sizeof(TB)>(row, soff, off[0]));
#pragma unroll
      for (int c = 0; c < VW; ++c) b[c] = (float)v[c];
    } else {
#pragma unroll
      for (int c = 0; c < VW; ++c) b[c] = (float)__builtin_bit_cast(TB, raw<(int)sizeof(TB)>(row, soff, off[c]));
    }
  }
};

// The lane's columns of a row of C (lanes at or beyond N repeat the last).
template <int VW, bool kVec>
__device__ __forceinline__ void load_cols(const float* __restrict__ row, int n0, int N, float (&s)[VW]) {
  const int lane = threadIdx.x & 63;
  if constexpr (kVec && VW > 1) {
    typedef float vec_t __attribute__((ext_vector_type(VW)));
    const vec_t v = *reinterpret_cast<const vec_t*>(row + min(n0 + VW * lane, N - VW));
#pragma unroll
    for (int c = 0; c < VW; ++c) s[c] = v[c];
  } else {
#pragma unroll
    for (int c = 0; c < VW; ++c) s[c] = row[min(n0 + lane + 64 * c, N - 1)];
  }
}

template <int VW, bool kVec>
__device__ __forceinline__ void store_cols(float* __restrict__ row, int n0, int N, const float (&s)[VW]) {
  const int lane = threadIdx.x & 63;
  if constexpr (kVec && VW > 1) {
    typedef float vec_t __attribute__((ext_vector_type(VW)));
    const int col = n0 + VW * lane;
    if (col < N) {
      vec_t v;
#pragma unroll
      for (int c = 0; c < VW; ++c) v[c] = s[c];
      *reinterpret_cast<vec_t*>(row + col) = v;
    }
  } else {
#pragma unroll
    for (int c = 0; c < VW; ++c)
      if (n0 + lane + 64 * c < N) row[n0 + lane + 64 * c] = s[c];
  }
}

template <int kBatch>
struct RowEntries {
  int k[kBatch];
  float v[kBatch];
  __device__ __forceinline__ void load(const int32_t* __restrict__ cols, const float* __restrict__ vals, int q) {
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      k[i] = cols[q + i];
      v[i] = vals[q + i];
    }
  }
};

// Entries [q0, q1), q0 < q1 (both wave-uniform), added to acc; at_end(q) is
// called before the entry at each position q is added.
// Reads the ids of up to 2 kBatch entries past q1 (of the next rows, or of the
// kRowPad padding entries behind the arrays); B rows of up to kBatch of them are
// gathered, and none is added.
template <int VW, typename Acc, int kBatch = kRowBatch, typename Reader, typename F>
__device__ __forceinline__ void run_entries(const int32_t* __restrict__ cols, const float* __restrict__ vals,
                                            const Reader& rd, int q0, int q1, Acc (&acc)[VW], F&& at_end) {
  float b0[kBatch][VW], b1[kBatch][VW];
  RowEntries<kBatch> e0, e1;
  auto gather = [&](const RowEntries<kBatch>& e, float (&b)[kBatch][VW]) {
#pragma unroll
    for (int i = 0; i < kBatch; ++i) rd.load(e.k[i], b[i]);
  };
  auto add = [&](const float (&v)[kBatch], const float (&b)[kBatch][VW], int q, int n) {
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      if (i < n) {
        at_end(q + i);
#pragma unroll
        for (int c = 0; c < VW; ++c) acc[c] += (Acc)v[i] * (Acc)b[i][c];
      }
    }
  };
  // Two register sets, no copies.  Every path from a batch's gathers to its use
  // issues the same loads in between: were the next gathers conditional, the
  // wait for the current ones would include them.
  e0.load(cols, vals, q0);
  gather(e0, b0);
  e1.load(cols, vals, q0 + kBatch);
  for (int q = q0;; q += 2 * kBatch) {
    float v[kBatch];
    if (q + kBatch >= q1) {
      add(e0.v, b0, q, q1 - q);
      break;
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) v[i] = e0.v[i];
    gather(e1, b1);
    e0.load(cols, vals, min(q + 2 * kBatch, q1));
    add(v, b0, q, kBatch);
    if (q + 2 * kBatch >= q1) {
      add(e1.v, b1, q + kBatch, q1 - q - kBatch);
      break;
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) v[i] = e1.v[i];
    gather(e0, b0);
    e1.load(cols, vals, min(q + 3 * kBatch, q1));
    add(v, b1, q + kBatch, kBatch);
  }
}

// Bytes B spans (K rows, N columns), or 0 when a buffer descriptor with 32-bit
// offsets cannot address them.
template <typename TB>
inline uint32_t b_bytes(int64_t K, int64_t ldb, int N) {
  const int64_t n = ((K - 1) * ldb + N) * (int64_t)sizeof(TB);
  return K > 0 && ldb < ((int64_t)1 << 30) && n < ((int64_t)1 << 32) ? (uint32_t)n : 0u;
}

}  // namespace stile
