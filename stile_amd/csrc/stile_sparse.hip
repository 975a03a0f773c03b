// Sparse rows of the hybrid SpMM (sparse-only windows and the pieces of long
// rows) for MI355X (gfx950).
#include "stile_device.h"

#include <algorithm>

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
// not 16-byte aligned): 932 -> 88 us for the whole product.
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
  __device__ __forceinline__ RowReader(const TB* __restrict__ Bp, int64_t ld, uint32_t bytes, int n0, int N)
      : B(Bp), ldb(ld) {
    const int lane = threadIdx.x & 63;
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

struct RowEntries {
  int k[kRowBatch];
  float v[kRowBatch];
  __device__ __forceinline__ void load(const int32_t* __restrict__ cols, const float* __restrict__ vals, int q) {
#pragma unroll
    for (int i = 0; i < kRowBatch; ++i) {
      k[i] = cols[q + i];
      v[i] = vals[q + i];
    }
  }
};

// Entries [q0, q1), q0 < q1 (both wave-uniform), added to acc; at_end(q) is
// called before the entry at each position q is added.
// Reads the ids of up to 2 kRowBatch entries past q1 (of the next rows, or of
// the kRowPad padding entries behind the arrays); B rows of up to kRowBatch of
// them are gathered, and none is added.
template <int VW, typename Acc, typename Reader, typename F>
__device__ __forceinline__ void run_entries(const int32_t* __restrict__ cols, const float* __restrict__ vals,
                                            const Reader& rd, int q0, int q1, Acc (&acc)[VW], F&& at_end) {
  float b0[kRowBatch][VW], b1[kRowBatch][VW];
  RowEntries e0, e1;
  auto gather = [&](const RowEntries& e, float (&b)[kRowBatch][VW]) {
#pragma unroll
    for (int i = 0; i < kRowBatch; ++i) rd.load(e.k[i], b[i]);
  };
  auto add = [&](const float (&v)[kRowBatch], const float (&b)[kRowBatch][VW], int q, int n) {
#pragma unroll
    for (int i = 0; i < kRowBatch; ++i) {
      if (i >= n) break;
      at_end(q + i);
#pragma unroll
      for (int c = 0; c < VW; ++c) acc[c] += (Acc)v[i] * (Acc)b[i][c];
    }
  };
  // Two register sets, no copies.  Every path from a batch's gathers to its use
  // issues the same loads in between: were the next gathers conditional, the
  // wait for the current ones would include them.
  e0.load(cols, vals, q0);
  gather(e0, b0);
  e1.load(cols, vals, q0 + kRowBatch);
  for (int q = q0;; q += 2 * kRowBatch) {
    float v[kRowBatch];
    if (q + kRowBatch >= q1) {
      add(e0.v, b0, q, q1 - q);
      break;
    }
#pragma unroll
    for (int i = 0; i < kRowBatch; ++i) v[i] = e0.v[i];
    gather(e1, b1);
    e0.load(cols, vals, min(q + 2 * kRowBatch, q1));
    add(v, b0, q, kRowBatch);
    if (q + 2 * kRowBatch >= q1) {
      add(e1.v, b1, q + kRowBatch, q1 - q - kRowBatch);
      break;
    }
#pragma unroll
    for (int i = 0; i < kRowBatch; ++i) v[i] = e1.v[i];
    gather(e0, b0);
    e1.load(cols, vals, min(q + 3 * kRowBatch, q1));
    add(v, b1, q + kRowBatch, kRowBatch);
  }
}

// One wave = (task, 64 * VW columns), column chunk by column chunk.  Task t =
// slots [x, y & 0x7fffffff) of the sparse-only windows: rows of at most
// kSplitNnz entries together, or the first kSplitNnz entries of one longer row
// (the rest are pieces).  Bit 31 of y: a row of more than kHubNnz entries,
// summed in FP64.
template <typename TB, int VW, bool kVec, bool kBuf>
__global__ __launch_bounds__(256, 4) void hyb_spmm_rows_kernel(
    const int2* __restrict__ tasks, int ntasks, const int32_t* __restrict__ res_ptr,
    const int32_t* __restrict__ cols, const float* __restrict__ vals, const int32_t* __restrict__ win_rows,
    const TB* __restrict__ B, int64_t ldb, uint32_t bbytes, int N, float* __restrict__ C, int64_t ldc, int nC) {
  const int wave = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cch = wave / ntasks;
  if (cch >= nC) return;
  const int2 t = tasks[wave - cch * ntasks];
  const int s0 = t.x, s1 = t.y & 0x7fffffff;
  const int n0 = cch * 64 * VW;
  const int q0 = res_ptr[s0];
  const int q1 = min(res_ptr[s1], q0 + (s1 == s0 + 1 ? kSplitNnz : INT32_MAX - q0));
  const RowReader<TB, VW, kVec, kBuf> rd(B, ldb, bbytes, n0, N);
  auto run = [&](auto zero) {
    typedef decltype(zero) Acc;
    Acc acc[VW];
#pragma unroll
    for (int c = 0; c < VW; ++c) acc[c] = zero;
    int slot = s0;
    // the row and the entry end of the current slot and the next, loaded one
    // slot ahead
    int row = win_rows[s0], end = min(res_ptr[s0 + 1], q1);
    int row1 = win_rows[min(s0 + 1, s1 - 1)], end1 = min(res_ptr[min(s0 + 2, s1)], q1);
    auto store = [&]() {
      if (row < 0) return;
      float o[VW];
#pragma unroll
      for (int c = 0; c < VW; ++c) o[c] = (float)acc[c];
      store_cols<VW, kVec>(C + (int64_t)row * ldc, n0, N, o);
    };
    auto next = [&]() {
#pragma unroll
      for (int c = 0; c < VW; ++c) acc[c] = zero;
      row = row1;
      end = end1;
      row1 = win_rows[min(slot + 1, s1 - 1)];
      end1 = min(res_ptr[min(slot + 2, s1)], q1);
    };
    if (q0 < q1)
      run_entries<VW, Acc>(cols, vals, rd, q0, q1, acc, [&](int q) {
        while (q == end) {
          store();
          ++slot;
          next();
        }
      });
    // the last row with entries and the empty ones behind it
    for (;;) {
      store();
      if (++slot == s1) break;
      next();
    }
  };
  if (t.y < 0)
    run(0.0);
  else
    run(0.f);
}

// Pieces of long rows, execution slots [pc0, pc1) (piece piece_exec[slot],
// ordered by first column so that pieces of different rows gathering the same
// B rows run together), column chunk by column chunk: summed in FP64 and added
// to C with atomicAdd (C already holds the row's first kSplitNnz entries), or,
// with ws (deterministic mode), stored to ws[piece][N] for the reduce kernel.
// One workgroup per piece and 64 * VW columns, a quarter of the entries per
// wave (a graph with few long rows has few pieces: 143 of them as one wave each
// took 36 us on N = 256, as four 15 us), the waves' sums added in wave order.
// FP64 sums: one conversion and one v_fma_f64 (as fast as v_fma_f32 here) per
// product against nine operations of a compensated FP32 sum, which bounded
// this kernel (1.31 M entries, N = 128: 58 us).
template <typename TB, int VW, bool kVec, bool kBuf>
__global__ __launch_bounds__(256, 4) void hyb_spmm_pieces_kernel(
    const int32_t* __restrict__ piece_exec, const int32_t* __restrict__ piece_row,
    const int32_t* __restrict__ piece_beg, const int32_t* __restrict__ piece_end, int pc0, int npc,
    const int32_t* __restrict__ cols, const float* __restrict__ vals, const TB* __restrict__ B, int64_t ldb,
    uint32_t bbytes, int N, float* __restrict__ C, int64_t ldc, float* __restrict__ ws) {
  __shared__ double part[3][VW][64];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int cch = (int)blockIdx.x / npc;
  const int pc = piece_exec[pc0 + ((int)blockIdx.x - cch * npc)];
  const int n0 = cch * 64 * VW;
  const int beg = piece_beg[pc], end = piece_end[pc];
  const int share = (end - beg + 3) >> 2;
  const int q0 = min(beg + wv * share, end), q1 = min(q0 + share, end);
  double acc[VW];
#pragma unroll
  for (int c = 0; c < VW; ++c) acc[c] = 0.0;
  if (q0 < q1) {
    const RowReader<TB, VW, kVec, kBuf> rd(B, ldb, bbytes, n0, N);
    run_entries<VW, double>(cols, vals, rd, q0, q1, acc, [](int) {});
  }
  if (wv > 0) {
#pragma unroll
    for (int c = 0; c < VW; ++c) part[wv - 1][c][lane] = acc[c];
  }
  __syncthreads();
  if (wv > 0) return;
  float s[VW];
#pragma unroll
  for (int c = 0; c < VW; ++c) s[c] = (float)(acc[c] + part[0][c][lane] + part[1][c][lane] + part[2][c][lane]);
  if (ws) {
    store_cols<VW, kVec>(ws + (int64_t)pc * N, n0, N, s);
    return;
  }
  float* cr = C + (int64_t)piece_row[pc] * ldc;
#pragma unroll
  for (int c = 0; c < VW; ++c) {
    const int col = kVec ? n0 + VW * lane + c : n0 + lane + 64 * c;
    if (col < N) atomicAdd(cr + col, s[c]);
  }
}

// Deterministic mode: C[row] += the row's pieces, for split rows [sr0, sr1).
// One workgroup per (split row, 64 columns): 16-lane group i sums pieces p0 + i,
// p0 + i + 16, ..., then group 0 adds the groups' sums in order to C.  (One
// group per row, its pieces one after the other: 21 us for R-MAT scale 17,
// whose hub row has 61 pieces, each read missing the L2.)
__global__ __launch_bounds__(256) void hyb_spmm_piece_reduce_kernel(SpmmPlanDev p, int N, float* __restrict__ C,
                                                                    int64_t ldc, int nC, bool vec, int sr0,
                                                                    const float* __restrict__ ws) {
  __shared__ float4 part[16][16];
  const int r = sr0 + (int)(blockIdx.x / nC);
  const int g = threadIdx.x >> 4, j = threadIdx.x & 15;
  const int col = (int)(blockIdx.x % nC) * 64 + 4 * j;
  const int p0 = p.srow_p0[r], p1 = p.srow_p1[r];
  with_vec(vec, [&](auto V) {
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int q = p0 + g; q < p1; q += 16) {
      const float4 v = load_b4(ws, N, q, col, N, V);
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    part[g][j] = s;
    __syncthreads();
    if (g > 0) return;
    const int row = p.srow_row[r];
    float4 c = load_b4(C, ldc, row, col, N, V);
    const int n = min(p1 - p0, 16);
    for (int i = 1; i < n; ++i) {
      const float4 v = part[i][j];
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    store_c4(C, ldc, row, col, N, V, make_float4(c.x + s.x, c.y + s.y, c.z + s.z, c.w + s.w));
  });
}

namespace {

// Columns per lane: the widest of 4, 2 and 1 that wastes no more lanes than
// the others (64 * VW columns per wave) and leaves at least kFewWaves waves
// for `waves` of them per column chunk (two per SIMD: below that a wave's
// latency is what the launch takes, and narrower waves are more of them).
constexpr int64_t kFewWaves = 2048;
int row_width(int N, int64_t waves) {
  auto chunks = [&](int vw) { return (N + 64 * vw - 1) / (64 * vw); };
  int best = 1;
  for (int vw = 2; vw <= 4; vw *= 2)
    if (chunks(vw) * vw <= chunks(best) * best && waves * chunks(vw) >= kFewWaves) best = vw;
  return best;
}

// f(VW, kVec, kBuf) with all three as compile-time constants.
template <typename F>
void with_width(int vw, bool vec, bool buf, F&& f) {
  auto g = [&](auto w) {
    auto h = [&](auto v) {
      if (buf)
        f(w, v, std::true_type{});
      else
        f(w, v, std::false_type{});
    };
    if (vec)
      h(std::true_type{});
    else
      h(std::false_type{});
  };
  if (vw == 4)
    g(std::integral_constant<int, 4>{});
  else if (vw == 2)
    g(std::integral_constant<int, 2>{});
  else
    g(std::integral_constant<int, 1>{});
}

// Bytes B spans, or 0 when a buffer descriptor cannot address them.
template <typename TB>
uint32_t b_bytes(const SpmmPlanDev& p, int64_t ldb, int N) {
  const int64_t n = ((int64_t)(p.K - 1) * ldb + N) * (int64_t)sizeof(TB);
  return p.K > 0 && ldb < ((int64_t)1 << 30) && n < ((int64_t)1 << 32) ? (uint32_t)n : 0u;
}

}  // namespace

template <typename TB>
hipError_t launch_sparse_rows(const SpmmPlanDev& p, const TB* B, int64_t ldb, int N, float* C, int64_t ldc, bool vec,
                         hipStream_t s) {
  const int vw = row_width(N, p.n_row_tasks);
  const int nC = (N + 64 * vw - 1) / (64 * vw);
  const int64_t blocks = ((int64_t)p.n_row_tasks * nC + 3) / 4;
  if (blocks > INT32_MAX / 4) return hipErrorInvalidValue;
  const uint32_t bytes = b_bytes<TB>(p, ldb, N);
  with_width(vw, vec, bytes > 0, [&](auto w, auto v, auto u) {
    hipLaunchKernelGGL((hyb_spmm_rows_kernel<TB, decltype(w)::value, decltype(v)::value, decltype(u)::value>),
                       dim3((unsigned)blocks), dim3(256), 0, s, p.row_tasks, p.n_row_tasks, p.res_ptr, p.res_cols,
                       p.res_vals, p.win_rows, B, ldb, bytes, N, C, ldc, nC);
  });
  return hipGetLastError();
}

template <typename TB>
hipError_t launch_sparse_pieces(const SpmmPlanDev& p, const TB* B, int64_t ldb, int N, float* C, int64_t ldc, bool vec,
                           int pc0, int pc1, float* ws, hipStream_t s) {
  const int vw = row_width(N, (int64_t)(pc1 - pc0) * 4);
  const int nC = (N + 64 * vw - 1) / (64 * vw);
  const int64_t blocks = (int64_t)(pc1 - pc0) * nC;
  if (blocks > INT32_MAX) return hipErrorInvalidValue;
  const uint32_t bytes = b_bytes<TB>(p, ldb, N);
  with_width(vw, vec, bytes > 0, [&](auto w, auto v, auto u) {
    hipLaunchKernelGGL((hyb_spmm_pieces_kernel<TB, decltype(w)::value, decltype(v)::value, decltype(u)::value>),
                       dim3((unsigned)blocks), dim3(256), 0, s, p.piece_exec, p.piece_row, p.piece_beg, p.piece_end,
                       pc0, pc1 - pc0, p.res_cols, p.res_vals, B, ldb, bytes, N, C, ldc, ws);
  });
  return hipGetLastError();
}

hipError_t launch_piece_reduce(const SpmmPlanDev& p, int N, float* C, int64_t ldc, bool vec, int sr0, const float* ws,
                               hipStream_t s) {
  const int nC = (N + 63) / 64;
  const int64_t blocks = (int64_t)(p.nsrows - sr0) * nC;
  if (blocks <= 0) return hipSuccess;
  if (blocks > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL(hyb_spmm_piece_reduce_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p, N, C, ldc, nC, vec, sr0,
                     ws);
  return hipGetLastError();
}

template hipError_t launch_sparse_rows<float>(const SpmmPlanDev&, const float*, int64_t, int, float*, int64_t, bool,
                                        hipStream_t);
template hipError_t launch_sparse_pieces<float>(const SpmmPlanDev&, const float*, int64_t, int, float*, int64_t, bool, int,
                                          int, float*, hipStream_t);
template hipError_t launch_sparse_rows<__bf16>(const SpmmPlanDev&, const __bf16*, int64_t, int, float*, int64_t, bool,
                                        hipStream_t);
template hipError_t launch_sparse_pieces<__bf16>(const SpmmPlanDev&, const __bf16*, int64_t, int, float*, int64_t, bool, int,
                                          int, float*, hipStream_t);
template hipError_t launch_sparse_rows<_Float16>(const SpmmPlanDev&, const _Float16*, int64_t, int, float*, int64_t, bool,
                                        hipStream_t);
template hipError_t launch_sparse_pieces<_Float16>(const SpmmPlanDev&, const _Float16*, int64_t, int, float*, int64_t, bool, int,
                                          int, float*, hipStream_t);

}  // namespace stile
