// Streaming kernel of the hybrid SpMM: dense windows whose B does not fit the
// B-stationary kernel (FP32 and FP16 blocks, K > kLdsMaxK), for MI355X (gfx950).
#include "stile_rows.h"

#include <algorithm>

namespace stile {

// ---------------------------------------------------------------------------
// hyb_spmm_stream_kernel: one workgroup, or half of one, = (window or part of a
// huge window, 16 * NT columns).  Each wave takes a contiguous share of the window's
// chunks and, in launches that fold the sparse parts, some of its 16 slots' sparse
// entries; the partial sums meet in LDS, are added in wave order and leave as whole
// rows of C.
//
// Lane l = 16g + j of a wave holds, for MFMA tile t, column col(j, t) of rows 4g
// .. 4g + 3 of the window: kVec (B rows aligned, N % 4 == 0) n0 + NT j + t, so
// that a row is one load of NT columns; otherwise n0 + 16t + j, NT loads of one
// column, each a contiguous run of 16 lanes at any alignment.
//
// Dense chunk (32 k-slots): k-slot 4e + g of lane l is column tc_cols[c][g][e]
// of A, A operand element e of lane l (the pairing of k-slots with operand
// elements is the same for A and B, which is all the MFMA needs).
//   BF16: one v_mfma_f32_16x16x32_bf16 per tile;
//   FP16: one v_mfma_f32_16x16x32_f16 per tile, times the chunk's scale;
//   FP32: eight v_mfma_f32_16x16x4_f32 per tile (MFMA e reduces k-slots
//         4e + 0..3; lane group g supplies k-slot 4e + g).
//
// What bounds it: the latency of ids -> B rows -> MFMA per group of chunks in
// flight, and the longest share.  With one wave per window of up to 8 chunks
// (eight per longer window) and a second launch for the sparse parts, a 1000 x
// 747 FP16 layer (63 windows, N = 321) ran on 48 workgroups in 17.7 us, the
// windows of an R-MAT scale 15 graph (N = 256, FP32) waited 78 us for 23 chunks
// in sequence, and a 1024 x 4096 BF16 layer (N = 512) took 24 us.  With four to
// eight waves per window, up to four chunks in flight, 32 columns a workgroup
// for windows of more than 16 chunks and the sparse parts in the same launch:
// 8.7, 38 and 14.9 us.  Launches that fill the GPU without all that have a kernel of
// their own (hyb_spmm_stream_full_kernel, full_launch): the 3072 x 768 FP16 layer at
// N = 4096 takes 33 us on it, 64 on several waves a window and 42 on the one-wave
// kernel before either; in FP32 65, 81 and 78.
// ---------------------------------------------------------------------------
// B elements of one chunk's eight rows for this lane, as loaded.
template <typename TB, int NT, bool kVec>
struct ChunkB {
  static constexpr int kWords = kVec ? NT * (int)sizeof(TB) / 4 : NT;  // 32-bit registers per row
  typedef uint32_t Words __attribute__((ext_vector_type(kWords)));
  Words w[8];
  __device__ __forceinline__ float f32(int e, int t) const {
    if constexpr (std::is_same<TB, float>::value) {
      return __uint_as_float(w[e][t]);
    } else {
      const uint32_t h = kVec ? (t & 1 ? w[e][t >> 1] >> 16 : w[e][t >> 1] & 0xffffu) : w[e][t];
      return (float)__builtin_bit_cast(TB, (uint16_t)h);
    }
  }
  // elements (e, t) and (e + 1, t) of 16-bit B as one register
  __device__ __forceinline__ uint32_t pair(int e, int t) const {
    if constexpr (kVec)
      return half_sel(w[e][t >> 1], w[e + 1][t >> 1], t & 1);
    else
      return half_sel(w[e][t], w[e + 1][t], 0);
  }
};

template <typename TB, int NT, bool kVec, bool kBuf>
struct ChunkReader {
  const TB* B;
  int64_t ldb;
  __amdgpu_buffer_rsrc_t rs;
  uint32_t row_bytes, off;  // kBuf: bytes per row, the lane's column offset
  int col[kVec ? 1 : NT];   // !kBuf: the lane's columns, clamped into the row
  __device__ __forceinline__ ChunkReader(const TB* __restrict__ Bp, int64_t ld, uint32_t bytes, int n0, int N)
      : B(Bp), ldb(ld) {
    const int j = threadIdx.x & 15;
    rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<TB*>(Bp), 0, bytes, 0x00020000);
    row_bytes = (uint32_t)ld * (uint32_t)sizeof(TB);
    // Columns at or beyond N read what follows (the next row, or 0 past B's
    // end): they only reach MFMA columns that are never stored.
    off = (uint32_t)(n0 + (kVec ? NT * j : j)) * (uint32_t)sizeof(TB);
    if constexpr (!kBuf) {
#pragma unroll
      for (int t = 0; t < (kVec ? 1 : NT); ++t) col[t] = min(n0 + 16 * t + j, N - 1);
    }
  }
  __device__ __forceinline__ void load(const int4& ka, const int4& kb, ChunkB<TB, NT, kVec>& b) const {
    const int k[8] = {ka.x, ka.y, ka.z, ka.w, kb.x, kb.y, kb.z, kb.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (kBuf) {
        const uint32_t o = __umul24((unsigned)k[e], row_bytes) + off;  // both below 2^24 (launch_stream)
        if constexpr (kVec) {
          constexpr int kB = NT * (int)sizeof(TB);
          if constexpr (kB == 16) {
            b.w[e] = __builtin_bit_cast(typename ChunkB<TB, NT, kVec>::Words,
                                        __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0));
          } else if constexpr (kB == 8) {
            b.w[e] = __builtin_bit_cast(typename ChunkB<TB, NT, kVec>::Words,
                                        __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, 0));
          } else {
            b.w[e][0] = __builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0);
          }
        } else {
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            if constexpr (sizeof(TB) == 4)
              b.w[e][t] = __builtin_amdgcn_raw_buffer_load_b32(rs, o + 64 * t, 0, 0);
            else
              b.w[e][t] = __builtin_amdgcn_raw_buffer_load_b16(rs, o + 32 * t, 0, 0);
          }
        }
      } else {
        static_assert(kBuf || !kVec, "the 64-bit path reads single columns");
        const TB* row = B + (int64_t)k[e] * ldb;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          if constexpr (sizeof(TB) == 4)
            b.w[e][t] = __float_as_uint(row[col[t]]);
          else
            b.w[e][t] = __builtin_bit_cast(uint16_t, row[col[t]]);
        }
      }
    }
  }
};

// The A operand of one chunk.
template <int MODE>
struct ChunkA {
  typename std::conditional<MODE == 0, float4, bf16x8>::type a0;
  float4 a1;
  float scale;
  __device__ __forceinline__ void load(const void* __restrict__ vals, const float* __restrict__ scales, int64_t c) {
    const int lane = threadIdx.x & 63;
    if constexpr (MODE == 0) {
      const float* ap = static_cast<const float*>(vals) + (c * 64 + lane) * 8;
      a0 = ld4(ap);
      a1 = ld4(ap + 4);
    } else {
      a0 = static_cast<const bf16x8*>(vals)[c * 64 + lane];
      if constexpr (MODE == 2) scale = scales[c];
    }
  }
};

template <int MODE, typename TB, int NT, bool kVec>
__device__ __forceinline__ void mfma_chunk(const ChunkA<MODE>& a, const ChunkB<TB, NT, kVec>& b, f32x4 (&acc)[NT]) {
  if constexpr (MODE == 0) {
    const float av[8] = {a.a0.x, a.a0.y, a.a0.z, a.a0.w, a.a1.x, a.a1.y, a.a1.z, a.a1.w};
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[e], b.f32(e, t), acc[t], 0, 0, 0);
  } else {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      u32x4 bt;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        if constexpr (MODE == 1) {
          if constexpr (std::is_same<TB, __bf16>::value)
            bt[e / 2] = b.pair(e, t);
          else
            bt[e / 2] = bf16_pair(b.f32(e, t), b.f32(e + 1, t));
        } else {
          if constexpr (std::is_same<TB, _Float16>::value) {
            bt[e / 2] = b.pair(e, t);
          } else {
            const f16x2 h = {(_Float16)b.f32(e, t), (_Float16)b.f32(e + 1, t)};
            bt[e / 2] = __builtin_bit_cast(uint32_t, h);
          }
        }
      }
      if constexpr (MODE == 1) {
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.a0, __builtin_bit_cast(bf16x8, bt), acc[t], 0, 0, 0);
      } else {
        const f32x4 tmp = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a.a0),
                                                                 __builtin_bit_cast(f16x8, bt),
                                                                 f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        acc[t] += a.scale * tmp;
      }
    }
  }
}

// What the kernel reads of a plan (a launch passes no more of it).
struct StreamArrays {
  const int32_t *tc_ptr, *tc_cols, *win_rows;
  const void* tc_vals;
  const float* tc_scale;
  const int32_t *part_win, *part_c0, *part_c1, *hw_p0;
  int32_t W_tc, W_long, W_big, W_huge, n_parts, fold_mix;
};

// Registers for the chunks in flight (four waves per SIMD).  16-bit rows with
// 16-bit blocks: 56 (two chunks of 64 columns, four of 32) measured 15.7 us on a
// 1024 x 4096 layer at N = 512, 80 registers 18.6 us, six waves per SIMD with
// 48 registers 24.7 us (spills).
template <int MODE, typename TB>
constexpr int stream_registers() { return sizeof(TB) == 2 && MODE != 0 ? 56 : 80; }

template <int MODE, typename TB, int NT, bool kVec, bool kBuf>
__device__ __forceinline__ void stream_window(const StreamArrays& A, const int32_t* __restrict__ res_ptr,
                                              const int32_t* __restrict__ res_cols,
                                              const float* __restrict__ res_vals, const TB* __restrict__ B,
                                              int64_t ldb, uint32_t bbytes, int N, float* __restrict__ C, int64_t ldc,
                                              int w, int n0, int c0, int c1, bool sparse, float* __restrict__ part,
                                              bool add, float* __restrict__ lds, int wv, int nw) {
  constexpr int CW = 16 * NT;
  // chunks in flight, by the registers their B rows and A operands take
  constexpr int D = std::min(4, stream_registers<MODE, TB>() / (8 * ChunkB<TB, NT, kVec>::kWords + (MODE == 0 ? 8 : 4)));
  static_assert(D >= 1);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, j = lane & 15;
  const int share = (c1 - c0 + nw - 1) / nw;
  const int nd = (c1 - c0 + share - 1) / share;  // waves with a share
  const int a = min(c0 + wv * share, c1), b = min(a + share, c1);
  // Sparse entries of the window's slots: on the waves without chunks when they
  // are at least half of them, else on all; consecutive slots [s0, s1) per wave.
  int s0 = 0, s1 = 0, q0 = 0, q1 = 0, end0 = 0;
  if (sparse) {
    const int first = nd * 2 <= nw ? nd : 0, per = (16 + nw - first - 1) / (nw - first);
    s0 = min(max(wv - first, 0) * per, 16);
    s1 = wv < first ? s0 : min(s0 + per, 16);
    q0 = res_ptr[w * 16 + s0];
    q1 = res_ptr[w * 16 + s1];
    end0 = res_ptr[min(w * 16 + s0 + 1, w * 16 + 16)];
  }
  if (a < b) {
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const ChunkReader<TB, NT, kVec, kBuf> rd(B, ldb, bbytes, n0, N);
    for (int c = a; c < b; c += D) {
      // the first chunk always, the others when the share reaches them
      int4 ka[D], kb[D];
      ChunkA<MODE> ca[D];
      ChunkB<TB, NT, kVec> cb[D];
#pragma unroll
      for (int u = 0; u < D; ++u)
        if (u == 0 || c + u < b) {
          const int4* cp = reinterpret_cast<const int4*>(A.tc_cols + (int64_t)(c + u) * 32 + g * 8);
          ka[u] = cp[0];
          kb[u] = cp[1];
          ca[u].load(A.tc_vals, A.tc_scale, c + u);
        }
#pragma unroll
      for (int u = 0; u < D; ++u)
        if (u == 0 || c + u < b) rd.load(ka[u], kb[u], cb[u]);
#pragma unroll
      for (int u = 0; u < D; ++u)
        if (u == 0 || c + u < b) mfma_chunk<MODE>(ca[u], cb[u], acc);
    }
    float* dp = lds + wv * 16 * CW;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float* at = dp + (4 * g + i) * CW;
      if constexpr (kVec && NT == 4)
        st4(at + 4 * j, make_float4(acc[0][i], acc[1][i], acc[2][i], acc[3][i]));
      else if constexpr (kVec)
        *reinterpret_cast<float2*>(at + 2 * j) = make_float2(acc[0][i], acc[1][i]);
      else
#pragma unroll
        for (int t = 0; t < NT; ++t) at[16 * t + j] = acc[t][i];
    }
  }
  float* sp = lds + nw * 16 * CW;
  if (s0 < s1) {
    // the wave's slots as one run of entries, whose gathers are pipelined across
    // the slots' ends
    float sum[1] = {0.f};
    int slot = s0, end = end0;
    auto store = [&]() {
      if (lane < CW) sp[slot * CW + lane] = sum[0];
      sum[0] = 0.f;
    };
    auto next = [&]() {
      ++slot;
      end = res_ptr[min(w * 16 + slot + 1, w * 16 + s1)];
    };
    if (q0 < q1) {
      const RowReader<TB, 1, false, kBuf> rr(B, ldb, bbytes, n0, N, lane & (CW - 1));
      run_entries<1, float, 16>(res_cols, res_vals, rr, q0, q1, sum, [&](int q) {
        while (q == end) {
          store();
          next();
        }
      });
    }
    for (;;) {
      store();
      if (slot + 1 == s1) break;
      next();
    }
  }
  __syncthreads();
  constexpr int Q = kVec ? 4 : 1;  // columns per thread and step
  for (int i = wv * 64 + lane; i < 16 * CW / Q; i += nw * 64) {
    const int r = i / (CW / Q), x = (i - r * (CW / Q)) * Q;
    const int row = A.win_rows[w * 16 + r];
    float o[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) o[q] = lds[r * CW + x + q];
    for (int v = 1; v < nd; ++v)
#pragma unroll
      for (int q = 0; q < Q; ++q) o[q] += lds[(v * 16 + r) * CW + x + q];
    if (sparse)
#pragma unroll
      for (int q = 0; q < Q; ++q) o[q] += sp[r * CW + x + q];
    if (n0 + x >= N) continue;
    if (part) {
      // partial rows of a huge window's part, summed by the reduce kernel
      float* at = part + (int64_t)r * N + n0 + x;
#pragma unroll
      for (int q = 0; q < Q; ++q) at[q] = o[q];
    } else if (row >= 0) {
      float* at = C + (int64_t)row * ldc + n0 + x;
      if (add) {
#pragma unroll
        for (int q = 0; q < Q; ++q) atomicAdd(at + q, o[q]);
      } else if constexpr (kVec) {
        st4(at, make_float4(o[0], o[1], o[2], o[3]));
      } else {
        at[0] = o[0];
      }
    }
  }
}

// Blocks [0, (n_parts + W_big - W_huge) * nC2) each run one (part of a huge
// window or other big window, 32 columns) on all its waves; the next ones run
// the (W_tc - W_big) * nC (window, 64 columns) on nw waves each.  Parts
// add into C with atomicAdd (C rows zeroed before), or, with ws (deterministic
// mode), store to ws[part][16][N]; the first part of a window brings its sparse
// part.
template <int MODE, typename TB, bool kVec, bool kBuf>
__global__ __launch_bounds__(kStreamWaves * 64, 4) void hyb_spmm_stream_kernel(
    StreamArrays p, const int32_t* __restrict__ res_ptr, const int32_t* __restrict__ res_cols,
    const float* __restrict__ res_vals, const TB* __restrict__ B, int64_t ldb, uint32_t bbytes, int N,
    float* __restrict__ C, int64_t ldc, int nC, int nC2, int nw, float* __restrict__ ws) {
  extern __shared__ float4 stream_lds[];
  float* lds = reinterpret_cast<float*>(stream_lds);
  const int block = (int)blockIdx.x;
  const int big = (p.n_parts + p.W_big - p.W_huge) * nC2;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool fold = p.fold_mix != 0;
  auto has_sparse = [&](int w) { return fold && res_ptr[w * 16] < res_ptr[w * 16 + 16]; };
  if (block < big) {
    const int i = block / nC2, n0 = (block - i * nC2) * 32;
    if (i < p.n_parts) {
      const int w = p.part_win[i];
      stream_window<MODE, TB, 2, kVec, kBuf>(p, res_ptr, res_cols, res_vals, B, ldb, bbytes, N, C, ldc, w, n0,
                                             p.part_c0[i], p.part_c1[i], i == p.hw_p0[w] && has_sparse(w),
                                             ws ? ws + (int64_t)i * 16 * N : nullptr, true, lds, wv, kStreamWaves);
    } else {
      const int w = p.W_huge + i - p.n_parts;
      stream_window<MODE, TB, 2, kVec, kBuf>(p, res_ptr, res_cols, res_vals, B, ldb, bbytes, N, C, ldc, w, n0,
                                             p.tc_ptr[w], p.tc_ptr[w + 1], has_sparse(w), nullptr, false, lds, wv,
                                             kStreamWaves);
    }
    return;
  }
  // kStreamWaves / nw windows side by side.  Waves of a last workgroup that have no
  // window left end here: the barrier waits for the waves that have not ended.
  const int sub = wv / nw;
  const int job = (block - big) * (kStreamWaves / nw) + sub;
  const int i = job / nC, n0 = (job - i * nC) * 64;
  const int w = p.W_big + i;
  if (w >= p.W_tc) return;
  stream_window<MODE, TB, 4, kVec, kBuf>(p, res_ptr, res_cols, res_vals, B, ldb, bbytes, N, C, ldc, w, n0,
                                         p.tc_ptr[w], p.tc_ptr[w + 1], has_sparse(w), nullptr, false,
                                         lds + sub * (nw + 1) * 16 * 64, wv - sub * nw, nw);
}

// Chunks [a, b) of a window into acc, two at a time, the column ids of the next
// two requested under the current ones' B rows.
template <int MODE, typename TB, bool kVec, bool kBuf>
__device__ __forceinline__ void full_chunks(const StreamArrays& A, const ChunkReader<TB, 4, kVec, kBuf>& rd, int a,
                                            int b, f32x4 (&acc)[4]) {
  const int g = (threadIdx.x & 63) >> 4;
  struct Ids {
    int4 ka, kb;
  };
  auto ids_of = [&](int c) {
    const int4* cp = reinterpret_cast<const int4*>(A.tc_cols + (int64_t)min(c, b - 1) * 32 + g * 8);
    return Ids{cp[0], cp[1]};
  };
  Ids i0 = ids_of(a), i1 = ids_of(a + 1);
  int c = a;
  for (; c + 1 < b; c += 2) {
    ChunkA<MODE> a0, a1;
    ChunkB<TB, 4, kVec> b0, b1;
    a0.load(A.tc_vals, A.tc_scale, c);
    a1.load(A.tc_vals, A.tc_scale, c + 1);
    rd.load(i0.ka, i0.kb, b0);
    rd.load(i1.ka, i1.kb, b1);
    i0 = ids_of(c + 2);
    i1 = ids_of(c + 3);
    mfma_chunk<MODE>(a0, b0, acc);
    mfma_chunk<MODE>(a1, b1, acc);
  }
  if (c < b) {
    ChunkA<MODE> a0;
    ChunkB<TB, 4, kVec> b0;
    a0.load(A.tc_vals, A.tc_scale, c);
    rd.load(i0.ka, i0.kb, b0);
    mfma_chunk<MODE>(a0, b0, acc);
  }
}

// Launches that fill the GPU with a wave per (window, 64 columns) (full_launch):
// blocks [0, (n_parts + W_long - W_huge) * nC) each run one (part, or window of
// more than kLongChunks chunks) on all their waves, a contiguous share each, whose
// sums the first wave adds in wave order; the next ones run kStreamWaves of the
// other (window, 64 columns), one per wave, stored from its registers.
template <int MODE, typename TB, bool kVec, bool kBuf>
__global__ __launch_bounds__(kStreamWaves * 64) void hyb_spmm_stream_full_kernel(
    StreamArrays p, const TB* __restrict__ B, int64_t ldb, uint32_t bbytes, int N, float* __restrict__ C, int64_t ldc,
    int nC, float* __restrict__ ws) {
  __shared__ f32x4 sums[kStreamWaves - 1][4][64];
  const int lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int shared = (p.n_parts + p.W_long - p.W_huge) * nC;
  const bool alone = (int)blockIdx.x >= shared;
  const int job = alone ? ((int)blockIdx.x - shared) * kStreamWaves + wv : (int)blockIdx.x;
  const int i = job / nC, n0 = (job - i * nC) * 64;
  const bool in_part = !alone && i < p.n_parts;
  const int w = alone ? p.W_long + i : in_part ? p.part_win[i] : p.W_huge + i - p.n_parts;
  if (alone && w >= p.W_tc) return;
  const int c0 = in_part ? p.part_c0[i] : p.tc_ptr[w], c1 = in_part ? p.part_c1[i] : p.tc_ptr[w + 1];
  const int share = (c1 - c0 + kStreamWaves - 1) / kStreamWaves;
  const int a = alone ? c0 : min(c0 + wv * share, c1), b = alone ? c1 : min(a + share, c1);
  // rows before any store: vector-memory counters complete in issue order
  int row[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) row[r] = p.win_rows[w * 16 + 4 * g + r];
  f32x4 acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (a < b) full_chunks<MODE>(p, ChunkReader<TB, 4, kVec, kBuf>(B, ldb, bbytes, n0, N), a, b, acc);
  if (!alone) {  // the whole workgroup
    if (wv > 0) {
#pragma unroll
      for (int t = 0; t < 4; ++t) sums[wv - 1][t][lane] = acc[t];
    }
    __syncthreads();
    if (wv > 0) return;
    for (int v = 0; v < kStreamWaves - 1; ++v)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t] += sums[v][t][lane];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float* at = in_part && ws ? ws + ((int64_t)i * 16 + 4 * g + r) * N : C + (int64_t)row[r] * ldc;
    const bool out = (in_part && ws) || row[r] >= 0;
    auto col = [&](int t) { return n0 + (kVec ? 4 * j + t : 16 * t + j); };
    if (in_part && !ws) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (out && col(t) < N) atomicAdd(at + col(t), acc[t][r]);
    } else if constexpr (kVec) {
      if (out && col(0) < N) {
        if (in_part) {  // rows of ws are aligned for a float only
#pragma unroll
          for (int t = 0; t < 4; ++t) at[col(t)] = acc[t][r];
        } else {
          st4(at + col(0), make_float4(acc[0][r], acc[1][r], acc[2][r], acc[3][r]));
        }
      }
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (out && col(t) < N) at[col(t)] = acc[t][r];
    }
  }
}

// Deterministic mode: C rows of huge window w = sum of its parts' partial
// rows in part order.  One wave per (huge window, 64 columns).
__global__ __launch_bounds__(256) void hyb_spmm_part_reduce_kernel(SpmmPlanDev p, int N, float* __restrict__ C,
                                                                   int64_t ldc, int nC, bool vec,
                                                                   const float* __restrict__ ws) {
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if (wave >= (int64_t)p.W_huge * nC) return;
  const int w = (int)(wave / nC);
  const int lane = threadIdx.x & 63, g = lane >> 4;
  const int col = (int)(wave - (int64_t)w * nC) * 64 + 4 * (lane & 15);
  const int q0 = p.hw_p0[w], q1 = p.hw_p0[w + 1];
  float4 acc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int q = q0; q < q1; ++q) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 v = load_b4(ws + (int64_t)q * 16 * N, N, 4 * g + i, col, N, vec);
      acc[i].x += v.x; acc[i].y += v.y; acc[i].z += v.z; acc[i].w += v.w;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = p.win_rows[w * 16 + 4 * g + i];
    if (row >= 0) store_c4(C, ldc, row, col, N, vec, acc[i]);
  }
}

// Waves per (window, 64 columns) of hyb_spmm_stream_kernel: half a workgroup's
// when the windows hold few chunks on average and there are enough of them to fill
// the GPU, else all.  Windows of four chunks, FP32, four waves / eight: 512
// (window, 64 columns) 6.0 / 6.0 us, 1,024 7.3 / 8.3; of eight chunks 7.1 / 6.3
// and 12.3 / 10.5.
static int waves_per_window(const SpmmPlanDev& p, int nC) {
  const int64_t small = p.W_tc - p.W_big;
  return small > 0 && p.chunks_small <= 4 * small && small * nC >= 512 ? kStreamWaves / 2 : kStreamWaves;
}

// Whether hyb_spmm_stream_full_kernel runs the dense windows.  Several waves per
// window and their sum through LDS are for launches that leave the GPU idle; with
// two waves per SIMD and more of one-wave (window, 64 columns) they only cost.
// Windows of one chunk, full / not: FP32, 1,024 of them 5.3 / 5.3 us, 2,048 5.3 /
// 8.3, 8,192 12.6 / 29.0; of eight chunks 15.5 / 12.3, 17.7 / 22.0 and 47 / 73;
// BF16 of eight chunks 8.4 / 7.6, 9.3 / 12.9 and 25.9 / 49.  A window that a whole
// workgroup shares counts as its eight waves where there are no others (17 chunks,
// FP32, 128 / 256 of them: 6.3 / 5.9 and 6.5 / 9.4), as one beside windows of up to
// eight chunks in one wave (2048 x 1024 FP16 layer, N = 512 9.4 / 8.1, N = 1024
// 10.5 / 13.3).  Up to two chunks in sequence it is never behind.
//
// With sparse parts in the windows a full launch leaves them to the row tasks: a
// launch (4 us) and a second pass over their rows of C (0.11 ns per row and 64
// columns), against 2.5 ns per (window, 64 columns) beyond 1,024.  3072 x 768 FP32
// layer, full / not: N = 1024 28.1 / 26.2 us, N = 2048 40.8 / 45.4, N = 4096 65 / 81.
// Not with windows of more than kLongChunks chunks beside them (graphs; R-MAT scale
// 15, N = 256: 97.6 / 86.9).
static bool full_launch(const SpmmPlanDev& p, int nC) {
  const int64_t alone = (int64_t)(p.W_tc - p.W_long) * nC;
  const int64_t shared = (int64_t)(p.n_parts + p.W_long - p.W_huge) * nC;
  if (p.nnz_mix == 0) return p.full_chain <= 2 || alone + shared * (alone == 0 ? kStreamWaves : 1) >= 1536;
  return p.W_long == 0 && 250 * (alone - 1024) >= 400000 + 11 * (int64_t)p.n_mix * nC;
}

// Whether the windows' sparse parts are summed by hyb_spmm_stream_kernel: up to
// kFoldWave entries per wave of a window on average, or kFoldTotal (entry, 64
// columns) in all.  Above, the row tasks' gathers of 128 columns and their balance
// are worth the second launch.  Folded / not: 64 BF16 windows of 100 columns, N =
// 512 (four waves), 128 entries a wave and 262,144 in all 9.2 / 10.4 us, twice as
// many 14.1 / 12.6; 512 of 40 columns, N = 128 (four waves), 32 a wave 8.6 / 10.7,
// 128 and 524,288 17.8 / 14.1, 512 54 / 27; 4096 x 4096 layer, FP32, N = 256 (eight
// waves, 73 a wave) 31.9 / 36.2.  One row of 16 with kFoldMaxLen entries, four in
// the others: 8.9 / 13.5.
constexpr int64_t kFoldWave = 96, kFoldTotal = 300000;

// The launch over columns [0, N) of B and C; ws as in launch_stream.
template <typename TB>
static hipError_t stream_columns(const SpmmPlanDev& p, const TB* B, int64_t ldb, int N, float* C, int64_t ldc,
                                 bool vec, float* ws, hipStream_t s, bool full, int fold) {
  const int nC = (N + 63) / 64, nC2 = (N + 31) / 32;
  const int64_t jobs = (int64_t)(p.W_tc - p.W_big) * nC;
  const int nw = waves_per_window(p, nC);
  const int per = kStreamWaves / nw;
  const int64_t blocks =
      full ? (int64_t)(p.n_parts + p.W_long - p.W_huge) * nC +
                 ((int64_t)(p.W_tc - p.W_long) * nC + kStreamWaves - 1) / kStreamWaves
           : (int64_t)(p.n_parts + p.W_big - p.W_huge) * nC2 + (jobs + per - 1) / per;
  if (blocks > max_blocks(kStreamWaves * 64) && N > 64) {
    // in column halves: each a product of its own, with its part of ws (an offset
    // of the blocks in the kernel would take scalar registers it does not have:
    // 1024 x 4096, N = 512 14.9 -> 15.5 us)
    const int n = nC / 2 * 64;
    const hipError_t e = stream_columns(p, B, ldb, n, C, ldc, vec, ws, s, full, fold);
    if (e != hipSuccess) return e;
    return stream_columns(p, B + n, ldb, N - n, C + n, ldc, vec, ws ? ws + (int64_t)p.n_parts * 16 * n : nullptr, s,
                          full, fold);
  }
  if (p.n_parts > 0 && !ws) {
    hipError_t e = launch_zero_window_rows(p, p.W_huge, C, ldc, N, s);
    if (e != hipSuccess) return e;
  }
  // 32-bit row offsets from 24-bit products
  uint32_t bytes = b_bytes<TB>(p.K, ldb, N);
  if (p.K > (1 << 24) || ldb * (int64_t)sizeof(TB) >= (1 << 24)) bytes = 0;
  const size_t lds = (size_t)(kStreamWaves + per) * 16 * 64 * 4;
  const StreamArrays arrays{p.tc_ptr,  p.tc_cols, p.win_rows, p.tc_vals, p.tc_scale, p.part_win, p.part_c0, p.part_c1,
                            p.hw_p0,   p.W_tc,    p.W_long,   p.W_big,   p.W_huge,   p.n_parts,  fold};
  auto go = [&](auto mode, auto v, auto u) {
    constexpr int kMode = decltype(mode)::value;
    constexpr bool kV = decltype(v)::value, kU = decltype(u)::value;
    if (full)
      hipLaunchKernelGGL((hyb_spmm_stream_full_kernel<kMode, TB, kV, kU>), dim3((unsigned)blocks),
                         dim3(kStreamWaves * 64), 0, s, arrays, B, ldb, bytes, N, C, ldc, nC, ws);
    else
      hipLaunchKernelGGL((hyb_spmm_stream_kernel<kMode, TB, kV, kU>), dim3((unsigned)blocks), dim3(kStreamWaves * 64),
                         lds, s, arrays, p.res_ptr, p.res_cols, p.res_vals, B, ldb, bytes, N, C, ldc, nC, nC2, nw, ws);
  };
  auto by_layout = [&](auto mode) {
    if (bytes > 0 && vec)
      go(mode, std::true_type{}, std::true_type{});
    else if (bytes > 0)
      go(mode, std::false_type{}, std::true_type{});
    else
      go(mode, std::false_type{}, std::false_type{});
  };
  if (p.blk_dtype == 1)
    by_layout(std::integral_constant<int, 1>{});
  else if (p.blk_dtype == 2)
    by_layout(std::integral_constant<int, 2>{});
  else
    by_layout(std::integral_constant<int, 0>{});
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (ws && p.W_huge > 0) {
    const int64_t waves = (int64_t)p.W_huge * nC;
    hipLaunchKernelGGL(hyb_spmm_part_reduce_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, p, N, C, ldc,
                       nC, vec, ws);
    e = hipGetLastError();
  }
  return e;
}

template <typename TB>
hipError_t launch_stream(const SpmmPlanDev& p, const TB* B, int64_t ldb, int N, float* C, int64_t ldc, bool vec,
                         float* ws, hipStream_t s, bool* folded) {
  const int nC = (N + 63) / 64;
  const bool full = full_launch(p, nC);
  *folded = p.fold_mix && !full &&
            (p.nnz_mix <= kFoldWave * waves_per_window(p, nC) * p.W_tc || (int64_t)p.nnz_mix * nC <= kFoldTotal);
  return p.W_tc > 0 ? stream_columns(p, B, ldb, N, C, ldc, vec, ws, s, full, *folded) : hipSuccess;
}

template hipError_t launch_stream<float>(const SpmmPlanDev&, const float*, int64_t, int, float*, int64_t, bool, float*,
                                         hipStream_t, bool*);
template hipError_t launch_stream<__bf16>(const SpmmPlanDev&, const __bf16*, int64_t, int, float*, int64_t, bool,
                                          float*, hipStream_t, bool*);
template hipError_t launch_stream<_Float16>(const SpmmPlanDev&, const _Float16*, int64_t, int, float*, int64_t, bool,
                                            float*, hipStream_t, bool*);

}  // namespace stile
