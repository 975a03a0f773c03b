// Streaming kernel of the hybrid SpMM: dense windows whose B does not fit the
// B-stationary kernel (FP32 and FP16 blocks, K > kLdsMaxK), for MI355X (gfx950).
#include "stile_rows.h"

#include <algorithm>

namespace stile {

// ---------------------------------------------------------------------------
// One workgroup = (window or part of a huge window, 16 * NT columns).  Each wave
// takes a contiguous share of the window's chunks and, in plans that fold the
// sparse parts, some of its 16 slots' sparse entries; the partial sums meet in
// LDS, are added in wave order and leave as whole rows of C.
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
// 8.7, 38 and 14.9 us.
// ---------------------------------------------------------------------------
constexpr int kStreamWaves = 8;

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
  int32_t W_tc, W_big, W_huge, n_parts, fold_mix;
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
  const int share = max((c1 - c0 + nw - 1) / nw, 1);  // (no chunks: see the kernel's last job)
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
  // kStreamWaves / nw windows side by side; a last workgroup with fewer left runs
  // the spare waves on no chunks and columns from N on, so that every wave meets
  // the others at the same barrier and stores nothing
  const int sub = wv / nw;
  const int job = (block - big) * (kStreamWaves / nw) + sub;
  const int i = job / nC;
  const bool live = p.W_big + i < p.W_tc;
  const int w = live ? p.W_big + i : p.W_tc - 1, n0 = live ? (job - i * nC) * 64 : N;
  const int c0 = p.tc_ptr[w], c1 = live ? p.tc_ptr[w + 1] : c0;
  stream_window<MODE, TB, 4, kVec, kBuf>(p, res_ptr, res_cols, res_vals, B, ldb, bbytes, N, C, ldc, w, n0, c0, c1,
                                         live && has_sparse(w), nullptr, false, lds + sub * (nw + 1) * 16 * 64,
                                         wv - sub * nw, nw);
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

template <typename TB>
hipError_t launch_stream(const SpmmPlanDev& p, const TB* B, int64_t ldb, int N, float* C, int64_t ldc, bool vec,
                         float* ws, hipStream_t s) {
  if (p.W_tc == 0) return hipSuccess;
  const int nC = (N + 63) / 64, nC2 = (N + 31) / 32;
  // Waves per (window, 64 columns): half a workgroup's when the windows hold few
  // chunks on average and there are enough of them to fill the GPU, else all.
  const int64_t jobs = (int64_t)(p.W_tc - p.W_big) * nC;
  const bool few = p.W_tc > p.W_big && p.chunks_small <= (int64_t)4 * (p.W_tc - p.W_big);
  const int nw = few && jobs >= 512 ? kStreamWaves / 2 : kStreamWaves;
  const int per = kStreamWaves / nw;
  const int64_t blocks = (int64_t)(p.n_parts + p.W_big - p.W_huge) * nC2 + (jobs + per - 1) / per;
  if (blocks > max_blocks(kStreamWaves * 64) && N > 64) {
    // in column halves: each a product of its own, with its part of ws (an offset
    // of the blocks in the kernel would take scalar registers it does not have:
    // 1024 x 4096, N = 512 14.9 -> 15.5 us)
    const int n = nC / 2 * 64;
    hipError_t e = launch_stream(p, B, ldb, n, C, ldc, vec, ws, s);
    if (e != hipSuccess) return e;
    return launch_stream(p, B + n, ldb, N - n, C + n, ldc, vec, ws ? ws + (int64_t)p.n_parts * 16 * n : nullptr, s);
  }
  if (p.n_parts > 0 && !ws) {
    hipError_t e = launch_zero_window_rows(p, p.W_huge, C, ldc, N, s);
    if (e != hipSuccess) return e;
  }
  // 32-bit row offsets from 24-bit products
  uint32_t bytes = b_bytes<TB>(p.K, ldb, N);
  if (p.K > (1 << 24) || ldb * (int64_t)sizeof(TB) >= (1 << 24)) bytes = 0;
  const size_t lds = (size_t)(kStreamWaves + per) * 16 * 64 * 4;
  const StreamArrays arrays{p.tc_ptr,  p.tc_cols, p.win_rows, p.tc_vals, p.tc_scale, p.part_win, p.part_c0,
                            p.part_c1, p.hw_p0,   p.W_tc,     p.W_big,   p.W_huge,   p.n_parts,  p.fold_mix};
  auto go = [&](auto mode, auto v, auto u) {
    hipLaunchKernelGGL((hyb_spmm_stream_kernel<decltype(mode)::value, TB, decltype(v)::value, decltype(u)::value>),
                       dim3((unsigned)blocks), dim3(kStreamWaves * 64), lds, s, arrays, p.res_ptr, p.res_cols, p.res_vals, B,
                       ldb, bytes, N, C, ldc, nC, nC2, nw, ws);
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

template hipError_t launch_stream<float>(const SpmmPlanDev&, const float*, int64_t, int, float*, int64_t, bool, float*,
                                         hipStream_t);
template hipError_t launch_stream<__bf16>(const SpmmPlanDev&, const __bf16*, int64_t, int, float*, int64_t, bool,
                                          float*, hipStream_t);
template hipError_t launch_stream<_Float16>(const SpmmPlanDev&, const _Float16*, int64_t, int, float*, int64_t, bool,
                                            float*, hipStream_t);

}  // namespace stile
