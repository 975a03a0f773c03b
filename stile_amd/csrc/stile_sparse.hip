// Sparse rows of the hybrid SpMM (sparse-only windows and the pieces of long
// rows) for MI355X (gfx950).
#include "stile_rows.h"

#include <algorithm>

namespace stile {

// One wave = (task, 64 * VW columns), column chunk by column chunk.  A task is a
// run of slots: rows of at most kSplitNnz entries together, or the first
// kSplitNnz entries of one longer row (the rest are pieces).  kTaskHub: a row of
// more than kHubNnz entries, summed in FP64.  kTaskAdd: slots of a dense window,
// whose rows the streaming kernel stored before: rows with entries are added to
// them (the row of C is requested when its first entry is reached).
template <typename TB, int VW, bool kVec, bool kBuf>
__global__ __launch_bounds__(256, 4) void hyb_spmm_rows_kernel(
    const int2* __restrict__ tasks, int ntasks, const int32_t* __restrict__ res_ptr,
    const int32_t* __restrict__ cols, const float* __restrict__ vals, const int32_t* __restrict__ win_rows,
    const TB* __restrict__ B, int64_t ldb, uint32_t bbytes, int N, float* __restrict__ C, int64_t ldc, int nC) {
  const int wave = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cch = wave / ntasks;
  if (cch >= nC) return;
  const int2 t = tasks[wave - cch * ntasks];
  const int s0 = t.x, s1 = t.y & kTaskSlots;
  const bool to_c = (t.y & kTaskAdd) != 0;
  const int n0 = cch * 64 * VW;
  const int q0 = res_ptr[s0];
  const int q1 = min(res_ptr[s1], q0 + (s1 == s0 + 1 ? kSplitNnz : INT32_MAX - q0));
  const RowReader<TB, VW, kVec, kBuf> rd(B, ldb, bbytes, n0, N, threadIdx.x & 63);
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
    float before[VW];
    int beg = q0;  // the current slot's first entry
    auto begin = [&]() {
      if (to_c && row >= 0 && beg < end) load_cols<VW, kVec>(C + (int64_t)row * ldc, n0, N, before);
    };
    auto store = [&]() {
      if (row < 0 || (to_c && beg == end)) return;
      float o[VW];
#pragma unroll
      for (int c = 0; c < VW; ++c) o[c] = (float)acc[c];
      if (to_c) {
#pragma unroll
        for (int c = 0; c < VW; ++c) o[c] += before[c];
      }
      store_cols<VW, kVec>(C + (int64_t)row * ldc, n0, N, o);
    };
    auto next = [&]() {
#pragma unroll
      for (int c = 0; c < VW; ++c) acc[c] = zero;
      row = row1;
      beg = end;
      end = end1;
      begin();
      row1 = win_rows[min(slot + 1, s1 - 1)];
      end1 = min(res_ptr[min(slot + 2, s1)], q1);
    };
    begin();
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
  if (t.y & kTaskHub)
    run(0.0);
  else
    run(0.f);
}

// Sparse-only rows of much the same lengths, FP32 B, aligned (even_rows): one row per
// 16-lane group and 64 columns, four columns per lane, column chunk by column chunk.
// Bound: the gather instructions; one of 16 bytes per lane brings four entries' 256
// bytes, where hyb_spmm_rows_kernel's brings 512 bytes of one entry.  That pays where
// the four rows end together (their wave goes on to the longest's end).  8192 x 4000,
// 600,000 uniform nonzeros, N = 128: 18.5 us, 23.4 by row tasks (19.1 with ids and
// gathers not as far ahead); 262144 x 262144, 5 M, N = 256: 713 and 764.
__global__ __launch_bounds__(256, 7) void hyb_spmm_even_rows_kernel(
    int slot0, int nslots, const int32_t* __restrict__ res_ptr, const int32_t* __restrict__ cols,
    const float* __restrict__ vals, const int32_t* __restrict__ win_rows, const float* __restrict__ B, int64_t ldb,
    int N, float* __restrict__ C, int64_t ldc, int nC) {
  const int wave = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = nslots / 4;  // slots of whole windows
  const int cch = wave / waves;
  if (cch >= nC) return;
  const int lane = threadIdx.x & 63;
  const int slot = slot0 + 4 * (wave - cch * waves) + (lane >> 4);
  const int col = cch * 64 + 4 * (lane & 15);
  const int row = win_rows[slot], r0 = res_ptr[slot], r1 = res_ptr[slot + 1];
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (r0 < r1) {
    // A step's ids and values are two loads each (kRowPad entries lie behind the
    // arrays); positions past the row's end gather its last B row and are not added.
    typedef int32_t i4 __attribute__((ext_vector_type(4), aligned(4)));
    typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
    i4 k0, k1;
    f4 v0, v1;
    auto ids = [&](int q) {
      k0 = *reinterpret_cast<const i4*>(cols + q);
      k1 = *reinterpret_cast<const i4*>(cols + q + 4);
      v0 = *reinterpret_cast<const f4*>(vals + q);
      v1 = *reinterpret_cast<const f4*>(vals + q + 4);
    };
    auto step = [&](int q, auto whole) {
      constexpr bool kWhole = decltype(whole)::value;
      float4 b[8];
      float v[8];
      int last = k0[0];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        last = kWhole || q + i < r1 ? (i < 4 ? k0[i & 3] : k1[i & 3]) : last;
        b[i] = load_b4(B, ldb, last, col, N, std::true_type{});
        v[i] = i < 4 ? v0[i & 3] : v1[i & 3];
      }
      if constexpr (kWhole) ids(q + 8);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (kWhole || q + i < r1) {
          s.x += v[i] * b[i].x;
          s.y += v[i] * b[i].y;
          s.z += v[i] * b[i].z;
          s.w += v[i] * b[i].w;
        }
    };
    ids(r0);
    int q = r0;
    for (; q + 8 <= r1; q += 8) step(q, std::true_type{});
    if (q < r1) step(q, std::false_type{});
  }
  if (row >= 0) store_c4(C, ldc, row, col, N, true, s);
}

// Pieces of long rows, execution slots [pc0, pc1) (piece piece_exec[slot],
// ordered by first column so that pieces of different rows gathering the same
// B rows run together), column chunk by column chunk: summed in FP64 and added
// to C with atomicAdd (C already holds the row's first kSplitNnz entries), or,
// with ws (deterministic mode), stored to ws[piece][N] for the reduce kernel.
// One workgroup per piece and 64 * VW columns, a quarter of the entries per
// wave, the waves' sums added in wave order: a graph with few long rows has few
// pieces, and as one wave each they made the GCN layer's products (R-MAT scale
// 16, N = 256) 12 us longer; in quarters the launch takes 6.6-7.1 us, 15.1
// with the compensated FP32 sums it had before.
// FP64 sums: one conversion and one v_fma_f64 (as fast as v_fma_f32 here) per
// product against nine operations of a compensated FP32 sum, which bounded
// this kernel (1.31 M entries, N = 128: 58 -> 49 us).
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
    const RowReader<TB, VW, kVec, kBuf> rd(B, ldb, bbytes, n0, N, threadIdx.x & 63);
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

// Columns per lane: 2 for more than 64 columns when that leaves at least
// kFewWaves waves (two per SIMD: below that a wave's latency is what the launch
// takes, and narrower waves are more of them), else 1.  (4 columns per lane: 105
// registers and half the waves in flight; R-MAT scale 16, N = 256: 172 against
// 161 us.  Sixteen entries a batch: 265 us, the scalar registers spill.  One
// slice of columns per XCD: no change.)
//
// FP32 B whose 128 columns are more than kWideBytes: 1 as well.  The launch runs column chunk by column chunk, and what one chunk's
// gathers touch, half as much of B, is then found in L2 and MALL more often.  A
// graph's whole product, FP32, N = 128, two columns per lane / one: scale 18 (128
// columns are 128 MB) 430 / 366 us; 19: 938 / 793; 20: 2005 / 1709, N = 256 4000
// / 3500.  Scale 17 (64 MB) gains or loses with the plan (with dense chunks 195 /
// 183, sparse only 173 / 175, N = 200 306 / 332), smaller ones lose (16, N = 256:
// 166 / 172).  16-bit B, whose two columns are those 256 bytes a gather, keeps
// two at every size: scale 17 125 / 170, 20 1070 / 1297.
// The line lies at 64 MB, where K = 131,072 (scale 17) is the last to take two: both
// widths are within 9 % of each other there, with the sign changing by plan and N.
constexpr int64_t kFewWaves = 2048;
constexpr int64_t kWideBytes = 64 << 20;
int row_width(int N, int K, int elem, int64_t waves) {
  const int64_t chunks = (N + 127) / 128;
  const bool wide = elem == 2 || (int64_t)K * 128 * elem <= kWideBytes;
  return wide && N > 64 && waves * chunks >= kFewWaves ? 2 : 1;
}

// f(VW, kVec, kBuf) with all three as compile-time constants.  One column per
// lane is the same code aligned or not.
template <typename F>
void with_width(int vw, bool vec, bool buf, F&& f) {
  auto g = [&](auto w, auto v) {
    if (buf)
      f(w, v, std::true_type{});
    else
      f(w, v, std::false_type{});
  };
  if (vw == 1)
    g(std::integral_constant<int, 1>{}, std::false_type{});
  else if (vec)
    g(std::integral_constant<int, 2>{}, std::true_type{});
  else
    g(std::integral_constant<int, 2>{}, std::false_type{});
}

}  // namespace

template <typename TB>
hipError_t launch_sparse_rows(const SpmmPlanDev& p, const TB* B, int64_t ldb, int N, float* C, int64_t ldc, bool vec,
                              int t0, int t1, hipStream_t s) {
  const int ntasks = t1 - t0;
  if (ntasks <= 0) return hipSuccess;
  const int vw = row_width(N, p.K, sizeof(TB), ntasks);
  const int nC = (N + 64 * vw - 1) / (64 * vw);
  const uint32_t bytes = b_bytes<TB>(p.K, ldb, N);
  hipError_t e = hipSuccess;
  const int per = (int)std::max<int64_t>(1, std::min<int64_t>(ntasks, max_blocks(256) * 4 / nC));
  for (int a = t0; a < t1 && e == hipSuccess; a += std::min(per, t1 - a)) {
    const int n = std::min(per, t1 - a);
    with_width(vw, vec, bytes > 0, [&](auto w, auto v, auto u) {
      hipLaunchKernelGGL((hyb_spmm_rows_kernel<TB, decltype(w)::value, decltype(v)::value, decltype(u)::value>),
                         dim3((unsigned)(((int64_t)n * nC + 3) / 4)), dim3(256), 0, s, p.row_tasks + a, n, p.res_ptr,
                         p.res_cols, p.res_vals, p.win_rows, B, ldb, bytes, N, C, ldc, nC);
    });
    e = hipGetLastError();
  }
  return e;
}

// Rows are even when they hold kEvenMean entries on average and four times the
// longest of each four comes to at most kEvenPercent of the entries: uniform draws
// of 16 entries a row come to 129 %, R-MAT graphs to 300 % and more (their rows: 28
// us by tasks, scale 13, N = 256, 95 one per lane group).  Nine entries a row, N = 512:
// 16.6 us here, 15.9 by tasks.  A last chunk of fewer than 64 columns leaves lanes
// idle, which shows once a chunk of B outgrows an L2 (65536 x 65536, 2 M, N = 100: 154
// and 129 us; 8192 x 8192 22.2 and 24.8).  16-bit B, of which an entry's 128 columns
// are one 256-byte gather: 25.1 and 17.2 (8192 x 8192, 671,088, N = 128).
bool even_rows_fit(const SpmmPlanDev& p, int N, bool vec) {
  return p.even_rows && vec && N > 64 && (N % 64 == 0 || (int64_t)p.K * 64 * 4 <= 4 << 20);
}

hipError_t launch_even_rows(const SpmmPlanDev& p, const float* B, int64_t ldb, int N, float* C, int64_t ldc,
                            hipStream_t s) {
  const int nC = (N + 63) / 64, s1 = p.W * 16;
  // launches of whole windows (max_blocks)
  const int64_t most = std::max<int64_t>(16, max_blocks(256) / nC * 16);
  hipError_t e = hipSuccess;
  for (int64_t a = (int64_t)p.W_tc * 16; a < s1 && e == hipSuccess; a += most) {
    const int n = (int)std::min(most, s1 - a);
    hipLaunchKernelGGL(hyb_spmm_even_rows_kernel, dim3((unsigned)(((int64_t)n / 4 * nC + 3) / 4)), dim3(256), 0, s,
                       (int)a, n, p.res_ptr, p.res_cols, p.res_vals, p.win_rows, B, ldb, N, C, ldc, nC);
    e = hipGetLastError();
  }
  return e;
}

template <typename TB>
hipError_t launch_sparse_pieces(const SpmmPlanDev& p, const TB* B, int64_t ldb, int N, float* C, int64_t ldc, bool vec,
                           int pc0, int pc1, float* ws, hipStream_t s) {
  const int vw = row_width(N, p.K, sizeof(TB), (int64_t)(pc1 - pc0) * 4);
  const int nC = (N + 64 * vw - 1) / (64 * vw);
  const uint32_t bytes = b_bytes<TB>(p.K, ldb, N);
  hipError_t e = hipSuccess;
  const int per = (int)std::max<int64_t>(1, std::min<int64_t>(pc1 - pc0, max_blocks(256) / nC));
  for (int a = pc0; a < pc1 && e == hipSuccess; a += std::min(per, pc1 - a)) {
    const int n = std::min(per, pc1 - a);
    with_width(vw, vec, bytes > 0, [&](auto w, auto v, auto u) {
      hipLaunchKernelGGL((hyb_spmm_pieces_kernel<TB, decltype(w)::value, decltype(v)::value, decltype(u)::value>),
                         dim3((unsigned)((int64_t)n * nC)), dim3(256), 0, s, p.piece_exec, p.piece_row, p.piece_beg,
                         p.piece_end, a, n, p.res_cols, p.res_vals, B, ldb, bytes, N, C, ldc, ws);
    });
    e = hipGetLastError();
  }
  return e;
}

hipError_t launch_piece_reduce(const SpmmPlanDev& p, int N, float* C, int64_t ldc, bool vec, int sr0, const float* ws,
                               hipStream_t s) {
  const int nC = (N + 63) / 64;
  hipError_t e = hipSuccess;
  const int per = (int)std::max<int64_t>(1, std::min<int64_t>(p.nsrows, max_blocks(256) / nC));
  for (int a = sr0; a < p.nsrows && e == hipSuccess; a += std::min(per, p.nsrows - a)) {
    const int n = std::min(per, p.nsrows - a);
    hipLaunchKernelGGL(hyb_spmm_piece_reduce_kernel, dim3((unsigned)((int64_t)n * nC)), dim3(256), 0, s, p, N, C, ldc,
                       nC, vec, a, ws);
    e = hipGetLastError();
  }
  return e;
}

template hipError_t launch_sparse_rows<float>(const SpmmPlanDev&, const float*, int64_t, int, float*, int64_t, bool, int,
                                        int, hipStream_t);
template hipError_t launch_sparse_pieces<float>(const SpmmPlanDev&, const float*, int64_t, int, float*, int64_t, bool, int,
                                          int, float*, hipStream_t);
template hipError_t launch_sparse_rows<__bf16>(const SpmmPlanDev&, const __bf16*, int64_t, int, float*, int64_t, bool,
                                        int, int, hipStream_t);
template hipError_t launch_sparse_pieces<__bf16>(const SpmmPlanDev&, const __bf16*, int64_t, int, float*, int64_t, bool, int,
                                          int, float*, hipStream_t);
template hipError_t launch_sparse_rows<_Float16>(const SpmmPlanDev&, const _Float16*, int64_t, int, float*, int64_t, bool,
                                        int, int, hipStream_t);
template hipError_t launch_sparse_pieces<_Float16>(const SpmmPlanDev&, const _Float16*, int64_t, int, float*, int64_t, bool, int,
                                          int, float*, hipStream_t);

}  // namespace stile
