// HIP kernels of libstile_hip.so for MI355X (gfx950, CDNA4, wave64).
//
// The kernels here:
//   csr_spmm_f32     plain CSR SpMM (the comparator; reference csrmm template,
//                    MY_sparse/my_fuse_formats.py:1106-1152)
//   csr_sddmm_f32    plain per-nonzero SDDMM (reference golden u_dot_v,
//                    my_fuse_formats.py:4331-4341)
//   hyb_spmm_lds     hybrid fused SpMM of BF16 plans with K <= kLdsMaxK: dense
//                    16-row blocks on MFMA against B staged in LDS + the FP32
//                    sparse part, every C row written once (replaces the fused
//                    ELL + TensorCore templates, my_fuse_formats.py:1162-1291,
//                    1444-1799, 2426-2465)
//   sparse_split     few sparse rows: one wave per row and 64 columns
//   row softmax, value refresh, ELL buckets (comparator), zero fills
// and launch_hyb_spmm, which picks a product's kernels: these, the streaming
// kernel (stile_stream.hip) and the sparse rows (stile_sparse.hip).  The SDDMM,
// the fused attention and the tall product have files of their own.
#include "stile_device.h"

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>

namespace stile {

// ---------------------------------------------------------------------------
// Plain CSR SpMM.  A segment of LPR lanes owns one row and CPL groups of
// 4*LPR consecutive columns (one float4 per lane per group); a wave holds
// 64/LPR rows.  Grid: (row groups) x (column blocks of 4*LPR*CPL).
// ---------------------------------------------------------------------------
template <int LPR, int CPL>
__global__ __launch_bounds__(256) void csr_spmm_f32_kernel(
    int M, int N, const int32_t* __restrict__ indptr,
    const int32_t* __restrict__ indices, const float* __restrict__ vals,
    const float* __restrict__ B, int64_t ldb, float* __restrict__ C,
    int64_t ldc, bool vec) {
  constexpr int RPW = 64 / LPR;
  const int lane = threadIdx.x & 63;
  const int sub = lane % LPR;
  const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int row = wave * RPW + lane / LPR;
  if (row >= M) return;
  const int col0 = blockIdx.y * (4 * LPR * CPL) + 4 * sub;
  const int p0 = indptr[row], p1 = indptr[row + 1];

  float4 acc[CPL];
#pragma unroll
  for (int q = 0; q < CPL; ++q) acc[q] = make_float4(0.f, 0.f, 0.f, 0.f);

  if (p1 - p0 <= kHubNnz) {
    int p = p0;
    for (; p + 4 <= p1; p += 4) {
      const int k0 = indices[p], k1 = indices[p + 1], k2 = indices[p + 2],
                k3 = indices[p + 3];
      const float v0 = vals[p], v1 = vals[p + 1], v2 = vals[p + 2],
                  v3 = vals[p + 3];
#pragma unroll
      for (int q = 0; q < CPL; ++q) {
        const int col = col0 + q * 4 * LPR;
        const float4 b0 = load_b4(B, ldb, k0, col, N, vec);
        const float4 b1 = load_b4(B, ldb, k1, col, N, vec);
        const float4 b2 = load_b4(B, ldb, k2, col, N, vec);
        const float4 b3 = load_b4(B, ldb, k3, col, N, vec);
        acc[q].x += v0 * b0.x; acc[q].y += v0 * b0.y; acc[q].z += v0 * b0.z; acc[q].w += v0 * b0.w;
        acc[q].x += v1 * b1.x; acc[q].y += v1 * b1.y; acc[q].z += v1 * b1.z; acc[q].w += v1 * b1.w;
        acc[q].x += v2 * b2.x; acc[q].y += v2 * b2.y; acc[q].z += v2 * b2.z; acc[q].w += v2 * b2.w;
        acc[q].x += v3 * b3.x; acc[q].y += v3 * b3.y; acc[q].z += v3 * b3.z; acc[q].w += v3 * b3.w;
      }
    }
    for (; p < p1; ++p) {
      const int k = indices[p];
      const float v = vals[p];
#pragma unroll
      for (int q = 0; q < CPL; ++q) {
        const float4 b = load_b4(B, ldb, k, col0 + q * 4 * LPR, N, vec);
        acc[q].x += v * b.x; acc[q].y += v * b.y; acc[q].z += v * b.z; acc[q].w += v * b.w;
      }
    }
  } else {
    // Hub row: compensated FP32 summation.
    float4 cc[CPL];
#pragma unroll
    for (int q = 0; q < CPL; ++q) cc[q] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int p = p0; p < p1; ++p) {
      const int k = indices[p];
      const float v = vals[p];
#pragma unroll
      for (int q = 0; q < CPL; ++q) {
        const float4 b = load_b4(B, ldb, k, col0 + q * 4 * LPR, N, vec);
        neu_add(acc[q].x, cc[q].x, v * b.x);
        neu_add(acc[q].y, cc[q].y, v * b.y);
        neu_add(acc[q].z, cc[q].z, v * b.z);
        neu_add(acc[q].w, cc[q].w, v * b.w);
      }
    }
#pragma unroll
    for (int q = 0; q < CPL; ++q) {
      acc[q].x += cc[q].x; acc[q].y += cc[q].y; acc[q].z += cc[q].z; acc[q].w += cc[q].w;
    }
  }
#pragma unroll
  for (int q = 0; q < CPL; ++q)
    store_c4(C, ldc, row, col0 + q * 4 * LPR, N, vec, acc[q]);
}

template <int LPR, int CPL>
static hipError_t launch_csr_spmm_cfg(int M, int N, const int32_t* indptr,
                                      const int32_t* indices,
                                      const float* vals, const float* B,
                                      int64_t ldb, float* C, int64_t ldc,
                                      bool vec, hipStream_t s) {
  constexpr int RPW = 64 / LPR;
  const int waves = (M + RPW - 1) / RPW;
  const int cb = 4 * LPR * CPL;
  dim3 grid((waves + 3) / 4, (N + cb - 1) / cb);
  hipLaunchKernelGGL((csr_spmm_f32_kernel<LPR, CPL>), grid, dim3(256), 0, s,
                     M, N, indptr, indices, vals, B, ldb, C, ldc, vec);
  return hipGetLastError();
}

hipError_t launch_csr_spmm_f32(int M, int N, const int32_t* indptr,
                               const int32_t* indices, const float* vals,
                               const float* B, int64_t ldb, float* C,
                               int64_t ldc, hipStream_t s) {
  if (M == 0 || N == 0) return hipSuccess;
  const bool vec = (N % 4 == 0) && (ldb % 4 == 0) && (ldc % 4 == 0) &&
                   ((reinterpret_cast<uintptr_t>(B) & 15) == 0) &&
                   ((reinterpret_cast<uintptr_t>(C) & 15) == 0);
  if (N <= 16)
    return launch_csr_spmm_cfg<4, 1>(M, N, indptr, indices, vals, B, ldb, C, ldc, vec, s);
  if (N <= 32)
    return launch_csr_spmm_cfg<8, 1>(M, N, indptr, indices, vals, B, ldb, C, ldc, vec, s);
  if (N <= 64)
    return launch_csr_spmm_cfg<16, 1>(M, N, indptr, indices, vals, B, ldb, C, ldc, vec, s);
  if (N <= 128)
    return launch_csr_spmm_cfg<32, 1>(M, N, indptr, indices, vals, B, ldb, C, ldc, vec, s);
  if (N <= 256)
    return launch_csr_spmm_cfg<64, 1>(M, N, indptr, indices, vals, B, ldb, C, ldc, vec, s);
  return launch_csr_spmm_cfg<64, 2>(M, N, indptr, indices, vals, B, ldb, C, ldc, vec, s);
}

// ---------------------------------------------------------------------------
// Plain CSR SDDMM: a segment of LPE lanes owns one nonzero; each lane loads
// float4 slices of X[row] and Y[col] and the segment reduces with xor
// shuffles.  The row of each nonzero is found by binary search in indptr.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int find_row(const int32_t* __restrict__ indptr,
                                        int M, int p) {
  int lo = 0, hi = M;  // indptr[lo] <= p < indptr[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (indptr[mid] <= p) lo = mid; else hi = mid;
  }
  return lo;
}

template <int LPE>
__device__ __forceinline__ float segment_dot(const float* __restrict__ x,
                                             const float* __restrict__ y,
                                             int Kf, int sub, bool vec) {
  float s = 0.f;
  if (vec) {
    for (int k = 4 * sub; k < Kf; k += 4 * LPE) {
      const float4 a = ld4(x + k), b = ld4(y + k);
      s += a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w;
    }
  } else {
    for (int k = sub; k < Kf; k += LPE) s += x[k] * y[k];
  }
#pragma unroll
  for (int off = LPE / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, LPE);
  return s;
}

template <int LPE>
__global__ __launch_bounds__(256) void csr_sddmm_f32_kernel(
    int M, int nnz, int Kf, const int32_t* __restrict__ indptr,
    const int32_t* __restrict__ indices, const float* __restrict__ X,
    int64_t ldx, const float* __restrict__ Y, int64_t ldy,
    float* __restrict__ out, bool vec) {
  constexpr int EPW = 64 / LPE;
  const int lane = threadIdx.x & 63;
  const int sub = lane % LPE;
  const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int p = wave * EPW + lane / LPE;
  if (p >= nnz) return;
  const int row = find_row(indptr, M, p);
  const int col = indices[p];
  const float s = segment_dot<LPE>(X + (int64_t)row * ldx,
                                   Y + (int64_t)col * ldy, Kf, sub, vec);
  if (sub == 0) out[p] = s;
}

hipError_t launch_csr_sddmm_f32(int M, int nnz, int Kf, const int32_t* indptr,
                                const int32_t* indices, const float* X,
                                int64_t ldx, const float* Y, int64_t ldy,
                                float* out, hipStream_t s) {
  if (nnz == 0) return hipSuccess;
  const bool vec = (Kf % 4 == 0) && (ldx % 4 == 0) && (ldy % 4 == 0) &&
                   ((reinterpret_cast<uintptr_t>(X) & 15) == 0) &&
                   ((reinterpret_cast<uintptr_t>(Y) & 15) == 0);
  int lpe = vec ? Kf / 4 : Kf;
  if (lpe > 16) lpe = 16;
  int l = 1;
  while (l * 2 <= lpe) l *= 2;
  lpe = l;
  const int epw = 64 / lpe;
  const int waves = (nnz + epw - 1) / epw;
  dim3 grid((waves + 3) / 4);
#define STILE_SDDMM_CASE(L)                                                  \
  case L:                                                                    \
    hipLaunchKernelGGL(csr_sddmm_f32_kernel<L>, grid, dim3(256), 0, s, M,    \
                       nnz, Kf, indptr, indices, X, ldx, Y, ldy, out, vec); \
    break;
  switch (lpe) {
    STILE_SDDMM_CASE(1)
    STILE_SDDMM_CASE(2)
    STILE_SDDMM_CASE(4)
    STILE_SDDMM_CASE(8)
    STILE_SDDMM_CASE(16)
  }
#undef STILE_SDDMM_CASE
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Hybrid fused SpMM.
//
// Kernels of one run, in stream order.  Plans on the B-stationary kernel
// (BF16 blocks, K <= kLdsMaxK): that kernel computes every dense window with
// its sparse part, and as its tail (when they are few) the sparse-only rows;
// otherwise the sparse-row kernels run the sparse-only rows.  Other plans: a
// streaming kernel (stile_stream.hip) stores the dense windows, with their sparse
// parts when those are few and short and the launch does not fill the GPU, and the
// sparse-row kernels (stile_sparse.hip) add the others and write the sparse-only
// windows.
// Last, the pieces of rows longer than kSplitNnz: added with atomicAdd, or, in
// the deterministic mode, summed into a workspace and added by a reduce kernel.
//
// B is FP32, BF16 or FP16 (TB); every product and sum of the sparse part is
// FP32 on B's exact values (FP64 sums for hub rows and pieces).
// ---------------------------------------------------------------------------

// The plan arrays that the B-stationary kernel and its tail of sparse rows read:
// what those launches pass of a plan.  The size of a launch's arguments shows in
// its time.  With the whole SpmmPlanDev among them the kernel's were 864 bytes,
// and two fields more in that structure (880 bytes, the kernel's instructions the
// same) made the block-pruned layer at N = 4096 slower, 12.97 -> 13.13 us a pass;
// with these arrays alone (464 bytes) it takes 13.00.
struct WindowArrays {
  int32_t W, W_tc;
  const int32_t *win_rows, *tc_cols;
  const void* tc_vals;
  const int2* sp_ent;
  const int32_t *res_ptr, *res_cols;
  const float* res_vals;
};
static_assert(sizeof(WindowArrays) == 64, "arguments of the B-stationary launch: see above");

static WindowArrays window_arrays(const SpmmPlanDev& p) {
  return {p.W, p.W_tc, p.win_rows, p.tc_cols, p.tc_vals, p.sp_ent, p.res_ptr, p.res_cols, p.res_vals};
}

// Output rows of the 4 slots a lane group stores.  Loaded before any of the
// window's C stores: vector-memory counters complete in issue order on
// CDNA, so a load issued after a store would wait for it.
struct SlotRows {
  int row[4];
};

__device__ __forceinline__ SlotRows load_rows(const WindowArrays& p, int slot0) {
  SlotRows sr;
#pragma unroll
  for (int i = 0; i < 4; ++i) sr.row[i] = p.win_rows[slot0 + i];
  return sr;
}

// Store the dense accumulators of the lane group's 4 rows (acc[t][i] is row
// 4g+i, column col+t).
template <bool NT = false>
__device__ __forceinline__ void store_window(float* __restrict__ C, int64_t ldc, int N, int col, bool vec,
                                             const SlotRows& sr, const f32x4 (&acc)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (sr.row[i] >= 0)
      store_c4<NT>(C, ldc, sr.row[i], col, N, vec, make_float4(acc[0][i], acc[1][i], acc[2][i], acc[3][i]));
}

// Sparse-only rows for launches with too few rows to fill the GPU at one row
// per 16-lane group: one wave per (row, 64 columns).  Task `wave` = (row
// wave / nC, column chunk wave % nC).  The row's nonzeros go 64 at a time:
// lane (g, j) loads nonzero base + 16g + j (column and value, one load each,
// so a round costs one index latency), lane group g's sixteen are passed to
// its lanes by shuffles, and the group's 16 B-row gathers are in flight
// together.  Positions past r1 read the row's last entry with weight 0.
// Fixed order: within a group u = 0..15 per round, then the xor-shuffle sum
// over the four groups.  Rows with more than kHubNnz sparse nonzeros sum with
// Neumaier compensation.
template <typename TB>
__device__ __forceinline__ void sparse_split_wave(const WindowArrays& p, const TB* __restrict__ B, int64_t ldb,
                                                  int N, float* __restrict__ C, int64_t ldc, int nC, bool vec,
                                                  int64_t wave) {
  const int lane = threadIdx.x & 63;
  const int64_t rows = (int64_t)(p.W - p.W_tc) * 16;
  if (wave >= rows * nC) return;
  const int64_t ri = wave / nC;
  const int n0 = (int)(wave - ri * nC) * 64;
  const int slot = p.W_tc * 16 + (int)ri;
  const int g = lane >> 4;
  const int col = n0 + 4 * (lane & 15);
  const int row = p.win_rows[slot];
  const int r0 = p.res_ptr[slot], rend = p.res_ptr[slot + 1];
  const int r1 = min(rend, r0 + kSplitNnz);
  const bool compensated = rend - r0 > kHubNnz;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f), cc = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int base = r0; base < r1; base += 64) {
    const int q = base + lane;  // = base + 16g + j
    const int qc = min(q, r1 - 1);
    const int kq = p.res_cols[qc];
    const float vq = q < r1 ? p.res_vals[qc] : 0.f;
    float4 b[16];
    float v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int src = (lane & 48) + u;
      const int k = __shfl(kq, src);
      v[u] = __shfl(vq, src);
      b[u] = load_b4(B, ldb, k, col, N, vec);
    }
    if (compensated) {
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        neu_add(s.x, cc.x, v[u] * b[u].x);
        neu_add(s.y, cc.y, v[u] * b[u].y);
        neu_add(s.z, cc.z, v[u] * b[u].z);
        neu_add(s.w, cc.w, v[u] * b[u].w);
      }
    } else {
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        s.x += v[u] * b[u].x;
        s.y += v[u] * b[u].y;
        s.z += v[u] * b[u].z;
        s.w += v[u] * b[u].w;
      }
    }
  }
  s.x += cc.x; s.y += cc.y; s.z += cc.z; s.w += cc.w;
#pragma unroll
  for (int off = 16; off <= 32; off <<= 1) {
    s.x += __shfl_xor(s.x, off);
    s.y += __shfl_xor(s.y, off);
    s.z += __shfl_xor(s.z, off);
    s.w += __shfl_xor(s.w, off);
  }
  if (g == 0 && row >= 0) store_c4(C, ldc, row, col, N, vec, s);
}

template <typename TB>
__global__ __launch_bounds__(256) void hyb_spmm_sparse_split_kernel(WindowArrays p, const TB* __restrict__ B,
                                                                    int64_t ldb, int N, float* __restrict__ C,
                                                                    int64_t ldc, int nC, bool vec) {
  with_vec(vec, [&](auto V) {
    sparse_split_wave(p, B, ldb, N, C, ldc, nC, V, (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6));
  });
}

// ---------------------------------------------------------------------------
// B-stationary variant for BF16 plans whose matrices all have K <= kLdsMaxK:
// a workgroup takes one work unit (a run of dense windows of one matrix,
// whose columns are B rows [koff, koff + ksz)) and one 64-column chunk,
// stages B[koff:koff+ksz, n0:n0+64] as BF16 in LDS and runs the unit's
// windows against it, a chunk-balanced run of windows per wave.  Each B row
// then leaves L2 once per workgroup instead of once per window.
//
// LDS row r (B row koff + r) starts at byte r * kLdsRowBytes and holds the
// 64 columns in the order position 16t + 4q + s <-> column n0 + 16q + 4s + t.
// The MFMA B operand of tile t is read with ds_read_b64_tr_b16: within each
// 16-lane group, result element e of lane i is element i % 4 of the 8 bytes
// that lane 4e + i / 4 of the group addresses.  Lane (g, 4e' + q) addresses
// row tc_cols[c][g][e'] (first read) and tc_cols[c][g][e' + 4] (second read)
// at position 16t + 4q, so lane j of group g receives B[col(g, e)][n0 + 4j +
// t] for e = 0..7 -- its MFMA B operand, with no repacking in registers, and
// the lane's four tiles hold four consecutive columns (each C store
// instruction writes four rows of 64 consecutive floats).  The 32 padding
// bytes per row put the 32 bytes one row contributes to a read at bank
// offset 40 r + 8 t (mod 64 banks): the 8 rows of a half-wave fall on
// distinct banks when their row ids differ mod 8, which the plan arranges
// (k-slot order within each chunk).
// ---------------------------------------------------------------------------

constexpr int kLdsThreads = 1024;

// Stage B[koff : koff + ksz, n0 : n0 + 64] into the LDS rows.  Consecutive
// threads take consecutive 16-byte pieces of the block, so every load
// instruction reads whole rows; each thread loads all its pieces (at most
// 8 of 16-bit B, 12 of FP32 B per round: one round up to K = 768) before
// writing them.  Columns at or beyond N are staged as 0.
//   16-bit B (vec16): piece (row r, columns 8b .. 8b + 7) -> for t = 0..3 the
//     pair of columns 8b + t, 8b + 4 + t to position 16t + 4(b / 2) + 2(b % 2)
//     (one v_perm_b32 and one 4-byte write each);
//   FP32 B: piece (row r, columns 4m .. 4m + 3) -> column 4m + t to position
//     16t + m (two packed conversions, four 2-byte writes).
// kStore == 2 (rows of B or C not aligned for a vector of columns): the same
// pieces at any alignment, 16-byte loads that need element alignment only; a
// piece that reaches past N is read from N - 8, or N - 4, on and shifted.  Only
// widths below one piece are read element by element, which is 8 times the
// loads (and as many store instructions, see store_window_lds): 3072 x 768
// times N = 4093, BF16 B: 36.3 us element by element, 18.3 so (N = 4096, every
// row aligned: 13.2); 1024 x 1000, N = 333: 12.8 and 7.4, FP32 B 20.6 and 11.7;
// 24-layer batch of 1024 x 4096 layers, N = 101: 95.5 and 70.6.
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

// Eight 16-bit columns from c0 on of a row of N >= 8, zero at or beyond N.
template <typename TB>
__device__ __forceinline__ uint4 load8_any(const TB* __restrict__ row, int c0, int N) {
  const int c = min(c0, N - 8);
  const u32x4_any d = *reinterpret_cast<const u32x4_any*>(row + c);
  uint64_t lo = ((uint64_t)d[1] << 32) | d[0], hi = ((uint64_t)d[3] << 32) | d[2];
  const int s = 16 * (c0 - c);  // bits to drop: 0 inside the row
  if (s > 0) {
    lo = s >= 64 ? hi >> (s & 63) : (lo >> s) | (hi << (64 - s));
    hi = s >= 64 ? 0 : hi >> s;
    if (s >= 128) lo = 0;
  }
  return make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
}

// Four FP32 columns from c0 on of a row of N >= 4, zero at or beyond N.
__device__ __forceinline__ float4 load4_any(const float* __restrict__ row, int c0, int N) {
  const int c = min(c0, N - 4), s = c0 - c;
  const f32x4_any d = *reinterpret_cast<const f32x4_any*>(row + c);
  float4 r = make_float4(d[0], d[1], d[2], d[3]);
  if (s & 1) r = make_float4(r.y, r.z, r.w, 0.f);
  if (s & 2) r = make_float4(r.z, r.w, 0.f, 0.f);
  return s >= 4 ? make_float4(0.f, 0.f, 0.f, 0.f) : r;
}

template <typename TB, int kStore>
__device__ __forceinline__ void stage_b(lds_u8* lds, const TB* __restrict__ B, int64_t ldb, int koff, int ksz,
                                        int n0, int N, bool vec, bool vec16) {
  constexpr bool kAny = kStore == 2;
  if constexpr (!std::is_same<TB, float>::value) {
    if (vec16 || (kAny && N >= 8)) {
      constexpr int U = kLdsMaxK * 8 / kLdsThreads;
      const int items = ksz * 8;
      uint4 d[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int it = min((int)threadIdx.x + u * kLdsThreads, items - 1);
        const int c0 = n0 + 8 * (it & 7);
        const TB* row = B + (int64_t)(koff + (it >> 3)) * ldb;
        if constexpr (kAny)
          d[u] = load8_any(row, c0, N);
        else
          d[u] = c0 < N ? *reinterpret_cast<const uint4*>(row + c0) : make_uint4(0, 0, 0, 0);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int it = threadIdx.x + u * kLdsThreads;
        if (it < items) {
          uint32_t dd[4] = {d[u].x, d[u].y, d[u].z, d[u].w};
          if constexpr (std::is_same<TB, _Float16>::value) {
            const float4 lo = cvt4<TB>(make_uint2(dd[0], dd[1])), hi = cvt4<TB>(make_uint2(dd[2], dd[3]));
            dd[0] = bf16_pair(lo.x, lo.y);
            dd[1] = bf16_pair(lo.z, lo.w);
            dd[2] = bf16_pair(hi.x, hi.y);
            dd[3] = bf16_pair(hi.z, hi.w);
          }
          const int b = it & 7;
          lds_u8* row = lds + (it >> 3) * kLdsRowBytes + 8 * (b >> 1) + 4 * (b & 1);
#pragma unroll
          for (int t = 0; t < 4; ++t)
            *reinterpret_cast<lds_u32*>(row + 32 * t) = half_sel(dd[t >> 1], dd[2 + (t >> 1)], t & 1);
        }
      }
      return;
    }
  }
  // 12 loads of 16 bytes in flight per thread: one round up to K = 768
  // (48 registers; the persistent variants have no room for 64); 8 for the
  // unaligned 16-bit fallback, which shares the kernel with the 16-byte path
  constexpr int U = std::is_same<TB, float>::value ? 12 : 8;
  const int items = ksz * 16;
  for (int base = threadIdx.x; base < items; base += U * kLdsThreads) {
    float4 f[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int it = min(base + u * kLdsThreads, items - 1);
      if constexpr (kAny && std::is_same<TB, float>::value)
        f[u] = N >= 4 ? load4_any(B + (int64_t)(koff + (it >> 4)) * ldb, n0 + 4 * (it & 15), N)
                      : load_b4(B, ldb, koff + (it >> 4), n0 + 4 * (it & 15), N, false);
      else
        f[u] = load_b4(B, ldb, koff + (it >> 4), n0 + 4 * (it & 15), N, vec);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int it = base + u * kLdsThreads;
      if (it < items) {
        lds_u8* pos = lds + (it >> 4) * kLdsRowBytes + 2 * (it & 15);
        const uint32_t p01 = bf16_pair(f[u].x, f[u].y), p23 = bf16_pair(f[u].z, f[u].w);
        *reinterpret_cast<lds_u16*>(pos) = (uint16_t)p01;
        *reinterpret_cast<lds_u16*>(pos + 32) = (uint16_t)(p01 >> 16);
        *reinterpret_cast<lds_u16*>(pos + 64) = (uint16_t)p23;
        *reinterpret_cast<lds_u16*>(pos + 96) = (uint16_t)(p23 >> 16);
      }
    }
  }
}

// Column ids of k-slots (g, e') and (g, e' + 4) (the rows this lane
// addresses in the transposed reads) and the lane's A operand of one chunk
// or, for a scatter chunk (sc, wave-uniform), the 16 bytes of k-slot words
// that hold the lane's one entry.
struct TrChunk {
  int k0, k1;
  bf16x8 a;
  bool sc;
};

__device__ __forceinline__ TrChunk load_tr_chunk(const WindowArrays& p, int c, int cidx, int lane, bool sc) {
  TrChunk r;
  const int32_t* cp = p.tc_cols + (int64_t)c * 32 + cidx;
  r.k0 = cp[0];
  r.k1 = cp[4];
  // scatter chunk: lane (G, row) needs the word of k-slot 8G + row % 8, in
  // 16-byte group 2G + (row % 8) / 4 of the chunk's A block
  const int q = sc ? 2 * (lane >> 4) + ((lane >> 2) & 1) : lane;
  r.a = reinterpret_cast<const bf16x8*>(p.tc_vals)[(int64_t)c * 64 + q];
  r.sc = sc;
  return r;
}

// The MFMA A operand of a scatter chunk for lane (G, row): element row % 8
// holds the value of k-slot 8G + row % 8 when that entry's row is this
// lane's (its word's bit 16 = row >= 8), every other element 0.
__device__ __forceinline__ bf16x8 scatter_operand(const bf16x8& raw, int lane) {
  const uint4 w4 = __builtin_bit_cast(uint4, raw);
  const int s = lane & 3;
  const uint32_t v = s == 0 ? w4.x : s == 1 ? w4.y : s == 2 ? w4.z : w4.w;
  const uint32_t val = ((v >> 16) & 1u) == (uint32_t)((lane >> 3) & 1) ? (v & 0xffffu) : 0u;
  const uint32_t h = (lane & 1) ? val << 16 : val;
  const int word = (lane >> 1) & 3;
  uint4 o;
  o.x = word == 0 ? h : 0u;
  o.y = word == 1 ? h : 0u;
  o.z = word == 2 ? h : 0u;
  o.w = word == 3 ? h : 0u;
  return __builtin_bit_cast(bf16x8, o);
}

// cst = 8q - koff * kLdsRowBytes: the lane's position offset within a row,
// and the unit's first B row
__device__ __forceinline__ void tr_chunk_mfma(lds_u8* lds, int cst, const TrChunk& r, f32x4 (&acc)[4]) {
  const bf16x8 a = r.sc ? scatter_operand(r.a, threadIdx.x & 63) : r.a;
  // 24-bit multiplies (column ids < 2^24): one full-rate v_mad_u32_u24 each
  lds_u8* p0 = lds + (int)(__umul24((unsigned)r.k0, (unsigned)kLdsRowBytes) + (unsigned)cst);
  lds_u8* p1 = lds + (int)(__umul24((unsigned)r.k1, (unsigned)kLdsRowBytes) + (unsigned)cst);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const i16x4 lo = lds_tr_read(p0 + 32 * t);
    const i16x4 hi = lds_tr_read(p1 + 32 * t);
    const i16x8 b = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, b), acc[t], 0, 0, 0);
  }
}

// Rows of the lane group's 4 window slots.
__device__ __forceinline__ SlotRows load_win(const WindowArrays& p, int slot0) { return load_rows(p, slot0); }

// One round of a window's sparse part (kMixed plans): e holds the round's
// entry of slot 4g + (lane & 3) (column, value bits); lane (g, j) adds
// v * B[col][n0 + 4j + t] of the group's four slots to acc[t][i].  BF16 B is
// read from the staged LDS block (position 16t + j of row col - koff), other
// B types from memory (FP32 products on B's exact values either way).
template <typename TB>
__device__ __forceinline__ void sparse_round(const TB* __restrict__ B, int64_t ldb, int N, int col, bool vec,
                                             lds_u8* lds, int koff, int2 e, f32x4 (&acc)[4]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int src = (lane & 48) + i;
    const int k = __shfl(e.x, src);
    const float v = __int_as_float(__shfl(e.y, src));
    float4 b;
    if constexpr (std::is_same<TB, __bf16>::value) {
      lds_u8* rp = lds + (k - koff) * kLdsRowBytes + 2 * (lane & 15);
      b.x = bf16_lo(*reinterpret_cast<lds_u16*>(rp));
      b.y = bf16_lo(*reinterpret_cast<lds_u16*>(rp + 32));
      b.z = bf16_lo(*reinterpret_cast<lds_u16*>(rp + 64));
      b.w = bf16_lo(*reinterpret_cast<lds_u16*>(rp + 96));
    } else {
      b = load_b4(B, ldb, k, col, N, vec);
    }
    acc[0][i] += v * b.x;
    acc[1][i] += v * b.y;
    acc[2][i] += v * b.z;
    acc[3][i] += v * b.w;
  }
}

// One work item (unit item / nC, column chunk item % nC) of the B-stationary
// kernel.  tc_ptr and sp_off are p.tc_ptr and p.sp_off, passed again as
// restrict parameters so that the compiler may read them with scalar loads
// inside the loop that stores C.  Returns early per wave (a wave with no
// windows) or per workgroup (an empty unit); the caller's barrier before the
// next item's staging keeps the LDS block until every wave is done with it.
// kMixed: windows may have sparse parts, added (in rounds, p.sp_ent) to the
// dense sums before the window's rows are stored; a window's first rounds
// (four, two with FP32 or FP16 B) are requested when it starts, later ones
// in batches of as many when it ends.  Scatter chunks (p.tc_kind) build their A operand from
// one k-slot word per lane.
typedef float f32v4_t __attribute__((ext_vector_type(4)));

// The window's rows as float4 stores of four columns each, one per row.
// kStore 1 (C rows 16-byte aligned, N a multiple of 4, C below 2 GiB): buffer
// stores with L2 write-through (sc1) over a descriptor of [C, C + cbytes),
// measured 4 % faster on the block-pruned layer at N = 4096 than
// non-temporal global stores; stores that fall outside C (rows of -1,
// columns at or beyond N) get an offset past the descriptor, which the
// hardware drops, so every lane issues the same stores on every path.
// Otherwise store_window.
// kStore 2 (any alignment and width): the quads that lie inside a row as
// unaligned 16-byte stores, the columns of the one that reaches past N one by
// one, in the items that hold it.
template <int kStore>
__device__ __forceinline__ void store_window_lds(float* __restrict__ C, int64_t ldc, int N, int col, bool vec,
                                                 int cbytes, const SlotRows& sr, const f32x4 (&acc)[4]) {
  if constexpr (kStore > 0) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(C, 0, cbytes, 0x00020000);
    constexpr uint32_t kOut = 0x80000000u;  // past every descriptor (cbytes < 2^31)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool ok = sr.row[i] >= 0 && (kStore == 1 ? col : col + 3) < N;
      const uint32_t off = ok ? ((uint32_t)sr.row[i] * (uint32_t)ldc + (uint32_t)col) * 4u : kOut;
      __builtin_amdgcn_raw_buffer_store_b128(f32v4_t{acc[0][i], acc[1][i], acc[2][i], acc[3][i]}, rs, (int)off, 0,
                                            16);
    }
    if constexpr (kStore == 2) {
      // wave-uniform: the item's 64 columns end past N inside a quad
      const int n0 = col - 4 * (int)(threadIdx.x & 15);
      if ((N & 3) && n0 + 64 > N) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int t = 0; t < 3; ++t) {
            const bool ok = sr.row[i] >= 0 && col + 3 >= N && col + t < N;
            const uint32_t off = ok ? ((uint32_t)sr.row[i] * (uint32_t)ldc + (uint32_t)(col + t)) * 4u : kOut;
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[t][i]), rs, (int)off, 0, 16);
          }
      }
    }
  } else {
    store_window<true>(C, ldc, N, col, vec, sr, acc);
  }
}

template <typename TB, bool kMixed, int kStore, bool kSc>
__device__ __forceinline__ void lds_item(const WindowArrays& p, const int32_t* __restrict__ tc_ptr,
                                         const int32_t* __restrict__ sp_off, const uint32_t* __restrict__ tc_kind,
                                         const int32_t* __restrict__ win_r0, const int4* __restrict__ units,
                                         const TB* __restrict__ B, int64_t ldb, int N, float* __restrict__ C,
                                         int64_t ldc, int nC, bool vec, bool vec16, int cbytes, int item,
                                         lds_u8* lds) {
  constexpr int kWaves = kLdsThreads / 64;
  const int chunk = item % nC;
  const int4 unit = units[item / nC];
  const int n0 = chunk * 64;
  const int koff = unit.z, ksz = unit.w;
  // The wave index is made visibly uniform so that the window and chunk
  // bookkeeping below lives in scalar registers and reads tc_ptr with scalar
  // loads: a vector load of the next window bound inside the loop would make
  // every step wait for all outstanding vector loads and stores.
  const int lane = threadIdx.x & 63, wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, j = lane & 15;
  const int col = n0 + 4 * j;  // the lane's columns: col .. col + 3
  const int cidx = g * 8 + ((lane >> 2) & 3);
  const int cst = 8 * (lane & 3) - koff * kLdsRowBytes;
  const int eidx = 4 * g + (lane & 3);  // slot of the round entry this lane requests
  // This wave's contiguous run of the unit's windows, balanced by chunk count.
  const int wg_beg = unit.x;
  const int wg_end = unit.y;
  if (wg_beg >= wg_end) return;  // the whole workgroup
  const int cb = tc_ptr[wg_beg], ce = tc_ptr[wg_end];
  auto window_at = [&](int target) {  // first window w in [wg_beg, wg_end] with tc_ptr[w] >= target
    int lo = wg_beg, hi = wg_end;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (tc_ptr[mid] < target) lo = mid + 1; else hi = mid;
    }
    return lo;
  };
  const int w_beg = window_at(cb + (int)(((int64_t)(ce - cb) * wib) / kWaves));
  const int w_end = window_at(cb + (int)(((int64_t)(ce - cb) * (wib + 1)) / kWaves));
  const bool has = w_beg < w_end;  // wave-uniform
  const int c_beg = has ? tc_ptr[w_beg] : 0, c_end = has ? tc_ptr[w_end] : 1;

  // The operands of chunk c + 3 are requested while chunk c is multiplied
  // (indices clamped to the wave's last chunk, so every load is
  // unconditional): a wave's loop is bound by the latency of these requests,
  // so three are kept in flight.  Four register sets rotate through a loop
  // unrolled by four, so no set is copied (a copy would wait for the newest
  // load).  Every window of the run holds at least one chunk, so at most one
  // window ends before each chunk.  The first two chunks' operands are
  // requested before the B block is staged, so their latency overlaps the
  // staging, the third one after it (fewer registers live while the staging
  // holds its loads).
  // A window's rows are not carried in registers: for consecutive rows they
  // are computed when the window is stored, from its first row (r0w, a
  // scalar load); other windows load theirs then.  (Rows loaded ahead into
  // registers that the consecutive path overwrites made every window end
  // wait for all loads in flight, the next chunks' operands included.)
  const int last = c_end - 1;
  // chunk kind (scatter or dense): kSc (the plan has scatter chunks, tc_kind
  // set) -- a scalar load of its word of tc_kind; otherwise dense, with no
  // per-chunk bookkeeping (measured 4 % of the block-pruned layer's launch)
  auto is_sc = [&](int idx) { return kSc && ((tc_kind[idx >> 5] >> (idx & 31)) & 1u) != 0; };
  int w = w_beg;
  int w_next = 0;
  int r0w = 0;
  TrChunk r0{}, r1{}, r2{};
  // kMixed: sp_off of the current window and the next, and the lane's
  // entries of the current window's rounds 0 .. kPfRounds - 1, requested when
  // the window starts and used when it ends.  The loads are unconditional
  // (indices clamped to the last entry; a plan with mixed windows has at
  // least one round), so the wait before their use is an exact count.
  constexpr int kPfRounds = std::is_same<TB, __bf16>::value ? 4 : 2;  // FP32 / FP16 B: fewer, for registers
  constexpr int kBatchRounds = std::is_same<TB, __bf16>::value ? 4 : 2;  // later rounds, per request batch
  int so0 = 0, so1 = 0;
  const int sp_last = kMixed ? sp_off[p.W_tc] - 1 : 0;
  int2 ecur[kPfRounds];
  auto request_rounds = [&](int so) {
#pragma unroll
    for (int u = 0; u < kPfRounds; ++u) ecur[u] = p.sp_ent[min(so + 16 * u + eidx, sp_last)];
  };
  if (has) {
    w_next = tc_ptr[w + 1];
    r0w = win_r0[w];
    r0 = load_tr_chunk(p, c_beg, cidx, lane, is_sc(c_beg));
    r1 = load_tr_chunk(p, min(c_beg + 1, last), cidx, lane, is_sc(min(c_beg + 1, last)));
    if constexpr (kMixed) {
      so0 = sp_off[w];
      so1 = sp_off[w + 1];
      request_rounds(so0);
    }
  }
  stage_b<TB, kStore>(lds, B, ldb, koff, ksz, n0, N, vec, vec16);
  if (has) r2 = load_tr_chunk(p, min(c_beg + 2, last), cidx, lane, is_sc(min(c_beg + 2, last)));
  __syncthreads();
  if (!has) return;
  f32x4 acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto finish = [&]() {
    if constexpr (kMixed) {
      const int rounds = (so1 - so0) >> 4;  // wave-uniform
      if (rounds > 0) {
#pragma unroll
        for (int u = 0; u < kPfRounds; ++u)
          if (u < rounds) sparse_round(B, ldb, N, col, vec, lds, koff, ecur[u], acc);
        // rounds beyond those: entries requested a batch at a time, one
        // memory latency per batch
        for (int r = kPfRounds; r < rounds; r += kBatchRounds) {
          int2 e[kBatchRounds];
#pragma unroll
          for (int u = 0; u < kBatchRounds; ++u)
            e[u] = r + u < rounds ? p.sp_ent[so0 + 16 * (r + u) + eidx] : make_int2(koff, 0);
#pragma unroll
          for (int u = 0; u < kBatchRounds; ++u)
            if (r + u < rounds) sparse_round(B, ldb, N, col, vec, lds, koff, e[u], acc);
        }
      }
    }
    SlotRows cur;
    if (r0w >= 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) cur.row[i] = r0w + 4 * g + i;
    } else {
      // The loaded rows are consumed inside this branch (the empty asm reads
      // them), so the wait for the load (and for the loads in flight before
      // it) stays on this path: where the branches join no load is pending
      // on the registers the consecutive path writes.
      cur = load_win(p, w * 16 + g * 4);
      asm volatile("" : "+v"(cur.row[0]), "+v"(cur.row[1]), "+v"(cur.row[2]), "+v"(cur.row[3]));
    }
    store_window_lds<kStore>(C, ldc, N, col, vec, cbytes, cur, acc);
  };
  TrChunk r3;
  int c = c_beg;
  auto step = [&](const TrChunk& use, TrChunk& fill) {
    fill = load_tr_chunk(p, min(c + 3, last), cidx, lane, is_sc(min(c + 3, last)));
    if (c >= w_next) {  // window w is complete: store it
      const int w_next2 = tc_ptr[w + 2];
      const int r0n = win_r0[w + 1];
      int so2 = 0;
      if constexpr (kMixed) so2 = sp_off[w + 2];
      finish();
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      ++w;
      w_next = w_next2;
      r0w = r0n;
      if constexpr (kMixed) {
        so0 = so1;
        so1 = so2;
        request_rounds(so0);
      }
    }
    tr_chunk_mfma(lds, cst, use, acc);
    ++c;
  };
  while (c + 4 <= c_end) {
    step(r0, r3);
    step(r1, r0);
    step(r2, r1);
    step(r3, r2);
  }
  if (c < c_end) step(r0, r3);
  if (c < c_end) step(r1, r0);
  if (c < c_end) step(r2, r1);
  finish();
}

// units: the work-unit list of this launch.  kLoop = false: one workgroup
// per item (grid = items <= compute units); true: persistent workgroups that
// restage the LDS block for each item they take: items blockIdx.x,
// blockIdx.x + gridDim.x, ... or, with xcd (grid a multiple of kXcds), items
// xr.start[x] + blockIdx.x / kXcds, + gridDim.x / kXcds, ... below
// xr.start[x + 1] for x = blockIdx.x % kXcds.  Two instantiations because
// the loop costs the one-item launches about 0.6 us (more registers live
// across the item body).
//
// Tail: the last tail_blocks workgroups of the grid then run the sparse-only
// rows' tasks (one wave per (row, 64 columns), as hyb_spmm_sparse_split_kernel)
// in place of a second launch: block gridDim.x - 1 - i takes tasks 16i ..
// 16i + 15 of tail_tasks.  Under the XCD grouping those are the last slot of
// each XCD, which holds the fewest items when a range does not divide evenly;
// one-item launches add tail blocks past the items when CUs are free.
template <bool kLoop, typename TB, bool kMixed, int kStore>
__global__ __launch_bounds__(kLdsThreads) void hyb_spmm_lds_bf16_kernel(WindowArrays p,
                                                                        const int32_t* __restrict__ tc_ptr,
                                                                        const int32_t* __restrict__ sp_off,
                                                                        const uint32_t* __restrict__ tc_kind,
                                                                        const int32_t* __restrict__ win_r0,
                                                                        const int4* __restrict__ units,
                                                                        const TB* __restrict__ B,
                                                                        int64_t ldb, int N, float* __restrict__ C,
                                                                        int64_t ldc, int nC, int n_items, bool vec,
                                                                        bool vec16, int cbytes, LdsXcdRanges xr,
                                                                        bool xcd, int tail_blocks, int tail_tasks) {
  extern __shared__ uint4 lds_dyn[];  // [ksz][kLdsRowBytes]
  lds_u8* lds = (lds_u8*)lds_dyn;
  const int tb = (int)gridDim.x - 1 - (int)blockIdx.x;
  auto run = [&](int item) {  // tc_kind: kernel-uniform
    if (tc_kind)
      lds_item<TB, kMixed, kStore, true>(p, tc_ptr, sp_off, tc_kind, win_r0, units, B, ldb, N, C, ldc, nC, vec, vec16,
                                       cbytes, item, lds);
    else
      lds_item<TB, kMixed, kStore, false>(p, tc_ptr, sp_off, tc_kind, win_r0, units, B, ldb, N, C, ldc, nC, vec,
                                        vec16, cbytes, item, lds);
  };
  if (!kLoop) {
    if ((int)blockIdx.x < n_items) run(blockIdx.x);
    if (tb < tail_blocks) {
      const int task = tb * (kLdsThreads / 64) + (int)(threadIdx.x >> 6);
      if (task < tail_tasks) with_vec(vec, [&](auto V) { sparse_split_wave(p, B, ldb, N, C, ldc, nC, V, task); });
    }
    return;
  }
  int beg = blockIdx.x, end = n_items, step = gridDim.x;
  if (xcd) {
    const int x = blockIdx.x % kXcds;
    int r0 = 0, r1 = 0;
#pragma unroll
    for (int i = 0; i < kXcds; ++i)  // selects, not a dynamically indexed copy
      if (i == x) {
        r0 = xr.start[i];
        r1 = xr.start[i + 1];
      }
    beg = r0 + (int)(blockIdx.x / kXcds);
    end = r1;
    step = gridDim.x / kXcds;
  }
  for (int item = beg; item < end; item += step) {
    __syncthreads();  // every wave is done reading the previous item's block
    run(item);
  }
  if (tb < tail_blocks) {
    const int task = tb * (kLdsThreads / 64) + (int)(threadIdx.x >> 6);
    if (task < tail_tasks) with_vec(vec, [&](auto V) { sparse_split_wave(p, B, ldb, N, C, ldc, nC, V, task); });
  }
}

template <bool kLoop, typename TB>
static void set_lds_bytes(int bytes) {
  for (const void* f : {reinterpret_cast<const void*>(hyb_spmm_lds_bf16_kernel<kLoop, TB, false, 0>),
                        reinterpret_cast<const void*>(hyb_spmm_lds_bf16_kernel<kLoop, TB, true, 0>),
                        reinterpret_cast<const void*>(hyb_spmm_lds_bf16_kernel<kLoop, TB, false, 1>),
                        reinterpret_cast<const void*>(hyb_spmm_lds_bf16_kernel<kLoop, TB, true, 1>),
                        reinterpret_cast<const void*>(hyb_spmm_lds_bf16_kernel<kLoop, TB, false, 2>),
                        reinterpret_cast<const void*>(hyb_spmm_lds_bf16_kernel<kLoop, TB, true, 2>)})
    (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

void prepare_spmm_kernels(const SpmmPlanDev& p) {
  const int bytes = p.lds_max_k * kLdsRowBytes;
  if (!p.lds_units || bytes <= 65536) return;
  set_lds_bytes<false, float>(bytes);
  set_lds_bytes<true, float>(bytes);
  set_lds_bytes<false, __bf16>(bytes);
  set_lds_bytes<true, __bf16>(bytes);
  set_lds_bytes<false, _Float16>(bytes);
  set_lds_bytes<true, _Float16>(bytes);
}

int device_cus() {
  // per-device cache; threads that race on the first query store the same value
  static std::atomic<int> cus[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cus[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

int64_t spmm_workspace_floats(const SpmmPlanDev& p, int N) {
  return ((int64_t)p.npieces + (int64_t)p.n_parts * 16) * N;
}

template <typename TB>
static hipError_t launch_hyb_spmm_t(const SpmmPlanDev& p, const TB* B, int64_t ldb, int N, float* C, int64_t ldc,
                                    bool det, float* ws, hipStream_t s) {
  const int eb = (int)sizeof(TB);
  const bool vec = (N % 4 == 0) && (ldb % 4 == 0) && (ldc % 4 == 0) &&
                   ((reinterpret_cast<uintptr_t>(B) & (4 * eb - 1)) == 0) &&
                   ((reinterpret_cast<uintptr_t>(C) & 15) == 0);
  const bool vec16 = eb == 2 && vec && N % 8 == 0 && ldb % 8 == 0 && ((reinterpret_cast<uintptr_t>(B) & 15) == 0);
  const int nC = (N + 63) / 64;
  // workspace regions of the deterministic mode: pieces, then huge-window parts
  float* ws_pieces = det ? ws : nullptr;
  float* ws_parts = det ? ws + (int64_t)p.npieces * N : nullptr;
  // B-stationary kernel for every BF16 plan whose matrices all have K <=
  // kLdsMaxK (measured on the block-pruned layer: 9.0 us vs 15.0 us
  // streaming at N = 128, 20.8 vs 82 us at N = 4096); otherwise the
  // streaming kernel.  Unit list: the plan's pick for nC column chunks (up to
  // kLdsPickMax), else the smallest list with at least one item per CU.
  // (launch options of the plan: opt_kernel 1 = streaming kernel, refused
  // at plan level for plans with scatter chunks; opt_lds_list >= 0 = that
  // unit list; opt_lds_xcd 0 = items round-robin instead of per-XCD ranges)
  bool lds = p.lds_units != nullptr && p.W_tc > 0;
  if (p.opt_kernel == 1 && !p.tc_kind) lds = false;
  // Sparse-only rows: with the LDS kernel and at most kLdsTailMaxTasks
  // (row, 64 columns) tasks they are the LDS launch's tail; otherwise a
  // launch of their own follows the dense kernels.
  const int64_t so_rows = (int64_t)(p.W - p.W_tc) * 16;
  const int cus = device_cus();
  const bool fold = lds && so_rows > 0 && so_rows * nC <= kLdsTailMaxTasks &&
                    (so_rows * nC + kLdsThreads / 64 - 1) / (kLdsThreads / 64) <= cus / kXcds * kXcds;
  // The LDS kernel runs every dense window with its sparse part; otherwise a
  // streaming kernel does the dense parts and, when the sparse parts are short
  // and the launch small, those too (folded); else the row tasks add them.
  bool folded = true;
  if (lds) {
    int t = p.opt_lds_list >= 0 && p.opt_lds_list < kLdsLists ? p.opt_lds_list : -1;
    if (t < 0 && nC <= kLdsPickMax) t = p.lds_pick[nC];
    if (t < 0) {
      t = 0;
      while (t + 1 < kLdsLists && (int64_t)p.lds_cnt[t] * nC < cus) ++t;
    }
    const int64_t items = (int64_t)p.lds_cnt[t] * nC;
    if (items > INT32_MAX) return hipErrorInvalidValue;
    // one workgroup per CU at most (each holds a staged block of LDS)
    int grid = (int)std::min<int64_t>(items, cus);
    LdsXcdRanges xr{};
    const bool xcd = items > cus && nC <= kLdsXcdMaxNC && cus >= kXcds && p.lds_xcd_host && p.opt_lds_xcd != 0;
    if (xcd) {
      const int32_t* st = p.lds_xcd_host + ((size_t)t * (kLdsXcdMaxNC + 1) + nC) * (kXcds + 1);
      if (st[0] != 0 || st[kXcds] != items) return hipErrorInvalidValue;  // ranges cover every item once
      for (int x = 0; x < kXcds; ++x)
        if (st[x + 1] < st[x]) return hipErrorInvalidValue;
      std::copy(st, st + kXcds + 1, xr.start);
      grid = cus / kXcds * kXcds;
    }
    const int tail_tasks = fold ? (int)(so_rows * nC) : 0;
    const int tail_blocks = (tail_tasks + kLdsThreads / 64 - 1) / (kLdsThreads / 64);
    // one-item launches: tail blocks of their own past the items while CUs
    // are free, else the last item blocks take the tail
    if (items <= cus && items + tail_blocks <= cus) grid = (int)items + tail_blocks;
    if (items <= cus) grid = std::max(grid, tail_blocks);
    const size_t lds_bytes = (size_t)p.lds_max_k * kLdsRowBytes;
    const int4* units = p.lds_units + p.lds_off[t];
    const bool mixed = p.n_mix > 0 && p.sp_off != nullptr;
    // C addressed by a buffer descriptor (kStore 1, 2) when its extent is below
    // 2 GiB
    const int64_t c_extent = ((int64_t)(p.M - 1) * ldc + N) * 4;
    const int cbytes = p.M > 0 && c_extent < ((int64_t)1 << 31) ? (int)c_extent : 0;
#define STILE_LDS_LAUNCH1(LOOP, MIX, VEC)                                                                    \
  hipLaunchKernelGGL((hyb_spmm_lds_bf16_kernel<LOOP, TB, MIX, VEC>), dim3(grid), dim3(kLdsThreads), lds_bytes, s, \
                     window_arrays(p),                                                                         \
                     p.tc_ptr, p.sp_off, p.tc_kind, p.win_r0, units, B, ldb, N, C, ldc, nC, (int)items, vec, vec16, \
                     cbytes, xr, LOOP && xcd, tail_blocks, tail_tasks)
#define STILE_LDS_LAUNCH(LOOP, MIX)                \
  do {                                             \
    if (vec && cbytes > 0)                         \
      STILE_LDS_LAUNCH1(LOOP, MIX, 1);             \
    else if (cbytes > 0)                           \
      STILE_LDS_LAUNCH1(LOOP, MIX, 2);             \
    else                                           \
      STILE_LDS_LAUNCH1(LOOP, MIX, 0);             \
  } while (0)
    if (items <= cus) {
      if (mixed) STILE_LDS_LAUNCH(false, true); else STILE_LDS_LAUNCH(false, false);
    } else {
      if (mixed) STILE_LDS_LAUNCH(true, true); else STILE_LDS_LAUNCH(true, false);
    }
#undef STILE_LDS_LAUNCH
#undef STILE_LDS_LAUNCH1
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  } else if (p.W_tc > 0) {
    hipError_t e = launch_stream(p, B, ldb, N, C, ldc, vec, ws_parts, s, &folded);
    if (e != hipSuccess) return e;
  }
  // Sparse-only rows (unless they were the LDS launch's tail) by wave tasks, or,
  // when there are fewer than 16,384 (row, 64 columns) of 8 or more nonzeros on
  // average, one of those per wave with all its gathers in flight at once, or one
  // row per lane group when they are even.  The sparse parts of dense windows come
  // first in the task list, when neither the LDS nor the streaming kernel added them.
  const int64_t so_left = fold ? 0 : so_rows;
  const bool split = so_left > 0 && so_left * nC / 4 < 4096 && p.nnz_sparse_only >= 8 * so_left;
  if (split) {
    const int64_t blocks = (so_rows * nC + 3) / 4;
    hipLaunchKernelGGL(hyb_spmm_sparse_split_kernel<TB>, dim3((unsigned)blocks), dim3(256), 0, s,
                       window_arrays(p), B, ldb, N, C, ldc, nC, vec);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  bool even = false;
  if constexpr (std::is_same<TB, float>::value) {
    even = so_left > 0 && !split && even_rows_fit(p, N, vec);
    if (even) {
      hipError_t e = launch_even_rows(p, B, ldb, N, C, ldc, s);
      if (e != hipSuccess) return e;
    }
  }
  {
    hipError_t e = launch_sparse_rows(p, B, ldb, N, C, ldc, vec, folded ? p.n_mix_tasks : 0,
                                      so_left > 0 && !split && !even ? p.n_row_tasks : p.n_mix_tasks, s);
    if (e != hipSuccess) return e;
  }
  // Pieces of long rows.  The LDS kernel summed its windows' rows whole, so
  // only the sparse-only rows' pieces remain after it.
  const int pc0 = lds ? p.npieces_dense : 0;
  if (p.npieces > pc0) {
    hipError_t e = launch_sparse_pieces(p, B, ldb, N, C, ldc, vec, pc0, p.npieces, ws_pieces, s);
    if (e != hipSuccess) return e;
    if (det) {
      e = launch_piece_reduce(p, N, C, ldc, vec, lds ? p.nsrows_dense : 0, ws_pieces, s);
      if (e != hipSuccess) return e;
    }
  }
  return hipSuccess;
}

hipError_t launch_hyb_spmm(const SpmmPlanDev& p, int b_dtype, const void* B, int64_t ldb, int N, float* C,
                           int64_t ldc, bool deterministic, float* ws, hipStream_t s) {
  if (p.W == 0 || N == 0) return hipSuccess;
  switch (b_dtype) {
    case 1:
      return launch_hyb_spmm_t(p, static_cast<const __bf16*>(B), ldb, N, C, ldc, deterministic, ws, s);
    case 2:
      return launch_hyb_spmm_t(p, static_cast<const _Float16*>(B), ldb, N, C, ldc, deterministic, ws, s);
    default:
      return launch_hyb_spmm_t(p, static_cast<const float*>(B), ldb, N, C, ldc, deterministic, ws, s);
  }
}

// ---------------------------------------------------------------------------
// Row softmax over CSR rows: one wave per row; max and sum reduced with xor
// shuffles across the 64 lanes.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void row_softmax_kernel(int M, const int32_t* __restrict__ indptr,
                                                          const float* in, float* out, float scale) {
  const int row = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  if (row >= M) return;
  const int lane = threadIdx.x & 63;
  const int p0 = indptr[row], p1 = indptr[row + 1];
  if (p0 >= p1) return;
  float m = -INFINITY;
  for (int p = p0 + lane; p < p1; p += 64) m = fmaxf(m, scale * in[p]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  float s = 0.f;
  for (int p = p0 + lane; p < p1; p += 64) s += __expf(scale * in[p] - m);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
  const float inv = 1.f / s;
  for (int p = p0 + lane; p < p1; p += 64) out[p] = __expf(scale * in[p] - m) * inv;
}

hipError_t launch_row_softmax(int M, const int32_t* indptr, const float* in, float* out, float scale,
                              hipStream_t s) {
  if (M == 0) return hipSuccess;
  const int64_t waves = M;
  hipLaunchKernelGGL(row_softmax_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, M, indptr, in, out,
                     scale);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// ELL-bucket SpMM (the SparseTIR hyb comparator): every ELL row of a bucket
// holds `width` (column, value) slots; C[row] += sum over slots v * B[col].
// One 16-lane group per ELL row and 64 columns; rows of C appear in several
// buckets (column parts, split long rows), so results are added with
// atomicAdd into a zero-filled C.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void ell_bucket_spmm_kernel(int rows, int width, const int32_t* __restrict__ orow,
                                                              const int32_t* __restrict__ cols,
                                                              const float* __restrict__ vals,
                                                              const float* __restrict__ B, int64_t ldb, int N,
                                                              float* __restrict__ C, int64_t ldc, int nC,
                                                              bool vec) {
  const int lane = threadIdx.x & 63;
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t item = wave * 4 + (lane >> 4);
  if (item >= (int64_t)rows * nC) return;
  const int r = (int)(item / nC);
  const int col = (int)(item - (int64_t)r * nC) * 64 + 4 * (lane & 15);
  if (col >= N) return;
  const int32_t* cr = cols + (int64_t)r * width;
  const float* vr = vals + (int64_t)r * width;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  int k = 0;
  for (; k + 4 <= width; k += 4) {
    const int k0 = cr[k], k1 = cr[k + 1], k2 = cr[k + 2], k3 = cr[k + 3];
    const float v0 = vr[k], v1 = vr[k + 1], v2 = vr[k + 2], v3 = vr[k + 3];
    const float4 b0 = load_b4(B, ldb, k0, col, N, vec), b1 = load_b4(B, ldb, k1, col, N, vec);
    const float4 b2 = load_b4(B, ldb, k2, col, N, vec), b3 = load_b4(B, ldb, k3, col, N, vec);
    s.x += v0 * b0.x + v1 * b1.x + v2 * b2.x + v3 * b3.x;
    s.y += v0 * b0.y + v1 * b1.y + v2 * b2.y + v3 * b3.y;
    s.z += v0 * b0.z + v1 * b1.z + v2 * b2.z + v3 * b3.z;
    s.w += v0 * b0.w + v1 * b1.w + v2 * b2.w + v3 * b3.w;
  }
  for (; k < width; ++k) {
    const float v = vr[k];
    const float4 b = load_b4(B, ldb, cr[k], col, N, vec);
    s.x += v * b.x; s.y += v * b.y; s.z += v * b.z; s.w += v * b.w;
  }
  float* c = C + (int64_t)orow[r] * ldc + col;
  atomicAdd(c, s.x);
  if (col + 1 < N) atomicAdd(c + 1, s.y);
  if (col + 2 < N) atomicAdd(c + 2, s.z);
  if (col + 3 < N) atomicAdd(c + 3, s.w);
}

hipError_t launch_ell_bucket_spmm(int rows, int width, const int32_t* orow, const int32_t* cols, const float* vals,
                                  const float* B, int64_t ldb, int N, float* C, int64_t ldc, hipStream_t s) {
  if (rows == 0 || N == 0) return hipSuccess;
  const bool vec = (N % 4 == 0) && (ldb % 4 == 0) && ((reinterpret_cast<uintptr_t>(B) & 15) == 0);
  const int nC = (N + 63) / 64;
  const int64_t items = (int64_t)rows * nC;
  const int64_t blocks = (items + 15) / 16;
  if (blocks > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL(ell_bucket_spmm_kernel, dim3((unsigned)blocks), dim3(256), 0, s, rows, width, orow, cols, vals,
                     B, ldb, N, C, ldc, nC, vec);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Value refresh.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void set_values_kernel(const float* __restrict__ vals,
                                                         const int32_t* __restrict__ tc_ids, int64_t n_tc,
                                                         void* tc_vals, int mode,
                                                         const int32_t* __restrict__ res_ids, int64_t n_res,
                                                         float* res_vals, const int32_t* __restrict__ sp_ids,
                                                         int64_t n_sp, int2* sp_ent) {
  const int64_t n = n_tc + n_res + n_sp;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    if (i < n_tc) {
      const int id = tc_ids[i];
      if (id == kKeepId) continue;
      const float v = id >= 0 ? vals[id] : 0.f;
      if (mode == 1)
        reinterpret_cast<__bf16*>(tc_vals)[i] = (__bf16)v;
      else
        reinterpret_cast<float*>(tc_vals)[i] = v;
    } else if (i < n_tc + n_res) {
      const int64_t j = i - n_tc;
      res_vals[j] = vals[res_ids[j]];
    } else {
      // the value half of a round entry; padding entries (id -1) stay 0
      const int64_t j = i - n_tc - n_res;
      const int id = sp_ids[j];
      reinterpret_cast<float*>(sp_ent)[2 * j + 1] = id >= 0 ? vals[id] : 0.f;
    }
  }
}

hipError_t launch_set_values(const SpmmPlanDev& p, const float* vals, const int32_t* tc_ids, int64_t n_tc,
                             const int32_t* res_ids, int64_t n_res, const int32_t* sp_ids, int64_t n_sp,
                             hipStream_t s) {
  const int64_t n = n_tc + n_res + n_sp;
  if (n == 0) return hipSuccess;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(set_values_kernel, dim3((unsigned)blocks), dim3(256), 0, s, vals, tc_ids, n_tc,
                     const_cast<void*>(p.tc_vals), p.blk_dtype, res_ids, n_res, const_cast<float*>(p.res_vals),
                     sp_ids, n_sp, const_cast<int2*>(p.sp_ent));
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Zero fill.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void fill_zero_2d_kernel(float* __restrict__ p, int rows, int cols,
                                                           int64_t ld) {
  const int64_t n = (int64_t)rows * cols;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / cols, c = i - r * cols;
    p[r * ld + c] = 0.f;
  }
}

// C rows of windows [0, nwin) set to zero (the huge windows' rows, before
// their parts add into them).  One block per row slot.
__global__ __launch_bounds__(256) void zero_window_rows_kernel(const int32_t* __restrict__ win_rows, float* C,
                                                               int64_t ldc, int N) {
  const int row = win_rows[blockIdx.x];
  if (row < 0) return;
  float* c = C + (int64_t)row * ldc;
  for (int i = threadIdx.x; i < N; i += blockDim.x) c[i] = 0.f;
}

hipError_t launch_zero_window_rows(const SpmmPlanDev& p, int nwin, float* C, int64_t ldc, int N, hipStream_t s) {
  if (nwin == 0 || N == 0) return hipSuccess;
  hipLaunchKernelGGL(zero_window_rows_kernel, dim3((unsigned)(nwin * 16)), dim3(256), 0, s, p.win_rows, C, ldc, N);
  return hipGetLastError();
}

hipError_t launch_fill_zero_2d(float* p, int rows, int cols, int64_t ld, hipStream_t s) {
  const int64_t n = (int64_t)rows * cols;
  if (n == 0) return hipSuccess;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(fill_zero_2d_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p, rows, cols, ld);
  return hipGetLastError();
}

hipError_t launch_fill_zero(float* p, int64_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  if (n <= INT32_MAX) return launch_fill_zero_2d(p, 1, (int)n, n, s);
  return hipErrorInvalidValue;
}

}  // namespace stile
