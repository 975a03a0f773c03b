// Tall FP32 products H^T G (the weight gradient of a tall dense layer) for
// MI355X (gfx950).
#include "stile_device.h"

#include <algorithm>

namespace stile {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// ---------------------------------------------------------------------------
// out[f][g] = sum over m of H[m][f] G[m][g], M >> F, Fg.
//
// One workgroup = (128 x 64 tile of out, slab of rows).  The operands of
// v_mfma_f32_32x32x2_f32 are rows of H and G as they lie in memory: lane l holds
// for k-slot l / 32 (row m + l / 32) one column per tile, so a row pair is one
// four-column load of H and one two-column load of G (kVec: tile t holds columns
// 4j + t and 2j + t of the tile; else 32t + j, one-column loads of any
// alignment), with the row offset in a scalar register and no arithmetic on
// addresses.  Eight MFMAs of 64 cycles follow each pair.  The slab's row pairs go
// round the four waves; their sums meet in LDS and the tile goes to
// ws[slab][F][Fg], summed over the slabs in order by tall_sum_kernel.
//
// Bound: the FP32 matrix rate (154 TFLOP/s measured on an 8192^3 product, 28 us
// for M = 32768, F = Fg = 256).  That product takes 50 us and the sum over 64
// slabs 6 us; the vendor's GEMM has 57 workgroups there and took 138 us.
// ---------------------------------------------------------------------------
constexpr int kTallF = 128, kTallG = 64;
constexpr int kTallDepth = 4;  // row pairs per wave requested together

template <bool kVec>
struct TallRows {
  float a[4], b[2];
};

template <bool kVec>
__global__ __launch_bounds__(256, 2) void tall_tn_kernel(const float* __restrict__ H, uint32_t hbytes, uint32_t ldh,
                                                         const float* __restrict__ G, uint32_t gbytes, uint32_t ldg,
                                                         int M, int F, int Fg, int tiles_g, int slab,
                                                         float* __restrict__ ws) {
  __shared__ float red[2 * 128 * 64];  // two waves' accumulators, [slot][register][lane]
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 31, h = lane >> 5;
  const int f0 = (int)(blockIdx.x / tiles_g) * kTallF, g0 = (int)(blockIdx.x % tiles_g) * kTallG;
  const __amdgpu_buffer_rsrc_t hr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(H), 0, hbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(G), 0, gbytes, 0x00020000);
  // Columns past F or Fg read what follows in memory: they only reach entries of
  // the tile that are never stored.  Rows past the slab are not read (below).
  const uint32_t ho = (h * ldh + f0 + (kVec ? 4 * j : j)) * 4u, go = (h * ldg + g0 + (kVec ? 2 * j : j)) * 4u;
  auto load = [&](int m, TallRows<kVec>& r) {
    const uint32_t hs = (uint32_t)m * ldh * 4u, gs = (uint32_t)m * ldg * 4u;
    if constexpr (kVec) {
      const f32x4 a = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(hr, ho, hs, 0));
      const auto b = __builtin_amdgcn_raw_buffer_load_b64(gr, go, gs, 0);
#pragma unroll
      for (int t = 0; t < 4; ++t) r.a[t] = a[t];
      r.b[0] = __uint_as_float(b[0]);
      r.b[1] = __uint_as_float(b[1]);
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        r.a[t] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(hr, ho + 128 * t, hs, 0));
#pragma unroll
      for (int t = 0; t < 2; ++t)
        r.b[t] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(gr, go + 128 * t, gs, 0));
    }
  };
  f32x16 acc[4][2];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][u][i] = 0.f;
  auto mul = [&](const TallRows<kVec>& r) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(r.a[t], r.b[u], acc[t][u], 0, 0, 0);
  };
  const int m0 = (int)blockIdx.y * slab, m1 = min(m0 + slab, M);
  const int pairs = (m1 - m0) >> 1;                    // whole row pairs of the slab
  const int mine = max((pairs - wv + 3) >> 2, 0);      // this wave's: wv, wv + 4, ...
  const int groups = mine / kTallDepth;                // full groups of kTallDepth pairs
  auto row = [&](int i) { return m0 + 2 * (wv + 4 * i); };
  TallRows<kVec> r0[kTallDepth], r1[kTallDepth];
  auto load_group = [&](int g, TallRows<kVec>(&r)[kTallDepth]) {
#pragma unroll
    for (int d = 0; d < kTallDepth; ++d) load(row(g * kTallDepth + d), r[d]);
  };
  auto mul_group = [&](const TallRows<kVec>(&r)[kTallDepth]) {
#pragma unroll
    for (int d = 0; d < kTallDepth; ++d) mul(r[d]);
  };
  // the next group's rows are requested before the current group is multiplied
  // (two register sets; the last request repeats the last group)
  if (groups > 0) {
    load_group(0, r0);
    int g = 0;
    while (g + 2 <= groups) {
      load_group(g + 1, r1);
      mul_group(r0);
      load_group(min(g + 2, groups - 1), r0);
      mul_group(r1);
      g += 2;
    }
    if (g < groups) mul_group(r0);
  }
  for (int i = groups * kTallDepth; i < mine; ++i) {
    load(row(i), r0[0]);
    mul(r0[0]);
  }
  // an odd last row: k-slot 1 is 0
  if (((m1 - m0) & 1) && wv == 0) {
    load(m1 - 1, r0[0]);
#pragma unroll
    for (int t = 0; t < 4; ++t) r0[0].a[t] = h == 0 ? r0[0].a[t] : 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t) r0[0].b[t] = h == 0 ? r0[0].b[t] : 0.f;
    mul(r0[0]);
  }
  // sums of the four waves: (0 + 2) + (1 + 3)
  auto at = [&](int slot, int k) -> float& { return red[(slot * 128 + k) * 64 + lane]; };
  if (wv >= 2)
#pragma unroll
    for (int k = 0; k < 128; ++k) at(wv - 2, k) = acc[k >> 5][(k >> 4) & 1][k & 15];
  __syncthreads();
  if (wv < 2)
#pragma unroll
    for (int k = 0; k < 128; ++k) acc[k >> 5][(k >> 4) & 1][k & 15] += at(wv, k);
  __syncthreads();
  if (wv == 1)
#pragma unroll
    for (int k = 0; k < 128; ++k) at(0, k) = acc[k >> 5][(k >> 4) & 1][k & 15];
  __syncthreads();
  if (wv != 0) return;
  float* part = ws + (int64_t)blockIdx.y * F * Fg;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = 8 * (i >> 2) + 4 * h + (i & 3);  // row of the 32 x 32 tile
      const int f = f0 + (kVec ? 4 * r + t : 32 * t + r);
      if (f >= F) continue;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int g = g0 + (kVec ? 2 * j + u : 32 * u + j);
        if (g < Fg) part[(int64_t)f * Fg + g] = acc[t][u][i] + at(0, (t * 2 + u) * 16 + i);
      }
    }
}

// out[f][g] = sum of ws[s][f][g] over the slabs in order, eight requested together.
__global__ __launch_bounds__(256) void tall_sum_kernel(const float* __restrict__ ws, int slabs, int F, int Fg,
                                                       float* __restrict__ out, int64_t ldo) {
  const int64_t n = (int64_t)F * Fg;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
  for (int q = 0; q < slabs; q += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = ws[(int64_t)min(q + u, slabs - 1) * n + i];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += q + u < slabs ? v[u] : 0.f;
  }
  out[i / Fg * ldo + i % Fg] = s;
}

// Slabs: two workgroups per CU, rows of a slab a multiple of 32 (each wave then
// has whole groups of row pairs) and at least 128.
int tall_slabs(int M, int F, int Fg, int* slab) {
  const int64_t tiles = (int64_t)((F + kTallF - 1) / kTallF) * ((Fg + kTallG - 1) / kTallG);
  const int64_t want = std::max<int64_t>(1, (2 * (int64_t)device_cus() + tiles - 1) / tiles);
  int64_t rows = ((int64_t)M + want - 1) / want;
  rows = std::max<int64_t>(128, (rows + 31) / 32 * 32);
  *slab = (int)std::min<int64_t>(rows, INT32_MAX / 2);
  return (int)(((int64_t)M + *slab - 1) / *slab);
}

hipError_t launch_tall_tn(int M, int F, int Fg, const float* H, int64_t ldh, const float* G, int64_t ldg, float* out,
                          int64_t ldo, float* ws, hipStream_t s) {
  int slab = 0;
  const int slabs = tall_slabs(M, F, Fg, &slab);
  const int tiles_f = (F + kTallF - 1) / kTallF, tiles_g = (Fg + kTallG - 1) / kTallG;
  const uint32_t hb = (uint32_t)(((int64_t)(M - 1) * ldh + F) * 4), gb = (uint32_t)(((int64_t)(M - 1) * ldg + Fg) * 4);
  const bool vec = F % 4 == 0 && Fg % 2 == 0 && ldh % 4 == 0 && ldg % 2 == 0 &&
                   (reinterpret_cast<uintptr_t>(H) & 15) == 0 && (reinterpret_cast<uintptr_t>(G) & 7) == 0;
  const dim3 grid((unsigned)(tiles_f * tiles_g), (unsigned)slabs);
  if (vec)
    hipLaunchKernelGGL(tall_tn_kernel<true>, grid, dim3(256), 0, s, H, hb, (uint32_t)ldh, G, gb, (uint32_t)ldg, M, F,
                       Fg, tiles_g, slab, ws);
  else
    hipLaunchKernelGGL(tall_tn_kernel<false>, grid, dim3(256), 0, s, H, hb, (uint32_t)ldh, G, gb, (uint32_t)ldg, M, F,
                       Fg, tiles_g, slab, ws);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t n = (int64_t)F * Fg;
  hipLaunchKernelGGL(tall_sum_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, ws, slabs, F, Fg, out, ldo);
  return hipGetLastError();
}

}  // namespace stile
