// Hybrid fused SDDMM of libstile_hip.so for MI355X (gfx950).
#include "stile_device.h"

namespace stile {

// ---------------------------------------------------------------------------
// Hybrid fused SDDMM.  Workgroups [0, blocks1d) run the 1D entries (segments of
// LPE lanes, kSddmmU consecutive entries each), the others dense 16x16 blocks:
// lane l = 16g + j loads quads of X[rows[j]] and Y[cols[j]] at features kb + 4g
// .. kb + 4g + 3 and feeds component e to MFMA e (v_mfma_f32_16x16x4_f32, so
// k-slot g of MFMA e is feature kb + 4g + e).  The 16x16 result goes through LDS
// to the sampled scatter.
// ---------------------------------------------------------------------------
constexpr int kSddmmU = 4;
// With more features than this the four waves of a workgroup share a dense block:
// one wave waits for Kf / 64 steps of loads in sequence (R-MAT scale 15, K = 163:
// 44.7 us, shared 34.4).  The line is not where sharing stops to pay (K = 64 13.4 us
// alone, 12.0 shared; 128 21.9 and 19.9): up to 128 features, attention heads, the
// sum stays one wave's in the order of the features, so that scores a softmax rounds
// to BF16 do not move.
constexpr int kSharedKf = 128;

// Sum over aligned segments of LPE <= 16 lanes, left in every lane: lanes 8, 4, 2
// and 1 apart are added in that order (scores that a softmax rounds to BF16
// later change visibly with the order).  The exchanges are DPP moves; a shuffle
// through LDS is four latencies in a row at the end of every entry.
template <int LPE>
__device__ __forceinline__ float segment_sum(float x) {
  auto dpp = [](float old, float v, auto ctrl, auto banks) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), decltype(ctrl)::value,
                                                      0xf, decltype(banks)::value, true));
  };
  typedef std::integral_constant<int, 0xf> all;
  if constexpr (LPE >= 16) {
    x += dpp(x, x, std::integral_constant<int, 0x128>{}, all{});  // row_ror:8
    x += dpp(x, x, std::integral_constant<int, 0x124>{}, all{});  // row_ror:4 (lanes 8 apart agree by now)
  } else if constexpr (LPE >= 8) {
    // row_shl:4 into the even quads, row_shr:4 into the odd ones
    float y = dpp(x, x, std::integral_constant<int, 0x104>{}, std::integral_constant<int, 0x5>{});
    y = dpp(y, x, std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xa>{});
    x += y;
  }
  if constexpr (LPE >= 4) x += dpp(x, x, std::integral_constant<int, 0x4E>{}, all{});  // quad_perm 2,3,0,1
  if constexpr (LPE >= 2) x += dpp(x, x, std::integral_constant<int, 0xB1>{}, all{});  // quad_perm 1,0,3,2
  return x;
}

// A row-major operand read by feature quads.  kSmall (it spans less than 4 GiB,
// rows and row bytes below 2^24): a 32-bit offset from the scalar base, one 24-bit
// product per row.
template <bool kSmall>
struct FeatureRows {
  const float* p;
  int64_t ld;
  typedef typename std::conditional<kSmall, uint32_t, const float*>::type Row;
  __device__ __forceinline__ Row row(int r) const {
    if constexpr (kSmall)
      return __umul24((unsigned)r, (unsigned)ld * 4u);
    else
      return p + (int64_t)r * ld;
  }
  __device__ __forceinline__ float4 quad(Row r, int k) const {  // features k .. k + 3, aligned
    if constexpr (kSmall)
      return *reinterpret_cast<const float4*>(reinterpret_cast<const unsigned char*>(p) + (uint32_t)(r + 4u * (unsigned)k));
    else
      return ld4(r + k);
  }
  __device__ __forceinline__ float one(Row r, int k) const {
    if constexpr (kSmall)
      return *reinterpret_cast<const float*>(reinterpret_cast<const unsigned char*>(p) + (uint32_t)(r + 4u * (unsigned)k));
    else
      return r[k];
  }
  // features k + S i, i = 0..3, zero at or beyond Kf
  template <int S>
  __device__ __forceinline__ float4 strided(Row r, int k, int Kf) const {
    float4 v;
    v.x = one(r, min(k, Kf - 1));
    v.y = one(r, min(k + S, Kf - 1));
    v.z = one(r, min(k + 2 * S, Kf - 1));
    v.w = one(r, min(k + 3 * S, Kf - 1));
    if (k >= Kf) v.x = 0.f;
    if (k + S >= Kf) v.y = 0.f;
    if (k + 2 * S >= Kf) v.z = 0.f;
    if (k + 3 * S >= Kf) v.w = 0.f;
    return v;
  }
};

// (256, 8): registers for 8 waves per SIMD, no spills; the 1D entries are
// latency-bound gathers and more waves in flight measured faster (R-MAT scale
// 16, K = 32: 16.3 -> 15.2 us with every entry in the 1D part).
// bpb: dense blocks per workgroup, 4 (one per wave) or 1 (its features shared by
// the four waves, whose sums are added in wave order through LDS).
template <int LPE, bool kVec, bool kSmall>
__global__ __launch_bounds__(256, 8) void hyb_sddmm_kernel(SddmmPlanDev p, const float* __restrict__ X, int64_t ldx,
                                                           const float* __restrict__ Y, int64_t ldy, int Kf,
                                                           float* __restrict__ out, int blocks1d, int bpb) {
  __shared__ float blk[4][256];
  const int lane = threadIdx.x & 63;
  const int wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const FeatureRows<kSmall> xs{X, ldx}, ys{Y, ldy};
  if ((int)blockIdx.x < blocks1d) {
    // a segment of LPE lanes computes kSddmmU consecutive entries, their
    // index loads and row gathers all in flight together
    constexpr int EPW = 64 / LPE;
    const int sub = lane % LPE;
    const int e0 = (((int)blockIdx.x * 4 + wib) * EPW + lane / LPE) * kSddmmU;
    if (e0 >= p.n1d) return;
    // four entries' ids in one load each (the arrays are padded to a multiple of
    // kSddmmU entries that repeat the last one)
    const int4 row4 = *reinterpret_cast<const int4*>(p.e_row + e0), col4 = *reinterpret_cast<const int4*>(p.e_col + e0),
               dst4 = *reinterpret_cast<const int4*>(p.e_out + e0);
    const int row[kSddmmU] = {row4.x, row4.y, row4.z, row4.w}, col[kSddmmU] = {col4.x, col4.y, col4.z, col4.w},
              dst[kSddmmU] = {dst4.x, dst4.y, dst4.z, dst4.w};
    typename FeatureRows<kSmall>::Row xr[kSddmmU], yr[kSddmmU];
    // consecutive entries of one row (CSR order) share the X load; an entry whose
    // row repeats skips its load and takes the previous X value in a select after
    // every load is issued (a copy inside the branch would wait for the previous
    // load before the next one)
    bool same[kSddmmU];
    float s[kSddmmU];
#pragma unroll
    for (int u = 0; u < kSddmmU; ++u) {
      xr[u] = xs.row(row[u]);
      yr[u] = ys.row(col[u]);
      same[u] = u > 0 && row[u] == row[u > 0 ? u - 1 : 0];
      s[u] = 0.f;
    }
    // kVec: lane sub holds features 4 sub .. + 3 of each step of 4 LPE; else
    // features sub + LPE i (any alignment, each load a run of LPE lanes)
    for (int k = kVec ? 4 * sub : sub; k < Kf; k += 4 * LPE) {
      float4 a[kSddmmU], b[kSddmmU];
#pragma unroll
      for (int u = 0; u < kSddmmU; ++u) {
        if constexpr (kVec) {
          if (!same[u]) a[u] = xs.quad(xr[u], k);
          b[u] = ys.quad(yr[u], k);
        } else {
          if (!same[u]) a[u] = xs.template strided<LPE>(xr[u], k, Kf);
          b[u] = ys.template strided<LPE>(yr[u], k, Kf);
        }
      }
#pragma unroll
      for (int u = 1; u < kSddmmU; ++u)
        if (same[u]) a[u] = a[u - 1];
#pragma unroll
      for (int u = 0; u < kSddmmU; ++u) s[u] += a[u].x * b[u].x + a[u].y * b[u].y + a[u].z * b[u].z + a[u].w * b[u].w;
    }
#pragma unroll
    for (int u = 0; u < kSddmmU; ++u) s[u] = segment_sum<LPE>(s[u]);
    if (sub == 0) {
#pragma unroll
      for (int u = 0; u < kSddmmU; ++u)
        if (e0 + u < p.n1d) out[dst[u]] = s[u];
    }
    return;
  }
  // Dense block: lane l = 16g + j loads features kb + 4g .. + 3 of X[rows[j]] and
  // Y[cols[j]], four steps of 16 features (64 with the block shared by the
  // waves) requested together.
  const int b = ((int)blockIdx.x - blocks1d) * bpb + (bpb == 1 ? 0 : wib);
  const bool shared_block = bpb == 1;
  const int g = lane >> 4, j = lane & 15;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  if (b < p.nblk) {
    const auto xr = xs.row(p.blk_rows[b * 16 + j]), yr = ys.row(p.blk_cols[b * 16 + j]);
    const int step = shared_block ? 64 : 16;
    for (int kb = shared_block ? 16 * wib : 0; kb < Kf; kb += 4 * step) {
      float4 xa[4], ya[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = kb + i * step + 4 * g;
        if (i > 0 && kb + i * step >= Kf) continue;
        if constexpr (kVec) {  // past the end: a clamped read, zeroed below
          const int kc = min(k, Kf - 4);
          xa[i] = xs.quad(xr, kc);
          ya[i] = ys.quad(yr, kc);
        } else {
          xa[i] = xs.template strided<1>(xr, k, Kf);
          ya[i] = ys.template strided<1>(yr, k, Kf);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i > 0 && kb + i * step >= Kf) continue;
        if constexpr (kVec) {
          const bool in = kb + i * step + 4 * g < Kf;
          xa[i] = make_float4(in ? xa[i].x : 0.f, in ? xa[i].y : 0.f, in ? xa[i].z : 0.f, in ? xa[i].w : 0.f);
          ya[i] = make_float4(in ? ya[i].x : 0.f, in ? ya[i].y : 0.f, in ? ya[i].z : 0.f, in ? ya[i].w : 0.f);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[i].x, ya[i].x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[i].y, ya[i].y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[i].z, ya[i].z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[i].w, ya[i].w, acc, 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) blk[wib][(4 * g + i) * 16 + j] = acc[i];
  __syncthreads();
  if (shared_block) {
    const int s0 = p.blk_ptr[b], s1 = p.blk_ptr[b + 1];
    for (int s = s0 + (int)threadIdx.x; s < s1; s += 256) {
      const int q = p.blk_pos[s];
      out[p.blk_out[s]] = ((blk[0][q] + blk[1][q]) + blk[2][q]) + blk[3][q];
    }
  } else if (b < p.nblk) {
    const int s0 = p.blk_ptr[b], s1 = p.blk_ptr[b + 1];
    for (int s = s0 + lane; s < s1; s += 64) out[p.blk_out[s]] = blk[wib][p.blk_pos[s]];
  }
}

hipError_t launch_hyb_sddmm(const SddmmPlanDev& p, const float* X,
                            int64_t ldx, const float* Y, int64_t ldy, int Kf,
                            float* out, hipStream_t s) {
  const bool vec = (Kf % 4 == 0) && (ldx % 4 == 0) && (ldy % 4 == 0) &&
                   ((reinterpret_cast<uintptr_t>(X) & 15) == 0) &&
                   ((reinterpret_cast<uintptr_t>(Y) & 15) == 0);
  // lanes per entry: a quarter of the features each, at most 16
  int lpe = 1;
  while (lpe < 16 && lpe * (vec ? 8 : 4) <= Kf) lpe *= 2;
  const int epw = 64 / lpe * kSddmmU;
  const int64_t waves1d = ((int64_t)p.n1d + epw - 1) / epw;
  const int64_t blocks1d = (waves1d + 3) / 4;
  const int bpb = Kf > kSharedKf && blocks1d + p.nblk <= max_blocks(256) ? 1 : 4;
  const int64_t blocks = blocks1d + ((int64_t)p.nblk + bpb - 1) / bpb;
  if (blocks == 0) return hipSuccess;
  auto small = [&](int64_t rows, int64_t ld) {
    return rows <= (1 << 24) && ld < (1 << 22) && ((rows - 1) * ld + Kf) * 4 < ((int64_t)1 << 32);
  };
  const bool fits = small(p.M, ldx) && small(p.N, ldy);
  auto go = [&](auto l, auto v, auto u) {
    hipLaunchKernelGGL((hyb_sddmm_kernel<decltype(l)::value, decltype(v)::value, decltype(u)::value>),
                       dim3((unsigned)blocks), dim3(256), 0, s, p, X, ldx, Y, ldy, Kf, out, (int)blocks1d, bpb);
  };
  auto by_layout = [&](auto l) {
    if (fits) {
      if (vec)
        go(l, std::true_type{}, std::true_type{});
      else
        go(l, std::false_type{}, std::true_type{});
    } else {
      if (vec)
        go(l, std::true_type{}, std::false_type{});
      else
        go(l, std::false_type{}, std::false_type{});
    }
  };
  switch (lpe) {
    case 1: by_layout(std::integral_constant<int, 1>{}); break;
    case 2: by_layout(std::integral_constant<int, 2>{}); break;
    case 4: by_layout(std::integral_constant<int, 4>{}); break;
    case 8: by_layout(std::integral_constant<int, 8>{}); break;
    default: by_layout(std::integral_constant<int, 16>{}); break;
  }
  return hipGetLastError();
}

}  // namespace stile
