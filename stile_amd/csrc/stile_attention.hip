// Fused sparse attention of libstile_hip.so for MI355X (gfx950).
#include "stile_device.h"

#include <algorithm>

namespace stile {

// ---------------------------------------------------------------------------
// Fused sparse attention: out = softmax(scale * Q K^T on the mask) V for BF16
// Q, K, V (rows x 64, leading dimension ld), FP32 out, over a plan built by
// stile_plan_create_attention (block-diagonal masks; tc_mask marks the mask
// entries among each chunk's k-slots).  One wave per window of 16 query rows;
// lane l holds query q = l & 15 and lane group g = l >> 4.
//
// Per chunk of 32 key columns (k-slots):
//   S^T = K Q^T as two 16x16 tiles (keys x queries), two v_mfma_f32_16x16x32_
//     bf16 each over the 64 features (lane group g carries features
//     32s + 8g .. +7 of step s for both operands, one 16-byte load each);
//     lane (g, q) then holds S[q][slot 16T + 4g + i], i = 0..3, T = 0, 1;
//   online softmax per query (running max m and sum l; the chunk max is
//     reduced over the four lanes of a query);
//   O^T += V^T P^T as four d-tiles of one v_mfma_f32_16x16x32_bf16: the
//     lane's eight probabilities are its B operand as they are (k-slot e of
//     lane group g = slot 4g + e for e < 4, 16 + 4g + e - 4 otherwise); the
//     V rows of the chunk are staged in LDS as they are and the A operand is
//     two transposed reads (ds_read_b64_tr_b16) per d-tile.
// Sparse entries of a window row (the plan's sparse part) come last, four
// lanes to a query (see below).
// Out row r = O[r] / l[r] (0 for a row without entries).
//
// What bounds it: the L1's cache accesses and the latency of the row fetches.
// With a K row's 16-byte pieces on lanes 16 apart (the MFMA operand order) and
// the sparse entries taken one a step, 64 masks of 640 to 5,120 rows (162,576
// rows, 23.0 M entries, 17 % of them sparse) took 225 us and 93 M cache
// accesses; with
// neighbouring lanes on one row everywhere (K through LDS), four sparse
// entries in flight a query and 32-bit row offsets they take 79 us and 30
// M.  One wave per workgroup: a window's length varies, and four waves of one
// workgroup hold its place until the longest is done (20,480 rows: 1.4 of
// 16 us).
// ---------------------------------------------------------------------------
// Bytes per K or V row staged in LDS: 160, so that the 32-byte runs one
// transposed read takes from eight consecutive rows, and the 16-byte pieces of
// eight consecutive K rows, start on distinct bank groups.
constexpr int kAttVRow = 160;
constexpr int kAttVBase = 32 * kAttVRow;  // V rows behind the K rows

// Exchanges between the four 16-lane groups of a wave (gfx950's
// v_permlane32_swap / v_permlane16_swap: the upper half, or the odd 16-lane
// rows, of one register with the lower half, or the even rows, of another).
struct Two {
  float a, b;
};
__device__ __forceinline__ Two swap32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
__device__ __forceinline__ Two swap16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
// max over lanes l, l ^ 32 / l, l ^ 16
__device__ __forceinline__ float max32(float x) {
  const Two r = swap32(x, x);
  return fmaxf(r.a, r.b);
}
__device__ __forceinline__ float max16(float x) {
  const Two r = swap16(x, x);
  return fmaxf(r.a, r.b);
}
// This wave's LDS accesses so far complete before those that follow.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// k-slot whose id is entry 4a + u of a chunk's 32 column ids (id i is slot
// 4 (i % 8) + i / 8).
__device__ __forceinline__ constexpr int att_slot(int a, int u) { return 16 * (a & 1) + 4 * u + (a >> 1); }

// Sum over the lanes of a quad, left in each of them (DPP operands).
__device__ __forceinline__ float sum4(float x) {
  auto dpp = [](float v, auto ctrl) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  x += dpp(x, std::integral_constant<int, 0xB1>{});  // quad_perm 1,0,3,2
  x += dpp(x, std::integral_constant<int, 0x4E>{});  // quad_perm 2,3,0,1
  return x;
}

// x if bit b of m is set, else -infinity
__device__ __forceinline__ float keep_if(uint32_t m, int b, float x) {
  const uint32_t all = (uint32_t)((int32_t)(m << (31 - b)) >> 31);
  return __uint_as_float((__float_as_uint(x) & all) | (0xff800000u & ~all));
}
// Pair e (elements 2e, 2e + 1) of eight BF16 values, and a.lo b.lo + a.hi b.hi
// + c in FP32 (v_dot2_f32_bf16).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pair_of(const bf16x8& v, int e) {
  const uint4 w = __builtin_bit_cast(uint4, v);
  return e == 0 ? w.x : e == 1 ? w.y : e == 2 ? w.z : w.w;
}
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}

// Whether any of eight BF16 values is an infinity or a NaN.
__device__ __forceinline__ bool not_finite(const bf16x8& v) {
  bool bad = false;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t w = pair_of(v, e);
    bad |= (w & 0x7f80u) == 0x7f80u || (w & 0x7f800000u) == 0x7f800000u;
  }
  return bad;
}

// Sparse entries of a query handled per step.
constexpr int kAttBatch = 4;
typedef int32_t i32x4_u __attribute__((ext_vector_type(4), aligned(4)));
// Row stride (floats) of the 16 x 64 block through which the dense part's
// sums change lanes: 68 puts the float4 reads of a lane group on 16 distinct
// bank quadruples.
constexpr int kAttOStride = 68;

// What the kernel reads of a plan (a launch passes no more of it).
struct AttArrays {
  const int32_t *win_rows, *tc_ptr, *tc_cols;
  const uint32_t* tc_mask;
  const int32_t *res_ptr, *res_cols;
};

template <bool kSmall>
__global__ __launch_bounds__(64, 3) void attention_fused_kernel(AttArrays p, AttOrder ord,
                                                                const __bf16* __restrict__ Qm,
                                                                const __bf16* __restrict__ Km,
                                                                const __bf16* __restrict__ Vm, int64_t ld,
                                                                float scale, float* __restrict__ out, int64_t ldo) {
  // the chunk's 32 K and 32 V rows; after them the sums on their way to the sparse part
  __shared__ __align__(16) unsigned char stage[64 * kAttVRow];
  static_assert(64 * kAttVRow >= 4 * 16 * kAttOStride);
  const int lane = threadIdx.x;
  const int x = blockIdx.x % kXcds;  // the XCD this workgroup is dispatched to
  int o0 = 0, o1 = 0;
#pragma unroll
  for (int i = 0; i < kXcds; ++i)  // selects, not a dynamically indexed copy
    if (i == x) {
      o0 = ord.start[i];
      o1 = ord.start[i + 1];
    }
  const int oi = o0 + (int)(blockIdx.x / kXcds);
  if (oi >= o1) return;
  const int w = __builtin_amdgcn_readfirstlane(ord.win[oi]);
  lds_u8* const vt = (lds_u8*)stage;
  // Eight values of a K, Q or V row from byte `at` of it.  kSmall: one 24-bit
  // multiply-add to a 32-bit offset from the (scalar) base, shared by the K and
  // V loads of an id; 64-bit products cost a dozen cycles per load more, as
  // much as the arithmetic on the loaded row.
  typedef typename std::conditional<kSmall, uint32_t, int64_t>::type Off;
  auto row_off = [&](int id, int at) -> Off {
    if constexpr (kSmall)
      return __umul24((unsigned)id, (unsigned)ld * 2u) + (unsigned)at;
    else
      return (int64_t)id * ld * 2 + at;
  };
  auto row8 = [&](const __bf16* base, Off off) {
    return *reinterpret_cast<const bf16x8*>(reinterpret_cast<const unsigned char*>(base) + off);
  };
  const int q = lane & 15, g = lane >> 4;
  const int row = p.win_rows[w * 16 + q];
  const Off qoff = row_off(max(row, 0), 16 * g);  // padding query rows compute on row 0, store nothing
  const bf16x8 qb0 = row8(Qm, qoff), qb1 = row8(Qm, qoff + 64);
  f32x4 acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, lsum = 0.f;
  const int c0 = p.tc_ptr[w], c1 = p.tc_ptr[w + 1];
  const int a = lane >> 3, o = lane & 7;
  // K and V rows of a chunk's slots att_slot(a, u): eight lanes read a row's
  // 128 bytes.  (K rows in MFMA operand order -- lane (g, q) 16 bytes of row q --
  // would be 64 separate cache accesses an instruction.)  The rows of chunk
  // c + 1 are requested before chunk c is processed (two register sets, loop
  // unrolled by two so neither is copied); column ids run one chunk further
  // ahead.
  i32x4_u cid;
  auto load_ids = [&](int c) { cid = *reinterpret_cast<const i32x4_u*>(p.tc_cols + (int64_t)c * 32 + 4 * a); };
  struct AttRegs {
    u32x4 kk[4], vv[4];
    uint32_t mw;
  };
  auto load_regs = [&](int c, AttRegs& r) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const Off off = row_off(cid[u], 16 * o);
      r.kk[u] = __builtin_bit_cast(u32x4, row8(Km, off));
      r.vv[u] = __builtin_bit_cast(u32x4, row8(Vm, off));
    }
    r.mw = p.tc_mask[(int64_t)c * 16 + q];
  };
  // Sparse rows of the window (see below): the query's entry range, Q and first
  // ids are requested before the chunks run.  A step's ids come in one load;
  // those past the row's end (of the next rows, or of the padding behind the
  // last one) are replaced by row 0 and take no part.
  const int sq = lane >> 2, s4 = lane & 3;
  const int r0 = p.res_ptr[w * 16 + sq], r1 = p.res_ptr[w * 16 + sq + 1];
  int n = r1 - r0;
#pragma unroll
  for (int off = 4; off < 64; off <<= 1) n = max(n, __shfl_xor(n, off));
  const Off sqoff = row_off(max(p.win_rows[w * 16 + sq], 0), 16 * s4);
  const bf16x8 qs0 = row8(Qm, sqoff), qs1 = row8(Qm, sqoff + 64);
  i32x4_u sid;
  auto load_cols = [&](int j) { sid = *reinterpret_cast<const i32x4_u*>(p.res_cols + min(r0 + j, r1)); };
  load_cols(0);
  const int last = c1 - 1;
  AttRegs R0, R1;
  if (c0 < c1) {
    load_ids(c0);
    load_regs(c0, R0);
    load_ids(min(c0 + 1, last));
  }
  auto process = [&](const AttRegs& r) {
    const uint32_t mw = r.mw;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      lds_u8* at = vt + att_slot(a, u) * kAttVRow + 16 * o;
      *reinterpret_cast<lds_u128*>(at) = r.kk[u];
      *reinterpret_cast<lds_u128*>(at + kAttVBase) = r.vv[u];
    }
    wave_lds_sync();
    // A operands of the scores: lane (g, q) features 8g .. and 32 + 8g .. of
    // slots q and 16 + q
    lds_u8* const kq = vt + q * kAttVRow + 16 * g;
    auto k8 = [&](int at) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<lds_u128*>(kq + at)); };
    const bf16x8 k00 = k8(0), k01 = k8(64), k10 = k8(16 * kAttVRow), k11 = k8(16 * kAttVRow + 64);
    f32x4 st0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k00, qb0, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    st0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k01, qb1, st0, 0, 0, 0);
    f32x4 st1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k10, qb0, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    st1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k11, qb1, st1, 0, 0, 0);
    // online softmax
    float sv[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sv[i] = keep_if(mw, 4 * g + i, st0[i]);
      sv[4 + i] = keep_if(mw, 16 + 4 * g + i, st1[i]);
    }
    float cm = sv[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) cm = fmaxf(cm, sv[i]);
    cm = max16(max32(cm));
    const float m_new = fmaxf(m, cm);
    const float mu = m_new == -INFINITY ? 0.f : m_new;  // nothing yet: every exponential below is 0
    const float alpha = __expf((m - mu) * scale);
    uint32_t pk[4];
    float psum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      pk[i] = bf16_pair(__expf((sv[2 * i] - mu) * scale), __expf((sv[2 * i + 1] - mu) * scale));
      // the sum uses the BF16-rounded probabilities the MFMA multiplies
      psum += bf16_lo(pk[i]) + bf16_hi(pk[i]);
    }
    lsum = lsum * alpha + psum;
    m = m_new;
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] *= alpha;
    const bf16x8 pb = __builtin_bit_cast(bf16x8, make_uint4(pk[0], pk[1], pk[2], pk[3]));
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      // lane (g, 4e + j) addresses features 16t + 4j .. + 3 of slot 4g + e (then
      // 16 + 4g + e); the transposed read hands lane q of the group feature
      // 16t + q of the four slots
      lds_u8* at = vt + kAttVBase + (4 * g + (q >> 2)) * kAttVRow + 32 * t + 8 * (q & 3);
      const i16x4 lo = lds_tr_read(at), hi = lds_tr_read(at + 16 * kAttVRow);
      const bf16x8 va = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, pb, acc[t], 0, 0, 0);
    }
    // the reads are done before the next chunk's rows overwrite these
    wave_lds_sync();
    };
  if (c0 < c1) {
    int c = c0;
    while (c + 2 <= c1) {
      load_regs(min(c + 1, last), R1);
      load_ids(min(c + 2, last));
      process(R0);
      ++c;
      load_regs(min(c + 1, last), R0);
      load_ids(min(c + 2, last));
      process(R1);
      ++c;
    }
    if (c < c1) process(R0);
  }
  float ltot = lsum + __shfl_xor(lsum, 16);
  ltot += __shfl_xor(ltot, 32);
  if (n == 0) {
    if (row < 0) return;
    const float inv = ltot > 0.f ? 1.f / ltot : 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
      st4(out + (int64_t)row * ldo + 16 * t + 4 * g,
          make_float4(acc[t][0] * inv, acc[t][1] * inv, acc[t][2] * inv, acc[t][3] * inv));
    return;
  }
  // Sparse part.  Four lanes share a query (query lane >> 2), lane s4 of them
  // holding features 8 s4 .. + 7 and 32 + 8 s4 .. + 7, so that a K or V row is
  // read in two 64-byte runs of four lanes; kAttBatch entries are in flight per
  // query.  The state of the dense part comes to these lanes through LDS.  Each
  // entry's probability is rounded to BF16 against the maximum of the row so
  // far, entry by entry, and then brought to the step's.
  {
    const bf16x8 z0 = row8(Vm, row_off(0, 16 * s4)), z1 = row8(Vm, row_off(0, 16 * s4 + 64));
    float* const os = reinterpret_cast<float*>(stage);  // [16][kAttOStride]
#pragma unroll
    for (int t = 0; t < 4; ++t)
      st4(os + q * kAttOStride + 16 * t + 4 * g, make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]));
    wave_lds_sync();
    float ms = __shfl(m, sq), ls = __shfl(ltot, sq), om[16];
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
      const float4 v = ld4(os + sq * kAttOStride + 8 * s4 + (e < 8 ? e : 24 + e));
      om[e] = v.x; om[e + 1] = v.y; om[e + 2] = v.z; om[e + 3] = v.w;
    }
    // Entries past a row's end read V's row 0 with probability 0: where that holds an
    // infinity or a NaN (0 times it is a NaN) their values are zeroed.  (3 masks of
    // 2,646 rows, 64 of 640 to 5,120: 11.6 and 77.0 us, 11.4 and 76.8 without; zeroed
    // always 11.6 and 77.2, by loads past a descriptor of V 12.2 and 77.0.)
    const bool spoilt = __any(not_finite(z0) || not_finite(z1));
    for (int j = 0; j < n; j += kAttBatch) {
      bf16x8 ka[kAttBatch], kb[kAttBatch], va[kAttBatch], vb[kAttBatch];
      bool on[kAttBatch];
#pragma unroll
      for (int u = 0; u < kAttBatch; ++u) {
        on[u] = r0 + j + u < r1;
        const Off off = row_off(on[u] ? sid[u] : 0, 16 * s4);
        ka[u] = row8(Km, off);
        kb[u] = row8(Km, off + 64);
        va[u] = row8(Vm, off);
        vb[u] = row8(Vm, off + 64);
      }
      load_cols(j + kAttBatch);
      __builtin_amdgcn_sched_barrier(0);  // every load of the step before its arithmetic
      float sval[kAttBatch], m_run = ms;
#pragma unroll
      for (int u = 0; u < kAttBatch; ++u) {
        float dot = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) dot += (float)qs0[e] * (float)ka[u][e] + (float)qs1[e] * (float)kb[u][e];
        dot = sum4(dot);
        sval[u] = on[u] ? dot : -INFINITY;
        m_run = fmaxf(m_run, sval[u]);
      }
      if (spoilt) {
#pragma unroll
        for (int u = 0; u < kAttBatch; ++u)
          if (!on[u]) va[u] = vb[u] = __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0));
      }
      auto prob = [&](float x, float mx) { return x == -INFINITY ? 0.f : __expf((x - mx) * scale); };
      if (__all(m_run == ms)) {
        // no row's maximum moved: entries two at a time (v_dot2_f32_bf16)
#pragma unroll
        for (int u = 0; u < kAttBatch; u += 2) {
          const uint32_t pp = bf16_pair(prob(sval[u], ms), prob(sval[u + 1], ms));
          ls += bf16_lo(pp) + bf16_hi(pp);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            om[e] = dot2(pp, half_sel(pair_of(va[u], e >> 1), pair_of(va[u + 1], e >> 1), e & 1), om[e]);
            om[8 + e] = dot2(pp, half_sel(pair_of(vb[u], e >> 1), pair_of(vb[u + 1], e >> 1), e & 1), om[8 + e]);
          }
        }
        continue;
      }
      const float mz = m_run == -INFINITY ? 0.f : m_run;
      const float alpha = __expf((ms - mz) * scale);
      float pe[kAttBatch], mu = ms;
      ls *= alpha;
#pragma unroll
      for (int u = 0; u < kAttBatch; ++u) {
        mu = fmaxf(mu, sval[u]);
        pe[u] = bf16_lo(bf16_pair(prob(sval[u], mu), 0.f)) * __expf((mu - mz) * scale);
        ls += pe[u];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float x = om[e] * alpha, y = om[8 + e] * alpha;
#pragma unroll
        for (int u = 0; u < kAttBatch; ++u) {
          x += pe[u] * (float)va[u][e];
          y += pe[u] * (float)vb[u][e];
        }
        om[e] = x;
        om[8 + e] = y;
      }
      ms = m_run;
    }
    const int srow = p.win_rows[w * 16 + sq];
    if (srow < 0) return;
    const float inv = ls > 0.f ? 1.f / ls : 0.f;
#pragma unroll
    for (int e = 0; e < 16; e += 4)
      st4(out + (int64_t)srow * ldo + 8 * s4 + (e < 8 ? e : 24 + e),
          make_float4(om[e] * inv, om[e + 1] * inv, om[e + 2] * inv, om[e + 3] * inv));
  }
}

hipError_t launch_attention(const SpmmPlanDev& p, const AttOrder& ord, const void* Q, const void* K, const void* V,
                            int64_t ld, float scale, float* out, int64_t ldo, hipStream_t s) {
  if (p.W == 0) return hipSuccess;
  int longest = 0;
  for (int x = 0; x < kXcds; ++x) longest = max(longest, ord.start[x + 1] - ord.start[x]);
  // 32-bit row offsets from 24-bit products: up to 2^24 rows and 4 GiB (of Q: M,
  // of K and V: K, equal in attention plans)
  const int64_t rows = max(p.M, p.K);
  const bool small = rows < (1 << 24) && ld < (1 << 23) && rows * ld * 2 < ((int64_t)1 << 32);
  const auto kernel = small ? attention_fused_kernel<true> : attention_fused_kernel<false>;
  const AttArrays arrays{p.win_rows, p.tc_ptr, p.tc_cols, p.tc_mask, p.res_ptr, p.res_cols};
  auto launch = [&](const AttOrder& o, int most) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(most * kXcds)), dim3(64), 0, s, arrays, o,
                       static_cast<const __bf16*>(Q), static_cast<const __bf16*>(K), static_cast<const __bf16*>(V),
                       ld, scale, out, ldo);
    return hipGetLastError();
  };
  constexpr int kMost = (int)(max_blocks(64) / kXcds);  // windows per XCD of one launch
  if (longest <= kMost) return launch(ord, longest);
  AttOrder part = ord;  // in launches of equally many windows per XCD
  for (int64_t a = 0; a < p.W; a = part.start[kXcds]) {
    const int64_t n = std::min<int64_t>(p.W - a, (int64_t)kMost * kXcds);
    for (int x = 0; x <= kXcds; ++x) part.start[x] = (int32_t)(a + n * x / kXcds);
    const hipError_t e = launch(part, (int)((n + kXcds - 1) / kXcds));
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace stile
