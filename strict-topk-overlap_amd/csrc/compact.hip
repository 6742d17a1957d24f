// Compact speculation (strict_topk/kernels.py:263-356,480-501) in two launches
// over the whole GPU.
//
// The reference runs a K-only mass pass, the grouping, then one program per
// head that walks every low block token by token in the low frame (and one
// per retained block).  That walk is one CU's work: 63 us at 32 heads x 64
// predicted blocks of 32 x 128 fp16, a third of the whole composed step.  Here
//   k_compact_states  one wave per (head, slot) reads the block's K and V once
//                     and writes its mass (m, l), its value sum u and the
//                     absolute sum of the same terms, both in the block's own
//                     frame;
//   k_compact_merge   one workgroup per head forms the groups as the hybrid
//                     grouping does, copies the retained blocks' states and
//                     sums the low blocks' rows rescaled by exp(m - low_m),
//                     which is the same sum over tokens: exp(s - low_m) =
//                     exp(s - m) exp(m - low_m).
// Every predicted block's V is needed in either form (retained or low), so no
// byte is read more than before; the rows pass through a workspace of
// 2 S D floats per head.  At the shape above the call's kernels take 7.8 + 4.8
// us instead of 7.3 (mass) + 6.0 (grouping) + 62.8 (values).
#include "states_tok.hpp"
#include "api.hpp"

namespace stk {

constexpr int kCompactThreads = 512;
constexpr int kCompactRows = 256;   // predicted blocks per head
constexpr int kCompactPF = 4;       // rows in flight per thread and pass

struct CompactStatesArgs {
  const void* q; const void* k; const void* v;
  const void* ids; int itype;
  int hq, hkv, n, b, d, s;
  float* m; float* l;   // [hq, s]
  float* w;             // [hq, s, 2, d]: u, then the absolute sums
};

template <typename T, int NCH, int UP, typename I>
__global__ __launch_bounds__(256, NCH <= 4 ? 4 : 2) void k_compact_states(CompactStatesArgs a) {
  using TT = TokTile<T, NCH, UP, true>;
  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t item = (int64_t)wg * (blockDim.x / STK_WAVE) + wave_id();
  if (item >= (int64_t)a.hq * a.s) return;
  const int h = (int)(item / a.s);
  TT t;
  t.init();
  uint32_t qw[TT::QW];
  t.load_q(reinterpret_cast<const T*>(a.q) + (size_t)h * TT::D, qw);
  const int64_t bid = reinterpret_cast<const I*>(a.ids)[item];
  const bool ok = bid >= 0 && bid < a.n;
  const int kv = h / (a.hq / a.hkv);
  const float scale = 1.0f / sqrtf((float)TT::D);
  const size_t off = (((size_t)kv * a.n + (ok ? (size_t)bid : 0)) * a.b) * TT::D;
  const T* kb = reinterpret_cast<const T*>(a.k) + off;
  const T* vb = reinterpret_cast<const T*>(a.v) + off;
  float m = -INFINITY, l = 0.f, acc[TT::DPL], aab[TT::DPL];
#pragma unroll
  for (int e = 0; e < TT::DPL; ++e) acc[e] = aab[e] = 0.f;
  uint32_t kw[UP][TT::QW], vw[TT::CH][TT::VW];
  if (ok) {
    for (int t0 = 0; t0 < a.b; t0 += TT::CH) {
      t.load(kb, vb, t0, kw, vw);
      __builtin_amdgcn_sched_barrier(0);   // every load before any arithmetic
      t.template update<false, true>(qw, kw, vw, t0, a.b, scale, m, l, acc, aab);
    }
  }
  if (lane_id() == 0) {
    a.m[item] = m;
    a.l[item] = l;
  }
  t.store(a.w + item * 2 * TT::D, acc);
  t.store(a.w + item * 2 * TT::D + TT::D, aab);
}

struct CompactMergeArgs {
  const void* ids; int itype;
  int s, d, c;
  float tau;
  const float* pm; const float* pl; const float* w;
  uint8_t* high; void* rids; uint8_t* overflow;
  float* lm; float* ll; float* lu; float* labs;
  float* m; float* l; float* u;
};

__global__ __launch_bounds__(kCompactThreads) void k_compact_merge(CompactMergeArgs a) {
  __shared__ float s_m[kCompactRows], s_l[kCompactRows], s_w[kCompactRows];
  __shared__ int s_rank[kCompactRows];   // retained row + 1, 0 for a low block
  __shared__ float4 s_pu[kCompactThreads], s_pa[kCompactThreads];
  const int h = blockIdx.x, tid = threadIdx.x, s = a.s, d = a.d;
  const int64_t row0 = (int64_t)h * s;
  const float mv = ld_or(a.pm, row0 + tid, tid < s, -INFINITY);
  const float lv = ld_or(a.pl, row0 + tid, tid < s, 0.f);
  const int64_t pid = tid < s ? load_id(a.ids, a.itype, row0 + tid) : -1;
  const int tpr = d >> 2, rgn = kCompactThreads / tpr;
  const int c4 = tid % tpr, rg = tid / tpr;
  const bool act = rg < rgn;
  float4 uu[kCompactPF], ua[kCompactPF];
  // every load is issued, rows past s reading row 0 (see k_hybrid_group1)
  auto fetch = [&](int pass) {
#pragma unroll
    for (int j = 0; j < kCompactPF; ++j) {
      const int r = rg + rgn * (pass * kCompactPF + j);
      const float* p = a.w + (row0 + (act && r < s ? r : 0)) * 2 * d + 4 * (act ? c4 : 0);
      uu[j] = *reinterpret_cast<const float4*>(p);
      ua[j] = *reinterpret_cast<const float4*>(p + d);
    }
  };
  fetch(0);
  if (tid < kCompactRows) {
    s_m[tid] = mv;
    s_l[tid] = lv;
  }
  __syncthreads();
  // ---- the groups, the same in every wave (lane l: rows l + 64 c):
  // high = mass >= tau * total, ranked in position order and capped at C
  float pm[4], pl[4], gm = -INFINITY, tot = 0.f, lm = -INFINITY, z = 0.f;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    pm[c] = s_m[c * STK_WAVE + lane_id()];
    pl[c] = s_l[c * STK_WAVE + lane_id()];
    gm = fmaxf(gm, pm[c]);
  }
  gm = wave_max_u(gm);
#pragma unroll
  for (int c = 0; c < 4; ++c) tot += wexp(pm[c], gm) * pl[c];
  const float thr = a.tau * wave_sum_u(tot);
  int rank[4], count = 0;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const bool in = c * STK_WAVE + lane_id() < s;
    const bool hi = in && wexp(pm[c], gm) * pl[c] >= thr;
    const uint64_t b = __ballot(hi);
    const int r = count + __popcll(b & lanemask_lt()) + 1;
    rank[c] = hi && r <= a.c ? r : 0;
    count += __popcll(b);
    lm = in && rank[c] == 0 ? fmaxf(lm, pm[c]) : lm;
  }
  lm = wave_max_u(lm);
  const float lowm = lm == -INFINITY ? 0.f : lm;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const bool low = c * STK_WAVE + lane_id() < s && rank[c] == 0;
    const float wt = low ? wexp(pm[c], lowm) : 0.f;
    z += wt * pl[c];
    if (wave_id() == 0) {
      s_rank[c * STK_WAVE + lane_id()] = rank[c];
      s_w[c * STK_WAVE + lane_id()] = wt;
    }
  }
  z = wave_sum_u(z);
  __syncthreads();
  const int kept = count < a.c ? count : a.c;
  if (tid < s) {
    const int r = s_rank[tid];
    a.high[row0 + tid] = r != 0;
    if (r) {
      store_id(a.rids, a.itype, (int64_t)h * a.c + r - 1, pid);
      a.m[(int64_t)h * a.c + r - 1] = mv;
      a.l[(int64_t)h * a.c + r - 1] = lv;
    }
  }
  for (int c = kept + tid; c < a.c; c += kCompactThreads) {
    store_id(a.rids, a.itype, (int64_t)h * a.c + c, -1);
    a.m[(int64_t)h * a.c + c] = -INFINITY;
    a.l[(int64_t)h * a.c + c] = 0.f;
  }
  if (tid == 0) {
    a.overflow[h] = count > a.c;
    a.lm[h] = lowm;
    a.ll[h] = z;
  }
  // ---- retained rows copied, low rows summed
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 lu = zero, la = zero;
  const int passes = (s + rgn * kCompactPF - 1) / (rgn * kCompactPF);
  for (int pass = 0; pass < passes; ++pass) {
    if (pass) fetch(pass);
#pragma unroll
    for (int j = 0; j < kCompactPF; ++j) {
      const int r = rg + rgn * (pass * kCompactPF + j);
      if (act && r < s) {
        const float4 x = uu[j], y = ua[j];
        if (const int k = s_rank[r]; k) {
          *reinterpret_cast<float4*>(a.u + ((int64_t)h * a.c + k - 1) * d + 4 * c4) = x;
        } else {
          const float wt = s_w[r];
          lu.x += wt * x.x; lu.y += wt * x.y; lu.z += wt * x.z; lu.w += wt * x.w;
          la.x += wt * y.x; la.y += wt * y.y; la.z += wt * y.z; la.w += wt * y.w;
        }
      }
    }
  }
  if (act)
    for (int c = kept + rg; c < a.c; c += rgn)
      *reinterpret_cast<float4*>(a.u + ((int64_t)h * a.c + c) * d + 4 * c4) = zero;
  s_pu[tid] = lu;
  s_pa[tid] = la;
  __syncthreads();
  if (tid < 2 * tpr) {
    const float4* part = tid < tpr ? s_pu : s_pa;
    float* dst = tid < tpr ? a.lu : a.labs;
    const int col = tid < tpr ? tid : tid - tpr;
    float4 su = zero;
    for (int g = 0; g < rgn; ++g) {
      const float4 x = part[g * tpr + col];
      su.x += x.x; su.y += x.y; su.z += x.z; su.w += x.w;
    }
    *reinterpret_cast<float4*>(dst + (size_t)h * d + 4 * col) = su;
  }
}

}  // namespace stk

using namespace stk;

// Whether the two launches cover the shape (the workspace and outputs are
// 16-byte aligned by the callers' allocations or checked below); a row of S
// blocks is one lane per block in k_compact_merge.
static int compact_nch(int dtype, int b, int d, int s, uintptr_t align) {
  if (dtype != DT_BF16 && dtype != DT_F16) return 0;
  return s >= 1 && s <= kCompactRows ? tok_nch(dtype, d, b, align) : 0;
}

extern "C" {

STK_API size_t stk_compact_workspace_bytes(int dtype, int hq, int b, int d, int s) {
  return compact_nch(dtype, b, d, s, 0) ? stk_align((size_t)hq * s * 2 * d * 4) : 0;
}

// strict_topk/kernels.py:480-501 with scratch memory
STK_API int stk_speculate_compact(const void* q, const void* k, const void* v, int dtype, int hq,
                                  int hkv, int n, int b, int d, const void* pred, int pred_dtype,
                                  int s, float tau, int capacity, float* m, float* l, float* u,
                                  uint8_t* high, float* low_m, float* low_l, float* low_u,
                                  float* low_abs, void* retained_ids, uint8_t* overflow,
                                  float* mass_m, float* mass_l, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  const uintptr_t bits = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
                         reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(u) |
                         reinterpret_cast<uintptr_t>(low_u) | reinterpret_cast<uintptr_t>(low_abs) |
                         reinterpret_cast<uintptr_t>(workspace);
  const int nch = compact_nch(dtype, b, d, s, bits);
  if (!nch || !workspace || workspace_bytes < stk_compact_workspace_bytes(dtype, hq, b, d, s))
    return stk_speculate(q, k, v, dtype, hq, hkv, n, b, d, pred, pred_dtype, s, 2, tau, capacity,
                         m, l, u, high, low_m, low_l, low_u, low_abs, retained_ids, overflow,
                         mass_m, mass_l, stream);
  STK_REQUIRE(stk_check_kv(dtype, hq, hkv, n, b, d));
  STK_REQUIRE(q && k && v && pred && m && l && u, "null pointer");
  STK_REQUIRE(tau >= 0.f && tau <= 1.f, "mass_threshold must be in [0,1]");
  STK_REQUIRE(high && low_m && low_l && low_u && low_abs && retained_ids && overflow && mass_m &&
                  mass_l,
              "null compact output");
  STK_REQUIRE(capacity >= 1 && capacity <= s, "bad compact capacity");
  STK_REQUIRE(pred_dtype == IT_I32 || pred_dtype == IT_I64, "bad ids");
  hipStream_t st = (hipStream_t)stream;
  float* w = static_cast<float*>(workspace);
  CompactStatesArgs sa{q, k, v, pred, pred_dtype, hq, hkv, n, b, d, s, mass_m, mass_l, w};
  const int grid = (int)(((int64_t)hq * s + 3) / 4);
  STK_DISPATCH_TOK(dtype, nch, {
    if constexpr (sizeof(T) == 2) {
      if (tok_up(b) == 1 && pred_dtype == IT_I64)
        hipLaunchKernelGGL((k_compact_states<T, NCH, 1, int64_t>), dim3(grid), dim3(256), 0, st, sa);
      else if (tok_up(b) == 1)
        hipLaunchKernelGGL((k_compact_states<T, NCH, 1, int32_t>), dim3(grid), dim3(256), 0, st, sa);
      else if (pred_dtype == IT_I64)
        hipLaunchKernelGGL((k_compact_states<T, NCH, 2, int64_t>), dim3(grid), dim3(256), 0, st, sa);
      else
        hipLaunchKernelGGL((k_compact_states<T, NCH, 2, int32_t>), dim3(grid), dim3(256), 0, st, sa);
    }
  });
  int rc = stk_check_launch("k_compact_states");
  if (rc) return rc;
  CompactMergeArgs ma{pred, pred_dtype, s, d, capacity, tau, mass_m, mass_l, w, high,
                      retained_ids, overflow, low_m, low_l, low_u, low_abs, m, l, u};
  hipLaunchKernelGGL(k_compact_merge, dim3(hq), dim3(kCompactThreads), 0, st, ma);
  return stk_check_launch("k_compact_merge");
}

}  // extern "C"
