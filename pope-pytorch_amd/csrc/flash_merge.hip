// Log-sum-exp merge of the key splits of one query row: the second launch of the decode and of the
// split flash forward (gfx950).
//
// A row's splits hold (m, l, O) in fp32: the reference max (log2 units), the sum of 2^(s - m) and
// the unnormalised output.  Thread = (row of the workgroup's, split group g, 4-dim quad q); group g
// takes every G-th split, eight splits' loads in flight at a time, and keeps a running (m, l, o)
// of its splits (one pass over the partials, no wait for a global maximum first); the groups'
// states then merge through LDS.  G is the number of splits where that leaves a workgroup (256
// threads) several rows, so few splits give many rows per workgroup and many splits of one row
// are read side by side: the pass is bound by the latency of its loads (4-5 us at 16 rows x 256
// splits as at 1,040 rows x 16).
#include "pope_common.hpp"
#include "pope_kernels.hpp"

namespace pope {

namespace {

constexpr int kThreads = 256;

template <typename T>
__global__ __launch_bounds__(kThreads) void flash_merge_kernel(FlashMergeParams p, int G, int RPB) {
  __shared__ float4 o_s[kThreads];
  __shared__ float2 ml_s[kThreads];
  const int tid = threadIdx.x;
  const int D = p.D, S = p.splits, qd = D / 4;
  const int q = tid % qd, t = tid / qd, rl = t % RPB, g = t / RPB;
  const int row = blockIdx.x * RPB + rl;
  const bool act = g < G && row < p.rows;
  float m = -INFINITY, l = 0.f;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  // folds one split into the running state; a split without a visible key has m = -inf, l = 0
  // and possibly an o that was never written, and leaves the state as it is.  One whose visible
  // scores are all NaN has m = -inf too (the maximum drops NaN) but l = NaN, and its NaN o counts:
  // the row is NaN, as in an unsplit kernel
  auto fold = [&](float2 ml, float4 v) {
    if (ml.x == -INFINITY && ml.y == 0.f) v = make_float4(0.f, 0.f, 0.f, 0.f);
    const float mn = fmaxf(m, ml.x);
    const float mu = mn == -INFINITY ? 0.f : mn;
    const float a = __builtin_amdgcn_exp2f(m - mu), w = __builtin_amdgcn_exp2f(ml.x - mu);
    acc.x = fmaf(acc.x, a, v.x * w);
    acc.y = fmaf(acc.y, a, v.y * w);
    acc.z = fmaf(acc.z, a, v.z * w);
    acc.w = fmaf(acc.w, a, v.w * w);
    l = fmaf(l, a, ml.y * w);
    m = mn;
  };
  if (act) {
    const float2* pml = reinterpret_cast<const float2*>(p.part_ml) + (int64_t)row * S;
    const float4* po4 = reinterpret_cast<const float4*>(p.part_o + (int64_t)row * S * D) + q;
    int s = g;
    for (; s + 7 * G < S; s += 8 * G) {
      float2 ml[8];
      float4 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        ml[u] = pml[s + u * G];
        v[u] = po4[(int64_t)(s + u * G) * qd];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) fold(ml[u], v[u]);
    }
    for (; s < S; s += G) fold(pml[s], po4[(int64_t)s * qd]);
  }
  o_s[tid] = acc;
  ml_s[tid] = make_float2(m, l);
  __syncthreads();
  if (g == 0 && row < p.rows) {
    const int st = RPB * qd;   // threads of one split group
    float M = -INFINITY;
    for (int g2 = 0; g2 < G; ++g2) M = fmaxf(M, ml_s[g2 * st + tid].x);
    const float Mu = M == -INFINITY ? 0.f : M;
    float L = 0.f;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int g2 = 0; g2 < G; ++g2) {
      const float2 sm = ml_s[g2 * st + tid];
      const float w = __builtin_amdgcn_exp2f(sm.x - Mu);
      const float4 v = o_s[g2 * st + tid];
      o.x = fmaf(v.x, w, o.x); o.y = fmaf(v.y, w, o.y); o.z = fmaf(v.z, w, o.z); o.w = fmaf(v.w, w, o.w);
      L = fmaf(sm.y, w, L);
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    const int bh = row / p.Nq, i = row % p.Nq;
    uint16_t* orow = p.o + (int64_t)(bh / p.Hq) * p.o_s[0] + (int64_t)(bh % p.Hq) * p.o_s[1] +
                     (int64_t)i * p.o_s[2] + 4 * q;
    u32x2 w2;   // rows are 16-byte aligned, D a multiple of 8
    w2[0] = T::pack2(o.x * inv, o.y * inv);
    w2[1] = T::pack2(o.z * inv, o.w * inv);
    *reinterpret_cast<u32x2*>(orow) = w2;
    if (q == 0) p.lse[row] = M == -INFINITY ? -INFINITY : (M + __builtin_amdgcn_logf(L)) * kLn2;
  }
}

}  // namespace

hipError_t launch_flash_merge(const FlashMergeParams& p, const char* name, int dtype, hipStream_t s) {
  const int tpr = kThreads / (p.D / 4);   // (row, split group) slots per workgroup: D <= 256
  const int G = p.splits < tpr ? p.splits : tpr;
  const int RPB = tpr / G;
  const dim3 grid((p.rows + RPB - 1) / RPB);
  return dtype == 2 ? launch_named(name, flash_merge_kernel<BF16>, grid, dim3(kThreads), s, p, G, RPB)
                    : launch_named(name, flash_merge_kernel<F16>, grid, dim3(kThreads), s, p, G, RPB);
}

}  // namespace pope
