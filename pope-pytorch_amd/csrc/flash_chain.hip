// Chain rule of the polar transform on raw expanded-row gradients (gfx950): the last launch of the
// wide-head backward (one raw row per key / query), and of a narrow backward whose jobs were split
// (flash_bwd_split: the partial rows of the splits are summed here, in split order, and dV with
// them).  Bound by HBM: 4 EP bytes per row and split, 4.2 TB/s at 32,768 rows each side of EP 512 (44.6 us).
// A thread keeps its four dims over the block's rows, so that dbias adds up in registers: with an LDS
// atomic per element the LDS was busy 80% of the time (64.7 us there).
#include "pope_common.hpp"
#include "pope_kernels.hpp"

namespace pope {

namespace {

// Blocks [0, nk): krows key rows of one (batch, kv head); blocks [nk, nk + nq): qrows query rows of
// one (batch, head).  With the raw expanded-row gradients U (cos column e = d, sin column
// e = R + d, pass-through column e = R + d) and the row's phase (keys F[j]; queries
// F[q_off + i] - bias, the bias on the query side as in the preparation):
//   dx = sigmoid(x) (cos U_c + sin U_s),  dphase = softplus(x) (cos U_s - sin U_c)
// and pass-through dims dx = U.  Key phase derivatives also sum into dbias (per block in LDS,
// then one atomic per dim).  A thread takes 4 consecutive dims per step (D and R are multiples of
// 8; the rows of q, k, dq, dk are 16-byte aligned): 16-byte loads of U, 8-byte loads and stores
// of the bf16 / fp16 rows.
template <typename T>
__device__ __forceinline__ void load4(const uint16_t* p, float* x) {
  const u32x2 w = *reinterpret_cast<const u32x2*>(p);
  x[0] = T::to_float((uint16_t)(w[0] & 0xffffu));
  x[1] = T::to_float((uint16_t)(w[0] >> 16));
  x[2] = T::to_float((uint16_t)(w[1] & 0xffffu));
  x[3] = T::to_float((uint16_t)(w[1] >> 16));
}
template <typename T>
__device__ __forceinline__ void store4(uint16_t* p, const float* g) {
  u32x2 w;
  w[0] = T::pack2(g[0], g[1]);
  w[1] = T::pack2(g[2], g[3]);
  *reinterpret_cast<u32x2*>(p) = w;
}
// Sum of 4 consecutive floats over S partial rows `stride` floats apart, in order.
__device__ __forceinline__ float4 sum4(const float* u, int S, int64_t stride) {
  float4 a = *reinterpret_cast<const float4*>(u);
#pragma unroll 4
  for (int s = 1; s < S; ++s) {
    const float4 b = *reinterpret_cast<const float4*>(u + s * stride);
    a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
  }
  return a;
}
template <typename T>
__global__ __launch_bounds__(256) void flash_chain_kernel(FlashBwdParams p, int nk, int krows, int qrows) {
  const float* wk = p.wk;
  const float* wq = p.wq;
  __shared__ float dsum[256];
  const int tid = threadIdx.x;
  const int D = p.D, R = p.R, EP = p.EP;
  const int D4 = D / 4, rpp = 256 / D4, r0 = tid / D4, d = 4 * (tid % D4);   // rpp rows per pass, threads past them idle
  if ((int)blockIdx.x < nk) {
    const int nkb = (p.Nk + krows - 1) / krows;
    const int k0 = krows * (blockIdx.x % nkb), bhk = blockIdx.x / nkb;
    const int b = bhk / p.Hk, hk = bhk % p.Hk;
    for (int e = tid; e < R; e += 256) dsum[e] = 0.f;
    __syncthreads();
    const uint16_t* kb = p.k + (int64_t)b * p.k_s[0] + (int64_t)hk * p.k_s[1];
    uint16_t* dkb = p.dk + (int64_t)b * p.dk_s[0] + (int64_t)hk * p.dk_s[1];
    const float2* tb = R ? p.table + (int64_t)b * p.t_sb + (int64_t)hk * p.t_sh : nullptr;
    float* dfb = p.dfreqs ? p.dfreqs + (int64_t)b * p.df_s[0] + (int64_t)hk * p.df_s[1] : nullptr;
    float* kpb = p.kpart ? p.kpart + (int64_t)bhk * p.Nk * R : nullptr;
    const float* wrow = wk + (int64_t)bhk * p.NkP * EP;
    const int S = p.kv_splits;
    const int64_t sk = (int64_t)p.B * p.Hk * p.NkP * EP;
    if (p.wv) {   // dV of the splits
      const int64_t sv = (int64_t)p.B * p.Hk * p.NkP * p.DV;
      const float* vrow = p.wv + (int64_t)bhk * p.NkP * p.DV;
      uint16_t* dvb = p.dv + (int64_t)b * p.dv_s[0] + (int64_t)hk * p.dv_s[1];
      if (r0 < rpp) {
#pragma unroll 2
        for (int key = k0 + r0; key < min(k0 + krows, p.Nk); key += rpp) {
          const float4 a = sum4(vrow + (int64_t)key * p.DV + d, S, sv);
          const float g[4] = {a.x, a.y, a.z, a.w};
          store4<T>(dvb + (int64_t)key * p.dv_s[2] + d, g);
        }
      }
    }
    float db[4] = {0.f, 0.f, 0.f, 0.f};
    if (r0 < rpp) {
#pragma unroll 2
      for (int r = r0; r < krows; r += rpp) {
        const int key = k0 + r;
        if (key >= p.Nk) break;
        const float* u = wrow + (int64_t)key * EP;
        float g[4];
        if (d < R) {   // R % 4 == 0: all four dims rotated
          float x[4];
          load4<T>(kb + (int64_t)key * p.k_s[2] + d, x);
          const float4 c01 = *reinterpret_cast<const float4*>(tb + (int64_t)key * R + d);
          const float4 c23 = *reinterpret_cast<const float4*>(tb + (int64_t)key * R + d + 2);
          const float4 uc = sum4(u + d, S, sk), us = sum4(u + R + d, S, sk);
          const float cs[4] = {c01.x, c01.z, c23.x, c23.z}, sn[4] = {c01.y, c01.w, c23.y, c23.w};
          const float ucv[4] = {uc.x, uc.y, uc.z, uc.w}, usv[4] = {us.x, us.y, us.z, us.w};
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            g[t] = sigmoid_f(x[t]) * (cs[t] * ucv[t] + sn[t] * usv[t]);
            const float dpsi = softplus_f(x[t]) * (cs[t] * usv[t] - sn[t] * ucv[t]);
            db[t] += dpsi;
            if (kpb) kpb[(int64_t)key * R + d + t] = dpsi;
            else if (dfb) atomicAdd(dfb + (int64_t)key * p.df_s[2] + d + t, dpsi);
          }
        } else {
          const float4 us = sum4(u + R + d, S, sk);
          g[0] = us.x; g[1] = us.y; g[2] = us.z; g[3] = us.w;
        }
        store4<T>(dkb + (int64_t)key * p.dk_s[2] + d, g);
      }
    }
    if (p.dbias && !kpb) {
      if (r0 < rpp && d < R) {
#pragma unroll
        for (int t = 0; t < 4; ++t) atomicAdd(&dsum[d + t], db[t]);
      }
      __syncthreads();
      for (int e = tid; e < R; e += 256) atomicAdd(p.dbias + (int64_t)hk * p.bias_sh + e, dsum[e]);
    }
    return;
  }
  const int nqb = (p.Nq + qrows - 1) / qrows, blk = blockIdx.x - nk;
  const int q0 = qrows * (blk % nqb), bh = blk / nqb;
  const int b = bh / p.Hq, h = bh % p.Hq, hk = h % p.Hk;
  const int q_off = p.Nk - p.Nq;
  const uint16_t* qb = p.q + (int64_t)b * p.q_s[0] + (int64_t)h * p.q_s[1];
  uint16_t* dqb = p.dq + (int64_t)b * p.dq_s[0] + (int64_t)h * p.dq_s[1];
  const float2* tq = R ? p.table + (int64_t)b * p.t_sb + (int64_t)h * p.t_sh : nullptr;
  const float2* bq = R ? p.btab + (p.Hb > 1 ? hk : 0) * R : nullptr;
  float* dfb = p.dfreqs ? p.dfreqs + (int64_t)b * p.df_s[0] + (int64_t)h * p.df_s[1] : nullptr;
  float* qpb = p.qpart && p.dfreqs ? p.qpart + (int64_t)bh * p.Nq * R : nullptr;
  const float* wrow = wq + (int64_t)bh * p.NqP * EP;
  const int S = p.q_splits;
  const int64_t sq = (int64_t)p.B * p.Hq * p.NqP * EP;
  if (r0 >= rpp) return;
  float2 tbv[4];
  if (d < R) {
#pragma unroll
    for (int t = 0; t < 4; ++t) tbv[t] = bq[d + t];
  }
#pragma unroll 2
  for (int r = r0; r < qrows; r += rpp) {
    const int i = q0 + r;
    if (i >= p.Nq) break;
    const float* u = wrow + (int64_t)i * EP;
    float g[4];
    if (d < R) {   // R % 4 == 0: all four dims rotated
      float x[4];
      load4<T>(qb + (int64_t)i * p.q_s[2] + d, x);
      const float4 f01 = *reinterpret_cast<const float4*>(tq + (int64_t)(q_off + i) * R + d);
      const float4 f23 = *reinterpret_cast<const float4*>(tq + (int64_t)(q_off + i) * R + d + 2);
      const float4 uc = sum4(u + d, S, sq), us = sum4(u + R + d, S, sq);
      const float tc[4] = {f01.x, f01.z, f23.x, f23.z}, ts[4] = {f01.y, f01.w, f23.y, f23.w};
      const float ucv[4] = {uc.x, uc.y, uc.z, uc.w}, usv[4] = {us.x, us.y, us.z, us.w};
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        // cos / sin(F[q_off + i] - bias) from the tables of F and of the bias
        const float cs = fmaf(tc[t], tbv[t].x, ts[t] * tbv[t].y), sn = fmaf(ts[t], tbv[t].x, -tc[t] * tbv[t].y);
        g[t] = sigmoid_f(x[t]) * (cs * ucv[t] + sn * usv[t]);
        const float dph = softplus_f(x[t]) * (cs * usv[t] - sn * ucv[t]);
        if (qpb) qpb[(int64_t)i * R + d + t] = dph;
        else if (dfb) atomicAdd(dfb + (int64_t)(q_off + i) * p.df_s[2] + d + t, dph);
      }
    } else {
      const float4 us = sum4(u + R + d, S, sq);
      g[0] = us.x; g[1] = us.y; g[2] = us.z; g[3] = us.w;
    }
    store4<T>(dqb + (int64_t)i * p.dq_s[2] + d, g);
  }
}

}  // namespace

hipError_t launch_flash_chain(const FlashBwdParams& p, const char* name, bool keys, bool queries, int dtype, hipStream_t s) {
  const auto nkey = [&](int rows) { return keys ? ((p.Nk + rows - 1) / rows) * p.B * p.Hk : 0; };
  const auto nquery = [&](int rows) { return queries ? ((p.Nq + rows - 1) / rows) * p.B * p.Hq : 0; };
  // A block's rows come one after another, a memory latency and one per split each: 8 rows a block where
  // blocks of 32 leave the chip idle (8 heads of 413 rows, D 250, R 62: 28 -> 12.5 us).  Every key block
  // adds to the same dbias row, 10 ns apiece: 3,410 keys of 4 batches on one row took 15.5 us at 32 and
  // 31.8 at 8, 2,999 keys of one batch 19 and 25, so keys keep 32 beyond kBiasAdds of them.
  constexpr int kBiasAdds = 192;
  const bool few = nkey(32) + nquery(32) < 1024;
  const int64_t adds = p.dbias ? (int64_t)((p.Nk + 7) / 8) * p.B * (p.Hb > 1 ? 1 : p.Hk) : 0;
  const int krows = few && adds <= kBiasAdds ? 8 : 32, qrows = few ? 8 : 32;
  const int nk = nkey(krows);
  const dim3 grid(nk + nquery(qrows));
  return dtype == 2 ? launch_named(name, flash_chain_kernel<BF16>, grid, dim3(256), s, p, nk, krows, qrows)
                    : launch_named(name, flash_chain_kernel<F16>, grid, dim3(256), s, p, nk, krows, qrows);
}

}  // namespace pope
