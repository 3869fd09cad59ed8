// Materialising PoPE polar transform on the device (gfx950): apply_pope_to_qk
// (pope.py:30-86) forward and backward.
//
//   q_hat[..., 2d]     = a_d cos(phi_d),  q_hat[..., 2d + 1] = a_d sin(phi_d)      d < R
//   q_hat[..., R + d]  = q_d                                                      d >= R
// with a = softplus(q) rounded to q's dtype (the reference applies F.softplus to the input
// tensor, pope.py:60, then multiplies by fp32 cos / sin, which promotes, :69-70), the query
// phase phi = F[q_off + i] (right-aligned rows, :64) and the key phase psi = fl(F[j] + bias[h])
// (the bias added in fp32 before cos / sin, :56).  Outputs are fp32 (B, H, N, D + R) rows.
//
// Backward, per rotated dim (g = the output gradient):
//   dq   = sigmoid(q) (cos phi g_2d + sin phi g_2d+1)          (in q's dtype)
//   dphi = a (cos phi g_2d+1 - sin phi g_2d)                    -> dfreqs rows, dbias (keys)
// Pass-through dims copy g.  dfreqs and dbias are fp32 and accumulated (atomics; dbias summed
// over the workgroup's rows first).
//
// Complex layout (return_complex, pope.py:49-51,66-67,74-75): rows of D (re, im) fp32 pairs, the
// memory layout of torch.polar's complex64 output.  The rotated dims are the same interleaved
// pairs; pass-through dim d is the pair (q_d, 0) at columns 2d, 2d + 1, and its gradient is
// sign(q_d) times the real part of the pair's gradient (torch.polar's backward for a possibly
// negative magnitude, which the reference's torch path differentiates).
//
// One thread per (row, 4 input dims); a workgroup covers 256 / (D / 4) rows at a time of one (batch,
// head), `iters` row groups one after another, so the dbias partial sums reduce in registers and LDS
// before one atomic per dim; both sides (q and k) in one launch.  Bound by HBM.  With one row group per
// workgroup the key side's 2,048 workgroups (2 x 8 heads x 2,048 rows, D 64, R 64) each added 64
// atomics to the same 512 floats: backward 2 x 21.7 us, now 17.9 for both; forward 2 x 8.9, now 12.3.
#include <type_traits>

#include "pope_common.hpp"
#include "pope_kernels.hpp"

namespace pope {

namespace {

constexpr int kThreads = 256;

template <typename T>
__device__ __forceinline__ void load4(const void* base, int64_t off, float* x) {
  if constexpr (std::is_same<T, float>::value) {
    const float4 v = *reinterpret_cast<const float4*>(static_cast<const float*>(base) + off);
    x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
  } else {
    const u32x2 w = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(base) + off);
    x[0] = T::to_float((uint16_t)(w[0] & 0xffffu));
    x[1] = T::to_float((uint16_t)(w[0] >> 16));
    x[2] = T::to_float((uint16_t)(w[1] & 0xffffu));
    x[3] = T::to_float((uint16_t)(w[1] >> 16));
  }
}

template <typename T>
__device__ __forceinline__ void store4(void* base, int64_t off, const float* x) {
  if constexpr (std::is_same<T, float>::value) {
    *reinterpret_cast<float4*>(static_cast<float*>(base) + off) = make_float4(x[0], x[1], x[2], x[3]);
  } else {
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(base) + off) = u32x2{T::pack2(x[0], x[1]), T::pack2(x[2], x[3])};
  }
}

// Rounds to T's precision (identity for fp32).
template <typename T>
__device__ __forceinline__ float round_to(float v) {
  if constexpr (std::is_same<T, float>::value) return v;
  else return T::to_float(T::bits(v));
}

struct Side {
  const void* x; int64_t xs0, xs1, xs2;   // q or k
  float* out;                             // (heads, N, D + R) fp32
  const float* gout;                      // its gradient (backward)
  void* dx; int64_t ds0, ds1, ds2;        // dq or dk (backward)
  int H, N, frow0, key;                   // heads, rows, first phase row, 1 = key side (bias)
};

// phases of the thread's 4 rotated dims
__device__ __forceinline__ void phases(const PolarParams& p, const Side& sd, int b, int h, int n, int d0, float* ph,
                                       int& frow) {
  frow = sd.frow0 + n;
  const float* f = p.freqs + (int64_t)b * p.f_s[0] + (int64_t)h * p.f_s[1] + (int64_t)frow * p.f_s[2] + d0;
#pragma unroll
  for (int t = 0; t < 4; ++t) ph[t] = f[t];
  if (sd.key) {
    const float* bb = p.bias + (int64_t)h * p.bias_sh + d0;
#pragma unroll
    for (int t = 0; t < 4; ++t) ph[t] = ph[t] + bb[t];
  }
}

struct Task {
  int u, r, rpb, b, h, bh, n0;   // 4-dim unit, row of a group, rows per group, head, first row
};
// The workgroup's side and rows: blocks [0, nq) the q side's, then the k side's.
__device__ __forceinline__ Task task_of(const PolarParams& p, const Side& sd, int blk, int iters) {
  Task t;
  const int U = p.D / 4;
  t.rpb = kThreads / U;
  t.u = threadIdx.x % U;
  t.r = threadIdx.x / U;
  const int per = (sd.N + t.rpb * iters - 1) / (t.rpb * iters);
  t.bh = blk / per;
  t.n0 = (blk % per) * t.rpb * iters;
  t.b = t.bh / sd.H;
  t.h = t.bh % sd.H;
  return t;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void polar_fwd_kernel(PolarParams p, Side sq, Side sk, int nq, int iters) {
  const bool key = (int)blockIdx.x >= nq;
  const Side& sd = key ? sk : sq;
  const Task t = task_of(p, sd, key ? (int)blockIdx.x - nq : (int)blockIdx.x, iters);
  const int d0 = 4 * t.u, E = p.cplx ? 2 * p.D : p.D + p.R;
  if (t.r >= t.rpb) return;
  for (int it = 0; it < iters; ++it) {
    const int n = t.n0 + it * t.rpb + t.r;
    if (n >= sd.N) return;
    float x[4];
    load4<T>(sd.x, (int64_t)t.b * sd.xs0 + (int64_t)t.h * sd.xs1 + (int64_t)n * sd.xs2 + d0, x);
    float* orow = sd.out + ((int64_t)t.bh * sd.N + n) * E;
    if (d0 < p.R) {
      float ph[4];
      int frow;
      phases(p, sd, t.b, t.h, n, d0, ph, frow);
      float o[8];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float sn, cs;
        sincos_acc(ph[c], &sn, &cs);
        const float a = round_to<T>(softplus_f(x[c]));
        o[2 * c] = a * cs;
        o[2 * c + 1] = a * sn;
      }
      *reinterpret_cast<float4*>(orow + 2 * d0) = make_float4(o[0], o[1], o[2], o[3]);
      *reinterpret_cast<float4*>(orow + 2 * d0 + 4) = make_float4(o[4], o[5], o[6], o[7]);
    } else if (p.cplx) {
      *reinterpret_cast<float4*>(orow + 2 * d0) = make_float4(x[0], 0.f, x[1], 0.f);
      *reinterpret_cast<float4*>(orow + 2 * d0 + 4) = make_float4(x[2], 0.f, x[3], 0.f);
    } else {
      *reinterpret_cast<float4*>(orow + p.R + d0) = make_float4(x[0], x[1], x[2], x[3]);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void polar_bwd_kernel(PolarParams p, Side sq, Side sk, int nq, int iters) {
  __shared__ float red[kThreads][4];
  const bool key = (int)blockIdx.x >= nq;
  const Side& sd = key ? sk : sq;
  const Task t = task_of(p, sd, key ? (int)blockIdx.x - nq : (int)blockIdx.x, iters);
  const int U = p.D / 4, d0 = 4 * t.u, E = p.cplx ? 2 * p.D : p.D + p.R;
  float dsum[4] = {0.f, 0.f, 0.f, 0.f};
  for (int it = 0; it < iters; ++it) {
    const int n = t.n0 + it * t.rpb + t.r;
    if (t.r >= t.rpb || n >= sd.N) break;
    float x[4];
    load4<T>(sd.x, (int64_t)t.b * sd.xs0 + (int64_t)t.h * sd.xs1 + (int64_t)n * sd.xs2 + d0, x);
    const float* grow = sd.gout + ((int64_t)t.bh * sd.N + n) * E;
    const int64_t doff = (int64_t)t.b * sd.ds0 + (int64_t)t.h * sd.ds1 + (int64_t)n * sd.ds2 + d0;
    float dx[4];
    if (d0 < p.R) {
      float ph[4], dph[4];
      int frow;
      phases(p, sd, t.b, t.h, n, d0, ph, frow);
      const float4 g0 = *reinterpret_cast<const float4*>(grow + 2 * d0);
      const float4 g1 = *reinterpret_cast<const float4*>(grow + 2 * d0 + 4);
      const float g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float sn, cs;
        sincos_acc(ph[c], &sn, &cs);
        const float a = round_to<T>(softplus_f(x[c]));
        dx[c] = sigmoid_f(x[c]) * (cs * g[2 * c] + sn * g[2 * c + 1]);
        dph[c] = a * (cs * g[2 * c + 1] - sn * g[2 * c]);
        dsum[c] += dph[c];
      }
      float* part = sd.key ? p.kpart : p.qpart;   // deterministic mode: written once, summed later
      if (part) {
        float* dst = part + (((int64_t)t.b * sd.H + t.h) * sd.N + n) * p.R + d0;
#pragma unroll
        for (int c = 0; c < 4; ++c) dst[c] = dph[c];
      } else if (p.dfreqs) {
        float* df = p.dfreqs + (int64_t)t.b * p.df_s[0] + (int64_t)t.h * p.df_s[1] + (int64_t)frow * p.df_s[2] + d0;
#pragma unroll
        for (int c = 0; c < 4; ++c) atomicAdd(df + c, dph[c]);
      }
    } else if (p.cplx) {
      // real parts of the (re, im) gradient pairs, times sign(x): the reference builds the pair
      // with torch.polar(x, 0) (pope.py:50-51), whose backward takes Re(g * conj(sgn(result)))
      const float4 g0 = *reinterpret_cast<const float4*>(grow + 2 * d0);
      const float4 g1 = *reinterpret_cast<const float4*>(grow + 2 * d0 + 4);
      const float gr[4] = {g0.x, g0.z, g1.x, g1.z};
#pragma unroll
      for (int c = 0; c < 4; ++c) dx[c] = x[c] > 0.f ? gr[c] : x[c] < 0.f ? -gr[c] : 0.f;
    } else {
      const float4 g = *reinterpret_cast<const float4*>(grow + p.R + d0);
      dx[0] = g.x; dx[1] = g.y; dx[2] = g.z; dx[3] = g.w;
    }
    store4<T>(sd.dx, doff, dx);
  }
  if (sd.key && p.dbias && !p.kpart) {   // sum the workgroup's rows per dim, one atomic per dim
#pragma unroll
    for (int c = 0; c < 4; ++c) red[threadIdx.x][c] = dsum[c];
    __syncthreads();
    if (t.r == 0 && d0 < p.R) {
      float s4[4] = {0.f, 0.f, 0.f, 0.f};
      for (int r2 = 0; r2 < t.rpb; ++r2)
#pragma unroll
        for (int c = 0; c < 4; ++c) s4[c] += red[r2 * U + t.u][c];
      float* db = p.dbias + (int64_t)t.h * p.bias_sh + d0;
#pragma unroll
      for (int c = 0; c < 4; ++c) atomicAdd(db + c, s4[c]);
    }
  }
}

template <typename T>
hipError_t launch_t(const PolarParams& p, bool bwd, hipStream_t s) {
  Side q{p.q, p.q_s[0], p.q_s[1], p.q_s[2], p.qh, p.gq, p.dq, p.dq_s[0], p.dq_s[1], p.dq_s[2],
         p.Hq, p.Nq, p.Nk - p.Nq, 0};
  Side k{p.k, p.k_s[0], p.k_s[1], p.k_s[2], p.kh, p.gk, p.dk, p.dk_s[0], p.dk_s[1], p.dk_s[2],
         p.Hk, p.Nk, 0, 1};
  const int rpb = kThreads / (p.D / 4);
  const auto blocks = [&](const Side& sd, int iters) {
    return (int64_t)((sd.N + rpb * iters - 1) / (rpb * iters)) * p.B * sd.H;
  };
  // row groups per workgroup: up to 8 while four workgroups per CU remain
  int iters = 1;
  while (iters < 8 && blocks(q, 2 * iters) + blocks(k, 2 * iters) >= 1024) iters *= 2;
  const int64_t nq = blocks(q, iters), nk = blocks(k, iters);
  if (nq + nk > INT32_MAX) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(nq + nk));
  if (bwd) return launch_named("polar_bwd", polar_bwd_kernel<T>, grid, dim3(kThreads), s, p, q, k, (int)nq, iters);
  return launch_named("polar_fwd", polar_fwd_kernel<T>, grid, dim3(kThreads), s, p, q, k, (int)nq, iters);
}

}  // namespace

hipError_t launch_polar(const PolarParams& p, int dtype, bool bwd, hipStream_t s) {
  if (dtype == 0) return launch_t<float>(p, bwd, s);
  if (dtype == 1) return launch_t<F16>(p, bwd, s);
  return launch_t<BF16>(p, bwd, s);
}

}  // namespace pope
