// fp32 -> fp16 conversion of the flash operands with their range check, one launch for q, k and v
// (gfx950).
//
// fp32 flash calls run on fp16 operands; a finite value beyond fp16's range must be reported, not
// become inf.  The conversion reads every element anyway, so the check rides along: a finite value
// beyond 65504 in magnitude (a little before the rounding reaches infinity, at 65520) sets the flag (one
// store by any lane that sees one; the flag may live in pinned host memory, where the caller reads it after
// an event).  As torch operators the check and the three casts were 22 launches and a readback in the
// middle of the call: 208-226 us by box for a (1, 8, 1024, 64) forward whose attention kernels take 25 us;
// with this launch of 6 us 43-49.
// Bound by HBM (6 bytes per element); at that size by its launch.
#include "pope_common.hpp"
#include "pope_kernels.hpp"

namespace pope {

namespace {

constexpr int kThreads = 256;

// Flat work items: VEC consecutive elements of one row, tensors one after another.
template <int VEC>
__global__ __launch_bounds__(kThreads) void cast_f16_kernel(CastParams p, float limit) {
  const int64_t step = (int64_t)gridDim.x * kThreads;
  bool bad = false;
  for (int64_t it = (int64_t)blockIdx.x * kThreads + threadIdx.x; it < p.items; it += step) {
    int64_t x = it;
    int t = 0;
    while (t + 1 < p.n && x >= p.t[t].items) x -= p.t[t++].items;
    const CastTensor& c = p.t[t];
    const int per = c.shape[3] / VEC;
    const int d = (int)(x % per) * VEC;
    int64_t r = x / per;
    const int n = (int)(r % c.shape[2]);
    r /= c.shape[2];
    const int h = (int)(r % c.shape[1]), b = (int)(r / c.shape[1]);
    const float* src = c.src + b * c.src_s[0] + h * c.src_s[1] + n * c.src_s[2] + d * c.src_s[3];
    uint16_t* dst = c.dst + b * c.dst_s[0] + h * c.dst_s[1] + n * c.dst_s[2] + d * c.dst_s[3];
    if constexpr (VEC == 4) {
      const float4 v = *reinterpret_cast<const float4*>(src);
      bad |= (fabsf(v.x) > limit && fabsf(v.x) < INFINITY) | (fabsf(v.y) > limit && fabsf(v.y) < INFINITY) |
             (fabsf(v.z) > limit && fabsf(v.z) < INFINITY) | (fabsf(v.w) > limit && fabsf(v.w) < INFINITY);
      *reinterpret_cast<u32x2*>(dst) = u32x2{F16::pack2(v.x, v.y), F16::pack2(v.z, v.w)};
    } else {
      const float v = *src;
      bad |= fabsf(v) > limit && fabsf(v) < INFINITY;
      *dst = F16::bits(v);
    }
  }
  if (bad) *p.flag = 1u;
}

}  // namespace

hipError_t launch_cast_f16(const CastParams& p0, float limit, hipStream_t s) {
  CastParams p = p0;
  // 4 elements per access where every row of every tensor allows it: unit feature strides, 16-byte
  // source and 8-byte destination rows
  bool vec = true;
  for (int t = 0; t < p.n; ++t) {
    const CastTensor& c = p.t[t];
    vec = vec && c.shape[3] % 4 == 0 && c.src_s[3] == 1 && c.dst_s[3] == 1 &&
          reinterpret_cast<uintptr_t>(c.src) % 16 == 0 && reinterpret_cast<uintptr_t>(c.dst) % 8 == 0;
    for (int i = 0; i < 3; ++i) vec = vec && c.src_s[i] % 4 == 0 && c.dst_s[i] % 4 == 0;
  }
  p.items = 0;
  for (int t = 0; t < p.n; ++t) {
    p.t[t].items = (int64_t)p.t[t].shape[0] * p.t[t].shape[1] * p.t[t].shape[2] * p.t[t].shape[3] / (vec ? 4 : 1);
    p.items += p.t[t].items;
  }
  if (p.items == 0) return hipSuccess;
  const int64_t blocks = (p.items + kThreads - 1) / kThreads;
  const dim3 grid((unsigned)(blocks < 4096 ? blocks : 4096));
  return vec ? launch_named("cast_f16", cast_f16_kernel<4>, grid, dim3(kThreads), s, p, limit)
             : launch_named("cast_f16", cast_f16_kernel<1>, grid, dim3(kThreads), s, p, limit);
}

}  // namespace pope
