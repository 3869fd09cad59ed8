// Rows of head / rotate dims that are not multiples of 8, moved between the caller's width and the
// kernels' padded width, one launch for up to six tensors (gfx950).
//
//   pad    column c of a padded row: source column c below `split`, `fill` in the `gap` columns after
//          it, source column c - gap up to the real width, 0 beyond
//   unpad  the inverse selection (gradients and outputs of the real columns)
//
// As torch operators (slices, fills, concatenations and their backward) a padded training step was 20
// to 30 launches and 230-290 us on the host around 30-60 us of kernels; here it is one launch before
// the forward, one for dO and one for the gradients.  Bound by HBM: a thread moves eight columns of a
// row, element by element on the unaligned side and with 16-byte stores where the destination's rows
// allow it.
#include "pope_common.hpp"
#include "pope_kernels.hpp"

namespace pope {

namespace {

constexpr int kThreads = 256;

template <typename E>
__device__ __forceinline__ void move8(const PadTensor& c, int64_t src_off, int64_t dst_off, int c0) {
  const E* src = static_cast<const E*>(c.src) + src_off;
  E* dst = static_cast<E*>(c.dst) + dst_off + c0;
  const int real = c.pad ? c.gap + c.cols : c.cols;   // columns at or past it are zero
  alignas(16) E v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int x = c0 + j;
    E e = (E)0;
    if (c.pad && x >= c.split && x < c.split + c.gap) e = (E)c.fill;
    else if (x < real) e = src[(int64_t)(x < c.split ? x : c.pad ? x - c.gap : x + c.gap) * c.src_s[3]];
    v[j] = e;
  }
  if (c.vec) {
    constexpr int N = sizeof(E) * 8 / 16;
    const u32x4* w = reinterpret_cast<const u32x4*>(v);
#pragma unroll
    for (int i = 0; i < N; ++i) reinterpret_cast<u32x4*>(dst)[i] = w[i];
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (c0 + j < c.dst_cols) dst[j] = v[j];
  }
}

// Flat work items: eight destination columns of one row, tensors one after another.
template <typename I>
__global__ __launch_bounds__(kThreads) void pad_rows_kernel(PadParams p) {
  const I step = (I)gridDim.x * kThreads;
  for (I it = (I)blockIdx.x * kThreads + threadIdx.x; it < (I)p.items; it += step) {
    I x = it;
    int t = 0;
    while (t + 1 < p.n && x >= (I)p.t[t].items) x -= (I)p.t[t++].items;
    const PadTensor& c = p.t[t];
    const I per = (I)((c.dst_cols + 7) / 8);
    const int c0 = 8 * (int)(x % per);
    I r = x / per;
    const int64_t n = (int64_t)(r % (I)c.shape[2]);
    r /= (I)c.shape[2];
    const int64_t h = (int64_t)(r % (I)c.shape[1]), b = (int64_t)(r / (I)c.shape[1]);
    const int64_t so = b * c.src_s[0] + h * c.src_s[1] + n * c.src_s[2];
    const int64_t d_o = b * c.dst_s[0] + h * c.dst_s[1] + n * c.dst_s[2];
    if (c.elem == 2) move8<uint16_t>(c, so, d_o, c0);
    else move8<uint32_t>(c, so, d_o, c0);
  }
}

}  // namespace

hipError_t launch_pad_rows(const PadParams& p0, hipStream_t s) {
  PadParams p = p0;
  p.items = 0;
  for (int t = 0; t < p.n; ++t) {
    PadTensor& c = p.t[t];
    c.vec = c.dst_cols % 8 == 0 && reinterpret_cast<uintptr_t>(c.dst) % 16 == 0;
    for (int i = 0; i < 3; ++i) c.vec = c.vec && c.dst_s[i] * c.elem % 16 == 0;
    c.items = (int64_t)c.shape[0] * c.shape[1] * c.shape[2] * ((c.dst_cols + 7) / 8);
    p.items += c.items;
  }
  if (p.items == 0) return hipSuccess;
  const int64_t blocks = (p.items + kThreads - 1) / kThreads;
  const dim3 grid((unsigned)(blocks < 16384 ? blocks : 16384));
  // 32-bit indexes leave room for one more grid's step past the last item
  return p.items < ((int64_t)1 << 31) ? launch_named("pad_rows", pad_rows_kernel<uint32_t>, grid, dim3(kThreads), s, p)
                                      : launch_named("pad_rows", pad_rows_kernel<uint64_t>, grid, dim3(kThreads), s, p);
}

}  // namespace pope
