// Flash attention backward, bf16 instances and the host side (kernels: flash_bwd.hpp).
#include <algorithm>
#include <cmath>

#include "flash_bwd.hpp"

namespace pope {

// How many workgroups share a job, and whether the chain rule runs in its own launch.
//
// A dK/dV job loops over the query heads of its group and the query steps, a dQ job over the key
// steps; one workgroup runs per CU.  With grouped heads, or few batches x heads, the longest jobs
// are longer than an even share of the work (per_cu) and CUs idle: 16 query heads on 4 kv heads,
// 2,999 tokens, D 128 run 96 dK/dV jobs of up to 188 steps unsplit, 499 us in flash_bwd.  Jobs split until
// the longest is about 1.2 even shares, or three 128-row steps where that is longer; the number of splits
// rounds up past a quarter, so a split can be as short as two steps.  (Measured 0.5, 0.65, 0.8, 1.0, 1.3
// shares: that case 238, 224, 237, 228, 228 us for kernel + merge; 4 heads x 2,048 tokens, D 64: 56, 56, 56,
// 49, 46 against 73 unsplit.)  The partial rows' traffic and the launch have to be worth it.
//
// A rotate dim that is no multiple of 32 takes the jobs' general epilogue, one wave at a time through
// LDS; where the raw rows are few, writing them and the separate chain-rule launch are faster.
FlashBwdSplit flash_bwd_split(int B, int Hq, int Hk, int Nq, int Nk, int R, int EP, int DV, bool causal) {
  const int job = bwd_job(EP, DV), bm = bwd_step(EP, DV);
  const auto up = [](int x, int m) { return (x + m - 1) / m; };
  // lengths of the longest jobs in 128-row steps of a dK/dV job (a dQ step does 0.8 of its products)
  const double unit = bm / 128.0;
  const double lk = (double)(Hq / Hk) * up(Nq, bm) * unit;
  const double lq = 0.8 * up(causal ? std::min(Nq, Nk) : Nk, bm) * unit;
  const double jobs_kv = (double)up(Nk, job) * B * Hk, jobs_q = (double)up(Nq, job) * B * Hq;
  const double per_cu = (causal ? 0.5 : 1.0) * (jobs_kv * lk + jobs_q * lq) / 256;
  const double goal = std::max(per_cu * 1.2, 3.0);
  const int kv = std::max(1, std::min(64, (int)std::ceil(lk / goal - 0.25)));
  const int q = std::max(1, std::min(64, (int)std::ceil(lq / goal - 0.25)));
  const double mb_k = 4e-6 * B * Hk * Nk * (EP + DV), mb_q = 4e-6 * B * Hq * Nq * EP;   // one partial, MB
  const auto cost_us = [&](int sk, int sq) { return 8 + 2 * (mb_k * sk + mb_q * sq) / 3; };   // written and read at 3 TB/s
  const double step_us = 4.5 * (EP + DV) / 160;
  const double gain_us = (std::max(std::max(lk, lq), per_cu) - std::max(std::max(lk / kv, lq / q), per_cu)) * step_us;
  if (gain_us >= 1.2 * cost_us(kv > 1 ? kv : 0, q > 1 ? q : 0)) return {kv, q, kv > 1, q > 1};
  if (R % 32 != 0 && cost_us(1, 1) < 14) return {1, 1, true, true};
  return {1, 1, false, false};
}

hipError_t launch_flash_bwd(const FlashBwdParams& p, int dtype, hipStream_t s) {
  return dtype == 2 ? flash_bwd_dispatch<BF16>(p, s) : launch_flash_bwd_f16(p, s);
}

hipError_t launch_flash_bwd_delta(const FlashBwdParams& p, int dtype, hipStream_t s) {
  const int64_t nrows = (int64_t)p.B * p.Hq * p.NqP;
  const dim3 grid((unsigned)((8 * nrows + 255) / 256));
  return dtype == 2 ? launch_named("flash_bwd_delta", bwd_delta_kernel<BF16>, grid, dim3(256), s, p)
                    : launch_named("flash_bwd_delta", bwd_delta_kernel<F16>, grid, dim3(256), s, p);
}

}  // namespace pope
