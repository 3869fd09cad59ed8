// Flash attention with PoPE for wide heads: head dims of 136 to 256 (after padding to a multiple
// of 8), expanded rows up to 512 features (gfx950, bf16 / fp16 MFMA).
//
// Reference semantics: triton_pope_flash_attn.py:23-117 (forward), :119-218 (backward), whose
// Triton kernels take any head dim (BD = next_pow2(D), :252-254); PyTorch path
// attention.py:106-145.
//
// The rows of these heads do not fit the register tiling of flash_fwd.hip / flash_bwd.hip (the
// backward's dK_hat accumulator alone is 256 registers per lane at E = 512), so the wide path
// trades speed for a plain structure: four waves per workgroup (one per SIMD, up to 512
// registers), 32 rows per wave, the backward's accumulators split into as few column chunks as the
// registers allow (each chunk recomputes the scores; the other waves take neighbouring row blocks),
// tiles shared by the four waves through LDS, and the polar transform's chain rule in a separate
// pass.  The streamed tiles go straight from global memory into LDS (global_load_lds_dwordx4) in
// three slots, two steps ahead of the step computed: a step's products take less time than the
// tile's fetch, and tiles staged through registers would hold registers these kernels do not
// have.  Each step's operand reads run as one ring over its products, with the addresses formed by an
// exclusive or from one base per tile, masks are applied on a side branch, and a head's jobs stay on
// one XCD.  What bounds the kernels: one operand read from LDS per product (1 KB per 32 cycles and
// SIMD), and the softmax of a wave's only row block, which nothing overlaps.  At (2, 8, 2048, 256),
// R 256, causal bf16 (two chunks): forward 205 -> 144 us, dK/dV 649 -> 168 (921 TFLOP/s of products),
// dQ 510 -> 167; before, every product group waited on reloads of spilled registers behind tile
// loads that missed the XCD's L2.
// Memory stays linear in the sequence length: no score matrix is stored.  Same workspace preparation as the narrow path
// (flash_prep.hip: K_hat, Q_hat pre-scaled by softmax_scale * log2 e, key visibility words,
// phase tables), with EP = E rounded up to 128 and DV = 256.
//   wide_fwd   one workgroup per (128 queries, batch * head): S^T = K_hat Q_hat^T, online softmax
//              in log2 units, O^T += V^T P^T with V read transposed (ds_read_b64_tr_b16); the
//              K_hat and V tiles of 32 keys streamed through LDS.
//   wide_kv    one workgroup per (key blocks, batch * kv head), wave = (32 keys, column chunk): S = Q_hat K_hat^T
//              - lse, dP = dO V^T - delta (Q_hat and dO tiles and the row terms streamed through
//              LDS), P = exp2 S,
//              dS = P dP; dV (the wave's chunk of D columns) += P^T dO and dK_hat (its chunk of E
//              columns) += dS^T Q_hat; writes dV and the raw dK_hat chunk (fp32 workspace).
//   wide_q     one workgroup per (query blocks, batch * head), wave = (32 queries, column chunk): S^T, dP^T with
//              the K_hat and V tiles in LDS, dQ_hat^T (its chunk) += K_hat^T dS^T; writes the raw
//              dQ_hat chunk.
//   flash_chain (flash_chain.hip) the chain rule of the polar transform from the raw rows: dk, dq,
//              dfreqs, dbias (deterministic mode: the per-row phase derivatives).
#include <algorithm>

#include "pope_common.hpp"
#include "pope_kernels.hpp"

namespace pope {

namespace {


__device__ __forceinline__ u32x4 ld16(const uint16_t* p) { return *reinterpret_cast<const u32x4*>(p); }
__device__ __forceinline__ u32x4 zero4() { return u32x4{0u, 0u, 0u, 0u}; }

typedef const __attribute__((address_space(4))) uint64_t cu64;
typedef const __attribute__((address_space(4))) int ci32;

// Registers [8 g, 8 g + 8) of an MFMA result, packed as an 8-element operand.
template <typename T>
__device__ __forceinline__ u32x4 pack8w(const f32x16& x, int g) {
  u32x4 w;
#pragma unroll
  for (int s = 0; s < 4; ++s) w[s] = T::pack2(x[8 * g + 2 * s], x[8 * g + 2 * s + 1]);
  return w;
}

__device__ __forceinline__ f32x16 splat16(float x) {
  f32x16 c;
#pragma unroll
  for (int r = 0; r < 16; ++r) c[r] = x;
  return c;
}

// Row offset within a 32-row block of register r of a 32x32 MFMA result in lane half hf.
__device__ __forceinline__ int res_row(int r, int hf) { return 8 * (r >> 2) + 4 * hf + (r & 3); }

// Growth of a row's running max (log2 units) that the forward absorbs without rescaling its
// accumulators: probabilities reach at most 2^lazy_max.  None at 512 features: the row's largest
// probability is exactly 1 there and adds no 16-bit rounding of its own (o's error against 64 bits
// 0.00239, with a growth of 8 absorbed 0.00241; the forward of the header's case 144 us against 117).
template <int EP>
constexpr float lazy_max() { return EP < 512 ? 8.f : 0.f; }

// LDS slots of the streamed tiles: tile t is computed from slot t % kSlots while tiles t + 1 and
// t + 2 load, so each tile has two steps of compute to arrive in.
constexpr int kSlots = 3;

// Job of a workgroup: (block, head) of nb blocks per head and `heads` heads.  Workgroup ids go
// round-robin over the 8 XCDs, each with its own 4 MB L2, and one head's streamed tiles are 3 MB at
// N 2048: where the heads divide over the XCDs, an XCD takes its heads one after the other, heaviest
// blocks first.  Otherwise the head index is fastest, so that a head stays on few XCDs.
__device__ __forceinline__ int2 wide_job(int id, int nb, int heads) {
  if (heads % 8 == 0) return make_int2(id / 8 % nb, id % 8 + 8 * (id / 8 / nb));
  return make_int2(id / heads, id % heads);
}

// Direct global -> LDS fill of one tile of 32 rows x U 16-byte units, stored unpadded with
// tile_swz (unit u of row r at position u ^ tile_swz(U, r)).  Load i of the thread fills position
// c = 64 (wave + 4 i) + lane (a wave's 64 lanes write 64 consecutive positions), in row c / U, with
// unit (c % U) ^ tile_swz(U, c / U) of that row.
//   dense rows of 8 U elements; U = 64: one row per wave load, so the row is scalar
template <int U>
__device__ __forceinline__ void fill_dense(uint32_t tile, int wave, int lane, const uint16_t* rows) {
  static_assert(32 * U % 256 == 0, "whole loads per thread");
#pragma unroll
  for (int i = 0; i < 32 * U / 256; ++i) {
    const int w = wave + 4 * i;
    if constexpr (U == 64) {
      load_lds16(rows + w * 8 * U, 16 * (lane ^ tile_swz(U, w)), tile + 1024 * w);
    } else {
      const int c = 64 * w + lane, r = c / U;
      load_lds16(rows, 16 * (r * U + ((c % U) ^ tile_swz(U, r))), tile + 1024 * w);
    }
  }
}
//   rows of a strided tensor from its row 0 of the tile: rows at or past `left` repeat the last one,
//   units at or past D the row's last unit
template <int U>
__device__ __forceinline__ void fill_strided(uint32_t tile, int wave, int lane, const uint16_t* rows, uint32_t row_bytes,
                                             int left, int D) {
  static_assert(64 % U == 0, "whole rows per wave load");
#pragma unroll
  for (int i = 0; i < 32 * U / 256; ++i) {
    const int w = wave + 4 * i, r = w * (64 / U) + lane / U;
    const uint32_t col = 2 * min(8 * ((lane % U) ^ tile_swz(U, r)), D - 8);
    load_lds16(rows, (uint32_t)min(r, left - 1) * row_bytes + col, tile + 1024 * w);
  }
}

// LDS byte addresses of a tile's operand reads, from one row-read and one transpose-read base per
// lane: with U % 16 == 0 and tiles on 256-byte boundaries, the swizzle turns the k step or column
// block within 256 bytes into an exclusive or on the base (TileOffsets has the layout).  The bases
// are opaque per step, so a step holds these two registers per tile and not one per address.
template <int U>
struct WideAddr {
  static_assert(U % 16 == 0, "rows of whole 256-byte groups");
  uint32_t row, tr;
  static __device__ __forceinline__ uint32_t lane_row(int lane) {
    const int lr = lane & 31, hf = lane >> 5;
    return 16 * (lr * U + (hf ^ tile_swz(U, lr)));
  }
  // of column blocks CH nb + ec
  static __device__ __forceinline__ uint32_t lane_tr(int lane, int ec) {
    const int j = lane & 15, hf = lane >> 5, u = 2 * ((lane >> 4) & 1) + ((j >> 1) & 1), r = 4 * hf + (j >> 2);
    return 16 * (r * U + ((u ^ tile_swz(U, r)) ^ (4 * ec))) + 8 * (j & 1);
  }
  __device__ __forceinline__ WideAddr(uint32_t tile, uint32_t lrow, uint32_t ltr)
      : row(opaque_u32(tile + lrow)), tr(opaque_u32(tile + ltr)) {}
  __device__ __forceinline__ u32x4 row_at(int kk) const { return lds_read16_at((row ^ (32 * (kk % 8))) + 256 * (kk / 8)); }
  // rows 16 g + (4 hf .. + 3) and + 8 of column block nb of the lane's chunk
  template <int CH>
  __device__ __forceinline__ u32x4 tr_at(int x, int g) const {
    const uint32_t nb = CH * x, o = 256 * (nb / 4) + 256 * U * g, lo = 64 * (nb % 4);
    return lds_tr8_at((tr ^ lo) + o, (tr ^ (lo ^ 32)) + o + 128 * U);
  }
};

// Operand reads kept in flight ahead of the product that takes them: as many of eight as leave the
// kernel's loop without spills (a reload waits for every tile load in flight behind it).
template <int EP>
constexpr int fwd_ring() { return EP >= 512 ? 6 : 8; }
constexpr int kKvRing = 4, kQRing = 8;

// ---- forward ---------------------------------------------------------------------------
// Four waves per workgroup, 128 query rows (wave w: rows q0 + 32 w ..); per 32-key tile the K_hat
// rows and the V rows go straight from global memory into LDS once for the four waves (unpadded,
// XOR-swizzled), in three slots: the loads of the next two tiles are in flight while the current
// tile is computed.
// SPLIT: one split of the key axis per workgroup, fp32 partials (as in flash_fwd.hip).
template <typename T, int EP, int DV, bool SPLIT>
__global__ __launch_bounds__(256) void wide_fwd_kernel(FlashFwdParams p) {
  constexpr int KS = EP / 16, NDB = DV / 32, kRing = fwd_ring<EP>();
  constexpr int KU = EP / 8, VU = DV / 8;              // 16-byte units per K_hat / V row
  constexpr int NL = 32 * (KU + VU) / 256;             // loads per thread and tile
  constexpr uint32_t KT = 64 * EP, SLOT = 64 * (EP + DV);   // bytes of the K_hat tile and of a slot
  typedef typename T::vec8 vec8;
  __shared__ __attribute__((aligned(256))) char smem[kSlots * SLOT];

  const int tid = threadIdx.x, wave = wave_id(), lane = tid & 63, lr = lane & 31, hf = lane >> 5;
  const int BH = p.B * p.Hq, nqb = (p.Nq + 127) / 128, splits = SPLIT ? p.splits : 1;
  const int2 job = wide_job(blockIdx.x, nqb * splits, BH);
  const int bh = job.y, sp = SPLIT ? job.x % splits : 0;
  const int q0 = 128 * (nqb - 1 - (SPLIT ? job.x / splits : job.x));   // heaviest causal blocks first
  const int b = bh / p.Hq, h = bh % p.Hq, hk = h % p.Hk;
  const int Nk = p.Nk, D = p.D, qw = q0 + 32 * wave, qi = qw + lr;

  int nkeys = min(((ci32*)p.kend)[b], Nk);
  if (p.causal) nkeys = min(nkeys, q0 + 128);
  const int t0 = SPLIT ? sp * (p.split_keys / 32) : 0;   // the workgroup's first tile
  if (SPLIT) nkeys = min(nkeys, (sp + 1) * p.split_keys);
  const uint16_t* khb = p.kh + (int64_t)(b * p.Hk + hk) * p.NkP * EP;   // rows padded to NkP
  const uint16_t* vb = p.v + (int64_t)b * p.v_s[0] + (int64_t)hk * p.v_s[1];
  cu64* mw = (cu64*)p.mwords + (int64_t)b * p.NW;
  const uint32_t lds0 = lds_addr(smem);
  const uint32_t krow = WideAddr<KU>::lane_row(lane), vtr = WideAddr<VU>::lane_tr(lane, 0);
  const uint32_t v_row = 2 * (uint32_t)p.v_s[2];

  // tile t into slot t % kSlots: K_hat rows are padded to NkP (no clamp); V rows past Nk repeat
  // the last one and V units at or past D repeat the row's last unit (they only reach the O rows
  // at or past D, which are not stored)
  auto issue = [&](int t) {
    const int j0 = 32 * (t0 + t);
    const uint32_t slot = lds0 + (t % kSlots) * SLOT;
    fill_dense<KU>(slot, wave, lane, khb + (int64_t)j0 * EP);
    fill_strided<VU>(slot + KT, wave, lane, vb + (int64_t)j0 * p.v_s[2], v_row, Nk - j0, D);
  };
  const int nt = max((nkeys + 31) / 32 - t0, 0);
  if (nt > 0) issue(0);
  if (nt > 1) issue(1);

  vec8 qreg[KS];
  {
    const uint16_t* qrow = p.qh + ((int64_t)bh * p.NqP + qi) * EP + 8 * hf;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) qreg[kk] = as_vec8<vec8>(ld16(qrow + 16 * kk));
  }
  // the Q_hat rows as loads the compiler sees complete: no use of them in the loop waits on the
  // tile loads in flight there
  settle_vector_loads();

  f32x16 oacc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) oacc[db] = splat16(0.f);
  float m = -INFINITY, l = 0.f;   // l: the lane half's share of the row sum
  const uint32_t ones = T::pack2(1.f, 1.f);
  uint32_t word = nt > 0 ? (uint32_t)(mw[t0 >> 1] >> (32 * (t0 & 1))) : 0u;   // visibility of the step's keys
  for (int t = 0; t < nt; ++t) {
    const int j0 = 32 * (t0 + t);
    if (t + 1 < nt) wait_vmcnt<NL>();   // this thread's loads of tile t landed (t + 1 may be in flight)
    else wait_vmcnt<0>();
    __syncthreads();                    // ... everyone's; and slot (t + 2) % kSlots was last read in step t - 1
    if (t + 2 < nt) issue(t + 2);
    const uint32_t wv = word;
    if (t + 1 < nt) word = (uint32_t)(mw[(t0 + t + 1) >> 1] >> (32 * ((t0 + t + 1) & 1)));
    const uint32_t slot = lds0 + (t % kSlots) * SLOT;
    const WideAddr<KU> ka(slot, krow, 0);
    const WideAddr<VU> va(slot + KT, 0, vtr);
    // one ring of operand reads over both products: S^T = K_hat Q_hat^T (rows = keys, lane = query,
    // log2 units), then O^T += V^T P^T; the first V operands arrive during the softmax
    constexpr int NP = KS + 2 * NDB;
    u32x4 f[kRing];
    auto operand = [&](int i) { return i < KS ? ka.row_at(i) : va.template tr_at<1>((i - KS) % NDB, (i - KS) / NDB); };
#pragma unroll
    for (int i = 0; i < kRing; ++i) f[i] = operand(i);
    __builtin_amdgcn_sched_barrier(0);
    f32x16 s = splat16(0.f);
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      s = T::mfma32(as_vec8<vec8>(f[i % kRing]), qreg[i], s);
      f[i % kRing] = operand(i + kRing);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (wv != 0xffffffffu || (p.causal && j0 + 31 > qw)) {   // a masked key, or the causal diagonal
      POPE_COLD_PATH();
      const int lim = qi - j0 - 4 * hf;   // causal: row offset <= lim
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kr_ = 8 * (r >> 2) + (r & 3);
        s[r] = ((wv >> (4 * hf + kr_)) & 1u) && (!p.causal || kr_ <= lim) ? s[r] : -INFINITY;
      }
    }
    float mt = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mt = fmaxf(mt, s[r]);
    mt = half_swap_max(mt);
    // lazy rescale: a row's reference max m moves only when the tile's max exceeds it by more than
    // lazy_max (log2 units), so the probabilities stay below 2^lazy_max and most steps skip
    // rescaling the O accumulators (the branch is taken when any row of the wave moves)
    const bool grow = mt > m + lazy_max<EP>();
    if (__ballot(grow)) {
      POPE_COLD_PATH();
      const float mn = grow ? mt : m;
      const float alpha = __builtin_amdgcn_exp2f(m - (mn == -INFINITY ? 0.f : mn));
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
      l *= alpha;
      m = mn;
    }
    const float mu = m == -INFINITY ? 0.f : m;
    u32x4 pw[2];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t w = T::pack2(__builtin_amdgcn_exp2f(s[8 * g + 2 * q] - mu),
                                    __builtin_amdgcn_exp2f(s[8 * g + 2 * q + 1] - mu));
        pw[g][q] = w;
        l = T::dot2(w, ones, l);   // the row sum of the probabilities the products use
      }
#pragma unroll
    for (int i = KS; i < NP; ++i) {
      const int db = (i - KS) % NDB;
      oacc[db] = T::mfma32(as_vec8<vec8>(f[i % kRing]), as_vec8<vec8>(pw[(i - KS) / NDB]), oacc[db]);
      if (i + kRing < NP) f[i % kRing] = operand(i + kRing);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  l += __shfl_xor(l, 32, 64);
  if (qi >= p.Nq) return;
  if constexpr (SPLIT) {
    const int64_t prow = (((int64_t)b * p.Hq + h) * p.Nq + qi) * p.splits + sp;
    float* po = p.part_o + prow * D;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d0 = 32 * db + 8 * g + 4 * hf;
        if (d0 < D)
          *reinterpret_cast<float4*>(po + d0) = make_float4(oacc[db][4 * g], oacc[db][4 * g + 1], oacc[db][4 * g + 2],
                                                            oacc[db][4 * g + 3]);
      }
    if (hf == 0) *reinterpret_cast<float2*>(p.part_ml + 2 * prow) = make_float2(m, l);
    return;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  uint16_t* orow = p.o + (int64_t)b * p.o_s[0] + (int64_t)h * p.o_s[1] + (int64_t)qi * p.o_s[2];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * db + 8 * g + 4 * hf;
      if (d0 < D) {
        u32x2 w;
        w[0] = T::pack2(oacc[db][4 * g] * inv, oacc[db][4 * g + 1] * inv);
        w[1] = T::pack2(oacc[db][4 * g + 2] * inv, oacc[db][4 * g + 3] * inv);
        *reinterpret_cast<u32x2*>(orow + d0) = w;
      }
    }
  if (hf == 0)
    p.lse[((int64_t)b * p.Hq + h) * p.Nq + qi] = m == -INFINITY ? -INFINITY : (m + __builtin_amdgcn_logf(l)) * kLn2;
}

// ---- backward: dK_hat / dV --------------------------------------------------------------
// One workgroup per (4 / CH blocks of 32 keys, batch * kv head); wave w takes key block w / CH and
// column chunk w % CH of the accumulators (CH chunks recompute the scores CH times; fewer where the
// registers allow).  The Q_hat and dO tiles of each 32-query step go straight from global memory
// into LDS once for the four waves, in three slots (two steps ahead of the step computed), with
// the step's -lse and -delta rows (one more load, wave 0).
// SPLIT: the workgroup takes one of kv_splits shares of the steps and leaves raw dV rows too (a run-time
// split count cost the unsplit kernels 5%).
template <typename T, int EP, int DV, int CH, bool SPLIT>
__global__ __launch_bounds__(256) void wide_kv_kernel(FlashBwdParams p) {
  constexpr int KS = EP / 16, DS = DV / 16, EBC = EP / 32 / CH, DBC = DV / 32 / CH, RB = 4 / CH;
  constexpr int QU = EP / 8, OU = DV / 8, NL = 32 * (QU + OU) / 256;
  constexpr uint32_t QT = 64 * EP, RT = 64 * (EP + DV), SLOT = RT + 1024;   // byte offsets in a slot: dO tile, row terms
  typedef typename T::vec8 vec8;
  __shared__ __attribute__((aligned(256))) char smem[kSlots * SLOT];

  const int tid = threadIdx.x, wave = wave_id(), lane = tid & 63, lr = lane & 31, hf = lane >> 5;
  const int nkb = p.NkP / (32 * RB);
  const int ec = wave % CH;   // the wave's column chunk
  const int S = SPLIT ? p.kv_splits : 1;
  const int2 job = wide_job(blockIdx.x, nkb * S, p.B * p.Hk);
  const int kb0 = 32 * RB * (SPLIT ? job.x / S : job.x), bhk = job.y;   // key block 0 (the heaviest causal one) first
  const int sp = SPLIT ? job.x % S : 0;
  const int k0 = kb0 + 32 * (wave / CH);   // the wave's keys
  const int b = bhk / p.Hk, hk = bhk % p.Hk;
  const int Nk = p.Nk, Nq = p.Nq, D = p.D, NqP = p.NqP;
  if (kb0 >= Nk) return;
  const int kj = k0 + lr;
  cu64* mw = (cu64*)p.mwords + (int64_t)b * p.NW;
  const bool kvis = kj < Nk && ((mw[kj >> 6] >> (kj & 63)) & 1ull);

  // the steps: (query head g of the kv head's group, 32-query block q0), flattened
  const int groups = p.Hq / p.Hk;
  const int qstart = p.causal ? kb0 : 0;   // the workgroup's first key block
  const int nsq = Nq > qstart ? (Nq - qstart + 31) / 32 : 0;
  const int nall = __syncthreads_or(kvis) ? groups * nsq : 0;   // uniform over the workgroup
  // the workgroup's share of the steps (split sp of kv_splits)
  const int st_lo = SPLIT ? (int)((int64_t)nall * sp / S) : 0;
  const int nsteps = SPLIT ? (int)((int64_t)nall * (sp + 1) / S) - st_lo : nall;
  const uint32_t lds0 = lds_addr(smem), do_row = 2 * (uint32_t)p.do_s[2];
  // the next step's tiles into the next slot: Q_hat rows padded to NqP (no clamp); dO rows past Nq
  // repeat the last one and dO units at or past D repeat the row's last unit (they meet zero V
  // columns in dP and reach only the dV columns at or past D, which are not stored)
  const int q_first = SPLIT && nall > 0 ? qstart + 32 * (st_lo % nsq) : qstart;
  int ih = hk + (SPLIT && nall > 0 ? p.Hk * (st_lo / nsq) : 0), iq = q_first, islot = 0;
  auto issue = [&]() {
    const uint32_t slot = lds0 + islot * SLOT;
    const int64_t row = (int64_t)(b * p.Hq + ih) * NqP + iq;
    fill_dense<QU>(slot, wave, lane, p.qh + row * EP);
    fill_strided<OU>(slot + QT, wave, lane,
                     p.dout + (int64_t)b * p.do_s[0] + (int64_t)ih * p.do_s[1] + (int64_t)iq * p.do_s[2], do_row, Nq - iq, D);
    // the row terms of the step's queries: lane units 0-7 -lse, 8-15 -delta (lanes past 15 repeat
    // them past float 64, unread)
    if (wave == 0) {
      const int u = lane & 15;
      load_lds16((u < 8 ? p.nl : p.nd) + row + 4 * (u & 7), slot + RT);
    }
    iq += 32;
    if (iq >= Nq) {
      iq = qstart;
      ih += p.Hk;
    }
    islot = islot == kSlots - 1 ? 0 : islot + 1;
  };
  if (nsteps > 0) issue();
  if (nsteps > 1) issue();

  vec8 kreg[KS], vreg[DS];
  {
    const uint16_t* khr = p.kh + ((int64_t)bhk * p.NkP + kj) * EP + 8 * hf;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) kreg[kk] = as_vec8<vec8>(ld16(khr + 16 * kk));
    const uint16_t* vr = p.v + (int64_t)b * p.v_s[0] + (int64_t)hk * p.v_s[1] + (int64_t)min(kj, Nk - 1) * p.v_s[2];
#pragma unroll
    for (int kk = 0; kk < DS; ++kk) {
      const int d0 = 16 * kk + 8 * hf;
      const u32x4 x = ld16(vr + min(d0, D - 8));   // no branch: a valid address always, the value selected
      vreg[kk] = as_vec8<vec8>((kj < Nk && d0 < D) ? x : zero4());
    }
  }
  // the K_hat / V rows as loads the compiler sees complete: no use of them in the loop waits on
  // the tile loads in flight there
  settle_vector_loads();
  f32x16 dka[EBC], dva[DBC];
#pragma unroll
  for (int x = 0; x < EBC; ++x) dka[x] = splat16(0.f);
#pragma unroll
  for (int x = 0; x < DBC; ++x) dva[x] = splat16(0.f);
  const uint32_t qrow = WideAddr<QU>::lane_row(lane), qtr = WideAddr<QU>::lane_tr(lane, ec);
  const uint32_t orow = WideAddr<OU>::lane_row(lane), otr = WideAddr<OU>::lane_tr(lane, ec);
  const bool wave_vis = __all(kvis);

  int q0 = q_first, buf = 0;
  for (int st = 0; st < nsteps; ++st) {
    // this thread's loads of step st landed (st + 1 may be in flight; wave 0 has one more per step)
    if (st + 1 < nsteps) {
      if (wave == 0) wait_vmcnt<NL + 1>();
      else wait_vmcnt<NL>();
    } else {
      wait_vmcnt<0>();
    }
    __syncthreads();                         // ... everyone's; and slot (st + 2) % kSlots was last read in step st - 1
    if (st + 2 < nsteps) issue();
    const uint32_t slot = lds0 + buf * SLOT;
    const WideAddr<QU> qa(slot, qrow, qtr);
    const WideAddr<OU> oa(slot + QT, orow, otr);
    // -lse and -delta of the result rows (queries q0 + res_row(r, hf); padded rows give P = 0)
    const uint32_t ra = slot + RT + 16 * hf;
    f32x16 s, dp;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 a = lds_read_f4_at(ra + 32 * q), c = lds_read_f4_at(ra + 128 + 32 * q);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        s[4 * q + x] = a[x];
        dp[4 * q + x] = c[x];
      }
    }
    // one ring of operand reads over the step's products: S = Q_hat K_hat^T - lse and
    // dP = dO V^T - delta (rows = queries, lane = key), then dV += P^T dO and dK_hat += dS^T Q_hat
    // by 16 queries; the first transposed operands arrive during the exponentials
    constexpr int N1 = KS + DS, NX = DBC + EBC, NP = N1 + 2 * NX;
    u32x4 f[kKvRing];
    auto operand = [&](int i) {
      if (i < KS) return qa.row_at(i);
      if (i < N1) return oa.row_at(i - KS);
      const int g = (i - N1) / NX, x = (i - N1) % NX;
      return x < DBC ? oa.template tr_at<CH>(x, g) : qa.template tr_at<CH>(x - DBC, g);
    };
#pragma unroll
    for (int i = 0; i < kKvRing; ++i) f[i] = operand(i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < N1; ++i) {
      if (i < KS) s = T::mfma32(as_vec8<vec8>(f[i % kKvRing]), kreg[i < KS ? i : 0], s);
      else dp = T::mfma32(as_vec8<vec8>(f[i % kKvRing]), vreg[i < KS ? 0 : i - KS], dp);
      f[i % kKvRing] = operand(i + kKvRing);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!wave_vis || (p.causal && q0 < k0 + 31)) {   // a masked key, or the causal diagonal
      POPE_COLD_PATH();
      const int lim = q0 + 4 * hf - kj;   // causal: row offset >= -lim
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[r] = (kvis && (!p.causal || 8 * (r >> 2) + (r & 3) + lim >= 0)) ? s[r] : -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float pv = __builtin_amdgcn_exp2f(s[r]);
      s[r] = pv;
      dp[r] = pv * dp[r];
    }
    vec8 ap[2], ads[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      ap[g] = as_vec8<vec8>(pack8w<T>(s, g));
      ads[g] = as_vec8<vec8>(pack8w<T>(dp, g));
    }
#pragma unroll
    for (int i = N1; i < NP; ++i) {
      const int g = (i - N1) / NX, x = (i - N1) % NX;
      if (x < DBC) dva[x < DBC ? x : 0] = T::mfma32(ap[g], as_vec8<vec8>(f[i % kKvRing]), dva[x < DBC ? x : 0]);
      else dka[x < DBC ? 0 : x - DBC] = T::mfma32(ads[g], as_vec8<vec8>(f[i % kKvRing]), dka[x < DBC ? 0 : x - DBC]);
      if (i + kKvRing < NP) f[i % kKvRing] = operand(i + kKvRing);
      __builtin_amdgcn_sched_barrier(0);
    }
    q0 += 32;
    if (q0 >= Nq) q0 = qstart;
    buf = buf == kSlots - 1 ? 0 : buf + 1;
  }
  // dV (lane = d column, registers = keys; a split's as raw fp32 rows); the raw dK_hat chunk, times
  // ln 2 (Q_hat carries log2 e)
  const int64_t row0 = ((int64_t)sp * p.B * p.Hk + bhk) * p.NkP;
  if constexpr (SPLIT) {
    float* wvb = p.wv + row0 * DV;
#pragma unroll
    for (int db = 0; db < DBC; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) wvb[(int64_t)(k0 + res_row(r, hf)) * DV + 32 * (CH * db + ec) + lr] = dva[db][r];
  } else {
    uint16_t* dvb = p.dv + (int64_t)b * p.dv_s[0] + (int64_t)hk * p.dv_s[1];
#pragma unroll
    for (int db = 0; db < DBC; ++db) {
      const int d = 32 * (CH * db + ec) + lr;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + res_row(r, hf);
        if (key < Nk && d < D) dvb[(int64_t)key * p.dv_s[2] + d] = T::bits(dva[db][r]);
      }
    }
  }
  float* wkb = p.wk + row0 * EP;
#pragma unroll
  for (int eb = 0; eb < EBC; ++eb) {
    const int e = 32 * (CH * eb + ec) + lr;
#pragma unroll
    for (int r = 0; r < 16; ++r) wkb[(int64_t)(k0 + res_row(r, hf)) * EP + e] = dka[eb][r] * kLn2;
  }
}

// ---- backward: dQ_hat -------------------------------------------------------------------
// One workgroup per (4 / CH blocks of 32 queries, batch * head); wave w takes query block w / CH
// and column chunk w % CH of the accumulator.  The K_hat and V tiles of each 32-key step go
// straight from global memory into LDS once for the four waves, in three slots (two steps ahead).
template <typename T, int EP, int DV, int CH, bool SPLIT>
__global__ __launch_bounds__(256) void wide_q_kernel(FlashBwdParams p) {
  constexpr int KS = EP / 16, DS = DV / 16, EBC = EP / 32 / CH, RB = 4 / CH;
  constexpr int KU = EP / 8, VU = DV / 8, NL = 32 * (KU + VU) / 256;
  constexpr uint32_t KT = 64 * EP, SLOT = 64 * (EP + DV);   // bytes of the K_hat tile and of a slot
  typedef typename T::vec8 vec8;
  __shared__ __attribute__((aligned(256))) char smem[kSlots * SLOT];

  const int tid = threadIdx.x, wave = wave_id(), lane = tid & 63, lr = lane & 31, hf = lane >> 5;
  const int nqb = p.NqP / (32 * RB);
  const int ec = wave % CH;   // the wave's column chunk
  const int S = SPLIT ? p.q_splits : 1;
  const int2 job = wide_job(blockIdx.x, nqb * S, p.B * p.Hq);
  const int qb0 = 32 * RB * (nqb - 1 - (SPLIT ? job.x / S : job.x)), bh = job.y;   // heaviest causal blocks first
  const int sp = SPLIT ? job.x % S : 0;
  const int q0 = qb0 + 32 * (wave / CH);   // the wave's queries
  const int b = bh / p.Hq, h = bh % p.Hq, hk = h % p.Hk;
  const int Nk = p.Nk, Nq = p.Nq, D = p.D;
  if (qb0 >= Nq) return;
  const int qi = q0 + lr;
  int nkeys = min(((ci32*)p.kend)[b], Nk);
  if (p.causal) nkeys = min(nkeys, qb0 + 32 * RB);   // the workgroup's last query block
  const uint16_t* khb = p.kh + (int64_t)(b * p.Hk + hk) * p.NkP * EP;   // rows padded to NkP
  const uint16_t* vb = p.v + (int64_t)b * p.v_s[0] + (int64_t)hk * p.v_s[1];
  // the workgroup's share of the tiles (split sp of q_splits): local tile t is tile t_lo + t
  const int nall = (nkeys + 31) / 32, t_lo = SPLIT ? (int)((int64_t)nall * sp / S) : 0;
  const int nt = SPLIT ? (int)((int64_t)nall * (sp + 1) / S) - t_lo : nall;
  const uint32_t lds0 = lds_addr(smem), v_row = 2 * (uint32_t)p.v_s[2];
  // tile t into slot t % kSlots: K_hat rows padded to NkP (no clamp); V rows past Nk repeat the
  // last one and V units at or past D repeat the row's last unit (they meet zero dO columns)
  auto issue = [&](int t) {
    const int j0 = 32 * (t_lo + t);
    const uint32_t slot = lds0 + (t % kSlots) * SLOT;
    fill_dense<KU>(slot, wave, lane, khb + (int64_t)j0 * EP);
    fill_strided<VU>(slot + KT, wave, lane, vb + (int64_t)j0 * p.v_s[2], v_row, Nk - j0, D);
  };
  if (nt > 0) issue(0);
  if (nt > 1) issue(1);

  vec8 qreg[KS], doreg[DS];
  {
    const uint16_t* qhr = p.qh + ((int64_t)bh * p.NqP + qi) * EP + 8 * hf;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) qreg[kk] = as_vec8<vec8>(ld16(qhr + 16 * kk));
    const uint16_t* dr = p.dout + (int64_t)b * p.do_s[0] + (int64_t)h * p.do_s[1] + (int64_t)min(qi, Nq - 1) * p.do_s[2];
#pragma unroll
    for (int kk = 0; kk < DS; ++kk) {
      const int d0 = 16 * kk + 8 * hf;
      const u32x4 x = ld16(dr + min(d0, D - 8));   // no branch: a valid address always, the value selected
      doreg[kk] = as_vec8<vec8>((qi < Nq && d0 < D) ? x : zero4());
    }
  }
  const float nls = p.nl[(int64_t)bh * p.NqP + qi], nds = p.nd[(int64_t)bh * p.NqP + qi];
  // the row loads as loads the compiler sees complete: no use of them in the loop waits on the
  // tile loads in flight there
  settle_vector_loads();
  f32x16 dqa[EBC];
#pragma unroll
  for (int x = 0; x < EBC; ++x) dqa[x] = splat16(0.f);
  cu64* mw = (cu64*)p.mwords + (int64_t)b * p.NW;
  const uint32_t krow = WideAddr<KU>::lane_row(lane), ktr = WideAddr<KU>::lane_tr(lane, ec);
  const uint32_t vrow = WideAddr<VU>::lane_row(lane);
  uint32_t word = nt > 0 ? (uint32_t)(mw[t_lo >> 1] >> (32 * (t_lo & 1))) : 0u;   // visibility of the step's keys
  for (int t = 0; t < nt; ++t) {
    const int j0 = 32 * (t_lo + t);
    if (t + 1 < nt) wait_vmcnt<NL>();   // this thread's loads of tile t landed (t + 1 may be in flight)
    else wait_vmcnt<0>();
    __syncthreads();                    // ... everyone's; and slot (t + 2) % kSlots was last read in step t - 1
    if (t + 2 < nt) issue(t + 2);
    const uint32_t wv = word;
    if (t + 1 < nt) word = (uint32_t)(mw[(t_lo + t + 1) >> 1] >> (32 * ((t_lo + t + 1) & 1)));
    const uint32_t slot = lds0 + (t % kSlots) * SLOT;
    const WideAddr<KU> ka(slot, krow, ktr);
    const WideAddr<VU> va(slot + KT, vrow, 0);
    // one ring of operand reads: S^T = K_hat Q_hat^T - lse and dP^T = V dO^T - delta (rows = keys,
    // lane = query), then dQ_hat^T += K_hat^T dS^T by 16 keys
    constexpr int N1 = KS + DS, NP = N1 + 2 * EBC;
    u32x4 f[kQRing];
    auto operand = [&](int i) {
      if (i < KS) return ka.row_at(i);
      if (i < N1) return va.row_at(i - KS);
      return ka.template tr_at<CH>((i - N1) % EBC, (i - N1) / EBC);
    };
#pragma unroll
    for (int i = 0; i < kQRing; ++i) f[i] = operand(i);
    __builtin_amdgcn_sched_barrier(0);
    f32x16 s = splat16(nls), dp = splat16(nds);
#pragma unroll
    for (int i = 0; i < N1; ++i) {
      if (i < KS) s = T::mfma32(as_vec8<vec8>(f[i % kQRing]), qreg[i < KS ? i : 0], s);
      else dp = T::mfma32(as_vec8<vec8>(f[i % kQRing]), doreg[i < KS ? 0 : i - KS], dp);
      f[i % kQRing] = operand(i + kQRing);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (wv != 0xffffffffu || (p.causal && j0 + 31 > q0)) {   // a masked key, or the causal diagonal
      POPE_COLD_PATH();
      const int lim = qi - j0 - 4 * hf;   // causal: row offset <= lim
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kr_ = 8 * (r >> 2) + (r & 3);
        s[r] = ((wv >> (4 * hf + kr_)) & 1u) && (!p.causal || kr_ <= lim) ? s[r] : -INFINITY;
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) dp[r] = __builtin_amdgcn_exp2f(s[r]) * dp[r];
    vec8 bds[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) bds[g] = as_vec8<vec8>(pack8w<T>(dp, g));
#pragma unroll
    for (int i = N1; i < NP; ++i) {
      const int g = (i - N1) / EBC, x = (i - N1) % EBC;
      dqa[x] = T::mfma32(as_vec8<vec8>(f[i % kQRing]), bds[g], dqa[x]);
      if (i + kQRing < NP) f[i % kQRing] = operand(i + kQRing);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the raw dQ_hat chunk (rows = e, lane = query), times softmax_scale
  float* wqb = p.wq + (((int64_t)sp * p.B * p.Hq + bh) * p.NqP + qi) * EP;
#pragma unroll
  for (int eb = 0; eb < EBC; ++eb)
#pragma unroll
    for (int r = 0; r < 16; ++r) wqb[32 * (CH * eb + ec) + res_row(r, hf)] = dqa[eb][r] * p.scale;
}

template <typename T, int EP, int DV>
hipError_t fwd_t(const FlashFwdParams& p, hipStream_t s) {
  const int blocks = ((p.Nq + 127) / 128) * p.B * p.Hq;
  if (p.splits > 1)
    return launch_named("flash_wide_fwd", wide_fwd_kernel<T, EP, DV, true>, dim3(blocks * p.splits), dim3(256), s, p);
  return launch_named("flash_wide_fwd", wide_fwd_kernel<T, EP, DV, false>, dim3(blocks), dim3(256), s, p);
}

// Column chunks per row block (each chunk recomputes the scores), as few as the registers hold: one
// at 256 features, two at 384 / 512.
constexpr int wide_chunks(int EP) { return EP <= 256 ? 1 : 2; }

template <typename T, int EP, int DV>
hipError_t bwd_t(const FlashBwdParams& p, hipStream_t s) {
  constexpr int CH = wide_chunks(EP);
  const dim3 gk((p.NkP / (128 / CH)) * p.B * p.Hk * p.kv_splits), gq((p.NqP / (128 / CH)) * p.B * p.Hq * p.q_splits);
  hipError_t e = p.kv_splits > 1 ? launch_named("flash_wide_kv", wide_kv_kernel<T, EP, DV, CH, true>, gk, dim3(256), s, p)
                                 : launch_named("flash_wide_kv", wide_kv_kernel<T, EP, DV, CH, false>, gk, dim3(256), s, p);
  if (e != hipSuccess) return e;
  e = p.q_splits > 1 ? launch_named("flash_wide_q", wide_q_kernel<T, EP, DV, CH, true>, gq, dim3(256), s, p)
                     : launch_named("flash_wide_q", wide_q_kernel<T, EP, DV, CH, false>, gq, dim3(256), s, p);
  if (e != hipSuccess) return e;
  FlashBwdParams c = p;   // both sides' raw rows; dV from the splits, or written already
  if (c.kv_splits == 1) c.wv = nullptr;
  return launch_flash_chain(c, "flash_wide_chain", true, true, T::kCode, s);
}

// Splits of n jobs with `steps` steps of 32 rows each (2.4 us a step) over the CUs they leave idle, one
// workgroup per CU, each split keeping kWideSplitSteps steps and the longest job losing kWideSplitGainUs
// (the chain rule reads a row per split).
constexpr int kWideSplitSteps = 4;
constexpr float kWideStepUs = 2.4f, kWideSplitGainUs = 8.f;
int wide_splits(int64_t n, int steps) {
  const int s = (int)std::min<int64_t>(256 / std::max<int64_t>(n, 1), steps / kWideSplitSteps);
  return s > 1 && (steps - (steps + s - 1) / s) * kWideStepUs >= kWideSplitGainUs ? s : 1;
}

}  // namespace

// Job splits of a wide backward (raw rows in any case: raw_kv and raw_q stay false).
FlashBwdSplit flash_wide_bwd_split(int B, int Hq, int Hk, int Nq, int Nk, int EP, bool causal) {
  const int rows = 128 / wide_chunks(EP);   // per workgroup
  FlashBwdSplit r{1, 1, false, false};
  r.kv = wide_splits((int64_t)((Nk + rows - 1) / rows) * B * Hk, Hq / Hk * ((Nq + 31) / 32));
  r.q = wide_splits((int64_t)((Nq + rows - 1) / rows) * B * Hq, ((causal ? std::min(Nq, Nk) : Nk) + 31) / 32);
  return r;
}

bool flash_wide_shape(int EP, int DV) { return DV == 256 && (EP == 256 || EP == 384 || EP == 512); }

hipError_t launch_flash_wide_fwd(const FlashFwdParams& p, int dtype, hipStream_t s) {
  if (!flash_wide_shape(p.EP, p.DV)) return hipErrorInvalidValue;
  if (dtype == 2) {
    if (p.EP == 256) return fwd_t<BF16, 256, 256>(p, s);
    if (p.EP == 384) return fwd_t<BF16, 384, 256>(p, s);
    return fwd_t<BF16, 512, 256>(p, s);
  }
  if (p.EP == 256) return fwd_t<F16, 256, 256>(p, s);
  if (p.EP == 384) return fwd_t<F16, 384, 256>(p, s);
  return fwd_t<F16, 512, 256>(p, s);
}

hipError_t launch_flash_wide_bwd(const FlashBwdParams& p, int dtype, hipStream_t s) {
  if (!flash_wide_shape(p.EP, p.DV)) return hipErrorInvalidValue;
  if (dtype == 2) {
    if (p.EP == 256) return bwd_t<BF16, 256, 256>(p, s);
    if (p.EP == 384) return bwd_t<BF16, 384, 256>(p, s);
    return bwd_t<BF16, 512, 256>(p, s);
  }
  if (p.EP == 256) return bwd_t<F16, 256, 256>(p, s);
  if (p.EP == 384) return bwd_t<F16, 384, 256>(p, s);
  return bwd_t<F16, 512, 256>(p, s);
}

}  // namespace pope
