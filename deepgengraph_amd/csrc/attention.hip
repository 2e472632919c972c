// Fused online-softmax attention for gfx950 (CDNA4): prefill forward (causal / sliding window / tanh soft-cap /
// GQA), the column-score passes of the selection cases (H2O, RoCo, SnapKV, Corm, KeyFormer) and KeyFormer's
// perturbed row log-sum-exp.
//
// Products. Both run on v_mfma_f32_32x32x16_{bf16,f16} with the scores computed transposed:
//   S^T (BN x 32)  = K (BN x D) . Q^T (D x 32)     A = K fragments from LDS, B = Q held in registers
//   O^T (D x 32)  += V^T (D x BN) . P^T (BN x 32)  A = V^T by transposing LDS reads (ds_read_b64_tr_b16) of the
//                                                   row-major V tile, B = P straight from the S^T accumulator
// One query per lane (column n = lane % 32): the row max and row sum are in-lane plus one cross-half exchange
// (v_permlane32_swap), and the accumulator, rounded to 16 bits, is already the B operand of P.V.
// Softmax runs in the exp2 domain with a lazily-updated row maximum: O and l are rescaled only when a row's
// maximum grows by more than 2^8.
//
// Kernels. attn_fwd_dma_kernel (attention_fwd.h; 16-bit forward at every head_dim, except that head_dim 256 with fp32
// scores runs on attention_d256.hip) copies K/V tiles global -> LDS with direct loads (global_load_lds_dwordx4) into a
// swizzled ring. Tiles a wave cannot see are skipped, and within masked tiles dead 32-key blocks skip their MFMAs.
// Here: attn_colsum_d128_kernel / attn_colsum_kernel recompute P = exp2(s - lse) with one key per lane and sum (or
// test) it over the queries; attn_kf_rowlse_kernel is the row pass of KeyFormer's perturbed softmax. Reference rounding
// (DGG_ATTN_REF_ROUNDING) rounds the scores as the reference does on the GPU: matmul result to the input dtype, then
// the fp32 multiply by the reciprocal of sqrt(D) (and of the soft-cap), rounded again.
// Workgroups are ordered longest-first and grouped by head inside each XCD so the K/V of a head stay in one L2.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"

#include "attention_common.h"

namespace {

using namespace dgg_attn;



// ------------------------------------------------------------------------------------------------
// KeyFormer pass 1 (kf.py:36-39): the base-2 log-sum-exp of the Gumbel-perturbed scores of each query row,
//   lse2'[b, h, i] = log2 sum_j exp2(y_ij),  y_ij = (s2_ij - log2 e_ij) / tau,
// over the keys j the row sees, with s2 the score in the exp2 domain (rounded as the reference rounds when
// REFROUND) and e the exp_rand input (gumbels = -log(e), kf.py:37). Four waves of 32 rows; S^T = K.Q^T puts one
// query per lane, so the row reduction stays in the lane (plus one cross-half step). K tiles of 64 keys are staged
// through double-buffered LDS; exp_rand is read once, as 16-byte loads when VEC (rows 16-byte aligned).
// ------------------------------------------------------------------------------------------------
template <typename T, int D, bool MASK, int REFROUND, bool VEC>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) attn_kf_rowlse_kernel(AttnParams p) {
  typedef typename T::scalar S;
  typedef typename T::vec8 V8;
  constexpr int BN = 64;
  constexpr int KP = D + 8;       // padded K row: 16-byte shift per row for the fragment reads
  constexpr int NKK = D / 16;
  constexpr int NMB = BN / 32;
  constexpr int CPT = BN * D / 8 / kThreads;  // 16-byte chunks per thread per tile
  static_assert(CPT * kThreads == BN * D / 8, "tile mapping");
  __shared__ __attribute__((aligned(16))) S Ks[2][BN][KP];

  int qt, bh;
  map_block<true>(p.n_tiles, p.B * p.Hq, true, qt, bh);
  const int b = bh / p.Hq, h = bh - b * p.Hq;
  const int hk = h / p.group;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int q0 = qt * kBM;
  const int qi = q0 + 32 * w + r;
  const int qc = min(qi, p.Sq - 1);
  const S* qp = static_cast<const S*>(p.q) + b * p.q_sb + h * p.q_sh;
  const S* kp = static_cast<const S*>(p.k) + b * p.k_sb + hk * p.k_sh;
  const float* erow = p.er + b * p.er_sb + h * p.er_sh + (int64_t)qc * p.er_ss;

  V8 qf[NKK];
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) qf[kk] = ld16<V8>(qp + (int64_t)qc * p.q_ss + 16 * kk + 8 * g);
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) {
    asm volatile("" : "+v"(qf[kk]));
    if (qi >= p.Sq) qf[kk] = V8{};
  }

  const int q_last = min(q0 + kBM, p.Sq) - 1;
  int k_begin = 0, k_end = p.Sk;
  if (p.causal) k_end = min(p.Sk, q_last + p.offset + 1);
  if (p.window > 0) k_begin = max(0, q0 + p.offset - p.window + 1);
  const int t_begin = k_begin / BN;
  const int t_end = k_end > k_begin ? (k_end + BN - 1) / BN : t_begin;
  int k_hi = p.Sk - 1, k_lo = 0;
  if (p.causal) k_hi = min(k_hi, qi + p.offset);
  if (p.window > 0) k_lo = max(k_lo, qi + p.offset - p.window + 1);

  // K staging: copy i of thread tid moves 16-byte chunk (tid + i * kThreads) of the tile, i.e. chunk c % (D/8) of
  // key row c / (D/8) (rows past the end read the last row). Consecutive lanes take consecutive chunks of a row, so
  // each store instruction writes whole rows and the lanes of one LDS pass hit distinct banks (a thread writing
  // CPT adjacent chunks, one instruction per chunk, put lanes 128 bytes apart on the same banks).
  V8 kreg[CPT];
  constexpr int CPR = D / 8;  // chunks per key row
  auto load = [&](int t) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = tid + i * kThreads;
      kreg[i] = ld16<V8>(kp + (int64_t)min(t * BN + c / CPR, p.Sk - 1) * p.k_ss + (c % CPR) * 8);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = tid + i * kThreads;
      *reinterpret_cast<V8*>(&Ks[buf][c / CPR][(c % CPR) * 8]) = kreg[i];
    }
  };

  // fp16 reference rounding keeps each pair of scores packed (two instructions per score instead of four)
  constexpr bool PK = REFROUND && std::is_same<T, F16>::value;
  const float cy = (PK ? kLog2e : score_coeff<false, REFROUND>(p)) * p.kf_inv_tau;  // score -> exp2 domain / tau
  f16x2 hpair;
  float m_run = -INFINITY, l_run = 0.f;
  // element (mb, j) of the S^T accumulators holds key t*BN + mb*32 + 8*(j/4) + 4g + j%4. The exp_rand values of
  // tile t+1 are loaded while tile t is computed (ev_next), so the stream stays in flight under the exp/log work.
  f32x4 ev[NMB][4], ev_next[NMB][4];
  // Tiles whose keys all exist (VEC: rows 16-byte aligned) load exp_rand coalesced: load i of lane l reads keys
  // 4 (l % 16) .. +3 of the wave's row 4 i + l / 16, 256 contiguous bytes per row (a load with one row per lane
  // would touch 64 rows, 16 bytes each), and restage() passes the tile through the wave's own LDS rows into the
  // one-row-per-lane layout. Other tiles load that layout directly, 4 bytes at a time.
  constexpr int EV_RS = BN + 4;  // padded LDS row, floats: consecutive rows 4 banks apart
  __shared__ __attribute__((aligned(16))) float Es[kThreads / 64][32 * EV_RS];
  const float* ebase = p.er + b * p.er_sb + h * p.er_sh;
  auto whole = [&](int t) { return VEC && (t + 1) * BN <= p.Sk; };
  auto load_ev = [&](int t, f32x4 (&dst)[NMB][4]) {
    const int kb = t * BN;
    if (whole(t)) {
#pragma unroll
      for (int i = 0; i < 2 * NMB * 2; ++i) {
        const int row = min(q0 + 32 * w + 4 * i + (lane >> 4), p.Sq - 1);
        dst[i >> 2][i & 3] = *reinterpret_cast<const f32x4*>(ebase + (int64_t)row * p.er_ss + kb + 4 * (lane & 15));
      }
      return;
    }
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) {
        const int key = kb + mb * 32 + 8 * jq + 4 * g;
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[mb][jq][e] = erow[min(key + e, p.Sk - 1)];
      }
  };
  // The coalesced addressing above (load i: row 4i + lane/16, keys 4*(lane%16)..+3) covers exactly the wave's 32 rows
  // by 64 keys: 2*NMB*2 loads of 4 rows, 16 lanes x 4 keys per row.
  static_assert(BN == 64 && 16 * 4 == BN && 4 * (2 * NMB * 2) == 32, "coalesced exp_rand layout assumes 64-key tiles");
  auto restage = [&](f32x4 (&x)[NMB][4]) {
    float* ew = Es[w];
#pragma unroll
    for (int i = 0; i < 2 * NMB * 2; ++i)
      *reinterpret_cast<f32x4*>(ew + (4 * i + (lane >> 4)) * EV_RS + 4 * (lane & 15)) = x[i >> 2][i & 3];
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq)
        x[mb][jq] = *reinterpret_cast<const f32x4*>(ew + r * EV_RS + mb * 32 + 8 * jq + 4 * g);
  };
  auto tile = [&](int t, int buf, auto masked) {
    const int kb = t * BN;
    if (whole(t)) restage(ev);
    f32x16 sacc[NMB];
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) sacc[mb] = f32x16{};
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk)
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb)
        sacc[mb] = mfma32(*reinterpret_cast<const V8*>(&Ks[buf][mb * 32 + r][16 * kk + 8 * g]), qf[kk], sacc[mb]);
    const int rel_hi = k_hi - (kb + 4 * g), rel_lo = k_lo - (kb + 4 * g);
    float mloc = -INFINITY;
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        // y = (x2 - log2 e) / tau as one fma of the score against per-launch constants: the score x in the natural
        // log domain times log2(e) / tau (PK: the reference-rounded fp16 pair, read by v_fma_mix), or x * c / tau
        float x;
        if constexpr (PK) {
          if ((j & 1) == 0) hpair = ref_scores_f16(sacc[mb][j], sacc[mb][j + 1], p);
          x = (float)hpair[j & 1];
        } else {
          x = score_value<T, false, REFROUND>(sacc[mb][j], p);
        }
        float y = fmaf(x, cy, -fast_log2(ev[mb][j >> 2][j & 3]) * p.kf_inv_tau);
        if constexpr (decltype(masked)::value) {
          const int o = mb * 32 + 8 * (j >> 2) + (j & 3);
          y = (o <= rel_hi && o >= rel_lo) ? y : -INFINITY;
        }
        sacc[mb][j] = y;
        mloc = fmaxf(mloc, y);
      }
    mloc = half_swap_max(mloc);
    const float m_new = fmaxf(m_run, mloc);
    if (m_new > m_run + kRescaleThreshold || (m_run == -INFINITY && m_new > -INFINITY)) {
      l_run *= fast_exp2(m_run - m_new);  // 0 while m_run is -inf
      m_run = m_new;
    }
    const float mu = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
      for (int j = 0; j < 16; ++j) l_run += fast_exp2(sacc[mb][j] - mu);
  };

  // Tiles [t_full0, t_full1) need no mask for any row of the workgroup.
  int t_full0 = t_begin, t_full1 = t_end;
  if constexpr (MASK) {
    if (p.window > 0) {
      const int lo_last = q_last + p.offset - p.window + 1;
      t_full0 = lo_last <= 0 ? t_begin : min(t_end, max(t_begin, (lo_last + BN - 1) / BN));
    }
    if (p.causal) {
      const int hi_first = q0 + p.offset;
      t_full1 = max(t_full0, min(t_end, hi_first < 0 ? t_begin : (hi_first + 1) / BN));
    }
  }
  if (t_full1 > t_full0 && t_full1 * BN > p.Sk) t_full1 = max(t_full0, p.Sk / BN);
  if (t_full1 < t_full0) t_full1 = t_full0;

  if (t_begin < t_end) {
    load(t_begin);
    load_ev(t_begin, ev);
    store(0);
  }
  __syncthreads();
  auto step = [&](int t, auto masked) {
    const int buf = (t - t_begin) & 1;
    const bool more = t + 1 < t_end;
    if (more) {
      load(t + 1);
      load_ev(t + 1, ev_next);
    }
    tile(t, buf, masked);
    if (more) store(buf ^ 1);
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) ev[mb][jq] = ev_next[mb][jq];
  };
  for (int t = t_begin; t < t_full0; ++t) step(t, std::true_type{});
  for (int t = t_full0; t < t_full1; ++t) step(t, std::false_type{});
  for (int t = t_full1; t < t_end; ++t) step(t, std::true_type{});

  const float l_tot = half_swap_sum(l_run);
  if (qi < p.Sq && g == 0) p.lse[(int64_t)bh * p.Sq + qi] = m_run == -INFINITY ? -INFINITY : m_run + fast_log2(l_tot);
}

// KeyFormer pass 1 for head_dim 128 and exp_rand rows of whole 16-byte chunks: the same reduction by 8 waves over 128
// rows, two waves (key groups) to the same 32 rows, each taking 32 keys of every 64-key tile. K tiles and exp_rand are
// copied global -> LDS directly. A wave's exp_rand (32 rows x 32 keys) is its own, so it needs no barrier and one buffer:
// it is read into registers at the start of a tile and the next tile's copies follow at once. Chunk c of row r of it
// sits at position c ^ (r / 2 % 8), so that 16 rows of one chunk are on distinct banks.
// What bounds it: with few rows the latency of a wave's chain (products, log2, maximum, exp2: ~1 us per 32 keys, hence
// the key groups and four waves per SIMD), with many the exp_rand stream. The tiles of a workgroup are taken from a
// starting point of its own: rows of a power-of-two length lie on few memory channels, and workgroups that all walk the
// columns in step keep hitting the same ones (S=2048, H=32, fp16, causal: 94.6 us without, 71.9 with; S=4096 218 / 227).
// Against the register-staged kernel above, same calls: S=1000 35.7 -> 29.1 us, S=2048 98 -> 72, S=4096 226 / 227.
template <typename T, bool MASK, int REFROUND>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4)))
attn_kf_rowlse_dma_kernel(AttnParams p) {
  typedef typename T::scalar S;
  typedef typename T::vec8 V8;
  constexpr int D = 128, NW = 8, KG = 2, NWR = NW / KG, BN = 32 * KG, BM = 32 * NWR;
  static_assert(BM == kBM, "rows per workgroup");
  typedef DmaLayout<D> L;
  constexpr int KT_B = (BN / 4) * L::GROUP_B;      // K tile
  constexpr int ET_B = 32 * 32 * 4;                // one wave's exp_rand
  constexpr int KPW = BN / 4 / NW, EPW = ET_B / 1024;  // copies per wave and tile
  constexpr int QSLOT_B = 8 * L::GROUP_B;
  static_assert(NWR * QSLOT_B <= 2 * KT_B, "the Q tile passes through the K ring");
  __shared__ __attribute__((aligned(1024))) char smem[2 * KT_B + NW * ET_B];

  int qt, bh;
  const int bid = p.block0 + blockIdx.x;
  map_block<true>(p.n_tiles, p.B * p.Hq, true, qt, bh, bid);
  const int b = bh / p.Hq, h = bh - b * p.Hq;
  const int hk = h / p.group;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = w % NWR, kg = w / NWR;  // row block and key group
  const int q0 = qt * BM, qw0 = q0 + 32 * wr;
  const int qi = qw0 + r;
  const char* qp = reinterpret_cast<const char*>(static_cast<const S*>(p.q) + b * p.q_sb + h * p.q_sh);
  const char* kp = reinterpret_cast<const char*>(static_cast<const S*>(p.k) + b * p.k_sb + hk * p.k_sh);
  const int64_t q_ss_b = p.q_ss * (int64_t)sizeof(S), k_ss_b = p.k_ss * (int64_t)sizeof(S);
  const uint32_t smem_base = (uint32_t)(size_t)((lds_char*)smem);
  const uint32_t e_slot = smem_base + (uint32_t)(2 * KT_B + w * ET_B);
  const int rr = lane >> 4;                                       // row of a 4-row group, in a Q / K copy
  const uint32_t chunk_b = 16u * (uint32_t)((lane & 15) ^ L::swizzle(rr));

  // Q through the K ring into registers, the two key groups copying half of a row block's rows each (rows past the end
  // read the last row and are zeroed below).
  const uint32_t q_slot = smem_base + (uint32_t)(wr * QSLOT_B);
#pragma unroll
  for (int i = 0; i < 8 / KG; ++i) {
    const int j = KG * i + kg;
    dma16(q_slot + j * L::GROUP_B, qp + (int64_t)min(qw0 + 4 * j + rr, p.Sq - 1) * q_ss_b + chunk_b);
  }

  const int q_last = min(q0 + BM, p.Sq) - 1;
  int k_begin = 0, k_end = p.Sk;
  if (p.causal) k_end = min(p.Sk, q_last + p.offset + 1);
  if (p.window > 0) k_begin = max(0, q0 + p.offset - p.window + 1);
  const int t_begin = k_begin / BN;
  const int n_t = k_end > k_begin ? (k_end + BN - 1) / BN - t_begin : 0;
  const int rot = n_t > 0 ? (int)((unsigned)(bid >> 3) * 7 % n_t) : 0;
  auto tile_of = [&](int i) { return t_begin + (i + rot < n_t ? i + rot : i + rot - n_t); };
  int k_hi = p.Sk - 1, k_lo = 0;
  if (p.causal) k_hi = min(k_hi, qi + p.offset);
  if (p.window > 0) k_lo = max(k_lo, qi + p.offset - p.window + 1);

  // exp_rand copy i of a tile: rows 8i + lane / 8 of the wave, position lane % 8 of the row. Where every row and key
  // exists: a scalar address plus one of two lane offsets (the swizzle of rows 8i.. differs between even and odd i).
  // At the edges: the last row, the last whole chunk of exp_rand, the last key of K (masked, finite: exactly 0).
  const char* eb = reinterpret_cast<const char*>(p.er + b * p.er_sb + h * p.er_sh);
  const int64_t er_ss_b = p.er_ss * 4;
  const bool rows_ok = qw0 + 32 <= p.Sq && p.er_lane32;
  uint32_t e_voff[2], k_voff = (uint32_t)(rr * k_ss_b) + chunk_b;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    e_voff[i] = (uint32_t)((lane >> 3) * er_ss_b) + 16u * (uint32_t)((lane & 7) ^ ((4 * i + (lane >> 4)) & 7));
  auto issue_e = [&](int t) __attribute__((always_inline)) {
    const int kb = t * BN + 32 * kg;
    if (rows_ok && kb + 32 <= p.Sk) {
      const char* base = eb + (int64_t)qw0 * er_ss_b + (int64_t)kb * 4;
#pragma unroll
      for (int i = 0; i < EPW; ++i) dma16(e_slot + 1024 * i, base + 8 * i * er_ss_b, e_voff[i & 1]);
    } else {
#pragma unroll
      for (int i = 0; i < EPW; ++i) {
        const int row = 8 * i + (lane >> 3), col = kb + 4 * ((lane & 7) ^ ((row >> 1) & 7));
        dma16(e_slot + 1024 * i, eb + ((int64_t)min(qw0 + row, p.Sq - 1) * p.er_ss + min(col, p.Sk - 4)) * 4);
      }
    }
  };
  auto issue_k = [&](int slot, int t) __attribute__((always_inline)) {
    const uint32_t dst = smem_base + (uint32_t)((slot & 1) * KT_B + KPW * w * L::GROUP_B);
    if ((t + 1) * BN <= p.Sk) {
      const char* base = kp + (int64_t)(t * BN + 4 * KPW * w) * k_ss_b;
#pragma unroll
      for (int j = 0; j < KPW; ++j) dma16(dst + j * L::GROUP_B, base + 4 * j * k_ss_b, k_voff);
    } else {
#pragma unroll
      for (int j = 0; j < KPW; ++j)
        dma16(dst + j * L::GROUP_B, kp + (int64_t)min(t * BN + 4 * (KPW * w + j) + rr, p.Sk - 1) * k_ss_b + chunk_b);
    }
  };

  const int s4 = r & 3;
  uint32_t xq[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) xq[i] = (uint32_t)((r >> 2) * L::GROUP_B + s4 * L::ROW_B + 16 * g + 64 * (i ^ s4));
  if (n_t > 0) issue_e(tile_of(0));
  V8 qf[D / 16];
  if (n_t > 0) wait_vmem<EPW>();
  else wait_vmem<0>();
  __syncthreads();
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) qf[kk] = lds_read<V8>(q_slot + xq[kk >> 1] + 32 * (kk & 1));
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    asm volatile("" : "+v"(qf[kk]));
    if (qi >= p.Sq) qf[kk] = V8{};
  }
  __syncthreads();  // every wave has its Q: the ring is free
  if (n_t > 0) issue_k(0, tile_of(0));

  // fp16 reference rounding keeps each pair of scores packed (two instructions per score instead of four)
  constexpr bool PK = REFROUND && std::is_same<T, F16>::value;
  const float cy = (PK ? kLog2e : score_coeff<false, REFROUND>(p)) * p.kf_inv_tau;  // score -> exp2 domain / tau
  float m_run = -INFINITY, l_run = 0.f;
  auto tile = [&](int t, f32x16& sacc, const f32x4 (&ev)[4], auto masked) __attribute__((always_inline)) {
    // element j holds key t*BN + 32*kg + 8*(j/4) + 4g + j%4
    const int kb4 = t * BN + 32 * kg + 4 * g;
    const int rel_hi = k_hi - kb4, rel_lo = k_lo - kb4;
    float mloc = -INFINITY;
    f16x2 hpair;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      // y = (x2 - log2 e) / tau as one fma of the score against per-launch constants: the score x in the natural log
      // domain times log2(e) / tau (PK: the reference-rounded fp16 pair, read by v_fma_mix), or x * c / tau
      float x;
      if constexpr (PK) {
        if ((j & 1) == 0) hpair = ref_scores_f16(sacc[j], sacc[j + 1], p);
        x = (float)hpair[j & 1];
      } else {
        x = score_value<T, false, REFROUND>(sacc[j], p);
      }
      float y = fmaf(x, cy, -fast_log2(ev[j >> 2][j & 3]) * p.kf_inv_tau);
      const int o = 8 * (j >> 2) + (j & 3);
      if constexpr (decltype(masked)::value) y = (o <= rel_hi && o >= rel_lo) ? y : -INFINITY;
      sacc[j] = y;
      mloc = fmaxf(mloc, y);
    }
    mloc = half_swap_max(mloc);
    const float m_new = fmaxf(m_run, mloc);
    if (m_new > m_run + kRescaleThreshold || (m_run == -INFINITY && m_new > -INFINITY)) {
      l_run *= fast_exp2(m_run - m_new);  // 0 while m_run is -inf
      m_run = m_new;
    }
    const float mu = m_run == -INFINITY ? 0.f : m_run;
    float part[2] = {0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 16; ++j) part[j & 1] += fast_exp2(sacc[j] - mu);
    l_run += part[0] + part[1];
  };

  // Keys [wk_begin, wk_end) are seen by some row of this wave, [f0, f1) by every one.
  int wk_begin = 0, wk_end = qw0 < p.Sq ? p.Sk : 0, f0 = 0, f1 = p.Sk;
  if constexpr (MASK) {
    const int wq_last = min(qw0 + 32, p.Sq) - 1;
    if (p.window > 0) {
      wk_begin = max(0, qw0 + p.offset - p.window + 1);
      f0 = max(0, wq_last + p.offset - p.window + 1);
    }
    if (p.causal) {
      wk_end = min(wk_end, wq_last + p.offset + 1);
      f1 = min(f1, qw0 + p.offset + 1);
    }
  }
  for (int i = 0; i < n_t; ++i) {
    wait_vmem<0>();
    __syncthreads();  // tile i of K is in the LDS; every wave has left tile i - 1
    if (i + 1 < n_t) issue_k(i + 1, tile_of(i + 1));
    const int t = tile_of(i), kb = t * BN + 32 * kg;
    const bool live = kb < wk_end && kb + 32 > wk_begin;
    f32x16 sacc = f32x16{};
    if (live) {
      const uint32_t st = smem_base + (uint32_t)((i & 1) * KT_B + kg * (KT_B / KG));
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) sacc = mfma32(lds_read<V8>(st + xq[kk >> 1] + 32 * (kk & 1)), qf[kk], sacc);
    }
    // exp_rand after the products (fewer registers at once: 128 are what four waves per SIMD have)
    f32x4 ev[4];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) ev[jq] = lds_read<f32x4>(e_slot + r * 128 + 16 * ((2 * jq + g) ^ ((r >> 1) & 7)));
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) asm volatile("" : "+v"(ev[jq]));  // read: the buffer may be overwritten
    if (i + 1 < n_t) issue_e(tile_of(i + 1));
    if (!live) continue;
    if (kb >= f0 && kb + 32 <= f1) tile(t, sacc, ev, std::false_type{});
    else tile(t, sacc, ev, std::true_type{});
  }
  float l_tot = half_swap_sum(l_run);
  __syncthreads();  // the ring is done with
  f32x2* ml = reinterpret_cast<f32x2*>(smem);  // key group 1's (maximum, sum) per row
  if (kg == 1 && g == 0) ml[32 * wr + r] = f32x2{m_run, l_tot};
  __syncthreads();
  if (kg == 0 && g == 0 && qi < p.Sq) {
    const f32x2 o = ml[32 * wr + r];
    const float m = fmaxf(m_run, o[0]), mu = m == -INFINITY ? 0.f : m;
    l_tot = l_tot * fast_exp2(m_run - mu) + o[1] * fast_exp2(o[0] - mu);
    p.lse[(int64_t)bh * p.Sq + qi] = m == -INFINITY ? -INFINITY : m + fast_log2(l_tot);
  }
}

// ------------------------------------------------------------------------------------------------
// Column-sum kernel: colsum[b,h,j] = sum_i exp(score_ij - lse_i). A workgroup owns 128 keys (32 per wave,
// held in VGPRs as the B operand); query tiles of 64 rows stream through double-buffered LDS together
// with their lse. S (64 x 32) = Q . K^T puts one key per lane, so each lane sums its own column.
// ------------------------------------------------------------------------------------------------
constexpr int kCBQ = 64;   // query rows per tile
constexpr int kCBK = 32 * kWaves;  // keys per workgroup

template <typename T, int D, bool MASK, bool SOFTCAP, int REFROUND, int EPI>
__global__ void __launch_bounds__(kThreads) attn_colsum_kernel(AttnParams p) {
  typedef typename T::scalar S;
  typedef typename T::vec8 V8;
  constexpr int QP = D + 8;
  constexpr int NKK = D / 16;
  constexpr int NMB = kCBQ / 32;
  constexpr int CHUNKS = kCBQ * D / 8;
  constexpr int CPT = (CHUNKS + kThreads - 1) / kThreads;

  __shared__ __attribute__((aligned(16))) S Qs[2][kCBQ][QP];
  __shared__ float Ls[2][kCBQ];

  int kt, bh;
  map_block(p.n_tiles, p.B * p.Hq, false, kt, bh);
  const int b = bh / p.Hq, h = bh - b * p.Hq;
  const int hk = h / p.group;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int k0 = kt * kCBK;
  const int kj = k0 + 32 * w + r;  // this lane's key

  const S* qp = static_cast<const S*>(p.q) + b * p.q_sb + h * p.q_sh;
  const S* kp = static_cast<const S*>(p.k) + b * p.k_sb + hk * p.k_sh;
  const float* lsep = p.lse + (int64_t)bh * p.Sq;

  V8 kf[NKK];
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk)  // back-to-back loads (keys past the end read the last key, zeroed below)
    kf[kk] = ld16<V8>(kp + (int64_t)min(kj, p.Sk - 1) * p.k_ss + 16 * kk + 8 * g);
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) {
    asm volatile("" : "+v"(kf[kk]));  // see the forward kernel
    if (kj >= p.Sk) kf[kk] = V8{};
  }

  // Query range that can see any key of this tile.
  const int k_last = min(k0 + kCBK, p.Sk) - 1;
  int q_begin = 0, q_end = p.Sq;
  if (p.causal) q_begin = max(0, k0 - p.offset);
  if (p.window > 0) q_end = min(p.Sq, k_last - p.offset + p.window);
  const int t_begin = q_begin / kCBQ;
  const int t_end = q_end > q_begin ? (q_end + kCBQ - 1) / kCBQ : t_begin;
  const float c = score_coeff<SOFTCAP, REFROUND>(p);

  V8 qreg[CPT];
  float lreg = 0.f;
  auto load_tile = [&](int t) {
    const int qb = t * kCBQ;
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int ch = tid + i * kThreads;
      if (CHUNKS % kThreads == 0 || ch < CHUNKS) {
        const int row = ch / (D / 8), dc = ch % (D / 8);
        const int qg = qb + row;
        qreg[i] = qg < p.Sq ? ld16<V8>(qp + (int64_t)qg * p.q_ss + dc * 8) : V8{};
      }
    }
    if (tid < kCBQ) {
      const int qg = qb + tid;
      // Rows past the end get +inf so that their probability is exp2(-inf) = 0.
      lreg = qg < p.Sq ? (p.lse_base2 ? lsep[qg] : lsep[qg] * kLog2e) : INFINITY;
    }
  };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int ch = tid + i * kThreads;
      if (CHUNKS % kThreads == 0 || ch < CHUNKS) {
        const int row = ch / (D / 8), dc = ch % (D / 8);
        *reinterpret_cast<V8*>(&Qs[buf][row][dc * 8]) = qreg[i];
      }
    }
    if (tid < kCBQ) Ls[buf][tid] = lreg;
  };

  if (t_begin < t_end) {
    load_tile(t_begin);
    store_tile(0);
  }
  __syncthreads();

  ColAcc<EPI> acc;
  const int kjc = min(kj, p.Sk - 1);
  const float* erp = EPI == kColKF ? p.er + b * p.er_sb + h * p.er_sh : nullptr;  // KeyFormer exp_rand of (b, h)
  for (int t = t_begin; t < t_end; ++t) {
    const int buf = (t - t_begin) & 1;
    const bool has_next = t + 1 < t_end;
    if (has_next) load_tile(t + 1);

    f32x16 sacc[NMB];
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) sacc[mb] = f32x16{};
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb) {
        const V8 a = *reinterpret_cast<const V8*>(&Qs[buf][mb * 32 + r][16 * kk + 8 * g]);
        sacc[mb] = mfma32(a, kf[kk], sacc[mb]);
      }
    }

    const int qb = t * kCBQ;
    bool need_mask = qb + kCBQ > p.Sq || k0 + kCBK > p.Sk;
    if constexpr (MASK) {
      if (p.causal && qb + p.offset < k_last) need_mask = true;
      if (p.window > 0 && qb + kCBQ - 1 + p.offset - k0 >= p.window) need_mask = true;
    }
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int row = mb * 32 + 8 * (j >> 2) + 4 * g + (j & 3);
        const float x = score_value<T, SOFTCAP, REFROUND>(sacc[mb][j], p);
        const int qg = qb + row;
        float pe;
        if constexpr (EPI == kColKF)
          pe = kf_prob(x * c, erp[(int64_t)min(qg, p.Sq - 1) * p.er_ss + kjc], Ls[buf][row], p);
        else
          pe = fast_exp2(fmaf(x, c, -Ls[buf][row]));
        bool vis = true;  // (qg, kj) a visible pair of an existing row and key
        if (need_mask) {
          bool ok = qg < p.Sq && kj < p.Sk;
          if constexpr (MASK) {
            const int rel = qg + p.offset - kj;
            if (p.causal) ok = ok && rel >= 0;
            if (p.window > 0) ok = ok && rel < p.window;
          }
          pe = ok ? pe : 0.f;
          vis = ok;
        }
        // Corm compares visible pairs here; the masked ones (p = 0) are ORed in by corm_masked_or_kernel
        acc.add(pe, EPI == kColAnyGe ? vis : qg < p.Sq, min(qg, p.Sq - 1), kjc, p);
      }
    }

    if (has_next) store_tile(buf ^ 1);
    __syncthreads();
  }
  acc.store(p, bh, kj, g);
}

// ------------------------------------------------------------------------------------------------
// Column-sum kernel for head_dim 128. A workgroup of NW waves owns 32*NW/NG keys, which each of its NG row groups
// covers; a wave keeps 32 of them in VGPRs as the B operand. Query tiles of BQ rows stream through a two-stage ring in LDS
// with the forward's swizzled layout and direct-to-LDS copies (the Q tile takes the place of the K tile),
// each stage followed by the BQ lse values of its rows (global_load_lds_dword, issued by the last wave).
// S (BQ x 32) = Q . K^T puts one key per lane: accumulator register j of block mb holds query row
// 32mb + 8(j/4) + 4(lane/32) + j%4, so each lane sums its key's column over its rows, and the partner
// lane (lane ^ 32) adds the other half at the end.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ void dma4(uint32_t lds, const void* vaddr) {
  // lane l's 4 bytes land at LDS byte address lds + 4*l (lanes switched off by EXEC write nothing)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds), "v"(vaddr)
               : "memory", "m0");
}

// NG: row groups of NW / NG waves. Each group covers every key of the workgroup (32 * NW / NG keys) and takes its own
// BQ / NG rows of each query tile; the groups' results are combined through the LDS at the end. OCC: waves per SIMD the
// register budget is sized for (4: two workgroups per CU, whose LDS fits).
template <typename T, int NW, int NG, int BQ, int OCC, bool MASK, bool SOFTCAP, int REFROUND, bool LSE2, int EPI>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(OCC, OCC)))
attn_colsum_d128_kernel(AttnParams p) {
  constexpr int D = 128;
  constexpr int ROW_B = DmaLayout<D>::ROW_B, GROUP_B = DmaLayout<D>::GROUP_B;
  typedef typename T::scalar S;
  typedef typename T::vec8 V8;
  constexpr int NWG = NW / NG;               // waves per row group
  constexpr int BQW = BQ / NG;               // query rows of a tile per row group
  constexpr int BK = 32 * NWG;               // keys per workgroup
  constexpr int NSTAGE = 2;                  // query tiles in the LDS ring
  constexpr int QT_B = (BQ / 4) * GROUP_B;   // bytes of one Q tile
  constexpr int STAGE_B = QT_B + 4 * BQ;     // Q tile, then its BQ lse values
  constexpr int GPW = (BQ / 4) / NW;         // 4-row groups of a Q tile copied by each wave
  constexpr int NLSE = BQ / 64;              // lse copies per tile (last wave only)
  constexpr int NMB = BQW / 32;              // 32-row query blocks of a wave's part of a tile
  static_assert(GPW >= 1 && GPW * NW == BQ / 4, "Q tile groups must split over the waves");
  static_assert(BQ % 64 == 0 && QT_B % 16 == 0 && BQW % 32 == 0 && NWG * NG == NW, "tile shape");
  static_assert(NG == 1 || NSTAGE * STAGE_B >= (NG - 1) * 2 * BK * 4, "the groups' sums are combined in the LDS");
  constexpr int KSLOT_B = 8 * GROUP_B;  // 32 keys on their way to the registers
  static_assert(NWG * KSLOT_B <= STAGE_B, "the workgroup's keys pass through the stage that no first copy fills");
  __shared__ __attribute__((aligned(1024))) char smem[NSTAGE * STAGE_B];

  int kt, bh;
  map_block<OCC == 4>(p.n_tiles, p.B * p.Hq, false, kt, bh, p.block0 + blockIdx.x);
  const int b = bh / p.Hq, h = bh - b * p.Hq;
  const int hk = h / p.group;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wi = w % NWG, gw = w / NWG;  // wave within its row group, row group
  const int rg0 = BQW * gw;              // first row of the group's part of a query tile
  const int k0 = kt * BK;
  const int kw0 = k0 + 32 * wi;  // first key of this wave
  const int kj = kw0 + r;             // this lane's key

  const S* kp = static_cast<const S*>(p.k) + b * p.k_sb + hk * p.k_sh;
  const char* qp = reinterpret_cast<const char*>(static_cast<const S*>(p.q) + b * p.q_sb + h * p.q_sh);
  const int64_t q_ss_b = p.q_ss * (int64_t)sizeof(S);
  const float* lsep = p.lse + (int64_t)bh * p.Sq;

  // Query tiles that see any key of the workgroup, and of this wave.
  const int k_last = min(k0 + BK, p.Sk) - 1;
  int q_begin = 0, q_end = p.Sq;
  if (p.causal) q_begin = max(0, k0 - p.offset);
  if (p.window > 0) q_end = min(p.Sq, k_last - p.offset + p.window);
  const int t_begin = q_begin / BQ;
  const int t_end = q_end > q_begin ? (q_end + BQ - 1) / BQ : t_begin;
  int wt_begin = t_begin, wt_end = t_begin;  // empty for a wave whose keys all lie past Sk
  if (kw0 < p.Sk) {
    const int wk_last = min(kw0 + 32, p.Sk) - 1;
    int wq_begin = 0, wq_end = p.Sq;
    if (p.causal) wq_begin = max(0, kw0 - p.offset);
    if (p.window > 0) wq_end = min(p.Sq, wk_last - p.offset + p.window);
    if (wq_end > wq_begin) {  // tiles whose rows [t BQ + rg0, t BQ + rg0 + BQW) meet [wq_begin, wq_end)
      const int y = wq_begin - rg0 - BQW + 1;
      wt_begin = max(t_begin, y <= 0 ? 0 : (y + BQ - 1) / BQ);
      const int z = wq_end - rg0;
      wt_end = min(t_end, z <= 0 ? 0 : (z + BQ - 1) / BQ);
      if (wt_end < wt_begin) wt_end = wt_begin;
    }
  }
  // Tiles [t_full0, t_full1) need no mask for this wave: every row < Sq of its part sees all of its 32 keys.
  int t_full0 = t_begin, t_full1 = t_end;
  if constexpr (MASK) {
    if (p.causal) {
      const int a = kw0 + 32 - 1 - p.offset - rg0;  // first row that sees the wave's last key, less rg0
      t_full0 = a <= 0 ? t_begin : min(t_end, max(t_begin, (a + BQ - 1) / BQ));
    }
    if (p.window > 0) {
      const int last = kw0 + p.window - p.offset - 1;  // last query row that sees the wave's first key
      const int v = last + 1 - rg0 - BQW + BQ;          // tiles t < v / BQ end their group rows by last
      t_full1 = v <= 0 ? t_full0 : min(t_end, v / BQ);
    }
  }
  if (t_full1 * BQ > p.Sq) t_full1 = p.Sq / BQ;  // ragged last tile
  if (EPI == kColKF && !p.er_lane32) t_full1 = t_full0;  // exp_rand offsets too wide for the full-tile loads
  if (EPI == kColAnyGe && !p.thr_lane32) t_full1 = t_full0;  // threshold offsets too wide for the full-tile loads
  if (t_full1 < t_full0) t_full1 = t_full0;

  // Direct-load lane constants (as the forward's K tiles).
  const int rr = lane >> 4;
  const uint32_t src_chunk = (uint32_t)((lane & 15) ^ (rr << 2));
  uint32_t q_voff = (uint32_t)(rr * q_ss_b) + src_chunk * 16u;
  asm volatile("" : "+v"(q_voff));
  const uint32_t smem_base = (uint32_t)(size_t)((lds_char*)smem);

  auto issue = [&](int t) {
    const uint32_t stage = smem_base + (uint32_t)((t % NSTAGE) * STAGE_B);
    const uint32_t qdst = stage + (uint32_t)(GPW * w * GROUP_B);
    const int row0 = t * BQ + 4 * GPW * w;
    if ((t + 1) * BQ <= p.Sq) {
      const char* qb = qp + (int64_t)row0 * q_ss_b;
#pragma unroll
      for (int j = 0; j < GPW; ++j) dma16(qdst + j * GROUP_B, qb + 4 * j * q_ss_b, q_voff);
    } else {  // ragged last tile: rows past the end re-read the last row (masked)
#pragma unroll
      for (int j = 0; j < GPW; ++j) {
        const int64_t row = min(row0 + 4 * j + rr, p.Sq - 1);
        dma16(qdst + j * GROUP_B, qp + row * q_ss_b + src_chunk * 16);
      }
    }
    if (w == NW - 1) {
#pragma unroll
      for (int i = 0; i < NLSE; ++i) dma4(stage + QT_B + 256 * i, lsep + min(t * BQ + 64 * i + lane, p.Sq - 1));
    }
  };

  // The keys: copied like the Q tiles (a fragment load straight from global memory has 64 lanes on 32 rows, ~64 cycles
  // of address processing each), the row groups taking turns at the 4-row groups of a slot. Keys past the end read the
  // last key and are zeroed.
  const uint32_t kslot = smem_base + (uint32_t)(((t_begin + NSTAGE - 1) % NSTAGE) * STAGE_B + wi * KSLOT_B);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (NG > 1 && j % NG != gw) continue;
    const int64_t key = min(kw0 + 4 * j + rr, p.Sk - 1);
    dma16(kslot + j * GROUP_B, reinterpret_cast<const char*>(kp + key * p.k_ss) + src_chunk * 16);
  }

  // Q fragment (row 32mb + r, chunk 2kk + g) addressing, as the forward's K fragments.
  const int s4 = r & 3;
  const uint32_t q_lane = (uint32_t)((rg0 / 4 + (r >> 2)) * GROUP_B + s4 * ROW_B + 16 * g);
  uint32_t xq[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) xq[i] = q_lane + 64u * (uint32_t)(i ^ s4);

  constexpr bool PK = REFROUND && !SOFTCAP && std::is_same<T, F16>::value;
  const float c = PK ? kLog2e : score_coeff<SOFTCAP, REFROUND>(p);
  const float cy = EPI == kColKF ? c * p.kf_inv_tau : 0.f;  // KeyFormer: score -> exp2 domain / tau
  ColAcc<EPI> acc;
  const int kjc = min(kj, p.Sk - 1);
  const float* erp = EPI == kColKF ? p.er + b * p.er_sb + h * p.er_sh : nullptr;  // KeyFormer exp_rand of (b, h)
  // KeyFormer exp_rand of (row, kjc) for tiles whose rows all exist: a wave-uniform tile address (scalar registers)
  // plus a 32-bit offset, this lane's part (rows 4g apart, column kjc) plus the row's, one add per load.
  const uint32_t er_lane_b = EPI == kColKF ? (uint32_t)((4 * g * p.er_ss + kjc) * 4) : 0u;
  // Corm's thresholds of (row, kjc), addressed the same way.
  const uint32_t thr_lane_b = EPI == kColAnyGe ? (uint32_t)((4 * g * p.thr_rs + kjc) * 4) : 0u;

  V8 kf[D / 16];  // this wave's keys (B operand), read below
  // S = Q . K^T of query tile t (its LDS stage) into s.
  auto qk_t = [&](const int t, f32x16 (&s)[NMB]) __attribute__((always_inline)) {
    const uint32_t st = smem_base + (uint32_t)((t % NSTAGE) * STAGE_B);
    uint32_t qb[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) qb[i] = st + xq[i];
#pragma unroll
    for (int i = 0; i < NMB; ++i) s[i] = f32x16{};
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk)
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb) {
        const V8 a = lds_read<V8>(qb[kk >> 1] + mb * 8 * GROUP_B + 32 * (kk & 1));
        s[mb] = mfma32(a, kf[kk], s[mb]);
      }
  };
  auto epi_t = [&](const int t, const f32x16 (&sacc)[NMB], const float (&ev)[NMB][16], const float (&tv)[NMB][16],
                   auto masked) __attribute__((always_inline)) {
    const uint32_t lb = smem_base + (uint32_t)((t % NSTAGE) * STAGE_B) + QT_B + 4 * rg0 + 16 * g;  // this lane's lse
    // Visibility of (row o of the tile, this lane's key): causal rel >= 0, window rel < window, row < Sq.
    const int rows_left = p.Sq - t * BQ - rg0 - 4 * g;
    const int rel0 = t * BQ + rg0 + 4 * g + p.offset - kj;
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) {
      f32x4 lv[4];
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) lv[jq] = lds_read<f32x4>(lb + 4 * (32 * mb + 8 * jq));
      f16x2 hs[8];
      if constexpr (PK) {
#pragma unroll
        for (int jp = 0; jp < 8; ++jp) hs[jp] = ref_scores_f16(sacc[mb][2 * jp], sacc[mb][2 * jp + 1], p);
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        float x;
        if constexpr (PK) x = (float)hs[j >> 1][j & 1];
        else x = score_value<T, SOFTCAP, REFROUND>(sacc[mb][j], p);
        const float l2 = LSE2 ? lv[j >> 2][j & 3] : lv[j >> 2][j & 3] * kLog2e;
        const int o = 32 * mb + 8 * (j >> 2) + (j & 3);
        float pe;
        if constexpr (EPI == kColKF)  // kf_prob with x * c folded into one fma against c / tau
          pe = __builtin_amdgcn_exp2f(fmaf(x, cy, -fmaf(__builtin_amdgcn_logf(ev[mb][j]), p.kf_inv_tau, l2)));
        else
          pe = fast_exp2(fmaf(x, c, -l2));
        bool valid = true, vis = true;
        if constexpr (decltype(masked)::value) {
          valid = o < rows_left;
          bool ok = valid;
          if constexpr (MASK) {
            if (p.causal) ok = ok && rel0 + o >= 0;
            if (p.window > 0) ok = ok && rel0 + o < p.window;
          }
          pe = ok ? pe : 0.f;
          vis = ok;
        }
        // Corm compares visible pairs here; the masked ones (p = 0) are ORed in by corm_masked_or_kernel
        if constexpr (EPI == kColAnyGe) acc.any |= vis && pe >= tv[mb][j];
        else acc.add(pe, valid, min(t * BQ + rg0 + 4 * g + o, p.Sq - 1), kjc, p);
      }
    }
  };

  auto tile = [&](const int t, auto masked) {
    float ev[NMB][16];
    if constexpr (EPI == kColKF) {
      if constexpr (!decltype(masked)::value) {  // every row of the tile exists (and er_lane32 holds)
        const char* rb = reinterpret_cast<const char*>(erp + (int64_t)(t * BQ + rg0) * p.er_ss);
        uint32_t ss_b = (uint32_t)(p.er_ss * 4);
        asm volatile("" : "+s"(ss_b));  // per tile: keeps the 64 offsets from being hoisted into registers
#pragma unroll
        for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const uint32_t row_b = (uint32_t)(32 * mb + 8 * (j >> 2) + (j & 3)) * ss_b;
            ev[mb][j] = *reinterpret_cast<const float*>(rb + (er_lane_b + row_b));
          }
      } else {  // rows past the end read the last row (their p is masked)
#pragma unroll
        for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
          for (int j = 0; j < 16; ++j)
            ev[mb][j] = erp[(int64_t)min(t * BQ + rg0 + 4 * g + 32 * mb + 8 * (j >> 2) + (j & 3), p.Sq - 1) * p.er_ss + kjc];
      }
    }
    // Corm: the tile's thresholds for this lane's key, requested before the QK^T MFMAs so that the loads overlap
    // them (corm.py:35-37 compares each p with thr[i][j])
    float tv[NMB][16];
    if constexpr (EPI == kColAnyGe) {
      if constexpr (!decltype(masked)::value) {  // every row of the tile exists (and thr_lane32 holds)
        const char* rb = reinterpret_cast<const char*>(p.thr + (int64_t)(t * BQ + rg0) * p.thr_rs);
        uint32_t ss_b = (uint32_t)(p.thr_rs * 4);
        asm volatile("" : "+s"(ss_b));  // per tile: keeps the 64 offsets from being hoisted into registers
#pragma unroll
        for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const uint32_t row_b = (uint32_t)(32 * mb + 8 * (j >> 2) + (j & 3)) * ss_b;
            tv[mb][j] = *reinterpret_cast<const float*>(rb + (thr_lane_b + row_b));
          }
      } else {  // rows past the end read the last row (they take no part)
#pragma unroll
        for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
          for (int j = 0; j < 16; ++j)
            tv[mb][j] = p.thr[(int64_t)min(t * BQ + rg0 + 4 * g + 32 * mb + 8 * (j >> 2) + (j & 3), p.Sq - 1) * p.thr_rs + kjc];
      }
    }
    f32x16 sacc[NMB];
    qk_t(t, sacc);
    epi_t(t, sacc, ev, tv, masked);
  };

#pragma unroll
  for (int i = 0; i < NSTAGE - 1; ++i)
    if (t_begin + i < t_end) issue(t_begin + i);
  // The key fragments, once their copies have landed (those of the first Q tile may stay in flight; the last wave
  // issued NLSE more of them).
  if (t_begin >= t_end) wait_vmem<0>();
  else if (w == NW - 1) wait_vmem<GPW + NLSE>();
  else wait_vmem<GPW>();
  if constexpr (NG > 1) __syncthreads();
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk)
    kf[kk] = lds_read<V8>(kslot + (uint32_t)((r >> 2) * GROUP_B + s4 * ROW_B + 16 * g) + 64 * ((kk >> 1) ^ s4) +
                          32 * (kk & 1));
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    asm volatile("" : "+v"(kf[kk]));
    if (kj >= p.Sk) kf[kk] = V8{};
  }
  // Corm: whether this wave's keys are all decided (no tile of its range left, or every key flagged).
  bool wave_done = wt_begin >= wt_end;
  // Waits for the copies of tile t, then the barrier after which tile t+1 is requested into the stage of tile t-1
  // (every wave has finished with it).
  auto sync = [&](const int t) -> bool {
    wait_vmem<0>();
    if constexpr (EPI == kColAnyGe) {
      // Corm ORs over the query rows: once every key of every wave is flagged, no later tile can change the
      // result, and the workgroup stops. The vote doubles as the tile's barrier; the copies of this tile have
      // landed and none is in flight yet, so nothing still writes into the LDS when it stops.
      if (__syncthreads_and(wave_done)) return false;
    } else {
      __syncthreads();
    }
    if (t + 1 < t_end) issue(t + 1);
    return true;
  };
  auto step = [&](const int t, auto masked) -> bool {
    if (!sync(t)) return false;
    if (t >= wt_begin && t < wt_end) {
      tile(t, masked);
      if constexpr (EPI == kColAnyGe) {
        // this lane's key is decided when either half of its rows flagged it (keys past the end count as decided)
        const bool decided = (acc.any | __shfl_xor(acc.any, 32, 64)) != 0 || kj >= p.Sk;
        wave_done = t + 1 >= wt_end || __all(decided);
      }
    }
    return true;
  };
  bool go = true;
  for (int t = t_begin; go && t < t_full0; ++t) go = step(t, std::true_type{});
  for (int t = t_full0; go && t < t_full1; ++t) go = step(t, std::false_type{});
  for (int t = t_full1; go && t < t_end; ++t) go = step(t, std::true_type{});

  if constexpr (NG == 1) {
    acc.store(p, bh, kj, g);
  } else {
    // Row groups 1 .. leave their results (lane halves combined) in the LDS; group 0 combines them with its own, in
    // group order, and stores.
    wait_vmem<0>();
    __syncthreads();  // every wave is done with the Q stages
    float* red = reinterpret_cast<float*>(smem);  // [group - 1][2][BK]
    const int key = 32 * wi + r;                  // key within the workgroup
    if constexpr (EPI == kColAnyGe) {
      acc.any |= __shfl_xor(acc.any, 32, 64);
    } else {
      acc.s += __shfl_xor(acc.s, 32, 64);
      if constexpr (EPI == kColSumSq) acc.s2 += __shfl_xor(acc.s2, 32, 64);
    }
    float t1 = EPI == kColAnyGe ? (acc.any ? 1.0f : 0.0f) : acc.s, t2 = acc.s2;
    if (gw > 0 && g == 0) {
      red[(gw - 1) * 2 * BK + key] = t1;
      if constexpr (EPI == kColSumSq) red[(gw - 1) * 2 * BK + BK + key] = t2;
    }
    __syncthreads();
    if (gw == 0 && g == 0 && kj < p.Sk) {
#pragma unroll
      for (int i = 0; i < NG - 1; ++i) {
        t1 += red[i * 2 * BK + key];
        if constexpr (EPI == kColSumSq) t2 += red[i * 2 * BK + BK + key];
      }
      if constexpr (EPI == kColAnyGe) {
        p.any_out[(int64_t)bh * p.Sk + kj] = t1 != 0.0f;
      } else {
        p.colsum[(int64_t)bh * p.Sk + kj] = t1;
        if constexpr (EPI == kColSumSq) p.colsum2[(int64_t)bh * p.Sk + kj] = t2;
      }
    }
  }
}

template <typename T, int D, bool MASK, bool SOFTCAP, int REFROUND, int EPI>
void launch_colsum(AttnParams p, hipStream_t st) {
  p.n_tiles = (p.Sk + kCBK - 1) / kCBK;
  const unsigned grid = (unsigned)p.n_tiles * p.B * p.Hq;
  hipLaunchKernelGGL((attn_colsum_kernel<T, D, MASK, SOFTCAP, REFROUND, EPI>), dim3(grid), dim3(kThreads), 0, st, p);
}

constexpr int kColMinKeys = 64;  // fewest keys per workgroup of a column pass

template <typename T, int NG, int OCC, bool MASK, bool SOFTCAP, int REFROUND, int EPI>
void launch_colsum_d128_form(AttnParams p, hipStream_t st) {
  constexpr int NW = 8, BQ = 128, BK = 32 * NW / NG;
  static_assert(BK >= kColMinKeys, "check_blocks");
  p.n_tiles = (p.Sk + BK - 1) / BK;
  launch_blocks(p, 64 * NW, [&](unsigned grid, const AttnParams& p) {
    if (p.lse_base2)
      hipLaunchKernelGGL((attn_colsum_d128_kernel<T, NW, NG, BQ, OCC, MASK, SOFTCAP, REFROUND, true, EPI>), dim3(grid),
                         dim3(64 * NW), 0, st, p);
    else
      hipLaunchKernelGGL((attn_colsum_d128_kernel<T, NW, NG, BQ, OCC, MASK, SOFTCAP, REFROUND, false, EPI>), dim3(grid),
                         dim3(64 * NW), 0, st, p);
  });
}

// head_dim 128 column passes: 8 waves, 128-row query tiles; 64 keys per workgroup in four row groups (NG 4) or 128 in
// two (NG 2). What counts is four waves per SIMD: each score costs ~6 vector instructions and one exponential against
// 1/32 of an MFMA, so waves at different points of their tiles fill the pipes better than any fixed order within one
// (fp16 reference-rounded sums, H=32, causal, S=4096: 92.3 us; 95.7 us for two waves per SIMD running the products of
// one tile under the exponentials of the previous, 256 keys per workgroup; 105 us for NG 2 at two waves per SIMD).
// * Sums: NG 4 up to 768 workgroups of 64 keys (S=1000: 12.6 us, NG 2 17.0; S=1536 19.9 / 21.5), NG 2 beyond, where
//   the chip is full and each query tile is read by half as many workgroups (2 x 1024: 17.3, NG 4 19.0).
// * Corm: NG 4 always (S=4096 44.3 us, NG 2 50.0 at its best, two waves per SIMD: its thresholds do not fit the
//   registers of four); the reference-rounded soft-cap likewise.
// * KeyFormer: NG 4 up to the same size (S=1000 19.7 us, NG 2 27.8); beyond, NG 2 at two waves per SIMD, whose rows of
//   exp_rand are read 512 bytes at a time (S=2048 64.9 us, NG 4 76.9; equal at S=4096).
template <typename T, bool MASK, bool SOFTCAP, int REFROUND, int EPI>
void launch_colsum_d128(const AttnParams& p, hipStream_t st) {
  const bool small = (int64_t)((p.Sk + 63) / 64) * p.B * p.Hq <= 768;
  constexpr bool NG4 = EPI == kColAnyGe || (SOFTCAP && REFROUND);
  if (NG4 || small) return launch_colsum_d128_form<T, 4, 4, MASK, SOFTCAP, REFROUND, EPI>(p, st);
  if constexpr (!NG4)
    launch_colsum_d128_form<T, 2, EPI == kColKF ? 2 : 4, MASK, SOFTCAP, REFROUND, EPI>(p, st);
}

template <typename T, int D, bool MASK, bool SOFTCAP, int REFROUND, int EPI>
void launch_col(const AttnParams& p, hipStream_t st) {
  if constexpr (D == 128) launch_colsum_d128<T, MASK, SOFTCAP, REFROUND, EPI>(p, st);
  else launch_colsum<T, D, MASK, SOFTCAP, REFROUND, EPI>(p, st);
}
template <typename T, int D, bool MASK, bool SOFTCAP>
void pick_col_ref(const AttnParams& p, bool ref, hipStream_t st) {
  with_ref_mode<D, SOFTCAP>(ref, p, [&](auto mode) {
    launch_col<T, D, MASK, SOFTCAP, decltype(mode)::value, kColSum>(p, st);
  });
}
// The RoCo / Corm epilogues exist for the mask-checking, soft-cap-free variants only (the reference cases are
// causal and have no soft-cap); the host rejects a soft-cap with them.
template <typename T, int D, int EPI>
void pick_col_epi(const AttnParams& p, bool ref, hipStream_t st) {
  with_ref_mode<D, false>(ref, p, [&](auto mode) { launch_col<T, D, true, false, decltype(mode)::value, EPI>(p, st); });
}
template <typename T, int D>
void pick_col(const AttnParams& p, bool ref, int epi, hipStream_t st) {
  if (epi == kColSumSq) return pick_col_epi<T, D, kColSumSq>(p, ref, st);
  if (epi == kColAnyGe) return pick_col_epi<T, D, kColAnyGe>(p, ref, st);
  if (epi == kColKF) return pick_col_epi<T, D, kColKF>(p, ref, st);
  const bool mask = p.causal || p.window > 0;
  const bool sc = p.softcap > 0.f;
  if (mask) {
    if (sc) pick_col_ref<T, D, true, true>(p, ref, st);
    else pick_col_ref<T, D, true, false>(p, ref, st);
  } else {
    if (sc) pick_col_ref<T, D, false, true>(p, ref, st);
    else pick_col_ref<T, D, false, false>(p, ref, st);
  }
}

template <typename T, int D, bool MASK, int REFROUND>
void launch_kf_rowlse(const AttnParams& p, bool vec, hipStream_t st) {
  if constexpr (D == 128) {
    // exp_rand as whole 16-byte chunks: aligned rows and a key count that ends on a chunk
    if (vec && p.Sk % 4 == 0) {
      launch_blocks(p, 512, [&](unsigned grid, const AttnParams& p) {
        hipLaunchKernelGGL((attn_kf_rowlse_dma_kernel<T, MASK, REFROUND>), dim3(grid), dim3(512), 0, st, p);
      });
      return;
    }
  }
  const unsigned grid = (unsigned)p.n_tiles * p.B * p.Hq;
  if (vec) hipLaunchKernelGGL((attn_kf_rowlse_kernel<T, D, MASK, REFROUND, true>), dim3(grid), dim3(kThreads), 0, st, p);
  else hipLaunchKernelGGL((attn_kf_rowlse_kernel<T, D, MASK, REFROUND, false>), dim3(grid), dim3(kThreads), 0, st, p);
}
template <typename T, int D>
void pick_kf_rowlse(const AttnParams& p, bool ref, bool vec, hipStream_t st) {
  const bool mask = p.causal || p.window > 0;
  with_ref_mode<D, false>(ref, p, [&](auto mode) {
    constexpr int R = decltype(mode)::value;
    if (mask) launch_kf_rowlse<T, D, true, R>(p, vec, st);
    else launch_kf_rowlse<T, D, false, R>(p, vec, st);
  });
}

}  // namespace

namespace dgg_attn {

// Shared host-side validation of the attention arguments.
int validate_attn(const char* op, const void* q, const void* k, int64_t B, int64_t Sq, int64_t Sk, int64_t Hq,
                  int64_t Hkv, int64_t D, const int64_t* strides, int nstrides, float scale, float softcap,
                  int64_t window, int dtype) {
  DGG_REQUIRE(dtype == DGG_F16 || dtype == DGG_BF16 || dtype == DGG_F32, DGG_ERR_DTYPE,
              "%s: dtype code %d not supported (attention kernels take f32, f16 or bf16)", op, dtype);
  DGG_REQUIRE(D == 64 || D == 128 || D == 256, DGG_ERR_UNSUPPORTED, "%s: head_dim %lld not supported (64, 128, 256)",
              op, (long long)D);
  DGG_REQUIRE(B >= 0 && Sq >= 0 && Sk >= 0, DGG_ERR_SHAPE, "%s: negative size", op);
  DGG_REQUIRE(Hq > 0 && Hkv > 0 && Hq % Hkv == 0, DGG_ERR_SHAPE,
              "%s: query heads (%lld) must be a positive multiple of kv heads (%lld)", op, (long long)Hq,
              (long long)Hkv);
  DGG_REQUIRE(Sq < (1ll << 30) && Sk < (1ll << 30) && B < (1ll << 20) && Hq < (1ll << 16), DGG_ERR_SHAPE,
              "%s: size too large", op);
  DGG_REQUIRE(B * Hq * ((std::max(Sq, Sk) + 127) / 128) < (1ll << 31), DGG_ERR_SHAPE, "%s: grid too large", op);
  DGG_REQUIRE(strides != nullptr, DGG_ERR_NULL, "%s: strides is NULL", op);
  for (int i = 0; i < nstrides; ++i) {
    DGG_REQUIRE(strides[i] >= 0 && strides[i] % 8 == 0, DGG_ERR_STRIDE,
                "%s: stride[%d] = %lld must be a non-negative multiple of 8 elements", op, i, (long long)strides[i]);
    // in-tile row offsets are 32-bit: 256 rows of the sequence stride must stay below 2^31 elements
    DGG_REQUIRE(i % 3 != 1 || strides[i] < (1ll << 23), DGG_ERR_STRIDE,
                "%s: sequence stride[%d] = %lld must be < 2^23 elements", op, i, (long long)strides[i]);
  }
  DGG_REQUIRE(std::isfinite(scale) && scale > 0.f, DGG_ERR_SHAPE, "%s: scale must be finite and > 0", op);
  DGG_REQUIRE(softcap >= 0.f && std::isfinite(softcap), DGG_ERR_SHAPE, "%s: softcap must be >= 0 (0 = off)", op);
  DGG_REQUIRE(window >= 0 && window < (1ll << 30), DGG_ERR_SHAPE, "%s: window must be >= 0 (0 = off)", op);
  // q is read whenever there are query rows (the forward kernels load it even when Sk == 0), k whenever there are
  // keys.
  if (B > 0 && Sq > 0) {
    DGG_REQUIRE(q != nullptr, DGG_ERR_NULL, "%s: null q pointer", op);
    DGG_REQUIRE(dgg::aligned16(q), DGG_ERR_ALIGN, "%s: q must be 16-byte aligned", op);
  }
  if (B > 0 && Sk > 0) {
    DGG_REQUIRE(k != nullptr, DGG_ERR_NULL, "%s: null k pointer", op);
    DGG_REQUIRE(dgg::aligned16(k), DGG_ERR_ALIGN, "%s: k must be 16-byte aligned", op);
  }
  return DGG_OK;
}

AttnParams make_params(const void* q, const void* k, const void* v, void* o, int64_t B, int64_t Sq, int64_t Sk,
                       int64_t Hq, int64_t Hkv, int64_t D, float scale, float softcap, int64_t window, uint32_t flags) {
  AttnParams p{};
  p.q = q;
  p.k = k;
  p.v = v;
  p.o = o;
  p.B = (int)B;
  p.Sq = (int)Sq;
  p.Sk = (int)Sk;
  p.Hq = (int)Hq;
  p.Hkv = (int)Hkv;
  p.group = (int)(Hq / Hkv);
  p.causal = (flags & DGG_ATTN_CAUSAL) ? 1 : 0;
  p.lse_base2 = (flags & DGG_ATTN_LSE_BASE2) ? 1 : 0;
  p.window = (int)window;
  p.offset = (int)(Sk - Sq);
  p.scale = scale;
  // The reference divides its scores by math.sqrt(D) (attn.py:29); torch takes that Python float to fp32 and
  // multiplies by the fp32 reciprocal. A scale other than the default is taken as 1 / divisor.
  const double root = std::sqrt((double)D);
  p.ref_div = scale == (float)(1.0 / root) ? (float)root : (float)(1.0 / (double)scale);
  p.ref_rcp = 1.0f / p.ref_div;
  p.c_fast = scale * kLog2e;
  p.softcap = softcap;
  p.inv_softcap = softcap > 0.f ? 1.0f / softcap : 0.f;
  p.sc_a = softcap > 0.f ? 2.0f * scale / softcap * kLog2e : 0.f;
  p.sc_b = softcap * kLog2e;
  return p;
}

}  // namespace dgg_attn

namespace {
// Shared body of dgg_attn_prefill and dgg_attn_prefill_rope (rope: rotate the query rows by the table rope_cs).
int prefill_impl(const char* op, const void* q, const void* k, const void* v, void* o, float* lse, int64_t B,
                 int64_t Sq, int64_t Sk, int64_t Hq, int64_t Hkv, int64_t D, const int64_t* strides, float scale,
                 float softcap, int64_t window, uint32_t flags, int dtype, bool rope, const float* rope_cs,
                 void* stream) {
  if (int rc = validate_attn(op, q, k, B, Sq, Sk, Hq, Hkv, D, strides, 12, scale, softcap, window, dtype)) return rc;
  if (rope)
    DGG_REQUIRE(D == 128 && dtype != DGG_F32, DGG_ERR_UNSUPPORTED,
                "%s: the fused rotary takes head_dim 128 (pos_encoding.cu:195) and 16-bit inputs", op);
  if (B == 0 || Sq == 0) return DGG_OK;
  DGG_REQUIRE(o && (v || Sk == 0), DGG_ERR_NULL, "%s: null v/o pointer", op);
  DGG_REQUIRE(dgg::aligned16(v) && dgg::aligned16(o), DGG_ERR_ALIGN, "%s: v/o must be 16-byte aligned", op);
  if (rope) {
    DGG_REQUIRE(rope_cs != nullptr, DGG_ERR_NULL, "%s: null rotary table", op);
    DGG_REQUIRE(((uintptr_t)rope_cs & 31u) == 0, DGG_ERR_ALIGN, "%s: the rotary table must be 32-byte aligned", op);
  }
  AttnParams p = make_params(q, k, v, o, B, Sq, Sk, Hq, Hkv, D, scale, softcap, window, flags);
  p.rope_cs = rope_cs;
  p.lse = lse;
  p.q_sb = strides[0]; p.q_ss = strides[1]; p.q_sh = strides[2];
  p.k_sb = strides[3]; p.k_ss = strides[4]; p.k_sh = strides[5];
  p.v_sb = strides[6]; p.v_ss = strides[7]; p.v_sh = strides[8];
  p.o_sb = strides[9]; p.o_ss = strides[10]; p.o_sh = strides[11];
  const bool ref = (flags & DGG_ATTN_REF_ROUNDING) != 0;
  hipStream_t st = dgg::as_stream(stream);
  // Sk == 0 still launches and writes o = 0 (the reference's P.V over an empty key axis) and lse = -inf.
  if (dtype == DGG_F32) {  // fp32 has no 16-bit rounding point: reference rounding changes nothing
    if (int rc = check_blocks(op, Sq, kF32Rows, B, Hq)) return rc;
    launch_attn_f32_fwd(p, (int)D, st);
    return dgg::check_launch(op);
  }
  if (dtype == DGG_BF16) launch_attn_fwd_bf16(p, (int)D, ref, st);
  else launch_attn_fwd_f16(p, (int)D, ref, st);
  return dgg::check_launch(op);
}
}  // namespace

extern "C" int dgg_attn_prefill(const void* q, const void* k, const void* v, void* o, float* lse, int64_t B,
                                int64_t Sq, int64_t Sk, int64_t Hq, int64_t Hkv, int64_t D, const int64_t* strides,
                                float scale, float softcap, int64_t window, uint32_t flags, int dtype, void* stream) {
  return prefill_impl("attn_prefill", q, k, v, o, lse, B, Sq, Sk, Hq, Hkv, D, strides, scale, softcap, window, flags,
                      dtype, false, nullptr, stream);
}

extern "C" int dgg_attn_prefill_rope(const void* q, const void* k, const void* v, void* o, float* lse, int64_t B,
                                     int64_t Sq, int64_t Sk, int64_t Hq, int64_t Hkv, int64_t D,
                                     const int64_t* strides, float scale, float softcap, int64_t window,
                                     uint32_t flags, int dtype, const float* q_cos_sin, void* stream) {
  return prefill_impl("attn_prefill_rope", q, k, v, o, lse, B, Sq, Sk, Hq, Hkv, D, strides, scale, softcap, window,
                      flags, dtype, true, q_cos_sin, stream);
}

namespace {
// Corm over the masked pairs (corm.py:35-37 compares every query row, masked pairs included): a masked pair of a
// row that sees at least one key has p = 0 (softmax of -inf), so it flags its key when thr[i][j] <= 0; a row that
// sees no key at all has NaN probabilities (0 / 0) and flags nothing. The column kernels compare the visible pairs
// only; this kernel, run after them on the same stream, sets any_out[bh][j] = 1 for every (batch, head) when some
// masked pair of a non-empty row has thr[i][j] <= 0 (the thresholds are shared by all heads). One thread per key and
// chunk of kMaskedRows rows, reading only the masked part of the chunk: for causal the rows before the key's
// diagonal, for a window the rows past its end. Flags are written only when found, as plain byte stores of 1.
constexpr int kMaskedRows = 64;
__global__ void __launch_bounds__(256) corm_masked_or_kernel(const float* __restrict__ thr, int64_t rs, int Sq, int Sk,
                                                             int offset, int causal, int window, uint8_t* any_out,
                                                             int64_t nbh) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= Sk) return;
  const int r0 = blockIdx.y * kMaskedRows, r1 = min(Sq, r0 + kMaskedRows);
  // masked rows of key j: [a0, a1) before the diagonal (rows i + offset < j that see a key: i + offset >= 0),
  // [b0, r1) past the window (i + offset - j >= window)
  int a0 = r1, a1 = r1, b0 = r1;
  const int64_t diag = (int64_t)j - offset;  // first row that sees key j (causal)
  if (causal) {
    a0 = (int)max<int64_t>(r0, max<int64_t>(0, -(int64_t)offset));
    a1 = (int)min<int64_t>(r1, diag);
  }
  if (window > 0) b0 = (int)min<int64_t>(r1, max<int64_t>(r0, diag + window));  // never overlaps [a0, a1)
  bool hit = false;
#pragma unroll 8
  for (int i = a0; i < a1; ++i) hit |= thr[(int64_t)i * rs + j] <= 0.f;
#pragma unroll 8
  for (int i = b0; i < r1; ++i) hit |= thr[(int64_t)i * rs + j] <= 0.f;
  if (hit)
    for (int64_t bh = 0; bh < nbh; ++bh) any_out[bh * Sk + j] = 1;
}

// Shared body of dgg_attn_colsum and dgg_attn_colscore.
int colscore(const char* op, const void* q, const void* k, const float* lse, int epi, float* out0, float* out1,
             uint8_t* out_any, const float* thr, int64_t thr_row_stride, int64_t B, int64_t Sq, int64_t Sk, int64_t Hq,
             int64_t Hkv, int64_t D, const int64_t* strides, float scale, float softcap, int64_t window, uint32_t flags,
             int dtype, void* stream) {
  if (int rc = validate_attn(op, q, k, B, Sq, Sk, Hq, Hkv, D, strides, 6, scale, softcap, window, dtype)) return rc;
  DGG_REQUIRE(epi == kColSum || epi == kColSumSq || epi == kColAnyGe, DGG_ERR_UNSUPPORTED, "%s: unknown epilogue %d", op,
              epi);
  DGG_REQUIRE(epi == kColSum || softcap == 0.f, DGG_ERR_UNSUPPORTED, "%s: epilogue %d takes no soft-cap", op, epi);
  if (B == 0 || Sk == 0) return DGG_OK;
  if (int rc = check_blocks(op, Sk, kColMinKeys, B, Hq)) return rc;
  if (epi == kColAnyGe) {
    DGG_REQUIRE(out_any != nullptr, DGG_ERR_NULL, "%s: null output pointer", op);
    DGG_REQUIRE(Sq == 0 || thr != nullptr, DGG_ERR_NULL, "%s: null threshold pointer", op);
    DGG_REQUIRE(Sq == 0 || (thr_row_stride >= Sk && thr_row_stride < (1ll << 40)), DGG_ERR_STRIDE,
                "%s: threshold row stride %lld must be >= Sk (%lld)", op, (long long)thr_row_stride, (long long)Sk);
  } else {
    DGG_REQUIRE(out0 != nullptr && (epi != kColSumSq || out1 != nullptr), DGG_ERR_NULL, "%s: null output pointer", op);
  }
  DGG_REQUIRE(Sq == 0 || lse != nullptr, DGG_ERR_NULL, "%s: null lse pointer", op);
  AttnParams p = make_params(q, k, nullptr, nullptr, B, Sq, Sk, Hq, Hkv, D, scale, softcap, window, flags);
  p.lse = const_cast<float*>(lse);
  p.colsum = out0;
  p.colsum2 = out1;
  p.any_out = out_any;
  p.thr = thr;
  p.thr_rs = thr_row_stride;
  p.thr_lane32 = (132 * thr_row_stride + Sk) * 4 < (1ll << 31) ? 1 : 0;
  p.q_sb = strides[0]; p.q_ss = strides[1]; p.q_sh = strides[2];
  p.k_sb = strides[3]; p.k_ss = strides[4]; p.k_sh = strides[5];
  hipStream_t st = dgg::as_stream(stream);
  if (dtype == DGG_F32) {
    p.n_tiles = (int)((Sk + f32_rows_per_tile() - 1) / f32_rows_per_tile());
    launch_attn_f32_col(p, (int)D, epi, st);
  } else {
    const bool ref = (flags & DGG_ATTN_REF_ROUNDING) != 0;
    if (dtype == DGG_BF16) {
      if (D == 64) pick_col<BF16, 64>(p, ref, epi, st);
      else if (D == 128) pick_col<BF16, 128>(p, ref, epi, st);
      else pick_col<BF16, 256>(p, ref, epi, st);
    } else {
      if (D == 64) pick_col<F16, 64>(p, ref, epi, st);
      else if (D == 128) pick_col<F16, 128>(p, ref, epi, st);
      else pick_col<F16, 256>(p, ref, epi, st);
    }
  }
  if (epi == kColAnyGe && Sq > 0 && (p.causal || p.window > 0)) {
    const dim3 grid((unsigned)((Sk + 255) / 256), (unsigned)((Sq + kMaskedRows - 1) / kMaskedRows));
    hipLaunchKernelGGL(corm_masked_or_kernel, grid, dim3(256), 0, st, thr, thr_row_stride, (int)Sq, (int)Sk, p.offset,
                       p.causal, p.window, out_any, B * Hq);
  }
  return dgg::check_launch(op);
}
}  // namespace

namespace {
// exp_rand [B, Hq, Sq, Sk] fp32 with element strides er_strides = {batch, head, row} and unit key stride.
int validate_exp_rand(const char* op, const float* er, const int64_t* er_strides, int64_t Sq, float tau) {
  DGG_REQUIRE(er != nullptr && er_strides != nullptr, DGG_ERR_NULL, "%s: null exp_rand / strides", op);
  DGG_REQUIRE(((uintptr_t)er & 3u) == 0, DGG_ERR_ALIGN, "%s: exp_rand must be 4-byte aligned", op);
  for (int i = 0; i < 3; ++i)
    DGG_REQUIRE(er_strides[i] >= 0 && er_strides[i] < (1ll << 40), DGG_ERR_STRIDE, "%s: exp_rand stride[%d] invalid", op,
                i);
  DGG_REQUIRE(Sq <= 1 || er_strides[2] > 0, DGG_ERR_STRIDE, "%s: exp_rand row stride must be > 0", op);
  DGG_REQUIRE(std::isfinite(tau) && tau > 0.f, DGG_ERR_SHAPE, "%s: tau must be finite and > 0", op);
  return DGG_OK;
}
void set_exp_rand(AttnParams& p, const float* er, const int64_t* er_strides, float tau) {
  p.er = er;
  p.er_sb = er_strides[0];
  p.er_sh = er_strides[1];
  p.er_ss = er_strides[2];
  p.kf_inv_tau = 1.0f / tau;
  p.er_lane32 = (132 * er_strides[2] + p.Sk) * 4 < (1ll << 31) ? 1 : 0;
}
}  // namespace

extern "C" int dgg_attn_kf_rowlse(const void* q, const void* k, const float* exp_rand, const int64_t* er_strides,
                                  float* lse2, int64_t B, int64_t Sq, int64_t Sk, int64_t Hq, int64_t Hkv, int64_t D,
                                  const int64_t* strides, float scale, float tau, int64_t window, uint32_t flags,
                                  int dtype, void* stream) {
  const char* op = "attn_kf_rowlse";
  DGG_REQUIRE(dtype == DGG_F16 || dtype == DGG_BF16, DGG_ERR_DTYPE,
              "%s: dtype code %d not supported (the KeyFormer passes take f16 or bf16)", op, dtype);
  if (int rc = validate_attn(op, q, k, B, Sq, Sk, Hq, Hkv, D, strides, 6, scale, 0.f, window, dtype)) return rc;
  if (B == 0 || Sq == 0) return DGG_OK;
  DGG_REQUIRE(lse2 != nullptr, DGG_ERR_NULL, "%s: null lse output", op);
  DGG_REQUIRE(Sk > 0, DGG_ERR_SHAPE, "%s: Sk must be > 0", op);
  if (int rc = validate_exp_rand(op, exp_rand, er_strides, Sq, tau)) return rc;
  AttnParams p = make_params(q, k, nullptr, nullptr, B, Sq, Sk, Hq, Hkv, D, scale, 0.f, window, flags);
  p.lse = lse2;
  p.q_sb = strides[0]; p.q_ss = strides[1]; p.q_sh = strides[2];
  p.k_sb = strides[3]; p.k_ss = strides[4]; p.k_sh = strides[5];
  set_exp_rand(p, exp_rand, er_strides, tau);
  p.n_tiles = (int)((Sq + kBM - 1) / kBM);
  const bool vec = dgg::aligned16(exp_rand) && er_strides[0] % 4 == 0 && er_strides[1] % 4 == 0 && er_strides[2] % 4 == 0;
  const bool ref = (flags & DGG_ATTN_REF_ROUNDING) != 0;
  hipStream_t st = dgg::as_stream(stream);
  if (dtype == DGG_BF16) {
    if (D == 64) pick_kf_rowlse<BF16, 64>(p, ref, vec, st);
    else if (D == 128) pick_kf_rowlse<BF16, 128>(p, ref, vec, st);
    else pick_kf_rowlse<BF16, 256>(p, ref, vec, st);
  } else {
    if (D == 64) pick_kf_rowlse<F16, 64>(p, ref, vec, st);
    else if (D == 128) pick_kf_rowlse<F16, 128>(p, ref, vec, st);
    else pick_kf_rowlse<F16, 256>(p, ref, vec, st);
  }
  return dgg::check_launch(op);
}

extern "C" int dgg_attn_kf_colsum(const void* q, const void* k, const float* exp_rand, const int64_t* er_strides,
                                  const float* lse2, float* kf_score, int64_t B, int64_t Sq, int64_t Sk, int64_t Hq,
                                  int64_t Hkv, int64_t D, const int64_t* strides, float scale, float tau,
                                  int64_t window, uint32_t flags, int dtype, void* stream) {
  const char* op = "attn_kf_colsum";
  DGG_REQUIRE(dtype == DGG_F16 || dtype == DGG_BF16, DGG_ERR_DTYPE,
              "%s: dtype code %d not supported (the KeyFormer passes take f16 or bf16)", op, dtype);
  if (int rc = validate_attn(op, q, k, B, Sq, Sk, Hq, Hkv, D, strides, 6, scale, 0.f, window, dtype)) return rc;
  if (B == 0 || Sk == 0) return DGG_OK;
  if (int rc = check_blocks(op, Sk, kColMinKeys, B, Hq)) return rc;
  DGG_REQUIRE(kf_score != nullptr, DGG_ERR_NULL, "%s: null output", op);
  DGG_REQUIRE(Sq == 0 || lse2 != nullptr, DGG_ERR_NULL, "%s: null lse pointer", op);
  if (Sq > 0)
    if (int rc = validate_exp_rand(op, exp_rand, er_strides, Sq, tau)) return rc;
  // The row lse of the perturbed scores is base 2 (as dgg_attn_kf_rowlse writes it).
  AttnParams p = make_params(q, k, nullptr, nullptr, B, Sq, Sk, Hq, Hkv, D, scale, 0.f, window,
                             flags | DGG_ATTN_LSE_BASE2);
  p.lse = const_cast<float*>(lse2);
  p.colsum = kf_score;
  p.q_sb = strides[0]; p.q_ss = strides[1]; p.q_sh = strides[2];
  p.k_sb = strides[3]; p.k_ss = strides[4]; p.k_sh = strides[5];
  if (Sq > 0) set_exp_rand(p, exp_rand, er_strides, tau);
  const bool ref = (flags & DGG_ATTN_REF_ROUNDING) != 0;
  hipStream_t st = dgg::as_stream(stream);
  if (dtype == DGG_BF16) {
    if (D == 64) pick_col<BF16, 64>(p, ref, kColKF, st);
    else if (D == 128) pick_col<BF16, 128>(p, ref, kColKF, st);
    else pick_col<BF16, 256>(p, ref, kColKF, st);
  } else {
    if (D == 64) pick_col<F16, 64>(p, ref, kColKF, st);
    else if (D == 128) pick_col<F16, 128>(p, ref, kColKF, st);
    else pick_col<F16, 256>(p, ref, kColKF, st);
  }
  return dgg::check_launch(op);
}

extern "C" int dgg_attn_colsum(const void* q, const void* k, const float* lse, float* colsum, int64_t B, int64_t Sq,
                               int64_t Sk, int64_t Hq, int64_t Hkv, int64_t D, const int64_t* strides, float scale,
                               float softcap, int64_t window, uint32_t flags, int dtype, void* stream) {
  return colscore("attn_colsum", q, k, lse, kColSum, colsum, nullptr, nullptr, nullptr, 0, B, Sq, Sk, Hq, Hkv, D, strides,
                  scale, softcap, window, flags, dtype, stream);
}

extern "C" int dgg_attn_colscore(const void* q, const void* k, const float* lse, int epilogue, float* out0, float* out1,
                                 uint8_t* out_any, const float* thr, int64_t thr_row_stride, int64_t B, int64_t Sq,
                                 int64_t Sk, int64_t Hq, int64_t Hkv, int64_t D, const int64_t* strides, float scale,
                                 float softcap, int64_t window, uint32_t flags, int dtype, void* stream) {
  return colscore("attn_colscore", q, k, lse, epilogue, out0, out1, out_any, thr, thr_row_stride, B, Sq, Sk, Hq, Hkv,
                  D, strides, scale, softcap, window, flags, dtype, stream);
}
