// Fused online-softmax attention forward for 16-bit inputs: kernels and launch rules, instantiated per storage type by
// attention_fwd_f16.hip and attention_fwd_bf16.hip (two translation units, so that they compile side by side).
#pragma once

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"

#include "attention_common.h"

// DGG_SPREAD_COPIES (default 1): mask-free tiles of the direct-load forward issue the next tile's copies among their
// QK^T MFMAs; 0 issues them all right after the barrier (for A/B measurements).
#ifndef DGG_SPREAD_COPIES
#define DGG_SPREAD_COPIES 1
#endif

namespace {

using namespace dgg_attn;

// Forward kernel: NW waves of 32 query rows over a ring of NSTAGE tiles of BN keys. KG: waves that share the same 32
// rows, each taking BN / KG keys of every tile (its own running maximum, row sum and O, combined through the LDS at the
// end), so a workgroup covers 32 * NW / KG rows. OCC: waves per SIMD the register budget is sized for. FASTSUM: the row
// sums add the 16-bit rounded probabilities two at a time (v_dot2); used at head_dim 128 and 256 when no lse is written,
// since the O normalisation tolerates the rounding but the column-sum pass needs the fp32 row sums.
template <typename T, int D, int NW, int KG, int BN, int NSTAGE, int OCC, bool MASK, bool SOFTCAP, int REFROUND, bool FASTSUM>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(OCC, OCC)))
attn_fwd_dma_kernel(AttnParams p) {
  typedef DmaLayout<D> L;
  constexpr int ROW_B = L::ROW_B, GROUP_B = L::GROUP_B, GR = L::GR, LPR = L::LPR, RPI = L::RPI, IPG = L::IPG;
  typedef typename T::scalar S;
  typedef typename T::vec8 V8;
  typedef typename T::vec4 V4;
  // 32-row query blocks per wave. One in every launch, as NSTAGE is 2; the loops over it and the waits for deeper rings stay
  // in the text because the compiler orders the same program without them worse (S=4096 causal, bf16: 134.9 -> 136.3 us).
  constexpr int NQB = 1;
  constexpr int QPW = 32 * NQB;                 // query rows per wave
  constexpr int NWR = NW / KG;                  // waves along the query rows
  constexpr int BM = QPW * NWR;                 // query rows per workgroup
  constexpr int SBN = BN / KG;                  // keys of a tile taken by each wave
  constexpr int TILE_B = (BN / GR) * GROUP_B;
  constexpr int STAGE_B = 2 * TILE_B;           // K tile, then V tile
  constexpr int GPW = (BN / GR) / NW;           // row groups of a tile copied by each wave (K and V each)
  constexpr int DMA_PER_TILE = 2 * GPW * IPG;   // direct loads per wave per tile
  static_assert(GPW >= 1 && GPW * NW == BN / GR, "tile groups must split over the waves");
  static_assert(NWR * KG == NW && SBN % 32 == 0 && D / 8 % KG == 0, "key groups");
  constexpr int OQ_B = 64 * 16 + 16;            // key groups' exchange: one quad of O registers of a wave + pad
  constexpr int SLOT_B = (D / 8) * OQ_B;        // one wave's O
  constexpr int SMEM_B = std::max(NSTAGE * STAGE_B, KG > 1 ? NW * (SLOT_B + 32 * 8) : 0);
  __shared__ __attribute__((aligned(1024))) char smem[SMEM_B];

  int qt, bh;
  map_block_kv(p.n_tiles, p.B, p.Hq, p.Hkv, true, qt, bh);
  const int b = bh / p.Hq, h = bh - b * p.Hq;
  const int hk = h / p.group;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q0 = qt * BM;
  const int wr = KG == 1 ? w : w % NWR, kg = KG == 1 ? 0 : w / NWR;  // row block and key group of this wave
  const int koff = SBN * kg;      // its keys within a tile: [koff, koff + SBN)
  const int qw0 = q0 + QPW * wr;  // first query row of this wave; lane rows qw0 + 32n + r

  const S* qp = static_cast<const S*>(p.q) + b * p.q_sb + h * p.q_sh;
  const char* kp = reinterpret_cast<const char*>(static_cast<const S*>(p.k) + b * p.k_sb + hk * p.k_sh);
  const char* vp = reinterpret_cast<const char*>(static_cast<const S*>(p.v) + b * p.v_sb + hk * p.v_sh);
  const int64_t k_ss_b = p.k_ss * (int64_t)sizeof(S), v_ss_b = p.v_ss * (int64_t)sizeof(S);

  V8 qf[NQB][D / 16];
  // BIAS (bf16 without soft-cap or reference rounding, no lse): Q is pre-scaled by scale*log2(e) and each score
  // accumulator starts from -m (the row's reference maximum) through one extra MFMA whose A fragment is the
  // constant column e_0 and whose B fragment holds -m in k-slot 0. The accumulator then holds s*c - m and
  // P = exp2(acc) needs no per-element arithmetic. The reference maxima are bf16 values so that -m is exact in
  // the B operand; the pre-scaled Q carries the same 2^-9 relative rounding as the reference's bf16 scores.
  constexpr bool BIAS = D == 128 && FASTSUM && !SOFTCAP && !REFROUND && std::is_same<T, BF16>::value;
  V8 abias = V8{};
  abias[0] = g == 0 ? to_s<S>(1.0f) : to_s<S>(0.0f);
  V8 bbias[NQB];
#pragma unroll
  for (int n = 0; n < NQB; ++n) bbias[n] = V8{};

  // Key tiles of the workgroup and of this wave.
  const int q_last = min(q0 + BM, p.Sq) - 1;
  int k_begin = 0, k_end = p.Sk;
  if (p.causal) k_end = min(p.Sk, q_last + p.offset + 1);
  if (p.window > 0) k_begin = max(0, q0 + p.offset - p.window + 1);
  const int t_begin = k_begin / BN;
  const int t_end = k_end > k_begin ? (k_end + BN - 1) / BN : t_begin;
  const int wq_last = min(qw0 + QPW, p.Sq) - 1;  // may be < qw0 for a wave past the end
  int wk_begin = 0, wk_end = p.Sk;
  if (p.causal) wk_end = min(p.Sk, wq_last + p.offset + 1);
  if (p.window > 0) wk_begin = max(0, qw0 + p.offset - p.window + 1);

  // Visible keys per lane row: lo <= key <= hi.
  int k_hi[NQB], k_lo[NQB];
#pragma unroll
  for (int n = 0; n < NQB; ++n) {
    const int qi = qw0 + 32 * n + r;
    k_hi[n] = p.Sk - 1;
    k_lo[n] = 0;
    if (p.causal) k_hi[n] = min(k_hi[n], qi + p.offset);
    if (p.window > 0) k_lo[n] = max(k_lo[n], qi + p.offset - p.window + 1);
  }

  // Direct-load lane constants: in load i of row group j of a tile, lane l fills LDS position l%LPR of the group's row
  // i*RPI + l/LPR, fetching the global chunk that the layout puts there. VI(j, i): the lane constants of that load.
  constexpr int NV = L::NV;
  auto VI = [](int j, int i) { return D == 64 ? j & 1 : i; };
  uint32_t src_chunk[NV], k_voff[NV], v_voff[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int grow = (D == 64 ? 0 : i * RPI) + lane / LPR;  // row within the group
    const int trow = D == 64 ? GR * (GPW * w + i) + grow : grow;  // (D == 64: the layout also looks at the group)
    src_chunk[i] = (uint32_t)((lane % LPR) ^ L::swizzle(trow));
    k_voff[i] = (uint32_t)(grow * k_ss_b) + src_chunk[i] * 16u;
    v_voff[i] = (uint32_t)(grow * v_ss_b) + src_chunk[i] * 16u;
    asm volatile("" : "+v"(k_voff[i]), "+v"(v_voff[i]));
  }
  const uint32_t smem_base = (uint32_t)(size_t)((lds_char*)smem);

  // Q tile: copied to the LDS stage that the first tile's step fills next (read into registers before that step's
  // barrier), 32 rows per row block in the tiles' layout, the KG waves of a row block taking the row groups in turn.
  // Loading the fragments straight from global memory takes D/16 loads per wave with 64 lanes on 32 rows each, ~64
  // cycles of address processing per load: 1.7-2.3 us per workgroup at head_dim 128 (measured with the real-time
  // counter), against 8 coalesced 1 KiB copies. Rows past the end read the last row and are zeroed afterwards.
  constexpr int QSLOT_B = (32 / GR) * GROUP_B;
  static_assert(NWR * QSLOT_B <= STAGE_B, "the Q tile fits one stage");
  const uint32_t q_slot = smem_base + (uint32_t)(((t_begin + NSTAGE - 1) % NSTAGE) * STAGE_B + wr * QSLOT_B);
  {
    const char* qb = reinterpret_cast<const char*>(qp);
#pragma unroll
    for (int j = 0; j < 32 / GR; ++j) {
      if (KG > 1 && j % KG != kg) continue;
#pragma unroll
      for (int i = 0; i < IPG; ++i) {
        const int trow = GR * j + i * RPI + lane / LPR;
        const int64_t row = min(qw0 + trow, p.Sq - 1);
        dma16(q_slot + j * GROUP_B + i * RPI * ROW_B,
              qb + row * (p.q_ss * (int64_t)sizeof(S)) + 16 * ((lane % LPR) ^ L::swizzle(trow)));
      }
    }
  }
  // Fused rotary of the query (head_dim 128): the (cos, sin) of this lane's 32 rotary pairs, requested with Q so
  // that the two latencies overlap. The lane holds elements 16kk + 8g + e of fragment kk and their pair partners (+64)
  // in fragment kk + 4, so it rotates its own pairs.
  constexpr int NRC = D == 128 ? NQB : 0;
  f32x8 rcos[NRC > 0 ? NRC : 1][4], rsin[NRC > 0 ? NRC : 1][4];
  const bool rope = D == 128 && p.rope_cs != nullptr;
  if constexpr (NRC > 0) {
    if (rope) {
#pragma unroll
      for (int n = 0; n < NQB; ++n) {
        const float* cs = p.rope_cs + ((int64_t)b * p.Sq + min(qw0 + 32 * n + r, p.Sq - 1)) * D + 8 * g;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          rcos[n][kk] = *reinterpret_cast<const f32x8*>(cs + 16 * kk);
          rsin[n][kk] = *reinterpret_cast<const f32x8*>(cs + 64 + 16 * kk);
        }
      }
    }
  }

  // Copies groups GPW*w .. GPW*w + GPW-1 of tile t into stage t % NSTAGE: DMA_PER_TILE loads per wave.
  auto issue = [&](int t) {
    const uint32_t kdst = smem_base + (uint32_t)((t % NSTAGE) * STAGE_B + GPW * w * GROUP_B);
    const uint32_t vdst = kdst + TILE_B;
    const int row0 = t * BN + GR * GPW * w;
    if ((t + 1) * BN <= p.Sk) {
      const char* kb = kp + (int64_t)row0 * k_ss_b;
      const char* vb = vp + (int64_t)row0 * v_ss_b;
#pragma unroll
      for (int j = 0; j < GPW; ++j)
#pragma unroll
        for (int i = 0; i < IPG; ++i) {
          dma16(kdst + j * GROUP_B + i * RPI * ROW_B, kb + GR * j * k_ss_b, k_voff[VI(j, i)]);
          dma16(vdst + j * GROUP_B + i * RPI * ROW_B, vb + GR * j * v_ss_b, v_voff[VI(j, i)]);
        }
    } else {  // ragged last tile: rows past the end re-read the last row (always masked, finite)
#pragma unroll
      for (int j = 0; j < GPW; ++j)
#pragma unroll
        for (int i = 0; i < IPG; ++i) {
          const int64_t row = min(row0 + GR * j + i * RPI + lane / LPR, p.Sk - 1);
          dma16(kdst + j * GROUP_B + i * RPI * ROW_B, kp + row * k_ss_b + src_chunk[VI(j, i)] * 16);
          dma16(vdst + j * GROUP_B + i * RPI * ROW_B, vp + row * v_ss_b + src_chunk[VI(j, i)] * 16);
        }
    }
  };

  // Load i (0 .. DMA_PER_TILE-1) of issue(t) for a tile whose rows all exist: the K loads, then the V loads. The
  // mask-free tiles issue the next tile's copies one per QK^T step with these, so that the copies' issue overlaps
  // the MFMAs instead of following the barrier as one burst (which held every wave of the workgroup at once).
  auto issue_one = [&](int t, int i) __attribute__((always_inline)) {
    const uint32_t kdst = smem_base + (uint32_t)((t % NSTAGE) * STAGE_B + GPW * w * GROUP_B);
    const int row0 = t * BN + GR * GPW * w;
    const int half = GPW * IPG, ii = i % half, j = ii / IPG, l = ii % IPG;
    if (i < half)
      dma16(kdst + j * GROUP_B + l * RPI * ROW_B, kp + (int64_t)row0 * k_ss_b + GR * j * k_ss_b, k_voff[VI(j, l)]);
    else
      dma16(kdst + TILE_B + j * GROUP_B + l * RPI * ROW_B, vp + (int64_t)row0 * v_ss_b + GR * j * v_ss_b, v_voff[VI(j, l)]);
  };
  constexpr int CPS = (DMA_PER_TILE + D / 16 - 1) / (D / 16);  // copies per QK^T step

  // LDS read addressing: a per-lane base (xk / xv), to which the tile loop adds the stage and a constant offset.
  // K fragment kk of key block mb: row mb*32 + r, chunk 2kk + g: base KI(kk), constant KO(mb, kk).
  // V transposing read (rows 16kk + 4g + (lane%16)/4, hi: + 8; head-dim column db*32 + 16*((lane/16)%2) +
  // 4*(lane%4)): base VB(db, hi), constant VO(kk, hi).
  constexpr int NKB = D == 64 ? D / 16 : D / 32, NVB = D == 64 ? 2 * (D / 32) : D / 32;
  auto KI = [](int kk) { return D == 64 ? kk : kk >> 1; };
  auto KO = [](int mb, int kk) { return mb * (32 / GR) * GROUP_B + (D == 64 ? 0 : 32 * (kk & 1)); };
  auto VB = [](int db, int hi) { return D == 64 ? 2 * db + hi : db; };
  auto VO = [](int kk, int hi) { return kk * (16 / GR) * GROUP_B + hi * (8 / GR) * GROUP_B; };
  const int m4 = (lane & 15) >> 2, m3 = lane & 3;
  uint32_t xq[NKB], xk[NKB], xv[NVB];
#pragma unroll
  for (int i = 0; i < NKB; ++i) {
    const int chunk = D == 64 ? 2 * i + g : 4 * i;  // (D >= 128: g and kk & 1 do not meet the swizzled bits)
    xq[i] = (uint32_t)((r / GR) * GROUP_B + (r % GR) * ROW_B + 16 * (chunk ^ L::swizzle(r)) + (D == 64 ? 0 : 16 * g));
    xk[i] = xq[i] + (koff / GR) * GROUP_B;
  }
#pragma unroll
  for (int i = 0; i < NVB; ++i) {
    const int row = 4 * g + m4 + (D == 64 ? 8 * (i & 1) : 0);  // hi reads of D == 64 swizzle differently
    const int chunk = 4 * (D == 64 ? i >> 1 : i) + 2 * ((lane >> 4) & 1) + (m3 >> 1);
    xv[i] = (uint32_t)(TILE_B + ((koff + (row & 7)) / GR) * GROUP_B + (row % GR) * ROW_B +
                       16 * (chunk ^ L::swizzle(row)) + 8 * (m3 & 1));
  }

  // Reads the Q fragments from the LDS (once their copies have landed; the first K / V copies stay in flight), zeroes
  // rows past the end, pre-scales for BIAS and pins the fragments in registers: AGPRs at one wave per SIMD (head_dim
  // 256: MFMA reads its B operand from there, the VGPRs stay free for the scores and the fragments read ahead).
  auto finish_q = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NQB; ++n) {
      const bool live = qw0 + 32 * n + r < p.Sq;
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) qf[n][kk] = lds_read<V8>(q_slot + xq[KI(kk)] + KO(0, kk));
      if constexpr (NRC > 0) {
        // pos_encoding.cu:90-112 on this lane's row: rotated in fp32, rounded to the storage type as the rotary
        // kernel stores it
        if (rope) {
#pragma unroll
          for (int kk = 0; kk < 4; ++kk) {
            const f32x8 c = rcos[n][kk], sn = rsin[n][kk];
            const f32x8 x = to_f32x8(qf[n][kk]), y = to_f32x8(qf[n][kk + 4]);
            f32x8 xo, yo;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              xo[e] = x[e] * c[e] - y[e] * sn[e];
              yo[e] = y[e] * c[e] + x[e] * sn[e];
            }
            qf[n][kk] = from_f32x8<V8>(xo);
            qf[n][kk + 4] = from_f32x8<V8>(yo);
          }
        }
      }
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) {
        if (!live) qf[n][kk] = V8{};
        if constexpr (BIAS) qf[n][kk] = from_f32x8<V8>(to_f32x8(qf[n][kk]) * p.c_fast);
        if constexpr (OCC == 1) asm volatile("" : "+a"(qf[n][kk]));
        else asm volatile("" : "+v"(qf[n][kk]));
      }
    }
  };

  f32x16 oacc[NQB][D / 32];
  float m_run[NQB], l_part[NQB][2];
#pragma unroll
  for (int n = 0; n < NQB; ++n) {
#pragma unroll
    for (int i = 0; i < D / 32; ++i) oacc[n][i] = f32x16{};
    m_run[n] = -INFINITY;
    l_part[n][0] = l_part[n][1] = 0.f;
  }
  // fp16 reference rounding without soft-cap keeps the scores as packed fp16 in the natural-log domain.
  constexpr bool PK = REFROUND && !SOFTCAP && std::is_same<T, F16>::value;
  const float c = PK ? kLog2e : score_coeff<SOFTCAP, REFROUND>(p);

  // SPREAD (mask-free tiles): the copies of tile t + NSTAGE - 1 are issued here, one per QK^T step.
  auto tile = [&](const int t, auto masked) {
    constexpr bool SPREAD = !decltype(masked)::value && DGG_SPREAD_COPIES;
    const uint32_t st = smem_base + (uint32_t)((t % NSTAGE) * STAGE_B);
    // Per-stage base addresses, opaque to the compiler so that every fragment read below is base + immediate
    // offset (otherwise it re-adds the stage offset for each read).
    uint32_t kbase[NKB], vbase[NVB];
    static_assert(NKB == NVB, "one base of each per step");
#pragma unroll
    for (int i = 0; i < NKB; ++i) {
      kbase[i] = st + xk[i];
      vbase[i] = st + xv[i];
      asm volatile("" : "+v"(kbase[i]), "+v"(vbase[i]));
    }
    constexpr int NMB = SBN / 32;
    constexpr bool MASKED = decltype(masked)::value;
    // Masked tiles: per 32-key block, whether any of the wave's rows sees any of its keys (live) and whether every
    // row sees every key (full). Dead blocks skip their MFMAs and exps, full blocks the per-element mask.
    bool blk_live[NMB], blk_full[NMB];
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) blk_live[mb] = blk_full[mb] = true;
    if constexpr (MASKED) {
      const int row_hi = max(qw0, min(qw0 + QPW, p.Sq) - 1);
      const int hi_min = p.causal ? min(p.Sk - 1, qw0 + p.offset) : p.Sk - 1;
      const int hi_max = p.causal ? min(p.Sk - 1, row_hi + p.offset) : p.Sk - 1;
      const int lo_min = p.window > 0 ? max(0, qw0 + p.offset - p.window + 1) : 0;
      const int lo_max = p.window > 0 ? max(0, row_hi + p.offset - p.window + 1) : 0;
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb) {
        const int kb0 = t * BN + koff + mb * 32;
        blk_live[mb] = kb0 <= hi_max && kb0 + 31 >= lo_min;
        blk_full[mb] = kb0 >= lo_max && kb0 + 31 <= hi_min;
      }
    }
    f32x16 sacc[NQB][NMB];
#pragma unroll
    for (int n = 0; n < NQB; ++n)
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb) {
        if constexpr (BIAS) sacc[n][mb] = mfma32(abias, bbias[n], f32x16{});  // every element = -m[n]
        else sacc[n][mb] = f32x16{};
      }
    if constexpr (MASKED) {
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb) {
        if (!blk_live[mb]) continue;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
          const V8 a = lds_read<V8>(kbase[KI(kk)] + KO(mb, kk));
#pragma unroll
          for (int n = 0; n < NQB; ++n) sacc[n][mb] = mfma32(a, qf[n][kk], sacc[n][mb]);
        }
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) {
        if constexpr (SPREAD) {
#pragma unroll
          for (int i = kk * CPS; i < std::min((kk + 1) * CPS, DMA_PER_TILE); ++i) issue_one(t + NSTAGE - 1, i);
        }
#pragma unroll
        for (int mb = 0; mb < NMB; ++mb) {
          const V8 a = lds_read<V8>(kbase[KI(kk)] + KO(mb, kk));
#pragma unroll
          for (int n = 0; n < NQB; ++n) sacc[n][mb] = mfma32(a, qf[n][kk], sacc[n][mb]);
        }
      }
    }
    const int kb4 = t * BN + koff + 4 * g;
    constexpr bool PKM = PK && !decltype(masked)::value;  // scores stay packed fp16 through the P stage
    f16x2 hs[NQB][NMB][8];
#pragma unroll
    for (int n = 0; n < NQB; ++n) {
      const int rel_hi = k_hi[n] - kb4, rel_lo = k_lo[n] - kb4;
      float mloc = -INFINITY;
      if constexpr (PK) {
#pragma unroll
        for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
          for (int jp = 0; jp < 8; ++jp) hs[n][mb][jp] = ref_scores_f16(sacc[n][mb][2 * jp], sacc[n][mb][2 * jp + 1], p);
      }
      if constexpr (PKM) {
        f16x2 mx = hs[n][0][0];
#pragma unroll
        for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
          for (int jp = 0; jp < 8; ++jp) mx = __builtin_elementwise_max(mx, hs[n][mb][jp]);
        mloc = fmaxf((float)mx[0], (float)mx[1]);
      } else {
#pragma unroll
        for (int mb = 0; mb < NMB; ++mb) {
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            float x;
            if constexpr (PK) x = (float)hs[n][mb][j >> 1][j & 1];
            else x = score_value<T, SOFTCAP, REFROUND>(sacc[n][mb][j], p);
            if constexpr (MASKED) {
              const int o = mb * 32 + 8 * (j >> 2) + (j & 3);
              if (!blk_live[mb]) x = -INFINITY;
              else if (!blk_full[mb]) x = (o <= rel_hi && o >= rel_lo) ? x : -INFINITY;
            }
            sacc[n][mb][j] = x;
            mloc = fmaxf(mloc, x);
          }
        }
      }
      mloc = half_swap_max(mloc);
      if constexpr (BIAS) {
        // mloc is relative to m_run (or absolute while m_run is still -inf and the bias is 0)
        const bool first = m_run[n] == -INFINITY;
        const bool need = first ? mloc > -INFINITY : mloc > kRescaleThreshold;
        if (__any(need)) {
          const float base = first ? 0.f : m_run[n];
          const float m_new = need ? to_f(to_s<S>(mloc + base)) : m_run[n];
          const float alpha = need ? fast_exp2(m_run[n] - m_new) : 1.0f;
          const float delta = need ? m_new - base : 0.f;
          m_run[n] = m_new;
          bbias[n][0] = g == 0 && m_new != -INFINITY ? to_s<S>(-m_new) : to_s<S>(0.0f);
          l_part[n][0] *= alpha;
          l_part[n][1] *= alpha;
#pragma unroll
          for (int i = 0; i < D / 32; ++i) oacc[n][i] *= alpha;
#pragma unroll
          for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
            for (int j = 0; j < 16; ++j) sacc[n][mb][j] -= delta;
        }
        continue;
      }
      const float m_new = fmaxf(m_run[n], mloc);
      const bool need = m_new * c > m_run[n] * c + kRescaleThreshold;
      if (__any(need)) {
        const float alpha = need ? fast_exp2((m_run[n] - m_new) * c) : 1.0f;
        if (need) m_run[n] = m_new;
        l_part[n][0] *= alpha;
        l_part[n][1] *= alpha;
#pragma unroll
        for (int i = 0; i < D / 32; ++i) oacc[n][i] *= alpha;
      }
    }
    float mcs[NQB];
#pragma unroll
    for (int n = 0; n < NQB; ++n) mcs[n] = BIAS || m_run[n] == -INFINITY ? 0.f : m_run[n] * c;
#pragma unroll
    for (int kk = 0; kk < SBN / 16; ++kk) {
      if (MASKED && !blk_live[kk >> 1]) continue;  // P = 0 there
      V8 pb[NQB];
#pragma unroll
      for (int n = 0; n < NQB; ++n) {
        const float mc = mcs[n];
        f32x8 pv;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float x;
          if constexpr (PKM) x = (float)hs[n][kk >> 1][4 * (kk & 1) + (e >> 1)][e & 1];
          else x = sacc[n][kk >> 1][8 * (kk & 1) + e];
          const float pe = BIAS ? fast_exp2(x) : fast_exp2(fmaf(x, c, -mc));
          if constexpr (!FASTSUM) l_part[n][e & 1] += pe;
          pv[e] = pe;
        }
        pb[n] = from_f32x8<V8>(pv);
        if constexpr (FASTSUM) l_part[n][kk & 1] = rowsum8(pb[n], l_part[n][kk & 1]);
      }
#pragma unroll
      for (int db = 0; db < D / 32; ++db) {
        const V4 lo = tr_read_at(vbase[VB(db, 0)] + VO(kk, 0), S{});
        const V4 hi = tr_read_at(vbase[VB(db, 1)] + VO(kk, 1), S{});
        const V8 a = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int n = 0; n < NQB; ++n) oacc[n][db] = mfma32(a, pb[n], oacc[n][db]);
      }
    }
  };

  // Tile classes, per wave: tiles outside [wk_begin, wk_end) are skipped by this
  // wave (it still takes part in the loads and barriers); [t_full0, t_full1) needs no mask for any of its rows.
  int t_full0 = t_begin, t_full1 = t_end;
  if constexpr (MASK) {
    if (p.window > 0) {
      const int lo_last = wq_last + p.offset - p.window + 1;
      t_full0 = lo_last <= koff ? t_begin : min(t_end, max(t_begin, (lo_last - koff + BN - 1) / BN));
    }
    if (p.causal) {
      const int x = qw0 + p.offset + 1 - koff - SBN;
      t_full1 = max(t_full0, min(t_end, x < 0 ? t_begin : x / BN + 1));
    }
  }
  if (t_full1 > t_full0 && t_full1 * BN > p.Sk) t_full1 = max(t_full0, p.Sk / BN);
  if (t_full1 < t_full0) t_full1 = t_full0;
  // A wave whose rows all lie past the end (qw0 >= Sq: the last workgroup of a ragged or short query range,
  // e.g. a single decode-like row) computes no tile; it still issues its share of the copies and meets the barriers.
  const int wt_begin = max(0, wk_begin - koff - SBN + BN) / BN;
  const int wt_end =
      max(wt_begin, qw0 < p.Sq && wk_end > wk_begin ? max(0, wk_end - koff + BN - 1) / BN : wt_begin);

  // Pipeline: tiles t+1 .. t+NSTAGE-2 may still be in flight while tile t is waited for; the copy of tile
  // t+NSTAGE-1 is issued after the barrier into the stage that held tile t-1.
#pragma unroll
  for (int i = 0; i < NSTAGE - 1; ++i)
    if (t_begin + i < t_end) issue(t_begin + i);
  {
    const int issued = min(NSTAGE - 1, t_end - t_begin);
    if (NSTAGE >= 4 && issued >= 3) wait_vmem<3 * DMA_PER_TILE>();
    else if (NSTAGE >= 3 && issued >= 2) wait_vmem<2 * DMA_PER_TILE>();
    else if (issued >= 1) wait_vmem<DMA_PER_TILE>();
    else wait_vmem<0>();
    if constexpr (KG > 1) __syncthreads();
  }
  finish_q();
  auto step = [&](const int t, auto masked) {
    const int after = min(NSTAGE - 2, t_end - 1 - t);
    if (NSTAGE >= 4 && after >= 2) wait_vmem<2 * DMA_PER_TILE>();
    else if (NSTAGE >= 3 && after >= 1) wait_vmem<DMA_PER_TILE>();
    else wait_vmem<0>();
    __syncthreads();
    constexpr bool SPREAD = !decltype(masked)::value && DGG_SPREAD_COPIES;
    if (!SPREAD && t + NSTAGE - 1 < t_end) issue(t + NSTAGE - 1);
    if (SPREAD || (t >= wt_begin && t < wt_end)) tile(t, masked);
  };
  // Mask-free steps issue their copies inside the tile, so they are the tiles this wave computes whose copy target
  // t + NSTAGE - 1 exists and is whole; the others (at most NSTAGE - 1 of them) take the masked step, which is
  // correct for any tile.
  int t_sp1 = t_full1;
  if (DGG_SPREAD_COPIES) t_sp1 = min(min(t_full1, wt_end), min(t_end, p.Sk / BN) - (NSTAGE - 1));
  const int t_sp0 = DGG_SPREAD_COPIES ? min(max(t_full0, wt_begin), t_end) : t_full0;
  t_sp1 = max(t_sp0, t_sp1);
  for (int t = t_begin; t < t_sp0; ++t) step(t, std::true_type{});
  for (int t = t_sp0; t < t_sp1; ++t) step(t, std::false_type{});
  for (int t = t_sp1; t < t_end; ++t) step(t, std::true_type{});

  if constexpr (KG > 1) {
    // The KG waves of a row block hold (m, l, O) over disjoint keys. Each leaves its state in the LDS (the tile ring
    // is done with), then combines one KG-th of the head dim over the groups:
    //   O = sum_i 2^(m_i - m) O_i / sum_i 2^(m_i - m) l_i, m = max_i m_i (a row that sees no key: 0 / 0 = NaN).
    constexpr int NDB = D / 32;
    const float l_own = half_swap_sum(l_part[0][0] + l_part[0][1]);
    __syncthreads();  // every wave is done with the tiles
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj)
        *reinterpret_cast<f32x4*>(smem + w * SLOT_B + (db * 4 + jj) * OQ_B + lane * 16) =
            f32x4{oacc[0][db][4 * jj], oacc[0][db][4 * jj + 1], oacc[0][db][4 * jj + 2], oacc[0][db][4 * jj + 3]};
    f32x2* ml = reinterpret_cast<f32x2*>(smem + NW * SLOT_B);
    if (g == 0) ml[w * 32 + r] = f32x2{BIAS ? m_run[0] : m_run[0] * c, l_own};
    __syncthreads();
    // Wave kg of the row block combines rows kg * 32 / KG .. of it, 8 head-dim elements (two quad halves) per lane, so
    // that the stores cover whole rows.
    constexpr int RW = 32 / KG, NE = D / 8;  // rows per wave, lanes per row
    static_assert(RW * NE % 64 == 0, "whole waves");
#pragma unroll
    for (int it = 0; it < RW * NE / 64; ++it) {
      const int row = kg * RW + (it * 64 + lane) / NE, quad = lane % NE;
      float wt[KG], m_all = -INFINITY, l_all = 0.f;
#pragma unroll
      for (int i = 0; i < KG; ++i) m_all = fmaxf(m_all, ml[(i * NWR + wr) * 32 + row][0]);
      const float mu = m_all == -INFINITY ? 0.f : m_all;
#pragma unroll
      for (int i = 0; i < KG; ++i) {
        const f32x2 x = ml[(i * NWR + wr) * 32 + row];
        wt[i] = fast_exp2(x[0] - mu);
        l_all = fmaf(wt[i], x[1], l_all);
      }
      const float inv = p.Sk == 0 ? 0.f : 1.0f / l_all;
      f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll
      for (int i = 0; i < KG; ++i) {
        const char* slot = smem + (i * NWR + wr) * SLOT_B + quad * OQ_B + row * 16;
        lo += wt[i] * *reinterpret_cast<const f32x4*>(slot);
        hi += wt[i] * *reinterpret_cast<const f32x4*>(slot + 32 * 16);
      }
      const int qi = qw0 + row;
      if (qi < p.Sq) {
        S* op = static_cast<S*>(p.o) + b * p.o_sb + (int64_t)qi * p.o_ss + h * p.o_sh;
        *reinterpret_cast<V8*>(op + 8 * quad) =
            from_f32x8<V8>(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7) * inv);
        if (p.lse != nullptr && quad == 0) {
          const float lse2 = m_all == -INFINITY ? -INFINITY : m_all + fast_log2(l_all);
          p.lse[(int64_t)bh * p.Sq + qi] = p.lse_base2 ? lse2 : lse2 * kLn2;
        }
      }
    }
    return;
  }
  // O goes out through the LDS: the accumulators hold 4 consecutive elements of a row per lane, whose direct stores
  // would touch 32 rows with 16 bytes each. Stage t_end % NSTAGE held tile t_end - NSTAGE, which every wave has left
  // (the last step's barrier), and each wave uses its own rows of it: no further barrier.
  const int qi = qw0 + r;
  const float l_tot = half_swap_sum(l_part[0][0] + l_part[0][1]);
  const float inv = p.Sk == 0 ? 0.f : 1.0f / l_tot;  // no keys at all: o = 0 (an empty P.V), lse = -inf
  const uint32_t o_off = (uint32_t)((t_end % NSTAGE) * STAGE_B + wr * QSLOT_B);
  char* o_row = smem + o_off + (r / GR) * GROUP_B + (r % GR) * ROW_B + 8 * g;
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      V4 ov;
#pragma unroll
      for (int e = 0; e < 4; ++e) ov[e] = to_s<S>(oacc[0][db][4 * jj + e] * inv);
      *reinterpret_cast<V4*>(o_row + 16 * ((4 * db + jj) ^ L::swizzle(r))) = ov;
    }
  if (p.lse != nullptr && g == 0 && qi < p.Sq) {
    const float lse2 = m_run[0] == -INFINITY ? -INFINITY : m_run[0] * c + fast_log2(l_tot);
    p.lse[(int64_t)bh * p.Sq + qi] = p.lse_base2 ? lse2 : lse2 * kLn2;
  }
  S* ob = static_cast<S*>(p.o) + b * p.o_sb + h * p.o_sh;
#pragma unroll
  for (int i = 0; i < 32 / RPI; ++i) {
    const int row = i * RPI + lane / LPR, chunk = lane % LPR;
    const V8 ov = *reinterpret_cast<const V8*>(smem + o_off + (row / GR) * GROUP_B + (row % GR) * ROW_B +
                                               16 * (chunk ^ L::swizzle(row)));
    if (qw0 + row < p.Sq) *reinterpret_cast<V8*>(ob + (int64_t)(qw0 + row) * p.o_ss + 8 * chunk) = ov;
  }
}

// One launch of the direct-load forward in the given form (32 * NW / KG query rows per workgroup).
template <typename T, int D, int NW, int KG, int BN, int NS, int OCC, bool MASK, bool SOFTCAP, int REFROUND>
void launch_fwd_form(AttnParams p, hipStream_t st) {
  constexpr int BM = 32 * NW / KG;
  p.n_tiles = (p.Sq + BM - 1) / BM;
  const unsigned grid = (unsigned)p.n_tiles * p.B * p.Hq;
  if constexpr (!REFROUND && D != 64) {
    if (p.lse == nullptr) {
      hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, NW, KG, BN, NS, OCC, MASK, SOFTCAP, REFROUND, true>), dim3(grid),
                         dim3(64 * NW), 0, st, p);
      return;
    }
  }
  hipLaunchKernelGGL((attn_fwd_dma_kernel<T, D, NW, KG, BN, NS, OCC, MASK, SOFTCAP, REFROUND, false>), dim3(grid),
                     dim3(64 * NW), 0, st, p);
}

// Workgroups of a launch with bm query rows each.
inline int64_t fwd_groups(const AttnParams& p, int bm) { return (int64_t)((p.Sq + bm - 1) / bm) * p.B * p.Hq; }
constexpr int kCUs = 256;

// head_dim 64. Large launches: 4 waves x 32 rows, 64-key tiles, 2 stages (32 KiB: three workgroups per CU at three
// waves per SIMD). The loop is bound by vector issue (a 32 x 32 block of scores takes 8 MFMAs and ~26 x 16 lanes of
// exp / fma / max / pack), and more waves hide more of it: fp16, B=8, S=1000, H=16 without a mask 60.4 -> 47.7 us
// against the kernel that staged tiles through registers; two workgroups of 8 waves 56 us, 64 rows per wave 49 us. The
// row sums are always of the fp32 probabilities (FASTSUM would gain nothing: 47.2 us either way).
// Launches that leave the chip idle split each tile's keys over KG waves instead: 32-row workgroups of 4 waves (KG 4)
// while one per CU suffices (1 x 300 x 16: 8.3 -> 6.4 us), 64-row workgroups of 8 waves (KG 4) up to one per CU
// (1 x 1024 x 16: 16.4 -> 11.3 us), and also up to two per CU when the rows are long (1 x 2048 x 16: 29.6 -> 27.2 us,
// causal 28.6 -> 19.6; 4 x 512 x 12 is better off without, 10.7 against 11.7 us).
template <typename T, bool MASK, bool SOFTCAP, int REFROUND>
void launch_fwd_d64(const AttnParams& p, hipStream_t st) {
  if (fwd_groups(p, 32) <= kCUs) return launch_fwd_form<T, 64, 4, 4, 128, 2, 2, MASK, SOFTCAP, REFROUND>(p, st);
  if (fwd_groups(p, 64) <= kCUs || (fwd_groups(p, 128) <= kCUs && p.Sk >= 1024))
    return launch_fwd_form<T, 64, 8, 4, 128, 2, 4, MASK, SOFTCAP, REFROUND>(p, st);
  launch_fwd_form<T, 64, 4, 1, 64, 2, 3, MASK, SOFTCAP, REFROUND>(p, st);
}

// head_dim 128: 8 waves, 128-key tiles, 2-stage ring, one workgroup per CU. Large launches give each wave 32 rows of
// its own (256 rows per workgroup). KG splits each tile's keys over KG waves of the same rows and adds their states at
// the end, so a workgroup covers 128 or 64 rows and a launch has 2 or 4 times as many:
// * KG 4 while that is at most one workgroup per CU (bf16 causal, H=32: S=509 18.1 -> 11.7 us, S=256 12.0 -> 8.7);
//   beyond one per CU the second round costs more than the shorter workgroups gain (S=768: 17.5 us, KG 2 17.1);
// * KG 2 while that is at most one per CU (S=1024 27.8 -> 20.7 us, without a mask 29.0 -> 22.4);
// * KG 2 also where 256-row workgroups would be at most one per CU but of very unequal length, i.e. a causal mask over
//   at least half of the keys and no window: the two rounds of 128-row workgroups pair long with short (S=1536
//   39.5 -> 29.5 us, S=2048 51.8 -> 42.3, 2 x 1024 31.0 -> 29.7; 4 x 512, with two lengths only, 20.6 against 23.7).
// With more workgroups the chip is full either way, and KG 1 has half the barriers per key and no exchange (S=4096:
// 126.3 us, KG 2 141.7).
template <typename T, bool MASK, bool SOFTCAP, int REFROUND>
void launch_fwd_d128(const AttnParams& p, hipStream_t st) {
  if (fwd_groups(p, 64) <= kCUs) return launch_fwd_form<T, 128, 8, 4, 128, 2, 2, MASK, SOFTCAP, REFROUND>(p, st);
  const bool unequal = p.causal && p.window == 0 && 2 * (int64_t)p.Sq >= p.Sk && p.Sq > 768;
  if (fwd_groups(p, 128) <= kCUs || (fwd_groups(p, 256) <= kCUs && unequal))
    return launch_fwd_form<T, 128, 8, 2, 128, 2, 2, MASK, SOFTCAP, REFROUND>(p, st);
  launch_fwd_form<T, 128, 8, 1, 128, 2, 2, MASK, SOFTCAP, REFROUND>(p, st);
}

// head_dim 256: 4 waves of one per SIMD. Scores kept in fp32 run on the software-pipelined kernel of attention_d256.hip
// (128 rows per workgroup), except where 64-row workgroups, two waves to the same rows (KG 2), are at most one per CU:
// these halve the serial chain of a row (bf16, soft-cap, 16 / 8 heads: S=256 15.0 -> 12.3 us, S=512 21.4 -> 17.5,
// S=1024 36.0 -> 28.4; 2 x 1280, 640 of them, stays at 47). Reference-rounded scores run on the direct-load kernel.
template <typename T, bool MASK, bool SOFTCAP, int REFROUND>
void launch_fwd_d256(AttnParams p, hipStream_t st) {
  if constexpr (REFROUND == 0) {
    if (fwd_groups(p, 64) <= kCUs) return launch_fwd_form<T, 256, 4, 2, 64, 2, 1, MASK, SOFTCAP, REFROUND>(p, st);
    p.n_tiles = (p.Sq + 127) / 128;
    launch_attn_d256_pipe(p, std::is_same<T, BF16>::value, st);
  } else {
    launch_fwd_form<T, 256, 4, 1, 64, 2, 1, MASK, SOFTCAP, REFROUND>(p, st);
  }
}

template <typename T, int D, bool MASK, bool SOFTCAP>
void pick_fwd_ref(const AttnParams& p, bool ref, hipStream_t st) {
  with_ref_mode<D, SOFTCAP>(ref, p, [&](auto mode) {
    constexpr int R = decltype(mode)::value;
    if constexpr (D == 128) launch_fwd_d128<T, MASK, SOFTCAP, R>(p, st);
    else if constexpr (D == 256) launch_fwd_d256<T, MASK, SOFTCAP, R>(p, st);
    else launch_fwd_d64<T, MASK, SOFTCAP, R>(p, st);
  });
}
template <typename T, int D>
void pick_fwd(const AttnParams& p, bool ref, hipStream_t st) {
  const bool mask = p.causal || p.window > 0;
  const bool sc = p.softcap > 0.f;
  if (mask) {
    if (sc) pick_fwd_ref<T, D, true, true>(p, ref, st);
    else pick_fwd_ref<T, D, true, false>(p, ref, st);
  } else {
    if (sc) pick_fwd_ref<T, D, false, true>(p, ref, st);
    else pick_fwd_ref<T, D, false, false>(p, ref, st);
  }
}
}  // namespace
