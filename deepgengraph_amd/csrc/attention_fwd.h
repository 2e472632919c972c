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

// ------------------------------------------------------------------------------------------------
// Forward kernel.
// ------------------------------------------------------------------------------------------------
template <typename T, int D, int BN, bool MASK, bool SOFTCAP, int REFROUND>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(D >= 256 ? 1 : 2, 2))) attn_fwd_kernel(AttnParams p) {
  typedef typename T::scalar S;
  typedef typename T::vec8 V8;
  typedef typename T::vec4 V4;
  constexpr int KP = D + 8;  // padded K row (elements): 16-byte shift per row for the fragment reads
  constexpr int VP = D + 8;  // padded V row (elements): 16-byte shift per row for the transposing reads
  constexpr int NKK = D / 16;      // MFMA k-steps over the head dim
  constexpr int NMB = BN / 32;     // 32-key blocks per tile
  constexpr int NDB = D / 32;      // 32-wide head-dim blocks of O^T
  constexpr int NPK = BN / 16;     // MFMA k-steps over keys in P.V
  constexpr int CHUNKS = BN * D / 8;
  constexpr int CPT = CHUNKS / kThreads;  // 16-byte chunks per thread per tile (K and V each)
  static_assert(CHUNKS % kThreads == 0, "tile must split evenly over the workgroup");

  __shared__ __attribute__((aligned(16))) S Ks[2][BN][KP];
  __shared__ __attribute__((aligned(16))) S Vs[2][BN][VP];

  int qt, bh;
  map_block(p.n_tiles, p.B * p.Hq, true, qt, bh);
  const int b = bh / p.Hq, h = bh - b * p.Hq;
  const int hk = h / p.group;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int q0 = qt * kBM;
  const int qi = q0 + 32 * w + r;  // this lane's query row
  const int tr_krow = (lane & 15) >> 2;                              // key row within a group of 4
  const int tr_dcol = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);     // head-dim column within a 32-wide block

  const S* qp = static_cast<const S*>(p.q) + b * p.q_sb + h * p.q_sh;
  const S* kp = static_cast<const S*>(p.k) + b * p.k_sb + hk * p.k_sh;
  const S* vp = static_cast<const S*>(p.v) + b * p.v_sb + hk * p.v_sh;

  // Q fragment (B operand of S^T = K.Q^T): lane holds query qi, head-dim elements 16kk + 8g .. +8.
  V8 qf[NKK];
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk)  // back-to-back loads (rows past the end read the last row, zeroed below)
    qf[kk] = ld16<V8>(qp + (int64_t)min(qi, p.Sq - 1) * p.q_ss + 16 * kk + 8 * g);
  // Re-define the Q registers here (after their loads complete) so that the main loop's wait counting does not
  // treat them as results of outstanding vector-memory loads.
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) {
    asm volatile("" : "+v"(qf[kk]));
    if (qi >= p.Sq) qf[kk] = V8{};
  }

  // Key range of this query tile.
  const int q_last = min(q0 + kBM, p.Sq) - 1;
  int k_begin = 0, k_end = p.Sk;
  if (p.causal) k_end = min(p.Sk, q_last + p.offset + 1);
  if (p.window > 0) k_begin = max(0, q0 + p.offset - p.window + 1);
  const int t_begin = k_begin / BN;
  const int t_end = k_end > k_begin ? (k_end + BN - 1) / BN : t_begin;

  f32x16 oacc[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i) oacc[i] = f32x16{};
  float m_run = -INFINITY;  // reference maximum (value units)
  const float c = score_coeff<SOFTCAP, REFROUND>(p);

  // Global -> register staging of one K/V tile: each thread owns CPT adjacent 16-byte chunks of one key row of
  // K and of V (coalesced rows; both stay row-major in LDS). Full tiles are addressed through two per-lane
  // pointers that advance by one tile right before each load (so a pointer register is never rewritten while
  // loads through it are in flight), the chunk index going into the immediate offset.
  V8 kreg[CPT], vreg[CPT];
  constexpr int TPR = (D / 8) / CPT;        // threads per row
  static_assert(TPR * CPT == D / 8 && kThreads / TPR == BN, "tile mapping");
  const int k_row0 = tid / TPR, k_c0 = (tid % TPR) * CPT;
  const int64_t k_step = (int64_t)BN * p.k_ss * (int64_t)sizeof(S), v_step = (int64_t)BN * p.v_ss * (int64_t)sizeof(S);
  // pointers of tile t_begin - 1 (advanced before use)
  gptr k_addr = to_gptr(kp + (int64_t)(k_row0 - BN) * p.k_ss + k_c0 * 8) + (int64_t)t_begin * k_step;
  gptr v_addr = to_gptr(vp + (int64_t)(k_row0 - BN) * p.v_ss + k_c0 * 8) + (int64_t)t_begin * v_step;
  auto load_full = [&]() {
    k_addr += k_step;
    v_addr += v_step;
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      kreg[i] = ldg16<V8>(k_addr + 16 * i);
      vreg[i] = ldg16<V8>(v_addr + 16 * i);
    }
  };
  // Ragged last tile: rows past the end are clamped to the last row (masked, finite: contributes exactly 0).
  auto load_ragged = [&](int t) {
    k_addr += k_step;
    v_addr += v_step;
    const int kb = t * BN;
    const int kr = min(k_row0, p.Sk - 1 - kb);  // >= 0 for every loaded tile
    const S* kt = kp + (int64_t)(kb + kr) * p.k_ss + k_c0 * 8;
    const S* vt = vp + (int64_t)(kb + kr) * p.v_ss + k_c0 * 8;
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      kreg[i] = ld16<V8>(kt + i * 8);
      vreg[i] = ld16<V8>(vt + i * 8);
    }
  };
  auto tile_full = [&](int t) { return (t + 1) * BN <= p.Sk; };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      *reinterpret_cast<V8*>(&Ks[buf][k_row0][(k_c0 + i) * 8]) = kreg[i];
      *reinterpret_cast<V8*>(&Vs[buf][k_row0][(k_c0 + i) * 8]) = vreg[i];
    }
  };

  if (t_begin < t_end) {
    if (tile_full(t_begin)) load_full();
    else load_ragged(t_begin);
    store_tile(0);
  }
  __syncthreads();

  // Visible keys of this lane's query: lo <= key <= hi (bottom-right causal, sliding window, ragged end).
  int k_hi = p.Sk - 1, k_lo = 0;
  if (p.causal) k_hi = min(k_hi, qi + p.offset);
  if (p.window > 0) k_lo = max(k_lo, qi + p.offset - p.window + 1);
  float l_part[4] = {0.f, 0.f, 0.f, 0.f};  // split row sums (breaks the dependent add chain)

  // One K/V tile: S^T = K.Q^T, scores, online softmax, O^T += V^T.P^T. MASKED tiles compare each key against
  // the lane's [k_lo, k_hi]; all other tiles run without any mask arithmetic.
  auto tile = [&](const int t, const int buf, auto masked) {
    f32x16 sacc[NMB];
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) sacc[mb] = f32x16{};
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb) {
        const V8 a = *reinterpret_cast<const V8*>(&Ks[buf][mb * 32 + r][16 * kk + 8 * g]);
        sacc[mb] = mfma32(a, qf[kk], sacc[mb]);
      }
    }
    // element (mb, j) holds key t*BN + mb*32 + 8*(j/4) + 4g + j%4
    const int rel_hi = k_hi - (t * BN + 4 * g), rel_lo = k_lo - (t * BN + 4 * g);
    float mloc = -INFINITY;
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        float x = score_value<T, SOFTCAP, REFROUND>(sacc[mb][j], p);
        if constexpr (decltype(masked)::value) {
          const int o = mb * 32 + 8 * (j >> 2) + (j & 3);
          x = (o <= rel_hi && o >= rel_lo) ? x : -INFINITY;
        }
        sacc[mb][j] = x;
        mloc = fmaxf(mloc, x);
      }
    }
    mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64));
    const float m_new = fmaxf(m_run, mloc);
    const bool need = m_new * c > m_run * c + kRescaleThreshold;
    if (__any(need)) {
      const float alpha = need ? fast_exp2((m_run - m_new) * c) : 1.0f;
      if (need) m_run = m_new;
#pragma unroll
      for (int i = 0; i < 4; ++i) l_part[i] *= alpha;
#pragma unroll
      for (int i = 0; i < NDB; ++i) oacc[i] *= alpha;
    }
    const float mc = m_run == -INFINITY ? 0.f : m_run * c;

    // P = exp2(v*c - m*c), row sums, pack to 16-bit B operands, O^T += V^T . P^T
#pragma unroll
    for (int kk = 0; kk < NPK; ++kk) {
      f32x8 pv;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float pe = fast_exp2(fmaf(sacc[kk >> 1][8 * (kk & 1) + e], c, -mc));
        l_part[e & 3] += pe;
        pv[e] = pe;
      }
      const V8 pb = from_f32x8<V8>(pv);
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        // A = V^T rows db*32 + r, keys 16kk + 4g + {0..3} and 16kk + 8 + 4g + {0..3} (the P operand's key order),
        // gathered from row-major V by the transposing read (lane m of each 16-lane group points at key row
        // m/4 and head-dim column 4*(m%4) of its 16-column slab).
        const S* vrow = &Vs[buf][16 * kk + 4 * g + tr_krow][db * 32 + tr_dcol];
        const V4 lo = tr_read(vrow);
        const V4 hi = tr_read(vrow + 8 * VP);
        const V8 a = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        oacc[db] = mfma32(a, pb, oacc[db]);
      }
    }
  };

  // Tiles [t_begin, t_full0) and [t_full1, t_end) straddle the window's lower edge or the causal diagonal (or the
  // ragged end of K) and evaluate the mask; tiles in between are visible to every row of the workgroup.
  int t_full0 = t_begin, t_full1 = t_end;
  if constexpr (MASK) {
    if (p.window > 0) {  // first tile whose first key is visible to the last row
      const int lo_last = q_last + p.offset - p.window + 1;
      t_full0 = lo_last <= 0 ? t_begin : min(t_end, max(t_begin, (lo_last + BN - 1) / BN));
    }
    if (p.causal) {  // first tile whose last key is hidden from the first row
      const int hi_first = q0 + p.offset;  // last key visible to the first row
      t_full1 = max(t_full0, min(t_end, hi_first < 0 ? t_begin : (hi_first + 1) / BN));
    }
  }
  if (t_full1 > t_full0 && t_full1 * BN > p.Sk) t_full1 = max(t_full0, p.Sk / BN);
  if (t_full1 < t_full0) t_full1 = t_full0;

  // Full next tiles are prefetched into registers before this tile's compute; the ragged last tile (at most one)
  // is loaded after it.
  const bool wave_live = q0 + 32 * w < p.Sq;  // wave-uniform: a wave past the end only stages tiles
  auto step = [&](const int t, auto masked) {
    const int buf = (t - t_begin) & 1;
    const int tn = t + 1;
    const bool prefetch = tn < t_end && tile_full(tn);
    if (prefetch) load_full();
    if (wave_live) tile(t, buf, masked);
    if (tn < t_end) {
      if (!prefetch) load_ragged(tn);
      store_tile(buf ^ 1);
    }
    __syncthreads();
  };
  for (int t = t_begin; t < t_full0; ++t) step(t, std::true_type{});
  for (int t = t_full0; t < t_full1; ++t) step(t, std::false_type{});
  for (int t = t_full1; t < t_end; ++t) step(t, std::true_type{});
  float l_run = (l_part[0] + l_part[1]) + (l_part[2] + l_part[3]);

  // Epilogue: full row sum, normalise, store O (4 consecutive head-dim elements per store) and lse.
  const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  const float inv = p.Sk == 0 ? 0.f : 1.0f / l_tot;  // no keys at all: o = 0 (an empty P.V), lse = -inf
  if (qi < p.Sq) {
    S* op = static_cast<S*>(p.o) + b * p.o_sb + (int64_t)qi * p.o_ss + h * p.o_sh;
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        V4 ov;
#pragma unroll
        for (int e = 0; e < 4; ++e) ov[e] = to_s<S>(oacc[db][4 * jj + e] * inv);
        *reinterpret_cast<V4*>(op + db * 32 + 8 * jj + 4 * g) = ov;
      }
    }
    if (p.lse != nullptr && g == 0) {
      const float lse2 = m_run == -INFINITY ? -INFINITY : m_run * c + fast_log2(l_tot);
      p.lse[(int64_t)bh * p.Sq + qi] = p.lse_base2 ? lse2 : lse2 * kLn2;
    }
  }
}



// NQB: 32-row query blocks per wave (each K / V fragment feeds NQB MFMAs); NW: waves per workgroup; BN: keys
// per tile; NSTAGE: tiles in the LDS ring; OCC: waves per SIMD the register budget is sized for. FASTSUM: the row
// sums add the 16-bit rounded probabilities two at a time (v_dot2); used when no lse is written, since the O
// normalisation tolerates the rounding but the column-sum pass needs the fp32 row sums.
template <typename T, int D, int NQB, int NW, int BN, int NSTAGE, int OCC, bool MASK, bool SOFTCAP, int REFROUND,
          bool FASTSUM>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(OCC, OCC)))
attn_fwd_dma_kernel(AttnParams p) {
  typedef DmaLayout<D> L;
  constexpr int ROW_B = L::ROW_B, GROUP_B = L::GROUP_B, LPR = L::LPR, RPI = L::RPI, IPG = L::IPG;
  typedef typename T::scalar S;
  typedef typename T::vec8 V8;
  typedef typename T::vec4 V4;
  constexpr int QPW = 32 * NQB;                 // query rows per wave
  constexpr int BM = QPW * NW;                  // query rows per workgroup
  constexpr int TILE_B = (BN / 4) * GROUP_B;
  constexpr int STAGE_B = 2 * TILE_B;           // K tile, then V tile
  constexpr int GPW = (BN / 4) / NW;            // 4-row groups of a tile copied by each wave (K and V each)
  constexpr int DMA_PER_TILE = 2 * GPW * IPG;   // direct loads per wave per tile
  static_assert(GPW >= 1 && GPW * NW == BN / 4, "tile groups must split over the waves");
  __shared__ __attribute__((aligned(1024))) char smem[NSTAGE * STAGE_B];

  int qt, bh;
  map_block_kv(p.n_tiles, p.B, p.Hq, p.Hkv, true, qt, bh);
  const int b = bh / p.Hq, h = bh - b * p.Hq;
  const int hk = h / p.group;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q0 = qt * BM;
  const int qw0 = q0 + QPW * w;  // first query row of this wave; lane rows qw0 + 32n + r, n = 0, 1

  const S* qp = static_cast<const S*>(p.q) + b * p.q_sb + h * p.q_sh;
  const char* kp = reinterpret_cast<const char*>(static_cast<const S*>(p.k) + b * p.k_sb + hk * p.k_sh);
  const char* vp = reinterpret_cast<const char*>(static_cast<const S*>(p.v) + b * p.v_sb + hk * p.v_sh);
  const int64_t k_ss_b = p.k_ss * (int64_t)sizeof(S), v_ss_b = p.v_ss * (int64_t)sizeof(S);

  // Q fragments: all loads issued back to back (rows past the end read the last row and are zeroed afterwards;
  // a load under a per-row branch would be waited for on its own).
  V8 qf[NQB][D / 16];
#pragma unroll
  for (int n = 0; n < NQB; ++n) {
    const int qi = min(qw0 + 32 * n + r, p.Sq - 1);
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) qf[n][kk] = ld16<V8>(qp + (int64_t)qi * p.q_ss + 16 * kk + 8 * g);
  }
  // Fused rotary of the query (head_dim 128): the (cos, sin) of this lane's 32 rotary pairs, loaded with Q so that
  // the two latencies overlap. The lane holds elements 16kk + 8g + e of fragment kk and their pair partners (+64)
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
  // BIAS (bf16 without soft-cap or reference rounding, no lse): Q is pre-scaled by scale*log2(e) and each score
  // accumulator starts from -m (the row's reference maximum) through one extra MFMA whose A fragment is the
  // constant column e_0 and whose B fragment holds -m in k-slot 0. The accumulator then holds s*c - m and
  // P = exp2(acc) needs no per-element arithmetic. The reference maxima are bf16 values so that -m is exact in
  // the B operand; the pre-scaled Q carries the same 2^-9 relative rounding as the reference's bf16 scores.
  constexpr bool BIAS = FASTSUM && !SOFTCAP && !REFROUND && std::is_same<T, BF16>::value;
  // Waits for the Q loads (after the first K / V copies are issued, so that the latencies overlap), zeroes rows
  // past the end, pre-scales for BIAS and pins the fragments in registers: AGPRs at one wave per SIMD (head_dim
  // 256: MFMA reads its B operand from there, the VGPRs stay free for the scores and the fragments read ahead).
  auto finish_q = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NQB; ++n) {
      const bool live = qw0 + 32 * n + r < p.Sq;
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) asm volatile("" : "+v"(qf[n][kk]));
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

  // Direct-load lane constants: in load i of a 4-row group, lane l fills LDS position l%LPR of group row
  // i*RPI + l/LPR, fetching global chunk (l%LPR) ^ 4*(group row).
  uint32_t src_chunk[IPG], k_voff[IPG], v_voff[IPG];
#pragma unroll
  for (int i = 0; i < IPG; ++i) {
    const int grow = i * RPI + lane / LPR;
    src_chunk[i] = (uint32_t)((lane % LPR) ^ (grow << 2));
    k_voff[i] = (uint32_t)(grow * k_ss_b) + src_chunk[i] * 16u;
    v_voff[i] = (uint32_t)(grow * v_ss_b) + src_chunk[i] * 16u;
    asm volatile("" : "+v"(k_voff[i]), "+v"(v_voff[i]));
  }
  const uint32_t smem_base = (uint32_t)(size_t)((lds_char*)smem);

  // Copies groups GPW*w .. GPW*w + GPW-1 of tile t into stage t % NSTAGE: DMA_PER_TILE loads per wave.
  auto issue = [&](int t) {
    const uint32_t kdst = smem_base + (uint32_t)((t % NSTAGE) * STAGE_B + GPW * w * GROUP_B);
    const uint32_t vdst = kdst + TILE_B;
    const int row0 = t * BN + 4 * GPW * w;
    if ((t + 1) * BN <= p.Sk) {
      const char* kb = kp + (int64_t)row0 * k_ss_b;
      const char* vb = vp + (int64_t)row0 * v_ss_b;
#pragma unroll
      for (int j = 0; j < GPW; ++j)
#pragma unroll
        for (int i = 0; i < IPG; ++i) {
          dma16(kdst + j * GROUP_B + i * RPI * ROW_B, kb + 4 * j * k_ss_b, k_voff[i]);
          dma16(vdst + j * GROUP_B + i * RPI * ROW_B, vb + 4 * j * v_ss_b, v_voff[i]);
        }
    } else {  // ragged last tile: rows past the end re-read the last row (always masked, finite)
#pragma unroll
      for (int j = 0; j < GPW; ++j)
#pragma unroll
        for (int i = 0; i < IPG; ++i) {
          const int64_t row = min(row0 + 4 * j + i * RPI + lane / LPR, p.Sk - 1);
          dma16(kdst + j * GROUP_B + i * RPI * ROW_B, kp + row * k_ss_b + src_chunk[i] * 16);
          dma16(vdst + j * GROUP_B + i * RPI * ROW_B, vp + row * v_ss_b + src_chunk[i] * 16);
        }
    }
  };

  // Load i (0 .. DMA_PER_TILE-1) of issue(t) for a tile whose rows all exist: the K loads, then the V loads. The
  // mask-free tiles issue the next tile's copies one per QK^T step with these, so that the copies' issue overlaps
  // the MFMAs instead of following the barrier as one burst (which held every wave of the workgroup at once).
  auto issue_one = [&](int t, int i) __attribute__((always_inline)) {
    const uint32_t kdst = smem_base + (uint32_t)((t % NSTAGE) * STAGE_B + GPW * w * GROUP_B);
    const int row0 = t * BN + 4 * GPW * w;
    const int half = GPW * IPG, ii = i % half, j = ii / IPG, l = ii % IPG;
    if (i < half)
      dma16(kdst + j * GROUP_B + l * RPI * ROW_B, kp + (int64_t)row0 * k_ss_b + 4 * j * k_ss_b, k_voff[l]);
    else
      dma16(kdst + TILE_B + j * GROUP_B + l * RPI * ROW_B, vp + (int64_t)row0 * v_ss_b + 4 * j * v_ss_b, v_voff[l]);
  };
  static_assert(DMA_PER_TILE <= D / 16, "one copy per QK^T step");

  // LDS read addressing. K fragment (row mb*32 + r, chunk 2kk + g): lane part + xk[kk/2] + constant.
  // V transposing read (rows 16kk + 4g + (lane%16)/4 (+8), head-dim column db*32 + 16*((lane/16)%2) + 4*(lane%4)):
  // lane part + xv[db] + constant.
  const int s4 = r & 3;
  const uint32_t k_lane = (uint32_t)((r >> 2) * GROUP_B + s4 * ROW_B + 16 * g);
  uint32_t xk[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) xk[i] = k_lane + 64u * (uint32_t)(i ^ s4);
  const int m4 = (lane & 15) >> 2, m3 = lane & 3;
  const uint32_t v_lane = (uint32_t)(TILE_B + g * GROUP_B + m4 * ROW_B + 32 * ((lane >> 4) & 1) + 16 * (m3 >> 1) +
                                     8 * (m3 & 1));
  uint32_t xv[D / 32];
#pragma unroll
  for (int db = 0; db < D / 32; ++db) xv[db] = v_lane + 64u * (uint32_t)(db ^ m4);

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
    uint32_t kbase[D / 32], vbase[D / 32];
#pragma unroll
    for (int i = 0; i < D / 32; ++i) {
      kbase[i] = st + xk[i];
      vbase[i] = st + xv[i];
      asm volatile("" : "+v"(kbase[i]), "+v"(vbase[i]));
    }
    constexpr int NMB = BN / 32;
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
        const int kb0 = t * BN + mb * 32;
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
          const V8 a = lds_read<V8>(kbase[kk >> 1] + mb * 8 * GROUP_B + 32 * (kk & 1));
#pragma unroll
          for (int n = 0; n < NQB; ++n) sacc[n][mb] = mfma32(a, qf[n][kk], sacc[n][mb]);
        }
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) {
        if constexpr (SPREAD) {
          if (kk < DMA_PER_TILE) issue_one(t + NSTAGE - 1, kk);
        }
#pragma unroll
        for (int mb = 0; mb < NMB; ++mb) {
          const V8 a = lds_read<V8>(kbase[kk >> 1] + mb * 8 * GROUP_B + 32 * (kk & 1));
#pragma unroll
          for (int n = 0; n < NQB; ++n) sacc[n][mb] = mfma32(a, qf[n][kk], sacc[n][mb]);
        }
      }
    }
    const int kb4 = t * BN + 4 * g;
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
    for (int kk = 0; kk < BN / 16; ++kk) {
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
        const V4 lo = tr_read_at(vbase[db] + kk * 4 * GROUP_B, S{});
        const V4 hi = tr_read_at(vbase[db] + kk * 4 * GROUP_B + 2 * GROUP_B, S{});
        const V8 a = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int n = 0; n < NQB; ++n) oacc[n][db] = mfma32(a, pb[n], oacc[n][db]);
      }
    }
  };

  // Tile classes, as in the generic kernel but per wave: tiles outside [wk_begin, wk_end) are skipped by this
  // wave (it still takes part in the loads and barriers); [t_full0, t_full1) needs no mask for any of its rows.
  int t_full0 = t_begin, t_full1 = t_end;
  if constexpr (MASK) {
    if (p.window > 0) {
      const int lo_last = wq_last + p.offset - p.window + 1;
      t_full0 = lo_last <= 0 ? t_begin : min(t_end, max(t_begin, (lo_last + BN - 1) / BN));
    }
    if (p.causal) {
      const int hi_first = qw0 + p.offset;
      t_full1 = max(t_full0, min(t_end, hi_first < 0 ? t_begin : (hi_first + 1) / BN));
    }
  }
  if (t_full1 > t_full0 && t_full1 * BN > p.Sk) t_full1 = max(t_full0, p.Sk / BN);
  if (t_full1 < t_full0) t_full1 = t_full0;
  // A wave whose rows all lie past the end (qw0 >= Sq: the last workgroup of a ragged or short query range,
  // e.g. a single decode-like row) computes no tile; it still issues its share of the copies and meets the barriers.
  const int wt_begin = wk_begin / BN;
  const int wt_end = qw0 < p.Sq && wk_end > wk_begin ? (wk_end + BN - 1) / BN : wt_begin;

  // Pipeline: tiles t+1 .. t+NSTAGE-2 may still be in flight while tile t is waited for; the copy of tile
  // t+NSTAGE-1 is issued after the barrier into the stage that held tile t-1.
#pragma unroll
  for (int i = 0; i < NSTAGE - 1; ++i)
    if (t_begin + i < t_end) issue(t_begin + i);
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

#pragma unroll
  for (int n = 0; n < NQB; ++n) {
    const int qi = qw0 + 32 * n + r;
    const float l_tot = half_swap_sum(l_part[n][0] + l_part[n][1]);
    const float inv = p.Sk == 0 ? 0.f : 1.0f / l_tot;  // no keys at all: o = 0 (an empty P.V), lse = -inf
    if (qi < p.Sq) {
      S* op = static_cast<S*>(p.o) + b * p.o_sb + (int64_t)qi * p.o_ss + h * p.o_sh;
#pragma unroll
      for (int db = 0; db < D / 32; ++db) {
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          V4 ov;
#pragma unroll
          for (int e = 0; e < 4; ++e) ov[e] = to_s<S>(oacc[n][db][4 * jj + e] * inv);
          *reinterpret_cast<V4*>(op + db * 32 + 8 * jj + 4 * g) = ov;
        }
      }
      if (p.lse != nullptr && g == 0) {
        const float lse2 = m_run[n] == -INFINITY ? -INFINITY : m_run[n] * c + fast_log2(l_tot);
        p.lse[(int64_t)bh * p.Sq + qi] = p.lse_base2 ? lse2 : lse2 * kLn2;
      }
    }
  }
}

template <typename T, int D, int BN, bool MASK, bool SOFTCAP, int REFROUND>
void launch_fwd(AttnParams p, hipStream_t st) {
  p.n_tiles = (p.Sq + kBM - 1) / kBM;
  const unsigned grid = (unsigned)p.n_tiles * p.B * p.Hq;
  hipLaunchKernelGGL((attn_fwd_kernel<T, D, BN, MASK, SOFTCAP, REFROUND>), dim3(grid), dim3(kThreads), 0, st, p);
}

// head_dim 128 configuration (measured on MI355X, config 2): 8 waves x 32 rows, 128-key tiles, 2-stage ring.
#ifndef DGG_D128_NW
#define DGG_D128_NW 8
#endif
#ifndef DGG_D128_BN
#define DGG_D128_BN 128
#endif
// DGG_D128_OCC: waves per SIMD the register budget is sized for (2; 3 with DGG_D128_NW=4 DGG_D128_BN=32 is the
// three-waves-per-SIMD form, whose LDS fits three workgroups per CU only at 32-key tiles).
#ifndef DGG_D128_OCC
#define DGG_D128_OCC 2
#endif
constexpr int kD128NQB = 1, kD128NW = DGG_D128_NW, kD128BN = DGG_D128_BN, kD128NS = 2;
constexpr int kD128BM = 32 * kD128NQB * kD128NW;  // query rows per workgroup (head_dim 128)

template <typename T, bool MASK, bool SOFTCAP, int REFROUND>
void launch_fwd_d128(AttnParams p, hipStream_t st) {
  p.n_tiles = (p.Sq + kD128BM - 1) / kD128BM;
  const unsigned grid = (unsigned)p.n_tiles * p.B * p.Hq;
  if (!REFROUND && p.lse == nullptr)
    hipLaunchKernelGGL(
        (attn_fwd_dma_kernel<T, 128, kD128NQB, kD128NW, kD128BN, kD128NS, DGG_D128_OCC, MASK, SOFTCAP, REFROUND, !REFROUND>),
        dim3(grid), dim3(64 * kD128NW), 0, st, p);
  else
    hipLaunchKernelGGL(
        (attn_fwd_dma_kernel<T, 128, kD128NQB, kD128NW, kD128BN, kD128NS, DGG_D128_OCC, MASK, SOFTCAP, REFROUND, false>),
        dim3(grid), dim3(64 * kD128NW), 0, st, p);
}

// head_dim 256 configuration: 4 waves x 32 rows (one wave per SIMD), DGG_D256_BN-key tiles, 2-stage ring.
#ifndef DGG_D256_BN
#define DGG_D256_BN 64
#endif
constexpr int kD256NW = 4, kD256BN = DGG_D256_BN, kD256NS = 2;
constexpr int kD256BM = 32 * kD256NW;

// DGG_D256_PIPE (default 1): the software-pipelined kernel of attention_d256.hip for the scores in fp32; 0 keeps
// every head_dim-256 launch on attn_fwd_dma_kernel (for A/B measurements).
#ifndef DGG_D256_PIPE
#define DGG_D256_PIPE 1
#endif

template <typename T, bool MASK, bool SOFTCAP, int REFROUND>
void launch_fwd_d256(AttnParams p, hipStream_t st) {
  p.n_tiles = (p.Sq + kD256BM - 1) / kD256BM;
  if (DGG_D256_PIPE && !REFROUND) return launch_attn_d256_pipe(p, std::is_same<T, BF16>::value, st);
  const unsigned grid = (unsigned)p.n_tiles * p.B * p.Hq;
  if (!REFROUND && p.lse == nullptr)
    hipLaunchKernelGGL((attn_fwd_dma_kernel<T, 256, 1, kD256NW, kD256BN, kD256NS, 1, MASK, SOFTCAP, REFROUND, !REFROUND>),
                       dim3(grid), dim3(64 * kD256NW), 0, st, p);
  else
    hipLaunchKernelGGL((attn_fwd_dma_kernel<T, 256, 1, kD256NW, kD256BN, kD256NS, 1, MASK, SOFTCAP, REFROUND, false>),
                       dim3(grid), dim3(64 * kD256NW), 0, st, p);
}

template <typename T, int D, bool MASK, bool SOFTCAP>
void pick_fwd_ref(const AttnParams& p, bool ref, hipStream_t st) {
  constexpr int BN = D >= 256 ? 32 : 64;
  with_ref_mode<D, SOFTCAP>(ref, p, [&](auto mode) {
    constexpr int R = decltype(mode)::value;
    if constexpr (D == 128) launch_fwd_d128<T, MASK, SOFTCAP, R>(p, st);
    else if constexpr (D == 256) launch_fwd_d256<T, MASK, SOFTCAP, R>(p, st);
    else launch_fwd<T, D, BN, MASK, SOFTCAP, R>(p, st);
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
