// fp32 attention: the forward (O and lse) and the column-score pass of the selection cases for fp32 inputs, the
// dtype of config 1 and of any case module the caller runs in fp32 (the reference's modules take any float
// dtype: attn.py:18-34 computes in the input dtype, so fp32 inputs give fp32 scores, an fp32 softmax and an fp32
// P.V with no 16-bit rounding anywhere).
//
// The forward runs on the fp32 MFMA. The column pass is a plain one: four adjacent lanes share one key, each holding a
// quarter of the head dimension in registers, the dot products are reduced over the four lanes with two cross-lane adds,
// and Q and its lse are staged through LDS in tiles of 32 rows. exp / log are the accurate device expf / logf.
#include "attention_common.h"

namespace dgg_attn {
namespace {

constexpr int kRows = 64;      // keys per workgroup (column pass)
constexpr int kThr = 4 * kRows;
constexpr int kTile = 32;      // query rows per LDS tile (column pass)

// Dot product of this lane's quarter with quarter `qd` of an LDS row, summed over the four lanes of the quad.
template <int D>
__device__ __forceinline__ float quad_dot(const float (&a)[D / 4], const float* row) {
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < D / 4; e += 4) {
    const f32x4 b = *reinterpret_cast<const f32x4*>(row + e);
    s = fmaf(a[e], b[0], s);
    s = fmaf(a[e + 1], b[1], s);
    s = fmaf(a[e + 2], b[2], s);
    s = fmaf(a[e + 3], b[3], s);
  }
  s += __shfl_xor(s, 1, 64);
  s += __shfl_xor(s, 2, 64);
  return s;
}

// The score as the reference computes it in fp32: the matmul result times the fp32 reciprocal of the divisor
// (torch's GPU division by a Python float), then softcap * tanh(s / softcap) (gemma2.py:31-33).
template <bool SOFTCAP>
__device__ __forceinline__ float f32_score(float dot, const AttnParams& p) {
  float s = dot * p.ref_rcp;
  if constexpr (SOFTCAP) s = tanhf(s * p.inv_softcap) * p.softcap;
  return s;
}

// Copies rows r0 .. r0 + kTile - 1 of a [rows, D] fp32 matrix (row stride rs elements) into lds[kTile][D + 4];
// rows at or past n are zero.
template <int D>
__device__ __forceinline__ void stage_rows(float (*lds)[D + 4], const float* src, int64_t rs, int r0, int n) {
  constexpr int C4 = D / 4;  // 16-byte chunks per row
  for (int c = threadIdx.x; c < kTile * C4; c += kThr) {
    const int r = c / C4, col = (c % C4) * 4;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (r0 + r < n) v = *reinterpret_cast<const f32x4*>(src + (int64_t)(r0 + r) * rs + col);
    *reinterpret_cast<f32x4*>(&lds[r][col]) = v;
  }
}

// Forward. Both products run on v_mfma_f32_16x16x4_f32 (fp32 operands and sums): S^T = K.Q^T puts one query per lane
// (lane % 16) with 4 keys of a 16-key block in its registers, and accumulator register i, rounded by nothing, is then the
// B operand of the i-th step of O^T += V^T.P^T (the keys 4g + i, g = lane / 16), whose A operand is one float of V per
// lane, read row-contiguous. Within a k-step the four lane groups may take any four head-dim elements as long as K and
// Q agree: group g holds elements g * D/4 .., so a fragment is D/16 16-byte reads.
// A workgroup is kKG = 4 waves on the same 16 query rows, wave kg taking every fourth 16-key block; their (m, l, O)
// are combined through the LDS at the end. K passes through wave-private LDS rows (coalesced loads, one block ahead), V is
// loaded in operand layout, so the loop has no barrier. What bounds it at the sizes fp32 is used at is the serial
// chain of a row's blocks, hence the four-way split of the keys and the small row blocks (32 rows per workgroup: 20.2 us
// where 16 take 13.1). Measured on MI355X against the kernel before, which had four lanes per row on the vector units:
// B=1, S=512, H=8, D=64, causal 121.4 -> 13.6 us; B=2, S=1024, D=128 420.7 -> 69.7; S=4096, H=32, D=128 4387 -> 1656.
// Relative error against 64 bits there: 2.6e-7 -> 1.5e-7 (S=512, D=64), 3.4e-7 -> 1.9e-7 (D=128).
constexpr int kKG = 4;

template <int D, bool SOFTCAP>
__global__ void __launch_bounds__(64 * kKG) attn_fwd_f32_kernel(AttnParams p) {
  static_assert(kF32Rows == 16, "one row per lane of 16");
  constexpr int NC = D / 16;             // 16-byte chunks of a fragment; 16-wide head-dim blocks of O^T
  constexpr int RS = D + 4;              // LDS row (floats): 16 rows of one chunk on distinct banks
  constexpr int SLOT = 16 * RS, OSLOT = NC * 64 * 4;  // floats: a wave's K block (at the start, Q); its O at the end
  constexpr int SMEM = kKG * (SLOT > OSLOT ? SLOT : OSLOT) + 2 * kKG * 16;
  __shared__ __attribute__((aligned(16))) float smem[SMEM];

  int qt, bh;
  map_block(p.n_tiles, p.B * p.Hq, true, qt, bh, p.block0 + blockIdx.x);
  const int b = bh / p.Hq, h = bh - b * p.Hq, hk = h / p.group;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int kg = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q0 = qt * 16;
  const float* qp = static_cast<const float*>(p.q) + b * p.q_sb + h * p.q_sh;
  const float* kp = static_cast<const float*>(p.k) + b * p.k_sb + hk * p.k_sh;
  const float* vp = static_cast<const float*>(p.v) + b * p.v_sb + hk * p.v_sh;
  float* slot = smem + kg * SLOT;  // wave-private

  // Keys of the workgroup, and of this lane's rows (bottom-right causal, window).
  const int q_last = min(q0 + 16, p.Sq) - 1;
  int k_begin = 0, k_end = p.Sk;
  if (p.causal) k_end = min(p.Sk, q_last + p.offset + 1);
  if (p.window > 0) k_begin = max(0, q0 + p.offset - p.window + 1);
  const int qi = q0 + r;
  int k_hi = p.Sk - 1, k_lo = 0;
  if (p.causal) k_hi = min(k_hi, qi + p.offset);
  if (p.window > 0) k_lo = max(k_lo, qi + p.offset - p.window + 1);
  const int b_begin = k_begin / 16 + kg, b_end = k_end > k_begin ? (k_end + 15) / 16 : 0;

  // Block loads: chunk c = lane + 64 i of a 16-row block is chunk c % (D/4) of row c / (D/4). Rows past the end read the
  // last row (masked).
  constexpr int CPR = D / 4;
  f32x4 kreg[NC];
  auto load_k = [&](int kb) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = lane + 64 * i;
      kreg[i] = *reinterpret_cast<const f32x4*>(kp + (int64_t)min(16 * kb + c / CPR, p.Sk - 1) * p.k_ss + 4 * (c % CPR));
    }
  };
  float vreg[4][NC];
  auto load_v = [&](int kb) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* row = vp + (int64_t)min(16 * kb + 4 * g + i, p.Sk - 1) * p.v_ss + r;
#pragma unroll
      for (int db = 0; db < NC; ++db) vreg[i][db] = row[16 * db];
    }
  };

  // Q through the slot into fragments: element j of chunk c of lane (r, g) is head-dim element g * D/4 + 4c + j.
  f32x4 qf[NC];
  {
    f32x4 x[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = lane + 64 * i;
      x[i] = *reinterpret_cast<const f32x4*>(qp + (int64_t)min(q0 + c / CPR, p.Sq - 1) * p.q_ss + 4 * (c % CPR));
    }
    if (b_begin < b_end) load_k(b_begin);
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = lane + 64 * i;
      *reinterpret_cast<f32x4*>(slot + (c / CPR) * RS + 4 * (c % CPR)) = x[i];
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) qf[c] = *reinterpret_cast<const f32x4*>(slot + r * RS + g * (D / 4) + 4 * c);
  }

  f32x4 o[NC];
  float m = -INFINITY, l = 0.f;
#pragma unroll
  for (int db = 0; db < NC; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int kb = b_begin; kb < b_end; kb += kKG) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = lane + 64 * i;
      *reinterpret_cast<f32x4*>(slot + (c / CPR) * RS + 4 * (c % CPR)) = kreg[i];
    }
    load_v(kb);
    if (kb + kKG < b_end) load_k(kb + kKG);
    // four partial sums per score (element j of every chunk), added pairwise: short chains, for speed and rounding
    f32x4 sp[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) sp[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const f32x4 kf = *reinterpret_cast<const f32x4*>(slot + r * RS + g * (D / 4) + 4 * c);
#pragma unroll
      for (int j = 0; j < 4; ++j) sp[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j], qf[c][j], sp[j], 0, 0, 0);
    }
    f32x4 s = (sp[0] + sp[1]) + (sp[2] + sp[3]);
    // register i: key 16 kb + 4g + i of query r
    float mt = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = 16 * kb + 4 * g + i;
      const float x = f32_score<SOFTCAP>(s[i], p);
      s[i] = key >= k_lo && key <= k_hi ? x : -INFINITY;
      mt = fmaxf(mt, s[i]);
    }
    mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    const float m_new = fmaxf(m, mt);
    if (__any(m_new > m)) {
      const float alpha = m_new > m ? expf(m - m_new) : 1.0f;  // 0 while m is -inf
      l *= alpha;
#pragma unroll
      for (int db = 0; db < NC; ++db) o[db] *= alpha;
      m = m_new;
    }
    const float mu = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = expf(s[i] - mu);
    l += (s[0] + s[1]) + (s[2] + s[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int db = 0; db < NC; ++db)
        o[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vreg[i][db], s[i], o[db], 0, 0, 0);
  }

  // Combine the waves: O = sum_w e^(m_w - m) O_w / sum_w e^(m_w - m) l_w. O register i of block db: head-dim element
  // 16 db + 4g + i of query r.
  __syncthreads();  // the K slots are done with
  float* ml = smem + SMEM - 2 * kKG * 16;
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (g == 0) {
    ml[kg * 32 + r] = m;
    ml[kg * 32 + 16 + r] = l;
  }
#pragma unroll
  for (int db = 0; db < NC; ++db) *reinterpret_cast<f32x4*>(smem + kg * OSLOT + (db * 64 + lane) * 4) = o[db];
  __syncthreads();
  float wt[kKG], mx = -INFINITY, lt = 0.f;
#pragma unroll
  for (int w = 0; w < kKG; ++w) mx = fmaxf(mx, ml[w * 32 + r]);
  const float mu = mx == -INFINITY ? 0.f : mx;
#pragma unroll
  for (int w = 0; w < kKG; ++w) {
    wt[w] = expf(ml[w * 32 + r] - mu);  // 0 for a wave that saw no key of the row
    lt = fmaf(wt[w], ml[w * 32 + 16 + r], lt);
  }
#pragma unroll
  for (int it = 0; it < NC / kKG; ++it) {
    const int db = it * kKG + kg;
    f32x4 ot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kKG; ++w) ot += wt[w] * *reinterpret_cast<const f32x4*>(smem + w * OSLOT + (db * 64 + lane) * 4);
    if (qi < p.Sq) {
      // no keys at all: o = 0 (an empty P.V); a row that sees no key: 0 * inf = NaN, the reference's softmax of -inf
      const float inv = p.Sk == 0 ? 0.f : 1.0f / lt;
      float* op = static_cast<float*>(p.o) + b * p.o_sb + (int64_t)qi * p.o_ss + h * p.o_sh;
      *reinterpret_cast<f32x4*>(op + 16 * db + 4 * g) = ot * inv;
      if (p.lse != nullptr && db == 0 && g == 0) {
        const float lse = mx == -INFINITY ? -INFINITY : mx + logf(lt);
        p.lse[(int64_t)bh * p.Sq + qi] = p.lse_base2 ? lse * kLog2e : lse;
      }
    }
  }
}

template <int D, bool SOFTCAP, int EPI>
__global__ void __launch_bounds__(kThr) attn_col_f32_kernel(AttnParams p) {
  constexpr int DQ = D / 4;
  __shared__ __attribute__((aligned(16))) float Qs[kTile][D + 4];
  __shared__ float Ls[kTile];
  int kt, bh;
  map_block(p.n_tiles, p.B * p.Hq, false, kt, bh);
  const int b = bh / p.Hq, h = bh - b * p.Hq, hk = h / p.group;
  const int col = threadIdx.x >> 2, qd = threadIdx.x & 3;
  const int k0 = kt * kRows, kj = k0 + col;
  const float* qp = static_cast<const float*>(p.q) + b * p.q_sb + h * p.q_sh;
  const float* kp = static_cast<const float*>(p.k) + b * p.k_sb + hk * p.k_sh;
  const float* lsep = p.lse + (int64_t)bh * p.Sq;

  float kv[DQ];
  const float* krow = kp + (int64_t)min(kj, p.Sk - 1) * p.k_ss + qd * DQ;
#pragma unroll
  for (int e = 0; e < DQ; e += 4) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(krow + e);
    kv[e] = v[0];
    kv[e + 1] = v[1];
    kv[e + 2] = v[2];
    kv[e + 3] = v[3];
  }

  // Query rows that can see any key of this workgroup.
  const int k_last = min(k0 + kRows, p.Sk) - 1;
  int q_begin = 0, q_end = p.Sq;
  if (p.causal) q_begin = max(0, k0 - p.offset);
  if (p.window > 0) q_end = min(p.Sq, k_last - p.offset + p.window);

  float sum = 0.f, sum2 = 0.f;
  int any = 0;
  for (int qb = (q_begin / kTile) * kTile; qb < q_end; qb += kTile) {
    __syncthreads();
    stage_rows<D>(Qs, qp, p.q_ss, qb, p.Sq);
    if (threadIdx.x < kTile) {
      const int qg = qb + threadIdx.x;
      Ls[threadIdx.x] = qg < p.Sq ? (p.lse_base2 ? lsep[qg] * kLn2 : lsep[qg]) : INFINITY;
    }
    __syncthreads();
#pragma unroll 4
    for (int i = 0; i < kTile; ++i) {
      const int qg = qb + i;
      const float x = f32_score<SOFTCAP>(quad_dot<D>(kv, &Qs[i][qd * DQ]), p);
      bool ok = qg < p.Sq && kj < p.Sk;
      if (p.causal) ok = ok && kj <= qg + p.offset;
      if (p.window > 0) ok = ok && qg + p.offset - kj < p.window;
      const float pe = ok ? expf(x - Ls[i]) : 0.f;
      if constexpr (EPI == kColAnyGe) {
        if (ok) any |= pe >= p.thr[(int64_t)qg * p.thr_rs + kj];  // masked pairs: corm_masked_or_kernel
      } else {
        sum += pe;
        if constexpr (EPI == kColSumSq) sum2 = fmaf(pe, pe, sum2);
      }
    }
  }
  if (qd == 0 && kj < p.Sk) {
    const int64_t idx = (int64_t)bh * p.Sk + kj;
    if constexpr (EPI == kColAnyGe) {
      p.any_out[idx] = (uint8_t)(any != 0);
    } else {
      p.colsum[idx] = sum;
      if constexpr (EPI == kColSumSq) p.colsum2[idx] = sum2;
    }
  }
}

template <int D>
void fwd_f32(AttnParams p, hipStream_t st) {
  p.n_tiles = (p.Sq + kF32Rows - 1) / kF32Rows;
  launch_blocks(p, 64 * kKG, [&](unsigned grid, const AttnParams& p) {
    if (p.softcap > 0.f) hipLaunchKernelGGL((attn_fwd_f32_kernel<D, true>), dim3(grid), dim3(64 * kKG), 0, st, p);
    else hipLaunchKernelGGL((attn_fwd_f32_kernel<D, false>), dim3(grid), dim3(64 * kKG), 0, st, p);
  });
}
template <int D, bool SOFTCAP, int EPI>
void launch_col_f32_d(const AttnParams& p, hipStream_t st) {
  const unsigned grid = (unsigned)p.n_tiles * p.B * p.Hq;
  hipLaunchKernelGGL((attn_col_f32_kernel<D, SOFTCAP, EPI>), dim3(grid), dim3(kThr), 0, st, p);
}
template <int D>
void col_f32(const AttnParams& p, int epi, hipStream_t st) {
  if (epi == kColSumSq) return launch_col_f32_d<D, false, kColSumSq>(p, st);
  if (epi == kColAnyGe) return launch_col_f32_d<D, false, kColAnyGe>(p, st);
  if (p.softcap > 0.f) launch_col_f32_d<D, true, kColSum>(p, st);
  else launch_col_f32_d<D, false, kColSum>(p, st);
}

}  // namespace

int f32_rows_per_tile() { return kRows; }

void launch_attn_f32_fwd(const AttnParams& p, int D, hipStream_t st) {
  if (D == 64) fwd_f32<64>(p, st);
  else if (D == 128) fwd_f32<128>(p, st);
  else fwd_f32<256>(p, st);
}

void launch_attn_f32_col(const AttnParams& p, int D, int epi, hipStream_t st) {
  if (D == 64) col_f32<64>(p, epi, st);
  else if (D == 128) col_f32<128>(p, epi, st);
  else col_f32<256>(p, epi, st);
}

}  // namespace dgg_attn
