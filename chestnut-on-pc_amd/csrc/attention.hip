// Non-causal multi-head attention for the token block of the driving model.
//
// The reference's attention lives in comma's pickle as WMMA GEMM kernels
// (NOTES.md:84-104); this is the gfx950 form of the same f16-input,
// f32-accumulate products with an f32 softmax between them.
//
// One workgroup = 32 queries of one head (T=512, 16 heads: 256 workgroups,
// one per CU), split over the keys: wave w owns keys [w*KPW, (w+1)*KPW) for
// all 32 queries and needs nothing from the other waves until the end:
//   1. S^T = K Q^T * scale*log2(e) for its keys with v_mfma_f32_16x16x32_f16
//      (A = 16 keys x 32 head dims of K, B = Q^T); lane (g = l/16, r = l%16)
//      holds keys 4g..4g+3 of every 16-key tile for query r;
//   2. a wave-local softmax numerator: per query the max m_w over the wave's
//      keys (lane-local, then xor-16/xor-32 exchanges), e = 2^(s - m_w) on
//      the hardware exp2, l_w = sum of e; e is rounded to f16 (values in
//      (0, 1]) and is, as it stands in the registers, the A operand of P.V:
//      the two 16-key tiles of a 32-key block give lane (g, r) the keys
//      {4g..4g+3, 16+4g..16+4g+3} of query r;
//   3. O_w = e . V over the wave's keys, B = V in the same permuted key order
//      (the QKV GEMM's fragment epilogue writes V that way);
//   4. each wave leaves O_w, m_w and l_w in LDS; after one barrier the
//      threads combine 4 features of one query at a time over the waves in
//      fixed order: M = max m_w, O = sum 2^(m_w - M) O_w / sum 2^(m_w - M) l_w
//      (with the O-projection: f16 P_w = O_w / l_w, weighted by 2^(m_w - M) l_w).
// The result is deterministic; each wave streams only its own K and V.
// Workgroups are regrouped by XCD (consecutive ids land on different XCDs):
// each XCD's L2 then serves the K/V of T*hd*2*2 bytes for 2 heads.
// MFMA 16x16x32 layout (lane l): A row l%16, k = 8*(l/16)..+7; B column
// l%16, same k; D element i of lane l is row 4*(l/16)+i, column l%16.
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace ck {
namespace {

constexpr int ATT_TMAX = 512;
constexpr int ATT_QB = 32;   // queries per workgroup

__device__ __forceinline__ float xor_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16));
  return fmaxf(v, __shfl_xor(v, 32));
}
__device__ __forceinline__ float xor_sum(float v) {
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}

// Row-layout operands.  An MFMA fragment wants lane (g, r) to hold 16-byte chunk g
// of row r.  A load in that order has neighbouring lanes on 16 different rows: 64
// pieces of 16 bytes for the address unit, which bounds the kernel.  So rows are
// loaded as they lie, RB bytes (128 or 64) of a row by RB / 16 neighbouring lanes,
// and turned through LDS that the wave owns (no barrier): row-major there, chunk c
// of a row at c ^ f(row), with f such that the 16 lanes served together hit 16
// different 16-byte bank groups, in the writes and in the fragment reads alike.
// Per launch against loads in fragment order (graph replays): 16 heads of 128 at
// 512 tokens 11.6 -> 8.5 us, 32 of them 22.5 -> 16.6, 8 at 320 7.1 -> 5.4, 16 heads
// of 64 at 512 7.0 -> 5.6, 8 at 256 4.2 -> 3.5, 4 at 64 2.6 either way.
template <int N, int RB>
__device__ __forceinline__ void rows_load(half8_t (&v)[N], const half_t* base, long stride, int lane) {
  constexpr int CH = RB / 16;
  const half_t* p = base + (lane / CH) * stride + (lane % CH) * 8;
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = *reinterpret_cast<const half8_t*>(p + (long)i * (64 / CH) * stride);
}
// byte of chunk c of a row; SWZ 0: fragments of 16 consecutive rows, 1: K's (rows 8q + 4p + i, q and i = 0..3)
template <int RB, int SWZ>
__device__ __forceinline__ int row_chunk(int row, int c) {
  const int f = RB == 64 ? (row >> 2) & 3 : SWZ ? ((row >> 1) & 1) | ((row >> 2) & 6) : (row >> 1) & 7;
  return row * RB + ((c ^ f) << 4);
}
template <int N, int RB, int SWZ>
__device__ __forceinline__ void rows_to_lds(char* st, const half8_t (&v)[N], int lane) {
  constexpr int CH = RB / 16;
  const int r = lane / CH, c = lane % CH;
#pragma unroll
  for (int i = 0; i < N; ++i) *reinterpret_cast<half8_t*>(st + row_chunk<RB, SWZ>(i * (64 / CH) + r, c)) = v[i];
}

// Waves per workgroup for T = 64*NKT keys: every wave owns 32 or 64 keys.
constexpr int att_waves(int nkt) { return nkt <= 4 ? 2 * nkt : nkt; }

// FRAG: qk / vt hold the operands in MFMA fragment order (written by the QKV
// GEMM's fragment epilogue): every fragment load of a wave is one contiguous
// KB.  Otherwise the row layouts: qk [T][2d], vt [d][T].  There the two 16-key
// tiles of a 32-key block take the keys 8q..8q+3 and 8q+4..8q+7 (q = 0..3) of
// the block as their rows, so that the softmax leaves lane (g, r) the keys
// 8g..8g+7: one 16-byte chunk of a V^T row.  The rows reach the fragments
// through LDS (rows_load).  Spreading a head over the XCDs measured slower
// (13.6 us against 12.9 with loads in fragment order).  All of a wave's loads
// (Q, its K, its V) are issued at entry, before any MFMA.
// QT: 16-query tiles per workgroup (2: 32 queries; 1: 16, twice the
// workgroups for short sequences that would leave most CUs idle).
// OTW > 0: the output projection rides along.  The workgroup's normalised
// f16 output (QB queries x HD features of head h) goes to LDS instead of
// memory, and wave w multiplies it by columns [h*HD, (h+1)*HD) of W_o
// ([d][d], row n = output feature) for output features
// [16*OTW*w, 16*OTW*(w+1)): P_h = O_h W_o[:, h]^T, an f32 plane per head,
// opart + h*T*d, [T][d].  The planes are the split-K partials of the
// O-projection over its K = d split by heads; the next LayerNorm sums them
// in head order with the bias.  W_o's fragments are loaded at entry with
// everything else.
template <int HD, int NKT, bool FRAG, int QT = 2, int OTW = 0>
__global__ __launch_bounds__(64 * att_waves(NKT)) void attention_kernel(const half_t* __restrict__ qk,
                                                                         const half_t* __restrict__ vt,
                                                                         half_t* __restrict__ out, int n_heads,
                                                                         float scale_log2e,
                                                                         const half_t* __restrict__ wo,
                                                                         float* __restrict__ opart) {
  constexpr int QB = 16 * QT;        // queries per workgroup
  constexpr int WAVES = att_waves(NKT);
  constexpr int T = 64 * NKT;
  constexpr int KS = HD / 32;        // k-steps of the q.k products
  constexpr int KPW = T / WAVES;     // keys per wave
  constexpr int KT = KPW / 16;       // 16-key tiles per wave
  constexpr int KB = KPW / 32;       // 32-key blocks (k-steps of P.V)
  constexpr int CT = HD / 16;        // 16-wide output tiles
  static_assert(KPW % 32 == 0, "every wave must own whole 32-key blocks");
  // The waves' partial outputs: f16 P_w = O_w / l_w where the O-projection
  // rides along (half the LDS bytes of the combine: 39M frame -0.75%), f32
  // O_w otherwise (the f16 form's extra conversions cost the 1B frame +0.6%).
  // Row pitch: f32 HD + 4 floats (the 4-row scatter of each lane's
  // accumulators hits distinct banks); f16 HD + 8 halves (4 banks mod 64, so
  // the 32 lanes of a half-wave writing 8 bytes each hit 64 distinct banks).
  constexpr bool P16 = OTW > 0;
  typedef std::conditional_t<P16, half_t, float> part_t;
  constexpr int OP = P16 ? HD + 8 : HD + 4;
  // row layout: each wave's area for turning K, Q and V^T into fragments, in the
  // same memory (the partial outputs come after the last fragment read)
  constexpr int TURN = FRAG ? 0 : (KPW > QB ? KPW : QB) * HD * 2;
  constexpr int SMEM = WAVES * QB * OP * (int)sizeof(part_t) > WAVES * TURN ? WAVES * QB * OP * (int)sizeof(part_t)
                                                                            : WAVES * TURN;
  __shared__ __attribute__((aligned(16))) char smem[SMEM];
  part_t (*const part)[QB][OP] = reinterpret_cast<part_t (*)[QB][OP]>(smem);
  __shared__ float mrow[WAVES][QB], lrow[WAVES][QB];
  constexpr int KSO = HD / 32;       // k-steps of the O-projection
  constexpr int OBP = HD + 8;        // f16 output row pitch in LDS (16-byte rows)
  __shared__ __attribute__((aligned(16))) half_t ob[OTW > 0 ? QB : 1][OBP];

  const int d = n_heads * HD;
  const int nqb = T / QB;
  const int total = nqb * n_heads;
  int L = blockIdx.x;
  if ((total & 7) == 0) L = (L & 7) * (total >> 3) + (L >> 3);
  const int h = L / nqb, q0 = (L % nqb) * QB;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, g = lane >> 4;
  const long ldq = 2L * d;
  const int kw0 = wave * KPW;

  // ---- all loads up front ----
  half8_t qf[QT][KS], kf[KT][KS], vb[KB][CT];
  constexpr int VRB = KPW * 2, NVL = HD * VRB / 1024;   // row layout: V^T rows of KPW keys, their loads
  half8_t vl[FRAG ? 1 : NVL];
  char* const turn = reinterpret_cast<char*>(smem) + wave * TURN;
  if constexpr (FRAG) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        kf[kt][ks] = *reinterpret_cast<const half8_t*>(
            qk + ((((long)(n_heads + h) * (T / 16) + kw0 / 16 + kt) * KS + ks) * 64 + lane) * 8);
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        qf[qt][ks] = *reinterpret_cast<const half8_t*>(
            qk + ((((long)h * (T / 16) + q0 / 16 + qt) * KS + ks) * 64 + lane) * 8);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        vb[kb][ct] = *reinterpret_cast<const half8_t*>(
            vt + ((((long)h * (HD / 16) + ct) * (T / 32) + kw0 / 32 + kb) * 64 + lane) * 8);
  } else {
    // halves of 64 head dims: 8 rows of 128 bytes per load
    constexpr int HH = HD / 64, NK = KPW / 8, NQ = QB / 8;
    half8_t kl[HH][NK], ql[HH][NQ];
#pragma unroll
    for (int f = 0; f < HH; ++f) rows_load<NK, 128>(kl[f], qk + (long)kw0 * ldq + d + h * HD + f * 64, ldq, lane);
#pragma unroll
    for (int f = 0; f < HH; ++f) rows_load<NQ, 128>(ql[f], qk + (long)q0 * ldq + h * HD + f * 64, ldq, lane);
    rows_load<NVL, VRB>(vl, vt + (long)h * HD * T + kw0, T, lane);
#pragma unroll
    for (int f = 0; f < HH; ++f) rows_to_lds<NK, 128, 1>(turn + f * KPW * 128, kl[f], lane);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)   // tile row r is key (r / 4) * 8 + (kt % 2) * 4 + r % 4 of its 32-key block
        kf[kt][ks] = *reinterpret_cast<const half8_t*>(
            turn + (ks >> 1) * KPW * 128 +
            row_chunk<128, 1>((kt >> 1) * 32 + (r16 >> 2) * 8 + (kt & 1) * 4 + (r16 & 3), (ks & 1) * 4 + g));
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int f = 0; f < HH; ++f) rows_to_lds<NQ, 128, 0>(turn + f * QB * 128, ql[f], lane);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        qf[qt][ks] = *reinterpret_cast<const half8_t*>(turn + (ks >> 1) * QB * 128 +
                                                       row_chunk<128, 0>(qt * 16 + r16, (ks & 1) * 4 + g));
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
  }
  // W_o fragments (MFMA A operand: row n = output feature, 8 k of head h's columns)
  half8_t wf[OTW > 0 ? OTW : 1][KSO];
  if constexpr (OTW > 0) {
#pragma unroll
    for (int t = 0; t < OTW; ++t)
#pragma unroll
      for (int ks = 0; ks < KSO; ++ks)
        wf[t][ks] = *reinterpret_cast<const half8_t*>(wo + (long)((wave * OTW + t) * 16 + r16) * d + h * HD +
                                                      ks * 32 + g * 8);
  }

  // ---- 1. S^T = K Q^T for this wave's keys (log2 domain) ----
  float4_t s[KT][QT];
#pragma unroll
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      float4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[kt][ks], qf[qt][ks], a, 0, 0, 0);
      s[kt][qt] = a * scale_log2e;
    }

  // ---- 2. wave-local softmax numerator per query (column r16 of q-tile qt) ----
  half8_t pa[KB][QT];
  float lw[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    float m = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) m = fmaxf(m, s[kt][qt][i]);
    m = xor_max(m);
    float acc = 0.f;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float e = __builtin_amdgcn_exp2f(s[2 * kb + i / 4][qt][i % 4] - m);
        acc += e;
        pa[kb][qt][i] = (half_t)e;
      }
    acc = xor_sum(acc);
    lw[qt] = acc;
    if (g == 0) {
      mrow[wave][qt * 16 + r16] = m;
      lrow[wave][qt * 16 + r16] = acc;
    }
  }

  if constexpr (!FRAG) {
    rows_to_lds<NVL, VRB, 0>(turn, vl, lane);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        vb[kb][ct] = *reinterpret_cast<const half8_t*>(turn + row_chunk<VRB, 0>(ct * 16 + r16, kb * 4 + g));
    // part overlaps the turning areas: every wave is past its V reads
    wait_vm_lgkm0<0>();
    lds_barrier();
  }
  // ---- 3. O_w = e V over this wave's keys ----
  if constexpr (P16) {
    // O_w^T = V^T e^T (operands swapped: lane (g, r16) ends with head dims
    // 16ct + 4g .. +3 of query 16qt + r16), divided by the wave's l_w: a convex
    // combination of V rows, so within V's range; one 8-byte write per tile
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const float rl = 1.0f / lw[qt];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        float4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) a = __builtin_amdgcn_mfma_f32_16x16x32_f16(vb[kb][ct], pa[kb][qt], a, 0, 0, 0);
        *reinterpret_cast<half4_t*>(&part[wave][qt * 16 + r16][ct * 16 + 4 * g]) =
            half4_t{(half_t)(a[0] * rl), (half_t)(a[1] * rl), (half_t)(a[2] * rl), (half_t)(a[3] * rl)};
      }
    }
  } else {
    float4_t o[QT][CT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        float4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) a = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[kb][qt], vb[kb][ct], a, 0, 0, 0);
        o[qt][ct] = a;
      }
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i) part[wave][qt * 16 + 4 * g + i][ct * 16 + r16] = o[qt][ct][i];
  }
  __syncthreads();

  // ---- 4. combine the waves: 4 features of one query per step, in fixed wave order ----
  for (int u = threadIdx.x; u < QB * HD / 4; u += 64 * WAVES) {
    const int q = u / (HD / 4), c = (u % (HD / 4)) * 4;
    float M = mrow[0][q];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) M = fmaxf(M, mrow[w][q]);
    float den = 0.f;
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float f = __builtin_amdgcn_exp2f(mrow[w][q] - M);
      if constexpr (P16) {
        const float fl = f * lrow[w][q];
        const half4_t pw = *reinterpret_cast<const half4_t*>(&part[w][q][c]);
        den += fl;
        acc += fl * float4_t{(float)pw[0], (float)pw[1], (float)pw[2], (float)pw[3]};
      } else {
        den += f * lrow[w][q];
        acc += f * *reinterpret_cast<const float4_t*>(&part[w][q][c]);
      }
    }
    const float rden = 1.0f / den;
    const half4_t v{(half_t)(acc[0] * rden), (half_t)(acc[1] * rden), (half_t)(acc[2] * rden), (half_t)(acc[3] * rden)};
    if constexpr (OTW > 0) {
      *reinterpret_cast<half4_t*>(&ob[q][c]) = v;
    } else {
      // device-scope cache policy for the output the O-projection reads next (-0.4% of the 1B frame)
      store_sc1(sc1_rsrc(out, 2L * T * d), ((long)(q0 + q) * d + h * HD + c) * 2, v);
    }
  }

  // ---- 5. (OTW > 0) P_h^T = W_o[n-tile, head h] O_h^T: lane (g, r16) ends with
  // output features 4g..4g+3 of the tile for query r16, one 16-byte store ----
  if constexpr (OTW > 0) {
    __syncthreads();
    half8_t of[QT][KSO];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int ks = 0; ks < KSO; ++ks)
        of[qt][ks] = *reinterpret_cast<const half8_t*>(&ob[qt * 16 + r16][ks * 32 + g * 8]);
    const auto pr = sc1_rsrc(opart + (long)h * T * d, 4L * T * d);
#pragma unroll
    for (int t = 0; t < OTW; ++t)
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        float4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KSO; ++ks) a = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[t][ks], of[qt][ks], a, 0, 0, 0);
        // device-scope cache policy: the LayerNorm reads the planes next
        store_sc1(pr, ((long)(q0 + qt * 16 + r16) * d + (wave * OTW + t) * 16 + 4 * g) * 4, a);
      }
  }
}

template <int HD, int NKT, bool FRAG>
void launch_t(int n_heads, const half_t* qk, const half_t* vt, half_t* out, float scale_log2e, hipStream_t s) {
  // 32 queries per workgroup, or 16 when that would leave more than half the CUs idle
  const int wg32 = (64 * NKT / ATT_QB) * n_heads;
  if (wg32 >= 128) {
    CK_LAUNCH((attention_kernel<HD, NKT, FRAG, 2>), dim3(wg32), dim3(64 * att_waves(NKT)), 0, s, qk, vt, out, n_heads,
              scale_log2e, nullptr, nullptr);
  } else {
    CK_LAUNCH((attention_kernel<HD, NKT, FRAG, 1>), dim3(2 * wg32), dim3(64 * att_waves(NKT)), 0, s, qk, vt, out,
              n_heads, scale_log2e, nullptr, nullptr);
  }
}

// With the O-projection: the same workgroup choice; OTW = d / 16 / waves
// output tiles per wave (checked by attention_oproj_tiles).
template <int HD, int NKT, int OTW>
void launch_o(int n_heads, const half_t* qk, const half_t* vt, const half_t* wo, float* opart, float scale_log2e,
              hipStream_t s) {
  const int wg32 = (64 * NKT / ATT_QB) * n_heads;
  if (wg32 >= 128) {
    CK_LAUNCH((attention_kernel<HD, NKT, true, 2, OTW>), dim3(wg32), dim3(64 * att_waves(NKT)), 0, s, qk, vt, nullptr,
              n_heads, scale_log2e, wo, opart);
  } else {
    CK_LAUNCH((attention_kernel<HD, NKT, true, 1, OTW>), dim3(2 * wg32), dim3(64 * att_waves(NKT)), 0, s, qk, vt,
              nullptr, n_heads, scale_log2e, wo, opart);
  }
}

template <int HD, int NKT>
void launch_o_t(int otw, int n_heads, const half_t* qk, const half_t* vt, const half_t* wo, float* opart,
                float scale_log2e, hipStream_t s) {
  switch (otw) {
    case 1: launch_o<HD, NKT, 1>(n_heads, qk, vt, wo, opart, scale_log2e, s); break;
    case 2: launch_o<HD, NKT, 2>(n_heads, qk, vt, wo, opart, scale_log2e, s); break;
    default: launch_o<HD, NKT, 4>(n_heads, qk, vt, wo, opart, scale_log2e, s); break;
  }
}

template <int HD>
void launch_o_hd(int T, int otw, int n_heads, const half_t* qk, const half_t* vt, const half_t* wo, float* opart,
                 float scale_log2e, hipStream_t s) {
  switch (T / 64) {
    case 1: launch_o_t<HD, 1>(otw, n_heads, qk, vt, wo, opart, scale_log2e, s); break;
    case 2: launch_o_t<HD, 2>(otw, n_heads, qk, vt, wo, opart, scale_log2e, s); break;
    case 3: launch_o_t<HD, 3>(otw, n_heads, qk, vt, wo, opart, scale_log2e, s); break;
    case 4: launch_o_t<HD, 4>(otw, n_heads, qk, vt, wo, opart, scale_log2e, s); break;
    case 5: launch_o_t<HD, 5>(otw, n_heads, qk, vt, wo, opart, scale_log2e, s); break;
    case 6: launch_o_t<HD, 6>(otw, n_heads, qk, vt, wo, opart, scale_log2e, s); break;
    case 7: launch_o_t<HD, 7>(otw, n_heads, qk, vt, wo, opart, scale_log2e, s); break;
    default: launch_o_t<HD, 8>(otw, n_heads, qk, vt, wo, opart, scale_log2e, s); break;
  }
}

template <int HD, bool FRAG>
void launch_hd(int T, int n_heads, const half_t* qk, const half_t* vt, half_t* out, float scale_log2e,
               hipStream_t s) {
  switch (T / 64) {
    case 1: launch_t<HD, 1, FRAG>(n_heads, qk, vt, out, scale_log2e, s); break;
    case 2: launch_t<HD, 2, FRAG>(n_heads, qk, vt, out, scale_log2e, s); break;
    case 3: launch_t<HD, 3, FRAG>(n_heads, qk, vt, out, scale_log2e, s); break;
    case 4: launch_t<HD, 4, FRAG>(n_heads, qk, vt, out, scale_log2e, s); break;
    case 5: launch_t<HD, 5, FRAG>(n_heads, qk, vt, out, scale_log2e, s); break;
    case 6: launch_t<HD, 6, FRAG>(n_heads, qk, vt, out, scale_log2e, s); break;
    case 7: launch_t<HD, 7, FRAG>(n_heads, qk, vt, out, scale_log2e, s); break;
    default: launch_t<HD, 8, FRAG>(n_heads, qk, vt, out, scale_log2e, s); break;
  }
}

}  // namespace

void launch_attention(const half_t* qk, const half_t* vt, half_t* out, int T, int n_heads, int head_dim, bool frag,
                      hipStream_t s) {
  CK_REQUIRE(qk && vt && out, "attention: null pointer");
  CK_REQUIRE(T > 0 && T % 64 == 0 && T <= ATT_TMAX, "attention: T must be a multiple of 64 and <= 512");
  CK_REQUIRE(head_dim == 64 || head_dim == 128, "attention: head_dim must be 64 or 128");
  CK_REQUIRE(n_heads > 0, "attention: n_heads must be positive");
  // the output leaves through raw buffer stores addressed by 32-bit offsets
  CK_REQUIRE(2L * T * n_heads * head_dim < (1L << 31), "attention: output must be under 2 GiB");
  CK_REQUIRE((reinterpret_cast<uintptr_t>(qk) & 15) == 0 && (reinterpret_cast<uintptr_t>(vt) & 15) == 0 &&
                 (reinterpret_cast<uintptr_t>(out) & 7) == 0,
             "attention: qk and vt must be 16-byte and out 8-byte aligned");
  // scores go straight to the exp2 domain: s * (1/sqrt(hd)) * log2(e)
  const float scale_log2e = 1.4426950408889634f / sqrtf((float)head_dim);
  if (frag) {
    if (head_dim == 64) launch_hd<64, true>(T, n_heads, qk, vt, out, scale_log2e, s);
    else launch_hd<128, true>(T, n_heads, qk, vt, out, scale_log2e, s);
  } else {
    if (head_dim == 64) launch_hd<64, false>(T, n_heads, qk, vt, out, scale_log2e, s);
    else launch_hd<128, false>(T, n_heads, qk, vt, out, scale_log2e, s);
  }
  CK_LAUNCHED("attention");
}

int attention_oproj_tiles(int T, int n_heads, int head_dim) {
  if (T <= 0 || T % 64 != 0 || T > ATT_TMAX || (head_dim != 64 && head_dim != 128) || n_heads <= 0) return 0;
  const int tiles = n_heads * head_dim / 16, waves = att_waves(T / 64);
  if (tiles % waves != 0) return 0;
  const int otw = tiles / waves;
  return (otw == 1 || otw == 2 || otw == 4) ? otw : 0;
}

void launch_attention_oproj(const half_t* qk, const half_t* vt, const half_t* wo, float* opart, int T, int n_heads,
                            int head_dim, hipStream_t s) {
  CK_REQUIRE(qk && vt && wo && opart, "attention_oproj: null pointer");
  const int otw = attention_oproj_tiles(T, n_heads, head_dim);
  CK_REQUIRE(otw > 0,
             "attention_oproj: needs T a multiple of 64 up to 512, head_dim 64 or 128, and 1, 2 or 4 output "
             "tiles of 16 features per wave");
  CK_REQUIRE(4L * T * n_heads * head_dim < (1L << 31), "attention_oproj: partial plane too large");
  CK_REQUIRE(((reinterpret_cast<uintptr_t>(qk) | reinterpret_cast<uintptr_t>(vt) | reinterpret_cast<uintptr_t>(wo) |
               reinterpret_cast<uintptr_t>(opart)) & 15) == 0,
             "attention_oproj: operands must be 16-byte aligned");
  const float scale_log2e = 1.4426950408889634f / sqrtf((float)head_dim);
  if (head_dim == 64) launch_o_hd<64>(T, otw, n_heads, qk, vt, wo, opart, scale_log2e, s);
  else launch_o_hd<128>(T, otw, n_heads, qk, vt, wo, opart, scale_log2e, s);
  CK_LAUNCHED("attention_oproj");
}

}  // namespace ck
