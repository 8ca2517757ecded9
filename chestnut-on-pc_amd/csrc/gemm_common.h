// Shared by the GEMM kernels (gemm.hip, gemm_pipe.hip): the parameter block,
// the per-element and LDS-staged epilogues, and the swizzle of a [K][N] stage.
#pragma once

#include "common.h"
#include "kernels.h"

namespace ck {

constexpr int BK = 64;

struct GemmParams {
  const half_t* A;
  const half_t* B;
  void* C;
  const float* bias;
  float* ws;
  half_t* vt;
  long lda, ldb, ldc, vt_ld;
  long sA, sB, sC, sBias;
  int M, N, K, kps;   // kps: K per split
  int split, batch, Mt, Nt;
  int qk_cols;
  int head_dim;       // EPI_QKV_FRAG
  int vec;            // 1: shapes/alignment allow the LDS-staged 16-byte epilogue
  const half_t* pos;  // EPI_EMBED
  const float* ctx;   // EPI_EMBED
  int cc_log2, ch, cw, cwo;   // implicit conv: log2(channels), input height/width, output width
  const half_t* zero;         // implicit conv: 16 zero bytes
  int c_nm;                   // the split-K reduce stores element (m, n) at C[n*ldc + m]
  unsigned* pair;             // split 2, f32 output: ticket counters of the in-kernel finish (null: a reduce follows)
};

template <int EPI>
__device__ __forceinline__ void epi_store(const GemmParams& p, void* C, const float* bias, int m, int n, float v) {
  if (EPI == EPI_F32) {
    if (bias) v += bias[n];
    static_cast<float*>(C)[(long)m * p.ldc + n] = v;
  } else if (EPI == EPI_EMBED) {
    if (bias) v += bias[n];
    static_cast<float*>(C)[(long)m * p.ldc + n] = v + ((float)p.pos[(long)m * p.ldc + n] + p.ctx[n]);
  } else if (EPI == EPI_F32_RESID) {
    if (bias) v += bias[n];
    float* c = static_cast<float*>(C) + (long)m * p.ldc + n;
    *c = *c + v;
  } else {
    if (bias) v += bias[n];
    if (EPI == EPI_F16_BIAS_RELU) v = fmaxf(v, 0.f);
    if (EPI == EPI_F16_BIAS_GELU) v = gelu_fast(v);
    if (EPI == EPI_QKV_FRAG) {
      return;   // unreachable: the host admits EPI_QKV_FRAG only with the staged epilogue
    } else if (EPI == EPI_QKV && n >= p.qk_cols) {
      p.vt[(long)(n - p.qk_cols) * p.vt_ld + m] = (half_t)v;
    } else if (p.c_nm) {
      static_cast<half_t*>(C)[(long)n * p.ldc + m] = (half_t)v;
    } else {
      static_cast<half_t*>(C)[(long)m * p.ldc + n] = (half_t)v;
    }
  }
}

// The epilogue of `per` summed values of row m, columns n.. (4 of them with v4):
// row-major outputs take 4 values in one 16-byte (f32) or 8-byte (f16) store
// where the address allows, the same values as epi_store.
template <int EPI>
__device__ __forceinline__ void store_reduced(const GemmParams& p, int bz, int m, int n, const float (&v)[4], int per,
                                              bool v4) {
  void* C = (EPI == EPI_F32 || EPI == EPI_F32_RESID || EPI == EPI_EMBED)
                ? static_cast<void*>(static_cast<float*>(p.C) + bz * p.sC)
                : static_cast<void*>(static_cast<half_t*>(p.C) + bz * p.sC);
  const float* bias = p.bias ? p.bias + bz * p.sBias : nullptr;
  if (v4 && (EPI == EPI_F32 || ((EPI == EPI_F16_BIAS || EPI == EPI_F16_BIAS_RELU || EPI == EPI_F16_BIAS_GELU) &&
                                !p.c_nm))) {
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = bias ? v[e] + bias[n + e] : v[e];
      if (EPI == EPI_F16_BIAS_RELU) o[e] = fmaxf(o[e], 0.f);
      if (EPI == EPI_F16_BIAS_GELU) o[e] = gelu_fast(o[e]);
    }
    if (EPI == EPI_F32) {
      float* c = static_cast<float*>(C) + (long)m * p.ldc + n;
      if ((reinterpret_cast<uintptr_t>(c) & 15) == 0) {
        *reinterpret_cast<float4_t*>(c) = float4_t{o[0], o[1], o[2], o[3]};
        return;
      }
    } else {
      half_t* c = static_cast<half_t*>(C) + (long)m * p.ldc + n;
      if ((reinterpret_cast<uintptr_t>(c) & 7) == 0) {
        *reinterpret_cast<half4_t*>(c) = half4_t{(half_t)o[0], (half_t)o[1], (half_t)o[2], (half_t)o[3]};
        return;
      }
    }
  }
  if (v4 && EPI == EPI_F32_RESID) {
    float4_t* c = reinterpret_cast<float4_t*>(static_cast<float*>(C) + (long)m * p.ldc + n);
    if ((reinterpret_cast<uintptr_t>(c) & 15) == 0) {
      float4_t o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = bias ? v[e] + bias[n + e] : v[e];
      *c = *c + o;
      return;
    }
  }
  for (int e = 0; e < per; ++e) epi_store<EPI>(p, C, bias, m, n + e, v[e]);
}

// Coalesced epilogue.  The MFMA accumulator layout gives a lane one column
// and scattered rows, so direct stores are 2- or 4-byte pieces spread over
// 32 rows per instruction (and, for the transposed V of the QKV epilogue,
// over 32 V^T rows).  Instead each wave puts its finished (WM x WN) sub-tile
// -- bias and activation applied, converted to the output type -- into a
// private LDS region and writes it out as whole 16-byte row chunks.  V
// columns are staged transposed ([n][m]), four consecutive rows of a lane
// forming one 8-byte LDS write, so V^T rows leave contiguously as well.
// Row pitches carry 16 bytes of padding so the two half-waves' staging
// writes (rows r and r+4) fall in different banks.  Every staged output --
// split-K partials, f32 outputs (plain, residual-add, embedding), row-major
// f16 outputs and the QKV fragments, all read by the next kernel -- leaves
// with the device-scope cache policy (store_sc1: -0.5%, -0.4% and -0.3% of
// the 1B frame for the partials, the f16 outputs and the fragments against
// non-temporal or default stores) wherever the region is addressable by a
// 32-bit buffer offset (sc1_ok), and with non-temporal stores otherwise.
// Requires (checked on the host, else the direct per-element stores run):
// N % 8 == 0, ldc / batch stride / base of C and ws 16-byte compatible,
// and for QKV qk_cols % BN == 0 (% 32 on the 128x96 tile), M % 8 == 0 and
// vt_ld % 8 == 0.
//
// EPI_QKV_FRAG writes the attention kernel's MFMA operands directly, in
// 16-byte chunks ordered so that one wave's fragment load is one contiguous
// KB (16 lanes x 16 B per row of the fragment would otherwise touch 16
// separate rows).  With T = M tokens, d = qk_cols / 2, hd = head_dim,
// H = d / hd, chunk c of a fragment holds 8 halves for lane l = 16*g + r:
//   Q, K (16x16x32 A/B operand: row r = token, 8 head dims from 8*g):
//     C chunk (((w*H + h) * T/16 + t/16) * hd/32 + j/32) * 64 + 16*((j%32)/8) + t%16
//     for token t, head dim j of head h; w = 0 for Q, 1 for K.
//   V (B operand of P.V: column r = head dim, tokens 4g..4g+3 and
//   16+4g..16+4g+3 of a 32-token block, the attention kernel's key order):
//     vt chunk ((h * hd/16 + j/16) * T/32 + t/32) * 64 + 16*((t%16)/4) + j%16,
//     element (t/16)*4 + t%4 of the chunk.
// SWP (every epilogue but the QKV ones): the accumulators hold D^T (the MFMA
// ran with its operands swapped), so element e of tile (i, j) is row
// i*32 + lane%32, column j*32 + 8*(e/4) + 4*(lane/32) + e%4: a lane's four
// consecutive e are four consecutive columns of one row, staged with one 8-
// or 16-byte LDS write instead of four scalar ones; bcol[j][e] is the bias
// of that column (bcol[j][0] of column j*32 + lane%32 otherwise).
template <int WM, int WN, int FM, int FN, int EPI, bool SWP, int NBC>
__device__ __forceinline__ void store_staged(const GemmParams& p, const float16_t (&acc)[FM][FN],
                                             const float (&bcol)[FN][NBC], char* region, int mw, int nw, int sp,
                                             int bz, int lane) {
  const bool to_ws = p.split > 1 || EPI == EPI_PARTIALS;
  if (to_ws || EPI == EPI_F32 || EPI == EPI_F32_RESID || EPI == EPI_EMBED) {
    constexpr int PF = WN + 8;   // floats
    float* st = reinterpret_cast<float*>(region);
    if constexpr (SWP) {
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            float4_t v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * k + e] + bcol[j][4 * k + e];
            *reinterpret_cast<float4_t*>(st + (i * 32 + (lane & 31)) * PF + j * 32 + 8 * k + 4 * (lane >> 5)) = v;
          }
    } else {
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int c = j * 32 + (lane & 31);
        const float bv = bcol[j][0];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            st[(i * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3)) * PF + c] = acc[i][j][e] + bv;
      }
    }
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
    constexpr int CPR = WN / 4;   // 16-byte chunks per row
    float* dst = to_ws ? p.ws + ((long)sp * p.batch + bz) * (long)p.M * p.N : static_cast<float*>(p.C) + bz * p.sC;
    const long ld = to_ws ? p.N : p.ldc;
    const long plane = to_ws ? 4L * p.M * p.N : 4L * ((long)(p.M - 1) * p.ldc + p.N);
    const bool sc1 = sc1_ok(plane);
    const __amdgpu_buffer_rsrc_t rs = sc1_rsrc(dst, sc1 ? plane : 0);
    if constexpr (EPI == EPI_F32_RESID) {
      // NB chunks at a time, the residual's old values all loaded before the first
      // is added: one memory round trip per NB chunks (221x4120x64 on 128x128
      // tiles 13.1 -> 8.7 us)
      constexpr int NQ = WM * CPR / 64, NB = NQ < 8 ? NQ : 8;
      static_assert(NQ * 64 == WM * CPR && NQ % NB == 0, "chunks per lane");
#pragma unroll
      for (int q0 = 0; q0 < NQ; q0 += NB) {
        float4_t old[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          const int q = lane + 64 * (q0 + i), m = mw + q / CPR, n = nw + (q % CPR) * 4;
          old[i] = !to_ws && m < p.M && n < p.N ? *reinterpret_cast<const float4_t*>(dst + (long)m * ld + n) : float4_t{};
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          const int q = lane + 64 * (q0 + i), r = q / CPR, c = (q % CPR) * 4;
          const int m = mw + r, n = nw + c;
          if (m >= p.M || n >= p.N) continue;
          float4_t v = *reinterpret_cast<const float4_t*>(st + r * PF + c);
          if (!to_ws) v += old[i];
          if (sc1) store_sc1(rs, ((long)m * ld + n) * 4, v);
          else __builtin_nontemporal_store(v, reinterpret_cast<float4_t*>(dst + (long)m * ld + n));
        }
      }
      return;
    }
#pragma unroll 4
    for (int q = lane; q < WM * CPR; q += 64) {
      const int r = q / CPR, c = (q % CPR) * 4;
      const int m = mw + r, n = nw + c;
      if (m >= p.M || n >= p.N) continue;
      float4_t v = *reinterpret_cast<const float4_t*>(st + r * PF + c);
      float4_t* g = reinterpret_cast<float4_t*>(dst + (long)m * ld + n);
      if (!to_ws && EPI == EPI_EMBED) {
        const half4_t ps = *reinterpret_cast<const half4_t*>(p.pos + (long)m * p.ldc + n);
        const float4_t cs = *reinterpret_cast<const float4_t*>(p.ctx + n);
        v += float4_t{(float)ps[0] + cs[0], (float)ps[1] + cs[1], (float)ps[2] + cs[2], (float)ps[3] + cs[3]};
      }
      if (sc1) store_sc1(rs, ((long)m * ld + n) * 4, v);
      else __builtin_nontemporal_store(v, g);
    }
    return;
  }
  half_t* st = reinterpret_cast<half_t*>(region);
  if ((EPI == EPI_QKV || EPI == EPI_QKV_FRAG) && nw >= p.qk_cols) {
    constexpr int PT = WM + 8;   // halves, transposed rows [n][m]
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int c = j * 32 + (lane & 31);
      const float bv = bcol[j][0];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          half4_t h;
#pragma unroll
          for (int e = 0; e < 4; ++e) h[e] = (half_t)(acc[i][j][4 * g4 + e] + bv);
          *reinterpret_cast<half4_t*>(st + c * PT + i * 32 + 8 * g4 + 4 * (lane >> 5)) = h;
        }
    }
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
    if (EPI == EPI_QKV_FRAG) {
      // V fragment blocks: 16 features x 32 tokens = 64 lanes x 8 tokens, one
      // contiguous KB per block (see the layout note at the epilogue modes)
      // The wave's WN columns lie in one head (head_dim is a power of two >= WN,
      // checked on the host), so the head and the first 16-feature block are
      // wave-uniform and the chunk index is shifts and adds.
      const int r = lane & 15, g = lane >> 4, hs = __builtin_ctz(p.head_dim);
      const int f0 = nw - p.qk_cols, h = f0 >> hs, c0 = f0 & (p.head_dim - 1);
      const long cbase = (long)(h << (hs - 4)) + (c0 >> 4);   // 16-feature block of the wave's first column
      const int tpb = p.M >> 5;                                 // 32-token blocks
#pragma unroll
      for (int blk = 0; blk < (WN / 16) * (WM / 32); ++blk) {
        const int cb = blk % (WN / 16), tb = blk / (WN / 16);
        if (mw + tb * 32 >= p.M) continue;
        // tokens 4g..4g+3 and 16+4g..16+4g+3 of the 32-token block: the key
        // order in which the attention kernel's P.V A operand leaves its softmax
        const int nl = cb * 16 + r, ml = tb * 32 + g * 4;
        const long chunk = ((cbase + cb) * tpb + (mw >> 5) + tb) * 64 + g * 16 + r;
        const half4_t lo = *reinterpret_cast<const half4_t*>(st + nl * PT + ml);
        const half4_t hi = *reinterpret_cast<const half4_t*>(st + nl * PT + ml + 16);
        store_sc1(sc1_rsrc(p.vt, 2L * p.M * (p.N - p.qk_cols)), chunk * 16,
                  half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
      }
      return;
    }
    constexpr int CPR = WM / 8;
#pragma unroll 4
    for (int q = lane; q < WN * CPR; q += 64) {
      const int r = q / CPR, c = (q % CPR) * 8;
      const int n = nw + r, m = mw + c;
      if (n >= p.N || m >= p.M) continue;
      *reinterpret_cast<half8_t*>(p.vt + (long)(n - p.qk_cols) * p.vt_ld + m) =
          *reinterpret_cast<const half8_t*>(st + r * PT + c);
    }
    return;
  }
  constexpr int PH = WN + 8;   // halves
  if constexpr (SWP) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          half4_t hv;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float v = acc[i][j][4 * k + e] + bcol[j][4 * k + e];
            if (EPI == EPI_F16_BIAS_RELU) v = fmaxf(v, 0.f);
            if (EPI == EPI_F16_BIAS_GELU) v = gelu_fast(v);
            hv[e] = (half_t)v;
          }
          *reinterpret_cast<half4_t*>(st + (i * 32 + (lane & 31)) * PH + j * 32 + 8 * k + 4 * (lane >> 5)) = hv;
        }
  } else {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int c = j * 32 + (lane & 31);
      const float bv = bcol[j][0];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          float v = acc[i][j][e] + bv;
          if (EPI == EPI_F16_BIAS_RELU) v = fmaxf(v, 0.f);
          if (EPI == EPI_F16_BIAS_GELU) v = gelu_fast(v);
          st[(i * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3)) * PH + c] = (half_t)v;
        }
    }
  }
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
  if (EPI == EPI_QKV_FRAG) {
    // Q / K fragment blocks: 16 tokens x 32 features = 64 lanes x 8 features
    // Q or K, the head and the first 32-feature block are wave-uniform (the
    // wave's WN columns lie in one head, as for V above).
    const int r = lane & 15, g = lane >> 4, hs = __builtin_ctz(p.head_dim), dh = p.qk_cols >> 1;
    const int which = nw >= dh, f0 = nw - which * dh, h = f0 >> hs, c0 = f0 & (p.head_dim - 1);
    const long hbase = (long)(which * (dh >> hs) + h) * (p.M >> 4);   // 16-token blocks before this head
    const int kpb = p.head_dim >> 5;                                  // 32-feature blocks per head
#pragma unroll
    for (int blk = 0; blk < (WM / 16) * (WN / 32); ++blk) {
      const int tb = blk % (WM / 16), kb = blk / (WM / 16);
      if (mw + tb * 16 >= p.M) continue;
      const int ml = tb * 16 + r, nl = kb * 32 + g * 8;
      const long chunk = ((hbase + (mw >> 4) + tb) * kpb + (c0 >> 5) + kb) * 64 + g * 16 + r;
      store_sc1(sc1_rsrc(p.C, 2L * p.M * p.qk_cols), chunk * 16, *reinterpret_cast<const half8_t*>(st + ml * PH + nl));
    }
    return;
  }
  constexpr int CPR = WN / 8;
  half_t* dst = static_cast<half_t*>(p.C) + bz * p.sC;
  const long span = 2L * ((long)(p.M - 1) * p.ldc + p.N);   // bytes of this batch's output
  const bool sc1 = sc1_ok(span);
  const __amdgpu_buffer_rsrc_t rs = sc1_rsrc(dst, sc1 ? span : 0);
#pragma unroll 4
  for (int q = lane; q < WM * CPR; q += 64) {
    const int r = q / CPR, c = (q % CPR) * 8;
    const int m = mw + r, n = nw + c;
    if (m >= p.M || n >= p.N) continue;
    const half8_t v = *reinterpret_cast<const half8_t*>(st + r * PH + c);
    if (sc1) store_sc1(rs, ((long)m * p.ldc + n) * 2, v);
    else __builtin_nontemporal_store(v, reinterpret_cast<half8_t*>(dst + (long)m * p.ldc + n));
  }
}

// Swizzle of a [K][N] B stage (rows of BN halves): physical 16-byte chunk =
// logical chunk ^ bt_swz(row).  The 64 lanes of one transposed fragment read
// cover rows r0..r0+3 and r0+8..r0+11 (r0 a multiple of 4) x 4 chunks.  Rows of
// 256 bytes (one bank window) or a multiple: the swizzle sends them to 16
// distinct chunks, two lanes' 8 bytes per chunk, the fewest passes 512 bytes
// take.  Rows of 128 bytes: rows of one parity share a half window, and the
// swizzle moves the two pairs of them 32 bytes (a read's piece of a row) apart.
template <int BN>
__device__ __forceinline__ int bt_swz(int row) {
  return BN >= 128 ? ((row & 3) << 2) | ((row >> 3) & 1) : ((row >> 1) & 3) << 1;
}

}  // namespace ck
