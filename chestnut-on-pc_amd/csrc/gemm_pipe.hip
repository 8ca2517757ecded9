// f16-input / f32-accumulate GEMM for products large enough to keep the matrix
// cores busy: 128x128 and 256x128 tiles with one workgroup per CU, and 64x64
// tiles for products with few of those; B as [N][K] or [K][N]; the K loop
// software-pipelined across its barrier.
//
// What bounds it.  A wave issues in order and an MFMA occupies the matrix core
// for 32 cycles, so every instruction that makes a wave wait between two MFMAs
// idles it.  gemm_dma_kernel (gemm.hip) reads the first two slices of a K-step
// after the step's barrier and waits for all of them before the first MFMA: a
// full LDS round trip per step.  And a 64x64 wave tile reads 4 fragments for 4
// MFMAs, so LDS bandwidth (128 bytes per cycle) is spent as fast as the matrix
// cores work.  Here
//   * the fragments of slice k+1 are read between the MFMAs of slice k, in a
//     second register set, and the last slice of a step runs after the barrier
//     that publishes the next stage, whose first slice it reads meanwhile: the
//     loop has one barrier per step and no exposed LDS latency;
//   * the refill loads (LDS-DMA, global_load_lds_dwordx4) of a stage go out
//     between the same MFMAs, starting right after the barrier that retires its
//     readers;
//   * larger tiles read each fragment for more MFMAs and fetch fewer operand
//     bytes per product (a CU takes about 20-35 bytes per cycle from L2).
// B as [K][N] is staged as it lies ([64][BN] rows) and read transposed
// (ds_read_b64_tr_b16).  The compiler holds such a read back until every
// LDS-DMA load in flight has landed (vmcnt(0)), which serialises the ring; the
// reads of a slice are therefore one asm block that ends with their own wait.
//
// Measured on one card, graph replays, us per launch (TFLOP/s), before = the
// 128x128 LDS-DMA tile with two K-groups.  Warm: two sets of operands, in the
// Infinity Cache where they fit; cold: 700 MB of them in turn.
//                              before        128x128         256x128
//   4096x4096x4096 [N][K] warm 246 (558)     156 (880)       132 (1040)
//                         cold 248 (555)     166 (826)       136 (1008)
//   4096x4096x4096 [K][N] warm 246 (559)     167 (821)       138 (1000)
//                         cold 251 (548)     174 (790)       142 (966)
//   2048x4096x2048 [N][K] warm 58.8 (584)    48.3 (711)      40.2 (855)
//                         cold 59.0          51.0            40.8
//   2048x4096x2048 [K][N] warm 66.1 (520)    50.9 (675)      41.4 (830)
//                         cold 67.9          52.0            41.4
//   512x8192x2048  [N][K] warm 31.2 (551)    26.1 (658)      29.6
//                         cold 29.2          27.8            35.2
//   512x8192x2048  [K][N] warm 34.3 (501)    27.3 (629)      32.6
//                         cold 32.2          27.4            34.7
//   1000x2184x1984 [N][K] warm 26.4 (328)    20.3 (427)      29.7
//                         cold 25.6          24.5            34.0
//   1000x2184x1984 [K][N] warm 32.3 (268)    22.9 (378)      32.7
//                         cold 31.3          26.5            37.0
// (4096x4096x4096, one set of operands for a second: 125 us on normal data, 119 on
// uniform, 88 on zeros; the power they draw sets the clock.)
// A 256x256 tile (8 waves, 113 us for 4096x4096x4096) has no registers for the
// second accumulator of each product that keeps the rounding error at what it was.
#include <type_traits>

#include "common.h"
#include "gemm_common.h"
#include "gemm_pipe.h"
#include "kernels.h"

namespace ck {
namespace {

typedef const __attribute__((address_space(1))) char* gptr_t;
typedef const __attribute__((address_space(3))) char* lrd_t;
typedef __attribute__((address_space(3))) char* lwr_t;

// Wait until at most `later` (<= MAX) whole K-steps of NI loads each are in flight.
template <int MAX, int NI>
__device__ __forceinline__ void wait_steps(int later) {
  if constexpr (MAX <= 0) {
    wait_vm_lgkm0<0>();
  } else {
    if (later >= MAX) wait_vm_lgkm0<MAX * NI>();
    else wait_steps<MAX - 1, NI>(later);
  }
}

// S: LDS ring stages; WGM x WGN: the wave grid over the tile; FRONT: all refill
// loads of a stage in the first two slices after its barrier (else spread over
// four); BT: B is [K][N].
template <int BM, int BN, int S, int WGM, int WGN, bool FRONT, int EPI, bool BT>
__global__ __launch_bounds__(64 * WGM * WGN, BM == 64 && S <= 4 ? 2 : 1) void gemm_pipe_kernel(const GemmParams p) {
  constexpr int NW = WGM * WGN;
  constexpr int STAGE_A = BM * BK * 2, STAGE = (BM + BN) * BK * 2;   // bytes
  constexpr int WM = BM / WGM, WN = BN / WGN, FM = WM / 32, FN = WN / 32, NM = FM * FN;
  constexpr int NIA = BM / (8 * NW), NIB = BN / (8 * NW), NI = NIA + NIB;
  constexpr int KS = BK / 16, NR = FM + FN;
  static_assert(FM * 32 == WM && FN * 32 == WN && NIA * 8 * NW == BM && NIB * 8 * NW == BN, "tile");
  static_assert((S - 1) * NI < 64, "vmcnt range");
  constexpr int REGION = 32 * (WN + 8) * 4;   // staged epilogue, bytes per wave
  static_assert(NW * REGION <= S * STAGE, "LDS ring too small for the staged epilogue");
  __shared__ __attribute__((aligned(1024))) char lds[S * STAGE];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  // ---- block -> tile: each XCD gets a contiguous run of the tile order, whose
  // runs cover GM M-tiles by as many N-tiles as they need ----
  const int per = p.Mt * p.Nt, total = per * p.split * p.batch;
  const int xcd = (int)blockIdx.x & 7, q8 = total >> 3, r8 = total & 7;
  int L = xcd * q8 + min(xcd, r8) + ((int)blockIdx.x >> 3);
  const int z = L / per;
  L -= z * per;
  const int sp = z % p.split, bz = z / p.split;
  constexpr int GM = 4;
  const int g = L / (GM * p.Nt), gm = min(GM, p.Mt - g * GM);
  L -= g * GM * p.Nt;
  const int mt = g * GM + L % gm, nt = L / gm;
  const int m0 = mt * BM, n0 = nt * BN, kbeg = sp * p.kps, nk = p.kps / BK;

  gptr_t ab = (gptr_t)(uintptr_t)(p.A + bz * p.sA + (long)m0 * p.lda + kbeg);
  gptr_t bb = BT ? (gptr_t)(uintptr_t)(p.B + bz * p.sB + (long)kbeg * p.ldb)
                 : (gptr_t)(uintptr_t)(p.B + bz * p.sB + (long)n0 * p.ldb + kbeg);
  const long astep = BK * 2, bstep = BT ? (long)BK * p.ldb * 2 : BK * 2;
  // per-lane byte offsets: physical chunk c of a stage row holds logical chunk c ^ swizzle(row);
  // rows and columns past the edge repeat the last ones (their products are not stored)
  long aoff[NIA], boff[NIB];
#pragma unroll
  for (int i = 0; i < NIA; ++i) {
    const int r = (wave * NIA + i) * 8 + (lane >> 3), q = (lane & 7) ^ ((r >> 1) & 7);
    aoff[i] = (long)min(r, p.M - 1 - m0) * p.lda * 2 + q * 16;
  }
#pragma unroll
  for (int i = 0; i < NIB; ++i) {
    if (BT) {
      constexpr int CH = BN / 8;   // 16-byte chunks per stage row
      const int c = (wave * NIB + i) * 64 + lane, r = c / CH, q = (c % CH) ^ bt_swz<BN>(r);
      boff[i] = (long)r * p.ldb * 2 + min(n0 + q * 8, p.N - 8) * 2;
    } else {
      const int r = (wave * NIB + i) * 8 + (lane >> 3), q = (lane & 7) ^ ((r >> 1) & 7);
      boff[i] = (long)min(r, p.N - 1 - n0) * p.ldb * 2 + q * 16;
    }
  }
  // load instruction i of a K-step: A rows first, then B rows
  auto dma = [&](int i, gptr_t a, gptr_t b, lwr_t st) {
    typedef const __attribute__((address_space(1))) void* src_t;
    if (i < NIA)
      __builtin_amdgcn_global_load_lds((src_t)(a + aoff[i < NIA ? i : 0]), (lds_ptr_t)(st + (wave * NIA + i) * 1024), 16,
                                       0, 0);
    else
      __builtin_amdgcn_global_load_lds((src_t)(b + boff[i >= NIA ? i - NIA : 0]),
                                       (lds_ptr_t)(st + STAGE_A + (wave * NIB + i - NIA) * 1024), 16, 0, 0);
  };

  // NCH accumulators per product, each taking every NCH-th k-slice: a chain of
  // roundings is that much shorter (relative error at K = 4096: one chain 4.1e-7,
  // two 2.9e-7).  The 64x64 tile, whose products leave room for
  // eight, then needs no split of K to be as exact as a split one was.
  constexpr int NCH = NM == 1 ? 8 : 2;
  float16_t acc[NCH][FM][1][FN];
#pragma unroll
  for (int c = 0; c < NCH; ++c)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[c][i][0][j] = float16_t{};

  // the bias of the lane's epilogue columns: older than every DMA, so it has
  // landed by the first wait
  float bcol[FN][16];
  {
    const float* bias = (p.split == 1 && EPI != EPI_PARTIALS && p.bias) ? p.bias + bz * p.sBias : nullptr;
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int n = n0 + wn * WN + j * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
        bcol[j][e] = (bias && n < p.N) ? bias[n] : 0.f;
      }
  }

  // ---- prologue: fill every stage ----
  const lwr_t lw = (lwr_t)lds;
#pragma unroll
  for (int t = 0; t < S; ++t)
    if (t < nk) {
#pragma unroll
      for (int i = 0; i < NI; ++i) dma(i, ab, bb, lw + t * STAGE);
      ab += astep;
      bb += bstep;
    }

  // ---- fragment reads ----
  const lrd_t lr = (lrd_t)lds;
  const unsigned sw = ((lane >> 5) ^ ((lane >> 1) & 7)) << 4;
  const unsigned arow = (wm * WM + (lane & 31)) * 128 + sw;
  const unsigned brow = STAGE_A + (wn * WN + (lane & 31)) * 128 + sw;
  unsigned btoff[FN][2];
  if (BT) {
    const int gq = lane >> 4, a = (lane >> 2) & 3, b = lane & 3;
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = 8 * (gq >> 1) + 4 * h + a;
        const int col = wn * WN + j * 32 + 16 * (gq & 1) + 4 * b;
        btoff[j][h] = STAGE_A + (row * BN + (((col >> 3) ^ bt_swz<BN>(row)) << 3) + (col & 7)) * 2;
      }
  }
  half8_t fa[2][FM], fb[2][FN];
  auto read_one = [&](auto BUF, auto KK, int r, unsigned so) {
    constexpr int bu = decltype(BUF)::value, kk = decltype(KK)::value;
    if (r < FM) {
      fa[bu][r < FM ? r : 0] =
          *(const __attribute__((address_space(3))) half8_t*)(lr + (((arow + so) ^ (kk << 5)) + r * 4096));
    } else {
      const int j = r >= FM ? r - FM : 0;
      fb[bu][j] = *(const __attribute__((address_space(3))) half8_t*)(lr + (((brow + so) ^ (kk << 5)) + j * 4096));
    }
  };
  // The transposed B reads of one slice (BT).  In one asm block with their
  // wait: the compiler would hold each ds_read_b64_tr_b16 back until every
  // LDS-DMA load in flight has landed, as it cannot tell the stages apart.
  auto read_bt = [&](auto BUF, auto KK, unsigned so) {
    constexpr int bu = decltype(BUF)::value, kk = decltype(KK)::value;
    static_assert(!BT || NM == 1 || FN == 2, "transposed reads are written for two column fragments");
    u32x2_t v0, v1, v2, v3;
    asm volatile(
        "ds_read_b64_tr_b16 %0, %4 offset:%8\n\t"
        "ds_read_b64_tr_b16 %1, %5 offset:%8\n\t"
        "ds_read_b64_tr_b16 %2, %6 offset:%8\n\t"
        "ds_read_b64_tr_b16 %3, %7 offset:%8\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(v0), "=&v"(v1), "=&v"(v2), "=&v"(v3)
        : "v"(btoff[0][0] + so), "v"(btoff[0][1] + so), "v"(btoff[FN - 1][0] + so), "v"(btoff[FN - 1][1] + so),
          "n"(kk * 16 * BN * 2));
    fb[bu][0] = __builtin_bit_cast(half8_t, u32x4_t{v0[0], v0[1], v1[0], v1[1]});
    fb[bu][FN - 1] = __builtin_bit_cast(half8_t, u32x4_t{v2[0], v2[1], v3[0], v3[1]});
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;

  // One k-slice: the MFMAs of the fragments in buffer KK & 1, the reads of the
  // next slice (slice RK of the stage at `rso`) and the refill loads [DLO, DHI)
  // of a K-step placed between them.
  auto slice = [&](auto KK, auto RK, bool reads, unsigned rso, bool refill, lwr_t rst, gptr_t ra, gptr_t rb, auto DLO, auto DHI) {
    constexpr int cur = decltype(KK)::value & 1;
    using NX = std::integral_constant<int, 1 - cur>;
    constexpr int dlo = decltype(DLO)::value, ND = decltype(DHI)::value - dlo;
    constexpr int RPM = (NR + NM - 1) / NM;   // reads per MFMA slot
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const int i = m / FN, j = m % FN;
      // operands swapped: the accumulators hold D^T (see store_staged)
      acc[cur][i][0][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[cur][j], fa[cur][i], acc[cur][i][0][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (reads) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if (r / RPM == m && (!BT || r < FM)) read_one(NX{}, RK, r, rso);
        if (BT && m == 0) read_bt(NX{}, RK, rso);
      }
      if (refill) {
#pragma unroll
        for (int d = 0; d < ND; ++d)
          if (d * NM / (ND > 0 ? ND : 1) == m) dma(dlo + d, ra, rb, rst);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  using F = std::false_type;
  using T = std::true_type;
  // stage offsets (bytes) of step t and, for the larger tiles, t - 1
  unsigned so = 0;
  wait_steps<S - 1, NI>(min(S, nk) - 1);   // step 0's loads
  lds_barrier();
  if constexpr (NM == 1) {
    // One product per wave: a slice's MFMA covers a quarter of an LDS round trip,
    // so the fragments of the whole next step are read while this step's MFMAs
    // run, in registers of the other parity.
    half8_t ga[2][KS], gb[2][KS];
    auto read_a = [&](auto BUF, unsigned o) {
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
        ga[decltype(BUF)::value][kk] = *(const __attribute__((address_space(3))) half8_t*)(lr + ((arow + o) ^ (kk << 5)));
    };
    auto read_b = [&](auto BUF, unsigned o) {
      constexpr int bu = decltype(BUF)::value;
      if constexpr (BT) {
        u32x2_t v[2 * KS];
        asm volatile(   // see read_bt
            "ds_read_b64_tr_b16 %0, %8\n\t"
            "ds_read_b64_tr_b16 %1, %9\n\t"
            "ds_read_b64_tr_b16 %2, %8 offset:%10\n\t"
            "ds_read_b64_tr_b16 %3, %9 offset:%10\n\t"
            "ds_read_b64_tr_b16 %4, %8 offset:%11\n\t"
            "ds_read_b64_tr_b16 %5, %9 offset:%11\n\t"
            "ds_read_b64_tr_b16 %6, %8 offset:%12\n\t"
            "ds_read_b64_tr_b16 %7, %9 offset:%12\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
            : "v"(btoff[0][0] + o), "v"(btoff[0][1] + o), "n"(16 * BN * 2), "n"(32 * BN * 2), "n"(48 * BN * 2));
#pragma unroll
        for (int kk = 0; kk < KS; ++kk)
          gb[bu][kk] = __builtin_bit_cast(half8_t, u32x4_t{v[2 * kk][0], v[2 * kk][1], v[2 * kk + 1][0], v[2 * kk + 1][1]});
      } else {
#pragma unroll
        for (int kk = 0; kk < KS; ++kk)
          gb[bu][kk] = *(const __attribute__((address_space(3))) half8_t*)(lr + ((brow + o) ^ (kk << 5)));
      }
    };
    read_a(I0{}, 0u);
    read_b(I0{}, 0u);
    // ab, bb point at step t + S
    auto step = [&](auto MAIN, auto PAR, int t) {
      constexpr bool main = decltype(MAIN)::value;
      constexpr int par = decltype(PAR)::value;
      using NX = std::integral_constant<int, 1 - par>;
      const bool ref = main || t + S < nk, more = main || t + 1 < nk;
      const unsigned son = so + STAGE == S * STAGE ? 0u : so + STAGE;
      if (more) {
        // step t + 1 has landed, and this wave's reads of stage t have
        if (main) wait_vm_lgkm0<(S - 2) * NI>();
        else wait_steps<S - 2, NI>(min(S - 2, nk - 2 - t));
        lds_barrier();
        read_a(NX{}, son);
        if (!BT) read_b(NX{}, son);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) {
        acc[4 * par + kk][0][0][0] =
            __builtin_amdgcn_mfma_f32_32x32x16_f16(gb[par][kk], ga[par][kk], acc[4 * par + kk][0][0][0], 0, 0, 0);
        if (ref) {
#pragma unroll
          for (int i = kk * NI / KS; i < (kk + 1) * NI / KS; ++i) dma(i, ab, bb, lw + so);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (ref) {
        ab += astep;
        bb += bstep;
      }
      if (BT && more) read_b(NX{}, son);
      so = son;
    };
    int t = 0;
    for (; t + 1 + S < nk; t += 2) {
      step(T{}, I0{}, t);
      step(T{}, I1{}, t + 1);
    }
    for (; t < nk; t += 2) {
      step(F{}, I0{}, t);
      if (t + 1 < nk) step(F{}, I1{}, t + 1);
    }
  } else {
    unsigned sop = 0;
#pragma unroll
    for (int r = 0; r < (BT ? FM : NR); ++r) read_one(I0{}, I0{}, r, 0u);
    if (BT) read_bt(I0{}, I0{}, 0u);

    // ab, bb point at the step whose refill is being issued: step t-1+S in slices 0..2 of step t
    // (its first quarter went out in slice 3 of step t-1), step t+S in slice 3
    // refill loads issued by the end of slices 3, 0 and 1 (slice 2 issues the rest)
    constexpr int E3 = FRONT ? NI / 2 : NI / 4, E0 = FRONT ? NI : NI / 2, E1 = FRONT ? NI : NI * 3 / 4;
    using D0 = std::integral_constant<int, 0>;
    using D1 = std::integral_constant<int, E3>;
    using D2 = std::integral_constant<int, E0>;
    using D3 = std::integral_constant<int, E1>;
    using D4 = std::integral_constant<int, NI>;
    auto step = [&](auto MAIN, int t) {
      constexpr bool main = decltype(MAIN)::value;
      const bool refp = main || (t >= 1 && t - 1 + S < nk), ref = main || t + S < nk, more = main || t + 1 < nk;
      const unsigned son = so + STAGE == S * STAGE ? 0u : so + STAGE;
      slice(I0{}, I1{}, true, so, refp, lw + sop, ab, bb, D1{}, D2{});
      slice(I1{}, I2{}, true, so, refp, lw + sop, ab, bb, D2{}, D3{});
      slice(I2{}, I3{}, true, so, refp, lw + sop, ab, bb, D3{}, D4{});
      if (refp) {
        ab += astep;
        bb += bstep;
      }
      if (more) {
        if (main) wait_vm_lgkm0<(S - 2) * NI>();
        else wait_steps<S - 2, NI>(min(S - 2, nk - 2 - t));
        lds_barrier();
      }
      slice(I3{}, I0{}, more, son, ref, lw + so, ab, bb, D0{}, D1{});
      sop = so;
      so = son;
    };
    int t = 1;
    step(F{}, 0);
    for (; t + S < nk; ++t) step(T{}, t);
    for (; t < nk; ++t) step(F{}, t);
  }

  // the chains' sum of product (i, j), by halves
  auto chain_sum = [&](int i, int j) {
    // (keeps the sums of later products behind this one's stores: all at once
    // they do not fit the registers of the larger tiles)
    if constexpr (NM > 1) asm volatile("" : "+a"(acc[1][i][0][j])::"memory");
#pragma unroll
    for (int w = 1; w < NCH; w *= 2)
#pragma unroll
      for (int c = 0; c + w < NCH; c += 2 * w) acc[c][i][0][j] += acc[c + w][i][0][j];
  };
  if (!p.vec) {   // shapes or addresses the 16-byte stores do not fit
    const bool to_ws = p.split > 1 || EPI == EPI_PARTIALS;
    float* ws = p.ws + ((long)sp * p.batch + bz) * (long)p.M * p.N;
    void* C = (EPI == EPI_F32 || EPI == EPI_F32_RESID || EPI == EPI_EMBED)
                  ? static_cast<void*>(static_cast<float*>(p.C) + bz * p.sC)
                  : static_cast<void*>(static_cast<half_t*>(p.C) + bz * p.sC);
    const float* bias = p.bias ? p.bias + bz * p.sBias : nullptr;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        chain_sum(i, j);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int m = m0 + wm * WM + i * 32 + (lane & 31);
          const int n = n0 + wn * WN + j * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
          if (m >= p.M || n >= p.N) continue;
          const float v = acc[0][i][0][j][e];
          if (to_ws) ws[(long)m * p.N + n] = v;
          else epi_store<EPI>(p, C, bias, m, n, v);
        }
      }
    return;
  }
  // ---- staged epilogue: 32 rows of the wave's sub-tile at a time through LDS,
  // once every wave is past its last fragment read ----
  wait_vm_lgkm0<0>();
  lds_barrier();
#pragma unroll
  for (int i = 0; i < FM; ++i) {
#pragma unroll
    for (int j = 0; j < FN; ++j) chain_sum(i, j);
    store_staged<32, WN, 1, FN, EPI, true, 16>(p, acc[0][i], bcol, lds + wave * REGION, m0 + wm * WM + i * 32, n0 + wn * WN,
                                               sp, bz, lane);
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
  }
}

template <int BM, int BN, int S, int WGM, int WGN, bool FRONT, int EPI>
void launch_t(bool b_kn, const GemmParams& p, hipStream_t s) {
  const dim3 grid(p.Mt * p.Nt * p.split * p.batch), block(64 * WGM * WGN);
  if constexpr (EPI == EPI_F32) {
    if (b_kn) {
      CK_LAUNCH((gemm_pipe_kernel<BM, BN, S, WGM, WGN, FRONT, EPI, true>), grid, block, 0, s, p);
      CK_LAUNCHED("gemm_pipe");
      return;
    }
  }
  CK_REQUIRE(!b_kn, "gemm: [K][N] B supports the f32 epilogue only");
  CK_LAUNCH((gemm_pipe_kernel<BM, BN, S, WGM, WGN, FRONT, EPI, false>), grid, block, 0, s, p);
  CK_LAUNCHED("gemm_pipe");
}

template <int EPI>
void launch_e(int bm, int bn, bool b_kn, const GemmParams& p, hipStream_t s) {
  if (bm == 256 && bn == 128) launch_t<256, 128, 3, 2, 2, true, EPI>(b_kn, p, s);
  else if (bm == 128 && bn == 128) launch_t<128, 128, 4, 2, 2, false, EPI>(b_kn, p, s);
  else if (bm == 64 && bn == 64 && p.Mt * p.Nt * p.split * p.batch <= 256) launch_t<64, 64, 8, 2, 2, false, EPI>(b_kn, p, s);
  else if (bm == 64 && bn == 64) launch_t<64, 64, 4, 2, 2, false, EPI>(b_kn, p, s);
  else throw Error("gemm: no pipelined kernel for this tile");
}

}  // namespace

void launch_gemm_pipe(int bm, int bn, bool b_kn, int epi, const GemmParams& p, hipStream_t s) {
  switch (epi) {
    case EPI_F32: launch_e<EPI_F32>(bm, bn, b_kn, p, s); break;
    case EPI_F16_BIAS: launch_e<EPI_F16_BIAS>(bm, bn, b_kn, p, s); break;
    case EPI_F16_BIAS_RELU: launch_e<EPI_F16_BIAS_RELU>(bm, bn, b_kn, p, s); break;
    case EPI_F16_BIAS_GELU: launch_e<EPI_F16_BIAS_GELU>(bm, bn, b_kn, p, s); break;
    case EPI_F32_RESID: launch_e<EPI_F32_RESID>(bm, bn, b_kn, p, s); break;
    case EPI_EMBED: launch_e<EPI_EMBED>(bm, bn, b_kn, p, s); break;
    case EPI_PARTIALS: launch_e<EPI_PARTIALS>(bm, bn, b_kn, p, s); break;
    default: throw Error("gemm: unknown epilogue");
  }
}

}  // namespace ck
