// f16 GEMM for few output tiles and a long K ([N][K] B): 32x32 tiles, K over the
// four waves of a workgroup (tile code 17).
//
// What bounds such a product is the operand stream of one CU: it keeps some 60
// cache lines in flight, so a 64x64 tile's 16 KB per 64-wide K-step take 0.2 to
// 0.3 us however deep the LDS ring is, and only more CUs help.  Splitting K over
// workgroups costs a reduce launch (3.4 us, and 4 us of host time).  Here the
// tile shrinks to 32x32 -- four times the workgroups, half the bytes per step --
// and wave w multiplies k-slice w of every K-step into accumulators of its own;
// the waves' sums meet in LDS at the end.  Every wave keeps four accumulators in
// turn, so an element is summed in sixteen chains: no less exact than a split in
// eight on two K-groups.
#include <type_traits>

#include "common.h"
#include "gemm_common.h"
#include "gemm_pipe.h"
#include "kernels.h"

namespace ck {
namespace {

typedef const __attribute__((address_space(1))) char* gptr_t;
typedef const __attribute__((address_space(1))) void* src_t;
typedef const __attribute__((address_space(3))) char* lrd_t;
typedef __attribute__((address_space(3))) char* lwr_t;

constexpr int SM_T = 32;                     // tile rows and columns
constexpr int SM_STAGE = 2 * SM_T * BK * 2;  // bytes of a K-step's A and B rows
constexpr int SM_S = 8;                      // ring stages: 64 KB, two workgroups per CU
constexpr int SM_PITCH = SM_T + 4;           // floats, the waves' sums

template <int MAX>
__device__ __forceinline__ void wait_later(int later) {   // 2 loads per wave and step
  if constexpr (MAX <= 0) {
    wait_vm_lgkm0<0>();
  } else {
    if (later >= MAX) wait_vm_lgkm0<2 * MAX>();
    else wait_later<MAX - 1>(later);
  }
}

template <int EPI>
__global__ __launch_bounds__(256, 2) void gemm_small_kernel(const GemmParams p) {
  constexpr int S = SM_S, STAGE = SM_STAGE;
  __shared__ __attribute__((aligned(1024))) char lds[S * STAGE];
  static_assert(4 * SM_T * SM_PITCH * 4 <= S * STAGE, "LDS ring too small for the waves' sums");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // each XCD gets a contiguous run of tiles, M fastest: the tiles that share
  // weight rows share its L2
  const int total = p.Mt * p.Nt * p.batch;
  const int xcd = (int)blockIdx.x & 7, q8 = total >> 3, r8 = total & 7;
  int L = xcd * q8 + min(xcd, r8) + ((int)blockIdx.x >> 3);
  const int mt = L % p.Mt; L /= p.Mt;
  const int nt = L % p.Nt, bz = L / p.Nt;
  const int m0 = mt * SM_T, n0 = nt * SM_T, nk = p.K / BK;

  // load instruction i (0: A, 1: B) of the wave: rows 8 wave .. +7 of the 32,
  // chunk c of a row at physical chunk c ^ ((row >> 1) & 7)
  gptr_t ab = (gptr_t)(uintptr_t)(p.A + bz * p.sA + (long)m0 * p.lda);
  gptr_t bb = (gptr_t)(uintptr_t)(p.B + bz * p.sB + (long)n0 * p.ldb);
  const int lr8 = wave * 8 + (lane >> 3), lq = ((lane & 7) ^ ((lr8 >> 1) & 7)) * 16;
  const long aoff = (long)min(lr8, p.M - 1 - m0) * p.lda * 2 + lq;
  const long boff = (long)min(lr8, p.N - 1 - n0) * p.ldb * 2 + lq;
  const lwr_t lw = (lwr_t)lds + wave * 1024;
  auto dma = [&](unsigned so) {
    __builtin_amdgcn_global_load_lds((src_t)(ab + aoff), (lds_ptr_t)(lw + so), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((src_t)(bb + boff), (lds_ptr_t)(lw + so + STAGE / 2), 16, 0, 0);
    ab += BK * 2;
    bb += BK * 2;
  };
#pragma unroll
  for (int t = 0; t < S; ++t)
    if (t < nk) dma(t * STAGE);

  // slice `wave` of a stage: row lane % 32, k 8 (lane / 32) .. +7 of the slice
  const lrd_t lr = (lrd_t)lds;
  const unsigned foff = (lane & 31) * 128 + (((wave * 2 + (lane >> 5)) ^ ((lane >> 1) & 7)) << 4);
  half8_t fa[2], fb[2];
  auto read = [&](auto BUF, unsigned so) {
    constexpr int bu = decltype(BUF)::value;
    fa[bu] = *(const __attribute__((address_space(3))) half8_t*)(lr + (foff + so));
    fb[bu] = *(const __attribute__((address_space(3))) half8_t*)(lr + (foff + so + STAGE / 2));
  };
  float16_t acc[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) acc[c] = float16_t{};

  unsigned so = 0;   // stage of step t
  wait_later<S - 1>(min(S, nk) - 1);
  lds_barrier();
  read(std::integral_constant<int, 0>{}, 0u);
  auto step = [&](auto MAIN, auto CH, int t) {
    constexpr bool main = decltype(MAIN)::value;
    constexpr int ch = decltype(CH)::value, cur = ch & 1;
    const unsigned son = so + STAGE == S * STAGE ? 0u : so + STAGE;
    if (main || t + 1 < nk) {
      // step t + 1 has landed and this wave has read its part of stage t
      if (main) wait_vm_lgkm0<2 * (S - 2)>();
      else wait_later<S - 2>(min(S - 2, nk - 2 - t));
      lds_barrier();
      read(std::integral_constant<int, 1 - cur>{}, son);
    }
    if (main || t + S < nk) dma(so);
    acc[ch] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[cur], fa[cur], acc[ch], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    so = son;
  };
  using F = std::false_type;
  using T = std::true_type;
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  using C2 = std::integral_constant<int, 2>;
  using C3 = std::integral_constant<int, 3>;
  int t = 0;
  for (; t + 3 + S < nk; t += 4) {
    step(T{}, C0{}, t);
    step(T{}, C1{}, t + 1);
    step(T{}, C2{}, t + 2);
    step(T{}, C3{}, t + 3);
  }
  for (; t < nk; t += 4) {
    step(F{}, C0{}, t);
    if (t + 1 < nk) step(F{}, C1{}, t + 1);
    if (t + 2 < nk) step(F{}, C2{}, t + 2);
    if (t + 3 < nk) step(F{}, C3{}, t + 3);
  }

  // ---- the waves' sums through LDS (operands swapped: lane holds row lane % 32,
  // columns 8k + 4 (lane / 32) .. +3), then one 4-column chunk per thread ----
  wait_vm_lgkm0<0>();
  lds_barrier();
  float* st = reinterpret_cast<float*>(lds);
  const float16_t w = (acc[0] + acc[1]) + (acc[2] + acc[3]);
#pragma unroll
  for (int k = 0; k < 4; ++k)
    *reinterpret_cast<float4_t*>(st + (wave * SM_T + (lane & 31)) * SM_PITCH + 8 * k + 4 * (lane >> 5)) =
        float4_t{w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]};
  wait_vm_lgkm0<0>();
  lds_barrier();
  const int r = tid >> 3, c = (tid & 7) * 4, m = m0 + r, n = n0 + c;
  if (m >= p.M || n >= p.N) return;
  float4_t q[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) q[i] = *reinterpret_cast<const float4_t*>(st + (i * SM_T + r) * SM_PITCH + c);
  const float4_t s = (q[0] + q[1]) + (q[2] + q[3]);
  const float v[4] = {s[0], s[1], s[2], s[3]};
  store_reduced<EPI>(p, bz, m, n, v, min(4, p.N - n), (p.N & 3) == 0);
}

template <int EPI>
void launch_s(const GemmParams& p, hipStream_t s) {
  CK_LAUNCH(gemm_small_kernel<EPI>, dim3(p.Mt * p.Nt * p.batch), dim3(256), 0, s, p);
  CK_LAUNCHED("gemm_small");
}

}  // namespace

void launch_gemm_small(int epi, const GemmParams& p, hipStream_t s) {
  CK_REQUIRE(p.split == 1, "gemm: tile 17 (32x32) does not split K");
  switch (epi) {
    case EPI_F32: launch_s<EPI_F32>(p, s); break;
    case EPI_F16_BIAS: launch_s<EPI_F16_BIAS>(p, s); break;
    case EPI_F16_BIAS_RELU: launch_s<EPI_F16_BIAS_RELU>(p, s); break;
    case EPI_F16_BIAS_GELU: launch_s<EPI_F16_BIAS_GELU>(p, s); break;
    case EPI_F32_RESID: launch_s<EPI_F32_RESID>(p, s); break;
    default: throw Error("gemm: tile 17 (32x32) has the f32, f16 and residual epilogues");
  }
}

}  // namespace ck
