// Launchers of the pipelined GEMM kernels (gemm_pipe.hip) and of the one for few
// tiles and a long K (gemm_small.hip).
#pragma once

#include "gemm_common.h"

namespace ck {

// C = A B^T (or A B with b_kn, f32 output only) on BM x BN tiles (p.Mt, p.Nt):
// 128x128, 256x128 or 64x64.  Every epilogue but the QKV ones.
void launch_gemm_pipe(int bm, int bn, bool b_kn, int epi, const GemmParams& p, hipStream_t s);

// C = A B^T on 32x32 tiles, K over the four waves; p.split 1, the f32, f16 and
// residual epilogues.
void launch_gemm_small(int epi, const GemmParams& p, hipStream_t s);

}  // namespace ck
