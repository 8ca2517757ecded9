// Launcher of the pipelined GEMM kernels (gemm_pipe.hip).
#pragma once

#include "gemm_common.h"

namespace ck {

// C = A B^T (or A B with b_kn, f32 output only) on BM x BN tiles (p.Mt, p.Nt):
// 128x128, 256x128 or 64x64.  Every epilogue but the QKV ones.
void launch_gemm_pipe(int bm, int bn, bool b_kn, int epi, const GemmParams& p, hipStream_t s);

}  // namespace ck
