// Launch of the small-tile GEMM kernels (gemm_pipe.hip) for lz_gemm.
#pragma once
#include "gemm_tiles.h"

// g as lz_gemm sets it up; bm x bn: 128x128, 64x128 or 64x64.  Any K that the
// layouts allow; operand spans as dma_span_fits; both operands K-major, B
// N-major, or both M/N-major.
int lz_gemm_pipe(const GemmArgs& g, bool f16, bool ak, bool bk, int bm, int bn, int splits, hipStream_t s);
