// fp32 GEMM on the fp16 matrix cores (gemm_split.hip).
#pragma once

#include "gemm_tile.hpp"

namespace aur {

// One launch of the bm×bn tile (256×256, 256×128, 128×128 or 64×64); `a` as
// for the fp32 kernels, k_chunk a multiple of 32.
void gemm_split_launch(const aurgemm::GemmArgs& a, int bm, int bn, bool a_kcontig, bool b_kcontig, int splits,
                       int batch, hipStream_t st);

}  // namespace aur
