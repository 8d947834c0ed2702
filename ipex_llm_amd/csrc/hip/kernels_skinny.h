// Host interface of the low-bit skinny GEMM (lowbit_skinny.cuh).
#pragma once
#include <hip/hip_runtime.h>

#include "gemv_args.h"

namespace illm {

// workgroup = nw waves (4 or 8) = nw weight tiles x 16 mt rows (mt 2 .. 4) x a.cpk chunks; grid =
// (column blocks x row blocks -- several row blocks: padded to groups of 8 column blocks --, slices)
template <int DK>
void launch_skinny_dk(bool bf16, int mt, int nw, int epi, dim3 grid, const GemvArgs& a, hipStream_t st);

}  // namespace illm
