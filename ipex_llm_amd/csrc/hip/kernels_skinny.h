// Host interface of the low-bit skinny GEMM (lowbit_skinny.cuh) and its small companion (lowbit_narrow.cuh).
#pragma once
#include <hip/hip_runtime.h>

#include "../common/formats.h"
#include "gemv_args.h"

namespace illm {

constexpr int SK_KW = 2;                       // waves along K
constexpr int SK_TPW = 2;                      // weight tiles per wave
constexpr int SK_STEP = SK_KW * CHUNK_K;       // k per step
// dynamic LDS of a workgroup: x of three steps, the table and, of one row tile, the rows' scales (bytes)
constexpr size_t skinny_shmem(int mt, int table) { return (size_t)3 * mt * 16 * SK_STEP * 2 + table + (mt == 1 ? 64 : 0); }
constexpr int skinny_table(bool lut, bool fine) { return !lut ? 0 : fine ? 2048 : 1024; }

// workgroup = nw waves (4 or 8) = nw weight tiles x 16 mt rows (mt 1 .. 4) x a.cpk chunks; grid =
// (column blocks x row blocks -- several row blocks: padded to groups of 8 column blocks or not at all --, slices)
// fine: table formats under bf16 x keep their table as bf16 pairs hi + lo (mt 3, 4)
template <int DK>
void launch_skinny_dk(bool bf16, int mt, int nw, int epi, dim3 grid, const GemvArgs& a, hipStream_t st, bool fine);

// workgroup = 4 waves = one weight tile (GLU: a gate / up pair) x all of a.M <= 64 rows (GLU: 32); grid = (tiles or pairs, slices)
template <int DK>
void launch_narrow_dk(bool bf16, int epi, dim3 grid, const GemvArgs& a, hipStream_t st);

}  // namespace illm
