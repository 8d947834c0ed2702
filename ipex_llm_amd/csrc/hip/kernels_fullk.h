// Host interface of the low-bit products that finish their rows (lowbit_fullk.cuh).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace illm {

// what a workgroup does with its 16 columns (FK_ROPE, FK_GLU: twice 16) of x W^T
enum FullkEpi : int {
  FK_NORM = 0,  // h = rnd(rnd(y) + res) -> res_out, rnd(w * h) -> xo, sums of squares of h by 16 columns -> ss
  FK_ROPE = 1,  // y * row scale (+ bias), columns below rcols rotated by the row's position -> out32, or q16 and the cache
  FK_GLU = 2,   // act(gate) * up of tile-interleaved rows, both times the row scale -> xo [M, N / 2]
};

struct FullkArgs {
  const uint16_t* x;       // [M, ldx] activations
  int M, K, ldx;
  const uint8_t* w;        // device blob (formats.h)
  int N, KC;               // rows of the weight, K chunks
  int lut_fmt;             // DK_LUT4: FMT_NF4 / FMT_NF3
  uint16_t* xo;            // FK_NORM [M, N], FK_GLU [M, N / 2]
  // FK_NORM
  const uint16_t* res;     // [M, N]
  uint16_t* res_out;       // [M, N], not res
  const uint16_t* nw;      // [N] norm weight (unit: stored as w - 1)
  int unit;
  float* ss;               // [M, ceil(N / 16)]
  float* zero;             // [M, N] to clear (an accumulator whose readers ran earlier in the stream), or null
  // FK_ROPE, FK_GLU: x is the input of a deferred norm whose rows' sums of squares have xpss_parts parts (0: 1 as scale)
  const float* xpss;
  int xpss_parts, xpss_n;
  float xpss_eps;
  int act;                 // FK_GLU: 0 = silu, 1 = gelu(tanh)
  // FK_ROPE: whole heads of rD (64, 128) columns, N a multiple of rD; cos / sin [max_pos][rD / 2][2]
  float* out32;            // [M, N]
  const uint16_t* bias;    // [N] or null
  const float* rcs;
  const int64_t* rpos;
  int rcols, rD;
  // ... instead of out32 (q16 not null): columns below qcols -> q16 [M, qcols], below rcols -> k_cache, then v_cache
  // [num_blocks, kv heads, bs, rD], the row of key lens[m] - 1; each rounded once
  uint16_t *q16, *k_cache, *v_cache;
  const int32_t *tables, *lens;   // [M, max_blocks], [M]
  int qcols, max_blocks, num_blocks, bs;
  uint32_t nib_mask, nib_magic;
};

template <int DK>
void launch_fullk_dk(bool bf16, int epi, const FullkArgs& a, hipStream_t st);

}  // namespace illm
