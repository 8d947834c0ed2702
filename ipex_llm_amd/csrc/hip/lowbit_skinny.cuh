// Low-bit weight x bf16/f16 activation product for 17 .. a few hundred rows
// (serving decode batches, speculative verify, short prompts) on gfx950 MFMA.
//
// Between the one-row-tile GEMV (lowbit_gemv5.cuh) and the compute-bound
// prefill GEMM the weight stream still bounds the product (a Llama-3-8B
// gate/up at 48 rows: 62 MB of codes and scales, 13 us at the rate of a large
// copy, beside 11 GFLOP), so the split is made for the stream:
//   * workgroup = NW = 8 (4) waves = 128 (64) output columns x R = MT * 16 rows;
//     wave (cg, kp) owns two 16-column weight tiles (cg) and every second 128-k
//     chunk (kp): codes go global -> registers in MFMA A-fragment order
//     (formats.h), PF chunks of both tiles in flight per wave, and no weight
//     is read twice by a row block;
//   * x is staged through LDS once per workgroup and 256-k step (two buffers,
//     the loads of a step requested two steps ahead), XOR-swizzled in 16-B
//     pieces so the 16 rows of a fragment read fall on distinct banks;
//   * codes stay raw in the A operand (exact in bf16 / f16); the block scale
//     is applied to the f32 block sum.  The offset of the integer formats is
//     one product of the block's x with the constant -offset: it comes out
//     broadcast over the tile's rows, i.e. it IS the accumulator input of the
//     code products (no per-row sums of x in memory, no subtract per value),
//     shared by the wave's two tiles;
//   * split-K over blockIdx.y writes f32 slabs summed by the consumer; row
//     blocks of one column block get ids that share id % 8, so a weight chunk
//     leaves HBM once per XCD.
// MI355X, sym_int4, against the kernel it replaced (every wave read its own x
// rows from L2 for one weight tile): gate/up [28672, 4096] 17 / 48 / 64 rows
// 51 / 111 / 144 -> 21 / 25 / 30 us, down [4096, 14336] 29 / 65 / 84 -> 12 / 15
// / 18, o [4096, 4096] 12 / 28 / 36 -> 6 / 7.5 / 9; fp8_e5m2 gate/up 51 / 108 /
// 142 -> 25 / 27 / 32 (4.8 TB/s at 17 rows).  What bounds it now is a step's
// own chain -- barrier, x fragments from LDS, products, scales, 0.6 to 0.9 us
// with two waves per SIMD -- not the stream: two steps in flight measured
// faster than four (o at 17 rows 5.9 vs 7.6 us, gate/up at 32 20.8 vs 22), and
// 128 registers for twice the waves spilled (gate/up at 32 rows 32 us).
#pragma once
#include <mutex>
#include <type_traits>

#include "../common/quant_block.h"
#include "gemv_args.h"
#include "illm_device.h"
#include "lowbit_raw.h"

namespace illm {

constexpr int SK_KW = 2;                       // waves along K
constexpr int SK_TPW = 2;                      // weight tiles per wave
constexpr int SK_STEP = SK_KW * CHUNK_K;       // k per step

// constant of the offset product: -offset for the formats whose codes carry
// one, 1 for unsigned codes with a block minimum (the plain sum of x)
template <int DK, typename T>
__host__ __device__ constexpr uint32_t skinny_const2() {
  constexpr bool b = std::is_same<T, BF16>::value;
  // bf16 -136 / -128 / 1, f16 -1032 / -1024 / -128 / 1
  return DK == DK_INT4S ? (b ? 0xC308C308u : 0xE408E408u)
       : DK == DK_INT4A ? (b ? 0xC300C300u : 0xE400E400u)
       : DK == DK_INT8S ? (b ? 0xC300C300u : 0xD800D800u)
       : (b ? 0x3F803F80u : 0x3C003C00u);
}

template <int DK, typename T, int MT, int NW>
__global__ void __launch_bounds__(NW * 64, 2) lowbit_skinny_kernel(const GemvArgs a, const int epi) {
  constexpr int BITS = dk_bits(DK);
  constexpr bool HASMIN = dk_has_min(DK);
  constexpr bool OFFS = dk_needx(DK) && DK != DK_INT8A;   // codes carry an offset
  constexpr bool NEEDX = OFFS || HASMIN;       // ... or the block minimum needs the sum of x
  constexpr int R = MT * 16;
  constexpr int SK_TILES = NW / SK_KW * SK_TPW;
  constexpr int PF = 2;                        // steps of weights in flight, and that x is requested ahead
  constexpr int XJ = MT * 8 / NW;              // 16-B pieces of x per thread and step
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  uint16_t* xs = (uint16_t*)smem;                                 // [2][R][SK_STEP]
  uint32_t* lut2 = (uint32_t*)(smem + 2 * R * SK_STEP * 2);       // DK_LUT4 only
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);      // uniform: weight addresses live in SGPRs
  const int g = lane >> 4, r16 = lane & 15;
  const int cg = wave >> 1, kp = wave & 1;

  // block -> (column block, row block): the MB row blocks of a column block share id % 8
  const int NT = (a.N * (epi == EPI_GLU ? 2 : 1) + 15) / 16;
  const int NB = (NT + SK_TILES - 1) / SK_TILES;
  const int MB = (a.M + R - 1) / R;
  int nb = blockIdx.x, mb = 0;
  if (MB > 1) {
    const int grp = blockIdx.x / (8 * MB), rem = blockIdx.x % (8 * MB);
    mb = rem / 8;
    nb = grp * 8 + rem % 8;
    if (nb >= NB) return;
  }
  const int m0 = mb * R;
  const int tile0 = nb * SK_TILES + cg * SK_TPW;

  const int KC = a.KC;
  const int cpk = a.cpk;                                          // chunks per split-K slice (even)
  const int c0 = blockIdx.y * cpk, c1 = min(KC, c0 + cpk);
  const int nstep = (c1 - c0 + SK_KW - 1) / SK_KW;

  if constexpr (DK == DK_LUT4) {
    if (tid < 256) lut2[tid] = pack2<T>(hd_lut4(a.lut_fmt, tid & 15), hd_lut4(a.lut_fmt, tid >> 4));
  }

  // ---- weights: this wave's chunk of a step is c0 + 2 step + kp
  const size_t TB = (size_t)dk_tile_bytes(DK, KC);
  const size_t soff = (size_t)KC * dk_code_chunk(DK), moff = soff + (size_t)16 * KC * 4;
  const uint32_t lq = lane * 16, ls = g * 16;                     // lane's codes; rows 4g..4g+3 of a scale record
  const uint8_t* tb[SK_TPW];
#pragma unroll
  for (int t = 0; t < SK_TPW; t++) tb[t] = a.w + (size_t)min(tile0 + t, NT - 1) * TB;
  struct Chunk {
    uint4 q[SK_TPW][BITS / 4];
    uint4 sc[SK_TPW];
    uint4 mn[HASMIN ? SK_TPW : 1];
  };
  auto load_w = [&](Chunk& ch, int step) {
    const int c = min(c0 + step * SK_KW + kp, c1 - 1);            // clamped: unconditional loads
#pragma unroll
    for (int t = 0; t < SK_TPW; t++) {
      const uint8_t* rec = tb[t] + (size_t)c * dk_code_chunk(DK);
      ch.q[t][0] = *(const uint4*)(rec + lq);
      if constexpr (BITS == 8) ch.q[t][1] = *(const uint4*)(rec + 1024 + lq);
      ch.sc[t] = *(const uint4*)(tb[t] + soff + (size_t)c * 64 + ls);
      if constexpr (HASMIN) ch.mn[t] = *(const uint4*)(tb[t] + moff + (size_t)c * 64 + ls);
    }
  };

  // ---- x: thread -> rows tid / 32 + 16 j, 16-B piece tid % 32 of the step
  const int xr0 = tid >> 5, xc = tid & 31;
  const int kend = min(a.K, c1 * CHUNK_K);
  uint32_t xo[XJ];                                                // byte offset of the row (host: < 4 GB)
#pragma unroll
  for (int j = 0; j < XJ; j++) xo[j] = (uint32_t)min(m0 + xr0 + NW * 2 * j, a.M - 1) * (uint32_t)a.ldx * 2u;
  auto load_x = [&](uint4 (&xr)[XJ], int step) {                  // unconditional (clamped); store_x zeroes past the slice
    const int k = (c0 + step * SK_KW) * CHUNK_K + xc * 8;
    const uint32_t ko = k < a.K ? (uint32_t)k * 2u : 0u;
#pragma unroll
    for (int j = 0; j < XJ; j++) xr[j] = *(const uint4*)((const uint8_t*)a.x + (xo[j] + ko));
  };
  // piece p of row r lives at piece p ^ (r & 15) (within its half of the step)
  auto store_x = [&](const uint4 (&xr)[XJ], int step, int buf) {
    const uint32_t keep = (c0 + step * SK_KW) * CHUNK_K + xc * 8 < kend ? ~0u : 0u;
#pragma unroll
    for (int j = 0; j < XJ; j++)
      *(uint4*)(xs + (size_t)(buf * R + xr0 + NW * 2 * j) * SK_STEP + ((xc & 16) | ((xc ^ (xr0 + NW * 2 * j)) & 15)) * 8) =
          make_uint4(xr[j].x & keep, xr[j].y & keep, xr[j].z & keep, xr[j].w & keep);
  };

  f32x4 acc[SK_TPW][MT];
#pragma unroll
  for (int t = 0; t < SK_TPW; t++)
#pragma unroll
    for (int mt = 0; mt < MT; mt++) acc[t][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t mask_s = a.nib_mask, magic_v = opaque_v(a.nib_magic);
  constexpr uint32_t cst = skinny_const2<DK, T>();
  const uint4 cA = make_uint4(cst, cst, cst, cst);

  auto read_x = [&](uint4 (&B)[2][MT][2], int buf) {
    const uint16_t* xb = xs + (size_t)(buf * R + r16) * SK_STEP + kp * CHUNK_K;
#pragma unroll
    for (int blk = 0; blk < 2; blk++) {
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        const uint16_t* xm = xb + (size_t)mt * 16 * SK_STEP;
        B[blk][mt][0] = *(const uint4*)(xm + (((8 * blk + g) ^ r16) * 8));
        B[blk][mt][1] = *(const uint4*)(xm + (((8 * blk + 4 + g) ^ r16) * 8));
      }
    }
  };
  auto compute = [&](const Chunk& ch, const uint4 (&B)[2][MT][2]) {
#pragma unroll
    for (int blk = 0; blk < 2; blk++) {
      uint4 A[SK_TPW][2];
#pragma unroll
      for (int t = 0; t < SK_TPW; t++)
#pragma unroll
        for (int ss = 0; ss < 2; ss++) {
          if constexpr (BITS == 4) {
            const uint4& q = ch.q[t][0];
            const uint32_t w = blk == 0 ? (ss == 0 ? q.x : q.y) : (ss == 0 ? q.z : q.w);
            A[t][ss] = raw_a4<DK, T>(w, mask_s, magic_v, lut2);
          } else {
            const uint4& q = ch.q[t][blk];
            A[t][ss] = ss == 0 ? raw_a8<DK, T>(q.x, q.y) : raw_a8<DK, T>(q.z, q.w);
          }
        }
      float d[SK_TPW][4], mn[SK_TPW][4];
#pragma unroll
      for (int t = 0; t < SK_TPW; t++) {
        const uint32_t sw[4] = {ch.sc[t].x, ch.sc[t].y, ch.sc[t].z, ch.sc[t].w};
#pragma unroll
        for (int i = 0; i < 4; i++) d[t][i] = f16_to_f32((uint16_t)(sw[i] >> (16 * blk)));
        if constexpr (HASMIN) {
          // times the sum of x: the offset product holds -offset * sum (exact power of two)
          constexpr float f = OFFS ? -1.f / (std::is_same<T, BF16>::value ? 128.f : 1024.f) : 1.f;
          const uint32_t mw[4] = {ch.mn[t].x, ch.mn[t].y, ch.mn[t].z, ch.mn[t].w};
#pragma unroll
          for (int i = 0; i < 4; i++) mn[t][i] = f * f16_to_f32((uint16_t)(mw[i] >> (16 * blk)));
        }
      }
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        const uint4 B0 = B[blk][mt][0], B1 = B[blk][mt][1];
        const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
        f32x4 X = zero;
        if constexpr (NEEDX) {
          X = mfma16<T>(cA, B0, zero);
          X = mfma16<T>(cA, B1, X);
        }
#pragma unroll
        for (int t = 0; t < SK_TPW; t++) {
          f32x4 P = mfma16<T>(A[t][0], B0, OFFS ? X : zero);
          P = mfma16<T>(A[t][1], B1, P);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            acc[t][mt][i] = __builtin_fmaf(d[t][i], P[i], acc[t][mt][i]);
            if constexpr (HASMIN) acc[t][mt][i] = __builtin_fmaf(mn[t][i], X[i], acc[t][mt][i]);
          }
        }
      }
    }
  };

  // ---- main loop.  Step s: stage x of s + 1 (requested PF steps before) into the
  // buffer that step s - 1 read (every wave is past that step's barrier), request
  // x of s + 1 + PF, compute s, request the weights of s + PF, barrier.  Loads
  // retire in order, so the wait for x of s + 1 leaves PF steps of weights in
  // flight (34 KB of 4-bit, 68 KB of 8-bit codes per CU).  Steps run in whole
  // groups of PF with no branch inside (hipcc keeps counted vmcnt waits); past
  // the slice's end they find zeros in the staged x.
  //
  // Two waves per SIMD leave the LDS reads (768 cycles of a 48-row step), the
  // decoding (1040) and the matrix work (1152) mostly one behind the other.  From
  // three row tiles on, a step reads all of its x first and stages the next
  // before its products, so that the decoding runs while LDS answers and no wave
  // waits for its own stores at the barrier, and half of the waves go first:
  // fp8_e5m2 300 rows gate/up [37888, 3584] 139 -> 133 us, down [3584, 18944]
  // 83.8 -> 79.8; sym_int4 48 rows gate/up 24.8 -> 24.3, down 15.4 -> 15.1.  Two
  // row tiles measured slower so (gate/up at 32 rows 18.9 -> 19.6); a barrier per
  // two steps (twice the LDS) gained nothing at any size.  Four-wave groups have no
  // registers left for it (one spilled) and one wave per SIMD to order.
  constexpr bool EARLY = MT >= 3 && NW == 8;
  uint4 xr[PF][XJ];
  Chunk ring[PF];
  load_x(xr[0], 0);
  __builtin_amdgcn_sched_barrier(0);           // (the order in which the loop requests and waits)
#pragma unroll
  for (int u = 0; u < PF; u++) {
    load_w(ring[u], u);
    __builtin_amdgcn_sched_barrier(0);
    if (u + 1 < PF) load_x(xr[u + 1], u + 1);
    __builtin_amdgcn_sched_barrier(0);
  }
  store_x(xr[0], 0, 0);
  load_x(xr[0], PF);
  __syncthreads();
  if (EARLY && wave < NW / 2) __builtin_amdgcn_s_setprio(1);
  for (int s0 = 0; s0 < nstep; s0 += PF) {
#pragma unroll
    for (int u = 0; u < PF; u++) {
      uint4 B[2][MT][2];
      read_x(B, u & 1);
      if constexpr (EARLY) {
        __builtin_amdgcn_sched_barrier(0);
        store_x(xr[(u + 1) % PF], s0 + u + 1, (u + 1) & 1);
        load_x(xr[(u + 1) % PF], s0 + u + 1 + PF);
      }
      compute(ring[u], B);
      __builtin_amdgcn_sched_barrier(0);       // the ring slot is free only after its compute: no second copy of it
      load_w(ring[u], s0 + u + PF);
      if constexpr (!EARLY) {
        __builtin_amdgcn_sched_barrier(0);
        store_x(xr[(u + 1) % PF], s0 + u + 1, (u + 1) & 1);
        load_x(xr[(u + 1) % PF], s0 + u + 1 + PF);
      }
      __syncthreads();
    }
  }

  // ---- the two k-parts through LDS (x is done: the last step's barrier is behind)
  float4* red = (float4*)smem;                                    // [4][SK_TPW][MT][64]
  if (kp == 1) {
#pragma unroll
    for (int t = 0; t < SK_TPW; t++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++)
        red[((cg * SK_TPW + t) * MT + mt) * 64 + lane] =
            make_float4(acc[t][mt][0], acc[t][mt][1], acc[t][mt][2], acc[t][mt][3]);
  }
  __syncthreads();
  if (kp != 0) return;
#pragma unroll
  for (int t = 0; t < SK_TPW; t++)
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      const float4 v = red[((cg * SK_TPW + t) * MT + mt) * 64 + lane];
      acc[t][mt][0] += v.x; acc[t][mt][1] += v.y; acc[t][mt][2] += v.z; acc[t][mt][3] += v.w;
    }

  // ---- epilogue: lane holds columns 16 tile + 4 g + i of row m0 + 16 mt + r16
  if (epi == EPI_GLU) {
    if (tile0 + 1 >= NT) return;                                  // whole gate / up pairs (NT even)
    const int n0 = (tile0 / 2) * 16 + 4 * g;
    if (n0 >= a.N) return;
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      const int m = m0 + mt * 16 + r16;
      if (m >= a.M) continue;
      float o[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float gv = acc[0][mt][i], uv = acc[1][mt][i];
        o[i] = (a.act == 0 ? silu_f(gv) : gelu_tanh_f(gv)) * uv;
      }
      uint16_t* y = (uint16_t*)a.out + (size_t)m * a.ldo + n0;
      if (n0 + 3 < a.N && ((a.ldo | n0) & 3) == 0) *(uint2*)y = make_uint2(pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]));
      else for (int i = 0; i < 4 && n0 + i < a.N; i++) y[i] = from_f32<T>(o[i]);
    }
    return;
  }
#pragma unroll
  for (int t = 0; t < SK_TPW; t++) {
    const int n0 = (tile0 + t) * 16 + 4 * g;
    if (tile0 + t >= NT || n0 >= a.N) continue;
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      const int m = m0 + mt * 16 + r16;
      if (m >= a.M) continue;
      float o[4] = {acc[t][mt][0], acc[t][mt][1], acc[t][mt][2], acc[t][mt][3]};
      if (epi == EPI_PARTIAL) {
        float* ws = (float*)a.out + ((size_t)blockIdx.y * a.M + m) * a.N + n0;
        if (n0 + 3 < a.N && (a.N & 3) == 0) *(float4*)ws = make_float4(o[0], o[1], o[2], o[3]);
        else for (int i = 0; i < 4 && n0 + i < a.N; i++) ws[i] = o[i];
      } else {
        if (a.bias) {
#pragma unroll
          for (int i = 0; i < 4; i++) o[i] += n0 + i < a.N ? to_f32<T>(a.bias[n0 + i]) : 0.f;
        }
        uint16_t* y = (uint16_t*)a.out + (size_t)m * a.ldo + n0;
        if (n0 + 3 < a.N && ((a.ldo | n0) & 3) == 0) *(uint2*)y = make_uint2(pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]));
        else for (int i = 0; i < 4 && n0 + i < a.N; i++) y[i] = from_f32<T>(o[i]);
      }
    }
  }
}

// dynamic LDS of one workgroup; a kernel asking for more than 64 KiB has its
// limit raised first (once per kernel)
inline size_t skinny_shmem(int mt, bool lut) { return (size_t)2 * mt * 16 * SK_STEP * 2 + (lut ? 1024 : 0); }

template <int DK, typename T, int MT, int NW>
void launch_skinny_t(int epi, dim3 grid, const GemvArgs& a, hipStream_t st) {
  const size_t shmem = skinny_shmem(MT, DK == DK_LUT4);
  if (shmem > 64 * 1024) {
    static std::once_flag once;
    std::call_once(once, [&] {
      if (hipFuncSetAttribute((const void*)lowbit_skinny_kernel<DK, T, MT, NW>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem) != hipSuccess)
        (void)hipGetLastError();
    });
  }
  hipLaunchKernelGGL((lowbit_skinny_kernel<DK, T, MT, NW>), grid, dim3(NW * 64), shmem, st, a, epi);
}

// mt: 16-row tiles per workgroup (one workgroup covers every row up to 64); nw: waves (4 or 8)
template <int DK, typename T>
void launch_skinny_mt(int mt, int nw, int epi, dim3 grid, const GemvArgs& a, hipStream_t st) {
  if (nw == 8) {
    if (mt <= 2) launch_skinny_t<DK, T, 2, 8>(epi, grid, a, st);
    else if (mt == 3) launch_skinny_t<DK, T, 3, 8>(epi, grid, a, st);
    else launch_skinny_t<DK, T, 4, 8>(epi, grid, a, st);
  } else {
    if (mt <= 2) launch_skinny_t<DK, T, 2, 4>(epi, grid, a, st);
    else if (mt == 3) launch_skinny_t<DK, T, 3, 4>(epi, grid, a, st);
    else launch_skinny_t<DK, T, 4, 4>(epi, grid, a, st);
  }
}
template <int DK>
void launch_skinny_dk(bool bf16, int mt, int nw, int epi, dim3 grid, const GemvArgs& a0, hipStream_t st) {
  GemvArgs a = a0;
  a.nib_mask = 0x000F000Fu;
  a.nib_magic = bf16 ? Raw<BF16>::k4 : Raw<F16>::k4;
  if (bf16) launch_skinny_mt<DK, BF16>(mt, nw, epi, grid, a, st);
  else launch_skinny_mt<DK, F16>(mt, nw, epi, grid, a, st);
}

}  // namespace illm
