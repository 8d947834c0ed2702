// Low-bit weight x bf16/f16 activations of 1 to 16 rows in launches that finish their rows (a decode step's projections) on
// gfx950 MFMA: o and down with the residual add and the deferred RMSNorm behind them, qkv with bias and rotation, gate/up
// with the activation.  One workgroup finishes 16 output columns (qkv: the two halves of 16 columns of a head; gate/up: a
// pair of tiles).
//
// A projection of 9 to 70 MB at few rows is bound by its chain of latencies, not by its bytes: launch, x from L2, weights,
// sum over K, and -- where K is cut over workgroups -- f32 atomics, a ticket and the sums read back before the row can be
// finished, 3 to 5 us of a 5 us product.  So K is not cut over workgroups:
//   * a workgroup's 8 (16) waves take an eighth (a 16th) of K each and meet once, in LDS; every wave stages its own x (a
//     piece = 4 chunks of 128 k; 2 from 9 rows on) in an LDS region of its own, so nothing waits for another wave before the
//     end, and requests its weights before it needs x: all of them where K is one piece a wave (to K = 4096), two pieces
//     ahead else.
//     A request out of range is not free (its turn in the address unit, 1 us over the 24 of a wave of K = 4096 whose ring
//     was 16 chunks deep), hence the exact ends;
//   * x is the A operand, raw codes the B operand, and the offset a product of x with a constant (lowbit_skinny.cuh), shared
//     by the workgroup's tiles: one scale per lane, one dword load for the four chunks of a piece;
//   * the rows' sums of squares go out as one number per tile, which the consumer's waves add (RowParts): no atomics, the
//     same bits each time.
// Alone, weights that no cache holds, us at 1 / 3 / 8 / 16 rows, split-K with atomics and the last group finishing the rows
// / this: sym_int4 [4096, 4096] 7.9 8.0 8.9 12.0 / 4.6 4.6 4.8 5.7, asym_int4 8.9 9.2 10.5 13.6 / 4.7 4.8 5.2 6.1, fp8_e5m2
// [3584, 3584] 9.2 9.4 10.3 12.7 / 4.6 4.8 5.2 6.3 (the split-K product without its rows 6.6 6.8 7.3 8.3).  A long K is
// bound by x, which every workgroup reads in full (sym_int4 [4096, 14336] 8.8 / 10.1 / 11.9 / 13.2, of 58 MB of x at 8 rows;
// the rules row_norm_takes, row_norm_o_takes, row_rope_takes and glu_rows_takes of csrc/torch/ops_hip.cpp, with qkv's and
// gate/up's figures).
// qkv that hands q on as the attention takes it and stores k and v in the cache (gemv_rope_kv): f32 sums / this, [6144, 4096]
// sym_int4 5.4 6.05 6.3 8.1 / 5.6 6.2 6.4 8.3 at 1 / 5 / 8 / 16 rows (with integer divisions for the addresses 6.1 7.0 7.1 8.4),
// for 0.5 to 1.5 us less of the attention: a step of 1 / 8 rows Llama-3-8B 1.018x / 1.011x of the tree without it and the shifts,
// 5 rows Qwen2.5-7B fp8_e5m2 1.013x.
// 16 waves of a K that 8 hold in one piece, or pieces four ahead, were slower.  A decode step, us: Llama-3-8B sym_int4,
// 1024 tokens, 1 / 4 / 8 rows 1572 1844 1981, with o and down here 1499 1635 1809, and qkv 1473 1599 1774, and gate/up 1379
// 1551 1769; Qwen2.5-7B fp8_e5m2, 1 / 5 rows 2149 2372, 1995 2182, 1887 2014, 1704 1886.
#pragma once
#include <mutex>
#include <type_traits>

#include "../common/quant_block.h"
#include "gemv_args.h"
#include "illm_device.h"
#include "kernels_fullk.h"
#include "lowbit_raw.h"

namespace illm {

// k-chunks staged at a time, LDS bytes of a staged row (+ 16: the 16 rows of a fragment read fall on distinct banks)
__host__ __device__ constexpr int fullk_pc(int mr) { return mr <= 8 ? 4 : 2; }
__host__ __device__ constexpr int fullk_row(int mr) { return fullk_pc(mr) * CHUNK_K * 2 + 16; }
// staged x of every wave, the waves' sums, the pair table
constexpr int FULLK_NW = 8;                                       // waves of a workgroup, each an eighth of K
constexpr int fullk_tiles(int epi) { return epi == FK_NORM ? 1 : 2; }
__host__ __device__ constexpr size_t fullk_shmem(int mr, int nw, int tiles, bool lut) {
  return (size_t)nw * mr * fullk_row(mr) + (size_t)tiles * nw * mr * 16 * 4 + (lut ? 1024 : 0);
}

// MR: rows of the instantiation (1, 2, 4, 8, 16), a.M <= MR; RG: pieces of weights in flight, no more than a wave has; NW:
// waves
template <int DK, typename T, int MR, int RG, int EPI, int NW = FULLK_NW>
__global__ void __launch_bounds__(NW * 64) lowbit_fullk_kernel(const FullkArgs a) {
  using C = typename std::conditional<DK == DK_LUT4, F16, T>::type;   // product type: table formats keep an f16 table
  constexpr int BITS = dk_bits(DK);
  constexpr bool HASMIN = dk_has_min(DK);
  constexpr bool OFFS = dk_needx(DK) && DK != DK_INT8A;           // codes carry an offset
  constexpr bool NEEDX = OFFS || HASMIN;
  constexpr int PC = fullk_pc(MR), ROW = fullk_row(MR);
  constexpr int XL = MR * PC / 4;                                 // 1-KB loads of a piece of x (PC chunks of MR rows)
  constexpr int QL = BITS / 4, NT = fullk_tiles(EPI);
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  uint8_t* xs = smem + (size_t)wave * MR * ROW;                   // this wave's alone: no barrier before the sums
  float* red = (float*)(smem + (size_t)NW * MR * ROW);            // [NT][NW][MR][16]
  uint32_t* lut2 = (uint32_t*)(red + NT * NW * MR * 16);

  // FK_ROPE: heads of 64 or 128 columns, shifts instead of divisions (an integer division is 0.1 us of the launch's chain
  // wherever it stands); tiles of a head's half
  const int dsh = EPI == FK_ROPE && a.rD == 128 ? 7 : 6, ht = EPI == FK_ROPE ? 1 << (dsh - 5) : 1;
  const int KC = a.KC;
  const int tile0 = EPI == FK_NORM ? blockIdx.x : EPI == FK_GLU ? 2 * blockIdx.x : (blockIdx.x >> (dsh - 5) << (dsh - 4)) + (blockIdx.x & (ht - 1));
  const int c0 = (int)((uint32_t)wave * KC / NW), c1 = (int)((uint32_t)(wave + 1) * KC / NW);

  // x: piece p of the wave is chunks c0 + PC p ..; rows past M and k past K or the wave's range: out of the descriptor, 0
  const __amdgpu_buffer_rsrc_t xd =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.x, 0, (int)((uint32_t)a.M * (uint32_t)a.ldx * 2u), 0x00020000);
  constexpr int LR = PC == 4 ? 1 : 2;                             // rows of a load
  const int xk = PC == 4 ? lane * 8 : (lane & 31) * 8, xrow = PC == 4 ? 0 : lane >> 5;
  const int kend = min(a.K, c1 * CHUNK_K);
  auto load_x = [&](uint4 (&v)[XL], int p) {
    const int k = (c0 + PC * p) * CHUNK_K + xk;
#pragma unroll
    for (int i = 0; i < XL; i++) {
      const int m = i * LR + xrow;
      v[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
          xd, m < a.M && k < kend ? ((uint32_t)m * (uint32_t)a.ldx + (uint32_t)k) * 2u : ~0u, 0, 0));
    }
  };
  auto store_x = [&](const uint4 (&v)[XL]) {
#pragma unroll
    for (int i = 0; i < XL; i++) {
      uint4 w = v[i];
      if constexpr (!std::is_same<C, T>::value) {                 // bf16 activations under an f16 table
        uint32_t* p = &w.x;
#pragma unroll
        for (int j = 0; j < 4; j++)
          p[j] = pack2<F16>(fminf(fmaxf(bf16_to_f32(p[j] & 0xffff), -65504.f), 65504.f),
                            fminf(fmaxf(bf16_to_f32(p[j] >> 16), -65504.f), 65504.f));
      }
      *(uint4*)(xs + (i * LR + xrow) * ROW + xk * 2) = w;
    }
  };

  // weights: two pieces in flight
  const size_t TB = (size_t)dk_tile_bytes(DK, KC);
  __amdgpu_buffer_rsrc_t wd[NT];
#pragma unroll
  for (int t = 0; t < NT; t++)
    wd[t] = __builtin_amdgcn_make_buffer_rsrc((void*)(a.w + (size_t)(tile0 + t * ht) * TB), 0, (int)TB, 0x00020000);
  const uint32_t soff = (uint32_t)KC * dk_code_chunk(DK), moff = soff + 16u * (uint32_t)KC * 4u;
  struct Piece {
    uint4 q[PC][NT][QL];
    uint32_t sc[NT], mn[NT];                                      // chunk c + lane / 16, column lane % 16
  };
  const int cl = g & (PC - 1);
  auto load_w1 = [&](Piece& w, int c, int i) {                    // (past the wave's range: zeros)
    const uint32_t cb = (uint32_t)(c + i) * dk_code_chunk(DK) + (uint32_t)lane * 16u;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int j = 0; j < QL; j++)
        w.q[i][t][j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(wd[t], c + i < c1 ? cb + j * 1024u : ~0u, 0, 2));
  };
  auto load_sc = [&](Piece& w, int c) {
    const uint32_t cs = c + cl < c1 ? soff + (uint32_t)(c + cl) * 64u + (uint32_t)r16 * 4u : ~0u;
#pragma unroll
    for (int t = 0; t < NT; t++) {
      w.sc[t] = __builtin_amdgcn_raw_buffer_load_b32(wd[t], cs, 0, 0);
      if constexpr (HASMIN) w.mn[t] = __builtin_amdgcn_raw_buffer_load_b32(wd[t], c + cl < c1 ? cs + (moff - soff) : ~0u, 0, 0);
    }
  };

  const int om = tid >> 4, on = tile0 * 16 + r16;                 // output of threads below 16 M; its (first) column
  const bool fin = tid < a.M * 16 && on < a.N;
  // FK_ROPE: the row's position and newest key ahead of all; what they lead to (cos / sin, the key's block) behind the weights'
  // requests, which its round trip would hold back -- of 9 to 16 rows ahead of them (us of 16 rows, ahead / behind: sym_int4 [6144,
  // 4096] 7.9 / 8.2, fp8_e5m2 [4608, 3584] 9.4 / 10.3; of 1 row 5.7 / 5.45)
  constexpr bool LATE = MR <= 8;
  const int mc = min(om, a.M - 1);                                // (in every thread: the counted waits of the loop stay exact)
  int64_t pos = 0, key = -1;
  if constexpr (EPI == FK_ROPE) {
    pos = a.rpos[mc];
    if (a.q16) key = (int64_t)a.lens[mc] - 1;
  }
  constexpr int XV = MR <= 4 ? RG : 1;                            // pieces of x ahead
  uint4 xv[XV][XL];
#pragma unroll
  for (int u = 0; u < XV; u++) load_x(xv[u], u);
  // what the last step reads: requested now
  uint32_t blk = ~0u, in_blk = 0;                                 // block of the new key, offset in it (below 2^32: host)
  uint16_t res16 = 0, nw16 = 0;
  float2 cs = make_float2(1.f, 0.f);
  float bias[NT] = {};
  auto lead = [&]() {
    const int d = on & ((1 << dsh) - 1);                          // (below half a head)
    cs = ((const float2*)a.rcs)[((size_t)pos << (dsh - 1)) + d];
    // (a key beyond the table, a bad block: left out here, reported by the attention, which reads them)
    if (on >= a.qcols && key >= 0 && key < (int64_t)a.max_blocks * a.bs) {
      const int bsh = (a.bs & (a.bs - 1)) == 0 ? 31 - __builtin_clz(a.bs) : -1;   // (a power of two but for odd configurations)
      const uint32_t bi = bsh >= 0 ? (uint32_t)key >> bsh : (uint32_t)key / (uint32_t)a.bs;
      blk = (uint32_t)a.tables[(size_t)mc * a.max_blocks + bi];
      const uint32_t head = (uint32_t)(on - (on < a.rcols ? a.qcols : a.rcols)) >> dsh;
      in_blk = ((head * (uint32_t)a.bs + ((uint32_t)key - bi * (uint32_t)a.bs)) << dsh) + d;
    }
  };
  RowParts<NW> parts;
  __shared__ float rscale[EPI == FK_NORM ? 1 : 16];
  if constexpr (EPI == FK_NORM) {
    if (fin) {
      if (a.zero) a.zero[(size_t)om * a.N + on] = 0.f;
      res16 = a.res[(size_t)om * a.N + on];
      nw16 = a.nw[on];
    }
  } else {
    parts.request(a, wave, lane);
    if constexpr (EPI == FK_ROPE) {
      if constexpr (!LATE) lead();
      if (fin) {
        if (a.bias) {
#pragma unroll
          for (int t = 0; t < NT; t++) bias[t] = to_f32<T>(a.bias[on + t * ht * 16]);
        }
      }
    }
  }
  asm volatile("" ::: "memory");
  Piece ring[RG];
#pragma unroll
  for (int u = 0; u < RG; u++) {
    load_sc(ring[u], c0 + u * PC);
#pragma unroll
    for (int i = 0; i < PC; i++) load_w1(ring[u], c0 + u * PC, i);
  }
  if constexpr (EPI == FK_ROPE) {
    asm volatile("" ::: "memory");
    if constexpr (LATE) lead();
    asm volatile("" : "+v"(in_blk));                              // (here, not behind the sums)
  }

  if constexpr (DK == DK_LUT4) {
    for (int i = tid; i < 256; i += NW * 64) lut2[i] = pack2<F16>(hd_lut4(a.lut_fmt, i & 15), hd_lut4(a.lut_fmt, i >> 4));
    __syncthreads();
  }
  const uint32_t mask_s = a.nib_mask, magic_v = opaque_v(a.nib_magic);
  constexpr uint32_t cst = raw_const2<DK, C>();
  const uint4 cA = make_uint4(cst, cst, cst, cst);
  const uint8_t* xf = xs + min(r16, MR - 1) * ROW + g * 16;       // rows past MR repeat the last one: never stored
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = zero;
  auto compute = [&](const Piece& w, int i) {
    const int from = (16 * i + r16) * 4;
    uint32_t sc[NT], mnw[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
      sc[t] = __builtin_amdgcn_ds_bpermute(from, w.sc[t]);
      mnw[t] = HASMIN ? __builtin_amdgcn_ds_bpermute(from, w.mn[t]) : 0;
    }
#pragma unroll
    for (int blk = 0; blk < 2; blk++) {
      const uint4 B0 = *(const uint4*)(xf + i * 256 + blk * 128), B1 = *(const uint4*)(xf + i * 256 + blk * 128 + 64);
      f32x4 X = zero;
      if constexpr (NEEDX) {
        X = mfma16<C>(B0, cA, X);
        X = mfma16<C>(B1, cA, X);
      }
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const uint4(&q)[QL] = w.q[i][t];
        uint4 A0, A1;
        if constexpr (BITS == 4) {
          A0 = raw_a4<DK, C>(blk == 0 ? q[0].x : q[0].z, mask_s, magic_v, lut2);
          A1 = raw_a4<DK, C>(blk == 0 ? q[0].y : q[0].w, mask_s, magic_v, lut2);
        } else {
          A0 = raw_a8<DK, C>(q[blk].x, q[blk].y);
          A1 = raw_a8<DK, C>(q[blk].z, q[blk].w);
        }
        f32x4 P = mfma16<C>(B0, A0, OFFS ? X : zero);
        P = mfma16<C>(B1, A1, P);
        const float d = f16_to_f32((uint16_t)(sc[t] >> (16 * blk)));
#pragma unroll
        for (int e = 0; e < 4; e++) acc[t][e] = __builtin_fmaf(d, P[e], acc[t][e]);
        if constexpr (HASMIN) {
          // X holds const * sum of x (const an exact power of two)
          constexpr float f = OFFS ? -1.f / (std::is_same<C, BF16>::value ? 128.f : 1024.f) : 1.f;
          const float mn = f * f16_to_f32((uint16_t)(mnw[t] >> (16 * blk)));
#pragma unroll
          for (int e = 0; e < 4; e++) acc[t][e] = __builtin_fmaf(mn, X[e], acc[t][e]);
        }
      }
    }
  };

  const int np = ((KC + NW - 1) / NW + PC - 1) / PC;              // pieces of the longest wave (host: RG <= np)
  // LDS operations of a wave are done in order: piece p + 1 is stored behind the reads of piece p without a wait
  auto piece = [&](auto U, int p, auto more) {
    Piece& w = ring[decltype(U)::value];
    uint4(&v)[XL] = xv[decltype(U)::value % XV];
    const int c = c0 + p * PC;
    asm volatile("" ::: "memory");
    store_x(v);
    asm volatile("" ::: "memory");
    if (decltype(more)::value || (XV < RG && p + 1 < np)) load_x(v, p + XV);
#pragma unroll
    for (int i = 0; i < PC; i++) {
      if (c + i < c1) compute(w, i);
      if constexpr (decltype(more)::value) load_w1(w, c + RG * PC, i);
    }
    if constexpr (decltype(more)::value) load_sc(w, c + RG * PC);
  };
  // requests run RG pieces ahead and stop at the last one: a load out of range costs its turn in the address unit
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  constexpr std::integral_constant<int, 0> u0{};
  constexpr std::integral_constant<int, RG - 1> u1{};
  if constexpr (RG == 1) {
    piece(u0, 0, no);
  } else {
    int p = 0;
    for (; p + 4 <= np; p += 2) {
      piece(u0, p, yes);
      piece(u1, p + 1, yes);
    }
    if (p + 3 == np) {
      piece(u0, p, yes);
      piece(u1, p + 1, no);
      piece(u0, p + 2, no);
    } else {
      piece(u0, p, no);
      piece(u1, p + 1, no);
    }
  }

  // ---- the waves' sums, in the order of K; lane holds column r16 of rows 4 g + e
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (4 * g + e < MR) red[((t * NW + wave) * MR + 4 * g + e) * 16 + r16] = acc[t][e];
  if constexpr (EPI != FK_NORM) parts.finish(a, wave, lane, rscale);
  __syncthreads();
  if (tid >= a.M * 16) return;                                    // (whole 16-lane groups)
  float y[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    y[t] = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) y[t] += red[((t * NW + w) * MR + om) * 16 + r16];
  }
  const float rs = EPI != FK_NORM && a.xpss_parts > 0 ? rscale[om & 15] : 1.f;
  auto rnd = [](float v) { return to_f32<T>(from_f32<T>(v)); };
  if constexpr (EPI == FK_NORM) {
    float h = 0.f;
    if (fin) {
      float wv = to_f32<T>(nw16);
      if (a.unit) wv = rnd(1.f + wv);
      h = rnd(rnd(y[0]) + to_f32<T>(res16));
      a.res_out[(size_t)om * a.N + on] = from_f32<T>(h);
      a.xo[(size_t)om * a.N + on] = from_f32<T>(wv * h);
    }
    float ss = h * h;
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 16);
    if (r16 == 0) a.ss[(size_t)om * gridDim.x + tile0] = ss;
  } else if constexpr (EPI == FK_ROPE) {
    if (!fin) return;
    const float c = rnd(cs.x), sn = rnd(cs.y);                    // as the model casts its tables
    const float y0 = __builtin_fmaf(y[0], rs, bias[0]), y1 = __builtin_fmaf(y[NT - 1], rs, bias[NT - 1]);
    const bool rot = on < a.rcols;                                // v: as it is (an infinity times a sine of 0 is no number)
    const float o0 = rot ? __builtin_fmaf(-y1, sn, y0 * c) : y0;  // (spelled out: one rounding in every instantiation)
    const float o1 = rot ? __builtin_fmaf(y0, sn, y1 * c) : y1;
    if (a.q16 == nullptr) {
      float* o = a.out32 + (size_t)om * a.N + on;
      o[0] = o0;
      o[ht * 16] = o1;
      return;
    }
    uint16_t* o = a.q16 + (size_t)om * a.qcols + on;
    if (on >= a.qcols) {
      if (blk >= (uint32_t)a.num_blocks) return;
      o = (rot ? a.k_cache : a.v_cache) + (size_t)blk * ((uint32_t)(a.rcols - a.qcols) * (uint32_t)a.bs) + in_blk;
    }
    o[0] = from_f32<T>(o0);
    o[ht * 16] = from_f32<T>(o1);
  } else {
    const float gv = y[0] * rs, uv = y[NT - 1] * rs;
    const int n = blockIdx.x * 16 + r16;
    if (fin) a.xo[(size_t)om * (a.N / 2) + n] = from_f32<T>((a.act == 0 ? silu_f(gv) : gelu_tanh_f(gv)) * uv);
  }
}

template <int DK, typename T, int MR, int RG, int EPI, int NW = FULLK_NW>
void launch_fullk_t(const FullkArgs& a, hipStream_t st) {
  constexpr int NT = fullk_tiles(EPI);
  constexpr size_t shmem = fullk_shmem(MR, NW, NT, DK == DK_LUT4);
  if (shmem > 64 * 1024) {
    static std::once_flag once;
    std::call_once(once, [&] {
      if (hipFuncSetAttribute((const void*)lowbit_fullk_kernel<DK, T, MR, RG, EPI, NW>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem) != hipSuccess)
        (void)hipGetLastError();
    });
  }
  hipLaunchKernelGGL((lowbit_fullk_kernel<DK, T, MR, RG, EPI, NW>), dim3(((a.N + 15) / 16) / NT), dim3(NW * 64), shmem, st, a);
}
template <int DK, typename T, int MR, int EPI>
void launch_fullk_r(const FullkArgs& a, hipStream_t st) {
  if ((a.KC + FULLK_NW - 1) / FULLK_NW <= fullk_pc(MR)) return launch_fullk_t<DK, T, MR, 1, EPI>(a, st);
  // down projections of few rows whose K is two pieces for each of 16 waves: what hides the second piece is the other
  // waves, where their registers (128) hold it.  8 / 16 waves, us at 1 / 2 / 3 rows: sym_int4 [4096, 14336] 9.1 9.1 10.3 /
  // 8.4 8.6 9.2, sym_int8 14.1 14.4 / 13.0 13.4 (3 rows spill: 15.1 / 21.4); three pieces, [3584, 18944], sym_int4 10.0 10.6
  // 11.6 / 10.3 10.6 11.3, fp8_e5m2 13.7 14.0 / 14.2 14.6; tables 12.6 12.9 / 13.3 14.2
  if constexpr (EPI == FK_NORM && MR <= (dk_bits(DK) == 4 ? 4 : 2) && DK != DK_LUT4) {
    if (a.KC > 16 * fullk_pc(MR) && a.KC <= 32 * fullk_pc(MR)) return launch_fullk_t<DK, T, MR, 2, EPI, 16>(a, st);
  }
  launch_fullk_t<DK, T, MR, 2, EPI>(a, st);
}
template <int DK, typename T, int EPI>
void launch_fullk_m(const FullkArgs& a, hipStream_t st) {
  if (a.M == 1) launch_fullk_r<DK, T, 1, EPI>(a, st);
  else if (a.M == 2) launch_fullk_r<DK, T, 2, EPI>(a, st);
  else if (a.M <= 4) launch_fullk_r<DK, T, 4, EPI>(a, st);
  else if (a.M <= 8) launch_fullk_r<DK, T, 8, EPI>(a, st);
  else launch_fullk_r<DK, T, 16, EPI>(a, st);
}
template <int DK, typename T>
void launch_fullk_e(int epi, const FullkArgs& a, hipStream_t st) {
  if (epi == FK_NORM) launch_fullk_m<DK, T, FK_NORM>(a, st);
  else if (epi == FK_ROPE) launch_fullk_m<DK, T, FK_ROPE>(a, st);
  else launch_fullk_m<DK, T, FK_GLU>(a, st);
}
template <int DK>
void launch_fullk_dk(bool bf16, int epi, const FullkArgs& a0, hipStream_t st) {
  FullkArgs a = a0;
  a.nib_mask = 0x000F000Fu;
  a.nib_magic = bf16 && DK != DK_LUT4 ? Raw<BF16>::k4 : Raw<F16>::k4;
  if (bf16) launch_fullk_e<DK, BF16>(epi, a, st);
  else launch_fullk_e<DK, F16>(epi, a, st);
}

}  // namespace illm
