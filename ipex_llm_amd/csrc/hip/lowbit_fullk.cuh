// Low-bit weight x bf16/f16 activations of 1 to 16 rows with the residual add and the deferred RMSNorm behind it (a
// decode step's o and down projections) on gfx950 MFMA: one workgroup finishes 16 output columns.
#pragma once
#include <mutex>
#include <type_traits>

#include "../common/quant_block.h"
#include "gemv_args.h"
#include "illm_device.h"
#include "lowbit_raw.h"

namespace illm {

// k-chunks staged at a time, LDS bytes of a staged row (+ 16: the 16 rows of a fragment read fall on distinct banks)
__host__ __device__ constexpr int fullk_pc(int mr) { return mr <= 8 ? 4 : 2; }
__host__ __device__ constexpr int fullk_row(int mr) { return fullk_pc(mr) * CHUNK_K * 2 + 16; }
// staged x of every wave, the waves' sums, the pair table
__host__ __device__ constexpr size_t fullk_shmem(int mr, int nw, bool lut) {
  return (size_t)nw * mr * fullk_row(mr) + (size_t)nw * mr * 16 * 4 + (lut ? 1024 : 0);
}

// MR: rows of the instantiation (1, 2, 4, 8, 16), a.M <= MR
template <int DK, typename T, int MR, int NW>
__global__ void __launch_bounds__(NW * 64) lowbit_fullk_kernel(const FullkArgs a) {
  using C = typename std::conditional<DK == DK_LUT4, F16, T>::type;   // product type: table formats keep an f16 table
  constexpr int BITS = dk_bits(DK);
  constexpr bool HASMIN = dk_has_min(DK);
  constexpr bool OFFS = dk_needx(DK) && DK != DK_INT8A;           // codes carry an offset
  constexpr bool NEEDX = OFFS || HASMIN;
  constexpr int PC = fullk_pc(MR), ROW = fullk_row(MR);
  constexpr int XL = MR * PC / 4;                                 // 1-KB loads of a piece of x (PC chunks of MR rows)
  constexpr int QL = BITS / 4;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  uint8_t* xs = smem + (size_t)wave * MR * ROW;                   // this wave's alone: no barrier before the sums
  float* red = (float*)(smem + (size_t)NW * MR * ROW);            // [NW][MR][16]
  uint32_t* lut2 = (uint32_t*)(red + NW * MR * 16);

  const int tile = blockIdx.x, KC = a.KC;
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
  const __amdgpu_buffer_rsrc_t wd =
      __builtin_amdgcn_make_buffer_rsrc((void*)(a.w + (size_t)tile * TB), 0, (int)TB, 0x00020000);
  const uint32_t soff = (uint32_t)KC * dk_code_chunk(DK), moff = soff + 16u * (uint32_t)KC * 4u;
  struct Chunk {
    uint4 q[QL];
    uint32_t sc, mn[HASMIN ? 1 : 0 + 1];
  };
  auto load_w = [&](Chunk& ch, int c) {                           // past the wave's range: no memory traffic, zeros
    const bool on = c < c1;
    const uint32_t cb = (uint32_t)c * dk_code_chunk(DK), cs = (uint32_t)c * 64u;
#pragma unroll
    for (int j = 0; j < QL; j++)
      ch.q[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
          wd, on ? cb + (uint32_t)lane * 16u + j * 1024u : ~0u, 0, 2));
    ch.sc = __builtin_amdgcn_raw_buffer_load_b32(wd, on ? soff + cs + (uint32_t)r16 * 4u : ~0u, 0, 0);
    if constexpr (HASMIN) ch.mn[0] = __builtin_amdgcn_raw_buffer_load_b32(wd, on ? moff + cs + (uint32_t)r16 * 4u : ~0u, 0, 0);
  };

  uint4 xv[XL];
  load_x(xv, 0);
  // what the last step reads: requested now
  const int om = tid >> 4, on = tile * 16 + r16;                  // output of threads below 16 M
  const bool fin = tid < a.M * 16 && on < a.N;
  uint16_t res16 = 0, nw16 = 0;
  if (fin) {
    res16 = a.res[(size_t)om * a.N + on];
    nw16 = a.nw[on];
  }
  asm volatile("" ::: "memory");
  Chunk ring[2][PC];
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int i = 0; i < PC; i++) load_w(ring[u][i], c0 + u * PC + i);

  if constexpr (DK == DK_LUT4) {
    for (int i = tid; i < 256; i += NW * 64) lut2[i] = pack2<F16>(hd_lut4(a.lut_fmt, i & 15), hd_lut4(a.lut_fmt, i >> 4));
    __syncthreads();
  }
  const uint32_t mask_s = a.nib_mask, magic_v = opaque_v(a.nib_magic);
  constexpr uint32_t cst = raw_const2<DK, C>();
  const uint4 cA = make_uint4(cst, cst, cst, cst);
  const uint8_t* xf = xs + min(r16, MR - 1) * ROW + g * 16;       // rows past MR repeat the last one: never stored
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 acc = zero;
  auto compute = [&](const Chunk& ch, int i) {
#pragma unroll
    for (int blk = 0; blk < 2; blk++) {
      const uint4 B0 = *(const uint4*)(xf + i * 256 + blk * 128), B1 = *(const uint4*)(xf + i * 256 + blk * 128 + 64);
      f32x4 X = zero;
      if constexpr (NEEDX) {
        X = mfma16<C>(B0, cA, X);
        X = mfma16<C>(B1, cA, X);
      }
      uint4 A0, A1;
      if constexpr (BITS == 4) {
        A0 = raw_a4<DK, C>(blk == 0 ? ch.q[0].x : ch.q[0].z, mask_s, magic_v, lut2);
        A1 = raw_a4<DK, C>(blk == 0 ? ch.q[0].y : ch.q[0].w, mask_s, magic_v, lut2);
      } else {
        A0 = raw_a8<DK, C>(ch.q[blk].x, ch.q[blk].y);
        A1 = raw_a8<DK, C>(ch.q[blk].z, ch.q[blk].w);
      }
      f32x4 P = mfma16<C>(B0, A0, OFFS ? X : zero);
      P = mfma16<C>(B1, A1, P);
      const float d = f16_to_f32((uint16_t)(ch.sc >> (16 * blk)));
#pragma unroll
      for (int e = 0; e < 4; e++) acc[e] = __builtin_fmaf(d, P[e], acc[e]);
      if constexpr (HASMIN) {
        // X holds const * sum of x (const an exact power of two)
        constexpr float f = OFFS ? -1.f / (std::is_same<C, BF16>::value ? 128.f : 1024.f) : 1.f;
        const float mn = f * f16_to_f32((uint16_t)(ch.mn[0] >> (16 * blk)));
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] = __builtin_fmaf(mn, X[e], acc[e]);
      }
    }
  };

  // LDS operations of a wave are done in order: piece p + 1 is stored behind the reads of piece p without a wait
  auto piece = [&](Chunk (&ch)[PC], int c) {
    store_x(xv);
    load_x(xv, (c - c0) / PC + 1);
#pragma unroll
    for (int i = 0; i < PC; i++) {
      if (c + i < c1) compute(ch[i], i);
      load_w(ch[i], c + 2 * PC + i);
    }
  };
  for (int c = c0; c < c1; c += 2 * PC) {
    piece(ring[0], c);
    if (c + PC < c1) piece(ring[1], c + PC);
  }

  // ---- the waves' sums, in the order of K; lane holds column r16 of rows 4 g + e
#pragma unroll
  for (int e = 0; e < 4; e++)
    if (4 * g + e < MR) red[(wave * MR + 4 * g + e) * 16 + r16] = acc[e];
  __syncthreads();
  if (tid >= a.M * 16) return;                                    // (whole 16-lane groups)
  float y = 0.f;
#pragma unroll
  for (int w = 0; w < NW; w++) y += red[(w * MR + om) * 16 + r16];
  auto rnd = [](float v) { return to_f32<T>(from_f32<T>(v)); };
  float h = 0.f;
  if (fin) {
    float wv = to_f32<T>(nw16);
    if (a.unit) wv = rnd(1.f + wv);
    h = rnd(rnd(y) + to_f32<T>(res16));
    a.res_out[(size_t)om * a.N + on] = from_f32<T>(h);
    a.xo[(size_t)om * a.N + on] = from_f32<T>(wv * h);
  }
  float ss = h * h;
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 16);
  if (r16 == 0) a.ss[(size_t)om * gridDim.x + tile] = ss;
}

template <int DK, typename T, int MR, int NW>
void launch_fullk_t(const FullkArgs& a, hipStream_t st) {
  constexpr size_t shmem = fullk_shmem(MR, NW, DK == DK_LUT4);
  if (shmem > 64 * 1024) {
    static std::once_flag once;
    std::call_once(once, [&] {
      if (hipFuncSetAttribute((const void*)lowbit_fullk_kernel<DK, T, MR, NW>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)shmem) != hipSuccess)
        (void)hipGetLastError();
    });
  }
  hipLaunchKernelGGL((lowbit_fullk_kernel<DK, T, MR, NW>), dim3((a.N + 15) / 16), dim3(NW * 64), shmem, st, a);
}
template <int DK, typename T, int NW>
void launch_fullk_m(const FullkArgs& a, hipStream_t st) {
  if (a.M == 1) launch_fullk_t<DK, T, 1, NW>(a, st);
  else if (a.M == 2) launch_fullk_t<DK, T, 2, NW>(a, st);
  else if (a.M <= 4) launch_fullk_t<DK, T, 4, NW>(a, st);
  else if (a.M <= 8) launch_fullk_t<DK, T, 8, NW>(a, st);
  else launch_fullk_t<DK, T, 16, NW>(a, st);
}
template <int DK>
void launch_fullk_dk(bool bf16, int nw, const FullkArgs& a0, hipStream_t st) {
  FullkArgs a = a0;
  a.nib_mask = 0x000F000Fu;
  a.nib_magic = bf16 && DK != DK_LUT4 ? Raw<BF16>::k4 : Raw<F16>::k4;
  if (bf16) nw == 16 ? launch_fullk_m<DK, BF16, 16>(a, st) : launch_fullk_m<DK, BF16, 8>(a, st);
  else nw == 16 ? launch_fullk_m<DK, F16, 16>(a, st) : launch_fullk_m<DK, F16, 8>(a, st);
}

}  // namespace illm
