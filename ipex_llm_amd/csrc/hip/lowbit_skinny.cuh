// Low-bit weight x bf16/f16 activation product for up to a few hundred rows
// (serving decode batches, speculative verify, short prompts) on gfx950 MFMA;
// up to 16 rows beside the decode kernel (skinny16 in csrc/torch/ops_hip.cpp says when).
//
// Between the one-row-tile GEMV (lowbit_gemv5.cuh) and the compute-bound
// prefill GEMM the weight stream still bounds the product (a Llama-3-8B
// gate/up at 48 rows: 62 MB of codes and scales, 13 us at the rate of a large
// copy, beside 11 GFLOP), so the split is made for the stream:
//   * workgroup = NW = 8 (4) waves = 128 (64) output columns x R = MT * 16 rows;
//     wave (cg, kp) owns two 16-column weight tiles (cg) and every second 128-k
//     chunk (kp): codes go global -> registers in MFMA fragment order
//     (formats.h), a ring of three chunks of both tiles per wave, requested two
//     steps ahead, and no weight is read twice by a row block;
//   * x is staged through LDS once per workgroup and 256-k step (three buffers: one is read, one is ahead, one is
//     stored into), XOR-swizzled in 16-B pieces so the 16 rows of a fragment read fall on distinct banks;
//   * x is the A operand and the codes are the B operand, raw (exact in bf16 / f16): a lane holds four rows of ONE
//     column, so a (tile, chunk) takes one scale dword per lane where the other order takes four (a 16-B load of 16
//     cycles in the address unit, as long as the codes' own);
//   * the block scale is applied to the f32 block sum.  The offset of the integer formats is one product of the
//     block's x with the constant -offset: it comes out broadcast over the tile's columns, i.e. it IS the
//     accumulator input of the code products (no per-row sums of x in memory, no subtract per value), shared by the
//     wave's two tiles;
//   * loads through buffer descriptors (lane constant + scalar: no address registers that a load in flight holds),
//     each in a place of its own among the products instead of in bursts, which stalled every wave of the step behind
//     the address unit at once;
//   * split-K over blockIdx.y writes f32 slabs summed by the consumer; row
//     blocks of one column block get ids that share id % 8, so a weight chunk
//     leaves HBM once per XCD.
// MI355X, us, back-to-back launches, bursts and four scales per lane / this: sym_int4 48 rows gate/up [28672, 4096]
// 25.1 / 23.1, down [4096, 14336] 15.6 / 14.7, qkv [6144, 4096] 11.7 / 9.5, o [4096, 4096] 8.3 / 7.3; gate/up of 32
// rows 20.2 / 18.6, 64 rows 30.3 / 27.6; fp8_e5m2 300 rows [3584, 18944] 78.4 / 67.5, [4608, 3584] 23.5 / 19.8; nf4
// gate/up of 48 rows 27.1 / 23.4, asym_int4 27.1 / 25.2, sym_int8 29.5 / 28.5, fp4 21.2 / 19.4; the pair table of 128
// rows [6144, 4096] 37.4 / 32.5.  What bounds it: issue, two waves per SIMD with 36 products (8 of an MFMA's 16 cycles
// each) and some 110 vector instructions a step, 13.9 us of the 18.1 that 16 steps of the gate/up pair take, the
// products alone 10.1.  Four steps of weights in flight measured no faster than three (23.9), nor did the bursts with
// the next step's decoding and reads between the products (26.1).
#pragma once
#include <mutex>
#include <type_traits>

#include "../common/quant_block.h"
#include "gemv_args.h"
#include "illm_device.h"
#include "kernels_skinny.h"
#include "lowbit_raw.h"

namespace illm {

// 16 B per lane through a buffer descriptor (reads past its range return 0)
__device__ __forceinline__ uint4 buf16(const __amdgpu_buffer_rsrc_t& r, uint32_t voff, int soff) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// FINE (a table weight under bf16 x): every entry as a bf16 pair hi + lo, two products each.  An entry is then
// 2^-17 off at most, where a bf16 table is 2^-9 and an f16 one 2^-12.  For the products of 65 rows and up that
// a kernel with an f16 table served: nf4 [6144, 4096], one entry / a pair / that kernel, 80 rows 20.5 / 24.3 / 42.6
// us, 256 rows 29 / 38 / 45 (twice the matrix work of a product that has no offsets, 8-B table reads)
template <int DK, typename T, int MT, int NW, bool FINE = false>
__global__ void __launch_bounds__(NW * 64, 2) lowbit_skinny_kernel(const GemvArgs a, const int epi) {
  constexpr int BITS = dk_bits(DK);
  constexpr bool HASMIN = dk_has_min(DK);
  constexpr bool OFFS = dk_needx(DK) && DK != DK_INT8A;   // codes carry an offset
  constexpr bool NEEDX = OFFS || HASMIN;       // ... or the block minimum needs the sum of x
  constexpr int R = MT * 16;
  constexpr int SK_TILES = NW / SK_KW * SK_TPW;
  constexpr int RG = 3;                        // steps in the rings of weights (registers) and of x (LDS)
  constexpr int XJ = MT * 8 / NW;              // 16-B pieces of x per thread and step
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  // x of three steps: [3][R][SK_STEP], then the table
  static_assert(!FINE || (DK == DK_LUT4 && std::is_same<T, BF16>::value), "the finer table: table formats in bf16");
  uint32_t* lut2 = (uint32_t*)(smem + 3 * R * SK_STEP * 2);       // DK_LUT4 only: [256] (FINE: {hi, lo})
  const uint2* lutf = (const uint2*)lut2;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);      // uniform: weight addresses live in SGPRs
  const int g = lane >> 4, r16 = lane & 15;
  const int cg = wave >> 1, kp = wave & 1;

  // block -> (column block, row block): the MB row blocks of a column block share id % 8, or, in a grid without
  // the padding that this takes, column blocks first (skinny_plan says when)
  const int NT = (a.N * (epi == EPI_GLU ? 2 : 1) + 15) / 16;
  const int NB = (NT + SK_TILES - 1) / SK_TILES;
  const int MB = (a.M + R - 1) / R;
  int nb = blockIdx.x, mb = 0;
  if (MB > 1 && NB % 8 != 0 && (int)gridDim.x == NB * MB) {
    mb = blockIdx.x / NB;
    nb = blockIdx.x % NB;
  } else if (MB > 1) {
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

  // x of a deferred norm: its rows' sums of squares, summed behind the first requests (one row tile: 1 to 16 rows; the sums
  // of more cost the gate/up product of 48 rows what the norm launch took)
  float* rsum = (float*)(smem + 3 * R * SK_STEP * 2 + skinny_table(DK == DK_LUT4, FINE));
  RowParts<NW> parts;
  if constexpr (MT == 1) parts.request(a, wave, lane);

  if constexpr (DK == DK_LUT4) {
    if (tid < 256) {
      const float v0 = hd_lut4(a.lut_fmt, tid & 15), v1 = hd_lut4(a.lut_fmt, tid >> 4);
      if constexpr (FINE)
        ((uint2*)lut2)[tid] = make_uint2(pack2<T>(v0, v1), pack2<T>(v0 - to_f32<T>(from_f32<T>(v0)),
                                                                    v1 - to_f32<T>(from_f32<T>(v1))));
      else
        lut2[tid] = pack2<T>(v0, v1);
    }
  }

  // ---- weights: this wave's chunk of a step is c0 + 2 step + kp
  const size_t TB = (size_t)dk_tile_bytes(DK, KC);
  const uint32_t soff = (uint32_t)KC * dk_code_chunk(DK), moff = soff + 16 * KC * 4;
  const uint32_t lq = lane * 16, ls = r16 * 4;                    // lane's codes; its column's scales
  // through buffer descriptors: a load's address is a lane constant + a scalar, no register of its own to wait for
  __amdgpu_buffer_rsrc_t wr[SK_TPW];
#pragma unroll
  for (int t = 0; t < SK_TPW; t++)
    wr[t] = __builtin_amdgcn_make_buffer_rsrc((void*)(a.w + (size_t)min(tile0 + t, NT - 1) * TB), 0, (int)TB, 0x00020000);
  struct Chunk {
    uint4 q[SK_TPW][BITS / 4];
    uint32_t sc[SK_TPW], mn[HASMIN ? SK_TPW : 1];
  };
  constexpr int WL = BITS / 4 + (HASMIN ? 2 : 1);                 // loads of a tile's chunk
  auto load_w1 = [&](Chunk& ch, int step, int i) {                // load i of SK_TPW * WL
    const int c = min(c0 + step * SK_KW + kp, c1 - 1), t = i / WL, j = i % WL;   // clamped: unconditional loads
    if (j == 0) ch.sc[t] = __builtin_amdgcn_raw_buffer_load_b32(wr[t], soff + ls, c * 64, 0);
    else if (j <= BITS / 4) ch.q[t][j - 1] = buf16(wr[t], lq + (j - 1) * 1024, c * dk_code_chunk(DK));
    else ch.mn[t] = __builtin_amdgcn_raw_buffer_load_b32(wr[t], moff + ls, c * 64, 0);
  };
  auto load_w = [&](Chunk& ch, int step) {
#pragma unroll
    for (int i = 0; i < SK_TPW * WL; i++) load_w1(ch, step, i);
  };

  // ---- x: thread -> rows tid / 32 + 16 j, 16-B piece tid % 32 of the step
  const int xr0 = tid >> 5, xc = tid & 31;
  const int kend = min(a.K, c1 * CHUNK_K);
  const __amdgpu_buffer_rsrc_t xd =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.x, 0, (int)((uint32_t)a.M * (uint32_t)a.ldx * 2u), 0x00020000);
  uint32_t xo[XJ];                                                // byte offset of the row's piece (host: < 4 GB)
#pragma unroll
  for (int j = 0; j < XJ; j++) xo[j] = (uint32_t)min(m0 + xr0 + NW * 2 * j, a.M - 1) * (uint32_t)a.ldx * 2u + xc * 16;
  auto load_x1 = [&](int step, int j) {                           // past the slice: out of the descriptor's range, zeros
    const int k = (c0 + step * SK_KW) * CHUNK_K;
    return buf16(xd, k + xc * 8 < kend ? xo[j] + (uint32_t)k * 2u : ~0u, 0);
  };
  // piece p of row r lives at piece p ^ (r & 15) (within its half of the step)
  auto store_x1 = [&](const uint4& v, uint32_t buf, int j) {
    const int row = xr0 + NW * 2 * j;
    *(uint4*)(smem + (buf + (uint32_t)row * SK_STEP * 2 + ((xc & 16) | ((xc ^ row) & 15)) * 16)) = v;
  };

  f32x4 acc[SK_TPW][MT];
#pragma unroll
  for (int t = 0; t < SK_TPW; t++)
#pragma unroll
    for (int mt = 0; mt < MT; mt++) acc[t][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t mask_s = a.nib_mask, magic_v = opaque_v(a.nib_magic);
  constexpr uint32_t cst = raw_const2<DK, T>();
  const uint4 cA = make_uint4(cst, cst, cst, cst);

  // ---- a phase = one 64-k block: products of the block's first 32 k (pass a), of its second (pass b), before them the
  // offset products where the codes carry one.  Beside a pass' products, in program order between them: the scales of
  // the block before, the decoding of the weights and the x reads of the pass after the next.
  constexpr int NP = SK_TPW * MT;                                 // products of a pass
  constexpr int NB1 = NEEDX ? 2 : 1;                              // (the offset products need both halves of x at once)
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 P[SK_TPW][MT], X[2][NEEDX ? MT : 1];
  uint4 A[SK_TPW][2], lo[FINE ? SK_TPW : 1][2], B0[MT], B1[NB1][MT];
  float d[2][SK_TPW], mn[2][HASMIN ? SK_TPW : 1];
#pragma unroll
  for (int t = 0; t < SK_TPW; t++)
#pragma unroll
    for (int mt = 0; mt < MT; mt++) P[t][mt] = zero;
#pragma unroll
  for (int t = 0; t < SK_TPW; t++) d[0][t] = d[1][t] = 0.f;
  if constexpr (HASMIN) {
#pragma unroll
    for (int t = 0; t < SK_TPW; t++) mn[0][t] = mn[1][t] = 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; mt++) X[0][mt] = X[1][mt] = zero;
  }
  const uint32_t xl = (uint32_t)r16 * SK_STEP * 2 + kp * CHUNK_K * 2;
  auto read_x = [&](uint32_t buf, int blk, int ss, int mt) {      // buf: byte offset of the step's x
    return *(const uint4*)(smem + (buf + xl + (uint32_t)(((8 * blk + 4 * ss + g) ^ r16) * 16)) + mt * 16 * SK_STEP * 2);
  };
  auto decode = [&](const Chunk& ch, int blk, int ss, int t, int c) {   // dword c of a fragment
    uint32_t v;
    if constexpr (BITS == 4) {
      const uint4& q = ch.q[t][0];
      const uint32_t w = blk == 0 ? (ss == 0 ? q.x : q.y) : (ss == 0 ? q.z : q.w);
      if constexpr (FINE) {
        const uint2 e = lutf[(w >> (8 * c)) & 0xff];
        v = e.x;
        uint4& l = lo[t][ss];
        (c == 0 ? l.x : c == 1 ? l.y : c == 2 ? l.z : l.w) = e.y;
      } else {
        v = raw_a4_at<DK, T>(w, c, mask_s, magic_v, lut2);
      }
    } else {
      const uint4& q = ch.q[t][blk];
      const uint32_t w = ss == 0 ? (c < 2 ? q.x : q.y) : (c < 2 ? q.z : q.w);
      v = raw_pair8<DK, T>(w, c & 1);
    }
    uint4& f = A[t][ss];
    (c == 0 ? f.x : c == 1 ? f.y : c == 2 ? f.z : f.w) = v;
  };
  auto scales = [&](const Chunk& ch, int blk, int t) {
    d[blk][t] = f16_to_f32((uint16_t)(ch.sc[t] >> (16 * blk)));
    if constexpr (HASMIN) {
      // times the sum of x: the offset product holds -offset * sum (exact power of two)
      constexpr float f = OFFS ? -1.f / (std::is_same<T, BF16>::value ? 128.f : 1024.f) : 1.f;
      mn[blk][t] = f * f16_to_f32((uint16_t)(ch.mn[t] >> (16 * blk)));
    }
  };
  auto scale_out = [&](int i, int blk) {                          // product i of block blk into the sums
    const int mt = i / SK_TPW, t = i % SK_TPW;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      acc[t][mt][e] = __builtin_fmaf(d[blk][t], P[t][mt][e], acc[t][mt][e]);
      if constexpr (HASMIN) acc[t][mt][e] = __builtin_fmaf(mn[blk][t], X[blk][mt][e], acc[t][mt][e]);
    }
  };
  constexpr int LATE = NEEDX ? 0 : NP / 2;                        // products scaled in their own pass b; the rest in the next phase
  // xb: this step's x, xn: the one of the next phase; ch: this chunk, nx: the next phase's
  constexpr int PH = (NEEDX ? 2 * MT : 0) + 2 * NP;               // slots of a phase
  auto phase = [&](const Chunk& ch, const Chunk& nx, int blk, uint32_t xb, uint32_t xn, auto&& fill) {
    const int nblk = blk ^ 1;
    if constexpr (NEEDX) {
#pragma unroll
      for (int j = 0; j < 2 * MT; j++) {
        const int mt = j % MT;
#pragma unroll
        for (int i = j * NP / (2 * MT); i < (j + 1) * NP / (2 * MT); i++) scale_out(i, nblk);
        X[blk][mt] = j < MT ? mfma16<T>(B0[mt], cA, zero) : mfma16<T>(B1[blk][mt], cA, X[blk][mt]);
        fill(j);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int j = 0; j < NP; j++) {
      const int mt = j / SK_TPW, t = j % SK_TPW;
      if (!NEEDX && j + LATE < NP) scale_out(j + LATE, nblk);
      P[t][mt] = mfma16<T>(B0[mt], A[t][0], OFFS ? X[blk][mt] : zero);
      if (!NEEDX && j < MT) B1[0][j] = read_x(xb, blk, 1, j);
#pragma unroll
      for (int c = j * 4 * SK_TPW / NP; c < (j + 1) * 4 * SK_TPW / NP; c++) decode(ch, blk, 1, c / 4, c % 4);
      if (j >= NP - SK_TPW) scales(ch, blk, j - (NP - SK_TPW));
      fill((NEEDX ? 2 * MT : 0) + j);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (FINE) {
#pragma unroll
      for (int j = 0; j < NP; j++) P[j % SK_TPW][j / SK_TPW] = mfma16<T>(B0[j / SK_TPW], lo[j % SK_TPW][0], P[j % SK_TPW][j / SK_TPW]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NP; j++) P[j % SK_TPW][j / SK_TPW] = mfma16<T>(B1[0][j / SK_TPW], lo[j % SK_TPW][1], P[j % SK_TPW][j / SK_TPW]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < NP; j++) {
      const int mt = j / SK_TPW, t = j % SK_TPW;
      P[t][mt] = mfma16<T>(B1[NEEDX ? blk : 0][mt], A[t][1], P[t][mt]);
      if (j < MT) {
        B0[j] = read_x(xn, nblk, 0, j);
        if constexpr (NEEDX) B1[nblk][j] = read_x(xn, nblk, 1, j);
      }
#pragma unroll
      for (int c = j * 4 * SK_TPW / NP; c < (j + 1) * 4 * SK_TPW / NP; c++) decode(nx, nblk, 0, c / 4, c % 4);
      if (!NEEDX && j >= NP - LATE) scale_out(j - (NP - LATE), blk);
      fill((NEEDX ? 2 * MT : 0) + NP + j);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- main loop.  Step s: store x of s + 2 (requested in step s - 1) into the buffer that step s - 1 read, request x
  // of s + 3 and the weights of s + 2, two phases, barrier: what a step reads ahead from the next one's x was stored
  // before the barrier behind it.
  constexpr uint32_t XBUF = R * SK_STEP * 2;
  uint4 xr[XJ];
  Chunk ring[RG];
  {
    uint4 x1[XJ];
#pragma unroll
    for (int j = 0; j < XJ; j++) xr[j] = load_x1(0, j);
#pragma unroll
    for (int j = 0; j < XJ; j++) x1[j] = load_x1(1, j);
    __builtin_amdgcn_sched_barrier(0);         // (the order in which the loop requests and waits)
    load_w(ring[0], 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < XJ; j++) store_x1(xr[j], 0, j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < XJ; j++) xr[j] = load_x1(2, j);
    __builtin_amdgcn_sched_barrier(0);
    load_w(ring[1], 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < XJ; j++) store_x1(x1[j], XBUF, j);
  }
  if constexpr (MT == 1) parts.finish(a, wave, lane, rsum);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < MT; j++) {
    B0[j] = read_x(0, 0, 0, j);
    if constexpr (NEEDX) B1[0][j] = read_x(0, 0, 1, j);
  }
#pragma unroll
  for (int c = 0; c < 4 * SK_TPW; c++) decode(ring[0], 0, 0, c / 4, c % 4);
  constexpr int NL = SK_TPW * WL, LS = 2 * PH - 2 * XJ - 1;      // weight loads of a step, slots they are spread over
  auto step = [&](int st, auto U) {
    constexpr int u = decltype(U)::value;
    auto fill = [&](int k) {                                      // slot k of the step's 2 PH
      if (k < XJ) store_x1(xr[k], (u + 2) % RG * XBUF, k);
      else if (k < 2 * XJ) xr[k - XJ] = load_x1(st + 3, k - XJ);
#pragma unroll
      for (int i = 0; i < NL; i++)
        if (k == 2 * XJ + (i * LS) / NL) load_w1(ring[(u + 2) % RG], st + 2, i);
    };
    phase(ring[u], ring[u], 0, u * XBUF, u * XBUF, [&](int k) { fill(k); });
    phase(ring[u], ring[(u + 1) % RG], 1, u * XBUF, (u + 1) % RG * XBUF, [&](int k) { fill(PH + k); });
    __syncthreads();
  };
  int s0 = 0;
  for (; s0 + RG <= nstep; s0 += RG) {                            // whole turns of the rings, no branch inside
    step(s0, std::integral_constant<int, 0>{});
    step(s0 + 1, std::integral_constant<int, 1>{});
    step(s0 + 2, std::integral_constant<int, 2>{});
  }
  if (s0 < nstep) step(s0, std::integral_constant<int, 0>{});
  if (s0 + 1 < nstep) step(s0 + 1, std::integral_constant<int, 1>{});
#pragma unroll
  for (int i = LATE; i < NP; i++) scale_out(i, 1);

  // ---- the two k-parts through LDS (x is done: the last step's barrier is behind): each wave of a pair finishes two of
  // the lane's four rows
  float2* red = (float2*)smem;                                    // [NW / 2][2][SK_TPW][MT][64]
  auto slot = [&](int part, int t, int mt) { return (((cg * 2 + part) * SK_TPW + t) * MT + mt) * 64 + lane; };
#pragma unroll
  for (int t = 0; t < SK_TPW; t++)
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
      red[slot(kp ^ 1, t, mt)] = kp == 0 ? make_float2(acc[t][mt][2], acc[t][mt][3]) : make_float2(acc[t][mt][0], acc[t][mt][1]);
  __syncthreads();
  float o[SK_TPW][MT][2];                                         // first k-part + second, whichever wave adds them
#pragma unroll
  for (int t = 0; t < SK_TPW; t++)
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      const float2 v = red[slot(kp, t, mt)];
      o[t][mt][0] = kp == 0 ? acc[t][mt][0] + v.x : v.x + acc[t][mt][2];
      o[t][mt][1] = kp == 0 ? acc[t][mt][1] + v.y : v.y + acc[t][mt][3];
    }

  // ---- epilogue: lane holds column 16 tile + r16 of rows m0 + 16 mt + 4 g + 2 kp + e
  const int mr = m0 + 4 * g + 2 * kp;
  if (epi == EPI_GLU) {
    const int n = (tile0 / 2) * 16 + r16;
    if (tile0 + 1 >= NT || n >= a.N) return;                      // whole gate / up pairs (NT even)
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const int m = mr + mt * 16 + e;
        if (m >= a.M) continue;
        // x of a deferred norm: its row's scale
        const float rs = MT == 1 && a.xpss_parts > 0 ? rsum[m & 15]
                         : a.xpss ? rsqrtf(a.xpss[m] / (float)a.xpss_n + a.xpss_eps) : 1.f;
        const float gv = o[0][mt][e] * rs, uv = o[1][mt][e] * rs;
        ((uint16_t*)a.out)[(size_t)m * a.ldo + n] = from_f32<T>((a.act == 0 ? silu_f(gv) : gelu_tanh_f(gv)) * uv);
      }
    return;
  }
#pragma unroll
  for (int t = 0; t < SK_TPW; t++) {
    const int n = (tile0 + t) * 16 + r16;
    if (tile0 + t >= NT) continue;
    const float bv = epi != EPI_PARTIAL && a.bias && n < a.N ? to_f32<T>(a.bias[n]) : 0.f;
    if constexpr (MT == 1) {
      if (epi == EPI_STORE && a.amax) {                           // maximum of the tile's stored values, first index on ties
#pragma unroll
        for (int e = 0; e < 2; e++) {
          const float v = to_f32<T>(from_f32<T>(o[t][0][e] + bv));
          const bool on = n < a.N && v > -INFINITY;               // (false for NaN)
          float best = on ? v : -INFINITY;
          int at = on ? n : 0x7fffffff;
#pragma unroll
          for (int off = 1; off < 16; off <<= 1) {
            const float ov = __shfl_xor(best, off, 64);
            const int oi = __shfl_xor(at, off, 64);
            if (ov > best || (ov == best && oi < at)) best = ov, at = oi;
          }
          if (r16 == 0 && mr + e < a.M) a.amax[(size_t)(tile0 + t) * a.M + mr + e] = make_float2(best, __int_as_float(at));
        }
      }
    }
    if (n >= a.N) continue;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const int m = mr + mt * 16 + e;
        if (m >= a.M) continue;
        if (epi == EPI_PARTIAL) ((float*)a.out)[((size_t)blockIdx.y * a.M + m) * a.N + n] = o[t][mt][e];
        else ((uint16_t*)a.out)[(size_t)m * a.ldo + n] = from_f32<T>(o[t][mt][e] + bv);
      }
  }
}

// a kernel asking for more than 64 KiB of dynamic LDS has its limit raised first (once per kernel)
template <int DK, typename T, int MT, int NW, bool FINE = false>
void launch_skinny_t(int epi, dim3 grid, const GemvArgs& a, hipStream_t st) {
  const size_t shmem = skinny_shmem(MT, skinny_table(DK == DK_LUT4, FINE));
  if (shmem > 64 * 1024) {
    static std::once_flag once;
    std::call_once(once, [&] {
      if (hipFuncSetAttribute((const void*)lowbit_skinny_kernel<DK, T, MT, NW, FINE>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem) != hipSuccess)
        (void)hipGetLastError();
    });
  }
  hipLaunchKernelGGL((lowbit_skinny_kernel<DK, T, MT, NW, FINE>), grid, dim3(NW * 64), shmem, st, a, epi);
}

// mt: 16-row tiles per workgroup (one workgroup covers every row up to 64); nw: waves (4 or 8)
template <int DK, typename T>
void launch_skinny_mt(int mt, int nw, int epi, dim3 grid, const GemvArgs& a, hipStream_t st) {
  if (nw == 8) {
    if (mt == 1) launch_skinny_t<DK, T, 1, 8>(epi, grid, a, st);
    else if (mt == 2) launch_skinny_t<DK, T, 2, 8>(epi, grid, a, st);
    else if (mt == 3) launch_skinny_t<DK, T, 3, 8>(epi, grid, a, st);
    else launch_skinny_t<DK, T, 4, 8>(epi, grid, a, st);
  } else {
    if (mt == 1) launch_skinny_t<DK, T, 1, 4>(epi, grid, a, st);
    else if (mt == 2) launch_skinny_t<DK, T, 2, 4>(epi, grid, a, st);
    else if (mt == 3) launch_skinny_t<DK, T, 3, 4>(epi, grid, a, st);
    else launch_skinny_t<DK, T, 4, 4>(epi, grid, a, st);
  }
}
template <int DK>
void launch_skinny_dk(bool bf16, int mt, int nw, int epi, dim3 grid, const GemvArgs& a0, hipStream_t st, bool fine) {
  GemvArgs a = a0;
  a.nib_mask = 0x000F000Fu;
  a.nib_magic = bf16 ? Raw<BF16>::k4 : Raw<F16>::k4;
  if constexpr (DK == DK_LUT4) {
    if (bf16 && fine) {                        // 65 rows and up: three row tiles, or four in 8 waves
      if (mt == 4) launch_skinny_t<DK, BF16, 4, 8, true>(epi, grid, a, st);
      else if (nw == 8) launch_skinny_t<DK, BF16, 3, 8, true>(epi, grid, a, st);
      else launch_skinny_t<DK, BF16, 3, 4, true>(epi, grid, a, st);
      return;
    }
  }
  if (bf16) launch_skinny_mt<DK, BF16>(mt, nw, epi, grid, a, st);
  else launch_skinny_mt<DK, F16>(mt, nw, epi, grid, a, st);
}

}  // namespace illm
