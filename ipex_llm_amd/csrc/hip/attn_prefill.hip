// Prefill / long-query attention straight over the paged KV cache
// (flash-attention forward, causal, GQA).
//
// Reference ops: xe_addons.sdp_causal / sdp_fp8_causal / sdp_non_causal
// (SRC/transformers/models/common.py:271-286), gemma2_sdp_causal (softcap,
// sliding window; models/gemma2.py:133-155) and the vLLM-XPU context
// (chunked-prefill) attention (VLLM_PATCH csrc/xpu).  Used for prefill,
// chunked prefill over a cached prefix and speculative / lookup verification
// (query chunks too wide for the decode kernel).
//
// MI355X design (gfx950, wave64, v_mfma_f32_16x16x32 bf16/f16):
//   * workgroup = 4 waves = 64 query rows of one head; wave w owns rows
//     16w..16w+15.  Causal q-blocks are issued heaviest first;
//   * K/V tiles of 64 keys are read once per workgroup straight from the
//     paged cache (a 64-key tile never crosses a cache block, bs % 64 == 0)
//     into LDS as [key][D] rows with a 16-byte XOR swizzle, by LDS-DMA: the
//     next tile is in flight while the current one is computed, with no
//     register, conversion or LDS store in between;
//   * swapped QK^T: S^T = K Q^T (A = K rows from LDS by ds_read_b128, B = the
//     wave's Q rows kept in registers), so a lane holds 16 scores of ONE query
//     row: the online-softmax row max / sum is a register reduction plus two
//     shuffles;
//   * P V as O^T = V^T P^T: the B operand (P^T) is the lane's own scores
//     converted to 16-bit (key order of the C layout, no lane movement), the
//     A operand (V^T) comes from ds_read_b64_tr_b16 transposed reads of the
//     row-major V tile in exactly that key order;
//   * fp8 KV caches go through registers and are converted to 16-bit on the
//     way to LDS.
// What bounds it: up to a grid of two workgroups per CU, one tile's chain in a
// wave (QK^T and PV each read the tile at LDS speed, 512 cycles, with the
// softmax between them and the staging's wait and barrier after), not the
// products.  Out of that chain came: the block-id round trip of every tile (ids
// are read 64 at a time), the waits for the tile in flight that hipcc placed
// before the first product (for Q, for zeros at the sequence end and for fp8
// conversions beside the load), the LDS stores, and half of the vector
// instructions (scale in one fma with the maximum, addresses by xor, row maximum
// by lane swaps).  MI355X, 32 / 8 heads of 128, before -> after: 1024 rows 32.6 ->
// 25.6 us, 8 x 1024 115 -> 100, 200 rows behind 1800 keys 56 -> 42, 300 rows of
// 28 / 4 heads 12.8 -> 10.2, 1024 rows on an e5m2 cache 50 -> 31, the same error.
// Slower or no better: keys of a tile split over 8 waves (23.5 at 1024 rows, 141 at
// 8 x 1024), K and V half a tile apart with a second barrier (26.4, 99), the next
// tile but one in flight, wave priorities around the products.
#include <cstdlib>

#include "../common/quant_block.h"
#include "illm_device.h"
#include "kernels.h"
#include "lds_dma.h"

namespace illm {

constexpr int PF_KT = 64;      // keys per tile
constexpr int PF_QB = 64;      // query rows per workgroup

// 8 cache elements as they lie, and as 16-bit values
template <int KVF> struct pf_raw { typedef uint2 type; };
template <> struct pf_raw<0> { typedef uint4 type; };

template <typename T, int KVF>
__device__ __forceinline__ uint4 pf_cvt8(const typename pf_raw<KVF>::type& u, float scale) {
  if constexpr (KVF == 0) {
    return u;
  } else {
    float v[8];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const uint32_t w = i ? u.y : u.x;
      auto f0 = KVF == 1 ? __builtin_amdgcn_cvt_pk_f32_bf8(w, false) : __builtin_amdgcn_cvt_pk_f32_fp8(w, false);
      auto f1 = KVF == 1 ? __builtin_amdgcn_cvt_pk_f32_bf8(w, true) : __builtin_amdgcn_cvt_pk_f32_fp8(w, true);
      v[4 * i + 0] = f0[0] * scale;
      v[4 * i + 1] = f0[1] * scale;
      v[4 * i + 2] = f1[0] * scale;
      v[4 * i + 3] = f1[1] * scale;
    }
    return make_uint4(pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]), pack2<T>(v[4], v[5]), pack2<T>(v[6], v[7]));
  }
}

// max over the four lanes of a query row (lane ^ 16, ^ 32)
__device__ __forceinline__ float xmax(float v) {
  auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
  p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
}

// HP = query heads per wave that share one kv head (GQA): every K fragment
// read from LDS and every transposed V read feeds HP MFMAs.
template <typename T, int D, int KVF, int HP, bool SOFTCAP>
__global__ void __launch_bounds__(256, 2) attn_prefill_kernel(const AttnPrefillArgs a) {
  constexpr int EB = KVF == 0 ? 2 : 1;            // cache bytes per element
  constexpr int KSTEP = D / 32;                   // MFMA k-steps over the head dim (QK^T)
  constexpr int DT = D / 16;                      // 16-wide d tiles of O^T
  constexpr int UPT = PF_KT * D / 8 / 256;        // 8-element staging units per thread per tile
  constexpr int TB = PF_KT * D * 2;               // bytes of a K or V tile in LDS
  // double-buffered K / V tiles (K0, K1, V0, V1): the next tile is written while the current
  // one is read, one workgroup barrier per tile
  __shared__ __attribute__((aligned(16))) uint8_t lds[4 * TB];

  // causal work per query block grows with its index.  Block order: heaviest
  // query blocks of every (head, batch) first (longest-processing-time first
  // for the dynamic dispatch); when the whole grid is resident at once (<= 2
  // workgroups per CU: 64 KiB of LDS each) the second half runs the light
  // blocks in ascending order instead, so workgroups i and i + grid/2 (one CU)
  // pair up to the same total (T = 1024: every CU 17 tiles instead of up to 32)
  const int nqb = gridDim.x, nother = gridDim.y * gridDim.z;
  const int lin = blockIdx.x + nqb * (blockIdx.y + gridDim.y * blockIdx.z);
  const int rank = lin / nother, other = lin % nother;
  const int half = (nqb + 1) / 2;
  const int qb = (nqb * nother <= 512 && rank >= half) ? rank - half : nqb - 1 - rank;
  const int hh = other % gridDim.y, b = other / gridDim.y;
  const int kvh = hh % a.Hkv, h0 = kvh * (a.Hq / a.Hkv) + hh / a.Hkv * HP;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, r16 = lane & 15;
  const int L = a.seq_lens[b];
  const int Tq = a.Tq;
  const int p0 = L - Tq;                          // position of query row 0
  const int qrow = qb * PF_QB + wave * 16 + r16;  // this lane's query row (B operand column)
  const int qpos = p0 + min(qrow, Tq - 1);

  // key range of the workgroup
  const int wg_q0 = p0 + qb * PF_QB;
  const int wg_q_last = min(Tq - 1, qb * PF_QB + PF_QB - 1);
  const int kend = min(L, p0 + wg_q_last + 1);
  int kbeg = 0;
  if (a.sliding_window > 0) kbeg = max(0, wg_q0 - a.sliding_window + 1) & ~(PF_KT - 1);
  const int ntile = kend > kbeg ? (kend - kbeg + PF_KT - 1) / PF_KT : 0;

  if (ntile == 0) {                               // no key: zeros
#pragma unroll
    for (int j = 0; j < HP; j++)
#pragma unroll
      for (int d = 0; d < DT; d++)
        if (qrow < Tq)
          *(uint2*)(a.out + ((size_t)(b * Tq + qrow) * a.Hq + h0 + j) * D + 16 * d + 4 * g) = make_uint2(0u, 0u);
    return;
  }

  // Q fragments (B operand of S^T = K Q^T): row qrow, dims 32 s + 8 g .. + 7
  uint4 qf[HP][KSTEP];
#pragma unroll
  for (int j = 0; j < HP; j++) {
    const uint16_t* qp = a.q + ((size_t)(b * Tq + min(qrow, Tq - 1)) * a.Hq + h0 + j) * D;
#pragma unroll
    for (int s = 0; s < KSTEP; s++) qf[j][s] = *(const uint4*)(qp + 32 * s + 8 * g);
  }

  // block ids: one load of 64 (lane i: block bi + i), read out lane by lane; an id and its tile
  // loaded in one step are two round trips
  const int* table = a.block_tables + (size_t)b * a.max_blocks;
  const int blast = (kend - 1) / a.bs;
  int bi = kbeg / a.bs, boff = kbeg % a.bs, bl = 0;       // block, offset and lane of the next tile to load
  int bids = table[min(bi + lane, blast)];
  size_t src = 0;                                         // its place in the caches, bytes
  auto next_src = [&] {
    int blk = __builtin_amdgcn_readlane(bids, bl);
    if (bad_block(blk, a.num_blocks)) {                  // read block 0 instead, report
      kerr(a.err, ERR_BLOCK_ID);
      blk = 0;
    }
    src = (((size_t)blk * a.Hkv + kvh) * a.bs + boff) * D * EB;
    boff += PF_KT;
    if (boff == a.bs) {
      boff = 0;
      bi++;
      if (++bl == 64) {
        bids = table[min(bi + lane, blast)];
        bl = 0;
      }
    }
  };
  // staging of a tile into buffer t & 1: 16-bit caches by LDS-DMA (piece i of a wave: 1 KB of LDS, the swizzle
  // on the source side), fp8 through registers, converted on the way to LDS
  using raw = typename pf_raw<KVF>::type;
  raw kreg[KVF ? UPT : 1], vreg[KVF ? UPT : 1];
  constexpr int RP = 512 / D;                     // rows of 1 KB
  const int dr = wave * RP + lane / (D / 8);
  const uint32_t doff = 2 * pf_off<D>(dr, lane % (D / 8));
  auto load_tile = [&](int t) {
    next_src();
    if constexpr (KVF == 0) {
      const dma_rsrc rk = make_dma_rsrc(a.k_cache + src, TB), rv = make_dma_rsrc(a.v_cache + src, TB);
      const uint8_t* dst = lds + (t & 1) * TB + wave * 1024;
#pragma unroll
      for (int i = 0; i < TB / 4096; i++) lds_dma16(rk, lds_addr(dst + i * 4096), doff, i * 4096);
#pragma unroll
      for (int i = 0; i < TB / 4096; i++) lds_dma16(rv, lds_addr(dst + 2 * TB + i * 4096), doff, i * 4096);
    } else {
#pragma unroll
      for (int j = 0; j < UPT; j++) {
        const int u = tid + 256 * j;
        kreg[j] = *(const raw*)(a.k_cache + src + (size_t)u * 8 * EB);
        vreg[j] = *(const raw*)(a.v_cache + src + (size_t)u * 8 * EB);
      }
    }
  };
  // the tile is in LDS for every wave.  V slots past the sequence end hold stale bytes (possibly NaN
  // patterns): p = 0 times NaN would still poison the P V product, so they are zeroed
  auto finish_tile = [&](int t) {
    const int buf = t & 1, last = L - (kbeg + t * PF_KT);       // rows of the tile that count
    if constexpr (KVF == 0) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (last < PF_KT) {
        __syncthreads();
        for (int u = tid; u < PF_KT * D / 8; u += 256)
          if (u / (D / 8) >= last) *(uint4*)(lds + (2 + buf) * TB + u * 16) = make_uint4(0, 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int j = 0; j < UPT; j++) {
        const int u = tid + 256 * j;
        const int r = u / (D / 8), c = u % (D / 8);
        const uint4 vv = pf_cvt8<T, KVF>(vreg[j], a.v_scale);
        *(uint4*)(lds + buf * TB + 2 * pf_off<D>(r, c)) = pf_cvt8<T, KVF>(kreg[j], a.k_scale);
        *(uint4*)(lds + (2 + buf) * TB + 2 * pf_off<D>(r, c)) = r < last ? vv : make_uint4(0, 0, 0, 0);
      }
    }
    __syncthreads();
  };

  f32x4 o[HP][DT];
#pragma unroll
  for (int j = 0; j < HP; j++)
#pragma unroll
    for (int d = 0; d < DT; d++) o[j][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  float mrow[HP], lpart[HP];
#pragma unroll
  for (int j = 0; j < HP; j++) { mrow[j] = -INFINITY; lpart[j] = 0.f; }
  const float sc = a.scale;
  constexpr float kLog2e = 1.4426950408889634f;
  const float sc2 = a.scale * kLog2e;
  // scores in the exp2 domain: p = exp2(st * mul - m), one fma each; the maximum is taken before the
  // factor, so a factor that is not positive and normal (and the soft cap) goes on beforehand and mul is 1
  const bool pre = SOFTCAP || !(sc2 >= 1.17549435e-38f);
  const float mul = pre ? 1.f : sc2;

  // LDS bytes of the lane's fragments: K row r16, chunk 4 s + g; V (transposed reads: lane 4 q + p of the
  // 16-lane group g addresses row 4 g + q, columns 16 d + 4 p).  The swizzle is an xor of the chunk, so
  // chunks s and d are an xor of bits 6.. and 5.. of the first one's address
  const uint32_t ko = 2 * pf_off<D>(r16, g);
  const uint32_t vo = 2 * pf_off<D>(4 * g + (r16 >> 2), (r16 & 3) >> 1) + 8 * (r16 & 1) + 2 * TB;

  load_tile(0);
  __builtin_amdgcn_s_waitcnt(0x0f70);           // Q too: a wait for it inside the loop would be one for the tile in flight
  finish_tile(0);
  for (int t = 0; t < ntile; t++) {
    const uint32_t bo = (t & 1) * TB;
    // next tile in flight during the compute (its buffer: read last in tile t - 1, free since the barrier)
    if (t + 1 < ntile) load_tile(t + 1);
    const int kt0 = kbeg + t * PF_KT;
    // tiles wholly below every query row of the workgroup need no mask
    const bool full = kt0 + PF_KT - 1 <= wg_q0 && kt0 + PF_KT <= L && a.sliding_window <= 0;

    // ---- S^T = K Q^T : lane holds keys 16 kb + 4 g + i of query row r16
    f32x4 st[HP][4];
#pragma unroll
    for (int kb = 0; kb < 4; kb++) {
#pragma unroll
      for (int j = 0; j < HP; j++) st[j][kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KSTEP; s++) {
        const uint4 kf = *(const uint4*)(lds + ((ko + bo) ^ (s << 6)) + kb * 16 * D * 2);
#pragma unroll
        for (int j = 0; j < HP; j++) st[j][kb] = mfma16<T>(kf, qf[j][s], st[j][kb]);
      }
    }
    // ---- soft-cap, causal / window / length mask, online softmax
    uint32_t pk[HP][4][2];                         // P^T fragments, 16-bit pairs
#pragma unroll
    for (int j = 0; j < HP; j++) {
      // soft-cap is a template flag and the mask one uniform branch per tile:
      // a per-score branch (tanhf's own control flow inlined 16 times) split
      // the tile loop into ~100 basic blocks, so no MFMA / VALU interleaving
      // across them (rocprofv3: 3 SALU and 10 VALU per MFMA)
      if (pre) {
#pragma unroll
        for (int kb = 0; kb < 4; kb++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            if constexpr (SOFTCAP) st[j][kb][i] = a.softcap * tanhf(st[j][kb][i] * sc / a.softcap) * kLog2e;
            else st[j][kb][i] *= sc2;
          }
      }
      if (!full) {
        const int win = a.sliding_window > 0 ? qpos - a.sliding_window : -1;
#pragma unroll
        for (int kb = 0; kb < 4; kb++) {
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const int key = kt0 + 16 * kb + 4 * g + i;
            const bool ok = key <= qpos && key < L && key > win;
            st[j][kb][i] = ok ? st[j][kb][i] : -INFINITY;
          }
        }
      }
      float tmax = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < 4; kb++)
#pragma unroll
        for (int i = 0; i < 4; i++) tmax = fmaxf(tmax, st[j][kb][i]);
      tmax = xmax(tmax) * mul;
      // O rescale only when some row max of the wave moved (wave-uniform).  Nothing seen yet
      // (mrow = -inf): exp2(-inf) = 0 clears the empty O; a row still fully masked keeps alpha 1
      if (__builtin_amdgcn_ballot_w64(tmax > mrow[j]) != 0) {
        const float mnew = fmaxf(mrow[j], tmax);
        const float alpha = mnew == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(mrow[j] - mnew);
        mrow[j] = mnew;
        lpart[j] *= alpha;
#pragma unroll
        for (int d = 0; d < DT; d++) {
          o[j][d][0] *= alpha; o[j][d][1] *= alpha; o[j][d][2] *= alpha; o[j][d][3] *= alpha;
        }
      }
      const float msafe = mrow[j] == -INFINITY ? 0.f : mrow[j];     // a finite base for the exp2 below
#pragma unroll
      for (int kb = 0; kb < 4; kb++) {
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; i++) p[i] = __builtin_amdgcn_exp2f(fmaf(st[j][kb][i], mul, -msafe));   // masked: 0
        lpart[j] += (p[0] + p[1]) + (p[2] + p[3]);
        pk[j][kb][0] = pack2<T>(p[0], p[1]);
        pk[j][kb][1] = pack2<T>(p[2], p[3]);
      }
    }
    // ---- O^T += V^T P^T over two 32-key steps (key blocks 2 kk, 2 kk + 1)
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
#pragma unroll
      for (int d = 0; d < DT; d++) {
        const uint8_t* vp = lds + ((vo + bo) ^ (d << 5)) + kk * 32 * D * 2;
        const uint2 v0 = ds_read_tr16((const uint16_t*)vp), v1 = ds_read_tr16((const uint16_t*)(vp + 16 * D * 2));
        const uint4 va = make_uint4(v0.x, v0.y, v1.x, v1.y);
#pragma unroll
        for (int j = 0; j < HP; j++) {
          const uint4 pb = make_uint4(pk[j][2 * kk][0], pk[j][2 * kk][1], pk[j][2 * kk + 1][0], pk[j][2 * kk + 1][1]);
          o[j][d] = mfma16<T>(va, pb, o[j][d]);
        }
      }
    }
    if (t + 1 < ntile) finish_tile(t + 1);
  }

  // ---- normalise and store: lane holds O^T[16 d + 4 g + i][row r16]
#pragma unroll
  for (int j = 0; j < HP; j++) {
    float l = lpart[j];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (qrow >= Tq) continue;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    uint16_t* op = a.out + ((size_t)(b * Tq + qrow) * a.Hq + h0 + j) * D;
#pragma unroll
    for (int d = 0; d < DT; d++) {
      *(uint2*)(op + 16 * d + 4 * g) = make_uint2(pack2<T>(o[j][d][0] * inv, o[j][d][1] * inv),
                                                  pack2<T>(o[j][d][2] * inv, o[j][d][3] * inv));
    }
  }
}

template <typename T, int D, int HP, bool SC>
static void launch_pf_sc(const AttnPrefillArgs& a, hipStream_t st) {
  dim3 grid((a.Tq + PF_QB - 1) / PF_QB, a.Hq / HP, a.B);
  if (a.kv_fp8 == 1) hipLaunchKernelGGL((attn_prefill_kernel<T, D, 1, HP, SC>), grid, dim3(256), 0, st, a);
  else if (a.kv_fp8 == 2) hipLaunchKernelGGL((attn_prefill_kernel<T, D, 2, HP, SC>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((attn_prefill_kernel<T, D, 0, HP, SC>), grid, dim3(256), 0, st, a);
}

template <typename T, int D, int HP>
static void launch_pf_hp(const AttnPrefillArgs& a, hipStream_t st) {
  if (a.softcap > 0.f) launch_pf_sc<T, D, HP, true>(a, st);
  else launch_pf_sc<T, D, HP, false>(a, st);
}

template <typename T, int D>
static void launch_pf_d(const AttnPrefillArgs& a, hipStream_t st) {
  // HP = 2: two query heads of one kv head per wave, so every K fragment and
  // transposed V read from LDS feeds two MFMAs (even GQA group).  It halves
  // the grid, so it is taken when the halved grid still covers the chip
  // twice (2 workgroups per CU).  Measured on MI355X (32 / 8 heads, HP = 1 / 2):
  // T = 4096 200 / 170 us, B = 8 x 1024 125 / 100, 3 x 1024 50 / 44, T = 2048 (512
  // workgroups) 59 / 63, with a window of 500 39 / 33; T = 1024 (256) 26 / 34, so
  // HP = 1 there.  ILLM_PREFILL_HP=1/2 forces either.
  static const int hp_env = getenv("ILLM_PREFILL_HP") ? atoi(getenv("ILLM_PREFILL_HP")) : 0;
  const bool even = (a.Hq / a.Hkv) % 2 == 0;
  const long wg2 = (long)((a.Tq + PF_QB - 1) / PF_QB) * (a.Hq / 2) * a.B;
  const bool hp2 = even && (hp_env == 2 || (hp_env == 0 && wg2 >= 512));
  if (hp2) launch_pf_hp<T, D, 2>(a, st);
  else launch_pf_hp<T, D, 1>(a, st);
}

template <typename T>
static void launch_pf_t(const AttnPrefillArgs& a, hipStream_t st) {
  if (a.D == 64) launch_pf_d<T, 64>(a, st);
  else launch_pf_d<T, 128>(a, st);
}

void launch_attn_prefill(bool bf16, const AttnPrefillArgs& a, hipStream_t st) {
  if (bf16) launch_pf_t<BF16>(a, st); else launch_pf_t<F16>(a, st);
}

}  // namespace illm
