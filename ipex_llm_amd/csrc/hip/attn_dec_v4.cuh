// Decode attention v4: a workgroup streams a (sequence, kv head)'s keys, whole rows throughout (included by attention.cuh).
//
// attn_dec_v3.cuh gives a wave one 32-key tile and merges the workgroups' partials: right for a few pairs of sequence and
// kv head, where the chain of round trips is the time (9 us of which the bytes of one sequence of 1024 keys take 1), but with
// many pairs the workgroups come in rounds that each pay that chain again, and the merge -- partials to memory, a ticket, the
// partials read back -- costs 2 to 3 us for sums that one workgroup could have kept.  Its variant of several tiles per wave
// asks for K as fragments (16 rows of 64 bytes a load: four times the address unit's time), for want of registers.  Here:
//   * NW = 8 (4) waves take the 32 NW-key tiles of the pair in turn (workgroup s of S: tiles s, s + S, ..., or 1 << v4_row
//     keys in a row, and those past the sequence's end leave at once); the waves meet once, at the end.  One workgroup: it
//     writes the result itself, no partials, no ticket, no second launch;
//   * a tile's 32 rows of K and of V are 8 KB in a row each: 16 loads of 1 KB through a buffer descriptor whose range ends
//     with the tile's keys (rows past them are zeros), the next tile's requested as soon as this one's are in the wave's LDS
//     rows, so 16 KB a wave and 128 KB a CU are in flight beside the products; 201 registers, 8 waves a CU.  Two tiles
//     ahead spilled, and a spill's reload waits for every request before it (1 x 8000, S = 16: 19.0 instead of 15.0 us);
//   * descriptors are scalar: the blocks of 64 tiles of a wave are one load, a lane each, read by lane;
//   * the new token's rows (pre-rotated q / k) go to the cache and, from LDS, over the tile's stale row.
// Bound by memory from some 30 MB on (48 sequences of up to 700 tokens, 101 MB: 25.3 us, 4.0 TB/s; 4.3 TB/s at 187 MB),
// below by the chain: 2.1 us a tile and wave with 8 waves on the CU, 1.3 with four.
#pragma once
#include <algorithm>
#include <climits>

namespace illm {

// RQ 3: the qkv product's f32 slabs [ks, B, ld], bias and rotation as in rope_kv.hip, the same bits.  An item is dims d, d + 1
// and their partners D / 2 on of one head, for a thread; q goes to LDS for all waves, k and v there and, from the workgroup
// that has the new key's tile, to the cache.  Only where a workgroup's tiles are in a row (attn_slabs_takes), so that all but
// the longest sequences have one: each of a pair rotates the same rows.  The rope launch takes 5.2 us
// for 0.5 us of bytes; this prologue, its loads ahead of the first tile's, 1.5 to 3: us a step, launch / this, Llama-3-8B 17 x 1024
// tokens 2374 / 2305, 24 x 600 2342 / 2262, 33 x 300 2597 / 2508, 64 x 900 asym_int4 4071 / 3980, 64 x 128 3013 / 2900, Qwen2.5-7B
// fp8_e5m2 40 x 500 2906 / 2868, 20 x 150 sym_int4 2082 / 1984, nf4 12 x 180 2680 / 2640.  (The block of the new key asked for behind
// the tile's requests, so that its wait is also for them: 0.7 us a launch more.)
template <typename T, int D>
struct V4Slabs {
  float2 f[4][2];                                                 // the first four slabs, in flight together
  uint16_t bias[2][2];
  float4 cs;
  int64_t pos, off;
  int hh, d, col, blk;
  __device__ void load(const AttnDecodeArgs& a, int b, int kvh, int group, int item) {
    const int it = min(item, (group + 2) * (D / 4) - 1);          // (past the last: not stored)
    hh = it / (D / 4) - group;                                    // below 0: a query head, 0: k, 1: v
    d = it % (D / 4) * 2;
    col = (hh < 0 ? kvh * group + hh + group : a.Hq + hh * a.Hkv + kvh) * D + d;
    pos = a.rq_pos[b];
    off = a.rq_pos_offset ? a.rq_pos_offset[b] : 0;
    const float* p = a.rq_part + (size_t)b * a.rq_ld + col;
    const size_t slab = (size_t)a.B * a.rq_ld;
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int h = 0; h < 2; h++) f[s][h] = *(const float2*)(p + min(s, a.rq_slabs - 1) * slab + h * (D / 2));
    const uint16_t* bp = a.rq_bias ? a.rq_bias + col : (const uint16_t*)p;
#pragma unroll
    for (int h = 0; h < 2; h++) bias[h][0] = bp[h * (D / 2)], bias[h][1] = bp[h * (D / 2) + 1];
  }
  // what the position leads to: ahead of the keys' requests, a wait is for all that was asked before
  __device__ void follow(const AttnDecodeArgs& a, int b) {
    cs = *(const float4*)(a.rq_cos_sin + ((size_t)pos * (D / 2) + d) * 2);
    const int64_t k = pos - off;
    const bool in = k >= 0 && k < (int64_t)a.max_blocks * a.bs;
    blk = a.block_tables[(size_t)b * a.max_blocks + (in ? (uint32_t)k / (uint32_t)a.bs : 0u)];
    blk = in ? blk : INT_MAX;
  }
  __device__ int key(int len) const {                             // index of the new key, -1: not among the len of the call
    const int64_t k = pos - off;
    return __builtin_amdgcn_readfirstlane(k >= 0 && k < len ? (int)k : -1);
  }
  __device__ void finish(const AttnDecodeArgs& a, int b, int kvh, int item, bool append, uint16_t (*q)[D], uint16_t (*kv)[D]) const {
    const int group = a.Hq / a.Hkv;
    if (item >= (group + 2) * (D / 4)) return;
    float v[2][2] = {};
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        v[h][0] = s < a.rq_slabs ? v[h][0] + f[s][h].x : v[h][0];
        v[h][1] = s < a.rq_slabs ? v[h][1] + f[s][h].y : v[h][1];
      }
    for (int s = 4; s < a.rq_slabs; s++) {
      const float* p = a.rq_part + ((size_t)s * a.B + b) * a.rq_ld + col;
      for (int h = 0; h < 2; h++) v[h][0] += p[h * (D / 2)], v[h][1] += p[h * (D / 2) + 1];
    }
    auto rnd = [](float x) { return to_f32<T>(from_f32<T>(x)); };
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int e = 0; e < 2; e++) {
        if (a.rq_bias) v[h][e] += to_f32<T>(bias[h][e]);
        v[h][e] = rnd(v[h][e]);
      }
    if (hh < 1) {                                                 // cos and sin in T, each product rounded to it
      const float osc = hh < 0 ? a.rq_qscale : 1.f;
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const float c = rnd(e ? cs.z : cs.x), sn = rnd(e ? cs.w : cs.y), x0 = v[0][e], x1 = v[1][e];
        v[0][e] = (rnd(x0 * c) - rnd(x1 * sn)) * osc;
        v[1][e] = (rnd(x1 * c) + rnd(x0 * sn)) * osc;
      }
    }
    const uint32_t o[2] = {pack2<T>(v[0][0], v[0][1]), pack2<T>(v[1][0], v[1][1])};
    uint16_t* l = hh < 0 ? q[hh + group] : kv[hh];
#pragma unroll
    for (int h = 0; h < 2; h++) *(uint32_t*)(l + d + h * (D / 2)) = o[h];
    if (hh < 0 || !append) return;
    const bool oob = blk >= a.num_blocks;
    if (oob) kerr(a.err, ERR_SLOT);
    if (blk < 0 || oob) return;                                   // a padding row
    uint16_t* c = (uint16_t*)(hh == 0 ? a.k_cache : a.v_cache) + (((size_t)blk * a.Hkv + kvh) * a.bs + (uint32_t)(pos - off) % (uint32_t)a.bs) * D + d;
#pragma unroll
    for (int h = 0; h < 2; h++) *(uint32_t*)(c + h * (D / 2)) = o[h];
  }
};

// ROW: a workgroup has 1 << v4_row keys in a row.  A kernel of its own: with both in one, tiles in turn took 0.2 to 0.6 us more
template <typename T, int D, int NW, int RQ, bool FUSE, bool ROW>
__global__ void __launch_bounds__(64 * NW, 2) attn_decode_v4_kernel(const AttnDecodeArgs a) {
  constexpr int SK = V3_KPW * NW;                  // keys of a tile
  constexpr int KSTEP = D / 32, DT = D / 16, VU = D / 8, KPJ = 64 / VU, VJ = V3_KPW / KPJ;
  static_assert(D == 64 || D == 128, "v4: head_dim 64 / 128");
  static_assert(RQ == 0 || ((RQ == 2 || RQ == 3) && D == 128), "v4: q from memory, pre-rotated or as slabs with head_dim 128");
  __shared__ __attribute__((aligned(16))) uint16_t vl[V3_KPW * NW * D];   // a wave's 32 K rows, then its V rows; the sums at the end
  __shared__ __attribute__((aligned(16))) uint16_t fresh[RQ != 0 ? 2 : 1][D];   // the new token's k and v rows
  __shared__ __attribute__((aligned(16))) uint16_t qrot[RQ == 3 ? 16 : 1][D];
  __shared__ float smx[NW][16], sml[NW][16];
  __shared__ int s_last;
  // (ROW: the workgroups of a pair far apart.  Beside each other, all first ones, the only ones of most sequences, fall to the
  // same XCDs: 31 x 500 and 1 x 16000 tokens 110 us instead of 52)
  const int split = ROW ? blockIdx.z : blockIdx.x, S = ROW ? gridDim.z : gridDim.x;
  const int kvh = ROW ? blockIdx.x : blockIdx.y, b = ROW ? blockIdx.y : blockIdx.z;
  const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = a.Hq / a.Hkv, R = group * a.Tq;
  const int kfirst = ROW ? split << a.v4_row : split * SK, kw0 = kfirst + V3_KPW * wv, step = ROW ? SK : S * SK;

  // blocks are a power of two tokens long but for odd configurations: no division on the way to an address
  const int bsh = (a.bs & (a.bs - 1)) == 0 ? 31 - __clz(a.bs) : -1;
  auto block_of = [&](uint32_t k) { return bsh >= 0 ? k >> bsh : k / (uint32_t)a.bs; };
  auto row_of = [&](uint32_t k) { return bsh >= 0 ? k & (uint32_t)(a.bs - 1) : k % (uint32_t)a.bs; };
  // ---- the length and the blocks of the wave's first 64 tiles, in flight together
  int len = a.seq_lens[b];
  auto entries = [&](int j) {                                     // lane: block of tile j + lane
    const uint32_t k = min((uint32_t)kw0 + (uint32_t)(j + lane) * (uint32_t)step, (uint32_t)a.max_blocks * (uint32_t)a.bs - 1u);
    return a.block_tables[(size_t)b * a.max_blocks + block_of(k)];
  };
  int ent = entries(0);                          // (of tiles j & ~63 ..)
  const int row = r16 < R ? r16 : 0;
  const int t = row / group, h = kvh * group + row % group;
  const V3Rope<T, D, true> rp(a, b, g, RQ == 2);
  typename V3Rope<T, D, true>::Raw qraw;
  uint4 qf[KSTEP];
  V4Slabs<T, D> sl;
  if constexpr (RQ == 3) {
    sl.load(a, b, kvh, group, threadIdx.x);
  } else if constexpr (RQ != 0) {
    if constexpr (D == 128) rp.load(h * D, qraw);
  } else {
    const uint16_t* qr = a.q + (((size_t)b * a.Tq + t) * a.Hq + h) * D;
#pragma unroll
    for (int s = 0; s < KSTEP; s++) qf[s] = *(const uint4*)(qr + 32 * s + 8 * g);
  }
  if ((int64_t)len > (int64_t)a.max_blocks * a.bs || (int64_t)a.nsplit * SPLIT < len) {
    if (split == 0 && threadIdx.x == 0) kerr(a.err, ERR_SEQ_LEN);
    len = min(min(len, a.max_blocks * a.bs), a.nsplit * SPLIT);
  }
  len = __builtin_amdgcn_readfirstlane(len);
  const int nsg = FUSE && ROW ? max(1, min(S, (len + (1 << a.v4_row) - 1) >> a.v4_row)) : S;
  if (split >= nsg) return;                      // (all of the workgroup; it is not among those that the ticket counts)
  const size_t prow = (((size_t)b * a.Hq + h) * a.Tq + t) * a.nsplit + split;
  const int win0 = a.sliding_window > 0 ? len - a.Tq - a.sliding_window : -1;   // keys up to here: no row sees them
  const int kend = ROW ? min(len, kfirst + (1 << a.v4_row)) : len, nt = kw0 < kend ? (kend - kw0 + step - 1) / step : 0;
  // (a window: the wave's first tile with a key in it)
  const int j0 = ROW && win0 - (V3_KPW - 1) >= kw0 ? min(nt, (win0 - (V3_KPW - 1) - kw0) / step + 1) : 0;
  if (j0 >= 64) ent = entries(j0 & ~63);

  // ---- tile j of the wave: keys that can be seen (0: none, a bad block, past the window) and where they start
  auto tile_at = [&](int j, int& kw, size_t& base, int& blk) {
    kw = kw0 + j * step;
    blk = __builtin_amdgcn_readlane(ent, j & 63);
    int n = min(V3_KPW, len - kw);
    if (kw + n - 1 <= win0) n = 0;
    if (n > 0 && bad_block(blk, a.num_blocks)) {
      if (lane == 0) kerr(a.err, ERR_BLOCK_ID);
      n = 0;
    }
    base = n > 0 ? (((size_t)blk * a.Hkv + kvh) * a.bs + row_of(kw)) * D * 2 : 0;
    return n;
  };
  // rows past the tile's keys are out of the descriptor's range: zeros
  auto load = [&](const uint8_t* cache, size_t base, int n, uint4 (&r)[VJ]) {
    const uint64_t p = (uint64_t)(cache + base);                  // the wave's: scalar registers, no loop over lanes
    const uint64_t ps = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(p >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)p);
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)ps, 0, __builtin_amdgcn_readfirstlane(n) * D * 2, 0x00020000);
#pragma unroll
    for (int j = 0; j < VJ; j++)
      r[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, lane * 16 + j * 1024, 0, 0));
  };
  auto store = [&](const uint4 (&r)[VJ], int kv, int at) {       // at: row that the new token's replaces (-1: none)
    int ln = lane;
    asm volatile("" : "+v"(ln));                 // addresses are recomputed per tile: hoisted, they spill
#pragma unroll
    for (int j = 0; j < VJ; j++) *(uint4*)(vl + pf_off<D>(V3_KPW * wv + j * KPJ + ln / VU, ln % VU)) = r[j];
    if (RQ != 0 && at >= 0) {
      v3_lds_order();
      if (lane < VU) *(uint4*)(vl + pf_off<D>(V3_KPW * wv + at, lane)) = *(const uint4*)(fresh[kv] + 8 * lane);
    }
  };

  if constexpr (RQ == 3) sl.follow(a, b);                        // (the position came with the length)
  uint4 kc[VJ], vc[VJ];
  auto request = [&](int j, uint4 (&k)[VJ], uint4 (&v)[VJ]) {
    int kw, blk;
    size_t base;
    const int n = tile_at(j, kw, base, blk);
    load(a.k_cache, base, n, k);
    load(a.v_cache, base, n, v);
  };
  if (j0 < nt) request(j0, kc, vc);

  // ---- the new token's rows (RQ): the wave whose last tile ends the sequence appends them and uses them from LDS
  const int newest = RQ == 3 ? sl.key(len) : len - 1;             // (slabs: -1, not among the keys)
  const bool mine = ROW ? max(newest, 0) >> a.v4_row == split : newest / SK % S == split;   // this workgroup's
  const bool holds_new = RQ != 0 && nt > 0 && newest >= 0 && mine && newest % SK / V3_KPW == wv;
  if constexpr (RQ == 3) {
    for (int it = threadIdx.x;;) {
      sl.finish(a, b, kvh, it, !ROW || mine, qrot, fresh);
      if ((it += NW * 64) >= (group + 2) * (D / 4)) break;
      sl.load(a, b, kvh, group, it);
      sl.follow(a, b);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < KSTEP; s++) qf[s] = *(const uint4*)(qrot[row] + 32 * s + 8 * g);
  } else if constexpr (RQ != 0) {
    const int d0 = 8 * (lane % VU);
    float4 k0, k1, v0, v1;
    uint4 nb;
    if (holds_new) {
      rp.vload((a.Hq + kvh) * D + d0, k0, k1, nb);
      rp.vload((a.Hq + a.Hkv + kvh) * D + d0, v0, v1, nb);
    }
    {
      float v[KSTEP][8];
      typename V3Rope<T, D, true>::CS cs;
      rp.vals(qraw, v);
      rp.frags(h * D, v, cs, a.rq_qscale, qf);
    }
    if (holds_new) {
      const float rsv = rp.rs();
      float kv[8], vv[8];
      rp.vals8(k0, k1, nb, rsv, kv);
      rp.vals8(v0, v1, nb, rsv, vv);
      const uint4 kn = make_uint4(pack2<T>(kv[0], kv[1]), pack2<T>(kv[2], kv[3]), pack2<T>(kv[4], kv[5]), pack2<T>(kv[6], kv[7]));
      const uint4 vn = make_uint4(pack2<T>(vv[0], vv[1]), pack2<T>(vv[2], vv[3]), pack2<T>(vv[4], vv[5]), pack2<T>(vv[6], vv[7]));
      const int blk = a.block_tables[(size_t)b * a.max_blocks + block_of(len - 1)];
      if (lane < VU) {
        *(uint4*)(fresh[0] + d0) = kn;
        *(uint4*)(fresh[RQ != 0 ? 1 : 0] + d0) = vn;
        if (!bad_block(blk, a.num_blocks)) {
          const size_t crow = (((size_t)blk * a.Hkv + kvh) * a.bs + row_of(len - 1)) * D + d0;
          *(uint4*)((uint16_t*)a.k_cache + crow) = kn;
          *(uint4*)((uint16_t*)a.v_cache + crow) = vn;
        }
      }
    }
  }
  if (r16 >= R)
#pragma unroll
    for (int s = 0; s < KSTEP; s++) qf[s] = make_uint4(0, 0, 0, 0);

  const int qpos = len - a.Tq + t;
  const int win = a.sliding_window > 0 ? qpos - a.sliding_window : -1;
  const float slope = a.alibi && r16 < R ? a.alibi[h] : 0.f;
  float m = -INFINITY, l = 0.f;                  // row r16: maximum; sum over this lane's keys
  f32x4 o[DT];
#pragma unroll
  for (int d = 0; d < DT; d++) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto tile = [&](int j, uint4 (&k)[VJ], uint4 (&v)[VJ]) __attribute__((always_inline)) {
    int kwc, blk;
    size_t base;
    const int nvis = tile_at(j, kwc, base, blk);
    const int at = holds_new && j == (RQ == 3 ? (newest - (ROW ? kfirst : 0)) / SK : nt - 1) && nvis > 0 ? newest - kwc : -1;
    v3_lds_order();
    store(k, 0, at);
    v3_lds_order();
    uint4 kf[2][KSTEP];
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
      for (int s = 0; s < KSTEP; s++) kf[kt][s] = *(const uint4*)(vl + pf_off<D>(V3_KPW * wv + kt * 16 + r16, 4 * s + g));
    v3_lds_order();
    store(v, RQ != 0 ? 1 : 0, at);
    v3_lds_order();
    if (j + 1 < nt) {
      if (((j + 1) & 63) == 0) ent = entries(j + 1);
      request(j + 1, k, v);
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- S^T tiles: lane holds (key = 16 kt + 4 g + i, row = r16)
    f32x4 st[2];
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KSTEP; s++) acc = mfma16<T>(kf[kt][s], qf[s], acc);
      st[kt] = acc;
    }
    const int klim = min(nvis, qpos - kwc + 1);                   // keys kk < klim are visible
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
      for (int i = 0; i < 4; i++) st[kt][i] *= a.scale;
    if (a.softcap > 0.f) {
#pragma unroll
      for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int i = 0; i < 4; i++) st[kt][i] = a.softcap * tanhf(st[kt][i] / a.softcap);
    }
    if (a.alibi) {
#pragma unroll
      for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int i = 0; i < 4; i++) st[kt][i] += slope * (float)(kwc + kt * 16 + 4 * g + i);
    }
    float mt = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int kk = kt * 16 + 4 * g + i;
        const bool ok = r16 < R && kk < klim && kwc + kk > win;
        st[kt][i] = ok ? st[kt][i] : -INFINITY;
        mt = fmaxf(mt, st[kt][i]);
      }
    mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    const float mn = fmaxf(m, mt);
    const float f = m == -INFINITY ? 0.f : __expf(m - mn);        // nothing summed yet: l and o are 0
    m = mn;
    l *= f;
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
      for (int i = 0; i < 4; i++) o[d][i] *= f;
    // ---- P (T precision, as the MFMA consumes it)
    uint32_t pk[2][2];
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      float p[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        p[i] = m == -INFINITY ? 0.f : __expf(st[kt][i] - m);
        l += p[i];
      }
      pk[kt][0] = pack2<T>(p[0], p[1]);
      pk[kt][1] = pack2<T>(p[2], p[3]);
    }
    // ---- O^T += V^T P^T over the tile's 32 keys
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int row0 = V3_KPW * wv + 4 * (ln >> 4) + ((ln & 15) >> 2), row1 = row0 + 16;
    const uint4 pb = make_uint4(pk[0][0], pk[0][1], pk[1][0], pk[1][1]);
#pragma unroll
    for (int d = 0; d < DT; d++) {
      const int col = 16 * d + 4 * (ln & 3);
      const uint2 v0 = ds_read_tr16(vl + pf_off<D>(row0, col >> 3) + (col & 7));
      const uint2 v1 = ds_read_tr16(vl + pf_off<D>(row1, col >> 3) + (col & 7));
      o[d] = mfma16<T>(make_uint4(v0.x, v0.y, v1.x, v1.y), pb, o[d]);
    }
  };
  for (int j = j0; j < nt; j++) tile(j, kc, vc);

  // ---- merge the waves: one common maximum, every wave's sums scaled to it
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (g == 0) smx[wv][r16] = m;
  __syncthreads();
  float M = m;
#pragma unroll
  for (int w = 0; w < NW; w++) M = fmaxf(M, smx[w][r16]);
  const float f = m == -INFINITY ? 0.f : __expf(m - M);
  if (g == 0) sml[wv][r16] = l * f;
  float* ob = (float*)vl;                        // [NW][DT][64] float4: wave w's own rows of vl
#pragma unroll
  for (int d = 0; d < DT; d++)
    *(float4*)(ob + ((size_t)(wv * DT + d) * 64 + lane) * 4) =
        make_float4(o[d][0] * f, o[d][1] * f, o[d][2] * f, o[d][3] * f);
  __syncthreads();
  if (r16 < R) {
    float L = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) L += sml[w][r16];
    const float inv = L > 0.f ? 1.f / L : 0.f;
    float* po = a.part_o + prow * D + 4 * g;
#pragma unroll
    for (int d = 0; d < DT; d++) {
      if (d % NW != wv) continue;
      float4 s4 = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int w = 0; w < NW; w++) {
        const float4 u = *(const float4*)(ob + ((size_t)(w * DT + d) * 64 + lane) * 4);
        s4.x += u.x; s4.y += u.y; s4.z += u.z; s4.w += u.w;
      }
      if (nsg == 1) {
        uint16_t* out = a.out + (((size_t)b * a.Tq + t) * a.Hq + h) * D + 16 * d + 4 * g;
        *(uint2*)out = make_uint2(pack2<T>(s4.x * inv, s4.y * inv), pack2<T>(s4.z * inv, s4.w * inv));
      } else if constexpr (FUSE) {
        st16_sc1(a.part_o, (size_t)(po - a.part_o) + 16 * d, s4);
      } else {
        *(float4*)(po + 16 * d) = s4;
      }
    }
    if (nsg > 1 && wv == 0 && g == 0) {
      if constexpr (FUSE) st8_sc1(a.part_ml + prow * 2, M, L);
      else *(float2*)(a.part_ml + prow * 2) = make_float2(M, L);
    }
  }
  if (nsg == 1) {
    if constexpr (RQ == 2) {
      // every wave has read its columns of the qkv sums: zero for the next layer's adds
      float* pr = (float*)a.rq_part + (size_t)b * a.rq_ld;
      for (int i = threadIdx.x * 4; i < (group + 2) * D; i += NW * 64 * 4) {
        const int hh = i / D, col = hh < group ? (kvh * group + hh) * D : (a.Hq + (hh - group) * a.Hkv + kvh) * D;
        *(float4*)(pr + col + i % D) = make_float4(0.f, 0.f, 0.f, 0.f);
      }
    }
    return;
  }
  if constexpr (FUSE) {
    // ---- the last workgroup of (b, kvh) to arrive merges every split
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's write-through stores are done
    __syncthreads();
    if (threadIdx.x == 0) {
      int* ctr = a.v3_counters + (size_t)b * a.Hkv + kvh;
      const int prev = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_last = prev == nsg - 1;
      if (s_last) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!s_last) return;
    v3_combine<T, true>(a, b, kvh, nsg, threadIdx.x, NW * 64);
  }
}

// waves of a workgroup and workgroups of a (sequence, kv head); groups 0: attn_dec_v3.cuh.  A function of batch, kv heads
// and split grid only, so a verify reduces as a one-token step of the same batch does -- one whose q lies in memory, rotated
// ahead or as slabs; steps that rotate in the attention stay on attn_dec_v3.cuh.  Sequences of half to all of these
// keys, 32 / 8 heads, us, the kernels of attn_dec_v3.cuh / this:
//   * from 136 pairs on one workgroup each, 8 waves while they are one per CU, else 4 (two per CU): 18 x 1024 29.3 / 19.8, 20 x
//     800 22.1 / 16.5, 24 x 1024 24.5 / 19.8, 32 x 600 21.6 / 16.9, 48 x 700 31.9 / 25.3 (8 waves 28.6), 64 x 256 19.0 / 14.5,
//     100 x 600 52.4 / 43.1, 28 x 2100 45.9 / 40.5 -- while the longest sequence that the grid is made for is no more than 10
//     tiles a wave (2560, 1280 keys).  Beyond, 1024 keys in a row each, 2048 .. where that makes more than 8192 workgroups or 32
//     a pair: with one long sequence among short ones a single workgroup streamed it while the others were done.  us with the rope
//     launch or the slabs here, attn_dec_v3.cuh / one workgroup / this: 31 x 500 and 1 x 16000 84 / 151 / 56, 39 and one 116 / 213 / 61,
//     56 x 300 and 8 x 8000 117 / 115 / 76, 16 x 500 and 1 x 16000 88 / 148 / 37, 63 x 200 and 1 x 30000 353 / 383 / 87, 47 x 300 and 1 x
//     4000 47 / 63 / 38, 39 x 300 and 1 x 2000 34 / 38 / 29, 28 / 4 heads 39 x 500 and 1 x 16000 105 / 148 / 49, a window of 4096 in
//     32 x 16000 295 / 145 / 126.  Up to 10 tiles one workgroup is no later than attn_dec_v3.cuh with those, either (17 x 300 and 1 x
//     2000 36 / 27, 31 and one 30 / 28), and ahead where the lengths are alike: 28 x 2100 48 / 42 / 45, 50 x 1200 55 / 45 / 47.  Above,
//     what rows of keys cost there: 20 x 3000 53 / 45 / 47, 17 x 3500 48 / 47 / 45, 24 x 4000 78 / 64 / 68, 40 x 1500 51 / 47 / 45, 33 x
//     2500 71 / 69 / 57, 64 x 2000 91 / 81 / 86, 32 x 8000 170 / 161 / 166, 28 / 4 heads 40 x 3000 51 / 45 / 47, 64 x 3000 76 / 64 / 73;
//   * fewer pairs of more than 8 sequences, so few keys that the merge is most of the time: 16 x 256 12.2 / 9.1, 16 x 800 (q
//     pre-rotated) 22.8 / 16.1, (from memory) 16.1 / 14.9.  Up to 8 sequences not, however many kv heads, though most are ahead (q pre-rotated 1 x 128 8.4 /
//     6.0, 8 x 400 10.8 / 10.1, 8 x 600 12.1 / 11.8, from memory 1 x 128 6.6 / 4.9, 32 kv heads 4 x 100 8.4 / 6.3, 5 x 250 10.3 / 8.4, 8 x 436 16.6 / 15.4; 1 x 400 even, 1 x 600
//     8.9 / 9.2, 32 kv heads 4 x 250 9.5 / 10.2, 4 x 1000 16.7 / 17.2): there, steps that rotate in the attention keep attn_dec_v3.cuh,
//     and p is rounded beside its wave's maximum here and its workgroup's there: 1.9e-3 between the two over 70 keys, and the
//     tokens of two ranks parted from those of one at a tie.  From `few` keys on the two do part (32 kv heads 5 x 950 22.5 / 18.4);
//   * long ones, where one tile a wave takes rounds: 4 waves and as many workgroups as make 512, at most 16 (32) a pair: 1 x
//     4200 14.8 / 11.8, 3 x 20000 45.7 / 42.0, 4 x 3000 19.3 / 16.2, 5 x 4200 23.5 / 20.2, 8 x 2400 31.0 / 20.5, 10 x 4200 35.0 /
//     33.7, 16 x 2000 41.0 / 27.0; from 64, 80 and 112 pairs on at fewer keys: 8 x 1024 15.0 / 14.0, 10 x 1300 17.1 / 16.9, 12 x
//     1300 23.2 / 17.8, 14 x 1024 22.8 / 17.9, 16 x 1024 24.2 / 18.7.  Between, one tile a wave has the shorter chain: 1 x 1100
//     9.1 / 9.3, 4 x 1500 12.7 / 12.8, 6 x 1300 13.8 / 13.8, 8 x 700 12.6 / 12.9, 12 x 1024 16.5 / 17.1.
struct V4Plan {
  int nw, groups, row;                           // row > 0: 1 << row keys in a row for each of the groups (4 waves)
};
inline V4Plan v4_plan(int B, int Hkv, int nsplit) {
  static const bool off = getenv("ILLM_ATTN_V3_NW") || getenv("ILLM_ATTN_V3_TILES") || (getenv("ILLM_ATTN_V4") && atoi(getenv("ILLM_ATTN_V4")) == 0);
  if (off) return {0, 0};                        // a forced form of attn_dec_v3.cuh (A/B runs)
  const long pairs = (long)B * Hkv, keys = (long)nsplit * SPLIT;
  const long few = pairs >= 136 ? 576 : pairs >= 112 ? 960 : pairs >= 80 ? 1152 : pairs >= 64 ? 1024 : 1920;
  if (B <= 8 && keys < few) return {0, 0};
  if (pairs >= 136) {
    const int nw = pairs <= 256 ? 8 : 4;
    if (keys <= 10 * V3_KPW * nw) return {nw, 1, 0};
    const long most = std::max(8L, std::min(32L, 8192 / pairs));
    int row = 10;
    while (keys > most << row) row++;
    return {4, (int)((keys + (1L << row) - 1) >> row), row};
  }
  if (B > 8 && keys <= (pairs >= 112 ? 896 : pairs >= 64 ? 704 : 512)) return {keys <= 192 ? 4 : 8, 1};
  if (keys < few) return {0, 0};
  const long s = std::min({512 / pairs, pairs >= 16 || keys < 16384 ? 16L : 32L, keys / (4 * V3_KPW)});
  return {4, (int)s};
}

template <typename T, int D, int NW, int RQ, bool ROW>
static void launch_v4_nw(const AttnDecodeArgs& a, int S, hipStream_t st) {
  const dim3 grid = ROW ? dim3(a.Hkv, a.B, S) : dim3(S, a.Hkv, a.B);
  if (RQ == 3 ? ROW : S == 1 || a.v3_counters != nullptr) {
    if constexpr (RQ != 3 || ROW) hipLaunchKernelGGL((attn_decode_v4_kernel<T, D, NW, RQ, true, ROW>), grid, dim3(64 * NW), 0, st, a);
  } else if constexpr (RQ == 3) {
    if constexpr (!ROW) hipLaunchKernelGGL((attn_decode_v4_kernel<T, D, NW, RQ, false, ROW>), grid, dim3(64 * NW), 0, st, a);
  } else {
    hipLaunchKernelGGL((attn_decode_v4_kernel<T, D, NW, RQ, false, ROW>), grid, dim3(64 * NW), 0, st, a);
    hipLaunchKernelGGL((attn_combine_v3_kernel<T>), dim3(a.Hkv, a.B), dim3(256), 0, st, a, S);
  }
}

template <typename T, int D, int RQ>
static bool launch_v4(const AttnDecodeArgs& a0, hipStream_t st) {
  const V4Plan p = v4_plan(a0.B, a0.Hkv, a0.nsplit);
  if (p.groups == 0) return false;
  AttnDecodeArgs a = a0;
  a.v4_row = p.row;
  if (p.row > 0) launch_v4_nw<T, D, 4, RQ, true>(a, p.groups, st);
  else if (p.nw == 8) launch_v4_nw<T, D, 8, RQ, false>(a, p.groups, st);
  else launch_v4_nw<T, D, 4, RQ, false>(a, p.groups, st);
  return true;
}

}  // namespace illm
