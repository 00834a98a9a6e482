// The attention kernel of the forward for fp32 operands, and its launch function.
#pragma once

#include "hbsa_common.h"

namespace hbsa {

// --------------------------------------------------------------------------------------
// fp32 kernel: fp32 operands, softmax and output, for callers that need the arithmetic of the reference's fp32 path (dot
// products without operand rounding, reference hbsattn/fwd_triton_auto_tile_size.py:205,225).
//
// A float is the sum of three bf16 numbers (8 + 8 + 8 significant bits, bf16 has fp32's exponents), so a product of two is the
// sum of nine products of bf16 numbers, which are exact and which the bf16 matrix instructions sum up in fp32.  Six of them are
// formed; the three left out are below 2^-26 of the product, a quarter of the rounding error of one fp32 operation.
// That is 6 x 32 cycles of a SIMD's matrix pipe for 32 x 32 x 16 multiplications against 8 x 64 of the fp32 instruction.
// Measured against the fp32 instructions throughout (v_mfma_f32_32x32x2_f32, 157 TFLOP/s at most): 4 sequences of 500 .. 3000
// tokens, 8 / 4 heads of 64, 64-key blocks, keep 0.5, causal, 110.8 -> 78.4 us; 2 x 1500 .. 2400, 16 / 2 heads of 32, 179 ->
// 123; 4 x 1200 .. 1700, 8 / 4 heads of 128, 178 -> 119; 40 calls of 10 .. 360 us 1.25 times as fast, none slower.  The
// error against 64-bit sums is 0.6 to 0.85 of what it was (relative error of the result 1.5e-7 for 2.7e-7 in the first of these).
// What bounds it now: products and vector instructions take about the same time (at D = 64, 32 keys and a wavefront 1536
// cycles of products, 1400 of softmax and splitting), two or three wavefronts a SIMD to cover one with the other.
//
// Same operand roles as the 16-bit kernel: S^T = K.Q^T with K rows from LDS and Q^T in registers, O^T += V^T.P^T with P^T
// taken from the S^T accumulator in place; K and V stand in LDS as three planes each, placed like the 16-bit kernel's tiles.
// What the split costs: K and V elements are split once a workgroup and tile on their way from registers to LDS (5.5 vector
// instructions an element and 1.5 times the bytes), Q once an item, P once a wavefront and tile.
// Tiles are KT keys in groups of 16, each group from any place of the sequence (blocks are multiples of 16 keys): blocks
// of 16 or 48 keys fill tiles like larger ones.  An item (kv head, q block, group of four wave slots) is cut into parts over its
// k blocks when there are few items (ItemParts), because a causal mask over ragged sequences makes the longest item several
// times the average and all of them are resident from the start.
//
// Infinities: an infinite element, or one that rounds to an infinite bf16, has a NaN among its parts, so a wavefront that
// met one (or a NaN) ends with a NaN among its sums, of the exponentials or of the output.  It then does its rows again with the
// fp32 matrix instructions (v_mfma_f32_32x32x2_f32) and operands straight from memory, and what an infinity gives is what fp32
// arithmetic gives.
// A 32x32x2 MFMA contracts over two indices, one per half of the wavefront; which two is free as long as both operands agree:
//   S: step (j, e), half g contracts over d = 8*j + 4*g + e, so a lane reads 4 consecutive floats of its K row per j;
//   PV: step i, half g contracts over key 8*(i/4) + 4*g + (i%4), which is exactly the key whose score the lane holds in
//      accumulator element i.
// --------------------------------------------------------------------------------------
template <int D>
struct F32Tile {
  static constexpr int RB = D * 2;                 // bytes of a row of a plane
  static constexpr int CPR = RB / 16;              // 16-byte chunks (8 elements) of it
  static constexpr int KT = D <= 32 ? 64 : 32;     // keys per tile
  static constexpr int GROUPS = KT / 16;
  static constexpr int PLANE = KT * RB;
  static constexpr int LDS_BYTES = 6 * PLANE;      // K planes (highest parts first), then V planes
  static constexpr int WG_PER_CU = D >= 256 ? 1 : D >= 128 ? 2 : 3;
};
// eight floats -> three operands of bf16 numbers whose sum they are
struct F32Split {
  short8v part[3];
  __device__ __forceinline__ F32Split() {}
  __device__ __forceinline__ explicit F32Split(const float *x) {
    u32x4 w[3];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float a = x[2 * j], b = x[2 * j + 1];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        w[t][j] = ElemBF16::pack2(a, b);
        if (t < 2) {   // (exact)
          a -= ElemBF16::lo(w[t][j]);
          b -= ElemBF16::hi(w[t][j]);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) part[t] = __builtin_bit_cast(short8v, w[t]);
  }
};

template <int D>
__global__ __launch_bounds__(kThreads, F32Tile<D>::WG_PER_CU) void hbsa_fwd_f32_kernel(FwdParams p, float c_signed) {
  using T = F32Tile<D>;
  using SW = FwdSwizzle<D>;
  constexpr int RB = T::RB, CPR = T::CPR, KT = T::KT, GROUPS = T::GROUPS, PLANE = T::PLANE;
  constexpr int KSTEPS = D / 16;  // MFMA steps of S (and of each of its six products)
  constexpr int DT = D / 32;      // accumulators of O^T
  constexpr int LOADS = KT * CPR / kThreads;   // chunks per lane, tile and operand
  constexpr int RPL = 64 / CPR;                // rows one load of a wavefront covers (inside one group)
  static_assert(LOADS >= 1 && RPL >= 1 && RPL <= 16, "a load stays inside a group of 16 keys");
  extern __shared__ __attribute__((aligned(1024))) char lds[];   // a tile
  __shared__ int last_flag;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g32 = lane >> 5, l32 = lane & 31;

  // Items: last q blocks (the heavy ones under a causal mask) first, the heads of a q block next to each other, and so
  // are its parts, which evens out the load of long items.  A small launch starts every item's first part before any
  // second one: what it waits for is the start of its workgroups, many of them without a part (2 x 64 .. 500 tokens
  // 25 -> 19 us; 4 x 1279 .. 2697 tokens at D = 128 215 us by item, 234 by part).
  uint32_t item;
  int part;
  if (p.parts_last) {
    part = (int)fast_div(blockIdx.x, p.div_items);
    item = blockIdx.x - (uint32_t)part * (gridDim.x / (uint32_t)p.max_parts);
  } else {
    item = fast_div(blockIdx.x, p.div_nparts);
    part = (int)(blockIdx.x - item * (uint32_t)p.max_parts);
  }
  const uint32_t t = fast_div(item, p.div_nsub);
  const int sub = (int)(item - t * (uint32_t)p.nsub);
  const uint32_t rev = fast_div(t, p.div_nhk);
  const int hk = (int)(t - rev * (uint32_t)p.nhead_k);
  const int qb = p.nqb - 1 - (int)rev;
  int kb0;
  const QBlockInfo inf = item_geometry(p, qb, lane, kb0);
  if (inf.rows <= 0 || sub * 4 * kWaveRows >= p.ratio * inf.rows) return;   // no entries (the same for every part)
  const int nvis = min(inf.nkblk, (inf.kmax + p.kbs - 1) / p.kbs);
  const ItemParts parts(p, nvis);
  if (part >= parts.count) return;
  const int blk_begin = part * parts.per, blk_end = min(nvis, blk_begin + parts.per);

  // entries: number = head of the group * rows + row; a wave slot takes 32 consecutive ones
  const int first = (sub * 4 + wave) * kWaveRows;
  const int n = min(kWaveRows, p.ratio * inf.rows - first);
  const bool active = n > 0;
  const int entry = first + min(l32, max(n - 1, 0));
  const int head = active ? entry / inf.rows : 0, row = active ? entry - head * inf.rows : 0;
  const int hq = hk * p.ratio + head;
  const int lane_kvis = inf.q_pos + row + inf.shift;   // last key position this query sees
  int wave_kvis_min = lane_kvis, wave_kvis_max = lane_kvis;
#pragma unroll
  for (int off = 1; off < 32; off <<= 1) {
    wave_kvis_min = min(wave_kvis_min, __shfl_xor(wave_kvis_min, off));
    wave_kvis_max = max(wave_kvis_max, __shfl_xor(wave_kvis_max, off));
  }
  wave_kvis_min = __builtin_amdgcn_readfirstlane(wave_kvis_min);
  wave_kvis_max = __builtin_amdgcn_readfirstlane(wave_kvis_max);

  // What the first tile needs is asked for before anything is waited for: the mask, then the query rows, K and V.
  const float *qrow = (const float *)(p.q + (int64_t)(inf.row_begin + row) * p.q_s + (int64_t)hq * p.q_h);
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  const char *kg = p.k + (int64_t)hk * p.k_h + (int64_t)inf.key_begin * p.k_s;
  const char *vg = p.v + (int64_t)hk * p.v_h + (int64_t)inf.key_begin * p.v_s;

  // ---- the sequence of 16-key groups of the kept blocks (the same in every wavefront)
  const KeptWindow window(p, hk, qb, kb0, lane);
  int win, blk, off;      // blocks win .. win + 63 are in `kept`; current block, position of its next group
  uint64_t kept;
  uint32_t ahead;         // the next window, on its way
  auto first_group = [&]() {
    win = blk_begin;
    blk = -1;
    off = 0;
    kept = KeptWindow::vote(window.load(win, blk_end));
    ahead = window.load(win + 64, blk_end);
  };
  first_group();
  auto next_group = [&](int &pos, int &valid) -> bool {
    if (blk < 0 || off >= p.kbs || blk * p.kbs + off >= inf.kmax) {
      while (kept == 0) {
        win += 64;
        if (win >= blk_end) return false;
        kept = KeptWindow::vote(ahead);
        ahead = window.load(win + 64, blk_end);
      }
      blk = win + __builtin_ctzll(kept);
      kept &= kept - 1;
      off = 0;
    }
    pos = blk * p.kbs + off;
    valid = min(16, inf.kmax - pos);
    off += 16;
    return true;
  };
  struct Tile {
    int pos[GROUPS], valid[GROUPS];   // groups past the last one: valid 0
    bool any;
  };
  auto next_tile = [&](Tile &tl) {
    tl.any = false;
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
      int pos = 0, valid = 0;
      const bool have = (g == 0 || tl.valid[g - 1] > 0) && next_group(pos, valid);
      tl.pos[g] = have ? pos : (g > 0 ? tl.pos[g - 1] : 0);
      tl.valid[g] = have ? valid : 0;
      if (g == 0) tl.any = have;
    }
  };

  // ---- tile loads: chunk i of a thread is eight elements of row RPL * (4 * i + wave) + lane / CPR.  K and V take turns in the
  // registers: a tile's V is on its way while its scores are formed, the next tile's K during the products with V.
  f32x4 raw[LOADS][2], first_k[LOADS][2];
  const int ld_row = RPL * wave + lane / CPR, ld_chunk = lane % CPR;
  const uint32_t k_s32 = (uint32_t)p.k_s, v_s32 = (uint32_t)p.v_s;   // row strides in bytes (the host checks they fit)
  auto fetch = [&](f32x4 (&raw)[LOADS][2], const char *base, int64_t stride, uint32_t stride32, const Tile &tl) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int g = __builtin_amdgcn_readfirstlane((RPL * (4 * i + wave)) >> 4);
      int pos = tl.pos[0], valid = tl.valid[0];
#pragma unroll
      for (int x = 1; x < GROUPS; ++x) {
        pos = g == x ? tl.pos[x] : pos;
        valid = g == x ? tl.valid[x] : valid;
      }
      const uint32_t in_group = (uint32_t)min((ld_row + 4 * RPL * i) & 15, max(valid, 1) - 1);   // rows past the end repeat the last one (masked below)
      const f32x4 *src = (const f32x4 *)(base + (int64_t)pos * stride + (in_group * stride32 + (uint32_t)ld_chunk * 32u));
      raw[i][0] = src[0];
      raw[i][1] = src[1];
    }
  };
  auto fetch_k = [&](const Tile &tl) { fetch(raw, kg, p.k_s, k_s32, tl); };
  auto fetch_v = [&](const Tile &tl) { fetch(raw, vg, p.v_s, v_s32, tl); };
  // splits what was fetched into the planes of K (false) or V (true)
  auto place = [&](auto v_, const f32x4 (&raw)[LOADS][2]) {
    constexpr bool V = decltype(v_)::value;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int r = ld_row + 4 * RPL * i;
      char *dst = lds + (V ? 3 * PLANE : 0) + r * RB + ((ld_chunk ^ (V ? SW::v(r) : SW::k(r))) << 4);
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = raw[i][e >> 2][e & 3];
      const F32Split s(x);
#pragma unroll
      for (int t = 0; t < 3; ++t) *(short8v *)(dst + t * PLANE) = s.part[t];
    }
  };
  // operand reads: K rows l32, V^T through the transposing read (within 16 lanes, lane r supplies the address of key r / 4,
  // dims 4 * (r % 4) .. + 3 and receives dim r of four keys)
  const int k_rd = l32 * RB;
  const int v_key = 4 * g32 + ((lane & 15) >> 2), v_lc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  const int v_rd = 3 * PLANE + v_key * RB + 8 * (lane & 1);

  auto half_of = [](const Tile &tl, int h) {   // half h of a tile of 64 keys, as the first of one
    Tile r = tl;
    r.pos[0] = h ? tl.pos[GROUPS - 2] : tl.pos[0];
    r.pos[1] = h ? tl.pos[GROUPS - 1] : tl.pos[1];
    r.valid[0] = h ? tl.valid[GROUPS - 2] : tl.valid[0];
    r.valid[1] = h ? tl.valid[GROUPS - 1] : tl.valid[1];
    return r;
  };
  auto half_used = [&](const Tile &tl, int h) { return active && tl.valid[2 * h] > 0 && (!p.causal || tl.pos[2 * h] <= wave_kvis_max); };
  // scores of half h of a tile -> exponentials, and the sums so far to their new reference
  auto softmax = [&](const Tile &tl, int h, f32x16 &sc) {
    const int pos0 = tl.pos[2 * h], pos1 = tl.pos[2 * h + 1], valid0 = tl.valid[2 * h], valid1 = tl.valid[2 * h + 1];
    const bool edge = valid1 < 16 || (p.causal && max(pos0, pos1) + 15 > wave_kvis_min);
    if (edge) {
      int lim0 = valid0, lim1 = valid1;   // keys of the groups below these are visible to this lane's query
      if (p.causal) {
        lim0 = min(lim0, lane_kvis - pos0 + 1);
        lim1 = min(lim1, lane_kvis - pos1 + 1);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (8 * ((i >> 2) & 1) + 4 * g32 + (i & 3) >= (i < 8 ? lim0 : lim1)) sc[i] = -INFINITY;
    }
    float mx = sc[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, sc[i]);
    mx = half_max(mx);
    // no branch on per-query values below: the MFMAs need every lane
    const float m_new = fmaxf(m_run, mx);
    const float m_ref = m_new == -INFINITY ? 0.f : m_new;       // a query that has seen no key yet
    if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0) {      // (otherwise every factor is one)
      const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_ref);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
    }
    m_run = m_new;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      sc[i] = __builtin_amdgcn_exp2f(sc[i] - m_ref);
      l_run += sc[i];
    }
  };
  F32Split qf[KSTEPS];
  // S^T of half h
  auto multiply_k = [&](int h, f32x16 &sc) {
    // the products with a second or third part first, then those of the first parts: few additions round at the sum's full size
    auto k_at = [&](int ks, int t) { return *(const short8v *)(lds + k_rd + 32 * h * RB + t * PLANE + (((2 * ks + g32) ^ SW::k(l32)) << 4)); };
    short8v k[3], ahead[3];
#pragma unroll
    for (int t = 0; t < 3; ++t) ahead[t] = k_at(0, t);
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      const short8v *q = qf[ks].part;
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        k[t] = ahead[t];
        if (ks + 1 < KSTEPS) ahead[t] = k_at(ks + 1, t);
        else if (t == 0) ahead[0] = k_at(0, 0);
      }
      sc = ElemBF16::mfma(k[2], q[0], sc);
      sc = ElemBF16::mfma(k[0], q[2], sc);
      sc = ElemBF16::mfma(k[1], q[1], sc);
      sc = ElemBF16::mfma(k[1], q[0], sc);
      sc = ElemBF16::mfma(k[0], q[1], sc);
      __builtin_amdgcn_sched_barrier(0);   // (or more steps' operands are read ahead than there are registers for)
    }
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      k[0] = ahead[0];
      if (ks + 1 < KSTEPS) ahead[0] = k_at(ks + 1, 0);
      sc = ElemBF16::mfma(k[0], qf[ks].part[0], sc);
    }
  };
  // O^T += V^T P^T of half h
  auto multiply_v = [&](int h, const f32x16 &sc) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {   // 16 keys at a time
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = sc[8 * j + e];
      const F32Split pp(x);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const char *at = lds + v_rd + (32 * h + 16 * j) * RB + (((4 * dt + v_lc) ^ SW::v(v_key)) << 4);
        short8v v[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          const short4v a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)HBSA_AS3(at + t * PLANE));
          const short4v b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)HBSA_AS3(at + t * PLANE + 8 * RB));
          v[t] = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
        }
        o[dt] = ElemBF16::mfma(v[2], pp.part[0], o[dt]);
        o[dt] = ElemBF16::mfma(v[0], pp.part[2], o[dt]);
        o[dt] = ElemBF16::mfma(v[1], pp.part[1], o[dt]);
        o[dt] = ElemBF16::mfma(v[1], pp.part[0], o[dt]);
        o[dt] = ElemBF16::mfma(v[0], pp.part[1], o[dt]);
        o[dt] = ElemBF16::mfma(v[0], pp.part[0], o[dt]);
      }
    }
  };

  Tile cur, nxt;
  next_tile(cur);
  f32x4 q_raw[KSTEPS][2];
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) {
    q_raw[ks][0] = q_raw[ks][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (active) {
      q_raw[ks][0] = *(const f32x4 *)(qrow + 16 * ks + 8 * g32);
      q_raw[ks][1] = *(const f32x4 *)(qrow + 16 * ks + 8 * g32 + 4);
    }
  }
  if (cur.any) {
    fetch(first_k, kg, p.k_s, k_s32, cur);
    fetch_v(cur);
  }
  // Q^T operands, pre-multiplied by softmax_scale * log2(e): scores come out in log2 units
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = q_raw[ks][e >> 2][e & 3] * c_signed;
    qf[ks] = F32Split(x);
  }
  if constexpr (KT == 64) {
    // Head dim 32: a tile's K and V are placed together, and its halves are two rounds of one loop, scores to products.  (What a
    // short call takes is, beside its loads, the way through the code: unrolled, two halves are 26 KB of it.)
    while (cur.any) {
      place(std::false_type{}, first_k);
      place(std::true_type{}, raw);
      next_tile(nxt);
      if (nxt.any) {
        fetch(first_k, kg, p.k_s, k_s32, nxt);
        fetch_v(nxt);
      }
      __syncthreads();   // the tile is in place
#pragma unroll 1
      for (int h = 0; h < KT / 32; ++h) {
        const Tile half = half_of(cur, h);
        if (!half_used(half, 0)) continue;
        f32x16 sc;
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] = 0.f;
        multiply_k(h, sc);
        softmax(half, 0, sc);
        multiply_v(h, sc);
      }
      __syncthreads();   // ... and has been read by all
      cur = nxt;
    }
  } else {
    if (cur.any) place(std::false_type{}, first_k);
    while (cur.any) {
      __syncthreads();   // the tile's K is in place, the V of the tile before has been read by all
      place(std::true_type{}, raw);
      next_tile(nxt);
      if (nxt.any) fetch_k(nxt);
      f32x16 scores[KT / 32];
#pragma unroll
      for (int h = 0; h < KT / 32; ++h) {   // ---- 32 keys at a time: scores
        f32x16 &sc = scores[h];
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] = 0.f;
        if (!half_used(cur, h)) continue;
        multiply_k(h, sc);
      }
      __syncthreads();   // the tile's V is in place, its K has been read by all
      if (nxt.any) {
        place(std::false_type{}, raw);
        fetch_v(nxt);
      }
#pragma unroll
      for (int h = 0; h < KT / 32; ++h) {   // ---- softmax and products with V
        if (!half_used(cur, h)) continue;
        softmax(cur, h, scores[h]);
        multiply_v(h, scores[h]);
      }
      cur = nxt;
    }
  }

  float any_nan = l_run;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) any_nan += o[dt][i] * 0.f;
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(any_nan != any_nan) != 0, 0)) {   // ---- again, with the fp32 instructions
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
    m_run = -INFINITY;
    l_run = 0.f;
    first_group();
    for (next_tile(cur); cur.any; next_tile(cur)) {
#pragma unroll 1
      for (int h = 0; h < KT / 32; ++h) {
        const Tile half = half_of(cur, h);
        if (!half_used(half, 0)) continue;
        auto row_at = [&](const char *base, int64_t stride, int key) {   // of key 0 .. 31 of the half, rows past the end repeat the last one
          return (const float *)(base + (int64_t)((key >> 4 ? half.pos[1] : half.pos[0]) +
                                                  min(key & 15, max(key >> 4 ? half.valid[1] : half.valid[0], 1) - 1)) * stride);
        };
        f32x16 sc;
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] = 0.f;
        const float *krow = row_at(kg, p.k_s, l32);
#pragma unroll 1
        for (int d = 4 * g32; d < D; d += 8) {
          const f32x4 kv = *(const f32x4 *)(krow + d), qv = *(const f32x4 *)(qrow + d) * c_signed;
#pragma unroll
          for (int e = 0; e < 4; ++e) sc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[e], qv[e], sc, 0, 0, 0);
        }
        softmax(half, 0, sc);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float *vrow = row_at(vg, p.v_s, 8 * (i >> 2) + 4 * g32 + (i & 3)) + l32;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vrow[32 * dt], sc[i], o[dt], 0, 0, 0);
        }
      }
    }
  }

  float l_tot = half_sum(l_run);
  if (parts.count > 1) {
    // ---- several parts: leave this one's result, and go on only if it is the last to arrive
    constexpr int REGS = DT * 16 + 2;
    const size_t stride = (size_t)REGS * 64;
    float *mine = p.parts + (((size_t)item * p.max_parts + part) * 4 + wave) * stride + lane;
    if (active && l32 < n) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) part_store(mine + (dt * 16 + i) * 64, o[dt][i]);
      part_store(mine + DT * 16 * 64, m_run);
      part_store(mine + (DT * 16 + 1) * 64, l_tot);
    }
    parts_arrived();
    __syncthreads();
    if (threadIdx.x == 0) {
      const uint32_t before = __hip_atomic_fetch_add(p.arrivals + item, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last_flag = before + 1 == (uint32_t)parts.count;
      if (last_flag) __hip_atomic_store(p.arrivals + item, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last_flag) return;
    parts_acquire();
    if (active && l32 < n) {
      const float *all = p.parts + ((size_t)item * p.max_parts * 4 + wave) * stride + lane;
      float m_all = -INFINITY;
#pragma unroll 8
      for (int pt = 0; pt < parts.count; ++pt) m_all = fmaxf(m_all, all[(size_t)pt * 4 * stride + DT * 16 * 64]);
      const float m_ref = m_all == -INFINITY ? 0.f : m_all;
      l_tot = 0.f;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
#pragma unroll 2
      for (int pt = 0; pt < parts.count; ++pt) {
        const float *q = all + (size_t)pt * 4 * stride;
        const float f = __builtin_amdgcn_exp2f(q[DT * 16 * 64] - m_ref);
        l_tot += f * q[(DT * 16 + 1) * 64];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[dt][i] += f * q[(dt * 16 + i) * 64];
      }
      m_run = m_all;
    }
  }

  if (!active || l32 >= n) return;
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  const int64_t out_row = inf.row_begin + row;
  if (p.lse != nullptr && g32 == 0)
    p.lse[out_row * p.lse_s + (int64_t)hq * p.lse_h] =
        l_tot > 0.f ? (m_run + __builtin_amdgcn_logf(l_tot)) * 0.69314718055994531f : -INFINITY;
  char *orow = p.out + out_row * p.o_s + (int64_t)hq * p.o_h;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4)
      *(f32x4 *)(orow + (32 * dt + 8 * i4 + 4 * g32) * 4) =
          f32x4{o[dt][4 * i4] * inv, o[dt][4 * i4 + 1] * inv, o[dt][4 * i4 + 2] * inv, o[dt][4 * i4 + 3] * inv};
}

template <int D>
int launch_fwd_f32(const FwdParams &fp, float c_signed, long long items, hipStream_t stream) {
  constexpr int lds_bytes = F32Tile<D>::LDS_BYTES;
  const void *kernel = reinterpret_cast<const void *>(&hbsa_fwd_f32_kernel<D>);
  static thread_local bool configured[kMaxDevices] = {};   // the attribute is per device
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fail(HBSA_ERR_UNSUPPORTED, "no current device, or device index above %d", kMaxDevices - 1);
  if (!configured[dev]) {
    hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) return fail((int)e, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    configured[dev] = true;
  }
  hipLaunchKernelGGL((hbsa_fwd_f32_kernel<D>), dim3((unsigned)(items * fp.max_parts)), dim3(kThreads), lds_bytes, stream, fp, c_signed);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail((int)e, "hbsa_fwd_f32_kernel launch: %s", hipGetErrorString(e));
  return 0;
}

}  // namespace hbsa
