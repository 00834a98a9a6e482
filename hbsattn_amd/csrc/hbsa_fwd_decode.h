// The attention kernel of the forward for few queries per (kv head, q block): decode steps and short verification or draft
// blocks against long key sequences.
#pragma once

#include "hbsa_common.h"

namespace hbsa {

// --------------------------------------------------------------------------------------
// What bounds it: the stream of K and V rows, each used by a few queries (16 on average and 64 at most; the 32-query wave slots
// of the other kernel would be mostly empty, and three of its four wavefronts idle).  So a workgroup is ONE wavefront with its own two tile
// buffers in LDS: no barriers, nothing shared, five of them on a CU at D = 128, each with up to two tiles of 32 keys
// (16 KB) on their way.  An item (kv head, q block) is cut into parts over its k blocks (ItemParts) whatever the lengths of the
// sequences; the part that arrives last combines them, or a second launch where items may have more than 16 queries.  32 sequences of 2000 .. 32000 keys, 32 / 8 heads of 128, bf16, keep
// 0.25: 151 us in the other kernel with a pre-pass, a split and a merge launch, 125 here (4.5 TB/s of K and V); 2 sequences
// of 3400 .. 8400 keys, 16 / 4 heads of 64: 35 and 12 us; 64 x 10000 .. 40000 keys, 32 heads: 5.7 TB/s.
//
// Operands (v_mfma_f32_16x16x32): S^T[16 keys, 16 queries] = K . Q^T with K rows from LDS (ds_read_b128), Q^T in registers; a
// lane then holds four keys of one query per 16 keys.  O^T[16 dims, 16 queries] += V^T . P^T over 32 keys, numbered so that
// the lane's eight P values (4 * g + i of the first and of the second 16 keys, g = lane / 16) are its operand as they
// are; V^T through transposing reads (ds_read_b64_tr_b16: rows 4 * g .. + 3, dim lane % 16).
// Tiles are two groups of 16 keys from any place, so blocks of 16 or 48 keys fill them like larger ones.
// LDS placement: chunk c (16 bytes) of K row r at c ^ k(r) as in the other kernel; of V row r at c ^ v(r), where v moves
// pairs of chunks: the eight rows x 32 bytes that half a wavefront's transposing read touches lie in different banks.
// --------------------------------------------------------------------------------------
template <int D>
struct DecodeTile {
  static constexpr int RB = D * 2, CPR = RB / 16;
  static constexpr int RPG = 16 / CPR > 0 ? 16 / CPR : 1;
  static constexpr int KT = 32;
  static constexpr int TILE_BYTES = KT * RB;           // of one operand
  static constexpr int LDS_BYTES = 4 * TILE_BYTES;     // two buffers of K and V
  static constexpr int LOADS = KT * CPR / 64;          // 16-byte loads per lane, tile and operand
  static constexpr int PAIRS = CPR / 2 < 8 ? CPR / 2 : 8;
  static __device__ __forceinline__ int k(int r) { return (r / RPG) % (CPR < 16 ? CPR : 16); }   // (the same for rows 16 apart)
  static __device__ __forceinline__ int v(int r) { return ((r / RPG) % PAIRS) << 1; }
};

struct Decode16BF16 {
  static __device__ __forceinline__ f32x4 mfma(short8v a, short8v b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
struct Decode16F16 {
  static __device__ __forceinline__ f32x4 mfma(short8v a, short8v b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

// combine over the four lanes that hold one query (lane % 16): lane ^ 16, then lane ^ 32
__device__ __forceinline__ float quad_max(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return half_max(fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1])));
}
__device__ __forceinline__ float quad_sum(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return half_sum(__builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]));
}

// The token row (of the q block) and q head of an item's entry: number = head of the group * rows + row
__device__ __forceinline__ void decode_entry(const FwdParams &p, const QBlockInfo &inf, int hk, int e, int &row, int &hq) {
  const int h = e / inf.rows;
  row = e - h * inf.rows;
  hq = hk * p.ratio + h;
}

// The output of the entries e_begin .. + 15 of an item (and of those e_step further on) from its parts, in the order of the parts.
// First the parts' weights, one (entry, part) per lane, into LDS; then four dims of one entry per lane at a time, with
// the same four of sixteen parts under way together (each a trip to memory of a microsecond or two: one after the
// other, 32 parts of four entries took 45 us, now 7).
constexpr int decode_combine_bytes = (16 * kDecodeMaxParts + 32) * 4;
template <int D, typename E, int THREADS>
__device__ __forceinline__ void decode_combine(const FwdParams &p, const QBlockInfo &inf, int hk, int count, int e_begin, int e_step,
                                               char *lds, int tid) {
  constexpr int kMaxParts = kDecodeMaxParts, CHUNK = 16;
  const int entries = p.ratio * inf.rows;
  const int64_t rows_all = (int64_t)p.total_q * p.nhead_q;
  const float *part_lse = p.parts + (size_t)p.max_parts * rows_all * D;
  float *weight = (float *)lds, *sum = weight + 16 * kMaxParts, *top = sum + 16;   // [entry of the pass][part]; [entry]
  auto sync = [] {
    if constexpr (THREADS > 64) __syncthreads();
    else asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");   // (one wavefront: its own writes)
  };
  for (int e0 = e_begin; e0 < entries; e0 += e_step) {
    const int n = min(16, entries - e0);
    for (int x = tid; x < n * kMaxParts; x += THREADS) {   // (32 lanes one entry)
      const int e = x / kMaxParts, pt = x % kMaxParts;
      int row, hq;
      decode_entry(p, inf, hk, e0 + e, row, hq);
      const int64_t at = (int64_t)pt * rows_all + (int64_t)(inf.row_begin + row) * p.nhead_q + hq;
      const float2 ml = pt < count ? *(const float2 *)(part_lse + 2 * at) : float2{-INFINITY, 0.f};
      float m_all = ml.x;
#pragma unroll
      for (int off = 1; off < kMaxParts; off <<= 1) m_all = fmaxf(m_all, __shfl_xor(m_all, off));
      const float f = __builtin_amdgcn_exp2f((ml.x - (m_all == -INFINITY ? 0.f : m_all)) * p.c);
      float l_tot = f * ml.y;
#pragma unroll
      for (int off = 1; off < kMaxParts; off <<= 1) l_tot += __shfl_xor(l_tot, off);
      weight[x] = f;
      if (pt == 0) {
        sum[e] = l_tot;
        top[e] = m_all;
      }
    }
    sync();
    for (int x = tid; x < n * (D / 4); x += THREADS) {
      const int e = x / (D / 4), dq = x % (D / 4);
      int row, hq;
      decode_entry(p, inf, hk, e0 + e, row, hq);
      const int64_t r = inf.row_begin + row;
      const float *src = p.parts + (r * p.nhead_q + hq) * D + 4 * dq;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      for (int base = 0; base < count; base += CHUNK) {
        f32x4 v[CHUNK], f[CHUNK / 4];
#pragma unroll
        for (int i = 0; i < CHUNK; ++i) v[i] = *(const f32x4 *)(src + (int64_t)min(base + i, count - 1) * rows_all * D);
#pragma unroll
        for (int i = 0; i < CHUNK / 4; ++i) f[i] = *(const f32x4 *)(weight + e * kMaxParts + base + 4 * i);
#pragma unroll
        for (int i = 0; i < CHUNK; ++i) acc += f[i / 4][i % 4] * (base + i < count ? v[i] : f32x4{0.f, 0.f, 0.f, 0.f});   // (no 0 * inf)
      }
      const float l_tot = sum[e], inv = l_tot > 0.f ? __builtin_amdgcn_rcpf(l_tot) : 0.f;
      if (p.lse != nullptr && dq == 0)
        p.lse[r * p.lse_s + (int64_t)hq * p.lse_h] = l_tot > 0.f ? (top[e] * p.c + __builtin_amdgcn_logf(l_tot)) * 0.69314718055994531f : -INFINITY;
      u32x2 w;
      w.x = E::pack2(acc[0] * inv, acc[1] * inv);
      w.y = E::pack2(acc[2] * inv, acc[3] * inv);
      *(u32x2 *)(p.out + r * p.o_s + (int64_t)hq * p.o_h + 8 * dq) = w;
    }
    sync();
  }
}

// NQ: groups of 16 entries a wavefront holds, 1 where no item has more than 16 entries.  Else a tile, once it is in LDS, serves
// all of an item's entries: its stream is what a step waits for, and the products of three more groups hide behind it.
// 25 single queries and 6 drafts of 16, 32 / 8 heads of 128 on 2000 .. 32000 keys: 210 us with one group at a time, each walking
// all tiles again, 154 in the other kernel, 134 here; 28 singles on 2000 .. 8000 keys and a draft of 16 on 32000: 154, 115, 89;
// 60 singles and a chunk of 64 in 16-row blocks, 16 / 4 heads of 64: 133, 109, 70.
template <int D, typename E, int NQ>
__global__ __launch_bounds__(64, (NQ > 1 && D > 128 ? 1 : 2)) void hbsa_fwd_decode_kernel(FwdParams p) {
  using T = DecodeTile<D>;
  using M = std::conditional_t<std::is_same<E, ElemBF16>::value, Decode16BF16, Decode16F16>;
  constexpr int RB = T::RB, CPR = T::CPR, KS = D / 32, DT = D / 16, LOADS = T::LOADS;
  extern __shared__ __attribute__((aligned(1024))) char lds[];   // K[2], V[2] tiles of 32 keys

  const int lane = threadIdx.x;
  const int l16 = lane & 15, g = lane >> 4;

  uint32_t item;
  int part;
  if (p.parts_last) {
    part = (int)fast_div(blockIdx.x, p.div_items);
    item = blockIdx.x - (uint32_t)part * (gridDim.x / (uint32_t)p.max_parts);
  } else {
    item = fast_div(blockIdx.x, p.div_nparts);
    part = (int)(blockIdx.x - item * (uint32_t)p.max_parts);
  }
  const uint32_t rev = fast_div(item, p.div_nhk);
  const int hk = (int)(item - rev * (uint32_t)p.nhead_k);
  const int qb = p.nqb - 1 - (int)rev;
  int kb0;
  const QBlockInfo inf = item_geometry(p, qb, lane, kb0);
  if (inf.rows <= 0) return;
  const int nvis = min(inf.nkblk, (inf.kmax + p.kbs - 1) / p.kbs);
  const ItemParts parts(p, nvis);
  if (part >= parts.count) return;
  const int blk_begin = part * parts.per, blk_end = min(nvis, blk_begin + parts.per);
  const int entries = p.ratio * inf.rows;
  const int64_t rows_all = (int64_t)p.total_q * p.nhead_q;
  float *part_lse = p.parts + (size_t)p.max_parts * rows_all * D;   // behind the results: (m, l) pairs

  const uint32_t lds_base = (uint32_t)(uintptr_t)HBSA_AS3(lds);
  const uint32_t k_s32 = (uint32_t)p.k_s, v_s32 = (uint32_t)p.v_s;   // row strides in bytes (the host checks they fit)
  const char *kg = p.k + (int64_t)hk * p.k_h + (int64_t)inf.key_begin * p.k_s;
  const char *vg = p.v + (int64_t)hk * p.v_h + (int64_t)inf.key_begin * p.v_s;

  auto store_out = [&](const f32x4 *o, float m, float l_tot, int row, int hq) {   // one lane: dims 16 * dt + 4 * g .. + 3 of its query
    const float inv = l_tot > 0.f ? __builtin_amdgcn_rcpf(l_tot) : 0.f;
    const int64_t r = inf.row_begin + row;
    if (p.lse != nullptr && g == 0)
      p.lse[r * p.lse_s + (int64_t)hq * p.lse_h] = l_tot > 0.f ? (m * p.c + __builtin_amdgcn_logf(l_tot)) * 0.69314718055994531f : -INFINITY;
    char *orow = p.out + r * p.o_s + (int64_t)hq * p.o_h + 8 * g;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      u32x2 w;
      w.x = E::pack2(o[dt][0] * inv, o[dt][1] * inv);
      w.y = E::pack2(o[dt][2] * inv, o[dt][3] * inv);
      *(u32x2 *)(orow + dt * 32) = w;
    }
  };

  const KeptWindow window(p, hk, qb, kb0, lane);
  for (int e0 = 0; e0 < entries; e0 += 16 * NQ) {   // (usually once)
    const int n = min(16 * NQ, entries - e0);
    const int groups = (n + 15) / 16;
    int row[NQ], hq[NQ], lane_kvis[NQ], kvis_min[NQ];
#pragma unroll
    for (int x = 0; x < NQ; ++x) {
      decode_entry(p, inf, hk, e0 + min(16 * x + l16, n - 1), row[x], hq[x]);
      lane_kvis[x] = inf.q_pos + row[x] + inf.shift;   // last key position this query sees
      kvis_min[x] = lane_kvis[x];
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) kvis_min[x] = min(kvis_min[x], __shfl_xor(kvis_min[x], off));
      kvis_min[x] = __builtin_amdgcn_readfirstlane(kvis_min[x]);
    }

    // ---- the sequence of 16-key groups of the kept blocks
    int win = blk_begin;
    uint32_t first_window = window.load(win, blk_end);
    uint32_t ahead = window.load(win + 64, blk_end);
    short8v qf[NQ][KS];   // Q^T operand: query l16, dims 32 * ks + 8 * g .. + 7
#pragma unroll
    for (int x = 0; x < NQ; ++x) {
      const char *qrow = p.q + (int64_t)(inf.row_begin + row[x]) * p.q_s + (int64_t)hq[x] * p.q_h + 16 * g;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[x][ks] = __builtin_bit_cast(short8v, *(const u32x4 *)(qrow + 64 * ks) ^ p.q_sign);
    }
    uint64_t kept = KeptWindow::vote(first_window);
    int blk = -1, off = 0;
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
      int pos0, pos1, valid0, valid1;   // valid0 == 0: no tile
    };
    auto next_tile = [&]() -> Tile {
      Tile t = {0, 0, 0, 0};
      if (next_group(t.pos0, t.valid0)) {
        t.pos1 = t.pos0;
        if (!next_group(t.pos1, t.valid1)) t.valid1 = 0;
      } else {
        t.valid0 = 0;
      }
      return t;
    };
    // a tile's chunks: load i fills 1024 bytes, rows i * 64 / CPR .. ; rows past a group's end repeat its last one
    auto fetch = [&](int buf, const Tile &t) {
      const uint32_t dst = lds_base + (uint32_t)(buf * T::TILE_BYTES);
      const char *k0 = kg + (int64_t)t.pos0 * p.k_s, *k1 = kg + (int64_t)t.pos1 * p.k_s;
      const char *v0 = vg + (int64_t)t.pos0 * p.v_s, *v1 = vg + (int64_t)t.pos1 * p.v_s;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const bool second = i >= (LOADS + 1) / 2;   // (rows 16 .. 31; with one load for the whole tile both groups are in it)
        const int r = i * (64 / CPR) + lane / CPR;
        if constexpr (LOADS >= 2) {
          const int in_group = min(r & 15, max(second ? t.valid1 : t.valid0, 1) - 1);
          const uint32_t ko = (uint32_t)in_group * k_s32 + (uint32_t)(((lane % CPR) ^ T::k(r)) * 16);
          const uint32_t vo = (uint32_t)in_group * v_s32 + (uint32_t)(((lane % CPR) ^ T::v(r)) * 16);
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(dst + i * 1024u), "v"(ko), "s"(second ? k1 : k0) : "memory", "m0");
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(dst + 2u * T::TILE_BYTES + i * 1024u), "v"(vo), "s"(second ? v1 : v0) : "memory", "m0");
        }
      }
    };
    static_assert(LOADS >= 2, "a load stays inside a group of 16 keys");

    f32x4 o[NQ][DT];
    float m_run[NQ], l_run[NQ];
#pragma unroll
    for (int x = 0; x < NQ; ++x) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[x][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
      m_run[x] = -INFINITY;
      l_run[x] = 0.f;
    }

    // per-lane LDS offsets inside a tile: K row l16, chunk 4 * ks + g; V row 4 * g + l16 / 4, chunk 2 * dt + (lane & 3) / 2
    const int v_row = 4 * g + (l16 >> 2);
    Tile cur = next_tile();
    int buf = 0;
    if (cur.valid0 > 0) fetch(0, cur);
    while (cur.valid0 > 0) {
      const Tile nxt = next_tile();
      if (nxt.valid0 > 0) {
        fetch(buf ^ 1, nxt);   // (what that buffer held has been read and used)
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * LOADS) : "memory");   // the current tile has landed
      } else {
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
      }
      const char *kt = lds + buf * T::TILE_BYTES, *vt = lds + (2 + buf) * T::TILE_BYTES;
#pragma unroll
      for (int x = 0; x < NQ; ++x) {
        if (NQ > 1 && x >= groups) continue;
        if (x > 0) asm volatile("" : : : "memory");   // (operands are read again for each group, not held in registers for all)
        f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
        {
          const char *krow = kt + l16 * RB;
          const int swz = T::k(l16);   // (the same for row l16 + 16)
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
            const int at = ((4 * ks + g) ^ swz) << 4;
            s0 = M::mfma(*(const short8v *)(krow + at), qf[x][ks], s0);
            s1 = M::mfma(*(const short8v *)(krow + 16 * RB + at), qf[x][ks], s1);
          }
        }
        if (cur.valid1 < 16 || cur.valid0 < 16 || (p.causal && max(cur.pos0, cur.pos1) + 15 > kvis_min[x])) {
          int lim0 = cur.valid0, lim1 = cur.valid1;
          if (p.causal) {
            lim0 = min(lim0, lane_kvis[x] - cur.pos0 + 1);
            lim1 = min(lim1, lane_kvis[x] - cur.pos1 + 1);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (4 * g + i >= lim0) s0[i] = -INFINITY;
            if (4 * g + i >= lim1) s1[i] = -INFINITY;
          }
        }
        float mx = fmaxf(fmaxf(fmaxf(s0[0], s0[1]), fmaxf(s0[2], s0[3])), fmaxf(fmaxf(s1[0], s1[1]), fmaxf(s1[2], s1[3])));
        mx = quad_max(mx);
        const bool grow = mx > m_run[x] + p.lag;   // the running max may lag the true one by 2^kLazyRescaleLog2
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
          const float m_new = grow ? mx : m_run[x];
          const float alpha = grow ? __builtin_amdgcn_exp2f((m_run[x] - m_new) * p.c) : 1.f;
          l_run[x] *= alpha;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[x][dt][i] *= alpha;
          m_run[x] = m_new;
        }
        const float mc = m_run[x] == -INFINITY ? 0.f : m_run[x] * p.c;
        u32x4 pw;
        {
          float e[8];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            e[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s0[i], p.c, -mc));
            e[4 + i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s1[i], p.c, -mc));
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            pw[i] = E::pack2(e[2 * i], e[2 * i + 1]);
            l_run[x] += e[2 * i] + e[2 * i + 1];
          }
        }
        const short8v pb = __builtin_bit_cast(short8v, pw);
        {
          const int swz = T::v(v_row);   // (the same for row v_row + 16)
          const char *vrow = vt + v_row * RB + 8 * (lane & 1);
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            const char *at = vrow + (((2 * dt + ((lane & 3) >> 1)) ^ swz) << 4);
            const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)HBSA_AS3(at));
            const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)HBSA_AS3(at + 16 * RB));
            o[x][dt] = M::mfma(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), pb, o[x][dt]);
          }
        }
      }
      // every read of this buffer has returned before the next tile's loads may overwrite it
      asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
      buf ^= 1;
      cur = nxt;
    }
#pragma unroll
    for (int x = 0; x < NQ; ++x) {
      if (NQ > 1 && x >= groups) continue;
      const float l_tot = quad_sum(l_run[x]);
      if (16 * x + l16 >= n) continue;
      if (parts.count == 1) {
        store_out(o[x], m_run[x], l_tot, row[x], hq[x]);
      } else {
        const int64_t rh = (int64_t)part * rows_all + (int64_t)(inf.row_begin + row[x]) * p.nhead_q + hq[x];
        float *dst = p.parts + rh * D + 4 * g;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          part_store4(dst + 16 * dt, o[x][dt]);
        if (g == 0) {
          part_store(part_lse + 2 * rh, m_run[x]);
          part_store(part_lse + 2 * rh + 1, l_tot);
        }
      }
    }
  }
  if (NQ > 1 || parts.count == 1) return;   // (NQ > 1: hbsa_fwd_decode_combine_kernel)

  // ---- several parts: the last one to arrive combines them, in their order
  parts_arrived();
  uint32_t before = 0;
  if (lane == 0) before = __hip_atomic_fetch_add(p.arrivals + item, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  before = (uint32_t)__builtin_amdgcn_readfirstlane((int)before);
  if (before + 1 != (uint32_t)parts.count) return;
  if (lane == 0) __hip_atomic_store(p.arrivals + item, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  parts_acquire();
  decode_combine<D, E, 64>(p, inf, hk, parts.count, 0, 16, lds, lane);
}

// The same for items of several groups (NQ > 1), a launch of its own: one workgroup per item and group of 16 entries, four
// wavefronts.  The last part's one wavefront, which has 16 KB under way at a time, took 50 us over 64 entries of 23 parts.
template <int D, typename E>
__global__ __launch_bounds__(256) void hbsa_fwd_decode_combine_kernel(FwdParams p) {
  __shared__ __attribute__((aligned(16))) char lds[decode_combine_bytes];
  const int hk = (int)(blockIdx.x % (uint32_t)p.nhead_k), qb = (int)(blockIdx.x / (uint32_t)p.nhead_k);
  int kb0;
  const QBlockInfo inf = item_geometry(p, qb, threadIdx.x & 63, kb0);
  if (inf.rows <= 0) return;
  const ItemParts parts(p, min(inf.nkblk, (inf.kmax + p.kbs - 1) / p.kbs));
  if (parts.count > 1) decode_combine<D, E, 256>(p, inf, hk, parts.count, 16 * (int)blockIdx.y, 16 * (int)gridDim.y, lds, threadIdx.x);
}

template <int D, typename E, int NQ>
int launch_fwd_decode_nq(const FwdParams &fp, long long items, hipStream_t stream) {
  constexpr int lds_bytes = DecodeTile<D>::LDS_BYTES;
  if (lds_bytes > 48 * 1024) {
    static thread_local bool configured[kMaxDevices] = {};   // the attribute is per device
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
      return fail(HBSA_ERR_UNSUPPORTED, "no current device, or device index above %d", kMaxDevices - 1);
    if (!configured[dev]) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&hbsa_fwd_decode_kernel<D, E, NQ>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
      if (e != hipSuccess) return fail((int)e, "hipFuncSetAttribute: %s", hipGetErrorString(e));
      configured[dev] = true;
    }
  }
  hipLaunchKernelGGL((hbsa_fwd_decode_kernel<D, E, NQ>), dim3((unsigned)(items * fp.max_parts)), dim3(64), lds_bytes, stream, fp);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail((int)e, "hbsa_fwd_decode_kernel launch: %s", hipGetErrorString(e));
  return 0;
}
// `most`: entries of an item at most.  Four groups fit the registers of two wavefronts a SIMD up to head dim 64, two from there on
// (four at 128, one wavefront a SIMD: 1 .. 4 queries on 2000 .. 32000 keys 159 us, with two 152).
template <int D, typename E>
int launch_fwd_decode(const FwdParams &fp, int most, long long items, hipStream_t stream) {
  if (most <= 16) return launch_fwd_decode_nq<D, E, 1>(fp, items, stream);
  if (int rc = launch_fwd_decode_nq<D, E, (D >= 128 ? 2 : 4)>(fp, items, stream)) return rc;
  if (fp.max_parts < 2) return 0;
  hipLaunchKernelGGL((hbsa_fwd_decode_combine_kernel<D, E>), dim3((unsigned)items, (unsigned)((most + 15) / 16)), dim3(256), 0, stream, fp);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : fail((int)e, "hbsa_fwd_decode_combine_kernel launch: %s", hipGetErrorString(e));
}

}  // namespace hbsa
