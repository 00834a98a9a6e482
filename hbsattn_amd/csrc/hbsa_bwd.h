// Block-sparse attention backward for gfx950: dQ, dK, dV from dO, the forward's output and its
// log-sum-exp.
//
// The reference stops at the forward (reference hbsattn/hbsa_interface.py:31-32 raises
// NotImplementedError in backward), so this follows the mathematics of that forward
// (reference hbsattn/reference.py:23-107): with S = scale * Q K^T masked like the forward,
// P = exp(S - lse), delta = rowsum(dO * O):
//     dV = P^T dO      dP = dO V^T      dS = P * (dP - delta)
//     dQ = scale * dS K                 dK = scale * dS^T Q
//
// Two launches per call, every output element written by exactly one workgroup, sums in a fixed order (few items are cut
// into parts that combine themselves, see bwd_last_part):
//   hbsa_bwd_dq_kernel    : one workgroup per (kv head, q block, group of four 32-row wave slots), the
//                           forward's decomposition; walks the kept k blocks of the q block's bit row.
//                           Per 64-key tile  S^T = K Q^T,  dP^T = V dO^T  (A = tile rows from LDS,
//                           B = Q^T / dO^T in registers),  dS^T in the accumulator layout is the B
//                           operand of  dQ^T += K^T dS^T  (A = K^T through transposing LDS reads).  It also forms
//                           delta of its rows (it holds their dO; their O is one more row load) and leaves
//                           it for the second launch.
//   hbsa_bwd_dkv_kernel   : (head dims up to 64; hbsa_bwd_dkv8_kernel is the form for D = 128) the same
//                           with the roles of queries and keys exchanged: one workgroup per
//                           (kv head, k block, group of four 32-key slots); K^T and V^T stay in
//                           registers, the Q and dO rows of every q block that keeps the k block (and of
//                           every q head of the group) stream through LDS in 64-row tiles:
//                           S = Q K^T,  dP = dO V^T,  dV^T += dO^T P,  dK^T += Q^T dS.
// Both recompute S.  The kept blocks of a mask row or column are found with one load per 32 or 64
// blocks, not one per block.  Tiles go from global memory straight into LDS (global_load_lds_dwordx4),
// two tiles ahead (V tiles of the dQ kernel one): tiles t + 1 and t + 2 travel while tile t is computed on, one barrier per
// tile (per two tiles, one ahead, for k blocks of up to 64 keys at head dims up to 64).  The dK/dV kernels walk the q blocks from the last to the first, so that the workgroups of a sequence, each of which
// a causal mask lets begin at another q block, start with the same tiles; the delta and the log-sum-exp of a tile's rows are
// consecutive floats of one q head.  A tile that is
// read both by rows and transposed is stored once, in a layout without bank conflicts for either
// (BwdTile::swz_both).  The operand reads from LDS are issued by
// hand, a fixed number ahead of the products that use them (BwdOperandOffsets).  The forward's persistent
// scheduling is not applied here: the grids already start their heaviest workgroups first, and what bounds
// both kernels at long sequences is the stream of tiles from memory next to the matrix work, not the tail.

#pragma once


#include "hbsa_common.h"

namespace hbsa {

// ---- shared pieces of the two main kernels ---------------------------------------------------------
template <int D>
struct BwdTile {
  static constexpr int RB = D * 2;            // row bytes
  static constexpr int CPR = RB / 16;         // 16-byte chunks per row
  static constexpr int RPG = 16 / CPR > 0 ? 16 / CPR : 1;
  static constexpr int TILE_BYTES = 64 * RB;
  static constexpr int KSTEPS = D / 16;
  static constexpr int DT = D / 32;
  // One chunk swizzle for a tile that is read both ways, so that it is stored once: chunk c of row r sits
  // at chunk position c ^ swz_both(r).  With a = (r / RPG) % CPR, the bits of a rotated so that its lowest
  // bits select the 64-byte column group.  Over any 16 consecutive rows the 16-byte slots of a chunk
  // column are all different (reads by rows), and rows 0-7 of a group spread evenly over the column
  // groups (transposing reads).
  static __host__ __device__ constexpr int swz_both(int r) {
    const int a = (r / RPG) % CPR;
    if constexpr (CPR == 16) return ((a & 3) << 2) | (a >> 2);
    else if constexpr (CPR == 8) return ((a & 1) << 2) | (a >> 1);
    else return a;
  }
};

// 16 bytes per lane from global memory (scalar base + 32-bit lane offset) straight into LDS at lds_addr + 16 * lane
__device__ __forceinline__ void bwd_dma16(uint32_t lds_addr, const char *sbase, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(voff), "s"(sbase) : "memory", "m0");
}

// 4 bytes per lane likewise, to lds_addr + 4 * lane
__device__ __forceinline__ void bwd_dma4(uint32_t lds_addr, const void *sbase, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(lds_addr), "v"(voff), "s"(sbase) : "memory", "m0");
}

// ---- Operand reads issued by hand (lds_read_b128 / lds_read_tr16_b64 of the forward, which explain the rules):
// the compiler puts a read next to the product that uses it, and a chain of products on one accumulator then
// waits out the LDS latency at every step.  Here a fixed number of reads is under way ahead of the products.
//
// Per-lane byte offsets of the operands inside a tile stored with BwdTile::swz_both, computed once per kernel:
//   rows[ks]   : row lane % 32 (+ 32 * h as an immediate), the 16 bytes of step ks for this lane's half of the step
//   tr[dt]     : the first of the two transposing reads of head dim slice dt for keys 16 * g .. (+ g * 16 rows as an
//                immediate); the second one, eight rows further down, sits at (tr[dt] ^ 32) + 8 rows: for every
//                head dim swz_both(key + 8) = swz_both(key) ^ 2 when key < 8
template <int D>
struct BwdOperandOffsets {
  using T = BwdTile<D>;
  uint32_t rows[T::KSTEPS], tr[T::DT];
  static constexpr bool second_read_is_xor_32() {
    for (int key = 0; key < 8; ++key)
      if (T::swz_both(key + 8) != (T::swz_both(key) ^ 2)) return false;
    return true;
  }
  static_assert(second_read_is_xor_32(), "the second transposing read's address is derived from the first one's");
  __device__ __forceinline__ void init(int lane) {
    const int l32 = lane & 31, g32 = lane >> 5;
    const int rd = l32 * T::RB + ((g32 ^ T::swz_both(l32)) << 4);
#pragma unroll
    for (int ks = 0; ks < T::KSTEPS; ++ks) rows[ks] = (uint32_t)(rd ^ (ks * 32));
    const int key = 4 * g32 + ((lane & 15) >> 2);
    const int lc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    const int t0 = key * T::RB + ((lc ^ T::swz_both(key)) << 4) + 8 * (lane & 1);
#pragma unroll
    for (int dt = 0; dt < T::DT; ++dt) tr[dt] = (uint32_t)(t0 ^ (dt * 64));
  }
};

// the 2 * DT transposing reads of key group G of the tile at LDS address tile (all head dim slices)
template <int D, int G>
__device__ __forceinline__ void bwd_issue_transposed(const BwdOperandOffsets<D> &off, uint32_t tile, short4v *dst) {
  using T = BwdTile<D>;
  static_for<0, T::DT>([&](auto dt_) {
    constexpr int dt = decltype(dt_)::value;
    dst[2 * dt] = lds_read_tr16_b64<G * 16 * T::RB>(off.tr[dt] + tile);
    dst[2 * dt + 1] = lds_read_tr16_b64<G * 16 * T::RB + 8 * T::RB>((off.tr[dt] ^ 32u) + tile);
  });
}
// returns once at most N LDS operations issued after those 2 * DT reads are outstanding
template <int D, int N>
__device__ __forceinline__ void bwd_wait_transposed(short4v *v) {
  constexpr int DT = BwdTile<D>::DT;
  static_assert(N <= 15, "the counter has four bits");
  if constexpr (DT == 4) lds_wait<N>(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]);
  else if constexpr (DT == 2) asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]) : "n"(N));
  else asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(v[0]), "+v"(v[1]) : "n"(N));
}
// acc[dt] += (those operands)^T . packed
template <int D, typename E>
__device__ __forceinline__ void bwd_transposed_products(const short4v *v, short8v packed, f32x16 *acc) {
#pragma unroll
  for (int dt = 0; dt < BwdTile<D>::DT; ++dt) {
    const short8v va = __builtin_shufflevector(v[2 * dt], v[2 * dt + 1], 0, 1, 2, 3, 4, 5, 6, 7);
    acc[dt] = E::mfma(va, packed, acc[dt]);
  }
}

// 16 accumulator values of one lane -> two B operands (rows 0-15 and 16-31 of the half tile)
template <typename E>
__device__ __forceinline__ void bwd_pack(const float *e, short8v &lo, short8v &hi) {
  u32x4 w[2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) w[j][q4] = E::pack2(e[8 * j + 2 * q4], e[8 * j + 2 * q4 + 1]);
  lo = __builtin_bit_cast(short8v, w[0]);
  hi = __builtin_bit_cast(short8v, w[1]);
}

// ---- A wavefront's 32 rows, read and written four lanes to 64 contiguous bytes of a row (as the forward's q and output rows): the
// operand layout has a lane on 16 bytes of every row of its own, the accumulators' on 8.  One instruction then covers 16 rows
// in place of 32.  What it saves is a workgroup's beginning and end: of an item of eight tiles at D = 128 the stores alone were 3400 of 51000
// cycles.  Training calls, one row a lane and as here: 4 x 8192 tokens, 32 heads of 128, a tenth kept, 1838 -> 1753 us; 64-key blocks, 5 x 4491 .. 8593,
// 16 heads, 1309 -> 1263; 4 x 4096, 32 / 8, 1059 -> 1020; 7 x 2143, 32 / 4, 716 -> 693; head dim 64, 6 x 660, 32 heads, 111.5 -> 106.6.
// Operand fragments of rows 0 .. 31 at `base` (those past `last` repeat it): lane i ends up with row i % 32, d = 16 * ks + 8 * (i / 32) .. + 7.
// With h = bit 4 of the lane, load 2k takes row i % 16, load 2k + 1 row 16 + i % 16, both at bytes 64 * k + 32 * h + 16 * (i / 32);
// then the h = 1 lanes of the first and the h = 0 lanes of the second trade places.
template <int D>
__device__ __forceinline__ void bwd_request_rows(const char *base, int64_t stride, int last, int lane, short8v *f) {
  const int l16 = lane & 15, at = (lane & 16) * 2 + (lane >> 5) * 16;
  const char *ra = base + min(l16, last) * stride + at, *rb = base + min(16 + l16, last) * stride + at;
#pragma unroll
  for (int k = 0; k < BwdTile<D>::KSTEPS / 2; ++k) {
    f[2 * k] = *(const short8v *)(ra + 64 * k);
    f[2 * k + 1] = *(const short8v *)(rb + 64 * k);
  }
}
template <int D>
__device__ __forceinline__ void bwd_place_rows(short8v *f) {
#pragma unroll
  for (int k = 0; k < BwdTile<D>::KSTEPS / 2; ++k) {
    u32x4 a = __builtin_bit_cast(u32x4, f[2 * k]), b = __builtin_bit_cast(u32x4, f[2 * k + 1]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const auto r = __builtin_amdgcn_permlane16_swap(a[j], b[j], false, false);
      a[j] = r[0];
      b[j] = r[1];
    }
    f[2 * k] = __builtin_bit_cast(short8v, a);
    f[2 * k + 1] = __builtin_bit_cast(short8v, b);
  }
}
// accumulators [d, row = lane % 32] * f -> rows 0 .. n - 1 at `base` (16-bit): lanes i and i + 32 (one row) trade halves, then
// lanes i and i + 16 the two 16-dim halves of a block
template <int D, typename E>
__device__ __forceinline__ void bwd_store_rows(char *base, int64_t stride, int n, const f32x16 *acc, float f, int lane) {
  const int l16 = lane & 15;
  char *row_x = base + l16 * stride + (lane & 16) * 2 + (lane >> 5) * 16, *row_y = row_x + 16 * stride;   // (a row past the end is not stored)
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) {
    u32x4 w[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      uint32_t x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = E::pack2(acc[dt][8 * m + 2 * j] * f, acc[dt][8 * m + 2 * j + 1] * f);
      const auto r0 = __builtin_amdgcn_permlane32_swap(x[0], x[2], false, false);
      const auto r1 = __builtin_amdgcn_permlane32_swap(x[1], x[3], false, false);
      w[m] = u32x4{(uint32_t)r0[0], (uint32_t)r1[0], (uint32_t)r0[1], (uint32_t)r1[1]};
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const auto r = __builtin_amdgcn_permlane16_swap(w[0][j], w[1][j], false, false);
      w[0][j] = r[0];
      w[1][j] = r[1];
    }
    if (l16 < n) *(u32x4 *)(row_x + dt * 64) = w[0];
    if (16 + l16 < n) *(u32x4 *)(row_y + dt * 64) = w[1];
  }
}

// The sequence a k block belongs to: what the dK/dV kernels need of it from the caller's arrays.  All three arrays are asked
// for at once, a sequence per lane (one wait in place of one per sequence passed and two more behind it).
struct BwdSequence {
  int k0, k1, kb0, qb0, qb1;   // keys [k0, k1), first k block, q blocks [qb0, qb1), those that there are records and bit rows of
  __device__ __forceinline__ BwdSequence(const BwdParams &p, int kb, int lane) {
    if (p.batch < 64) {
      const int i = min(lane, p.batch);
      const int nkb = p.cu_num_k_block[i], k = p.cu_k[i], nqb = p.cu_num_q_block[i];
      // the last sequence reached from the first one by steps to a sequence that starts at or before kb
      const uint64_t starts = __builtin_amdgcn_ballot_w64(lane >= 1 && lane < p.batch && nkb <= kb);
      const int b = __builtin_ctzll(~(starts >> 1));
      k0 = __builtin_amdgcn_readlane(k, b);
      k1 = __builtin_amdgcn_readlane(k, b + 1);
      kb0 = __builtin_amdgcn_readlane(nkb, b);
      qb0 = __builtin_amdgcn_readlane(nqb, b);
      qb1 = __builtin_amdgcn_readlane(nqb, b + 1);
    } else {   // 64 sequences at a time (dK/dV of 250 x 20 .. 128 tokens, 4 heads of 128: one at a time 127 us, so 60)
      int b = 0;
      for (;; b += 64) {
        const int i = b + 1 + lane;
        const uint64_t starts = __builtin_amdgcn_ballot_w64(i < p.batch && p.cu_num_k_block[min(i, p.batch)] <= kb);
        if (~starts != 0) {
          b += __builtin_ctzll(~starts);
          break;
        }
      }
      k0 = p.cu_k[b];
      k1 = p.cu_k[b + 1];
      kb0 = p.cu_num_k_block[b];
      qb0 = p.cu_num_q_block[b];
      qb1 = p.cu_num_q_block[b + 1];
    }
    qb1 = min(qb1, p.nqb);
  }
  // the sequence's keys lie inside the tensors, and the k block inside the sequence's numbering
  __device__ __forceinline__ bool fits(const BwdParams &p, int kb) const { return k0 >= 0 && k1 >= k0 && k1 <= p.total_k && kb >= kb0; }
};
// The record of the sequence's first q block, a word per lane (nullptr words: no q blocks).
__device__ __forceinline__ uint32_t bwd_first_record(const BwdParams &p, const BwdSequence &s, int lane) {
  return s.qb0 < s.qb1 && lane < 12 ? ((const uint32_t *)(p.info + s.qb0))[lane] : 0u;
}
// Whether that record is of the sequence's first q block and not flagged by the pre-pass.  With the keys and the position it
// states, all rows of the sequence as the kernels count them lie inside the tensors (the pre-pass has checked the record's own).
__device__ __forceinline__ bool bwd_record_holds(const BwdSequence &s, uint32_t record) {
  auto word = [&](int i) { return __builtin_amdgcn_readlane((int)record, i); };   // 2: key_begin, 3: klen, 4: q_pos, 9: flags
  return word(9) == 0 && word(2) == s.k0 && word(3) == s.k1 - s.k0 && word(4) == 0;
}
// A sequence the pre-pass found not to fit the tensors (flagged q block records, no bit rows) takes no part: its keys get zero
// gradients where they lie inside dk and dv.
template <int D, int KEYS>   // of a workgroup
__device__ __forceinline__ void bwd_zero_keys(const BwdParams &p, const BwdSequence &s, int kb, int sub, int hk) {
  const int64_t k0 = s.k0, k1 = s.k1;
  const int kbl = kb - s.kb0;
  if (k0 < 0 || k1 <= k0 || kbl < 0) return;
  const int64_t first = k0 + (int64_t)kbl * p.kbs + (int64_t)sub * KEYS;
  int64_t stop = k0 + (int64_t)(kbl + 1) * p.kbs;
  stop = stop < k1 ? stop : k1;
  stop = stop < first + KEYS ? stop : first + KEYS;
  stop = stop < p.total_k ? stop : (int64_t)p.total_k;
  const u32x4 zero = {0u, 0u, 0u, 0u};
  for (int64_t i = threadIdx.x; i < (stop - first) * (D / 8); i += blockDim.x) {
    const int64_t row = first + i / (D / 8);
    const int c = (int)(i % (D / 8));
    *(u32x4 *)(p.dk + row * p.dk_s + (int64_t)hk * p.dk_h + c * 16) = zero;
    *(u32x4 *)(p.dv + row * p.dv_s + (int64_t)hk * p.dv_h + c * 16) = zero;
  }
}

// ---- Items cut into parts (PARTS instantiations) -------------------------------------------------------
// One workgroup per item leaves the chip idle when there are few items, and under a causal mask over ragged sequences
// the longest item is several times the average.  An item's range of blocks is then cut into parts, one workgroup
// each; all leave their fp32 accumulators in the workspace and the one that arrives last adds them up in the order of
// the parts, so the result does not depend on the order of arrival (the stores and the counter as in ItemParts).
// Accumulators of a wavefront at `at` (+ 4 * lane): NT blocks of 16 registers, [register / 4][lane][4].
template <int NT>
__device__ __forceinline__ void bwd_leave_part(const f32x16 *acc, float *at) {
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4)
      part_store4(at + (t * 4 + i4) * 256, f32x4{acc[t][4 * i4], acc[t][4 * i4 + 1], acc[t][4 * i4 + 2], acc[t][4 * i4 + 3]});
}
// whether this workgroup is the last of the item's `count` to arrive; `flag` is a word of LDS nobody reads any more
// after the barrier at the start
__device__ __forceinline__ bool bwd_last_part(uint32_t *counter, int count, int *flag) {
  parts_arrived();
  __syncthreads();
  if (threadIdx.x == 0) {
    const bool last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == (uint32_t)count;
    if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = last;
  }
  __syncthreads();
  if (!*flag) return false;
  parts_acquire();
  return true;
}
template <int NT>
__device__ __forceinline__ void bwd_sum_parts(f32x16 *acc, const float *first, size_t stride, int count) {
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
#pragma unroll 2
  for (int pt = 0; pt < count; ++pt) {
    const float *at = first + (size_t)pt * stride;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const f32x4 v = *(const f32x4 *)(at + (t * 4 + i4) * 256);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[t][4 * i4 + j] += v[j];
      }
  }
}
// Cut of n blocks into at most max_parts parts of at least min_len (part i: blocks i * per .. )
struct BwdCut {
  int per, count;
  __device__ __forceinline__ BwdCut(int n, int max_parts, int min_len) {
    const int even = (n + max_parts - 1) / max_parts;
    per = even > min_len ? even : min_len;
    count = (n + per - 1) / per;
    if (count < 1) count = 1;
  }
};
// What a workgroup of the D = 128 dK/dV kernel keeps of its part in LDS, where no registers are left for it.
struct BwdPartRecord {
  float *first;        // partial accumulators of the item's first part
  uint32_t *counter;
  int part, count;
};
// The dK/dV kernels' share of a k block: the (q block, q head of the group) pairs, q block by q block, from the first
// q block with a row that sees a key of the workgroup (causal) to the sequence's last; one part's are [u0, u1) of them.
struct BwdKeyPart {
  int qb_first, r_first, qb_last, r_last_end;   // q blocks qb_first .. qb_last, heads r_first .. of the first, .. r_last_end - 1 of the last
  int count;
  __device__ __forceinline__ BwdKeyPart(const BwdParams &p, int qb_begin, int qb_end, int shift, int wg_first_key, int part) {
    int skip = 0;
    if (p.causal) skip = min(max(0, wg_first_key - shift) / p.qbs, qb_end - qb_begin);
    const int units = (qb_end - qb_begin - skip) * p.ratio;
    const BwdCut cut(units, p.parts_k, p.min_units_k);
    count = cut.count;
    const int u0 = min(part * cut.per, units), u1 = min(u0 + cut.per, units);
    const int first = u0 / p.ratio, last = (u1 - 1) / p.ratio;
    qb_first = qb_begin + skip + first;
    r_first = u0 - first * p.ratio;
    qb_last = u1 > u0 ? qb_begin + skip + last : qb_first - 1;
    r_last_end = u1 - last * p.ratio;
  }
};

// The kv head and the workgroup of that head (of per_head).  Workgroup ids go round the eight XCDs, each with its own L2.
// With a multiple of eight kv heads XCD x works on the heads x, x + 8, ..., one after the other: the workgroups that share an
// L2 then read one head of one sequence at a time, and every XCD has the same amount of work whatever the sequence lengths.
// Any other number of heads goes round with the ids: with 1, 2 or 4 of them an XCD still sees one head only, and the
// heaviest workgroups of all heads start before the light ones of any (4 heads: 228 -> 195 and 533 -> 456 us backward).
__device__ __forceinline__ void bwd_decode_grid(const BwdParams &p, unsigned per_head, int &hk, int &bx) {
  const unsigned nhk = gridDim.x / per_head;
  if (p.xcd_heads) {
    const unsigned t = blockIdx.x >> 3;
    hk = (int)(blockIdx.x & 7u) + 8 * (int)(t / per_head);
    bx = (int)(t % per_head);
  } else if (nhk > 1) {
    hk = (int)(blockIdx.x % nhk);
    bx = (int)(blockIdx.x / nhk);
  } else {
    hk = blockIdx.y;
    bx = blockIdx.x;
  }
}

// ---- dQ ----------------------------------------------------------------------------------------------
template <int D, typename E, bool PARTS>
__global__ __launch_bounds__(kThreads, 2) void hbsa_bwd_dq_kernel(BwdParams p) {
  using T = BwdTile<D>;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  // three K tiles and two V tiles, filled straight from global memory, in the layout that serves the reads by
  // rows and the transposing reads (BwdTile::swz_both)

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g32 = lane >> 5, l32 = lane & 31;
  int hk, bx;
  bwd_decode_grid(p, (unsigned)(p.nqb * p.nsub) * (PARTS ? (unsigned)p.parts_q : 1u), hk, bx);
  int part = 0, nparts = 1;
  const int per_part = p.nqb * p.nsub;
  if constexpr (PARTS) {
    part = bx / per_part;
    bx -= part * per_part;
  }
  // last q blocks first: under a causal mask they are the long ones, and the grid should not end on them
  const int qb_rev = bx / p.nsub, sub = bx - qb_rev * p.nsub;
  const int qb = p.nqb - 1 - qb_rev;
  const uint32_t *bits = p.bits + ((size_t)hk * p.nqb + qb) * p.wpr;
  const uint32_t first_words = !PARTS && lane < p.wpr ? bits[lane] : 0u;
  const QBlockInfo inf = p.info[qb];
  if (inf.rows <= 0) return;   // a q block with no row inside the tensors (its sequence did not fit them)
  int blk_begin = 0, blk_end = inf.nkblk;   // k blocks of this part
  if constexpr (PARTS) {
    const BwdCut cut(min(inf.nkblk, (inf.kmax + p.kbs - 1) / p.kbs), p.parts_q, p.min_blocks_q);
    nparts = cut.count;
    if (part >= nparts) return;
    blk_begin = part * cut.per;
    blk_end = min(inf.nkblk, blk_begin + cut.per);
  }

  const int slot = sub * 4 + wave;
  const int head_in_group = slot / p.wps;
  const int row0 = (slot % p.wps) * kWaveRows;
  const int nrows = min(kWaveRows, inf.rows - row0);
  const bool active = head_in_group < p.ratio && nrows > 0;
  const int hq = hk * p.ratio + head_in_group;

  // Asked for together: the rows of Q, dO and O, and below the first tiles.  (One after the other they cost every workgroup two
  // waits for memory before its first product.)
  short8v qf[T::KSTEPS], dof[T::KSTEPS], of[T::KSTEPS];   // Q^T, dO^T and O^T fragments: lane holds row l32, d = 16*ks + 8*g32 .. +7
  float row_lse = 0.f;
  const int my_row = inf.row_begin + min(row0 + l32, inf.rows - 1);
  if (active) {
    const int64_t first = inf.row_begin + row0;
    row_lse = p.lse[(int64_t)my_row * p.nhead_q + hq];
    bwd_request_rows<D>(p.dout + first * p.do_s + (int64_t)hq * p.do_h, p.do_s, nrows - 1, lane, dof);
    bwd_request_rows<D>(p.out + first * p.o_s + (int64_t)hq * p.o_h, p.o_s, nrows - 1, lane, of);
    bwd_request_rows<D>(p.q + first * p.q_s + (int64_t)hq * p.q_h, p.q_s, nrows - 1, lane, qf);
  } else {
#pragma unroll
    for (int ks = 0; ks < T::KSTEPS; ++ks) { qf[ks] = short8v{0, 0, 0, 0, 0, 0, 0, 0}; dof[ks] = of[ks] = qf[ks]; }
  }
  const int lane_kvis = inf.q_pos + min(row0 + l32, inf.rows - 1) + inf.shift;   // last key position the row sees (causal)
  const int wave_kvis_min = inf.q_pos + min(row0, inf.rows - 1) + inf.shift;      // ... the wavefront's first row sees
  const char *kg = p.k + (int64_t)hk * p.k_h + (int64_t)inf.key_begin * p.k_s;
  const char *vg = p.v + (int64_t)hk * p.v_h + (int64_t)inf.key_begin * p.v_s;

  // the tile sequence: 64-key tiles of the kept k blocks, cut at the last key any row of the block sees
  int j = -1, kpos = 0;
  int word_base = (PARTS ? blk_begin & ~31 : 0) - 32;      // k block of bit 0 of the word being walked
  uint32_t word_left = 0;   // its kept blocks not visited yet
  // The bit row is read once, a word per lane (64 words = 2048 k blocks at a time), so that no load and its wait
  // stand between two tiles.
  const int last_word = (blk_end - 1) >> 5;
  const int word_at = PARTS ? ((blk_begin >> 5) & ~63) + lane : lane;
  uint32_t row_words = PARTS ? (word_at <= last_word ? bits[word_at] : 0u) : first_words;
  if (word_at > last_word) row_words = 0u;   // (only the words of the sequence's blocks have been written)
  auto next_tile = [&]() -> bool {
    if (j >= 0) {
      kpos += kTileKeys;
      if (kpos < min((j + 1) * p.kbs, inf.kmax)) return true;
    }
    while (word_left == 0) {   // next word of the bit row: 32 k blocks, kept or not
      word_base += 32;
      if (word_base >= blk_end) return false;
      const int w = word_base >> 5;
      if (w >= 64 && (w & 63) == 0) {   // beyond 2048 k blocks: the next 64 words, waited for here so that no other path waits
        row_words = w + lane <= last_word ? bits[w + lane] : 0u;
        __builtin_amdgcn_s_waitcnt(0x0F70);
      }
      word_left = (uint32_t)__builtin_amdgcn_readlane((int)row_words, w & 63);
      if constexpr (PARTS) {
        if (word_base < blk_begin) word_left &= ~0u << (blk_begin - word_base);
        if (word_base + 32 > blk_end) word_left &= ~0u >> (word_base + 32 - blk_end);
      }
    }
    j = word_base + __builtin_ctz(word_left);
    word_left &= word_left - 1;
    kpos = j * p.kbs;   // below kmax: the pre-pass cleared the bits of blocks no row can see
    return true;
  };
  auto tile_valid = [&]() { return min(kTileKeys, min((j + 1) * p.kbs, inf.kmax) - kpos); };
  // A tile's chunks over four wavefronts: one load of a wavefront fills 1024 bytes (RPL rows); load i of
  // wavefront w the rows RPL * (4 * i + w) .. + RPL - 1; lane l the chunk position l % CPR of row l / CPR
  // of those, which holds the row's chunk (l % CPR) ^ swz_both(row).
  constexpr int RPL = 1024 / T::RB, LOADS = 64 / (4 * RPL);
  const int ld_row = RPL * wave + lane / T::CPR;                                  // + 4 * RPL * i
  const uint32_t ld_chunk = (uint32_t)(((lane % T::CPR) ^ T::swz_both(ld_row)) * 16);
  const uint32_t k_s32 = (uint32_t)p.k_s, v_s32 = (uint32_t)p.v_s;              // the host checks that they fit
  const uint32_t k_voff = (uint32_t)ld_row * k_s32 + ld_chunk, v_voff = (uint32_t)ld_row * v_s32 + ld_chunk;   // of a full tile's first load
  const uint32_t tiles_addr = (uint32_t)(uintptr_t)HBSA_AS3(lds) + (uint32_t)wave * 1024u;
  // LDS: three K tiles, then two V tiles.  K tiles are requested two tiles ahead, V tiles one (with two workgroups
  // of 5 tiles of D = 128 a CU's LDS is full).
  auto fetch_one = [&](uint32_t dst, const char *src, int64_t stride, uint32_t s32, uint32_t full_voff, int valid) {
    if (valid == kTileKeys) {   // a full tile: the loads differ in their scalar base only
#pragma unroll
      for (int i = 0; i < LOADS; ++i) bwd_dma16(dst + (uint32_t)(i * 4 * 1024), src + (int64_t)(4 * RPL * i) * stride, full_voff);
    } else {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const uint32_t rr = (uint32_t)min(ld_row + 4 * RPL * i, valid - 1);   // rows past the end repeat the last one (masked later)
        bwd_dma16(dst + (uint32_t)(i * 4 * 1024), src, rr * s32 + ld_chunk);
      }
    }
  };
  auto fetch_k = [&](int kb, int at, int valid) {
    fetch_one(tiles_addr + (uint32_t)(kb * T::TILE_BYTES), kg + (int64_t)at * p.k_s, p.k_s, k_s32, k_voff, valid);
  };
  auto fetch_v = [&](int vb, int at, int valid) {
    fetch_one(tiles_addr + (uint32_t)((3 + vb) * T::TILE_BYTES), vg + (int64_t)at * p.v_s, p.v_s, v_s32, v_voff, valid);
  };
  bool have_c = next_tile(), have_n = false;   // the current tile exists; the one after it exists (its K is requested)
  int kpos_c = 0, valid_c = 0, kpos_n = 0, valid_n = 0;
  int kb = 0, vb = 0;   // K and V buffer of the current tile
  if (have_c) {
    kpos_c = kpos;
    valid_c = tile_valid();
    fetch_k(0, kpos_c, valid_c);
    fetch_v(0, kpos_c, valid_c);
    have_n = next_tile();
    if (have_n) {
      kpos_n = kpos;
      valid_n = tile_valid();
      fetch_k(1, kpos_n, valid_n);
    }
  }
  float lse2 = INFINITY, dlt = 0.f;         // a row that takes no part gets P = exp2(-inf) = 0
  if (active) {
    lse2 = row_lse == -INFINITY ? INFINITY : row_lse * kLog2e;
    bwd_place_rows<D>(dof);
    bwd_place_rows<D>(of);
    bwd_place_rows<D>(qf);
    // delta = sum over d of dO * O of the row: this lane's half of the head dim, then the other half's from lane + 32.
    // Every (row, q head) belongs to exactly one wavefront of this grid, which also leaves it for the dK/dV kernel.
#pragma unroll
    for (int ks = 0; ks < T::KSTEPS; ++ks) {
      const u32x4 a = __builtin_bit_cast(u32x4, dof[ks]), b = __builtin_bit_cast(u32x4, of[ks]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        dlt += E::lo(a[j]) * E::lo(b[j]);
        dlt += E::hi(a[j]) * E::hi(b[j]);
      }
    }
    dlt = half_sum(dlt);
    if (g32 == 0 && l32 < nrows && (!PARTS || part == 0)) {
      p.delta[(int64_t)hq * p.total_q + my_row] = -dlt;
      p.lse2[(int64_t)hq * p.total_q + my_row] = lse2;
    }
  }
  f32x16 acc[T::DT];
#pragma unroll
  for (int dt = 0; dt < T::DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;

  // Operand addresses of the K tile in use: they move to the next buffer with one addition per tile instead of
  // one per read (the V tile's reads add the distance between the two buffers in use).
  BwdOperandOffsets<D> off;
  off.init(lane);
  {
    const uint32_t lds_base = (uint32_t)(uintptr_t)HBSA_AS3(lds);
#pragma unroll
    for (int ks = 0; ks < T::KSTEPS; ++ks) off.rows[ks] += lds_base;
#pragma unroll
    for (int dt = 0; dt < T::DT; ++dt) off.tr[dt] += lds_base;   // a multiple of 64: the second read's "^ 32" still holds
  }
  int off_buf = 0;   // the buffer they point to
  // Reads of one half tile's two chains S^T = K Q^T and dP^T = V dO^T: K and V rows in turn, PF under way
  constexpr int PF = 4, NC = 2 * T::KSTEPS;
  static_assert(NC >= PF, "the first reads of a half are issued as one group");
  static_assert(LOADS <= 15, "vmcnt immediate");
  // What was loaded so far (the rows' Q above all, first used in the loop) has arrived before the loop begins, and with it the
  // tiles requested behind it: the compiler counts only the loads it knows, and a wait of its own for them inside the loop would
  // also wait for every tile under way.
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
  while (have_c) {
    const int cur_kpos = kpos_c, valid = valid_c, cur_kb = kb, cur_vb = vb;
    // This wavefront's part of the tile has landed; the K loads of the tile after it (requested last; a
    // wavefront's loads return in order) may still be under way.
    if (have_n) __builtin_amdgcn_s_waitcnt(0x0F70 | LOADS);   // vmcnt(LOADS)
    else __builtin_amdgcn_s_waitcnt(0x0F70);                  // vmcnt(0)
    __syncthreads();   // ... every wavefront's, and the buffers of the tile before have been read by all
    if (have_n) fetch_v(vb ^ 1, kpos_n, valid_n);
    const bool have_nn = have_n && next_tile();
    kpos_c = kpos_n;
    valid_c = valid_n;
    have_c = have_n;
    if (have_nn) {
      kpos_n = kpos;
      valid_n = tile_valid();
      fetch_k(kb == 0 ? 2 : kb - 1, kpos_n, valid_n);   // two tiles ahead
    }
    have_n = have_nn;
    kb = kb == 2 ? 0 : kb + 1;
    vb ^= 1;
    if (!active) continue;
    if (off_buf != cur_kb) {
      const uint32_t step = (uint32_t)((cur_kb - off_buf) * T::TILE_BYTES);
#pragma unroll
      for (int ks = 0; ks < T::KSTEPS; ++ks) off.rows[ks] += step;
#pragma unroll
      for (int dt = 0; dt < T::DT; ++dt) off.tr[dt] += step;
      off_buf = cur_kb;
    }
    const uint32_t v_from_k = (uint32_t)((3 + cur_vb - cur_kb) * T::TILE_BYTES);   // from a K tile address to the V tile's
    int lim = valid;   // keys of the tile below lim are visible to this lane's row
    if (p.causal) lim = min(lim, lane_kvis - cur_kpos + 1);
    lim -= 4 * g32;
    short8v rb[PF];
    auto chain_read = [&](auto h_, auto i_) {
      constexpr int h = decltype(h_)::value, i = decltype(i_)::value;
      if constexpr (i & 1) rb[i % PF] = lds_read_b128<h * 32 * T::RB>(off.rows[i >> 1] + v_from_k);
      else rb[i % PF] = lds_read_b128<h * 32 * T::RB>(off.rows[i >> 1]);
    };
    // edge: some key of the tile is hidden from some row of the wavefront (the tile's end, or the causal
    // diagonal); elsewhere the per-element comparison and select are left out.  Rows past the block's end
    // have lse2 = +inf and so P = 0 either way.
    const bool edge = valid < kTileKeys || (p.causal && cur_kpos + valid - 1 > wave_kvis_min);
    auto half = [&](auto h_) {
      constexpr int h = decltype(h_)::value;
      f32x16 s, dp;
#pragma unroll
      for (int i = 0; i < 16; ++i) { s[i] = 0.f; dp[i] = 0.f; }
      static_for<0, NC>([&](auto i_) {
        constexpr int i = decltype(i_)::value;
        constexpr int ahead = (NC - 1 - i) < (PF - 1) ? (NC - 1 - i) : (PF - 1);
        lds_wait1<ahead>(rb[i % PF]);
        if constexpr (i & 1) dp = E::mfma(rb[i % PF], dof[i >> 1], dp);
        else s = E::mfma(rb[i % PF], qf[i >> 1], s);
        if constexpr (i + PF < NC) chain_read(h_, std::integral_constant<int, i + PF>{});
      });
      // The K^T operands of this half's first dQ products are on their way while the vector ALU forms dS, and
      // behind them (first half) the first reads of the second half's chains.
      short4v tb[2][2 * T::DT];
      bwd_issue_transposed<D, 2 * h>(off, 0u, tb[0]);
      if constexpr (h == 0)
        static_for<0, PF>([&](auto i_) { chain_read(std::integral_constant<int, 1>{}, i_); });
      short8v lo, hi;
      auto form_ds = [&](auto edge_) {
        float e[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], p.c, -lse2));
          if constexpr (decltype(edge_)::value) pv = 32 * h + 8 * (i >> 2) + (i & 3) < lim ? pv : 0.f;
          e[i] = pv * (dp[i] - dlt);
        }
        bwd_pack<E>(e, lo, hi);
      };
      if (edge) form_ds(std::true_type{});
      else form_ds(std::false_type{});
      // the second key group's operands travel during the first group's products (the registers for both
      // at once, next to dS in the making, are not there)
      bwd_issue_transposed<D, 2 * h + 1>(off, 0u, tb[1]);
      bwd_wait_transposed<D, 2 * T::DT + (h == 0 ? PF : 0)>(tb[0]);
      bwd_transposed_products<D, E>(tb[0], lo, acc);
      bwd_wait_transposed<D, 0>(tb[1]);
      bwd_transposed_products<D, E>(tb[1], hi, acc);
    };
    static_for<0, PF>([&](auto i_) { chain_read(std::integral_constant<int, 0>{}, i_); });
    half(std::integral_constant<int, 0>{});
    half(std::integral_constant<int, 1>{});
  }
  if constexpr (PARTS) {
    if (nparts > 1) {
      constexpr size_t kWaveFloats = (size_t)T::DT * 1024;   // of one wavefront's accumulators
      const uint32_t item = (uint32_t)hk * (uint32_t)per_part + (uint32_t)bx;
      float *first = p.parts + ((size_t)item * p.parts_q * 4 + wave) * kWaveFloats + lane * 4;
      if (active) bwd_leave_part<T::DT>(acc, first + (size_t)part * 4 * kWaveFloats);
      if (!bwd_last_part(p.arrivals + item, nparts, (int *)lds)) return;
      if (active) bwd_sum_parts<T::DT>(acc, first, 4 * kWaveFloats, nparts);
    }
  }
  if (active) bwd_store_rows<D, E>(p.dq + (int64_t)(inf.row_begin + row0) * p.dq_s + (int64_t)hq * p.dq_h, p.dq_s, nrows, acc, p.scale, lane);
}

// ---- The tiles of a k block, for the dK/dV kernels: a list in LDS, made once by one wavefront.  (With every
// wavefront walking the mask column tile by tile, a third of what it issued was that walk: 148 scalar instructions a tile.)
constexpr int kBwdListCap = 256;   // entries: in-sequence position of the first row | q head of the group << 7, rows; a multiple of 64
struct BwdTileRange {
  int qb_begin;         // the sequence's first q block
  int qb_low, qb_end;   // q blocks of the list
  int row0, qlen;       // first query row and query count of the sequence
  int r_last_end;       // q heads of the group below it are the last block's, ...
  int r_first;          // ... those from it on the first one's (a part's share; the others' are all)
  int first_row;        // in-sequence position of the first row that sees a key of the workgroup
};
// lane i: the word at bit row qb_end - 1 - i (by falling q block) of a mask column, zero outside of [low, end)
__device__ __forceinline__ uint32_t bwd_column_word(const BwdParams &p, const uint32_t *column, int first, int low, int end, int lane) {
  const int g = first + 63 - lane;
  return g >= low && g < end ? column[(size_t)g * p.wpr] : 0u;
}
// Entries [chunk_base, chunk_base + kBwdListCap) of the tiles, last q block first, to `list`; returns how many there are in all.
// first: the column's words of the last 64 q blocks, if they have been loaded.
template <int ROWS>   // of a tile
__device__ __forceinline__ int bwd_key_tiles(const BwdParams &p, const BwdTileRange &t, const uint32_t *column, int bit, const uint32_t *first,
                                             int chunk_base, u32x2 *list, int lane) {
  int total = 0;
  for (int base = t.qb_end - 64; base + 63 >= t.qb_low; base -= 64) {
    const uint32_t word = first != nullptr && base == t.qb_end - 64 ? *first : bwd_column_word(p, column, base, t.qb_low, t.qb_end, lane);
    const int qb = base + 63 - lane, pos = (qb - t.qb_begin) * p.qbs;
    const int rows = min(p.qbs, t.qlen - pos), skip = max(0, t.first_row - pos);   // rows of the block, and those before the first that sees a key
    int heads = 0, tiles = 0, r0 = 0;
    if (((word >> bit) & 1u) != 0 && skip < rows) {
      r0 = qb == t.qb_low ? t.r_first : 0;
      heads = (qb == t.qb_end - 1 ? t.r_last_end : p.ratio) - r0;
      tiles = (rows + ROWS - 1) / ROWS - skip / ROWS;
    }
    const int mine = max(heads, 0) * tiles;
    int incl = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(incl, off);
      if (lane >= off) incl += y;
    }
    int to = total + incl - mine - chunk_base;
    for (int r = r0; r < r0 + heads; ++r)
      for (int row = skip & ~(ROWS - 1); row < rows; row += ROWS, ++to)
        if (tiles > 0 && to >= 0 && to < kBwdListCap) list[to] = u32x2{(uint32_t)(pos + row), (uint32_t)r << 7 | (uint32_t)min(ROWS, rows - row)};
    total += __builtin_amdgcn_readlane(incl, 63);
  }
  return total;
}

// ---- dK, dV (head dims up to 64) ---------------------------------------------------------------------
// Four wavefronts; K^T and V^T of a wavefront's 32 keys stay in registers.  The Q and dO tiles go straight
// into LDS like the dQ kernel's (one layout, one barrier a step).  k blocks of up to 64 keys fill two 32-key slots (SPLIT):
// two wavefronts work on one 64-row tile and the other two on the next one, a step is two tiles, and the two sums are added through
// LDS at the end; two buffers, one step ahead.  Larger blocks fill four slots with one tile a step in three buffers, two
// steps ahead; in the narrow rest of a block (at most two slots) two wavefronts share a slot and take the upper and lower 32
// rows of every tile.
// What bounds it: a tile is one chain from S to dK, and the wavefronts on the longest k blocks have a SIMD to themselves when the
// others have ended, so that it is what one wavefront issues and waits for: of 3270 cycles a tile and wavefront 1530
// were instructions (590 of them the walk over the mask, a tile at a time), 1120 waits for LDS and the barrier, one read after another.  Hence
// the tile list (bwd_key_tiles), two tiles a barrier, operand reads issued by hand, dP started at -delta, both halves of a tile
// unrolled, the second one's first reads before the first one's last products.  6 x 300 .. 4000 tokens, 16 / 4 heads, 64-key
// blocks, keep 0.4: 141 us, with the list and two tiles a step by a workgroup of eight wavefronts 124, in this form 115, dP from
// -delta and no refill of the list inside the loop 109, halves unrolled 100.  dQ + dK/dV + forward: 1 x 8000, 32 / 1 heads, 838 ->
// 713; 6 x 4000, 16 / 4, 531 -> 497; 4 x 8192, 16 heads, 128-key blocks, 1537 -> 1521; head dim 32, 4 x 8192, 1008 -> 959.
// (217 registers at head dim 64, two wavefronts a SIMD.  Three of 165 registers were the better form of the kernel before where there
// were more than 4.5 items a CU; this one is faster there, too: 8 x 500 .. 3000, 32 / 8, 128-key blocks, 489 -> 466.)
template <int D, typename E, bool PARTS, bool SPLIT>
__global__ __launch_bounds__(kThreads, 2) void hbsa_bwd_dkv_kernel(BwdParams p) {
  static_assert(D <= 64, "head dim 128 has its own kernel");
  using T = BwdTile<D>;
  // SPLIT (k blocks of up to 64 keys, two slots of 32): two wavefronts work on one tile and the other two on the next one
  constexpr int TEAMS = SPLIT ? 2 : 1, WAVES = 4 / TEAMS, BUFS = SPLIT ? 2 : 3;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  // buffer s of a team's tiles (BUFS of them): Q rows at (s * TEAMS + team) * 2 * TILE_BYTES, dO rows one tile further
  float *rowv = (float *)(lds + TEAMS * BUFS * 2 * T::TILE_BYTES);    // and of it: [64] log2-domain log-sum-exp of the tile's rows, [64] their -delta
  u32x2 *list = (u32x2 *)(rowv + TEAMS * BUFS * 128);             // [kBwdListCap] tiles, see bwd_key_tiles
  int *list_total = (int *)(list + kBwdListCap);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) % WAVES;   // of the team
  const int team = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / WAVES;
  const int g32 = lane >> 5, l32 = lane & 31;
  int hk, bx;
  bwd_decode_grid(p, (unsigned)(p.nkb * p.nsub_k) * (PARTS ? (unsigned)p.parts_k : 1u), hk, bx);
  int part = 0;
  const int per_part = p.nkb * p.nsub_k;
  if constexpr (PARTS) {
    part = bx / per_part;
    bx -= part * per_part;
  }
  const int kb_at = bx / p.nsub_k, sub = bx - kb_at * p.nsub_k;
  const int kb = p.order_k != nullptr ? p.order_k[kb_at] : kb_at;

  const BwdSequence seq(p, kb, lane);
  if (seq.qb0 < 0 || seq.qb0 > p.nqb) return;   // (== nqb: sequences without queries at the batch's end, whose keys get zeros)
  // asked for together: the sequence's record, the mask column's first 64 words, the resident operands
  const uint32_t record = bwd_first_record(p, seq, lane);
  const int kbl = kb - seq.kb0;                      // in-sequence index of the k block
  const int k0 = seq.k0, klen = seq.k1 - k0;
  const bool fits = seq.fits(p, kb);
  const uint32_t first_word = !PARTS && fits ? bwd_column_word(p, p.bits + (size_t)hk * p.nqb * p.wpr + (kbl >> 5), seq.qb1 - 64, seq.qb0, seq.qb1, lane) : 0u;
  const int krows = min(p.kbs, klen - kbl * p.kbs);  // keys in the block
  const int wg_keys = min(4 * kWaveRows, p.kbs - sub * 4 * kWaveRows);   // by the block size: the same for every k block
  const bool shared_slots = !SPLIT && wg_keys <= 2 * kWaveRows;          // two wavefronts per 32-key slot
  const int slot = shared_slots ? (wave & 1) : wave;
  const int rows_half = shared_slots ? (wave >> 1) : 0;                  // which 32 rows of a tile (shared slots)
  const int row0 = (sub * 4 + slot) * kWaveRows;
  const int nrows = min(kWaveRows, krows - row0);
  const bool active = nrows > 0;
  const int key_pos = kbl * p.kbs + min(row0 + l32, krows - 1);   // in-sequence position of this lane's key
  const int wg_first_key = kbl * p.kbs + sub * 4 * kWaveRows;     // of the workgroup's first key
  const int wave_key_max = kbl * p.kbs + min(row0 + kWaveRows - 1, krows - 1);   // position of the wavefront's last key

  short8v kf[T::KSTEPS], vf[T::KSTEPS];   // K^T and V^T fragments: lane holds key l32, d = 16*ks + 8*g32 .. +7
  if (active && fits) {
    const int64_t first = k0 + kbl * p.kbs + row0;
    bwd_request_rows<D>(p.k + first * p.k_s + (int64_t)hk * p.k_h, p.k_s, nrows - 1, lane, kf);
    bwd_request_rows<D>(p.v + first * p.v_s + (int64_t)hk * p.v_h, p.v_s, nrows - 1, lane, vf);
  } else {
#pragma unroll
    for (int ks = 0; ks < T::KSTEPS; ++ks) { kf[ks] = short8v{0, 0, 0, 0, 0, 0, 0, 0}; vf[ks] = kf[ks]; }
  }
  f32x16 acc_k[T::DT], acc_v[T::DT];
#pragma unroll
  for (int dt = 0; dt < T::DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) { acc_k[dt][i] = 0.f; acc_v[dt][i] = 0.f; }

  // the tile sequence: for every q block of the sequence that keeps this k block, for every q head of
  // the group, the block's rows in 64-row tiles (under a causal mask only those with a row that sees a
  // key of this workgroup)
  int shift = 0, nparts = 1, total = 0;
  BwdTileRange range = {seq.qb0, seq.qb0, 0, 0, 0, p.ratio, 0, 0};
  if (seq.qb0 < seq.qb1) {
    if (!bwd_record_holds(seq, record)) {
      bwd_zero_keys<D, 4 * kWaveRows>(p, seq, kb, sub, hk);
      return;
    }
    shift = __builtin_amdgcn_readlane((int)record, 5);
    range.row0 = __builtin_amdgcn_readlane((int)record, 0);
    range.qlen = klen - shift;
    range.qb_end = seq.qb1;
    range.first_row = p.causal ? wg_first_key - shift : 0;
  }
  if (!fits) return;   // (a sequence without queries that lies outside of the tensors)
  int qb_low = seq.qb0;
  if constexpr (PARTS) {
    const BwdKeyPart share(p, seq.qb0, range.qb_end, shift, wg_first_key, part);
    nparts = share.count;
    if (part >= nparts) return;
    qb_low = share.qb_first;
    range.r_first = share.r_first;
    range.r_last_end = share.r_last_end;
    range.qb_end = share.qb_last + 1;
  }
  range.qb_low = qb_low;
  const uint32_t *column = p.bits + (size_t)hk * p.nqb * p.wpr + (kbl >> 5);
  if (range.qb_low < range.qb_end && range.qlen > 0) {
    if (threadIdx.x < 64) {
      const int n = bwd_key_tiles<64>(p, range, column, kbl & 31, PARTS ? nullptr : &first_word, 0, list, lane);
      if (lane == 0) *list_total = n;
    }
    __syncthreads();
    total = __builtin_amdgcn_readfirstlane(*list_total);
  }
  // (placement of a tile's chunks over the four wavefronts: see hbsa_bwd_dq_kernel)
  constexpr int RPL = 1024 / T::RB, LOADS = 64 / (WAVES * RPL);
  const int ld_row = RPL * wave + lane / T::CPR;
  const uint32_t ld_chunk = (uint32_t)(((lane % T::CPR) ^ T::swz_both(ld_row)) * 16);
  const uint32_t q_s32 = (uint32_t)p.q_s, do_s32 = (uint32_t)p.do_s;   // the host checks that they fit
  const uint32_t q_voff = (uint32_t)ld_row * q_s32 + ld_chunk, do_voff = (uint32_t)ld_row * do_s32 + ld_chunk;   // of a full tile's first load
  const char *q_base = p.q + (int64_t)range.row0 * p.q_s + (int64_t)hk * p.ratio * p.q_h, *g_base = p.dout + (int64_t)range.row0 * p.do_s + (int64_t)hk * p.ratio * p.do_h;
  const int64_t row_base = (int64_t)hk * p.ratio * p.total_q + range.row0;
  const uint32_t tiles_addr = (uint32_t)(uintptr_t)HBSA_AS3(lds) + (uint32_t)(team * 2 * T::TILE_BYTES + wave * 1024);
  const uint32_t row_addr = (uint32_t)(uintptr_t)HBSA_AS3(rowv) + (uint32_t)team * 512u;
  // Loads of one tile per wavefront: LOADS of Q and of dO, and in wavefront 0 the two of the rows' values
  auto fetch = [&](int buf, int pos, int valid, int r) {   // `valid` rows of q head r of the group, from in-sequence position pos on
    const char *qsrc = q_base + (uint64_t)(uint32_t)pos * q_s32 + (int64_t)r * p.q_h;
    const char *gsrc = g_base + (uint64_t)(uint32_t)pos * do_s32 + (int64_t)r * p.do_h;
    const uint32_t dst = tiles_addr + (uint32_t)(buf * TEAMS * 2 * T::TILE_BYTES);
    if (valid == 64) {   // a full tile: the loads differ in their scalar base only
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        bwd_dma16(dst + (uint32_t)(i * WAVES * 1024), qsrc + (uint64_t)(uint32_t)(WAVES * RPL * i) * q_s32, q_voff);
        bwd_dma16(dst + (uint32_t)(T::TILE_BYTES + i * WAVES * 1024), gsrc + (uint64_t)(uint32_t)(WAVES * RPL * i) * do_s32, do_voff);
      }
    } else {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const uint32_t rr = (uint32_t)min(ld_row + WAVES * RPL * i, valid - 1);   // rows past the block's end repeat its last row
        bwd_dma16(dst + (uint32_t)(i * WAVES * 1024), qsrc, rr * q_s32 + ld_chunk);
        bwd_dma16(dst + (uint32_t)(T::TILE_BYTES + i * WAVES * 1024), gsrc, rr * do_s32 + ld_chunk);
      }
    }
    if (wave == 0) {
      const uint32_t rvoff = (uint32_t)min(lane, valid - 1) * 4u;
      const int64_t row_at = row_base + (int64_t)r * p.total_q + pos;
      bwd_dma4(row_addr + (uint32_t)(buf * TEAMS * 512), p.lse2 + row_at, rvoff);
      bwd_dma4(row_addr + (uint32_t)(buf * TEAMS * 512 + 256), p.delta + row_at, rvoff);
    }
  };
  BwdOperandOffsets<D> off;
  off.init(lane);
  const uint32_t lds_base = (uint32_t)(uintptr_t)HBSA_AS3(lds);
  const int h_begin = shared_slots ? rows_half : 0, h_end = shared_slots ? rows_half + 1 : 2;   // 32-row halves of a tile
  for (int chunk_base = 0; chunk_base < total;) {   // ---- chunks of the tile list (usually one)
  const int entries = min(total - chunk_base, kBwdListCap);
  int n_ahead = 0;                               // tiles (of each team) fetched and not computed on yet
  int buf_f = 0, buf = 0;                        // buffer of the next fetch, and of the current tile
  int fq_a = 0, fq_b = 0, va_a = 64, va_b = 64;  // first query position and row count of those tiles (a: the older); no rows: there is none
  int at = team;                                 // this team's next entry
  u32x2 held = {0u, 0u};                         // lane i: entry i of the list's current 64
  auto issue = [&]() {   // fetches the team's next tile
    if (at - team < entries && ((at - team) & 63) == 0) {
      held = list[min(at - team + lane, kBwdListCap - 1)];
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): here, not on every tile's path
    }
    int fq = 0, va = 0;
    if (TEAMS == 1 || at < entries) {
      const uint32_t y = (uint32_t)__builtin_amdgcn_readlane((int)held.y, at & 63);
      fq = __builtin_amdgcn_readlane((int)held.x, at & 63);
      va = (int)(y & 127u);
      fetch(buf_f, fq, va, (int)(y >> 7));
    }
    if (n_ahead == 0) { fq_a = fq; va_a = va; } else { fq_b = fq; va_b = va; }
    buf_f = buf_f == BUFS - 1 ? 0 : buf_f + 1;
    ++n_ahead;
    at += TEAMS;
  };
  auto more = [&]() { return at - team < entries; };
  issue();
  if (BUFS == 3 && more()) issue();
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the resident operands have arrived, and the tiles (see hbsa_bwd_dkv8_kernel)
  if (chunk_base == 0) {
    bwd_place_rows<D>(kf);
    bwd_place_rows<D>(vf);
  }
  while (n_ahead > 0) {
    const int first_q_pos = fq_a, valid = va_a;
    // This wavefront's part of the tile has landed; the loads of the tile after it (a wavefront's loads return in
    // order) may still be under way.
    if (n_ahead >= 2 && (TEAMS == 1 || va_b > 0)) {
      if (wave == 0) __builtin_amdgcn_s_waitcnt(0x0F70 | (2 * LOADS + 2));
      else __builtin_amdgcn_s_waitcnt(0x0F70 | (2 * LOADS));
    } else {
      __builtin_amdgcn_s_waitcnt(0x0F70);
    }
    __syncthreads();   // ... every wavefront's, and the buffer of the tile before has been read by all
    const uint32_t tile_lds = lds_base + (uint32_t)((buf * TEAMS + team) * 2 * T::TILE_BYTES);
    const uint32_t rows_lds = lds_base + (uint32_t)(TEAMS * BUFS * 2 * T::TILE_BYTES + (buf * TEAMS + team) * 512);
    buf = buf == BUFS - 1 ? 0 : buf + 1;
    fq_a = fq_b;
    va_a = va_b;
    --n_ahead;
    if (more()) issue();   // ahead by one buffer less than there are
    if (!active || (TEAMS > 1 && valid == 0)) continue;
    // rows first_vis .. valid - 1 of the tile see this lane's key (what lanes without a key sum up is not stored);
    // comparisons and selects are left out where all 64 rows see all of the wavefront's keys
    int first_vis = 0;
    if (p.causal) first_vis = max(0, key_pos - shift - first_q_pos);
    const bool diagonal = p.causal && wave_key_max - shift - first_q_pos > 0;
    // Operand reads are issued by hand (BwdOperandOffsets), in the order the products need them and as far ahead as the counter
    // (15 of them) and the registers allow: with a read next to every product, a tile was 16 round trips to LDS one after another.
    const uint32_t q_t = tile_lds, g_t = q_t + (uint32_t)T::TILE_BYTES;
    constexpr int KS = T::KSTEPS, DT = T::DT;
    short8v qr[KS];
    auto half = [&](auto h_) {
      constexpr int h = decltype(h_)::value;
      constexpr bool NEXT = SPLIT && h == 0;   // the other half follows: the first reads of it go out before this one's last products
      const uint32_t h_rows = (uint32_t)h * (32 * T::RB), v_at = rows_lds + (uint32_t)(128 * h + 16 * g32);
      short8v gr[KS], lv[4], dl[4];
      short4v tg[2][2 * DT], tq[2][2 * DT];
      if constexpr (!(SPLIT && h == 1))
        static_for<0, KS>([&](auto i_) { qr[decltype(i_)::value] = lds_read_b128<0>(off.rows[decltype(i_)::value] + q_t + h_rows); });
      static_for<0, 4>([&](auto i_) { lv[decltype(i_)::value] = lds_read_b128<32 * decltype(i_)::value>(v_at); });
      static_for<0, KS>([&](auto i_) { gr[decltype(i_)::value] = lds_read_b128<0>(off.rows[decltype(i_)::value] + g_t + h_rows); });
      f32x16 s, dp;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.f;
      static_for<0, KS>([&](auto i_) {
        constexpr int i = decltype(i_)::value;
        lds_wait1<(2 * KS + 3 - i)>(qr[i]);
        s = E::mfma(qr[i], kf[i], s);
      });
      static_for<0, 4>([&](auto i_) { dl[decltype(i_)::value] = lds_read_b128<256 + 32 * decltype(i_)::value>(v_at); });
      bwd_issue_transposed<D, 0>(off, g_t + h_rows, tg[0]);
      asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(dl[0]), "+v"(dl[1]), "+v"(dl[2]), "+v"(dl[3]) : "n"(2 * DT));
#pragma unroll
      for (int i = 0; i < 16; ++i) dp[i] = __builtin_bit_cast(f32x4, dl[i >> 2])[i & 3];   // (dP starts at -delta)
      static_for<0, KS>([&](auto i_) {
        constexpr int i = decltype(i_)::value;
        lds_wait1<(2 * DT)>(gr[i]);
        dp = E::mfma(gr[i], vf[i], dp);
      });
      bwd_issue_transposed<D, 1>(off, g_t + h_rows, tg[1]);
      asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(lv[0]), "+v"(lv[1]), "+v"(lv[2]), "+v"(lv[3]) : "n"(4 * DT));
      // P and its product with dO, then dS and its product with Q
      float e[16];
      auto form_p = [&](auto short_, auto diagonal_) {
        const int left = valid - 32 * h - 4 * g32, before = first_vis - 32 * h - 4 * g32;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const f32x4 l4 = __builtin_bit_cast(f32x4, lv[a]);
#pragma unroll
          for (int bq = 0; bq < 4; ++bq) {
            float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(s[4 * a + bq], p.c, -l4[bq]));
            if constexpr (decltype(short_)::value) pv = 8 * a + bq < left ? pv : 0.f;   // (rows past the end repeat the last one)
            if constexpr (decltype(diagonal_)::value) pv = 8 * a + bq >= before ? pv : 0.f;
            e[4 * a + bq] = pv;
          }
        }
      };
      if (diagonal) form_p(std::true_type{}, std::true_type{});
      else if (valid < 64) form_p(std::true_type{}, std::false_type{});
      else form_p(std::false_type{}, std::false_type{});
      short8v lo, hi;
      bwd_pack<E>(e, lo, hi);
      bwd_wait_transposed<D, 2 * DT>(tg[0]);
      bwd_transposed_products<D, E>(tg[0], lo, acc_v);
      bwd_issue_transposed<D, 0>(off, q_t + h_rows, tq[0]);
      bwd_wait_transposed<D, 2 * DT>(tg[1]);
      bwd_transposed_products<D, E>(tg[1], hi, acc_v);
      bwd_issue_transposed<D, 1>(off, q_t + h_rows, tq[1]);
#pragma unroll
      for (int i = 0; i < 16; ++i) e[i] *= dp[i];
      bwd_pack<E>(e, lo, hi);
      if constexpr (NEXT)
        static_for<0, KS>([&](auto i_) { qr[decltype(i_)::value] = lds_read_b128<0>(off.rows[decltype(i_)::value] + q_t + (uint32_t)(32 * T::RB)); });
      bwd_wait_transposed<D, 2 * DT + (NEXT ? KS : 0)>(tq[0]);
      bwd_transposed_products<D, E>(tq[0], lo, acc_k);
      bwd_wait_transposed<D, NEXT ? KS : 0>(tq[1]);
      bwd_transposed_products<D, E>(tq[1], hi, acc_k);
    };
    if (SPLIT || h_begin == 0) half(std::integral_constant<int, 0>{});
    if (SPLIT || h_end == 2) half(std::integral_constant<int, 1>{});
  }
  chunk_base += kBwdListCap;
  if (chunk_base < total) {
    __syncthreads();
    if (threadIdx.x < 64) (void)bwd_key_tiles<64>(p, range, column, kbl & 31, nullptr, chunk_base, list, lane);
    __syncthreads();
  }
  }
  // the sums of the wavefronts that share a slot (the upper and lower rows' of a tile, the teams') go to the first of them
  // through LDS: [wavefront][slot][register][lane] floats
  const int sharers = TEAMS * (shared_slots ? 2 : 1), sharer = team * (shared_slots ? 2 : 1) + rows_half;
  if (sharers > 1) {
    constexpr int REGS = 2 * T::DT * 16;
    const int slots = shared_slots ? 2 : 4;
    __syncthreads();
    float *xch = (float *)lds + (size_t)slot * REGS * 64 + lane;
    if (sharer > 0) {
      float *mine = xch + (size_t)(sharer - 1) * slots * REGS * 64;
#pragma unroll
      for (int dt = 0; dt < T::DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          mine[(dt * 16 + i) * 64] = acc_k[dt][i];
          mine[((T::DT + dt) * 16 + i) * 64] = acc_v[dt][i];
        }
    }
    __syncthreads();
    if (sharer == 0) {
#pragma unroll 1
      for (int x = 1; x < sharers; ++x) {
        const float *theirs = xch + (size_t)(x - 1) * slots * REGS * 64;
#pragma unroll
        for (int dt = 0; dt < T::DT; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            acc_k[dt][i] += theirs[(dt * 16 + i) * 64];
            acc_v[dt][i] += theirs[((T::DT + dt) * 16 + i) * 64];
          }
      }
    }
  }
  if constexpr (PARTS) {
    if (nparts > 1) {
      constexpr size_t kWaveFloats = (size_t)2 * T::DT * 1024;   // of one slot's accumulators
      const uint32_t item = (uint32_t)hk * (uint32_t)per_part + (uint32_t)bx;
      float *at = p.parts + ((size_t)item * p.parts_k * 4 + slot) * kWaveFloats + lane * 4;
      if (sharer == 0 && active) {
        bwd_leave_part<T::DT>(acc_k, at + (size_t)part * 4 * kWaveFloats);
        bwd_leave_part<T::DT>(acc_v, at + (size_t)part * 4 * kWaveFloats + kWaveFloats / 2);
      }
      if (!bwd_last_part(p.arrivals + item, nparts, (int *)lds)) return;
      if (sharer == 0 && active) {
        bwd_sum_parts<T::DT>(acc_k, at, 4 * kWaveFloats, nparts);
        bwd_sum_parts<T::DT>(acc_v, at + kWaveFloats / 2, 4 * kWaveFloats, nparts);
      }
    }
  }
  if (sharer == 0 && active) {
    const int64_t row = k0 + kbl * p.kbs + row0;
    bwd_store_rows<D, E>(p.dk + row * p.dk_s + (int64_t)hk * p.dk_h, p.dk_s, nrows, acc_k, p.scale, lane);
    bwd_store_rows<D, E>(p.dv + row * p.dv_s + (int64_t)hk * p.dv_h, p.dv_s, nrows, acc_v, 1.f, lane);
  }
}

// ---- dK, dV at D = 128: wavefronts in two roles ---------------------------------------------------------
// The kernel above would hold K^T, V^T and both accumulators of a wavefront in registers: 256 + 238 at
// D = 128, one wavefront per SIMD.  Here two wavefronts share a 32-key slot (and a SIMD) and split the four
// products between them, each with one operand and one accumulator in registers:
//   the P wavefront  keeps K^T:  S = Q K^T,  P = exp(S - lse) (masked),   dV^T += dO^T P,   hands P over;
//   the dS wavefront keeps V^T:  dP = dO V^T,  dS = P * (dP - delta),      dK^T += Q^T dS.
// P travels through LDS in the element type, as the P wavefront packs it for its own product (4 KB per slot and
// tile), and one tile late: in the iteration in which the P wavefront works on tile t, the dS wavefront
// finishes tile t - 1 (whose dP it kept in registers) and forms dP of tile t, so one barrier per tile orders
// everything.  Tiles go from global memory straight into LDS, stored once in the layout of BwdTile::swz_both,
// and two tiles ahead (one workgroup per CU has nobody else to cover its waits for memory): four Q buffers
// (tile t - 1 is still read while tile t + 2 arrives), three for dO, and with them three sets of the
// rows' log-sum-exp and delta, which wavefront 0 loads into LDS the same way.
// What bounds it: the two roles' chains between two barriers, of which the matrix instructions are 2050 cycles a SIMD and tile, and what
// a workgroup does before its first tile, which nothing covers (at 8192 tokens with a tenth kept 8.3 us of 28.5 for 8.3 tiles).  The tiles
// come from a list (bwd_key_tiles; all eight wavefronts had walked the mask tile by tile), whose next entry is read while the barrier is waited for;
// dP starts at -delta, and the rows' values and P are read by hand ahead of the transposed operands, behind which the compiler's own reads had
// to wait for all of them.  Whole training calls, before and after: 1 x 32768 tokens, 8 heads, a tenth kept, 1255 -> 1211 us; 4 x 8192, 32
// heads, 1858 -> 1825; 64-key blocks (the shared form), 5 x 4491 .. 8593, 16 heads, 80-row blocks, 1418 -> 1315; 4 x 4096, 32 / 8 heads, 1080 -> 1029; 48-key blocks,
// 5 x 823 .. 2209, 8 / 4 heads, 186 -> 173; few items, 6 x 1734, 2 heads, 128 -> 121.
// Of the forms (which of them when, with figures: bwd_form) the narrow one has two workgroups a CU, of four wavefronts on 64 keys and tiles of 32
// rows: 66 KB of LDS and 222 registers.  In the shared one eight wavefronts do as little between two barriers, 16 products each, and all wait.
struct BwdListRecord {   // what a further chunk of the list is made from, kept in LDS: in registers over the tile loop it would spill
  BwdTileRange range;
  const uint32_t *column;
  int bit, total;
};
// Its three forms (bwd_form): rows of a tile, wavefronts and keys of a workgroup
constexpr int bwd_dkv8_rows(int form) { return form == kBwdNarrow ? 32 : 64; }
constexpr int bwd_dkv8_threads(int form) { return form == kBwdNarrow ? 256 : 512; }
constexpr int bwd_dkv8_lds(int form) {   // tiles, P records (two parities), the rows' values, the list
  return 7 * bwd_dkv8_rows(form) * 256 + 2 * (bwd_dkv8_threads(form) / 128) * (form == kBwdWide ? 2 : 1) * 2048 + 1536 + kBwdListCap * 8 +
         (int)sizeof(BwdListRecord) + (int)sizeof(BwdPartRecord);
}
template <typename E, bool PARTS, int FORM>
__global__ __launch_bounds__(bwd_dkv8_threads(FORM), FORM == kBwdNarrow ? 2 : 1) void hbsa_bwd_dkv8_kernel(BwdParams p) {
  constexpr int D = 128;
  using T = BwdTile<D>;
  constexpr int ROWS = bwd_dkv8_rows(FORM), WAVES = bwd_dkv8_threads(FORM) / 64, SLOTS = WAVES / 2;
  constexpr int NH = FORM == kBwdWide ? 2 : 1;       // 32-row halves of a tile a wavefront works on
  constexpr int KEY_SLOTS = FORM == kBwdWide ? 4 : 2;
  constexpr int TILE_BYTES = ROWS * T::RB, P_BYTES = SLOTS * NH * 2048;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  char *q_buf = lds;                                   // [4] Q tiles
  char *g_buf = lds + 4 * TILE_BYTES;                  // [3] dO tiles
  char *p_buf = lds + 7 * TILE_BYTES;                  // [2 tile parities][SLOTS][NH][2][64 lanes] eight 16-bit values
  float *rows_s = (float *)(p_buf + 2 * P_BYTES);      // [3] of the dO buffer's rows: [64] log2-domain log-sum-exp, [64] -delta
  u32x2 *list = (u32x2 *)(rows_s + 3 * 128);           // [kBwdListCap] tiles, see bwd_key_tiles
  BwdListRecord *list_s = (BwdListRecord *)(list + kBwdListCap);
  BwdPartRecord *part_s = (BwdPartRecord *)(list_s + 1);   // PARTS

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slot = wave % SLOTS, role = wave / SLOTS;   // pair of wavefronts; 0: the P wavefront, 1: the dS wavefront
  // Pair i has keys 32 i .. 32 i + 31; in the shared form pairs 0 and 2, 1 and 3 have the same 32 keys, the first ones the upper 32 rows of
  // every tile and the others the lower ones, whose sums are added through LDS at the end.
  const int key_slot = slot % KEY_SLOTS, first_row = FORM == kBwdShared ? 32 * (slot / KEY_SLOTS) : 0;
  const int g32 = lane >> 5, l32 = lane & 31;
  int hk, bx;
  bwd_decode_grid(p, (unsigned)(p.nkb * p.nsub_k) * (PARTS ? (unsigned)p.parts_k : 1u), hk, bx);
  int part = 0;
  const int per_part = p.nkb * p.nsub_k;
  if constexpr (PARTS) {
    part = bx / per_part;
    bx -= part * per_part;
  }
  const int kb_at = bx / p.nsub_k, sub = bx - kb_at * p.nsub_k;
  const int kb = p.order_k != nullptr ? p.order_k[kb_at] : kb_at;

  const BwdSequence seq(p, kb, lane);
  if (seq.qb0 < 0 || seq.qb0 > p.nqb) return;   // (== nqb: sequences without queries at the batch's end, whose keys get zeros)
  // Asked for together: the sequence's record, the mask column's first 64 words, the resident operand.  With one workgroup
  // per CU nothing covers the loads a workgroup begins with, and it has some eight tiles where 8K sequences keep a tenth.
  const uint32_t record = bwd_first_record(p, seq, lane);
  const int kbl = kb - seq.kb0;
  const int k0 = seq.k0, klen = seq.k1 - k0;
  const bool fits = seq.fits(p, kb);
  const uint32_t *column = p.bits + (size_t)hk * p.nqb * p.wpr + (kbl >> 5);
  const uint32_t first_word = !PARTS && fits ? bwd_column_word(p, column, seq.qb1 - 64, seq.qb0, seq.qb1, lane) : 0u;
  const int krows = min(p.kbs, klen - kbl * p.kbs);
  const int wg_row0 = sub * KEY_SLOTS * kWaveRows;             // first key of the workgroup inside the block
  const int row0 = wg_row0 + key_slot * kWaveRows;
  const int nrows = min(kWaveRows, krows - row0);
  const bool active = nrows > 0;
  const int key_pos = kbl * p.kbs + min(row0 + l32, krows - 1);
  const int wg_first_key = kbl * p.kbs + wg_row0;
  const int wave_key_max = kbl * p.kbs + min(row0 + kWaveRows - 1, krows - 1);   // position of the wavefront's last key

  // this wavefront's resident operand: K^T (P wavefront) or V^T (dS wavefront) of its 32 keys; lane holds
  // key l32, d = 16 * ks + 8 * g32 .. + 7
  short8v frag[T::KSTEPS];
  if (active && fits) {
    const int64_t first = k0 + kbl * p.kbs + row0;
    const int64_t stride = role == 0 ? p.k_s : p.v_s;
    bwd_request_rows<D>((role == 0 ? p.k + (int64_t)hk * p.k_h : p.v + (int64_t)hk * p.v_h) + first * stride, stride, nrows - 1, lane, frag);
  } else {
#pragma unroll
    for (int ks = 0; ks < T::KSTEPS; ++ks) frag[ks] = short8v{0, 0, 0, 0, 0, 0, 0, 0};
  }
  f32x16 acc[T::DT];   // dV^T (P wavefront) or dK^T (dS wavefront) of the 32 keys
#pragma unroll
  for (int dt = 0; dt < T::DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;

  int shift = 0, total = 0;
  BwdTileRange range = {seq.qb0, seq.qb0, seq.qb0, 0, 0, p.ratio, 0, 0};
  if (seq.qb0 < seq.qb1) {
    if (!bwd_record_holds(seq, record)) {
      bwd_zero_keys<D, KEY_SLOTS * kWaveRows>(p, seq, kb, sub, hk);
      return;
    }
    shift = __builtin_amdgcn_readlane((int)record, 5);
    range.row0 = __builtin_amdgcn_readlane((int)record, 0);
    range.qlen = klen - shift;
    range.qb_end = seq.qb1;
    range.first_row = p.causal ? wg_first_key - shift : 0;
  }
  if (!fits) return;   // (a sequence without queries that lies outside of the tensors)
  if constexpr (PARTS) {
    const BwdKeyPart share(p, seq.qb0, range.qb_end, shift, wg_first_key, part);
    if (part >= share.count) return;
    if (threadIdx.x == 0) {
      const size_t item = (size_t)hk * per_part + bx;
      *part_s = BwdPartRecord{p.parts + item * p.parts_k * WAVES * (T::DT * 1024), p.arrivals + item, part, share.count};
    }
    range.qb_low = share.qb_first;
    range.r_first = share.r_first;
    range.r_last_end = share.r_last_end;
    range.qb_end = share.qb_last + 1;
  }
  if (PARTS || (range.qb_low < range.qb_end && range.qlen > 0)) {
    if (threadIdx.x < 64) {
      const int n = range.qlen > 0 ? bwd_key_tiles<ROWS>(p, range, column, kbl & 31, PARTS ? nullptr : &first_word, 0, list, lane) : 0;
      if (lane == 0) *list_s = BwdListRecord{range, column, kbl & 31, n};
    }
    __syncthreads();
    total = __builtin_amdgcn_readfirstlane(list_s->total);
  }
  // A tile's chunks over the wavefronts: wavefront w fills rows 4 * (WAVES * i + w) .. + 3 with load i
  // (i = 0, 1), lane l the 16 bytes at chunk position l % 16 of row l / 16 of those, which hold the
  // row's chunk (l % 16) ^ swz_both(row).
  const int ld_row = 4 * wave + (lane >> 4);                              // + 4 * WAVES * i
  const uint32_t ld_chunk = (uint32_t)(((lane & 15) ^ T::swz_both(ld_row & 15)) * 16);
  const uint32_t q_s32 = (uint32_t)p.q_s, do_s32 = (uint32_t)p.do_s;      // the host checks that they fit
  const uint32_t q_addr = (uint32_t)(uintptr_t)HBSA_AS3(q_buf) + (uint32_t)wave * 1024u;
  const uint32_t g_addr = (uint32_t)(uintptr_t)HBSA_AS3(g_buf) + (uint32_t)wave * 1024u;
  const uint32_t q_voff = (uint32_t)ld_row * q_s32 + ld_chunk, g_voff = (uint32_t)ld_row * do_s32 + ld_chunk;   // of a full tile's first load
  const uint32_t row_addr = (uint32_t)(uintptr_t)HBSA_AS3(rows_s);
  const char *q_base = p.q + (int64_t)range.row0 * p.q_s + (int64_t)hk * p.ratio * p.q_h, *g_base = p.dout + (int64_t)range.row0 * p.do_s + (int64_t)hk * p.ratio * p.do_h;
  const int64_t row_base = (int64_t)hk * p.ratio * p.total_q + range.row0;
  // Loads of one tile per wavefront: two Q and two dO loads, and in wavefront 0 the two loads of the rows' values
  auto fetch = [&](int qi, int gi, int pos, int valid, int r) {   // `valid` rows of q head r of the group, from in-sequence position pos on, into Q buffer qi and dO buffer gi
    const char *qsrc = q_base + (uint64_t)(uint32_t)pos * q_s32 + (int64_t)r * p.q_h;
    const char *gsrc = g_base + (uint64_t)(uint32_t)pos * do_s32 + (int64_t)r * p.do_h;
    if (valid == ROWS) {   // a full tile: the loads differ in their scalar base only
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        bwd_dma16(q_addr + (uint32_t)(qi * TILE_BYTES + i * WAVES * 1024), qsrc + (uint64_t)(4u * WAVES * i) * q_s32, q_voff);
        bwd_dma16(g_addr + (uint32_t)(gi * TILE_BYTES + i * WAVES * 1024), gsrc + (uint64_t)(4u * WAVES * i) * do_s32, g_voff);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t rr = (uint32_t)min(ld_row + 4 * WAVES * i, valid - 1);   // rows past the block's end repeat its last row
        bwd_dma16(q_addr + (uint32_t)(qi * TILE_BYTES + i * WAVES * 1024), qsrc, rr * q_s32 + ld_chunk);
        bwd_dma16(g_addr + (uint32_t)(gi * TILE_BYTES + i * WAVES * 1024), gsrc, rr * do_s32 + ld_chunk);
      }
    }
    if (wave == 0) {   // the rows' log-sum-exp and delta, one row per lane (rows past the block's end repeat its last row)
      const uint32_t rvoff = (uint32_t)min(lane, valid - 1) * 4u;
      const int64_t row_at = row_base + (int64_t)r * p.total_q + pos;
      bwd_dma4(row_addr + (uint32_t)(gi * 512), p.lse2 + row_at, rvoff);
      bwd_dma4(row_addr + (uint32_t)(gi * 512 + 256), p.delta + row_at, rvoff);
    }
  };
  // this lane's 2 x 16 bytes of a (tile parity, slot, half) record of P
  char *p_mine = p_buf + (size_t)slot * (NH * 2048) + lane * 16;
  const uint32_t p_lds = (uint32_t)(uintptr_t)HBSA_AS3(p_mine);

  BwdOperandOffsets<D> off;
  off.init(lane);
  const uint32_t lds_base = (uint32_t)(uintptr_t)HBSA_AS3(lds);   // Q tiles at 0 .. 3 tile sizes, dO tiles at 4 .. 6
  // The loop exists once per role (the same barriers in both): with the roles as branches of one loop body the
  // register allocator keeps both roles' temporaries apart and spills.
  auto run = [&](auto role_) {
  constexpr int ROLE = decltype(role_)::value;
  for (int chunk_base = 0; chunk_base < total;) {   // ---- chunks of the tile list (usually one)
  const int entries = min(total - chunk_base, kBwdListCap);
  // Tiles are fetched two ahead: tile t lives in Q buffer t % 4 and dO buffer t % 3 (the dS wavefront still reads
  // Q of tile t - 1 in the iteration in which tile t + 2 arrives).
  int n_ahead = 0;                               // tiles fetched and not computed on yet
  int qi_f = 0, gi_f = 0;                        // buffers of the next fetch
  int fq_a = 0, fq_b = 0, va_a = ROWS, va_b = ROWS;  // first query position and row count of those tiles (a: the older)
  int at = 0;                                    // the next entry
  auto issue = [&](u32x2 entry) {   // fetches the next tile, entry `at` of the list
    const uint32_t y = (uint32_t)__builtin_amdgcn_readfirstlane((int)entry.y);
    const int fq = __builtin_amdgcn_readfirstlane((int)entry.x), va = (int)(y & 127u);
    if (n_ahead == 0) { fq_a = fq; va_a = va; } else { fq_b = fq; va_b = va; }
    fetch(qi_f, gi_f, fq, va, (int)(y >> 7));
    qi_f = (qi_f + 1) & 3;
    gi_f = gi_f == 2 ? 0 : gi_f + 1;
    ++n_ahead;
    ++at;
  };
  issue(list[0]);
  if (at < entries) issue(list[1]);
  // The resident operand has arrived before the loop begins (and with it the first two tiles, requested behind it): the
  // compiler counts only the loads it knows, and a wait of its own for it inside the loop would also wait for every tile under way.
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
  if (chunk_base == 0) bwd_place_rows<D>(frag);
  bool prev = false;        // the tile before the current one exists: its dK part is still due
  int qi = 0, gi = 0, par = 0;   // Q buffer, dO buffer and parity of the current tile
  f32x16 dp_prev[NH];       // dS wavefront: dP - delta of the previous tile
#pragma unroll
  for (int h = 0; h < NH; ++h)
#pragma unroll
    for (int i = 0; i < 16; ++i) dp_prev[h][i] = 0.f;
  while (n_ahead > 0 || prev) {
    const bool had = n_ahead > 0;
    const int first_q_pos = fq_a, valid = va_a;   // of the current tile (if any)
    const u32x2 entry = list[min(at, kBwdListCap - 1)];   // (arrives while the barrier is waited for)
    // This wavefront's part of the current tile has landed; the loads of the tile after it (a wavefront's loads
    // return in order) may still be under way.
    if (n_ahead >= 2) {
      if (wave == 0) __builtin_amdgcn_s_waitcnt(0x0F76);   // vmcnt(6)
      else __builtin_amdgcn_s_waitcnt(0x0F74);             // vmcnt(4)
    } else {
      __builtin_amdgcn_s_waitcnt(0x0F70);                  // vmcnt(0)
    }
    __syncthreads();   // ... every wavefront's; what the iteration before read and wrote is settled
    const int q_now = qi, q_before = (qi + 3) & 3;
    if (had) {
      fq_a = fq_b;
      va_a = va_b;
      --n_ahead;
      if (at < entries) issue(entry);   // two tiles ahead: the buffers it fills were last read an iteration ago
    }
    if (active) {
      // Operand reads are issued by hand (BwdOperandOffsets): PF reads of a pair of chains under way ahead of
      // their products, the transposing reads of a key group before the vector ALU work that precedes their
      // products.  The counts in the waits name only reads that every path issues.
      constexpr int PF = 4, NC = NH * T::KSTEPS, TR = 2 * T::DT;
      const uint32_t half_base = lds_base + (uint32_t)(first_row * T::RB);
      const uint32_t v_at = row_addr + (uint32_t)(gi * 512 + first_row * 4 + 16 * g32);   // the rows' values
      short8v rb[PF];
      short4v tb[2][TR];
      if constexpr (ROLE == 0) {
        if (had) {   // ---- P wavefront, current tile
          const uint32_t q_t = half_base + (uint32_t)(q_now * TILE_BYTES), g_t = half_base + (uint32_t)((4 + gi) * TILE_BYTES);
          // rows first_vis .. left - 1 of the tile, counted from the lane's first, see its key
          const int lane_row = first_row + 4 * g32, left = valid - lane_row, first_vis = p.causal ? key_pos - shift - first_q_pos - lane_row : -64;
          // S = Q K^T, the steps of the halves in turn (read i: half i % NH, step i / NH)
          auto chain_read = [&](auto i_) {
            constexpr int i = decltype(i_)::value;
            rb[i % PF] = lds_read_b128<(i % NH) * 32 * T::RB>(off.rows[i / NH] + q_t);
          };
          static_for<0, PF>(chain_read);
          f32x16 sv[NH];
#pragma unroll
          for (int i = 0; i < 16; ++i) { sv[0][i] = 0.f; sv[NH - 1][i] = 0.f; }
          static_for<0, NC>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            constexpr int ahead = (NC - 1 - i) < (PF - 1) ? (NC - 1 - i) : (PF - 1);
            lds_wait1<ahead>(rb[i % PF]);
            sv[i % NH] = E::mfma(rb[i % PF], frag[i / NH], sv[i % NH]);
            if constexpr (i + PF < NC) chain_read(std::integral_constant<int, i + PF>{});
          });
          short8v lv[4];   // log-sum-exp of a half's rows
          auto read_lse = [&](auto h_) {
            static_for<0, 4>([&](auto a_) { lv[decltype(a_)::value] = lds_read_b128<128 * decltype(h_)::value + 32 * decltype(a_)::value>(v_at); });
          };
          read_lse(std::integral_constant<int, 0>{});
          bwd_issue_transposed<D, 0>(off, g_t, tb[0]);
          // edge: some row of the tile does not see some key of the wavefront (the causal diagonal, a slot with
          // fewer than 32 keys, a tile with fewer than 64 rows); elsewhere the per-element comparison and select
          // are left out.
          const bool edge = valid < ROWS || (p.causal && wave_key_max - shift - first_q_pos > 0);
          auto half = [&](auto h_) {
            constexpr int h = decltype(h_)::value;
            constexpr bool NEXT = h + 1 < NH;
            asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(lv[0]), "+v"(lv[1]), "+v"(lv[2]), "+v"(lv[3]) : "n"(TR));
            float ep[16];
            auto form_p = [&](auto edge_) {
#pragma unroll
              for (int a = 0; a < 4; ++a) {
                const f32x4 l4 = __builtin_bit_cast(f32x4, lv[a]);
#pragma unroll
                for (int bq = 0; bq < 4; ++bq) {
                  float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[h][4 * a + bq], p.c, -l4[bq]));
                  if constexpr (decltype(edge_)::value) pv = (32 * h + 8 * a + bq >= first_vis && 32 * h + 8 * a + bq < left) ? pv : 0.f;   // rows past the block's end repeat its last row
                  ep[4 * a + bq] = pv;
                }
              }
            };
            if (edge) form_p(std::true_type{});
            else form_p(std::false_type{});
            bwd_issue_transposed<D, 2 * h + 1>(off, g_t, tb[1]);
            short8v plo, phi;
            bwd_pack<E>(ep, plo, phi);
            *(short8v *)(p_mine + par * P_BYTES + h * 2048) = plo;
            *(short8v *)(p_mine + par * P_BYTES + h * 2048 + 1024) = phi;
            if constexpr (NEXT) read_lse(std::integral_constant<int, h + 1>{});
            bwd_wait_transposed<D, TR + (NEXT ? 4 : 0)>(tb[0]);
            bwd_transposed_products<D, E>(tb[0], plo, acc);
            if constexpr (NEXT) bwd_issue_transposed<D, 2>(off, g_t, tb[0]);
            bwd_wait_transposed<D, (NEXT ? 4 + TR : 0)>(tb[1]);
            bwd_transposed_products<D, E>(tb[1], phi, acc);
          };
          static_for<0, NH>(half);
        }
      } else {
        const uint32_t q_t = half_base + (uint32_t)(q_before * TILE_BYTES), g_t = half_base + (uint32_t)((4 + gi) * TILE_BYTES);
        auto chain_read = [&](auto i_) {   // dP = dO V^T of both halves of the current tile, as above
          constexpr int i = decltype(i_)::value;
          rb[i % PF] = lds_read_b128<(i % NH) * 32 * T::RB>(off.rows[i / NH] + g_t);
        };
        if (prev) {   // ---- dS wavefront, the tile before: dS = P * (dP - delta), dK^T += Q^T dS
          const uint32_t p_at = p_lds + (uint32_t)((par ^ 1) * P_BYTES);
          short8v pw[2];   // P of a half
          auto read_p = [&](auto h_) {
            pw[0] = lds_read_b128<2048 * decltype(h_)::value>(p_at);
            pw[1] = lds_read_b128<2048 * decltype(h_)::value + 1024>(p_at);
          };
          read_p(std::integral_constant<int, 0>{});
          bwd_issue_transposed<D, 0>(off, q_t, tb[0]);
          auto half = [&](auto h_) {
            constexpr int h = decltype(h_)::value;
            constexpr bool NEXT = h + 1 < NH;
            asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(pw[0]), "+v"(pw[1]) : "n"(TR));
            bwd_issue_transposed<D, 2 * h + 1>(off, q_t, tb[1]);
            float ed[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const uint32_t w = __builtin_bit_cast(u32x4, pw[i >> 3])[(i & 7) >> 1];
              ed[i] = ((i & 1) ? E::hi(w) : E::lo(w)) * dp_prev[h][i];
            }
            short8v dlo, dhi;
            bwd_pack<E>(ed, dlo, dhi);
            if constexpr (NEXT) read_p(std::integral_constant<int, h + 1>{});
            bwd_wait_transposed<D, TR + (NEXT ? 2 : 0)>(tb[0]);
            bwd_transposed_products<D, E>(tb[0], dlo, acc);
            if constexpr (NEXT) bwd_issue_transposed<D, 2>(off, q_t, tb[0]);
            bwd_wait_transposed<D, (NEXT ? 2 + TR : 0)>(tb[1]);
            bwd_transposed_products<D, E>(tb[1], dhi, acc);
          };
          static_for<0, NH>(half);
        }
        if (had) {   // ---- dS wavefront, current tile: dP - delta = dO V^T - delta, kept for the next iteration
          short8v dl[NH][4];
          static_for<0, 4 * NH>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            dl[i / 4][i % 4] = lds_read_b128<256 + 128 * (i / 4) + 32 * (i % 4)>(v_at);
          });
          static_for<0, PF>(chain_read);
#pragma unroll
          for (int h = 0; h < NH; ++h) {
            asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(dl[h][0]), "+v"(dl[h][1]), "+v"(dl[h][2]), "+v"(dl[h][3]) : "n"(PF));
#pragma unroll
            for (int i = 0; i < 16; ++i) dp_prev[h][i] = __builtin_bit_cast(f32x4, dl[h][i >> 2])[i & 3];
          }
          static_for<0, NC>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            constexpr int ahead = (NC - 1 - i) < (PF - 1) ? (NC - 1 - i) : (PF - 1);
            lds_wait1<ahead>(rb[i % PF]);
            dp_prev[i % NH] = E::mfma(rb[i % PF], frag[i / NH], dp_prev[i % NH]);
            if constexpr (i + PF < NC) chain_read(std::integral_constant<int, i + PF>{});
          });
        }
      }
    }
    prev = had;
    qi = (qi + 1) & 3;
    gi = gi == 2 ? 0 : gi + 1;
    par ^= 1;
  }
  chunk_base += kBwdListCap;
  if (chunk_base < total) {
    __syncthreads();
    if (wave == 0) {
      int l = threadIdx.x;
      asm volatile("" : "+v"(l));   // (nothing of this is to be prepared ahead of the tile loop)
      const BwdListRecord rec = *list_s;
      (void)bwd_key_tiles<ROWS>(p, rec.range, rec.column, rec.bit, nullptr, chunk_base, list, l);
    }
    __syncthreads();
  }
  }
  if constexpr (FORM == kBwdShared) {   // the lower rows' sums go to the pair with the upper rows: [pair % 2][role][register][lane] floats
    // (the record of the part lies behind what this overwrites)
    __syncthreads();
    float *xch = (float *)lds + (size_t)(key_slot * 2 + ROLE) * (T::DT * 16) * 64 + lane;
    if (slot >= 2) {
#pragma unroll
      for (int dt = 0; dt < T::DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) xch[(dt * 16 + i) * 64] = acc[dt][i];
    }
    __syncthreads();
    if (slot < 2) {
#pragma unroll
      for (int dt = 0; dt < T::DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[dt][i] += xch[(dt * 16 + i) * 64];
    }
  }
  const bool owner = active && slot < KEY_SLOTS;   // of the sums of 32 keys
  if constexpr (PARTS) {
    const BwdPartRecord rec = *part_s;
    const int count = __builtin_amdgcn_readfirstlane(rec.count);
    if (count > 1) {
      constexpr size_t kWaveFloats = (size_t)T::DT * 1024;   // of one wavefront's accumulators
      float *at = rec.first + (size_t)wave * kWaveFloats + lane * 4;
      if (owner) bwd_leave_part<T::DT>(acc, at + (size_t)rec.part * WAVES * kWaveFloats);
      if (!bwd_last_part(rec.counter, count, (int *)lds)) return;
      if (owner) bwd_sum_parts<T::DT>(acc, at, WAVES * kWaveFloats, count);
    }
  }
  if (owner) {
    const int64_t row = k0 + kbl * p.kbs + row0;
    if constexpr (ROLE == 0) bwd_store_rows<D, E>(p.dv + row * p.dv_s + (int64_t)hk * p.dv_h, p.dv_s, nrows, acc, 1.f, lane);
    else bwd_store_rows<D, E>(p.dk + row * p.dk_s + (int64_t)hk * p.dk_h, p.dk_s, nrows, acc, p.scale, lane);
  }
  };
  if (role == 0) run(std::integral_constant<int, 0>{});
  else run(std::integral_constant<int, 1>{});
}

// FORM: of the dK/dV kernel (kBwdShared is SPLIT at head dims up to 64)
template <int D, typename E, bool PARTS_Q, bool PARTS_K, int FORM>
int launch_bwd_kernels(const BwdParams &bp, int nhead_k, int num_k_block, hipStream_t stream) {
  using T = BwdTile<D>;
  // LDS: the dQ kernel's three K and two V tiles; the dK/dV kernels' tile buffers, P records and row values
  constexpr int lds_dq = 5 * T::TILE_BYTES, lds_dkv = D == 128 ? bwd_dkv8_lds(FORM) : (FORM == kBwdShared ? 4 : 3) * (2 * T::TILE_BYTES + 512) + kBwdListCap * 8 + 16;
  if constexpr (lds_dkv > 48 * 1024) {
    static thread_local bool raised[kMaxDevices] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
      return fail(HBSA_ERR_UNSUPPORTED, "no current device, or device index above %d", kMaxDevices - 1);
    if (!raised[dev]) {
      const void *dkv = nullptr;
      if constexpr (D == 128) dkv = reinterpret_cast<const void *>(&hbsa_bwd_dkv8_kernel<E, PARTS_K, FORM>);
      else dkv = reinterpret_cast<const void *>(&hbsa_bwd_dkv_kernel<D, E, PARTS_K, FORM == kBwdShared>);
      hipError_t e = hipFuncSetAttribute(dkv, hipFuncAttributeMaxDynamicSharedMemorySize, lds_dkv);
      if (e == hipSuccess)
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(&hbsa_bwd_dq_kernel<D, E, PARTS_Q>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds_dq);
      if (e != hipSuccess) return (int)e;
      raised[dev] = true;
    }
  }
  const unsigned q_wgs = (unsigned)(bp.nqb * bp.nsub * (PARTS_Q ? bp.parts_q : 1));
  const unsigned k_wgs = (unsigned)(num_k_block * bp.nsub_k * (PARTS_K ? bp.parts_k : 1));
  const dim3 q_grid = bp.flat_grid ? dim3(q_wgs * (unsigned)nhead_k) : dim3(q_wgs, (unsigned)nhead_k);
  const dim3 kv_grid = bp.flat_grid ? dim3(k_wgs * (unsigned)nhead_k) : dim3(k_wgs, (unsigned)nhead_k);
  hipLaunchKernelGGL((hbsa_bwd_dq_kernel<D, E, PARTS_Q>), q_grid, dim3(kThreads), lds_dq, stream, bp);
  if constexpr (D == 128) hipLaunchKernelGGL((hbsa_bwd_dkv8_kernel<E, PARTS_K, FORM>), kv_grid, dim3(bwd_dkv8_threads(FORM)), lds_dkv, stream, bp);
  else hipLaunchKernelGGL((hbsa_bwd_dkv_kernel<D, E, PARTS_K, FORM == kBwdShared>), kv_grid, dim3(kThreads), lds_dkv, stream, bp);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

template <int D, typename E, int FORM>
int launch_bwd_parts(const BwdParams &bp, int nhead_k, int num_k_block, hipStream_t stream) {
  const bool pq = bp.parts_q > 1, pk = bp.parts_k > 1;
  if (pq && pk) return launch_bwd_kernels<D, E, true, true, FORM>(bp, nhead_k, num_k_block, stream);
  if (pk) return launch_bwd_kernels<D, E, false, true, FORM>(bp, nhead_k, num_k_block, stream);
  if (pq) return launch_bwd_kernels<D, E, true, false, FORM>(bp, nhead_k, num_k_block, stream);
  return launch_bwd_kernels<D, E, false, false, FORM>(bp, nhead_k, num_k_block, stream);
}
template <int D, typename E>
int launch_bwd(const BwdParams &bp, int nhead_k, int num_k_block, hipStream_t stream) {
  if constexpr (D == 128)
    if (bp.form_k == kBwdNarrow) return launch_bwd_parts<D, E, kBwdNarrow>(bp, nhead_k, num_k_block, stream);
  if (bp.form_k == kBwdShared) return launch_bwd_parts<D, E, kBwdShared>(bp, nhead_k, num_k_block, stream);
  return launch_bwd_parts<D, E, kBwdWide>(bp, nhead_k, num_k_block, stream);
}

}  // namespace hbsa
