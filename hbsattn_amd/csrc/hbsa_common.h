// Types, element policies and device helpers shared by the kernels of the library, the kernel parameter blocks,
// and the declarations of the launch functions.  The attention kernels are templates over head dim and element type;
// each (head dim, element type) is a translation unit of its own (hbsa_inst.hip), so that they compile side by side.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "hbsattn_amd.h"

namespace hbsa {

typedef short short4v __attribute__((ext_vector_type(4)));
typedef short short8v __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

#define HBSA_AS1(p) ((const __attribute__((address_space(1))) void *)(p))
#define HBSA_AS3(p) ((__attribute__((address_space(3))) void *)(p))

constexpr int kThreads = 256;   // 4 wavefronts
constexpr int kWaveRows = 32;   // query rows per wavefront (the MFMA N dimension)
constexpr int kTileKeys = 64;   // keys per main-loop step
constexpr int kWalkReportTiles = 8;   // an item adds its progress to its walk clock every so many tiles (a power of two)
constexpr float kLog2e = 1.4426950408889634f;
// One-launch form: sequences whose boundaries the scheduler keeps in LDS (batch + 1 entries of four arrays)
constexpr int kSeqCap = 128;
constexpr int kDecodeMaxParts = 32;    // parts of an item of the decode kernel
constexpr int kDecodeEntries = 64;     // (q head, row) entries of an item of the decode kernel, as the host bounds them
constexpr int kMaxPartItems = 4096;   // items of a launch that may be cut into parts (its arrival counters)
// Up to this many items per resident workgroup are handed out without the per-XCD work queues, in a fixed order
// (see claim() in hbsa_fwd_kernel).  Measured against the queues: 8 x 512 tokens 71 -> 45 us, 8 x 1024 113 -> 99,
// 8 x 2048 causal 200 -> 189, C5 0.33 -> 0.245 ms; at sixteen per workgroup 8 x 4096 tokens lose 5 % and at 64
// C2 and C3 lose 5-8 % (the queues keep one head's K/V in one XCD's L2).
constexpr int kStaticShare = 8;
constexpr int kMaxDevices = 64;            // devices of one process the launch caches cover
constexpr float kLazyRescaleLog2 = 8.0f;  // the reference of a row's exponentials may lag the true maximum by 2^8

// Geometry of one q block, written by the pre-pass (48 bytes).
struct QBlockInfo {
  int32_t row_begin;   // token row of the block's first query
  int32_t rows;        // queries in the block (ragged last block of a sequence)
  int32_t key_begin;   // token row of the sequence's first key
  int32_t klen;        // keys in the sequence
  int32_t q_pos;       // in-sequence position of the block's first query
  int32_t shift;       // k_len - q_len: bottom-right causal alignment
  int32_t nkblk;       // k blocks in the sequence
  int32_t kmax;        // exclusive in-sequence bound of keys any row of the block may see
  int32_t seq;         // first q block of the block's sequence: identifies the sequence by a number below num_q_block
                       // (the batch index can exceed it when the batch holds sequences without queries)
  int32_t flags;       // 1: the block's sequence did not fit the tensors; it has no keys (and perhaps no rows)
  int32_t pad[2];
};
static_assert(sizeof(QBlockInfo) == 48, "QBlockInfo is read as twelve 32-bit words");

struct Sched;

struct PrepParams {
  const int32_t *cu_q, *cu_k, *q_block_to_batch, *cu_num_q_block, *cu_num_k_block;
  const uint8_t *mask;
  int64_t ms_h, ms_q, ms_k;
  QBlockInfo *info;
  uint32_t *bits;
  struct Sched *sched;
  unsigned long long *clock;
  int32_t nqb, qbs, kbs, wpr, causal;
  int32_t batch, nkb, total_q, total_k;   // bounds the sequences' boundaries are checked against
  uint32_t *order;         // order of the items (see OrderRoom), nullptr: not wanted
  struct OrderRoom *room;  // the stream's room for making it, nullptr: the order without weights is written
  int32_t nhead_k, weight_shift;
  int32_t *order_k;        // [nkb]: the k blocks by falling number of query rows that can see them
  int32_t weigh_k;         // 0: in their own order
  int32_t shared_tiles;    // for the launch record
};

// Division by a launch constant d, exact for 0 <= n < 2^31: n / d == (n * m) >> s with
// s = 31 + ceil(log2 d), m = ceil(2^s / d) (which fits 32 bits).  Three scalar instructions where
// a hardware-less integer division takes about forty.
struct FastDiv {
  uint32_t m, s;
};
__host__ __device__ inline uint32_t fast_div(uint32_t n, FastDiv f) { return (uint32_t)(((uint64_t)n * f.m) >> f.s); }
inline FastDiv make_fast_div(uint32_t d) {
  uint32_t l = 0;
  while (((uint64_t)1 << l) < d) ++l;
  FastDiv f;
  f.s = 31 + l;
  f.m = (uint32_t)((((uint64_t)1 << f.s) + d - 1) / d);
  return f;
}

// (Fields are appended at the end, never inserted: the compiler fetches the kernel arguments in aligned groups,
// and a layout that splits the fields the tile loop uses makes it fetch some of them again inside that loop,
// where a scalar load's wait also waits for every hand-issued LDS read; measured, 0.8 % of T for one such shift.)
struct FwdParams {
  const char *q, *k, *v;
  char *out;
  const QBlockInfo *info;
  const uint32_t *bits;
  int64_t q_s, q_h, k_s, k_h, v_s, v_h, o_s, o_h;  // bytes
  int32_t nqb, ratio, kbs, wpr, causal;
  int32_t wps;    // wave slots per q head = ceil(q_block_size / 32)
  int32_t nw;     // wavefronts per workgroup (4 or 8)
  int32_t nsub;   // workgroups per (kv head, q block) = ceil(ratio * wps / nw)
  uint32_t q_sign;  // 0x80008000 when softmax_scale < 0 (Q is negated, |scale| used)
  float c;        // |softmax_scale| * log2(e)
  float lag;      // kLazyRescaleLog2 / c: how far the decode kernel's running max may lag, in raw score units
  FastDiv div_nsub, div_nqb, div_kbs;   // divisions on the scheduler's path
  int32_t f32;    // fp32 inputs staged as fp16: the softmax constants come from the launch record, where
                  // the setup kernel derived them from the tensors' maxima
  int32_t nhead_k;
  int32_t one_each;   // > 0: the number of work items, handed out without queues: workgroup i of G takes items i, 2G - 1 - i, 2G + i, ...
  struct Sched *sched;
  // Walk order of the kept k blocks (see the kernel's comment).  walk != 0: the workgroups that work on
  // one (kv head, sequence) keep near each other in key space through a shared clock, so that they find
  // each other's K/V blocks in the L2; the summation order, and with it the last bits of the result,
  // then depend on timing.  walk == 0: every item walks its blocks in ascending order (deterministic).
  unsigned long long *clock;   // [nhead_k, num_q_block]: clock of (kv head, first q block of the sequence)
  int32_t walk;
  float *lse;             // optional [total_q, nhead_q] log-sum-exp output (nullptr: none)
  int64_t lse_s, lse_h;   // its strides in elements
  // Split over key blocks (few, long work items): every (kv head, q block, slot group) becomes
  // nparts items.  Part i sees its share of the kept k blocks and stores a normalised fp32 partial result and its log-sum-exp;
  // hbsa_merge_kernel combines them.  An item of few keys has fewer parts (the others find nothing to do), or one, which
  // writes the output itself.
  int32_t nparts;         // 1: no split
  FastDiv div_nparts;
  // One-launch form whose caller has not counted the blocks (the COUNTED kernels, in the place of what a split needs: 16 bytes more of
  // arguments cost every short call 0.2 us): the sides of count_info[1] (1: queries, 2: keys; cu_nqb, cu_nkb then point to something that
  // can be read) are counted by every workgroup for itself, and the first writes counts[2] = whether the totals are nqb and
  // nkb_total, counts[3] = count_info[0], the caller's ticket, in one 8-byte store.
  union {
    float *part_out;        // [nparts, total_q, nhead_q, D]
    int32_t *counts;
  };
  union {
    float *part_lse;        // [nparts, total_q, nhead_q], and behind them int32 [total_q, nhead_q], the rows' numbers of parts
    int32_t count_info[2];
  };
  int32_t total_q, nhead_q;
  // One-launch form (the kernel instantiated with FUSED): no pre-pass has run, `info` and `bits` are unused,
  // and the scheduler derives every item's geometry and bit row itself from the caller's arrays.
  const int32_t *cu_q, *cu_k, *cu_nqb, *cu_nkb;   // int32[batch + 1] each
  const uint8_t *mask;                            // block_mask bytes, innermost (k block) stride 1
  int64_t ms_h, ms_q;                             // its head and q block strides
  int32_t batch, nkb_total, total_k, qbs;
  int32_t pack;   // host side only: the launch uses the kernel whose wave slots are packed across the q heads of a GQA group
  FastDiv div_nhk;   // division by nhead_k (items handed out without queues)
  int32_t ncol;      // 16-byte chunks of a row (the COLS form of the kernel)
  // Kernels that cut an item's k blocks into parts, one workgroup each, and combine them themselves (see ItemParts)
  int64_t ms_k;          // stride of the mask's innermost dimension
  int32_t max_parts;     // parts of an item at most (1: items are whole)
  int32_t min_blocks;    // k blocks of a part at least
  float *parts;          // partial results
  FastDiv div_items;     // division by the number of items
  int32_t parts_last;    // workgroups are numbered by part first (else: the parts of an item are neighbours)
  uint32_t *arrivals;    // one counter per item, zero before and after every launch
  int32_t split;         // host side only: parts of the split over key blocks that pay (fwd_split)
  // host side only, 32 bits in all (the arguments grow by nothing): two teams for the tiles of every item (fwd_teams); what the two unions hold (put_parts,
  // put_counts); tiles of 16-key groups (the GROUPED form of the kernel)
  int8_t teams, unions;
  int16_t grouped;
  // Items handed out without queues in the order of their weights (see OrderRoom), nullptr: last q blocks first
  const uint32_t *order;         // [num_q_block * nhead_k]: q block << 16 | kv head, heaviest first
};

// The only writers of the unions of FwdParams; false where the other one has been there (once a split's pointers were written over, and its kernel
// stored its results at address zero and up).  Every launch asks unions_fit first.
enum : int8_t { kUnionsEmpty, kUnionsParts, kUnionsCounts };
inline bool put_parts(FwdParams &fp, float *out, float *lse) {
  if (fp.unions == kUnionsCounts) return false;
  fp.unions = kUnionsParts;
  fp.part_out = out;
  fp.part_lse = lse;
  return true;
}
inline bool put_counts(FwdParams &fp, int32_t *counts, int32_t ticket, int32_t sides) {
  if (fp.unions == kUnionsParts) return false;
  fp.unions = kUnionsCounts;
  fp.counts = counts;
  fp.count_info[0] = ticket;
  fp.count_info[1] = sides;
  return true;
}
// counted: the kernel counts blocks.  (nparts > 1: it writes partial results)
inline bool unions_fit(const FwdParams &fp, bool counted) {
  return counted ? fp.unions == kUnionsCounts && fp.nparts == 1 : fp.unions == (fp.nparts > 1 ? kUnionsParts : kUnionsEmpty);
}

// Boundaries of one sequence of the packed batch, as read from the caller's device arrays.
struct SeqBounds {
  int32_t q0, q1;     // cu_q_seqlens[b], [b + 1]
  int32_t k0, k1;     // cu_k_seqlens[b], [b + 1]
  int32_t kb0, kb1;   // cu_num_k_block[b], [b + 1]
  int32_t qb0;        // cu_num_q_block[b]
};

// Geometry record of q block g.  The sequence boundaries are device data the host cannot check, so they
// are checked here against the token counts of q and k/v and the block counts.  A sequence that does
// not fit (a wrong cu_seqlens, q/k/v shorter than it says, inconsistent block metadata) gets no keys:
// nothing of k, v or the mask is read for it, and those of its query rows that lie inside q and out are
// written as zeros, like any row that sees no key (flags = 1 marks such a block).  When not even the
// query side makes sense (have == false: the block's sequence index is outside the batch) the block
// has no rows and nothing is written for it.  kb0: first global k block of the sequence.
__host__ __device__ inline QBlockInfo q_block_geometry(int g, bool have, SeqBounds s, int qbs, int kbs, int causal,
                                                      int nkb_total, int total_q, int total_k, int &kb0) {
  const int qlen = s.q1 - s.q0, klen_in = s.k1 - s.k0, nkb_in = s.kb1 - s.kb0;
  const int q_pos = (g - s.qb0) * qbs;
  const bool q_ok = have && s.q0 >= 0 && qlen > 0 && s.qb0 >= 0 && g >= s.qb0 && q_pos >= 0 && q_pos < qlen &&
                    (int64_t)s.q0 + q_pos < total_q;
  const bool ok = q_ok && (int64_t)s.q0 + qlen <= total_q && s.k0 >= 0 && klen_in >= 0 && (int64_t)s.k0 + klen_in <= total_k &&
                  s.kb0 >= 0 && nkb_in >= 0 && (int64_t)s.kb0 + nkb_in <= nkb_total && (int64_t)nkb_in * kbs >= klen_in;
  QBlockInfo r;
  r.row_begin = q_ok ? s.q0 + q_pos : 0;
  int rows = 0;
  if (q_ok) {
    rows = qlen - q_pos < qbs ? qlen - q_pos : qbs;
    if (rows > total_q - r.row_begin) rows = total_q - r.row_begin;
  }
  r.rows = rows;
  r.key_begin = ok ? s.k0 : 0;
  r.klen = ok ? klen_in : 0;
  r.q_pos = q_ok ? q_pos : 0;
  r.shift = ok ? klen_in - qlen : 0;
  r.nkblk = ok ? nkb_in : 0;
  int kmax = 0;
  if (ok) {
    kmax = klen_in;
    if (causal && q_pos + rows + r.shift < kmax) kmax = q_pos + rows + r.shift;
    if (kmax < 0) kmax = 0;
  }
  r.kmax = kmax;
  r.seq = q_ok ? s.qb0 : 0;
  r.flags = ok ? 0 : 1;
  r.pad[0] = r.pad[1] = 0;
  kb0 = ok ? s.kb0 : 0;
  return r;
}

// --------------------------------------------------------------------------------------
// Element-type policies.
// --------------------------------------------------------------------------------------
struct ElemBF16 {
  static __device__ __forceinline__ f32x16 mfma(short8v a, short8v b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    bf16x2 v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
  }
  static __device__ __forceinline__ float lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
  static __device__ __forceinline__ float hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }
};
struct ElemF16 {
  static __device__ __forceinline__ f32x16 mfma(short8v a, short8v b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    f16x2 v = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, v);
  }
  static __device__ __forceinline__ float lo(uint32_t w) { return (float)__builtin_bit_cast(f16x2, w).x; }
  static __device__ __forceinline__ float hi(uint32_t w) { return (float)__builtin_bit_cast(f16x2, w).y; }
};

// exchange-and-combine between lane i and lane i^32
__device__ __forceinline__ float half_max(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}
__device__ __forceinline__ float half_sum(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}

struct Sched {
  uint32_t qnext[8];   // next unclaimed entry of each queue
  uint32_t done;       // workgroups of the running attention launch that have made their last claim
  // fp32 inputs staged as fp16 only (written by hbsa_setup_kernel, read by the attention kernel at its start):
  float c;             // |softmax_scale| * log2(e), divided by the q and k staging multipliers
  float out_mul;       // 1 / (v staging multiplier)
  // bit patterns of max|x| over q, k, v and the power-of-two staging multipliers
  uint32_t amax[3];
  float in_mul[3];
  uint32_t shared_tiles;   // prepared masks: teams may share an item's tiles (team_sequences)
  uint32_t pad[46];
};
static_assert(sizeof(Sched) == 256, "Sched is one 256-byte slot of the workspace");

// ---- LDS reads issued by hand.  The compiler neither waits for these nor knows they touch LDS,
// so each result must pass through lds_wait<N>() before it is used: LDS operations of a
// wavefront complete in order, and lds_wait<N> returns once at most N of them are outstanding.
// (The transposing read is issued this way because the compiler otherwise waits for every
// outstanding global->LDS load before it; the K reads so that their issue distance is fixed.)
// HAND = false gives the same reads as ordinary loads the compiler schedules and waits for itself (the
// lds_wait calls then do nothing): the form for instantiations that move registers to the accumulation half, where a
// register with a hand-issued read in flight could be moved before its data arrives.
template <int OFF, bool HAND = true>
__device__ __forceinline__ short8v lds_read_b128(uint32_t addr) {
  if constexpr (HAND) {
    short8v r;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(r) : "v"(addr), "n"(OFF));
    return r;
  } else {
    return *(const __attribute__((address_space(3))) short8v *)(uintptr_t)(addr + (uint32_t)OFF);
  }
}
template <int OFF, bool HAND = true>
__device__ __forceinline__ short4v lds_read_tr16_b64(uint32_t addr) {
  if constexpr (HAND) {
    short4v r;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=&v"(r) : "v"(addr), "n"(OFF));
    return r;
  } else {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(uintptr_t)(addr + (uint32_t)OFF));
  }
}
template <int N>
__device__ __forceinline__ void lds_wait1(short8v &a) {
  asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(a) : "n"(N));
}
template <int N>
__device__ __forceinline__ void lds_wait(short4v &a, short4v &b, short4v &c, short4v &d, short4v &e, short4v &f, short4v &g,
                                         short4v &h) {
  asm volatile("s_waitcnt lgkmcnt(%8)" : "+v"(a), "+v"(b), "+v"(c), "+v"(d), "+v"(e), "+v"(f), "+v"(g), "+v"(h) : "n"(N));
}

// Placement of a K / V tile's rows in LDS: 16-byte chunk c of row r sits at chunk position c ^ k(r) (K), c ^ v(r) (V).
// Rows by 16 consecutive ones (K, one chunk column at a time) then start at 16 different 16-byte slots of the 256-byte
// bank sweep, and the 4 rows x 64 bytes of a transposing V read cover it once.  With a row of 4, 8, 16 or 32 chunks
// that takes an exclusive or over all chunk bits; rows of 12, 20 and 24 chunks already step by 12, 4 and 8 slots, so
// that the low two or three bits are enough (and the exchange stays inside the row).
template <int D>
struct FwdSwizzle {
  static constexpr int CPR = D / 8;
  static constexpr int RPG = 16 / CPR > 0 ? 16 / CPR : 1;   // rows per 256-byte bank sweep
  static constexpr bool POW2 = (CPR & (CPR - 1)) == 0;
  static constexpr int PERIOD = RPG * CPR;   // rows after which the placement repeats (POW2)
  static __device__ __forceinline__ int k(int r) { return POW2 ? (r / RPG) % CPR : CPR % 8 == 0 ? (r >> 1) & 7 : (r >> 2) & 3; }
  static __device__ __forceinline__ int v(int r) {
    return POW2 ? (CPR >= 8 ? ((r / RPG) % (CPR / 4)) << 2 : 0) : CPR % 8 == 0 ? ((r >> 1) & 1) << 2 : 0;
  }
};

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// Arguments of the backward kernels (hbsa_bwd.h).
struct BwdParams {
  const char *q, *k, *v, *out, *dout;
  char *dq, *dk, *dv;
  const float *lse;           // [total_q, nhead_q], contiguous
  // [nhead_q, total_q]: what the dQ kernel leaves for the dK/dV kernels, whose tiles are consecutive rows of one q head
  float *delta;               // -rowsum(dO * O)
  float *lse2;                // lse * log2(e), +inf where lse is -inf
  const QBlockInfo *info;
  const uint32_t *bits;
  const int32_t *cu_k, *cu_num_q_block, *cu_num_k_block;
  int64_t q_s, q_h, k_s, k_h, v_s, v_h, o_s, o_h, do_s, do_h, dq_s, dq_h, dk_s, dk_h, dv_s, dv_h;   // bytes
  int32_t nqb, nkb, xcd_heads, batch, ratio, nhead_q, qbs, kbs, wpr, causal;   // xcd_heads: see the dK/dV kernels
  int32_t total_k;
  int32_t wps, nsub;     // q side: wave slots per q head and workgroups per (kv head, q block), as in the forward
  int32_t nsub_k;        // k side: workgroups per (kv head, k block), of 128 keys or (form_k == kBwdNarrow) 64
  float c;               // softmax_scale * log2(e), signed
  float scale;
  // Items cut into parts (see BwdCut): at most parts_q k block ranges a dQ item, of min_blocks_q k blocks at least, and parts_k
  // ranges of (q block, q head) pairs a dK/dV item, of min_units_k pairs at least; 1: whole
  int32_t parts_q, min_blocks_q, parts_k, min_units_k;
  int32_t total_q;
  int32_t flat_grid;     // one-dimensional grids (bwd_decode_grid)
  float *parts;          // partial accumulators, shared by the two launches
  uint32_t *arrivals;    // one counter per item, zero before and after every launch
  const int32_t *order_k;   // k blocks by falling number of query rows that can see them, nullptr: in their own order
  int32_t form_k;         // of the dK/dV kernel (bwd_form, bwd_pairs)
};
constexpr int kBwdWide = 0, kBwdShared = 1, kBwdNarrow = 2, kBwdHalves = 3;

// ---- Items of the kernels without a scheduler: geometry and kept blocks straight from the caller's arrays (bits == nullptr)
// or from a prepared workspace.  Everything here is uniform over the calling wavefront.
__device__ __forceinline__ QBlockInfo item_geometry(const FwdParams &p, int qb, int lane, int &kb0) {
  if (p.bits != nullptr) {
    const uint32_t w = lane < 12 ? ((const uint32_t *)(p.info + qb))[lane] : 0u;
    QBlockInfo r;
    int32_t *f = (int32_t *)&r;
#pragma unroll
    for (int i = 0; i < 12; ++i) f[i] = __builtin_amdgcn_readlane((int)w, i);
    kb0 = 0;
    return r;
  }
  int b = 0;   // sequences that start at or before qb, minus one
  for (int base = 0; base < p.batch; base += 64) {
    const int i = base + lane + 1;
    const int first_qb = i <= p.batch ? p.cu_nqb[i] : 0x7fffffff;
    b += __builtin_popcountll(__builtin_amdgcn_ballot_w64(first_qb <= qb));
  }
  const bool have = b < p.batch;
  SeqBounds s = {0, 0, 0, 0, 0, 0, 0};
  if (have) {   // seven numbers, one load
    const int32_t *at = lane < 2 ? p.cu_q + b + lane : lane < 4 ? p.cu_k + b + lane - 2 : lane < 6 ? p.cu_nkb + b + lane - 4 : p.cu_nqb + b;
    const int v = lane < 7 ? *at : 0;
    s.q0 = __builtin_amdgcn_readlane(v, 0); s.q1 = __builtin_amdgcn_readlane(v, 1);
    s.k0 = __builtin_amdgcn_readlane(v, 2); s.k1 = __builtin_amdgcn_readlane(v, 3);
    s.kb0 = __builtin_amdgcn_readlane(v, 4); s.kb1 = __builtin_amdgcn_readlane(v, 5);
    s.qb0 = __builtin_amdgcn_readlane(v, 6);
  }
  return q_block_geometry(qb, have, s, p.qbs, p.kbs, p.causal, p.nkb_total, p.total_q, p.total_k, kb0);
}

// Kept k blocks among blocks first .. first + 63 of the q block's own sequence, those below `end` only.  The load and the
// vote are apart, so that the load can be on its way while something else is done.
struct KeptWindow {
  const FwdParams &p;
  const uint32_t *row;     // prepared bit row, or
  const uint8_t *mrow;     // mask byte of the sequence's first k block
  int lane;
  __device__ __forceinline__ KeptWindow(const FwdParams &p_, int hk, int qb, int kb0, int lane_) : p(p_), lane(lane_) {
    row = p.bits != nullptr ? p.bits + ((size_t)hk * p.nqb + qb) * p.wpr : nullptr;
    mrow = p.mask + (int64_t)hk * p.ms_h + (int64_t)qb * p.ms_q + (int64_t)kb0 * p.ms_k;
  }
  __device__ __forceinline__ uint32_t load(int first, int end) const {
    const int j = first + lane;
    if (j >= end) return 0u;
    return row != nullptr ? (row[j >> 5] >> (j & 31)) & 1u : (uint32_t)mrow[(int64_t)j * p.ms_k];
  }
  static __device__ __forceinline__ uint64_t vote(uint32_t loaded) { return __builtin_amdgcn_ballot_w64(loaded != 0); }
};

// An item's visible k blocks [0, nvis) cut into parts of `per` blocks: as few as keep a part at min_blocks or more, at most
// max_parts.  Every part is one workgroup; the one that arrives last combines the others' partial results with its own, in
// the order of the parts, so the result does not depend on the order of arrival.
struct ItemParts {
  int per, count;
  __device__ __forceinline__ ItemParts(const FwdParams &p, int nvis) {
    const int even = (nvis + p.max_parts - 1) / p.max_parts;
    per = even > p.min_blocks ? even : p.min_blocks;
    count = (nvis + per - 1) / per;
    if (count < 1) count = 1;
  }
  __device__ __forceinline__ uint32_t word_mask(int part, int j0) const {   // of a part's blocks among j0 .. j0 + 31
    const int a = max(part * per - j0, 0), b = min((part + 1) * per - j0, 32);
    return a < b ? (~0u << a) & (~0u >> (32 - b)) : 0u;
  }
};

// Partial results travel between workgroups, and so between the chip's eight dies, whose L2 caches know nothing of each
// other.  They are stored through to the memory all dies share (agent scope, as an atomic store of that scope is done): such
// a store has arrived once its wavefront has waited for it.  The workgroup that combines them first drops what its own
// caches hold (an acquire of that scope) and may then load plainly, many at a time: with loads of agent scope, each waited
// for by itself, combining 32 parts took longer (50 us) than everything before it.
__device__ __forceinline__ void part_store(float *at, float v) {
  __hip_atomic_store((uint32_t *)at, __builtin_bit_cast(uint32_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// 16-byte aligned.  The two wait states belong to the store: it still reads its data registers when the next instruction is
// issued, and the compiler, which keeps vector instructions from writing them too early after its own wide stores, does not
// know this one (measured without them: the first registers of a part, lanes 12-15 of every 16, replaced by what came next).
__device__ __forceinline__ void part_store4(float *at, f32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(at), "v"(v) : "memory");
}
__device__ __forceinline__ void parts_arrived() { asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); }
__device__ __forceinline__ void parts_acquire() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent"); }

// ---- Items in the order of their weights.  A launch whose workgroups take two to eight items each in a fixed order ends when
// the unluckiest workgroup does: a Bernoulli mask, ragged sequences and a causal mask make items differ by factors.  So the
// (q block, kv head) pairs are counted (their kept keys) and sorted, heaviest first; the fixed order (forwards, then backwards
// through the list) then gives every workgroup about the same.  One wavefront counts each pair, the workgroup that arrives last
// sorts by counting; the order among equals is left to chance, and no result depends on it.
// Measured, forward kernels: 6 x 300 .. 4000 tokens, 16 / 4 heads of 64, 1.8 items a place, 67 -> 48 us, the pre-pass 4.7 -> 7.7.
// The one-launch form has no pre-pass, and a launch for the order alone took 8 to 11 us: of what it gives, 8 x 2050 tokens, 16 heads of
// 192, not causal, 221 -> 199, C5's shape 276 -> 262, 11 and 6 us would be left, and shorter calls lose.  That form takes no order.
constexpr int kMaxOrderItems = 4096;   // pairs (of 8192, 4 x 8192 tokens with 32 heads, no launch takes the order, and sorting them costs 10 us)
constexpr int kOrderBins = 2 * kThreads;   // weights told apart
constexpr int kOrderCopies = 4;            // counters of one weight, by lane: equal weights otherwise queue at one word of LDS
struct OrderRoom {   // a stream's
  uint32_t weight[kMaxOrderItems];
  uint32_t arrived, pad[63];   // zero before and after every launch
};
struct OrderLds {
  uint32_t count[kOrderCopies][kOrderBins];
  uint16_t bin[kMaxOrderItems];
  uint32_t sums[kThreads / 64], last;
};
__device__ __forceinline__ void order_note(OrderRoom *room, int pair, int keys, int shift) {
  __hip_atomic_store(&room->weight[pair], (uint32_t)min(kOrderBins - 1, (keys + (1 << shift) - 1) >> shift), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
// Behind the notes: every workgroup of kThreads threads arrives, the last of `workgroups` sorts.
__device__ __forceinline__ void order_arrive(OrderRoom *room, uint32_t *order, int pairs, int nhead_k, uint32_t workgroups, OrderLds &lds) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const bool last = __hip_atomic_fetch_add(&room->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == workgroups;
    if (last) __hip_atomic_store(&room->arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    lds.last = last;
  }
  for (int i = threadIdx.x; i < kOrderCopies * kOrderBins; i += kThreads) (&lds.count[0][0])[i] = 0;
  __syncthreads();
  if (!lds.last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  const int copy = lane & (kOrderCopies - 1);   // (pair i is always thread i % kThreads's)
  for (int base = threadIdx.x; base < pairs; base += 8 * kThreads) {   // (eight loads under way: each comes from beyond the L2)
    uint32_t w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = room->weight[min(base + j * kThreads, pairs - 1)];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = base + j * kThreads, bin = kOrderBins - 1 - (int)w[j];
      if (i < pairs) {
        lds.bin[i] = (uint16_t)bin;
        atomicAdd(&lds.count[copy][bin], 1u);
      }
    }
  }
  __syncthreads();
  // places of the first of every (weight, copy): two weights a thread
  uint32_t n[2][kOrderCopies], sum = 0;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int c = 0; c < kOrderCopies; ++c) sum += n[x][c] = lds.count[c][2 * threadIdx.x + x];
  uint32_t incl = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(incl, off);
    if (lane >= off) incl += y;
  }
  if (lane == 63) lds.sums[wave] = incl;
  __syncthreads();
  uint32_t before = incl - sum;
  for (int w = 0; w < wave; ++w) before += lds.sums[w];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int c = 0; c < kOrderCopies; ++c) {
      lds.count[c][2 * threadIdx.x + x] = before;
      before += n[x][c];
    }
  __syncthreads();
  for (int i = threadIdx.x; i < pairs; i += kThreads) {
    const int qb = i / nhead_k;
    order[atomicAdd(&lds.count[copy][lds.bin[i]], 1u)] = (uint32_t)qb << 16 | (uint32_t)(i - qb * nhead_k);
  }
}

// Keeps the message hbsa_last_error() returns and gives back `code` (defined in hbsa_fwd.hip).
int fail(int code, const char *fmt, ...);

// Launches, defined in hbsa_fwd_kernel.h, hbsa_fwd_f32.h and hbsa_bwd.h, instantiated by hbsa_inst.hip.
template <int D, typename E, bool OUT32>
int launch_fwd(const FwdParams &fp, long long items, hipStream_t stream);
template <int D, typename E>
int launch_fwd_fused(const FwdParams &fp, long long items, hipStream_t stream);
template <int D, typename E>
int launch_packed_eights(const FwdParams &fp, long long items, hipStream_t stream);
template <int D, typename E>
int launch_fwd_counted(const FwdParams &fp, long long items, hipStream_t stream);
template <int D, typename E, bool PARTS, int TEAMS>
int launch_fwd_cols(const FwdParams &fp, long long items, hipStream_t stream);
template <int D, typename E>
int launch_fwd_teams(const FwdParams &fp, long long items, hipStream_t stream);
template <int D, typename E>
int launch_fwd_parts(const FwdParams &fp, long long items, hipStream_t stream);
template <int D, typename E>
int launch_fwd_prepared_parts(const FwdParams &fp, long long items, hipStream_t stream);
template <int D, typename E>
int launch_fwd_decode(const FwdParams &fp, int most, long long items, hipStream_t stream);
template <int D>
int launch_fwd_f32(const FwdParams &fp, float c_signed, long long items, hipStream_t stream);
template <int D, typename E>
int launch_bwd(const BwdParams &bp, int nhead_k, int num_k_block, hipStream_t stream);

}  // namespace hbsa
