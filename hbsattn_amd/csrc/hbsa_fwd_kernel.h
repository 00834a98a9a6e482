// The attention kernel of the forward for 16-bit operands, and its launch functions.
#pragma once

#include "hbsa_common.h"

namespace hbsa {

// --------------------------------------------------------------------------------------
// Main kernel (persistent).  D = head dim (32, 64, 128 or 256); rows of K/V tiles are D*2 bytes.  At D = 256 a
// wavefront's output accumulator and query operand alone are 192 registers, so a CU runs one workgroup of four
// wavefronts, each with the 512 registers of a SIMD (the output in the AGPR half; hbsattn_amd/build.py), and its two 128 KB of K/V
// tile buffers take most of the LDS.
//
// Scheduling.  The grid is as many workgroups as fit the device at once and every workgroup
// loops over work items it claims from eight queues, one per XCD (the chip's eight dies, each
// with its own L2).  Queue v holds, head-major, the items of the kv heads h with h % 8 == v:
// for each such head every q block of the packed batch from the last to the first (under a
// causal mask the heaviest blocks of each sequence come first), and for each q block its
// groups of four wave slots.  The queues need no storage: entry idx of queue v decodes
// arithmetically, and one atomic counter per queue hands entries out.  A workgroup reads the
// id of the XCD it runs on from the hardware and drains that XCD's queue, so at any time the
// workgroups that share an L2 walk the K/V of one (or few) kv heads; when its queue is empty it
// takes from the other queues, which balances the tail.  A workgroup ends after at most eight
// consecutive failed claims, one per queue.
//
// Division of labour.  Wavefront 0 is also the workgroup's scheduler: one item ahead it
// claims a queue entry, fetches that item's geometry record and mask bits, and expands the
// bits into a list of 64-key tiles in LDS (adjacent kept k blocks merge into key runs).  The
// main loop of every wavefront then only steps through that list: no mask logic, no global
// metadata loads and no divergent control flow remain on the per-tile path.
//
// Pipelining.  K/V tiles stream through two LDS buffers without a bubble at item borders:
// while the last tile of an item is being computed the first tile of the next item is
// already on its way and the next item's Q rows are being fetched.
//
// LDS: K[2][64][D] then V[2][64][D] (double-buffered 64-key tiles), 16-byte chunks of
// every row XOR-swizzled so that both the K reads (16 rows x one chunk per 16 lanes) and
// the transposing V reads (4 rows x 64 bytes per 32 lanes) spread over all banks; then two
// item headers and two tile lists.
// --------------------------------------------------------------------------------------
constexpr int kListCap = 1024;   // tile entries per list; longer items are expanded in chunks
constexpr int kGroupCap = 2 * kListCap;   // GROUPED: 16-bit entries of a list, one per 16 keys
// Bytes of the one-launch form's staging area for one row of block_mask bytes (2048 blocks and the alignment slack)
constexpr int kMaskWindow = 2048;
constexpr int kMaskStage = kMaskWindow + 256;
constexpr int kTeamTiles = 6;   // tiles of an item that teams share, at least
constexpr float kMostSum = 256.f;   // 2^kLazyRescaleLog2
static_assert(kLazyRescaleLog2 == 8.0f, "kMostSum");

// Item header in LDS (16 ints).
enum { H_HK = 0, H_QB, H_SUB, H_TOTAL, H_ROW_BEGIN, H_ROWS, H_KEY_BEGIN, H_Q_POS, H_SHIFT, H_PART, H_T0, H_SEQ, H_NKBLK, H_GROUPS, H_KMAX, H_WORDS = 16 };

__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// A tile entry packs the in-sequence position of the tile's first key (a multiple of 16) and
// the number of valid keys (1..64).
__device__ __forceinline__ int pack_tile(int pos, int valid) { return ((pos >> 4) << 6) | (valid - 1); }

// Expands one item's kept-block bits into tile entries [chunk_base, chunk_base + kListCap) of
// the item's tile sequence, written to list[0..); returns the item's total tile count.
// Executed by one whole wavefront; `first_words`: lane i holds bit word i of the row.  Rows longer than
// 2048 blocks ask `more_words(window)` for the words window * 64 + lane (lane i: word window * 64 + i, zero
// past the row's end), arrived and ready to use.
template <int KT, typename MoreWords>
__device__ __forceinline__ int build_tile_list(int *list, int chunk_base, MoreWords &&more_words, int nwords, int kbs,
                                                FastDiv div_kbs, int kmax, uint32_t first_words, int lane) {
  if (kmax <= 0 || nwords <= 0) return 0;
  int total = 0;
  if ((kbs & (KT - 1)) == 0) {
    // Blocks are whole tiles: every kept block yields kbs / KT tiles (those starting at or past
    // kmax are dropped; they would be the last of the list).  Two bit words are expanded per
    // step: lane l looks at bit (l & 31) of word 2*step + (l >> 5), and its tiles go right after
    // the tiles of the kept blocks below it.
    constexpr int kShift = KT == 64 ? 6 : 5;
    static_assert(1 << kShift == KT, "tiles of 64 or 32 keys");
    const int tpb = kbs >> kShift;
    const int half = lane >> 5, bit = lane & 31;
    const int j_last = (int)fast_div((uint32_t)(kmax - 1), div_kbs);   // no bit above this block is set
    int window = 0;
    uint32_t held = lane < nwords ? first_words : 0u;
    for (int w2 = 0; w2 < nwords; w2 += 2) {
      if ((w2 >> 6) != window) {   // rows longer than 2048 blocks only
        window = w2 >> 6;
        held = more_words(window);
      }
      const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)held, w2 & 63);
      const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)held, (w2 + 1) & 63);   // nwords is even
      if ((lo | hi) == 0) continue;
      const uint32_t mine = half ? hi : lo;
      if ((mine >> bit) & 1u) {
        const int below = __builtin_popcount(mine & ((1u << bit) - 1u)) + (half ? __builtin_popcount(lo) : 0);
        const int j = (w2 + half) * 32 + bit;
        int off = total + below * tpb - chunk_base;
        for (int t = 0; t < tpb; ++t, ++off) {
          const int pos = j * kbs + KT * t;
          if (pos < kmax && off >= 0 && off < kListCap) list[off] = pack_tile(pos, min(KT, kmax - pos));
        }
      }
      total += (__builtin_popcount(lo) + __builtin_popcount(hi)) * tpb;
      if ((j_last >> 6) == (w2 >> 1)) {   // tiles dropped at the end of the last visible block
        const uint32_t wsel = (j_last & 32) ? hi : lo;
        if ((wsel >> (j_last & 31)) & 1u) total -= tpb - ((kmax - j_last * kbs + KT - 1) >> kShift);
      }
    }
  } else {
    // General block sizes: walk the runs of adjacent kept blocks serially (wavefront-uniform).
    int window = 0;
    uint32_t held = lane < nwords ? first_words : 0u;
    auto word = [&](int w) -> uint32_t {
      if ((w >> 6) != window) {   // rows longer than 2048 blocks only
        window = w >> 6;
        held = more_words(window);
      }
      return (uint32_t)__builtin_amdgcn_readlane((int)held, w & 63);
    };
    int blk = 0;
    for (;;) {
      int w = blk >> 5;
      if (w >= nwords) break;
      uint32_t cur = word(w) & (~0u << (blk & 31));
      while (cur == 0) {
        if (++w >= nwords) break;
        cur = word(w);
      }
      if (w >= nwords) break;
      const int first = w * 32 + __builtin_ctz(cur);
      uint32_t inv = ~word(w) & (~0u << (first & 31));
      while (inv == 0) {
        if (++w >= nwords) break;
        inv = ~word(w);
      }
      const int stop = (w >= nwords) ? nwords * 32 : w * 32 + __builtin_ctz(inv);
      blk = stop;
      const int end = min(stop * kbs, kmax);
      for (int pos = first * kbs; pos < end; pos += KT) {
        const int off = total - chunk_base;
        if (lane == 0 && off >= 0 && off < kListCap) list[off] = pack_tile(pos, min(KT, end - pos));
        ++total;
      }
      if (end >= kmax) break;
    }
  }
  return total;
}

// The same for tiles of 16-key groups: the kept blocks' groups (their in-sequence position / 16) one after another, entries
// [chunk_base, chunk_base + kGroupCap) of them to list[0..); returns the item's number of groups.  Whole wavefront; block sizes
// that are any multiple of 16.
template <typename MoreWords>
__device__ __forceinline__ int build_group_list(uint16_t *list, int chunk_base, MoreWords &&more_words, int nwords, int kbs,
                                                FastDiv div_kbs, int kmax, uint32_t first_words, int lane) {
  if (kmax <= 0 || nwords <= 0) return 0;
  const int gpb = kbs >> 4;
  const int half = lane >> 5, bit = lane & 31;
  const int j_last = (int)fast_div((uint32_t)(kmax - 1), div_kbs);   // no bit above this block is set
  int total = 0, window = 0;
  uint32_t held = lane < nwords ? first_words : 0u;
  for (int w2 = 0; w2 < nwords; w2 += 2) {   // 64 blocks a step, as above
    if ((w2 >> 6) != window) {
      window = w2 >> 6;
      held = more_words(window);
    }
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)held, w2 & 63);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)held, (w2 + 1) & 63);
    if ((lo | hi) == 0) continue;
    const uint32_t mine = half ? hi : lo;
    if ((mine >> bit) & 1u) {
      const int below = __builtin_popcount(mine & ((1u << bit) - 1u)) + (half ? __builtin_popcount(lo) : 0);
      const int first = ((w2 + half) * 32 + bit) * gpb;
      int off = total + below * gpb - chunk_base;
      for (int g = 0; g < gpb; ++g, ++off)
        if ((first + g) * 16 < kmax && off >= 0 && off < kGroupCap) list[off] = (uint16_t)(first + g);
    }
    total += (__builtin_popcount(lo) + __builtin_popcount(hi)) * gpb;
    if ((j_last >> 6) == (w2 >> 1)) {   // groups dropped at the end of the last visible block
      const uint32_t wsel = (j_last & 32) ? hi : lo;
      if ((wsel >> (j_last & 31)) & 1u) total -= gpb - ((kmax - j_last * kbs + 15) >> 4);
    }
  }
  return total;
}

template <int D, typename E, bool OUT32, int NW, bool EXTRAS, bool FUSED, bool PACK, bool COLS, bool GROUPED, bool COUNTED, bool ONE, int TEAMS>
__global__ __launch_bounds__(NW * TEAMS * 64, TEAMS > 1 || D > 192 ? 1 : D > 64 ? 8 / NW : D > 32 ? 3 : 4) void hbsa_fwd_kernel(FwdParams p) {
  // OUT32: fp32 output (the fp32-input path; q/k/v are then fp16 staging copies)
  // EXTRAS: the split over key blocks is compiled in, and (not FUSED) the clocked walk and the log-sum-exp output.  The
  // plain call uses none of them, and its kernel is a tenth shorter without them (1-2 % faster: eight
  // wavefronts in different parts of a long kernel share one instruction cache).
  // FUSED: the one-launch form.  No pre-pass has run: wavefront 0 derives an item's geometry from the
  // sequence boundaries (kept in LDS) and its bit row from the item's own block_mask bytes, which it
  // fetches into an LDS staging area one item ahead, where the other form fetches the prepared records.
  // PACK: wave slots packed across the q heads of a GQA group (see slot_of below).  Either placement of the queries gives the
  // same results bit for bit; a prepared mask's launch has packed ones where it is cut over key blocks or has teams.
  // COLS: the tensors' rows hold p.ncol <= D / 8 chunks of eight elements (a head dim that is no D of its own).  The
  // columns past them are zero in LDS (cleared once, never loaded) and in the Q operand, and not stored: in place of
  // zero-padded copies of q, k, v and a copy of the output.
  // GROUPED: tiles are made of groups of 16 keys from any places, for block sizes that are no multiple of the tile.  Otherwise a
  // tile is consecutive keys of one run of kept blocks, and the end of every run is a tile that is partly empty and has to be
  // masked (blocks of 48 keys, half of them kept: 120 keys' worth of tiles for 96, half of the tiles masked).
  // COUNTED: (FUSED) the caller has not counted the blocks; see FwdParams::counts.  Kernels of their own: compiled in everywhere, the
  // counting cost calls that do not use it 1 % (16 x 40 .. 500 tokens, 32 / 8 heads, 37.7 -> 38.0 us; 8 x 2050, 16 of 192, 227.6 -> 229.7).
  // ONE: (FUSED) no workgroup has a second item: nothing is staged, listed or claimed for one, and there is that much less code to fetch
  // before the first tile, at 0.1 us a cold line.  A third of a call of a few tiles is the scheduler's code: us, before and after, 2 x 27 tokens, 16 / 8
  // heads of 32, 8.0 -> 7.2; 2 x 54 .. 72, 32 / 16, 9.3 -> 8.4; 8 x 149 .. 240, 2 heads, 10.6 -> 9.7; 1 x 204 .. 512, 32 / 16 of 128, 15.2 -> 14.5.
  // (A kernel of its own, with packed slots, which give the same bits: as a branch it cost launches of two and more items 0.7 % at head dim
  // 128, 35.0 -> 35.3 and 64.0 -> 64.5; the COUNTED and COLS kernels and the split ones of four wavefronts,
  // where nothing got slower, have the branch; split ones of eight, whose items are long, lost 1 % with it.)
  // TEAMS: (ONE) the item's tiles are shared out among this many teams of NW wavefronts, each with tile buffers of its own, tile i to team
  // i % TEAMS; their sums are put together through LDS at the end.  For launches that leave SIMDs with one wavefront: alone there, its tile is a
  // chain of matrix products, exponentials and LDS reads with nothing beside them (see fwd_teams).
  // NW: wavefronts (wave slots) of a workgroup, 4 or 8.  Eight are used when the q heads of a GQA group
  // and the 32-row slices of a q block give an item more than four wave slots: one workgroup per CU then
  // stages every K/V tile once for all of them instead of two workgroups staging it each (D = 128 only, and
  // where the items fill the device: see fwd_split).
  constexpr int RB = D * 2;            // row bytes
  constexpr int CPR = RB / 16;         // 16-byte chunks per row
  // Keys per tile.  At head dims 160 and 192 tiles of 32 keys let two workgroups share a CU (their LDS, and the
  // registers of a wavefront with one half tile in the making): 8 x ~2000 tokens, 16 heads of 192, fp16, keep 0.3: see
  // launch_fwd_cols for the measurement.
  constexpr int KT = D > 128 && D <= 192 ? 32 : 64;
  constexpr int TILE_BYTES = KT * RB;
  constexpr int LOADS = (CPR * KT + 64 * NW - 1) / (64 * NW);   // 16-byte loads per thread per tile per operand
  constexpr bool LAST_PART = CPR * KT % (64 * NW) != 0;         // the last round is for the first wavefronts only
  using SW = FwdSwizzle<D>;
  constexpr int KSTEPS = D / 16;       // MFMA k-steps of Q.K^T
  constexpr int DT = D / 32;           // 32-row tiles of O^T
  constexpr bool WALK = EXTRAS && !FUSED && !ONE, LSE = EXTRAS && !FUSED;
  static_assert(TEAMS == 1 || ONE, "the tiles of one item");
  constexpr bool HAND = D <= 192;      // operand reads from LDS issued and waited for by hand (see lds_read_b128)

  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int team = TEAMS > 1 ? wave_all / NW : 0, wave = TEAMS > 1 ? wave_all % NW : wave_all;
  char *lds_k = lds + team * 4 * TILE_BYTES;
  int *lds_hdr = (int *)(lds + TEAMS * 4 * TILE_BYTES);     // [2][H_WORDS]
  int *lds_list = lds_hdr + 2 * H_WORDS;            // [2][kListCap]
  int *lds_seq = lds_list + 2 * kListCap;           // FUSED: [4][kSeqCap] cu_q, cu_k, cu_num_q_block, cu_num_k_block
  uint8_t *lds_mask = (uint8_t *)(lds_seq + 4 * kSeqCap);   // FUSED: [kMaskStage] block_mask bytes of the staged item
  auto hdr_word = [&](int c_, int i) { return __builtin_amdgcn_readfirstlane(lds_hdr[c_ * H_WORDS + i]); };

  const int lane = threadIdx.x & 63;
  const int g32 = lane >> 5;   // which half of the wavefront
  const int l32 = lane & 31;   // query within the wave slot / key row within a sub-tile

  // The launch's arguments, for what is done once an item: read again (scalar loads) each time.  Held in scalar registers over
  // the tile loop they do not fit: 100 to 240 of them went to lanes of vector registers.
  auto fresh_args = [&]() -> const FwdParams & {
    auto at = (const __attribute__((address_space(4))) FwdParams *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(at));
    return *(const FwdParams *)at;
  };

  // softmax constants of this launch (uniform): kernel arguments, or for fp32 inputs staged as fp16 what
  // the setup kernel that precedes this launch derived on the device
  float sm_c = p.c, sm_out_mul = 1.f;
  if (p.f32) {
    sm_c = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, p.sched->c)));
    sm_out_mul = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, p.sched->out_mul)));
  }
  // Leaving: wavefront 0 makes every claim of its workgroup.  Once its last claim has been performed it
  // counts the workgroup as done, and the workgroup that completes the count puts the queue counters
  // back to zero, so the next launch on this work description needs no preparation of its own.
  auto leave = [&]() {
    if (wave != 0 || p.one_each) return;   // (items without queues: no counter was touched)
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this workgroup's last claim has returned
    if (lane == 0) {
      const uint32_t before = atomicAdd(&p.sched->done, 1u);
      if (before + 1 == gridDim.x) {
#pragma unroll
        for (int i = 0; i < 8; ++i) atomicExch(&p.sched->qnext[i], 0u);
        atomicExch(&p.sched->done, 0u);
      }
    }
  };

  // ------------------------------------------------------------------ scheduler (wavefront 0)
  const int nq = p.nhead_k < 8 ? p.nhead_k : 8;                       // queues that hold work
  const int home = __builtin_amdgcn_s_getreg((3 << 11) | 20) & 7;    // HW_REG_XCC_ID
  const int first_queue = home < nq ? home : home % nq;
  int tries = 0;                    // queues found empty so far
  uint32_t pending = 0xffffffffu;   // queue index claimed for the item after the staged one
  int st_hk = -1, st_qb = 0, st_sub = 0, st_part = 0;   // staged item: claimed, records fetched, list not built
  uint32_t st_info = 0, st_bits = 0;       // lane i: word i of its QBlockInfo / of its bit row

  auto queue_len = [&](int v) -> uint32_t {
    const FwdParams &p = fresh_args();
    const int heads = v < p.nhead_k ? (p.nhead_k - v + 7) / 8 : 0;
    return (uint32_t)heads * (uint32_t)p.nqb * (uint32_t)p.nsub * (uint32_t)p.nparts;
  };
  // Without queues (few items per workgroup).  The items are numbered last q blocks first, the heads of a q block
  // next to each other (decode_free_entry), so under a causal mask their weights fall with the number.  Workgroup
  // i of G takes item i, then 2G - 1 - i, 2G + i, 4G - 1 - i, ...: every second round runs backwards, so the
  // lightest item of a round goes to the workgroup that got the heaviest of the round before, and the
  // workgroups (those of one CU, too) end at about the same time.  Nothing is claimed: measured against a shared
  // counter for the later rounds, 8 x 1024 tokens 106 -> 99 us and C5 0.258 -> 0.241 ms.
  int own_claims = 0, pending_sub = 0;
  auto claim = [&]() -> uint32_t {   // the value is looked at an item later, so its latency is hidden
    const FwdParams &p = fresh_args();
    uint32_t r = 0xffffffffu;
    if (p.one_each) {
      r = (own_claims & 1) ? (uint32_t)(own_claims + 1) * gridDim.x - 1u - blockIdx.x : (uint32_t)own_claims * gridDim.x + blockIdx.x;
      ++own_claims;
      if (p.order != nullptr) {   // the place in the order -> the item; a load that is waited for when the value is looked at
        const uint32_t whole = fast_div(r, p.div_nsub);
        pending_sub = (int)(r - whole * (uint32_t)p.nsub);
        r = r < (uint32_t)p.one_each ? p.order[whole] : 0xffffffffu;
      }
    } else if (tries < 8) {
      if (lane == 0) r = atomicAdd(&p.sched->qnext[(first_queue + tries) & 7], 1u);
    }
    return r;
  };
  // (kv head, q block, slot group, part) of entry `claimed` of a head-major list that starts at kv head
  // `head0` and holds every `head_step`-th head
  auto decode_entry = [&](uint32_t claimed, int head0, int head_step) {
    const FwdParams &p = fresh_args();
    const uint32_t whole = fast_div(claimed, p.div_nparts);   // parts of one item are neighbours
    st_part = (int)(claimed - whole * (uint32_t)p.nparts);
    const uint32_t t = fast_div(whole, p.div_nsub);
    st_sub = (int)(whole - t * (uint32_t)p.nsub);
    const uint32_t h = fast_div(t, p.div_nqb);
    st_hk = head0 + head_step * (int)h;
    st_qb = p.nqb - 1 - (int)(t - h * (uint32_t)p.nqb);
  };
  // (kv head, q block, slot group, part) of item `claimed` of the numbering without queues: parts, slot groups and
  // kv heads of a q block are neighbours, the last q block comes first
  auto decode_free_entry = [&](uint32_t claimed) {
    const FwdParams &p = fresh_args();
    const uint32_t whole = fast_div(claimed, p.div_nparts);
    st_part = (int)(claimed - whole * (uint32_t)p.nparts);
    const uint32_t t = fast_div(whole, p.div_nsub);
    st_sub = (int)(whole - t * (uint32_t)p.nsub);
    const uint32_t b = fast_div(t, p.div_nhk);
    st_hk = (int)(t - b * (uint32_t)p.nhead_k);
    st_qb = p.nqb - 1 - (int)b;
  };
  // ---- one-launch form: geometry and mask bits without a pre-pass (wavefront 0)
  const uint8_t *st_mrow = nullptr;   // staged item: address of the mask byte of its sequence's first k block
  int st_nvis = 0, st_ms = 0;         // its k blocks below the causal bound; offset of the first one's byte in the staging area
  // geometry of q block qb from the boundaries in LDS (uniform values); kb0: first global k block of its sequence.
  // Consecutive items of a queue mostly belong to one sequence, so the last sequence's boundaries are kept.
  SeqBounds seq_sb = {0, 0, 0, 0, 0, 0, 0};
  int seq_qb_end = -1;      // q blocks [seq_sb.qb0, seq_qb_end) belong to the kept sequence (none at first)
  bool seq_have = false;
  auto fused_geometry = [&](int qb, int &kb0) -> QBlockInfo {
    const FwdParams &p = fresh_args();
    if (!(qb >= seq_sb.qb0 && qb < seq_qb_end)) {
      int b = 0;   // sequences that start at or before qb, minus one
      for (int base = 0; base < p.batch; base += 64) {
        const int i = base + lane + 1;
        const int first_qb = i <= p.batch ? lds_seq[2 * kSeqCap + i] : 0x7fffffff;
        b += __builtin_popcountll(__builtin_amdgcn_ballot_w64(first_qb <= qb));
      }
      seq_have = b < p.batch;
      seq_sb = SeqBounds{0, 0, 0, 0, 0, 0, 0};
      seq_qb_end = -1;
      if (seq_have) {
        auto at = [&](int arr, int i) { return __builtin_amdgcn_readfirstlane(lds_seq[arr * kSeqCap + i]); };
        seq_sb.q0 = at(0, b); seq_sb.q1 = at(0, b + 1);
        seq_sb.k0 = at(1, b); seq_sb.k1 = at(1, b + 1);
        seq_sb.qb0 = at(2, b); seq_qb_end = at(2, b + 1);
        seq_sb.kb0 = at(3, b); seq_sb.kb1 = at(3, b + 1);
      }
    }
    return q_block_geometry(qb, seq_have, seq_sb, p.qbs, p.kbs, p.causal, p.nkb_total, p.total_q, p.total_k, kb0);
  };
  const uint32_t lds_mask_addr = (uint32_t)(uintptr_t)HBSA_AS3(lds_mask);
  // Requests the mask bytes of blocks [first, first + count), count <= kMaskWindow, of the row at `mrow`: whole
  // aligned dwords, four bytes per lane, straight into the staging area (a dword that holds a byte of the
  // row lies inside the mask's allocation).  Returns the offset of block `first`'s byte in the staging area.
  auto mask_dma = [&](const uint8_t *mrow, int first, int count) -> int {
    const uintptr_t a = (uintptr_t)(mrow + first);
    const int sh = (int)(a & 3);
    const char *base = (const char *)(a - sh);
    const uint32_t last = (uint32_t)(sh + count - 1) & ~3u;   // offset of the last dword needed
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");        // what was read from the staging area before has arrived
    for (uint32_t i = 0; i <= last; i += 256) {
      const uint32_t off = min(i + 4u * (uint32_t)lane, last);   // every lane loads: lanes past the end repeat the last dword
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                   :
                   : "s"(lds_mask_addr + i), "v"(off), "s"(base)
                   : "memory", "m0");
    }
    return sh;
  };
  // bit words of the staged bytes: lane i gets word i (blocks 32 * i .. + 31 of the window; zero from `count` on)
  auto staged_words = [&](int sh, int count) -> uint32_t {
    uint32_t words = 0;
    for (int w64 = 0; w64 * 64 < count; ++w64) {
      const int j = w64 * 64 + lane;
      const bool keep = j < count && lds_mask[sh + j] != 0;
      const uint64_t bal = __builtin_amdgcn_ballot_w64(keep);
      if (lane == 2 * w64) words = (uint32_t)bal;
      if (lane == 2 * w64 + 1) words = (uint32_t)(bal >> 32);
    }
    return words;
  };
  // words of a later window of a row (rows longer than kMaskWindow blocks): fetched and waited for on the spot
  auto fused_more_words = [&](const uint8_t *mrow, int nvis, int part) {
    return [&, mrow, nvis, part](int window) -> uint32_t {
      const int first = window * kMaskWindow;
      const int count = min(kMaskWindow, nvis - first);
      if (count <= 0) return 0u;
      const int sh = mask_dma(mrow, first, count);
      __builtin_amdgcn_s_waitcnt(0x0F70);
      asm volatile("" : : : "memory");
      uint32_t words = staged_words(sh, count);
      if constexpr (EXTRAS) {   // (a row of several windows: cut by position)
        if (nvis > kMaskWindow) words &= ItemParts(fresh_args(), nvis).word_mask(part, 32 * (window * 64 + lane));
      }
      return words;
    };
  };
  // the same for a prepared bit row in the workspace
  auto prepared_more_words = [&](const uint32_t *row, int nwords, int part, int kmax, int nkblk) {
    return [=](int window) -> uint32_t {
      const int i = window * 64 + lane;
      uint32_t held = i < nwords ? row[i] : 0u;
      __builtin_amdgcn_s_waitcnt(0x0F70);   // wait here, not (for everything in flight) on the common path
      asm volatile("" : "+v"(held));
      if constexpr (EXTRAS) {
        const FwdParams &p = fresh_args();
        const int nvis = min(nkblk, (int)fast_div((uint32_t)(kmax + p.kbs - 1), p.div_kbs));
        if (p.nparts > 1 && nvis > kMaskWindow) held &= ItemParts(p, nvis).word_mask(part, 32 * i);
      }
      return held;
    };
  };

  // turn `pending` into the staged item (claiming again from the next queues when the one it
  // came from is exhausted) and start fetching the item's records
  auto stage = [&]() {
    const FwdParams &p = fresh_args();
    uint32_t claimed = (uint32_t)__builtin_amdgcn_readfirstlane((int)pending);
    st_hk = -1;
    if (p.one_each) {
      if (p.order != nullptr) {
        if (claimed != 0xffffffffu) {
          st_hk = (int)(claimed & 0xffffu);
          st_qb = (int)(claimed >> 16);
          st_sub = pending_sub;
          st_part = 0;
        }
      } else if (claimed < (uint32_t)p.one_each) {
        decode_free_entry(claimed);
      }
    } else {
      while (tries < 8) {
        const int v = (first_queue + tries) & 7;
        if (claimed < queue_len(v)) {
          decode_entry(claimed, v, 8);
          break;
        }
        // This queue has run dry (the tail of the kernel).  Look at the other queues' counters first, all at
        // once, and claim only from one that still shows work: a workgroup then ends after one load instead
        // of seven failed claims in a row, each a round trip to a counter every other workgroup is hitting.
        uint32_t seen = 0xffffffffu;
        if (lane < 8) seen = __hip_atomic_load(&p.sched->qnext[(first_queue + lane) & 7], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_waitcnt(0x0F70);
        asm volatile("" : "+v"(seen));
        const bool open = lane > tries && lane < 8 && seen < queue_len((first_queue + lane) & 7);
        const uint64_t open_mask = __builtin_amdgcn_ballot_w64(open);
        if (open_mask == 0) {
          tries = 8;
          break;
        }
        tries = __builtin_ctzll(open_mask);
        uint32_t r = 0;
        if (lane == 0) r = atomicAdd(&p.sched->qnext[(first_queue + tries) & 7], 1u);
        __builtin_amdgcn_s_waitcnt(0x0F70);
        asm volatile("" : "+v"(r));
        claimed = (uint32_t)__builtin_amdgcn_readfirstlane((int)r);
      }
    }
    if (st_hk >= 0) {
      if constexpr (FUSED) {
        int kb0;
        const QBlockInfo r = fused_geometry(st_qb, kb0);
        st_info = (uint32_t)(lane == 0 ? r.row_begin : lane == 1 ? r.rows : lane == 2 ? r.key_begin : lane == 3 ? r.klen
                             : lane == 4 ? r.q_pos : lane == 5 ? r.shift : lane == 6 ? r.nkblk : lane == 7 ? r.kmax
                             : lane == 8 ? r.seq : 0);
        st_nvis = min(r.nkblk, (int)fast_div((uint32_t)(r.kmax + p.kbs - 1), p.div_kbs));
        st_mrow = p.mask + (int64_t)st_hk * p.ms_h + (int64_t)st_qb * p.ms_q + kb0;
        st_ms = st_nvis > 0 ? mask_dma(st_mrow, 0, min(st_nvis, kMaskWindow)) : 0;
      } else {
        st_info = lane < 12 ? ((const uint32_t *)(p.info + st_qb))[lane] : 0u;
        st_bits = lane < p.wpr ? p.bits[((size_t)st_hk * p.nqb + st_qb) * p.wpr + lane] : 0u;
      }
    }
  };
  // the tiles (GROUPED: groups) [chunk_base, ..) of an item into list `c`; returns how many the item has
  auto list_of = [&](int c, int chunk_base, auto &&more_words, int nwords, int kmax, uint32_t first_words) -> int {
    const FwdParams &p = fresh_args();
    if constexpr (GROUPED)
      return build_group_list((uint16_t *)(lds_list + c * kListCap), chunk_base * (KT / 16), more_words, nwords, p.kbs, p.div_kbs, kmax, first_words, lane);
    else
      return build_tile_list<KT>(lds_list + c * kListCap, chunk_base, more_words, nwords, p.kbs, p.div_kbs, kmax, first_words, lane);
  };
  // Split over key blocks: part `part` sees a share of the item's kept k blocks, counted from the bit row, so that parts are of one
  // length and an item of few keys is whole; a row of several windows of words is cut by position.
  // words: lane i's word i of the row (of blocks below nvis); returns the part's, and how many parts the item has.
  auto part_words = [&](uint32_t words, int nvis, int part, int &parts) -> uint32_t {
    const FwdParams &p = fresh_args();
    if (32 * lane >= nvis) words = 0u;   // (a prepared row is written as far as its sequence goes)
    if (nvis > kMaskWindow) {
      const ItemParts cut(p, nvis);
      parts = cut.count;
      return words & cut.word_mask(part, 32 * lane);
    }
    const int mine = __builtin_popcount(words);
    int upto = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int x = __shfl_up(upto, off);
      if (lane >= off) upto += x;
    }
    const ItemParts cut(p, __builtin_amdgcn_readlane(upto, 63));
    parts = cut.count;
    // kept blocks of this word before and after the part
    int skip = min(max(part * cut.per - (upto - mine), 0), mine), drop = min(max(upto - (part + 1) * cut.per, 0), mine);
    if (part >= parts || skip + drop >= mine) return 0u;
    for (; skip > 0; --skip) words &= words - 1u;
    for (; drop > 0; --drop) words &= ~(0x80000000u >> __builtin_clz(words));
    return words;
  };
  // expand the staged item into list `c` and write its header
  auto build = [&](int c) {
    const FwdParams &p = fresh_args();
    int *hdr = lds_hdr + c * H_WORDS;
    int total = 0, parts = 1;
    if (st_hk >= 0) {
      const int nkblk = __builtin_amdgcn_readlane((int)st_info, 6);
      const int kmax = __builtin_amdgcn_readlane((int)st_info, 7);
      // packed slots behind the q block's entries: no rows, so no tiles
      auto rowless = [&]() { return st_sub * NW * kWaveRows >= p.ratio * __builtin_amdgcn_readlane((int)st_info, 1); };
      if constexpr (FUSED) {
        // the staged bytes arrived with the wait of a tile, or one of the waits before the first item, since stage()
        st_bits = st_nvis > 0 ? staged_words(st_ms, min(st_nvis, kMaskWindow)) : 0u;
        if constexpr (EXTRAS) {
          st_bits = part_words(st_bits, st_nvis, st_part, parts);
          if (rowless()) parts = 0;
        }
        if (!EXTRAS || st_part < parts)
          total = list_of(c, 0, fused_more_words(st_mrow, st_nvis, st_part), 2 * ((st_nvis + 63) >> 6), kmax, st_bits);
      } else {
        const int nwords = 2 * ((nkblk + 63) >> 6);
        if (EXTRAS && p.nparts > 1) st_bits = part_words(st_bits, min(nkblk, (int)fast_div((uint32_t)(kmax + p.kbs - 1), p.div_kbs)), st_part, parts);
        if (EXTRAS && PACK && rowless()) parts = 0;
        if (!EXTRAS || st_part < parts)
          total = list_of(c, 0, prepared_more_words(p.bits + ((size_t)st_hk * p.nqb + st_qb) * p.wpr, nwords, st_part, kmax, nkblk), nwords, kmax, st_bits);
      }
    }
    if (lane == 0) {
      hdr[H_HK] = st_hk; hdr[H_QB] = st_qb; hdr[H_SUB] = st_sub;
      hdr[H_PART] = EXTRAS ? st_part | parts << 8 : 0;
      hdr[H_TOTAL] = GROUPED ? (total + KT / 16 - 1) / (KT / 16) : total;
      if (GROUPED) hdr[H_GROUPS] = total;
      hdr[H_T0] = 0;   // the item's walk starts at its first tile unless next_start() decides otherwise
    }
    if (lane < 9) {   // QBlockInfo words: row_begin, rows, key_begin, klen, q_pos, shift, nkblk, kmax, seq
      const int dst = lane == 0 ? H_ROW_BEGIN : lane == 1 ? H_ROWS : lane == 2 ? H_KEY_BEGIN : lane == 4 ? H_Q_POS
                      : lane == 5 ? H_SHIFT : lane == 6 ? H_NKBLK : lane == 7 ? H_KMAX : lane == 8 ? H_SEQ : -1;
      if (dst >= 0) hdr[dst] = (int)st_info;
    }
  };

  // ---- the walk clock (wavefront 0; p.walk != 0 only).  The online softmax does not care in which
  // order an item's tiles are taken, and the workgroups that share an L2 (one XCD) work on items of
  // one (kv head, sequence) at a time.  They keep near each other in key space, so that a K/V tile one
  // of them fetched is still in the L2 when the others ask for it: every (kv head, sequence) has a
  // clock word that holds, for the workgroups inside its items, their number (low 16 bits) and the sum
  // of their positions (upper 48 bits; a position counts 64-key tiles of the sequence's key space and
  // keeps growing over laps); one 64-bit atomic add updates both and returns both.  An item starts its
  // walk at the first of its tiles at or after the clock's mean position, walks upwards, wraps to its
  // first tile and ends where it began; it adds every step to the clock.  The start is decided two
  // tiles before the item begins (its first tile is requested one tile before).
  unsigned long long w_clk = 0;          // lane 0: the next item's clock as read three tiles before this item's end
  unsigned long long *w_ptr = nullptr;   // this item's clock word, nullptr when it takes no part
  int w_lap = 0, w_told = 0;             // the lap this item started in; the position its clock holds for it
  int w_next_lap = 0;                    // lap the next item starts in (-1: it takes no part); the workgroup's
                                         // first item finds the clocks empty: lap 0, first tile
  int w_lt = 1;                          // 64-key tiles of this item's sequence (the length of a lap)
  // what wavefront 0 remembers of the two items whose lists are in LDS (slot c_): clock word, lap length,
  // and whether the item may take part (its tile list is a single chunk of at least three tiles)
  unsigned long long *w_clock_of[2] = {nullptr, nullptr};
  int w_tiles_of[2] = {1, 1};
  bool w_part_of[2] = {false, false};
  auto note_item = [&](int c_, int total_) {   // right after build(c_), from the staged records
    const FwdParams &p = fresh_args();
    const int nkblk = __builtin_amdgcn_readlane((int)st_info, 6);
    const int seq = __builtin_amdgcn_readlane((int)st_info, 8);
    w_part_of[c_] = WALK && p.walk != 0 && st_hk >= 0 && total_ >= 3 && total_ <= kListCap;
    w_clock_of[c_] = p.clock + (size_t)(st_hk < 0 ? 0 : st_hk) * p.nqb + seq;
    w_tiles_of[c_] = (nkblk * p.kbs + kTileKeys - 1) >> 6;
  };
  // three tiles before this item ends: read the next item's clock (a load that bypasses the CU's own
  // cache; the clock words live in the XCD's L2, where the atomics on them are performed)
  auto peek_next = [&](int cn) {
    w_next_lap = -1;
    if (!w_part_of[cn]) return;
    if (lane == 0) w_clk = __hip_atomic_load(w_clock_of[cn], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    w_next_lap = 0;
  };
  // two tiles before it ends: the next item's start, from the clock's mean position
  auto next_start = [&](int cn) {
    if (w_next_lap < 0) return;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)w_clk);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(w_clk >> 32));
    const uint32_t members = lo & 0xffffu;
    if (members == 0) return;   // nobody there: start at the first tile, in lap 0
    const float sum = (float)hi * 65536.f + (float)(lo >> 16);
    int mean = __builtin_amdgcn_readfirstlane((int)(sum * __builtin_amdgcn_rcpf((float)members)));
    const int lt = w_tiles_of[cn];
    int lap = __builtin_amdgcn_readfirstlane((int)((float)mean * __builtin_amdgcn_rcpf((float)lt)));
    int pos = mean - lap * lt;
    while (pos < 0) { pos += lt; --lap; }
    while (pos >= lt) { pos -= lt; ++lap; }
    // entries of the (ascending) list below that position
    const int n = hdr_word(cn, H_TOTAL);
    int below = 0;
    for (int i = 0; i < n; i += 64) {
      const bool less = i + lane < n && (lds_list[cn * kListCap + i + lane] >> 8) < pos;   // entry >> 6 = key >> 4
      below += __builtin_popcountll(__builtin_amdgcn_ballot_w64(less));
    }
    if (below >= n) {   // every tile of the item lies below: it starts the next lap at its first tile
      below = 0;
      ++lap;
    }
    if (lane == 0) lds_hdr[cn * H_WORDS + H_T0] = below;
    w_next_lap = lap;
  };
  // first tile of an item: join its clock; later: add the progress since the last report (the atomics
  // return nothing).  wraps: how often the walk has passed the end of the list (0 or 1).
  auto report = [&](int c_, int kpos, bool first, int wraps) {
    if (first) {
      w_ptr = nullptr;
      const int lap0 = w_next_lap;
      w_next_lap = -1;   // the item after this one takes part only if peek_next() says so
      if (lap0 < 0 || !w_part_of[c_]) return;
      w_ptr = w_clock_of[c_];
      w_lt = w_tiles_of[c_];
      w_lap = lap0;
      w_told = w_lap * w_lt + (kpos >> 6);
      if (lane == 0) atomicAdd(w_ptr, ((unsigned long long)(uint32_t)w_told << 16) + 1ull);
      return;
    }
    if (w_ptr == nullptr) return;
    const int now = (w_lap + wraps) * w_lt + (kpos >> 6);
    if (now != w_told && lane == 0) atomicAdd(w_ptr, (unsigned long long)(uint32_t)(now - w_told) << 16);
    w_told = now;
  };
  auto leave_clock = [&]() {
    if (w_ptr == nullptr) return;
    if (lane == 0) atomicAdd(w_ptr, 0ull - (((unsigned long long)(uint32_t)w_told << 16) + 1ull));
    w_ptr = nullptr;
  };

  constexpr bool MAY_ONE = COUNTED || COLS || (FUSED && EXTRAS && NW == 4);
  const bool one = ONE || (MAY_ONE && p.one_each != 0 && p.one_each <= (int)gridDim.x);
  const bool schedules = wave_all == 0 && !one;
  if constexpr (COLS) {
    for (int i = threadIdx.x; i < TEAMS * 4 * TILE_BYTES / 16; i += NW * TEAMS * 64) *(u32x4 *)(lds + i * 16) = u32x4{0u, 0u, 0u, 0u};
  }
  if (wave_all == 0) {
    if constexpr (FUSED) {   // the sequences' boundaries, for fused_geometry()
      for (int i = lane; i <= p.batch; i += 64) {
        lds_seq[i] = p.cu_q[i];
        lds_seq[kSeqCap + i] = p.cu_k[i];
        lds_seq[2 * kSeqCap + i] = p.cu_nqb[i];   // (either array where the caller has not counted: replaced below)
        lds_seq[3 * kSeqCap + i] = p.cu_nkb[i];
      }
      // (lanes read what others have written, here and in fused_geometry(): no read is to move up, no write down)
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if constexpr (COUNTED) {   // as hbsa_block_counts_kernel, whose launch was 2.6 us of a call's 13.5 (5 x 32 tokens, 8 / 2 heads of 32)
        const int l = lane;
        bool bad = false;
#pragma unroll
        for (int side = 0; side < 2; ++side) {
          if (!((p.count_info[1] >> side) & 1)) continue;
          const int *cu = lds_seq + side * kSeqCap;
          int *first = lds_seq + (2 + side) * kSeqCap, before = 0;
          const uint32_t size = (uint32_t)(side == 0 ? p.qbs : p.kbs);
          for (int base = 0; base <= p.batch; base += 64) {
            const int i = base + l;
            int n = 0;
            if (i < p.batch) {
              const int64_t len = (int64_t)cu[i + 1] - cu[i];
              if (len < 0) bad = true;
              else n = (int)((uint32_t)(len + size - 1) / size);
            }
            int incl = n;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
              const int x = __shfl_up(incl, off);
              if (l >= off) incl += x;
            }
            if (i <= p.batch) first[i] = before + incl - n;
            before += __builtin_amdgcn_readlane(incl, 63);
          }
          if (before != (side == 0 ? p.nqb : p.nkb_total)) bad = true;
        }
        bad = __builtin_amdgcn_ballot_w64(bad) != 0;
        if (bad)   // the mask does not fit: sequences without blocks, nothing is read for them
          for (int i = l; i <= p.batch; i += 64) {
            if (p.count_info[1] & 1) lds_seq[2 * kSeqCap + i] = 0;
            if (p.count_info[1] & 2) lds_seq[3 * kSeqCap + i] = 0;
          }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (blockIdx.x == 0 && l == 0)
          __hip_atomic_store((uint64_t *)(p.counts + 2), (uint64_t)(uint32_t)p.count_info[0] << 32 | (bad ? 0u : 1u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
    pending = claim();
    stage();
    if constexpr (FUSED) {   // the first item's mask bytes
      __builtin_amdgcn_s_waitcnt(0x0F70);
      asm volatile("" : : : "memory");
    }
    build(0);
    note_item(0, hdr_word(0, H_TOTAL));
    if (schedules) {
      pending = claim();
      stage();
      pending = claim();
    } else if (lane == 0) {
      lds_hdr[H_WORDS + H_HK] = -1;
    }
  }

  // ------------------------------------------------------------------ per-thread constants
  // tile loads: thread -> (row, 16-byte chunk) of the tile, same for every tile
  // Rounds of the workgroup's loads that are a whole number of rows after which the chunk placement repeats apart differ in
  // their scalar base only: load i takes offset i % OFFSETS, ahead_rows(i) rows on (at head dim 256, whose rounds are a quarter of
  // the period, four offsets in place of eight: 8 x 2050 tokens, 16 heads of 208, 412 -> 310 us when the kernel still spilled, 225
  // now).  Where rows are no power of two long every load has its offset in a register.
  constexpr int ROUND_ROWS = SW::POW2 ? 64 * NW / CPR : 0;
  constexpr int OFFSETS = !SW::POW2 ? LOADS : ROUND_ROWS >= SW::PERIOD ? 1 : SW::PERIOD / ROUND_ROWS < LOADS ? SW::PERIOD / ROUND_ROWS : LOADS;
  static_assert(!SW::POW2 || (OFFSETS == LOADS || OFFSETS * ROUND_ROWS % SW::PERIOD == 0), "loads that share an offset share their chunk");
  auto ahead_rows = [](int i) constexpr { return i / OFFSETS * OFFSETS * ROUND_ROWS; };
  uint32_t ld_koff[OFFSETS], ld_voff[OFFSETS];   // byte offset of the thread's chunk from the tile's (GROUPED: the group's) first row
  bool ld_kin[OFFSETS], ld_vin[OFFSETS];         // COLS: the chunk is one of the row's
  const uint32_t ks32 = (uint32_t)p.k_s, vs32 = (uint32_t)p.v_s;   // row strides in bytes (the host checks they fit)
  auto ld_place = [&](int i, int &r, uint32_t &kchunk, uint32_t &vchunk) {
    const int c = (i * NW + wave) * 64 + lane;
    const int pc = c % CPR;
    r = c / CPR;
    kchunk = (uint32_t)((pc ^ SW::k(r)) * 16);
    vchunk = (uint32_t)((pc ^ SW::v(r)) * 16);
  };
#pragma unroll
  for (int i = 0; i < OFFSETS; ++i) {
    int r; uint32_t kc, vc;
    ld_place(i, r, kc, vc);
    const uint32_t from = GROUPED ? (uint32_t)r & 15u : (uint32_t)r;
    ld_koff[i] = from * ks32 + kc;
    ld_voff[i] = from * vs32 + vc;
    ld_kin[i] = !COLS || kc < (uint32_t)p.ncol * 16u;
    ld_vin[i] = !COLS || vc < (uint32_t)p.ncol * 16u;
  }
  const uint32_t lds_k_addr = (uint32_t)(uintptr_t)HBSA_AS3(lds_k);
  // kbase / vbase: wavefront-uniform address of the tile's first key row (for this kv head).
  // 16 bytes per lane go straight from global memory into LDS at (M0 + 16 * lane); the global
  // address is a scalar base plus a 32-bit per-lane offset.  The V buffers follow the K buffers.
  auto dma16 = [&](auto off_, const char *sbase, uint32_t voff, uint32_t lds_addr) {
    constexpr int off = decltype(off_)::value;
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(sbase), "n"(off)
                 : "memory", "m0", "scc");
  };
  auto tile_ptr = [&](const char *base, int tok, uint32_t stride) {   // tok >= 0
    return base + (uint64_t)(uint32_t)tok * (uint64_t)stride;
  };
  // A tile as the wavefronts know it: keys 0 .. valid - 1 of it exist, key x is the sequence's key pos(x / 16) + x % 16.
  // Plain: consecutive keys from `first` on.  GROUPED: sixteen bits per group of 16 keys, their position / 16.
  struct TileRef {
    int first, valid;
    uint32_t lo, hi;
    __device__ __forceinline__ int pos(int g) const {
      if constexpr (GROUPED) return (int)(((g < 2 ? lo : hi) >> (16 * (g & 1))) & 0xffffu) << 4;
      else return first + 16 * g;
    }
  };
  // step `at` (of all steps) of the item with header c_, from its list entry (GROUPED: 64 bits, four groups; 32 with two)
  auto tile_ref = [&](uint32_t lo, uint32_t hi, int c_, int at, int total) -> TileRef {
    TileRef r;
    if constexpr (GROUPED) {
      r.lo = lo;
      r.hi = hi;
      r.valid = KT;
      r.first = r.pos(0);
      if (at + 1 >= total) {   // the item's last tile: groups may be missing, and keys of the last group
        const int n = hdr_word(c_, H_GROUPS) - at * (KT / 16);
        int last = r.pos(0);
#pragma unroll
        for (int g = 1; g < KT / 16; ++g) last = n > g ? r.pos(g) : last;
        r.valid = 16 * (n - 1) + min(16, hdr_word(c_, H_KMAX) - last);
      }
    } else {
      r.first = (int)(lo >> 6) << 4;
      r.valid = (int)(lo & 63u) + 1;
      r.lo = r.hi = 0;
    }
    return r;
  };
  auto group_entry = [&](int c_, int at) -> u32x2 {   // GROUPED: entry `at` of list c_, the tile's groups
    const int *list = lds_list + c_ * kListCap + at * (KT / 32);
    if constexpr (KT == 64) return *(const u32x2 *)list;
    else return u32x2{(uint32_t)*list, 0u};
  };
  // the tile of list entry `at` (of the list's chunk, which starts at step chunk_base)
  auto listed_tile = [&](int c_, int at, int chunk_base) -> TileRef {
    const int total = GROUPED ? hdr_word(c_, H_TOTAL) : 0;
    if constexpr (GROUPED) {
      const u32x2 w = group_entry(c_, at);
      return tile_ref((uint32_t)__builtin_amdgcn_readfirstlane((int)w.x), (uint32_t)__builtin_amdgcn_readfirstlane((int)w.y), c_, chunk_base + at, total);
    } else {
      return tile_ref((uint32_t)__builtin_amdgcn_readfirstlane(lds_list[c_ * kListCap + at]), 0u, c_, chunk_base + at, total);
    }
  };
  static_assert(!GROUPED || 1024 % RB != 0 || NW * 64 / CPR % 16 == 0 || 16 % (NW * 64 / CPR) == 0, "no load is rows of two groups");
  // One operand's half of a tile's loads.  V_PART selects the V buffers (which follow the K buffers).
  // base: of the sequence's first key (for this kv head)
  auto issue_part = [&](auto v_part_, int buf, const char *base, const TileRef &tile) {
    constexpr bool V_PART = decltype(v_part_)::value;
    constexpr int lds_off = V_PART ? 2 * TILE_BYTES : 0;
    const uint32_t l0 = lds_k_addr + (uint32_t)(buf * TILE_BYTES) + (uint32_t)wave * 1024u;
    const int valid = tile.valid;
    const uint32_t stride = V_PART ? vs32 : ks32;
    if constexpr (GROUPED) {
      // Load i of this wavefront is rows of one group (g), or of two where a row is no power of two long.  The lane offsets
      // count from the row's group.  Rows past the tile's end re-read the last valid row (masked later).
      const uint64_t groups = (uint64_t)tile.hi << 32 | tile.lo;
      int wave_ = wave;
      if constexpr (KT == 32) asm volatile("" : "+s"(wave_));   // (or what follows from it is kept in registers for every load)
      auto group_at = [&](int g) -> uint32_t { return ((uint32_t)(groups >> (16 * g)) & 0xffffu) << 4; };
      if constexpr (KT == 32) {   // two groups: one scalar base, and the second group's lanes go on by the distance
        const uint32_t apart = valid > 16 ? (uint32_t)(tile.pos(1) - tile.pos(0)) * stride : 0u;
        base += (uint64_t)(uint32_t)tile.pos(0) * (uint64_t)stride;
        static_for<0, LOADS>([&](auto i_) {
          constexpr int i = decltype(i_)::value;
          uint32_t voff = (V_PART ? ld_voff[i % OFFSETS] : ld_koff[i % OFFSETS]) +
                          (lane >= 16 * CPR - (i * NW + wave_) * 64 ? apart : 0u);
          if (valid < KT) {
            const int row = ((i * NW + wave_) * 64 + lane) / CPR;
            uint32_t step = (uint32_t)((min(row, valid - 1) & 15) - (row & 15)) * stride;
            asm volatile("" : "+v"(step));
            voff += step;
          }
          if ((!LAST_PART || i < LOADS - 1 || (i * NW + wave) * 64 < CPR * KT) && (!COLS || (V_PART ? ld_vin[i % OFFSETS] : ld_kin[i % OFFSETS])))
            dma16(std::integral_constant<int, lds_off + i * NW * 1024>{}, base, voff, l0);
        });
        return;
      }
      static_for<0, LOADS>([&](auto i_) {
        constexpr int i = decltype(i_)::value;
        constexpr bool WHOLE = 1024 % RB == 0;
        constexpr int ROUND = NW * 64 / CPR;   // rows between two loads
        const int row = ((i * NW + wave_) * 64 + lane) / CPR;
        int g = WHOLE ? ((wave_ * 64 / CPR) >> 4) + i * ROUND / 16 : ((i * NW + wave_) * 64 / CPR) >> 4;
        uint32_t voff = V_PART ? ld_voff[i % OFFSETS] : ld_koff[i % OFFSETS];
        if (valid < KT) {
          g = min(g, (valid - 1) >> 4);
          uint32_t step = (uint32_t)((min(row, valid - 1) & 15) - (row & 15)) * stride;
          asm volatile("" : "+v"(step));   // (or a 64-bit multiply-add is formed, and its 64-bit addend kept in registers)
          voff += step;
        }
        const uint32_t pos = group_at(g);
        if constexpr (!WHOLE) {
          const int second = 16 * (g + 1) * CPR - (i * NW + wave_) * 64;   // first lane of the second group, if one of them is
          voff += lane >= second ? (group_at(min(g + 1, (valid - 1) >> 4)) - pos) * stride : 0u;
        }
        if ((!LAST_PART || i < LOADS - 1 || (i * NW + wave) * 64 < CPR * KT) && (!COLS || (V_PART ? ld_vin[i % OFFSETS] : ld_kin[i % OFFSETS])))
          dma16(std::integral_constant<int, lds_off + i * NW * 1024>{},
                base + (uint64_t)(pos + ((uint32_t)ahead_rows(i) & 15u)) * (uint64_t)stride, voff, l0);
      });
      return;
    }
    base = tile_ptr(base, tile.first, stride);
    if (__builtin_expect(valid == KT, 1)) {
      static_for<0, LOADS>([&](auto i_) {
        constexpr int i = decltype(i_)::value;
        if ((!LAST_PART || i < LOADS - 1 || (i * NW + wave) * 64 < CPR * KT) && (!COLS || (V_PART ? ld_vin[i % OFFSETS] : ld_kin[i % OFFSETS])))   // (a lane that loads nothing leaves its 16 bytes of LDS alone)
        dma16(std::integral_constant<int, lds_off + i * NW * 1024>{}, base + (uint64_t)(uint32_t)ahead_rows(i) * (V_PART ? vs32 : ks32),
              V_PART ? ld_voff[i % OFFSETS] : ld_koff[i % OFFSETS], l0);
      });
    } else {   // ragged tail of a run: rows past the end re-read the last valid row (masked later)
      static_for<0, LOADS>([&](auto i_) {
        constexpr int i = decltype(i_)::value;
        const int r0 = (i % OFFSETS * NW * 64 + wave * 64 + lane) / CPR;
        uint32_t step = (uint32_t)(min(r0 + ahead_rows(i), valid - 1) - r0) * (V_PART ? vs32 : ks32);
        asm volatile("" : "+v"(step));   // (or a 64-bit multiply-add is formed, and its 64-bit addend kept in registers)
        if ((!LAST_PART || i < LOADS - 1 || (i * NW + wave) * 64 < CPR * KT) && (!COLS || (V_PART ? ld_vin[i % OFFSETS] : ld_kin[i % OFFSETS])))
        dma16(std::integral_constant<int, lds_off + i * NW * 1024>{}, base, (V_PART ? ld_voff[i % OFFSETS] : ld_koff[i % OFFSETS]) + step, l0);
      });
    }
  };
  auto issue_k = [&](int buf, const char *kbase, const TileRef &tile) { issue_part(std::false_type{}, buf, kbase, tile); };
  auto issue_v = [&](int buf, const char *vbase, const TileRef &tile) { issue_part(std::true_type{}, buf, vbase, tile); };
  // the first keys of the sequence of the item with header c_
  auto item_k = [&](int c_) -> const char * {
    const FwdParams &pn = fresh_args();
    return tile_ptr(pn.k + (int64_t)hdr_word(c_, H_HK) * pn.k_h, hdr_word(c_, H_KEY_BEGIN), ks32);
  };
  auto item_v = [&](int c_) -> const char * {
    const FwdParams &pn = fresh_args();
    return tile_ptr(pn.v + (int64_t)hdr_word(c_, H_HK) * pn.v_h, hdr_word(c_, H_KEY_BEGIN), vs32);
  };
  auto issue_first = [&](int buf, int c_) {   // the first tile of an item that starts at its list's first entry
    const TileRef tile = listed_tile(c_, 0, 0);
    issue_k(buf, item_k(c_), tile);
    issue_v(buf, item_v(c_), tile);
  };

  // per-lane LDS read addresses
  // K (A operand of S^T): row l32 (+32), chunk (2*ks + g32) ^ swz(row)
  // V^T (A operand of O^T) through ds_read_b64_tr_b16: within a group of 16 lanes, lane r
  // supplies the address of key (r / 4), dims 4*(r % 4) .. +3 and receives dim r of 4 keys.
  const int v_key = 4 * g32 + ((lane & 15) >> 2);
  const int v_lc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  const int v_rd = v_key * RB + 8 * (lane & 1);

  // Absolute LDS addresses of this lane's operand reads in the CURRENT tile buffer: one per k-step
  // for K, one per 32-dim block for V.  flip_buffers() moves them to the other buffer with one add
  // each (the two buffers of K, and of V, are TILE_BYTES apart), so the per-tile path has no
  // address arithmetic besides that.
  // (Where the swizzle touches the low chunk bits only, k-steps and blocks further on are immediate offsets.)
  constexpr int KADDR = SW::POW2 ? KSTEPS : CPR % 8 == 0 ? 4 : 2, VADDR = SW::POW2 ? DT : CPR % 8 == 0 ? 2 : 1;
  uint32_t k_addr[KADDR], v_addr[VADDR];
#pragma unroll
  for (int ks = 0; ks < KADDR; ++ks) k_addr[ks] = lds_k_addr + (uint32_t)(l32 * RB + (((2 * ks + g32) ^ SW::k(l32)) << 4));
#pragma unroll
  for (int dt = 0; dt < VADDR; ++dt) v_addr[dt] = lds_k_addr + 2 * TILE_BYTES + (uint32_t)(v_rd + (((4 * dt + v_lc) ^ SW::v(v_key)) << 4));
  int buf = 0;
  auto flip_buffers = [&]() {
    buf ^= 1;
    const uint32_t step = buf ? (uint32_t)TILE_BYTES : (uint32_t)-TILE_BYTES;
#pragma unroll
    for (int ks = 0; ks < KADDR; ++ks) {
      k_addr[ks] += step;
      asm volatile("" : "+v"(k_addr[ks]));   // keep it in its register instead of recomputing it per read
    }
#pragma unroll
    for (int dt = 0; dt < VADDR; ++dt) {
      v_addr[dt] += step;
      asm volatile("" : "+v"(v_addr[dt]));
    }
  };

  // This wavefront's slot of an item.  A wave slot holds up to 32 (q head of the GQA group, query row of the
  // q block) entries.  Plain form: the 32-row slices of one head after another (slot = head * wps + slice), a
  // q block of 80 rows filling 32 + 32 + 16 entries per head.  Packed form (PACK: q_block_size no multiple
  // of 32 and several q heads per kv head): entry number = head * rows + row, every slot takes the next 32
  // numbers, so a slot may hold the last rows of one head and the first rows of the next and only an item's
  // last slot is partly empty.  Every lane works on one query with its own pointers and causal limit, and
  // all heads of the group see the same K/V tiles, so nothing else changes.
  struct Slot {
    int first;          // first entry number (packed) / first row of the slice (plain)
    int n;              // entries held, <= 0: none
    int min_r, max_r;   // smallest and largest query row among them
    int hq;             // plain form: the slot's q head; packed form: the group's first q head
  };
  // a / b for 0 <= a < 2^20 (kPackedEntries), b > 0.  Exact: (a + 0.5) / b is 0.5 / b or more from the whole numbers, a relative distance of 2^-21 of
  // what is at most 2^20 / b, and the reciprocal (1 ulp) and the product (half of one) are off by 1.5 * 2^-23 of it.  (Above 2^22 it is not exact.)
  auto quotient = [](int a, int b) {
    return (int)(((float)a + 0.5f) * __builtin_amdgcn_rcpf((float)b));
  };
  auto slot_of = [&](int hk, int sub, int rows) -> Slot {
    const FwdParams &p = fresh_args();
    const int slot = sub * NW + wave;
    Slot sl;
    if constexpr (PACK) {
      sl.hq = hk * p.ratio;
      sl.first = slot * kWaveRows;
      sl.n = min(kWaveRows, p.ratio * rows - sl.first);
      sl.min_r = 0;
      sl.max_r = rows - 1;
      if (sl.n > 0) {
        const int h0 = __builtin_amdgcn_readfirstlane(quotient(sl.first, rows));
        const int h1 = __builtin_amdgcn_readfirstlane(quotient(sl.first + sl.n - 1, rows));
        if (h0 == h1) {   // all entries belong to one head
          sl.min_r = sl.first - h0 * rows;
          sl.max_r = sl.min_r + sl.n - 1;
        }
      }
    } else {
      const int head = slot / p.wps;
      sl.hq = hk * p.ratio + head;
      sl.first = (slot % p.wps) * kWaveRows;
      sl.n = head < p.ratio ? min(kWaveRows, rows - sl.first) : 0;
      sl.min_r = sl.first;
      sl.max_r = sl.first + sl.n - 1;
    }
    return sl;
  };
  // q head and row (inside the q block) of entry idx of a slot with entries; idx past the last entry repeats it.
  // (The plain form needs nothing but the slot: what stays live through an item's tiles is as little as it can be.)
  auto slot_entry = [&](const Slot &sl, int idx, int rows, int &hq, int &r) {
    const int e = sl.first + min(idx, sl.n - 1);
    if constexpr (PACK) {
      const int h = quotient(e, rows);
      hq = sl.hq + h;
      r = e - h * rows;
    } else {
      hq = sl.hq;
      r = e;
    }
  };

  // Q^T fragments (B operand) of one item: lane (l32, g32) ends up with, per k-step ks, the 16 bytes
  // d = 16*ks + 8*g32 .. +7 of query row l32.  Fetched so that four lanes read 64 contiguous bytes
  // of a row (16 rows per instruction instead of 32, half the memory requests): with h = bit 4 of
  // the lane, load A_k takes row (lane % 16), load B_k row 16 + (lane % 16), both at bytes
  // 64*k + 32*h + 16*g32; then the h = 1 lanes of A_k and the h = 0 lanes of B_k trade places
  // (v_permlane16_swap), which leaves k-step 2k in A_k and k-step 2k+1 in B_k.
  // The loads go out when the item before has formed its last scores; place_q() waits for them when the item begins.
  short8v qf[KSTEPS];
  static_assert(KSTEPS % 2 == 0, "the loads come in pairs of k-steps");
  auto request_q = [&](int hk, int sub, int row_begin, int rows) {
    const FwdParams &p = fresh_args();
    const Slot sl = slot_of(hk, sub, rows);
    if (sl.n <= 0) return;   // this wavefront has no rows: qf is never used
    const int l16 = lane & 15;
    int hq_a, r_a, hq_b, r_b;
    slot_entry(sl, l16, rows, hq_a, r_a);
    slot_entry(sl, 16 + l16, rows, hq_b, r_b);
    const char *base = p.q + (lane & 16) * 2 + g32 * 16;
    const char *ra = base + (int64_t)(row_begin + r_a) * p.q_s + (int64_t)hq_a * p.q_h;
    const char *rb = base + (int64_t)(row_begin + r_b) * p.q_s + (int64_t)hq_b * p.q_h;
#pragma unroll
    for (int k = 0; k < KSTEPS / 2; ++k) {
      u32x4 a = {0u, 0u, 0u, 0u}, b = a;
      if (!COLS || 4 * k + ((lane >> 4) & 1) * 2 + g32 < p.ncol) {
        a = *(const u32x4 *)(ra + 64 * k);
        b = *(const u32x4 *)(rb + 64 * k);
      }
      qf[2 * k] = __builtin_bit_cast(short8v, a);
      qf[2 * k + 1] = __builtin_bit_cast(short8v, b);
    }
  };
  auto place_q = [&]() {
    const FwdParams &p = fresh_args();
#pragma unroll
    for (int k = 0; k < KSTEPS / 2; ++k) {
      u32x4 a = __builtin_bit_cast(u32x4, qf[2 * k]) ^ p.q_sign, b = __builtin_bit_cast(u32x4, qf[2 * k + 1]) ^ p.q_sign;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const auto r = __builtin_amdgcn_permlane16_swap(a[j], b[j], false, false);
        a[j] = r[0];
        b[j] = r[1];
      }
      qf[2 * k] = __builtin_bit_cast(short8v, a);
      qf[2 * k + 1] = __builtin_bit_cast(short8v, b);
    }
  };

  // ------------------------------------------------------------------ first item
  __syncthreads();   // (the other wavefronts have done what is above while wavefront 0 made the list, and its code is there)
  int c = 0;   // list / header of the current item
  if (hdr_word(0, H_HK) < 0) {
    if (!ONE) leave();
    return;
  }
  // tiles of a step of all teams; a short list is the first team's alone
  const int step = TEAMS > 1 && hdr_word(0, H_TOTAL) >= kTeamTiles && (FUSED || p.sched->shared_tiles != 0) ? TEAMS : 1;
  const int off = step > 1 ? team : team > 0 ? 0x3fffffff : 0;   // the team's first tile
  if constexpr (TEAMS > 1) {
    if (off < hdr_word(0, H_TOTAL)) {
      const TileRef tile = listed_tile(0, off, 0);
      issue_k(0, item_k(0), tile);
      issue_v(0, item_v(0), tile);
    }
  } else if (hdr_word(0, H_TOTAL) > 0) {
    issue_first(0, 0);
  }
  if (TEAMS == 1 || team == 0 || step > 1) request_q(hdr_word(0, H_HK), hdr_word(0, H_SUB), hdr_word(0, H_ROW_BEGIN), hdr_word(0, H_ROWS));
  // What this wavefront asked for so far has arrived, the scheduler's records included: the compiler is told here, or it
  // waits for ALL outstanding memory traffic where they are first read.
  bool settled = false;   // ... since the scheduler last asked for something
  auto settle = [&]() {
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
    asm volatile("" : "+v"(st_info), "+v"(st_bits), "+v"(pending), "+v"(w_clk));
    settled = true;
  };

  for (;;) {   // ------------------------------------------------------ one iteration per work item
    const int cur_hk = hdr_word(c, H_HK);
    const int cur_sub = hdr_word(c, H_SUB);
    const int cur_part = EXTRAS ? hdr_word(c, H_PART) & 255 : 0, cur_parts = EXTRAS ? hdr_word(c, H_PART) >> 8 : 1;   // read now: wavefront 0 rewrites the header while others finish this item
    const int total = hdr_word(c, H_TOTAL);
    const int row_begin = hdr_word(c, H_ROW_BEGIN);
    const int rows = hdr_word(c, H_ROWS);
    const int key_begin = hdr_word(c, H_KEY_BEGIN);
    const int q_pos = hdr_word(c, H_Q_POS);
    const int shift = hdr_word(c, H_SHIFT);

    // The q rows were requested after the item's first tile, and a wavefront's loads return in order: once it has put them in
    // place its part of that tile is there as well.  What the scheduler asks for below then has the first tile's time to arrive.
    // (In every wavefront: the compiler then knows that these loads have arrived.)
    place_q();
    if (schedules) {   // stay one item ahead: expand the staged item, stage the one after it
      if (!settled) settle();   // (the staged item's mask bytes among what it waits for: no tile of the item before may have been waited for)
      build(c ^ 1);
      if (WALK && p.walk) note_item(c ^ 1, hdr_word(c ^ 1, H_TOTAL));
      stage();
      pending = claim();
      settled = false;
    }

    const Slot slot = slot_of(cur_hk, cur_sub, rows);
    const int nrows = slot.n;   // lanes l32 < nrows hold a query
    // last key position this lane's query / any query of the wavefront sees (causal): key position <= q_pos + row + shift
    int lane_kvis;
    if constexpr (PACK) {
      int hq_mine, r_mine = 0;
      if (nrows > 0) slot_entry(slot, l32, rows, hq_mine, r_mine);
      lane_kvis = q_pos + r_mine + shift;
    } else {
      lane_kvis = q_pos + slot.first + min(l32, nrows - 1) + shift;   // (a wavefront without queries never looks at it)
    }
    const int wave_kvis_min = q_pos + slot.min_r + shift;
    const int wave_kvis_max = q_pos + slot.max_r + shift;
    const bool active = nrows > 0 && (TEAMS == 1 || team == 0 || step > 1);

    f32x16 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
    float m_ref = -INFINITY;  // reference the row's exponentials are formed against, times c (log2 units)
    float l_run = 0.f;        // this lane's share of the row sum

    const FwdParams &pi = fresh_args();
    const char *kg = pi.k + (int64_t)cur_hk * pi.k_h + (int64_t)key_begin * pi.k_s;
    const char *vg = pi.v + (int64_t)cur_hk * pi.v_h + (int64_t)key_begin * pi.v_s;

    int nxt_hk = -1;          // known once the last tile is reached
    int chunk_base = 0;
    // the walk starts at entry t0 of the (ascending) list and wraps: step t takes entry rot(t)
    constexpr int kCap = GROUPED ? kGroupCap / (KT / 16) : kListCap;   // tiles of a list
    const int t0 = !GROUPED && total <= kListCap ? hdr_word(c, H_T0) : 0;
    for (;;) {   // ---------------------------------------------------- chunks of the tile list (usually one)
      const int n = min(kCap, total - chunk_base);
      auto rot = [&](int x) { return x + t0 >= n ? x + t0 - n : x + t0; };   // x < n
      u32x2 held = {0u, 0u};  // lane i: entry of step (window * 64 + i) of the current chunk
      auto entry_of = [&](int x) -> u32x2 {   // lane i: that of step x + i
        u32x2 w = {0u, 0u};
        if (x + lane < n) {
          if constexpr (GROUPED) w = group_entry(c, x + lane);
          else w.x = (uint32_t)lds_list[c * kListCap + rot(x + lane)];
        }
        return w;
      };
      auto held_tile = [&](const u32x2 &from, int lane_at, int x) -> TileRef {
        return tile_ref((uint32_t)__builtin_amdgcn_readlane((int)from.x, lane_at),
                        GROUPED ? (uint32_t)__builtin_amdgcn_readlane((int)from.y, lane_at) : 0u, c, chunk_base + x, total);
      };
      held = entry_of(0);
      TileRef nx_tile = {0, 0, 0u, 0u};
      if (TEAMS == 1 || off < n) nx_tile = held_tile(held, TEAMS > 1 ? off : 0, TEAMS > 1 ? off : 0);
      for (int t = 0; t < n; t += TEAMS > 1 ? step : 1) {   // ---------------------------------- one iteration per 64-key tile
        const TileRef tile = nx_tile;
        const int kpos = tile.first, valid = tile.valid;
        const int t_next = TEAMS > 1 ? t + off + step : t + 1;
        const bool more = t_next < n, last = chunk_base + t + 1 == total;
        // The next tile is looked up before the wait, and what is rare stands out of line: between the barrier and the tile's first
        // products none of the workgroup's wavefronts has work for the matrix cores, and scalar code there, taken branches above
        // all, is paid by every one of them (some 70 scalar instructions and six taken branches before, 30 and one here: 16 x 40 .. 500
        // tokens, 32 / 8 heads of 128, 35.4 -> 34.7 us; two chunks on 65000 keys 268 -> 262; 8 x 2050, 16 heads of 192, 215 -> 211).
        TileRef nx = {0, 0, 0u, 0u};      // valid > 0: a next tile exists and its loads go out during this tile
        if (__builtin_expect(more, 1)) {
          if (__builtin_expect((t_next & 63) < (TEAMS > 1 ? step : 1), 0)) held = entry_of(t_next & ~63);
          nx = held_tile(held, t_next & 63, t_next);
        }
        const char *nx_k = kg, *nx_v = vg;
        const bool compute = active && (TEAMS == 1 || t + off < n) && (!p.causal || kpos <= wave_kvis_max);
        // keys that are missing, or (causal) a last key that some lane's query does not see
        const bool edge = valid < KT || (p.causal && tile.pos(KT / 16 - 1) + 15 > wave_kvis_min);

        if (t > 0 || chunk_base > 0 || !active) settle();   // the current tile has landed in LDS
        __syncthreads();                     // ... for every wave, and the other buffers are free

        // The clock is dealt with on few tiles only (wavefront 0; any work it does alone on every tile
        // makes the other three wait at the next barrier): the item's first tile, every eighth, and
        // the last three.
        if (WALK && p.walk && wave == 0 && ((t & (kWalkReportTiles - 1)) == 0 || chunk_base + t + 3 >= total)) {
          report(c, kpos, chunk_base + t == 0, t + t0 >= n ? 1 : 0);
          if (chunk_base + t + 3 == total) peek_next(c ^ 1);
          if (chunk_base + t + 2 == total) next_start(c ^ 1);
          if (last) leave_clock();
        }
        if (!ONE && __builtin_expect(last, 0)) {
          nxt_hk = hdr_word(c ^ 1, H_HK);
          if (nxt_hk >= 0 && hdr_word(c ^ 1, H_TOTAL) > 0) {
            nx = listed_tile(c ^ 1, GROUPED ? 0 : hdr_word(c ^ 1, H_T0), 0);
            nx_k = item_k(c ^ 1);
            nx_v = item_v(c ^ 1);
          }
        }
        nx_tile = nx;
        // The next tile's K is requested right after this tile's first operand reads, its V only after
        // the first MFMA block: the wavefronts then do not all queue at the load unit at once.

        if (!compute && nx.valid > 0) {
          issue_k(buf ^ 1, nx_k, nx);
          issue_v(buf ^ 1, nx_v, nx);
        }
        if (compute) {
          // The tile is processed as two halves of 32 keys so that, inside one wavefront, the
          // matrix cores always have work queued while the vector ALU does the softmax of the
          // other half:   S0 | S1 + exp(S0) | PV0 + exp(S1) | PV1.   (A maximum, of S0, is formed for an item's first tile alone:
          // see settle_half.)
          const bool first = chunk_base + t == 0;   // the item's first tile gives the reference
          f32x16 s0, s1;
#pragma unroll
          for (int i = 0; i < 16; ++i) { s0[i] = 0.f; s1[i] = 0.f; }

          // ---- K operand reads: 2 * KSTEPS reads (all k-steps of the first 32 keys, then of the
          // second 32), PF of them in flight, each consumed by one MFMA
          constexpr int PF = 4;
          constexpr int NK = KT / 32 * KSTEPS;
          short8v kb[PF];
          auto read_k = [&](auto i_) {
            constexpr int i = decltype(i_)::value;
            constexpr int ks = i % KSTEPS;
            constexpr int off = ks / KADDR * KADDR * 32;
            if constexpr (i < KSTEPS) kb[i % PF] = lds_read_b128<off, HAND>(k_addr[ks % KADDR]);
            else kb[i % PF] = lds_read_b128<off + 32 * RB, HAND>(k_addr[ks % KADDR]);
          };
          static_for<0, PF>(read_k);
          // the next tile's K is requested while this tile's first operands are on their way from LDS
          if (nx.valid > 0) issue_k(buf ^ 1, nx_k, nx);
          // ---- S0 = K[0:32] . Q^T
          static_for<0, KSTEPS>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            constexpr int ahead = (NK - 1 - i) < (PF - 1) ? (NK - 1 - i) : (PF - 1);
            if constexpr (HAND) lds_wait1<ahead>(kb[i % PF]);
            s0 = E::mfma(kb[i % PF], qf[i % KSTEPS], s0);
            if constexpr (i + PF < NK) read_k(std::integral_constant<int, i + PF>{});
          });

          if (nx.valid > 0) issue_v(buf ^ 1, nx_v, nx);

          // Largest score of one half in log2 units.  The first reduction step is an instruction the compiler knows, so
          // that it inserts the wait states an MFMA result needs before the vector ALU may read it; the
          // hand-written v_max3 steps all depend on that first result.
          auto half_rowmax = [&](const f32x16 &sh) {
            float mx = __builtin_amdgcn_fmed3f(sh[0], sh[1], INFINITY);   // = max(sh[0], sh[1])
#pragma unroll
            for (int i = 2; i < 16; i += 2) mx = max3(mx, sh[i], sh[i + 1]);
            return half_max(mx) * sm_c;
          };
          auto hide = [&](f32x16 &sh, int half) {   // keys this lane's query does not see
            if (edge) {
              int lim[2];   // keys of the half's two groups below lim are visible
#pragma unroll
              for (int g = 0; g < 2; ++g) {
                lim[g] = valid - 32 * half - 16 * g;
                if (p.causal) lim[g] = min(lim[g], lane_kvis - tile.pos(2 * half + g) + 1);
                lim[g] -= 4 * g32;
              }
#pragma unroll
              for (int i = 0; i < 16; ++i)
                if (8 * ((i >> 2) & 1) + (i & 3) >= lim[i >> 3]) sh[i] = -INFINITY;
            }
          };
          // exponentials of one half against reference m, packed to the element type (two groups of 16 keys); their sum
          auto half_exp = [&](const f32x16 &sh, float m, short8v &p_lo, short8v &p_hi) {
            u32x4 w[2];
            float sum = 0.f;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
#pragma unroll
              for (int q4 = 0; q4 < 4; ++q4) {
                const float e0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sh[8 * j + 2 * q4], sm_c, -m));
                const float e1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sh[8 * j + 2 * q4 + 1], sm_c, -m));
                w[j][q4] = E::pack2(e0, e1);
                // fp32 adds, not v_dot2c: the dot instructions share the matrix pipeline and would
                // stall the MFMAs of the wavefront's neighbour on the SIMD
                sum += e0 + e1;
              }
              asm volatile("" : "+v"(w[j]));   // packed here, or the 32-bit exponentials stay alive until their sum has been looked at
            }
            p_lo = __builtin_bit_cast(short8v, w[0]);
            p_hi = __builtin_bit_cast(short8v, w[1]);
            return sum;
          };
          // Whether the reference was good enough for a half, and if not (rarely, or with a NaN) a better one.  No maximum
          // is formed: the exponentials are taken against the reference of the halves before, and only a sum (which
          // has to be formed anyway) above 2^kLazyRescaleLog2 can hide an exponential above it.  Then the maximum is looked
          // for, the reference of the rows that ask for it moved there, O and l rescaled and the exponentials formed again.
          // In place of a maximum of every half (eight v_max3 in a chain, an exchange between half wavefronts, a rescaled P),
          // which the exponentials had to wait for.  (Sixteen exponentials reach that sum at 2^4 each, so the reference moves
          // whenever this is entered: left where no exponential alone exceeds 2^8, a plateau of later scores that lie 2^4 to 2^8
          // above the first tile's comes back here for every half: scores of deviation 0.3 with the first key block's 4 below the
          // rest, 8 x 8192 tokens, 32 heads of 128, 1112 -> 929 us (918 without the step), 4 x 4096, 16 heads of 64, 164 -> 114
          // (112).  A row whose own sums did not ask keeps its reference, so its bits do not depend on its neighbours.)
          auto settle_half = [&](const f32x16 &sh, float sum, short8v &p_lo, short8v &p_hi) {
            const uint64_t asked = __builtin_amdgcn_ballot_w64(!(sum <= kMostSum));
            if (__builtin_expect(asked != 0, 0)) {
              const float mx = half_rowmax(sh);
              const bool grow = (((uint32_t)asked | (uint32_t)(asked >> 32)) >> l32 & 1u) != 0 && mx > m_ref;
              const float m_new = grow ? mx : m_ref;
              const float alpha = grow ? __builtin_amdgcn_exp2f(m_ref - m_new) : 1.f;
              l_run *= alpha;
#pragma unroll
              for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
              m_ref = m_new;
              sum = half_exp(sh, m_ref == -INFINITY ? 0.f : m_ref, p_lo, p_hi);   // (a row that has seen no key yet)
            }
            l_run += sum;
          };
          auto read_vgroup = [&](auto g_, short4v *dst) {   // V^T operands of keys 16*g .. 16*g+15
            constexpr int g = decltype(g_)::value;
            static_for<0, DT>([&](auto dt_) {
              constexpr int dt = decltype(dt_)::value;
              constexpr int off = g * 16 * RB + dt / VADDR * VADDR * 64;
              dst[2 * dt] = lds_read_tr16_b64<off, HAND>(v_addr[dt % VADDR]);
              dst[2 * dt + 1] = lds_read_tr16_b64<off + 8 * RB, HAND>(v_addr[dt % VADDR]);
            });
          };
          auto wait_vgroup = [&](auto n_, short4v *v) {
            constexpr int n = decltype(n_)::value;
            if constexpr (!HAND) {
              (void)v;   // the compiler waits for its own reads
            } else if constexpr (DT == 4) {
              lds_wait<n>(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]);
            } else if constexpr (DT == 6) {
              asm volatile("s_waitcnt lgkmcnt(%12)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]),
                           "+v"(v[6]), "+v"(v[7]), "+v"(v[8]), "+v"(v[9]), "+v"(v[10]), "+v"(v[11]) : "n"(n));
            } else if constexpr (DT == 5) {
              asm volatile("s_waitcnt lgkmcnt(%10)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]),
                           "+v"(v[6]), "+v"(v[7]), "+v"(v[8]), "+v"(v[9]) : "n"(n));
            } else if constexpr (DT == 3) {
              asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]) : "n"(n));
            } else if constexpr (DT == 2) {
              asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]) : "n"(n));
            } else {
              static_assert(DT == 1, "one statement waits and names every register of the reads it waits for");
              asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(v[0]), "+v"(v[1]) : "n"(n));
            }
          };
          auto pv_group = [&](const short8v &pb, const short4v *v) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
              const short8v va = __builtin_shufflevector(v[2 * dt], v[2 * dt + 1], 0, 1, 2, 3, 4, 5, 6, 7);
              o[dt] = E::mfma(va, pb, o[dt]);
            }
          };

          if constexpr (KT == 32) {
            // one half: its V operands are on their way while the vector ALU does the softmax
            short8v p0a, p0b;
            short4v vb[2 * DT];
            read_vgroup(std::integral_constant<int, 0>{}, vb);
            hide(s0, 0);
            if (first) m_ref = half_rowmax(s0);
            settle_half(s0, half_exp(s0, m_ref, p0a, p0b), p0a, p0b);
            wait_vgroup(std::integral_constant<int, 0>{}, vb);
            pv_group(p0a, vb);
            read_vgroup(std::integral_constant<int, 1>{}, vb);
            wait_vgroup(std::integral_constant<int, 0>{}, vb);
            pv_group(p0b, vb);
          } else {
          hide(s0, 0);
          if (first) m_ref = half_rowmax(s0);

          // ---- S1 = K[32:64] . Q^T   interleaved with   P0 = exp(S0)
          short8v p0a, p0b, p1a, p1b;
          static_for<KSTEPS, NK>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            constexpr int ahead = (NK - 1 - i) < (PF - 1) ? (NK - 1 - i) : (PF - 1);
            if constexpr (HAND) lds_wait1<ahead>(kb[i % PF]);
            s1 = E::mfma(kb[i % PF], qf[i % KSTEPS], s1);
            if constexpr (i + PF < NK) read_k(std::integral_constant<int, i + PF>{});
          });
          short4v vb[2][2 * DT];
          read_vgroup(std::integral_constant<int, 0>{}, vb[0]);
          read_vgroup(std::integral_constant<int, 1>{}, vb[1]);
          settle_half(s0, half_exp(s0, m_ref, p0a, p0b), p0a, p0b);
          hide(s1, 1);

          // ---- O^T += V^T[:, 0:32] . P0   interleaved with   P1 = exp(S1)
          wait_vgroup(std::integral_constant<int, 2 * DT>{}, vb[0]);
          pv_group(p0a, vb[0]);
          read_vgroup(std::integral_constant<int, 2>{}, vb[0]);
          wait_vgroup(std::integral_constant<int, 2 * DT>{}, vb[1]);
          pv_group(p0b, vb[1]);
          read_vgroup(std::integral_constant<int, 3>{}, vb[1]);
          settle_half(s1, half_exp(s1, m_ref, p1a, p1b), p1a, p1b);

          // ---- O^T += V^T[:, 32:64] . P1
          wait_vgroup(std::integral_constant<int, 2 * DT>{}, vb[0]);
          pv_group(p1a, vb[0]);
          wait_vgroup(std::integral_constant<int, 0>{}, vb[1]);
          pv_group(p1b, vb[1]);
          }
        }
        flip_buffers();
      }
      chunk_base += n;
      if (chunk_base >= total) break;
      // a longer item: expand the next chunk of its tile list in place
      __syncthreads();
      if (wave_all == 0) {
        // (the staged records now belong to a later item, so this item's are fetched again)
        const FwdParams &p = fresh_args();
        const int qb = hdr_word(c, H_QB);
        if constexpr (FUSED) {
          int kb0;
          const QBlockInfo inf = fused_geometry(qb, kb0);
          const int nvis = min(inf.nkblk, (int)fast_div((uint32_t)(inf.kmax + p.kbs - 1), p.div_kbs));
          auto more = fused_more_words(p.mask + (int64_t)cur_hk * p.ms_h + (int64_t)qb * p.ms_q + kb0, nvis, cur_part);
          uint32_t first = more(0);
          if constexpr (EXTRAS) {
            int parts;
            first = part_words(first, nvis, cur_part, parts);
          }
          (void)list_of(c, chunk_base, more, 2 * ((nvis + 63) >> 6), inf.kmax, first);
          // the staging area held the staged item's bytes: request them again (they arrive with the next tile's wait)
          if (!ONE && st_hk >= 0 && st_nvis > 0) st_ms = mask_dma(st_mrow, 0, min(st_nvis, kMaskWindow));
        } else {
          const QBlockInfo inf = p.info[qb];
          const uint32_t *row = p.bits + ((size_t)cur_hk * p.nqb + qb) * p.wpr;
          const int nwords = 2 * ((inf.nkblk + 63) >> 6);
          uint32_t first = lane < nwords ? row[lane] : 0u;
          if (EXTRAS && p.nparts > 1) {
            int parts;
            first = part_words(first, min(inf.nkblk, (int)fast_div((uint32_t)(inf.kmax + p.kbs - 1), p.div_kbs)), cur_part, parts);
          }
          (void)list_of(c, chunk_base, prepared_more_words(row, nwords, cur_part, inf.kmax, inf.nkblk), nwords, inf.kmax, first);
        }
      }
      __syncthreads();
      if (TEAMS == 1 || off < total - chunk_base) {   // nothing is in flight here: fetch the chunk's first tile
        const TileRef tile = listed_tile(c, TEAMS > 1 ? off : 0, chunk_base);
        issue_k(buf, kg, tile);
        issue_v(buf, vg, tile);
      }
    }

    // Q of this item is no longer needed: the next item's rows are requested while the last MFMAs drain and the epilogue runs
    // (outside of the tile loop, or the compiler waits for them inside it)
    if (nxt_hk >= 0) request_q(nxt_hk, hdr_word(c ^ 1, H_SUB), hdr_word(c ^ 1, H_ROW_BEGIN), hdr_word(c ^ 1, H_ROWS));

    if constexpr (TEAMS > 1) {   // the teams' sums: to the larger of their references, in the order of the teams
      static_assert((DT * 4 + 1) * 1024 <= 8 * TILE_BYTES / (TEAMS > 1 ? NW : 1), "the sums of a team fit its and the first team's tile buffers");
      if (step > 1) {
        f32x4 *sums = (f32x4 *)lds + wave * (DT * 4 + 1) * 64 + lane;
        __syncthreads();   // no tile is read any more
        if (team > 0 && active) {
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) sums[(dt * 4 + i) * 64] = f32x4{o[dt][4 * i], o[dt][4 * i + 1], o[dt][4 * i + 2], o[dt][4 * i + 3]};
          sums[DT * 4 * 64] = f32x4{m_ref, l_run, 0.f, 0.f};
        }
        __syncthreads();
        if (team == 0 && active) {
          const f32x4 ml = sums[DT * 4 * 64];
          const float m = fmaxf(m_ref, ml[0]);
          const float mine = m_ref == m ? 1.f : __builtin_amdgcn_exp2f(m_ref - m), other = ml[0] == m ? 1.f : __builtin_amdgcn_exp2f(ml[0] - m);
          m_ref = m;
          l_run = l_run * mine + ml[1] * other;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const f32x4 x = sums[(dt * 4 + i) * 64];
#pragma unroll
              for (int j = 0; j < 4; ++j) o[dt][4 * i + j] = o[dt][4 * i + j] * mine + x[j] * other;
            }
        }
      }
    }

    // ---- epilogue: normalise, convert, store (rows with no visible key store exact zeros)
    if (active && (TEAMS == 1 || team == 0) && (!EXTRAS || cur_part < cur_parts)) {
      const FwdParams &p = fresh_args();
      int hq, my_r;   // this lane's query (lanes l32 >= nrows repeat the last one and store nothing)
      slot_entry(slot, l32, rows, hq, my_r);
      const float l_tot = half_sum(l_run);
      const float inv = l_tot > 0.f ? __builtin_amdgcn_rcpf(l_tot) : 0.f;   // 1 ulp; a full division is ten instructions
      if (EXTRAS && p.nparts > 1 && cur_part == 0 && g32 == 0 && l32 < nrows)   // the row's number of parts, behind the log-sum-exps
        ((int32_t *)p.part_lse)[((int64_t)p.nparts * p.total_q + (row_begin + my_r)) * p.nhead_q + hq] = cur_parts;
      if (EXTRAS && cur_parts > 1) {
        // split over key blocks: this part's normalised result and log-sum-exp, for the merge kernel
        if (l32 < nrows) {
          const int64_t rh = ((int64_t)cur_part * p.total_q + (row_begin + my_r)) * p.nhead_q + hq;
          if (g32 == 0)   // (-inf: no key; inf: NaN, which would be left out of the merge's maximum.  Its weight there is exp(inf - inf))
            p.part_lse[rh] = l_tot > 0.f ? (m_ref + __builtin_amdgcn_logf(l_tot)) * 0.69314718055994531f : l_tot == 0.f ? -INFINITY : INFINITY;
          float *dst = p.part_out + rh * (COLS ? 8 * p.ncol : D);
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
              f32x4 w = {o[dt][4 * i4 + 0] * inv, o[dt][4 * i4 + 1] * inv, o[dt][4 * i4 + 2] * inv, o[dt][4 * i4 + 3] * inv};
              if (!COLS || 4 * dt + i4 < p.ncol) *(f32x4 *)(dst + dt * 32 + 8 * i4 + 4 * g32) = w;
            }
        }
      } else {
      if (LSE && p.lse != nullptr && g32 == 0 && l32 < nrows) {
        // natural-log sum over the row's visible keys of exp(scale * q.k); m_ref is the (possibly
        // lagging) reference maximum the row sum was accumulated under, which makes this exact
        const float lse = l_tot > 0.f ? (m_ref + __builtin_amdgcn_logf(l_tot)) * 0.69314718055994531f : -INFINITY;
        p.lse[(int64_t)(row_begin + my_r) * p.lse_s + (int64_t)hq * p.lse_h] = lse;
      }
      if constexpr (OUT32) {
        if (l32 < nrows) {
          char *orow = p.out + (int64_t)(row_begin + my_r) * p.o_s + (int64_t)hq * p.o_h;
          const float f = inv * sm_out_mul;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
              f32x4 w = {o[dt][4 * i4 + 0] * f, o[dt][4 * i4 + 1] * f, o[dt][4 * i4 + 2] * f, o[dt][4 * i4 + 3] * f};
              *(f32x4 *)(orow + (dt * 32 + 8 * i4 + 4 * g32) * 4) = w;
            }
        }
      } else {
        // A lane holds dims 8*i4 + 4*g32 .. +3 of row l32, per 32-dim block.  Two exchanges turn that
        // into 64 contiguous bytes of a row across four lanes, so that one store instruction covers
        // 16 rows instead of 32 and the memory system sees a quarter of the write requests:
        // lanes i and i+32 (same row) trade halves (16 contiguous bytes per lane), then lanes with
        // bit 4 clear / set (rows l and 16 + l) trade the two 16-dim halves of the block.
        const int l16 = lane & 15;
        int hq_x, r_x, hq_y, r_y;   // the slot's entries l16 and 16 + l16
        slot_entry(slot, l16, rows, hq_x, r_x);
        slot_entry(slot, 16 + l16, rows, hq_y, r_y);
        char *row_x = p.out + (int64_t)(row_begin + r_x) * p.o_s + (int64_t)hq_x * p.o_h + (lane & 16) * 2 + g32 * 16;
        char *row_y = PACK ? p.out + (int64_t)(row_begin + r_y) * p.o_s + (int64_t)hq_y * p.o_h + (lane & 16) * 2 + g32 * 16
                           : row_x + (int64_t)16 * p.o_s;   // (a row past the block's end is not stored)
        const bool st_x = l16 < nrows, st_y = 16 + l16 < nrows;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          u32x4 w[2];
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            const uint32_t ax = E::pack2(o[dt][8 * m + 0] * inv, o[dt][8 * m + 1] * inv);
            const uint32_t ay = E::pack2(o[dt][8 * m + 2] * inv, o[dt][8 * m + 3] * inv);
            const uint32_t bx = E::pack2(o[dt][8 * m + 4] * inv, o[dt][8 * m + 5] * inv);
            const uint32_t by = E::pack2(o[dt][8 * m + 6] * inv, o[dt][8 * m + 7] * inv);
            const auto rx = __builtin_amdgcn_permlane32_swap(ax, bx, false, false);
            const auto ry = __builtin_amdgcn_permlane32_swap(ay, by, false, false);
            w[m] = u32x4{(uint32_t)rx[0], (uint32_t)ry[0], (uint32_t)rx[1], (uint32_t)ry[1]};
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const auto r = __builtin_amdgcn_permlane16_swap(w[0][j], w[1][j], false, false);
            w[0][j] = r[0];
            w[1][j] = r[1];
          }
          const bool in = !COLS || 4 * dt + ((lane >> 4) & 1) * 2 + g32 < p.ncol;
          if (st_x && in) *(u32x4 *)(row_x + dt * 64) = w[0];
          if (st_y && in) *(u32x4 *)(row_y + dt * 64) = w[1];
        }
      }
      }
    }

    // ---- move on to the next item
    if (!ONE && total == 0) {
      // No tile, hence no barrier since this item began: the next list may still be being written,
      // and nothing of the next item has been requested yet.
      w_next_lap = -1;   // (nor has its walk been given a start: it takes no part in the clock)
      settle();
      __syncthreads();
      nxt_hk = hdr_word(c ^ 1, H_HK);
      if (nxt_hk >= 0) {
        if (hdr_word(c ^ 1, H_TOTAL) > 0) issue_first(buf, c ^ 1);
        request_q(nxt_hk, hdr_word(c ^ 1, H_SUB), hdr_word(c ^ 1, H_ROW_BEGIN), hdr_word(c ^ 1, H_ROWS));
      }
      __syncthreads();   // wave 0 rewrites this item's list next; every wave has read its header by now
    }
    if (ONE || nxt_hk < 0) break;
    c ^= 1;
  }
  if (!ONE) leave();
}

inline int persistent_grid(const void *kernel, int lds_bytes, int threads) {
  int dev = 0, cus = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, lds_bytes) != hipSuccess) return 0;
  if (per_cu < 1) return 0;
  if (per_cu > 4) per_cu = 4;
  return cus * per_cu;
}

template <int D, typename E, bool OUT32, int NW, bool EXTRAS, bool FUSED = false, bool PACK = false, bool COLS = false, bool GROUPED = false,
          bool COUNTED = false, bool ONE = false, int TEAMS = 1>
int launch_fwd_nw(const FwdParams &fp, long long items, hipStream_t stream) {
  constexpr int lds_bytes = TEAMS * 4 * (D > 128 && D <= 192 ? 32 : 64) * D * 2 + 2 * H_WORDS * 4 + 2 * kListCap * 4 + (FUSED ? 4 * kSeqCap * 4 + kMaskStage : 0);
  const void *kernel = reinterpret_cast<const void *>(&hbsa_fwd_kernel<D, E, OUT32, NW, EXTRAS, FUSED, PACK, COLS, GROUPED, COUNTED, ONE, TEAMS>);
  if (!unions_fit(fp, COUNTED) || (!EXTRAS && fp.nparts > 1)) return fail(HBSA_ERR_UNSUPPORTED, "partial results or counts that the kernel has no place for");
  // workgroups that fit the current device at once; the attribute and the occupancy are per device
  static thread_local int resident_of[kMaxDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fail(HBSA_ERR_UNSUPPORTED, "no current device, or device index above %d", kMaxDevices - 1);
  int &resident = resident_of[dev];
  if (resident == 0) {
    hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) return fail((int)e, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    resident = persistent_grid(kernel, lds_bytes, NW * TEAMS * 64);
    if (resident <= 0) return fail(HBSA_ERR_UNSUPPORTED, "could not size the persistent grid");
  }
  if constexpr (FUSED && NW == 4 && !EXTRAS && !COLS && !COUNTED && !ONE) {
    if (items <= resident) return launch_fwd_nw<D, E, false, 4, false, true, true, false, GROUPED, false, true>(fp, items, stream);
  }
  const int grid = (int)(ONE || items < resident ? items : resident);
  FwdParams launch = fp;
  // Few items per workgroup: a fixed order instead of the per-XCD queues, whose round trips (and, with few kv
  // heads, the crowd at few counters) would be a good part of such a launch.
  launch.one_each = ONE || items <= (long long)kStaticShare * resident ? (int)items : 0;
  if (launch.one_each == 0 || launch.nparts != 1 || items <= resident) launch.order = nullptr;
  hipLaunchKernelGGL((hbsa_fwd_kernel<D, E, OUT32, NW, EXTRAS, FUSED, PACK, COLS, GROUPED, COUNTED, ONE, TEAMS>), dim3(grid), dim3(NW * TEAMS * 64), lds_bytes, stream, launch);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail((int)e, "hbsa_fwd_kernel launch: %s", hipGetErrorString(e));
  return 0;
}
template <int D, typename E, bool OUT32, bool GROUPED>
int launch_fwd_tiles(const FwdParams &fp, long long items, hipStream_t stream) {
  const bool extras = fp.walk != 0 || fp.nparts > 1 || fp.lse != nullptr;
  if constexpr (D == 128) {
    if (fp.nw == 8)
      return extras ? launch_fwd_nw<D, E, OUT32, 8, true, false, false, false, GROUPED>(fp, items, stream)
                    : launch_fwd_nw<D, E, OUT32, 8, false, false, false, false, GROUPED>(fp, items, stream);
  }
  return extras ? launch_fwd_nw<D, E, OUT32, 4, true, false, false, false, GROUPED>(fp, items, stream)
                : launch_fwd_nw<D, E, OUT32, 4, false, false, false, false, GROUPED>(fp, items, stream);
}
template <int D, typename E, bool OUT32>
int launch_fwd(const FwdParams &fp, long long items, hipStream_t stream) {
  return fp.grouped ? launch_fwd_tiles<D, E, OUT32, true>(fp, items, stream) : launch_fwd_tiles<D, E, OUT32, false>(fp, items, stream);
}
// the one-launch form (16-bit tensors, none of the extras; eight wavefronts and packed slots: launch_packed_eights)
template <int D, typename E, bool GROUPED>
int launch_fused_tiles(const FwdParams &fp, long long items, hipStream_t stream) {
  if constexpr (D == 128) {
    if (fp.nw == 8) return launch_fwd_nw<D, E, false, 8, false, true, false, false, GROUPED>(fp, items, stream);
  }
  return fp.pack ? launch_fwd_nw<D, E, false, 4, false, true, true, false, GROUPED>(fp, items, stream)
                 : launch_fwd_nw<D, E, false, 4, false, true, false, false, GROUPED>(fp, items, stream);
}
template <int D, typename E>
int launch_fwd_fused(const FwdParams &fp, long long items, hipStream_t stream) {
  return fp.grouped ? launch_fused_tiles<D, E, true>(fp, items, stream) : launch_fused_tiles<D, E, false>(fp, items, stream);
}

// The one-launch form cut over key blocks: fp.nparts parts an item at most, put together by hbsa_merge_kernel.  In place of pre-pass, a bit row
// copy for each part, attention and merge: three launches, and the mask read and written once more.  Slots are packed here, which leaves
// whole workgroups of ragged q blocks without rows and so without tiles.  us, before and after, one job: 2 x 300 .. 512 queries on 65000
// keys, 32 / 8 heads of 128, 267 -> 234 (q blocks of 4 and 70 rows among them); 512 on 32000 93 -> 79; 2 x 146 .. 292 on 9000 .. 17000, 32 / 8 of
// 64, 35.5 -> 27.2; 40 .. 80 on 8000, 8 / 1 of 64, 19.3 -> 15.8; head dim 80, 4 x 2700 .. 3900 tokens, one head, 84 -> 27.
template <int D, typename E>
int launch_fwd_parts(const FwdParams &fp, long long items, hipStream_t stream) {
  if constexpr (D == 128) {
    if (fp.nw == 8)
      return fp.grouped ? launch_fwd_nw<D, E, false, 8, true, true, true, false, true>(fp, items, stream)
                        : launch_fwd_nw<D, E, false, 8, true, true, true>(fp, items, stream);
  }
  return fp.grouped ? launch_fwd_nw<D, E, false, 4, true, true, true, false, true>(fp, items, stream)
                    : launch_fwd_nw<D, E, false, 4, true, true, true>(fp, items, stream);
}

// The same on a prepared mask, where the slots are packed (plain ones: launch_fwd)
template <int D, typename E>
int launch_fwd_prepared_parts(const FwdParams &fp, long long items, hipStream_t stream) {
  if constexpr (D == 128) {
    if (fp.nw == 8)
      return fp.grouped ? launch_fwd_nw<D, E, false, 8, true, false, true, false, true>(fp, items, stream)
                        : launch_fwd_nw<D, E, false, 8, true, false, true>(fp, items, stream);
  }
  return fp.grouped ? launch_fwd_nw<D, E, false, 4, true, false, true, false, true>(fp, items, stream)
                    : launch_fwd_nw<D, E, false, 4, true, false, true>(fp, items, stream);
}

// The one-launch form, packed slots, eight wavefronts (a unit of its own: see ALIGNED in hbsattn_amd/build.py)
template <int D, typename E>
int launch_packed_eights(const FwdParams &fp, long long items, hipStream_t stream) {
  return fp.grouped ? launch_fwd_nw<D, E, false, 8, false, true, true, false, true>(fp, items, stream)
                    : launch_fwd_nw<D, E, false, 8, false, true, true>(fp, items, stream);
}

// the one-launch form that counts the blocks itself, workgroups of four wavefronts
template <int D, typename E>
int launch_fwd_counted(const FwdParams &fp, long long items, hipStream_t stream) {
  if (fp.grouped)
    return fp.pack ? launch_fwd_nw<D, E, false, 4, false, true, true, false, true, true>(fp, items, stream)
                   : launch_fwd_nw<D, E, false, 4, false, true, false, false, true, true>(fp, items, stream);
  return fp.pack ? launch_fwd_nw<D, E, false, 4, false, true, true, false, false, true>(fp, items, stream)
                 : launch_fwd_nw<D, E, false, 4, false, true, false, false, false, true>(fp, items, stream);
}

// Two teams for the tiles of an item (see fwd_teams): the one-launch form, that counts the blocks or not, and the prepared form
template <int D, typename E, bool GROUPED>
int launch_prepared_teams(const FwdParams &fp, long long items, hipStream_t stream) {
  return fp.pack ? launch_fwd_nw<D, E, false, 4, true, false, true, false, GROUPED, false, true, 2>(fp, items, stream)
                 : launch_fwd_nw<D, E, false, 4, true, false, false, false, GROUPED, false, true, 2>(fp, items, stream);
}
template <int D, typename E>
int launch_fwd_teams(const FwdParams &fp, long long items, hipStream_t stream) {
  if (fp.info != nullptr)
    return fp.grouped ? launch_prepared_teams<D, E, true>(fp, items, stream) : launch_prepared_teams<D, E, false>(fp, items, stream);
  if (fp.unions == kUnionsCounts)
    return fp.grouped ? launch_fwd_nw<D, E, false, 4, false, true, true, false, true, true, true, 2>(fp, items, stream)
                      : launch_fwd_nw<D, E, false, 4, false, true, true, false, false, true, true, 2>(fp, items, stream);
  return fp.grouped ? launch_fwd_nw<D, E, false, 4, false, true, true, false, true, false, true, 2>(fp, items, stream)
                    : launch_fwd_nw<D, E, false, 4, false, true, true, false, false, false, true, 2>(fp, items, stream);
}

// the one-launch form for tensors whose head dim (fp.ncol chunks of eight elements) is D or less
template <int D, typename E, bool PARTS, int TEAMS>
int launch_fwd_cols(const FwdParams &fp, long long items, hipStream_t stream) {
  // (a load of rows whose length is no power of two can span two groups: the lanes' offsets have to reach from one to the other)
  const bool reaches = 1024 % (2 * D) == 0 || (uint64_t)fp.wpr * 32u * (uint64_t)fp.kbs * (uint64_t)std::max(fp.k_s, fp.v_s) < (1ull << 32);
  if (fp.grouped && reaches) return launch_fwd_nw<D, E, false, 4, PARTS, true, true, true, true, false, (TEAMS > 1), TEAMS>(fp, items, stream);
  return launch_fwd_nw<D, E, false, 4, PARTS, true, true, true, false, false, (TEAMS > 1), TEAMS>(fp, items, stream);
}

}  // namespace hbsa
