// The attention kernel of the forward for fp32 operands (fp32 matrix instructions), and its launch function.
#pragma once

#include "hbsa_common.h"

namespace hbsa {

// --------------------------------------------------------------------------------------
// fp32 kernel: fp32 operands, fp32 MFMA (v_mfma_f32_32x32x2_f32), fp32 softmax and output, for
// callers that need the arithmetic of the reference's fp32 path (dot products without operand
// rounding, reference hbsattn/fwd_triton_auto_tile_size.py:205,225).
//
// What bounds it: the fp32 matrix rate, a sixteenth of the bf16 one (a 32x32x2 product occupies a SIMD for 64 cycles; the
// softmax of 32 keys is a few hundred cycles beside 4096 of products at D = 64), as long as operands arrive in time and
// every CU has as much work as the next.  So: tiles go from memory straight into LDS, one tile ahead; an operand read from
// LDS feeds four products; and an item (kv head, q block, group of four wave slots) is cut into parts over its k blocks when
// there are few items (ItemParts), because a causal mask over ragged sequences makes the longest item several times the
// average and all of them are resident from the start.  4 sequences of 1279 .. 2697 tokens, 8 / 4 heads of 64, keep 0.5,
// causal: 200 us with single-buffered tiles through registers and whole items, 117 now (73 TFLOP/s; 98 on uniform lengths,
// where the matrix pipeline is busy 82 % of the time).
//
// Same operand roles as the 16-bit kernel: S^T = K.Q^T with K rows from LDS and Q^T in registers,
// O^T += V^T.P^T with P^T taken from the S^T accumulator in place.  A 32x32x2 MFMA contracts over
// two indices, one per half of the wavefront; which two is free as long as both operands agree:
//   S: step (j, e), half g contracts over d = 8*j + 4*g + e, so a lane reads 4 consecutive floats of
//      its K row per j (one ds_read_b128) and holds Q the same way;
//   PV: step i, half g contracts over key 8*(i/4) + 4*g + (i%4), which is exactly the key whose
//      score the lane holds in accumulator element i.  The 32 rows of the product that fills accumulator dt are the
//      head dims W * m + dt (m the row, W = 4 at D = 128), so a lane's W consecutive floats of a V row serve W products.
// Tiles are KT keys in groups of 16, each group from any place of the sequence (blocks are multiples of 16 keys): blocks
// of 16 or 48 keys fill tiles like larger ones.
// LDS: K tiles with chunk c (16 bytes) of row r at c ^ (r's place in the bank sweep), V tiles as they come.
// --------------------------------------------------------------------------------------
template <int D>
struct F32Tile {
  static constexpr int RB = D * 4;                 // row bytes
  static constexpr int CPR = RB / 16;              // 16-byte chunks per row
  static constexpr int RPG = 16 / CPR > 0 ? 16 / CPR : 1;
  static constexpr int KT = D <= 32 ? 64 : 32;     // keys per tile
  static constexpr int GROUPS = KT / 16;
  static constexpr int TILE_BYTES = KT * RB;
  static constexpr int W = D >= 128 ? 4 : D / 32;  // floats of a V row per lane and read
  static constexpr int VR = D / 32 / W;            // such reads per row
  static constexpr int LDS_BYTES = 4 * TILE_BYTES;
  static constexpr int WG_PER_CU = D >= 256 ? 1 : D >= 128 ? 2 : 3;
  static __device__ __forceinline__ int swz(int r) { return (r / RPG) % CPR; }
};

template <int D>
__global__ __launch_bounds__(kThreads, F32Tile<D>::WG_PER_CU) void hbsa_fwd_f32_kernel(FwdParams p, float c_signed) {
  using T = F32Tile<D>;
  constexpr int RB = T::RB, CPR = T::CPR, KT = T::KT, GROUPS = T::GROUPS;
  constexpr int DJ = D / 8;       // ds_read_b128 steps of S
  constexpr int DT = D / 32;      // accumulators of O^T
  constexpr int LOADS = KT * CPR / kThreads;   // 16-byte loads per lane, tile and operand
  constexpr int RPL = 64 / CPR;                // rows one load of a wavefront covers (1 .. 8: inside one group)
  static_assert(LOADS >= 1 && RPL >= 1 && RPL <= 16, "a load stays inside a group of 16 keys");
  extern __shared__ __attribute__((aligned(1024))) char lds[];   // K[2] tiles, V[2] tiles
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

  // Q^T fragments, pre-multiplied by softmax_scale * log2(e): scores come out in log2 units
  f32x4 qf[DJ];
  {
    const char *qrow = p.q + (int64_t)(inf.row_begin + row) * p.q_s + (int64_t)hq * p.q_h;
#pragma unroll
    for (int j = 0; j < DJ; ++j) {
      f32x4 x = {0.f, 0.f, 0.f, 0.f};
      if (active) x = *(const f32x4 *)(qrow + (8 * j + 4 * g32) * 4);
      qf[j] = x * c_signed;
    }
  }
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
  int win = blk_begin;                                     // blocks win .. win + 63 are in `kept`
  uint64_t kept = KeptWindow::vote(window.load(win, blk_end));
  uint32_t ahead = window.load(win + 64, blk_end);         // the next window, on its way
  int blk = -1, off = 0;                                   // current block, position of its next group
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

  // ---- tile loads: load i of wavefront w covers rows RPL * (4 * i + w) .. + RPL - 1
  const uint32_t lds_base = (uint32_t)(uintptr_t)HBSA_AS3(lds) + (uint32_t)wave * 1024u;
  const int ld_row = RPL * wave + lane / CPR;
  const uint32_t k_s32 = (uint32_t)p.k_s, v_s32 = (uint32_t)p.v_s;   // row strides in bytes (the host checks they fit)
  auto dma16 = [&](uint32_t dst, const char *sbase, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(dst), "v"(voff), "s"(sbase) : "memory", "m0");
  };
  auto fetch = [&](int buf, const Tile &tl) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int r = ld_row + 4 * RPL * i;                           // row of the tile
      const int g = __builtin_amdgcn_readfirstlane((RPL * (4 * i + wave)) >> 4);
      int pos = tl.pos[0], valid = tl.valid[0];
#pragma unroll
      for (int x = 1; x < GROUPS; ++x) {
        pos = g == x ? tl.pos[x] : pos;
        valid = g == x ? tl.valid[x] : valid;
      }
      const int in_group = min(r & 15, max(valid, 1) - 1);          // rows past the end repeat the last one (masked below)
      const uint32_t dst = lds_base + (uint32_t)(buf * T::TILE_BYTES + i * 4096);
      dma16(dst, kg + (int64_t)pos * p.k_s, (uint32_t)in_group * k_s32 + (uint32_t)(((lane % CPR) ^ T::swz(r)) * 16));
      dma16(dst + 2 * T::TILE_BYTES, vg + (int64_t)pos * p.v_s, (uint32_t)in_group * v_s32 + (uint32_t)((lane % CPR) * 16));
    }
  };

  Tile cur;
  next_tile(cur);
  int buf = 0;
  if (cur.any) fetch(0, cur);
  while (cur.any) {
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this wavefront's part of the tile has landed
    __syncthreads();                      // ... every wavefront's, and the other buffers have been read by all
    Tile nxt;
    next_tile(nxt);
    if (nxt.any) fetch(buf ^ 1, nxt);
    const float *kt = (const float *)(lds + buf * T::TILE_BYTES), *vt = (const float *)(lds + (2 + buf) * T::TILE_BYTES);
    if (active) {
#pragma unroll
      for (int h = 0; h < KT / 32; ++h) {   // ---- 32 keys at a time
        const int pos0 = cur.pos[2 * h], pos1 = cur.pos[2 * h + 1], valid0 = cur.valid[2 * h], valid1 = cur.valid[2 * h + 1];
        if (valid0 <= 0 || (p.causal && pos0 > wave_kvis_max)) continue;
        f32x16 sc;
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] = 0.f;
        const float *krow = kt + (32 * h + l32) * D;
        const int swz = T::swz(l32);   // (the same for rows 32 apart)
#pragma unroll
        for (int jj = 0; jj < DJ; ++jj) {
          const f32x4 kv = *(const f32x4 *)(krow + (((2 * jj + g32) ^ swz) << 2));
#pragma unroll
          for (int e = 0; e < 4; ++e) sc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[e], qf[jj][e], sc, 0, 0, 0);
        }
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
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float *vrow = vt + (32 * h + 8 * (i >> 2) + 4 * g32 + (i & 3)) * D + T::W * l32;
#pragma unroll
          for (int vr = 0; vr < T::VR; ++vr) {
            float a[T::W];
            if constexpr (T::W == 4) {
              const f32x4 x = *(const f32x4 *)(vrow + 128 * vr);
              a[0] = x[0]; a[1] = x[1]; a[2] = x[2]; a[3] = x[3];
            } else if constexpr (T::W == 2) {
              const float2 x = *(const float2 *)vrow;
              a[0] = x.x; a[1] = x.y;
            } else {
              a[0] = *vrow;
            }
#pragma unroll
            for (int w = 0; w < T::W; ++w)
              o[vr * T::W + w] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[w], sc[i], o[vr * T::W + w], 0, 0, 0);
          }
        }
      }
    }
    buf ^= 1;
    cur = nxt;
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
  for (int vr = 0; vr < T::VR; ++vr)
#pragma unroll
    for (int i = 0; i < 16; ++i) {   // accumulator element i holds row m of the products: head dims W * m .. + W - 1
      const int m = 8 * (i >> 2) + 4 * g32 + (i & 3);
      float *dst = (float *)(orow + (128 * vr + T::W * m) * 4);
      if constexpr (T::W == 4) *(f32x4 *)dst = f32x4{o[4 * vr][i] * inv, o[4 * vr + 1][i] * inv, o[4 * vr + 2][i] * inv, o[4 * vr + 3][i] * inv};
      else if constexpr (T::W == 2) *(float2 *)dst = float2{o[0][i] * inv, o[1][i] * inv};
      else *dst = o[0][i] * inv;
    }
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
