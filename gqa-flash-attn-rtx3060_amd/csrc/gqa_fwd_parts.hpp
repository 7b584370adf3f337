// gqa_fwd_parts.hpp — what the two single-pass kernels (gqa_fwd.hip,
// gqa_short.hip) share: the online softmax of one 64-key tile, the instruction
// schedule of an MFMA phase, and the loads of a tile in each K/V form.
#pragma once

#include "gqa_common.hpp"
#include "gqa_lds.hpp"
#include "gqa_params.hpp"

namespace gqa {

// Work item w (XCD x takes items [x * total / 8, ...), xcd_remap) as item idx
// of the (b, kv head) pair bh: pair after pair, or, with several pairs per XCD
// (FwdParams::xcd_heads), pairs dealt to the XCDs in turn and an XCD's items
// in the order first of each pair, second of each pair, ...  Dealt, a pair's
// heavy items no longer start behind the light ones of the pair before it, and
// the sequences of a batch of unequal lengths spread over all XCDs instead of
// each filling XCDs of its own.  Measured (us, pair after pair / dealt), more
// items than CUs:
// * head_dim 64 (items handed out by the hardware as workgroups end): causal
//   3 x 2999 tokens 131 / 117, 2 x 4096 153 / 138, 8 x 700 35.7 / 30.5.
// * Paged, 512 query tokens over [1700, 5262] keys: 82 / 71, short form 80 /
//   66; [600, 5000, 2000] with 400: 122 / 74; 4 x 17000 with 382: 399 / 384.
// * Contiguous head_dim 128, causal, fixed lists: sorted heavy first over all
//   the XCD's pairs, the snake order hands every workgroup the same work;
//   pair after pair, what met what was chance.  2 x 1300 tokens 42.3 / 35.9, 2
//   x 3700 236 / 190, 3 x 900 39.7 / 29.6, 3 x 1800 109 / 84, 4 x 1300 91 / 66,
//   6 x 1300 124 / 93, 2 x 4096 231 / 227.  With many items per workgroup
//   (claimed as it goes), and key chunks: pair after pair, fewer pairs' keys
//   in each L2.
// * Many pairs per XCD (kDealPairs): nothing is shared in L2 any more.  Paged
//   head_dim 128, 34 pairs, 197 tokens over 2755 keys 358 / 418, 28 pairs 183
//   over 8184 662 / 727; contiguous 28 pairs 376 over 4341 1.20 times; head_dim
//   64 36 pairs 134 over 7635 448 / 509.  Means of dealt / pair after pair,
//   head_dim 128 with 13-24 pairs: paged, equal lengths 1.00 (22 pairs 659 over
//   689 keys 1.07), unequal 0.93 (568 tokens over 590-4076 484 / 399), contiguous
//   0.98 (14 pairs 168 tokens 26.4 / 21.7); with 25-32: 1.04, 0.96 and 1.06.
//   head_dim 64 with 25-32: 0.97, 0.94 and 0.98 (worst 295 over 10192 1.17);
//   with more, equal lengths 1.06.
// * At most one item per CU, all start together: paged head_dim 64, 13 pairs
//   21.8 / 23.5, 14 pairs 20.2 / 21.7; contiguous 10 pairs 13.0 / 14.0.  Paged
//   head_dim 128 only the spread over the XCDs counts: 8 x 200 tokens over
//   2850-26921 keys 645 / 554, 32 batches of up to 12 pairs with unequal lengths 0.96-0.99
//   in the mean, equal ones and more pairs within 1 %.
// * Key chunks, paged head_dim 128: 97 tokens of [4223, 9688] keys 49.5 / 44.7,
//   equal lengths alike; head_dim 64 35 tokens over 1981 keys 18.9 / 22.6, 127
//   over 4834 32.9 / 35.7, so pair after pair there.
// * Without a mask, contiguous, only the split blocks need it (dispatch.py
//   FWD_SPLIT_MAX_ROUNDS): head_dim 64 4 x 1025 54.8 / 55.1, 25 pairs 2194
//   tokens 954 / 1010.
// * The short form gains once its workgroups no longer start together: 4 x 300
//   tokens (320 workgroups) 16.8 / 15.8, 8 x 300 over 16/4 heads 16.3 / 14.9;
//   2 x 512 (256) 12.4 / 12.8.
__device__ inline void item_of(const FwdParams& p, int w, int n_items, int& bh, int& idx) {
  if (p.xcd_heads > 0) {
    const int x = fast_div(w, p.div_share.mul, p.div_share.shift);
    const int e = w - x * (p.xcd_heads * n_items);
    idx = fast_div(e, p.div_heads.mul, p.div_heads.shift);
    bh = (e - idx * p.xcd_heads) * 8 + x;
  } else {
    bh = fast_div(w, p.div_items.mul, p.div_items.shift);
    idx = w - bh * n_items;
  }
}

// ---------------------------------------------------------------------------
// Online softmax of one 64-key S^T tile held as two 32-key blocks (16 values
// per lane and block; the two lane halves hold the other 16 keys of the
// same row), exp2 domain.
//
// Lazy rescaling: the reference point m_ref of a row is kept as long as the
// probabilities computed against it stay at most 2^kRescaleLog2, which
// bf16/fp16 P and fp32 l/acc hold as exactly as probabilities <= 1.  A tile's
// exponentials are first computed against the current m_ref, with no row
// max; a lane's partial row sum bounds each of its probabilities, so only
// when some lane's sum exceeds 2^kRescaleLog2 (or is NaN / inf), or some row
// has no reference yet, does the wave take the tile's exact row max, raise
// m_ref to it, rescale l and the accumulators, and recompute the tile's
// exponentials.  The decision is wave-uniform, so in steady state neither a
// max tree nor the O accumulators cost VALU work.  The result o = acc / l is
// unchanged (both are relative to the same m_ref).  A row whose m_ref is
// still -inf after the exact pass (every key masked so far) uses 0 as the
// reference, so a fully masked tile contributes p = 0, never NaN.
// ---------------------------------------------------------------------------
constexpr float kRescaleSum = 256.0f;  // 2^8

// Exact pass: the tile's row max (a max3 tree), m_ref raised to it, l and the
// accumulators rescaled.  Returns -m_ref * c, the offset of the exponent.
template <int NACC>
__device__ inline float softmax_rebase(const f32x16 (&s)[2], float& m_ref, float& l_run, f32x16 (&acc)[NACC],
                                       float c) {
  float m1[11];
#pragma unroll
  for (int k = 0; k < 10; ++k) {
    const int i0 = 3 * k, i1 = 3 * k + 1, i2 = 3 * k + 2;
    m1[k] = vmax3(s[i0 >> 4][i0 & 15], s[i1 >> 4][i1 & 15], s[i2 >> 4][i2 & 15]);
  }
  m1[10] = vmax3(s[1][14], s[1][15], s[1][15]);
  const float n0 = vmax3(m1[0], m1[1], m1[2]), n1 = vmax3(m1[3], m1[4], m1[5]);
  const float n2 = vmax3(m1[6], m1[7], m1[8]), n3 = vmax3(m1[9], m1[10], m1[10]);
  const float mx = xhalf_max(vmax3(vmax3(n0, n1, n2), n3, n3));
  const float m_new = fmaxf(m_ref, mx);
  const float m_new_use = (m_new == -__builtin_inff()) ? 0.f : m_new;
  const float alpha = fast_exp2((m_ref - m_new_use) * c);
  l_run *= alpha;
#pragma unroll
  for (int db = 0; db < NACC; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[db][v] *= alpha;
  m_ref = m_new;
  return -m_new_use * c;
}

// Scores of keys a row may not see become -inf.  lim: the row's visible keys
// counted from the tile's first, less 8 for the upper lane half (its register
// v holds the key 8 past the lower half's, key_of), so that each score is
// compared with a constant.
__device__ inline void mask_tile(f32x16 (&s)[2], int lim) {
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int v = 0; v < 16; ++v) s[mb][v] = 32 * mb + key_of(v, 0) >= lim ? -__builtin_inff() : s[mb][v];
}

// One 32-key block: p = 2^(s*c - m_ref*c) in fp32, rounded to the input type
// and packed as the P^T operand; returns the fp32 row sum (a tree).
template <int DT>
__device__ inline float softmax_exp(const f32x16& s, float nmc, float c, u32x4 (&pk)[2]) {
  using E = Elem<DT>;
  float pv[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) pv[v] = fast_exp2(__builtin_fmaf(s[v], c, nmc));
  float s8[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) s8[j] = pv[2 * j] + pv[2 * j + 1];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int e = 0; e < 4; ++e) pk[kk][e] = E::pack2(pv[8 * kk + 2 * e], pv[8 * kk + 2 * e + 1]);
  return ((s8[0] + s8[1]) + (s8[2] + s8[3])) + ((s8[4] + s8[5]) + (s8[6] + s8[7]));
}

// ---------------------------------------------------------------------------
// Instruction schedule of an MFMA phase: slot j is one MFMA; the LDS reads of
// slot j + P are issued right after MFMA j (P slots ahead, to cover the LDS
// latency).  Slots [0, NRD2) are P*V MFMAs with two transposing reads each,
// the rest S^T MFMAs with one 16-byte read each.
// ---------------------------------------------------------------------------
template <int NRD2, int NSLOT, int P, int J>
__device__ __forceinline__ void mphase_prefetch() {
  if constexpr (J < P && J < NSLOT) {
    __builtin_amdgcn_sched_group_barrier(0x100, (J < NRD2) ? 2 : 1, 0);  // LDS reads
    mphase_prefetch<NRD2, NSLOT, P, J + 1>();
  }
}
template <int NRD2, int NSLOT, int P, int J>
__device__ __forceinline__ void mphase_pipe() {
  if constexpr (J < NSLOT) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
    if constexpr (J + P < NSLOT) __builtin_amdgcn_sched_group_barrier(0x100, (J + P < NRD2) ? 2 : 1, 0);
    mphase_pipe<NRD2, NSLOT, P, J + 1>();
  }
}

// ---------------------------------------------------------------------------
// Tile loads.  PG, the form of K and V: 0 contiguous; 1 a paged cache through
// the block table with pages of >= 64 keys (one buffer descriptor per 64-key
// tile, ending at the sequence's last key); 2 pages of RPI..8 keys (RPI = 512 /
// D rows per LDS-DMA instruction: each instruction's rows lie in one page, and
// every instruction gets its own descriptor); 3 pages of 16 or 32 keys (each
// wave loads 16 consecutive rows of a tile, which lie in one page: one table
// read and one descriptor per wave and tile).
// ---------------------------------------------------------------------------

// Block ids a wave needs per tile: one, or (PG 2) one per LDS-DMA instruction
// it issues.
template <int D, int PG> struct FwdTileBlocks { int id[PG == 2 ? FwdStage<D>::NI : 1]; };

// The block(s) holding tile `tile`, or wave gw's rows of it (read only for
// rows that start below key `skv`).
template <int D, int PG>
__device__ __forceinline__ FwdTileBlocks<D, PG> tile_blocks(const int* table_row, int block_shift, int skv, int tile,
                                                            int gw) {
  using ST = FwdStage<D>;
  FwdTileBlocks<D, PG> tbk;
  const int key0 = tile * ST::kKeys;
  if constexpr (PG == 2) {
#pragma unroll
    for (int j = 0; j < ST::NI; ++j) {
      const int key = key0 + (j * 4 + gw) * ST::RPI;  // first row of instruction j
      tbk.id[j] = key < skv ? load_uniform(table_row + (key >> block_shift)) : 0;
    }
  } else if constexpr (PG == 3) {
    const int key = key0 + 16 * gw;  // first of this wave's 16 rows
    tbk.id[0] = key < skv ? load_uniform(table_row + (key >> block_shift)) : 0;
  } else {
    tbk.id[0] = (PG != 0 && key0 < skv) ? load_uniform(table_row + (key0 >> block_shift)) : 0;
  }
  return tbk;
}

// Issue wave gw's (of four) share of the K or V tile `tile` into `lds`.
// Contiguous: rsrc, whose extent ends at the last row to read.  Paged: rows of
// the kv head at `head`; a descriptor starts at the tile's (wave share's,
// instruction's) first row and ends at key skv - 1, so rows past it (and whole
// tiles past it, which read no table entry) load as zeros.  off: the lane's
// offset, its row in an instruction times the row stride plus its swizzled
// chunk (FwdStage).
template <int D, int PG>
__device__ __forceinline__ void issue_fwd_tile(char* lds, const char* head, __amdgpu_buffer_rsrc_t rsrc, uint32_t rowb,
                                               uint32_t off, int64_t blk_stride, int block_shift, int skv, int tile,
                                               const FwdTileBlocks<D, PG>& blk, bool is_k, int gw, int lane) {
  using ST = FwdStage<D>;
  constexpr int CPR = ST::CPR;
  typedef __attribute__((address_space(3))) void lds_void;
  const int key0 = tile * ST::kKeys;
  if constexpr (PG == 3) {
    // This wave's rows [key, key + 16) of the tile, one run in one page:
    // instruction j loads rows key + j * RPI + 0..RPI-1 (scalar offset) into
    // LDS rows 16 gw + j * RPI + ...  Both swizzles are linear in the row
    // bits: V's depends on the lane's row lrow alone (off as given); K's
    // chunk is (lane % CPR) ^ gk(lrow) ^ gk(j * RPI).
    const int key = key0 + 16 * gw;
    const int rows = skv - key;
    __amdgpu_buffer_rsrc_t rt = make_rsrc(head, 0u);
    if (rows > 0) {
      const char* base =
          head + 2 * ((int64_t)blk.id[0] * blk_stride + (int64_t)(key & ((1 << block_shift) - 1)) * (rowb >> 1));
      rt = make_rsrc(base, (uint32_t)(min(rows, 16) - 1) * rowb + 2 * D);
    }
    if constexpr (D == 64) {
      // Derived from `off` (the lane's offset for LDS rows gw * RPI + lr),
      // so no offsets of their own stay live across the loop: sv depends
      // on lr alone, so V's is `off` for both instructions; gk(gw * RPI +
      // lr) = gk(lr) ^ gk(8 (gw & 1)) with gk(8) = 2, so K's is `off` for
      // instruction j = gw & 1 and `off` with chunk bit 1 flipped (byte
      // offset ^ 32, as lr * rowb is a multiple of 64: the host takes
      // this path only for such row strides) for the other.
      // The empty asm keeps the XOR here: hoisted out of the tile loop, its
      // result would hold a register across the loop.
      uint32_t flip = off;
      if (is_k) {
        asm volatile("" : "+v"(flip));
        flip ^= 32u;
      }
      const uint32_t other = flip;
#pragma unroll
      for (int j = 0; j < ST::NI; ++j) {
        const uint32_t o = (j == (gw & 1)) ? off : other;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rt, (lds_void*)(lds + (gw * ST::NI + j) * 1024), 16, o,
                                                 (uint32_t)(j * ST::RPI) * rowb, 0, 0);
      }
    } else {
      const int lr = lane / CPR, lc = lane % CPR;
#pragma unroll
      for (int j = 0; j < ST::NI; ++j) {
        const int sw = is_k ? (ST::gk(lr) ^ ST::gk(j * ST::RPI)) : ST::sv(lr);
        const uint32_t o = (uint32_t)(lr * rowb) + 16u * (uint32_t)(lc ^ sw);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rt, (lds_void*)(lds + (gw * ST::NI + j) * 1024), 16, o,
                                                 (uint32_t)(j * ST::RPI) * rowb, 0, 0);
      }
    }
  } else if constexpr (PG == 2) {
    // Instruction j loads rows [key, key + RPI) of the tile, one run in
    // one page (key is a multiple of RPI and pages hold >= RPI keys); its
    // descriptor ends at the sequence's last key.
#pragma unroll
    for (int j = 0; j < ST::NI; ++j) {
      const int step = j * 4 + gw;
      const int key = key0 + step * ST::RPI;
      const int rows = skv - key;
      __amdgpu_buffer_rsrc_t rt = make_rsrc(head, 0u);
      if (rows > 0) {
        const char* base =
            head + 2 * ((int64_t)blk.id[j] * blk_stride + (int64_t)(key & ((1 << block_shift) - 1)) * (rowb >> 1));
        rt = make_rsrc(base, (uint32_t)(min(rows, ST::RPI) - 1) * rowb + 2 * D);
      }
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rt, (lds_void*)(lds + step * 1024), 16, off, 0, 0, 0);
    }
  } else if constexpr (PG == 1) {
    const int rows = skv - key0;
    __amdgpu_buffer_rsrc_t rt = make_rsrc(head, 0u);
    if (rows > 0) {
      const char* base =
          head + 2 * ((int64_t)blk.id[0] * blk_stride + (int64_t)(key0 & ((1 << block_shift) - 1)) * (rowb >> 1));
      rt = make_rsrc(base, (uint32_t)(min(rows, ST::kKeys) - 1) * rowb + 2 * D);
    }
    issue_tile_dma<D>(lds, rt, 0u, rowb, off, gw);
  } else {
    issue_tile_dma<D>(lds, rsrc, (uint32_t)key0 * rowb, rowb, off, gw);
  }
}

}  // namespace gqa
