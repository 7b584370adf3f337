// gqa_fwd.hip — single-pass group-packed GQA forward for gfx950.
//
// Replaces the Triton kernel gqa_fwd_kernel (reference
// gqa_kernels/gqa_fwd.py:33-109).  One workgroup = 8 waves = 256 packed query
// rows of ONE (batch, kv head): G query heads x block_m positions (row r ->
// head r / block_m, position r % block_m, as gqa_fwd.py:58-63), so each K/V
// tile staged in LDS feeds the whole query group.  Per 64-key tile and wave
// (32 rows):
//   S^T = K Q^T        (bf16/f16 MFMA 32x32x16, fp32 accumulate)
//   online softmax     (exp2 domain, scale applied in fp32, gqa_fwd.py:98-101)
//   O^T += V^T P^T     (P rounded to the input type, gqa_fwd.py:103)
// Causal: the key loop stops at the workgroup's last visible key
// (gqa_fwd.py:70-73) and masks only the tiles that cross the diagonal or the
// end of the keys.
//
// Schedule ("ping-pong").  The waves form two groups of four, A = waves 0-3
// and B = waves 4-7; wave w and wave w+4 share a SIMD.  Work alternates
// between MFMA phases (the P*V product of the previous tile and S^T of the
// current one: 32 MFMAs per wave) and softmax phases (VALU only), and the two
// groups run one phase apart, separated by workgroup barriers: while one
// group's MFMAs occupy the matrix core of a SIMD, the other group's softmax
// runs on the same SIMD's vector ALU.
//
//   phase:   0       1       2       3       4     ...
//   A:     S(0)    sm(0)   PV(0)   sm(1)   PV(1)
//                          +S(1)           +S(2)
//   B:     (idle)  S(0)    sm(0)   PV(0)   sm(1)
//                                  +S(1)
//
// K and V tiles are both loaded straight into LDS (buffer loads in their
// LDS-DMA form) through a ring of three stages; stage t holds K(t) and
// V(t-1), the operands of MFMA phase t.  Each softmax phase issues the loads
// two tiles ahead (group A: K, group B: V) and waits for the ones issued one
// softmax phase earlier, so a load has two phases to land and the ring never
// overwrites a stage that is still read.
#include <algorithm>
#include <type_traits>

#include "gqa_common.hpp"
#include "gqa_fwd_parts.hpp"
#include "gqa_lds.hpp"
#include "gqa_params.hpp"

namespace gqa {

// PG: the form of K and V (gqa_fwd_parts.hpp).
// D = 64 keeps to 128 VGPRs (four waves per SIMD): two workgroups share a
// compute unit, which outweighs the shorter LDS-read lookahead it needs.
//
// Contiguous K/V at D = 128 (one workgroup per compute unit) runs
// persistent: p.n_wg workgroups each work through a list of items (below),
// and an item's start overlaps the previous item's end: as soon as the
// finished item's output has left the LDS stages, the workgroup issues the
// next item's first K/V tiles and Q, and the output stores drain while
// those loads are in flight.  The workgroup launch between items leaves the
// critical path.
// KC: key chunks (FwdParams::kv_splits > 0), a separate instance so the
// others keep their registers.
template <int DT, int D, int PG, bool KC = false>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(D == 64 ? 4 : 2))) void gqa_fwd_kernel(
    FwdParams p) {
  using E = Elem<DT>;
  using T = typename E::T;
  using ST = FwdStage<D>;
  constexpr int CPR = ST::CPR;
  constexpr bool PAGED = PG != 0;
  constexpr bool PERSIST = PG == 0 && D == 128;
  using TileBlocks = FwdTileBlocks<D, PG>;
  constexpr int NDB = D / 32;  // 32-wide d blocks of O^T
  constexpr int NKS = D / 16;  // k-steps of S^T
  constexpr int PF = (D == 64) ? 3 : 6;  // MFMA slots of LDS-read lookahead
  // Six separate arrays (not one): the compiler can then tell the LDS-DMA
  // targets of later tiles from the buffers being read, and does not wait for
  // those loads before the reads.
  // The V stages take the low 48 KiB: an MFMA phase reads V with twice as
  // many LDS instructions as K, and below 64 KiB a stage's address fits the
  // 16-bit offset field of ds_read, so those reads need no VALU address
  // arithmetic (which would compete with the other wave's softmax on the
  // SIMD).  The compiler lays kernel LDS variables out in name order.
  __shared__ __attribute__((aligned(1024))) char lds0_v0[ST::kTileBytes];
  __shared__ __attribute__((aligned(1024))) char lds0_v1[ST::kTileBytes];
  __shared__ __attribute__((aligned(1024))) char lds0_v2[ST::kTileBytes];
  __shared__ __attribute__((aligned(1024))) char lds1_k0[ST::kTileBytes];
  __shared__ __attribute__((aligned(1024))) char lds1_k1[ST::kTileBytes];
  __shared__ __attribute__((aligned(1024))) char lds1_k2[ST::kTileBytes];
  __shared__ int s_last;

  const Dims& dm = p.dm;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6) & 7;  // wave-uniform (SGPR)
  const int grp = wave >> 2;                                     // 0: group A, 1: group B
  const int gw = wave & 3;                                       // wave index in its group
  const int i = lane & 31, hh = lane >> 5;
  const bool varlen = p.q_len != nullptr;

  // Work items: heavy (late) query blocks first under causal, and every XCD
  // gets a contiguous range of items (same kv head -> same L2).  With a key
  // split, the n_split heaviest blocks of each (b, kv head) come as two
  // items: first the upper halves of their key ranges, then (in the usual
  // order) the lower halves and the unsplit blocks.  Without a mask all
  // blocks are as long and the halves fill the last round: the unsplit
  // blocks, then the upper and the lower halves of the last n_split.
  // Key chunks: kv_splits items per query block, the blocks of one chunk
  // consecutive (they read the same keys).
  constexpr bool chunked = KC;
  const int n_items = chunked ? p.n_mblk * p.kv_splits : p.n_mblk + p.n_split;
  const int total = n_items * dm.Hkv * dm.B;
  // The k-th item of this workgroup (-1: none).  One item per workgroup
  // (xcd_remap), or persistent: the workgroups of XCD x (hardware ids x,
  // x + 8, ...) take the XCD's item range round by round in snake order
  // (round j: slot c takes item j*S + c, or j*S + S-1-c in odd rounds), so
  // the heavy-first order hands every slot a mix of heavy and light items.
  const int n_wg = PERSIST ? p.n_wg : total;
  // Item range of XCD x: [lo, lo + n), served by its S workgroups.
  auto xrange = [&](int x, int& lo, int& n, int& S) {
    S = (n_wg - x + 7) >> 3;
    const int q = total >> 3, r = total & 7;
    lo = x * q + min(x, r);
    n = q + (x < r ? 1 : 0);
  };
  auto item_at = [&](int k) -> int {
    if (!PERSIST) return k == 0 ? xcd_remap(blockIdx.x, total) : -1;
    const int x = blockIdx.x & 7, slot = blockIdx.x >> 3;
    int lo, n, S;
    xrange(x, lo, n, S);
    const int j = k;
    const int e = j * S + ((j & 1) ? S - 1 - slot : slot);
    return e < n ? lo + e : -1;
  };
  // Dynamic schedule (persistent kernel, p.sched set): the XCDs run at
  // different speeds under sustained MFMA load (their workgroups end up to
  // 6 % apart on a static schedule), so after its first item (slot c of XCD
  // x takes item c of x's range, as above) a workgroup claims the next one
  // from its own XCD's queue — items S, S + 1, ... of the range, heavy
  // first — and, once that is empty, from the other XCDs' queues.  One
  // thread claims with an agent-scope atomic issued as the epilogue begins
  // and resolves it after the output stores, so its latency is hidden.
  // Items are independent (a split block's halves merge in a fixed order),
  // so the outputs do not depend on who computes what.  p.sched: 8 queue
  // counters, 8 + 1 counts of workgroups done, zero on entry; the last
  // workgroup to finish leaves them zero.  The counters' address waits in
  // LDS (kept in registers, it would add to those held across the tile
  // loop).
  __shared__ int s_next;
  __shared__ int* s_sched;
  if (PERSIST && t == 0) s_sched = p.sched;

  // One work item's parameters.
  struct Item {
    int b, kvh, bh, pid_m, part;  // part: -1 whole key range, 0 lower half, 1 upper half
    int skv, sq, tb, ntiles, qpos_lo;
    int64_t tok0;
    int pos, head, vis;  // this lane's query row; the keys it sees, as mask_tile counts them
    bool valid;
    const char* kbh;
    const char* vbh;
    __amdgpu_buffer_rsrc_t rk, rv;
    const int* table_row;
  };
  const uint32_t kssb = (uint32_t)(2 * p.k.ss), vssb = (uint32_t)(2 * p.v.ss);
  auto decode = [&](int w, int i, int block_m) __attribute__((always_inline)) -> Item {
    Item x;
    int idx;
    item_of(p, w, n_items, x.bh, idx);
    int chunk = 0;
    if constexpr (chunked) {
      chunk = fast_div(idx, p.div_mblk.mul, p.div_mblk.shift);
      idx -= chunk * p.n_mblk;
    }
    const int up = idx - (dm.causal ? 0 : p.n_mblk - p.n_split);  // place among the upper halves
    if (up >= 0 && up < p.n_split) {
      x.pid_m = p.n_mblk - 1 - up;
      x.part = 1;
    } else {
      const int mrank = up < 0 ? idx : idx - p.n_split;
      x.pid_m = dm.causal ? (p.n_mblk - 1 - mrank) : mrank;
      x.part = (x.pid_m >= p.n_mblk - p.n_split) ? 0 : -1;
    }
    x.b = fast_div(x.bh, p.div_hkv.mul, p.div_hkv.shift);
    x.kvh = x.bh - x.b * dm.Hkv;
    // Keys of this sequence (paged: its own length, clamped to [0, Skv]),
    // and its query rows (variable lengths: q_len[b], tokens from q_start[b]).
    x.skv = PAGED ? min(max(load_uniform(p.seq_lens + x.b), 0), dm.Skv) : dm.Skv;
    x.sq = varlen ? min(max(load_uniform(p.q_len + x.b), 0), dm.Sq) : dm.Sq;
    x.tok0 = varlen ? (int64_t)load_uniform(p.q_start + x.b) : 0;
    // This lane's query row.
    const int r = wave * 32 + i;
    const int g = (int)(__umul24(r, p.bm_mul) >> 16), ml = r - g * block_m;
    x.pos = x.pid_m * block_m + ml;
    x.valid = (g < dm.G) && (x.pos < x.sq);
    x.head = x.kvh * dm.G + (g < dm.G ? g : 0);
    x.vis = (dm.causal ? min(x.skv, x.pos + (x.skv - x.sq) + 1) : x.skv) - 8 * hh;
    // Key range of this item: tiles [tb, tb + ntiles).
    const int pos_lo = x.pid_m * block_m;
    const int pos_hi = min(pos_lo + block_m, x.sq) - 1;
    int kv_end = x.skv;
    if (dm.causal) kv_end = min(x.skv, pos_hi + (x.skv - x.sq) + 1);
    kv_end = max(kv_end, 0);
    const int ntiles_all = (kv_end + ST::kKeys - 1) / ST::kKeys;
    const int tsplit = ntiles_all >> 1;
    x.tb = (x.part == 1) ? tsplit : 0;
    x.ntiles = (x.part == 0) ? tsplit : ntiles_all - x.tb;
    if constexpr (chunked) {
      // Tiles [chunk * ct, (chunk + 1) * ct) of the block's range (none
      // for a chunk past it: an empty partial).
      x.tb = chunk * p.kv_chunk_tiles;
      x.ntiles = max(min(ntiles_all - x.tb, p.kv_chunk_tiles), 0);
    }
    x.qpos_lo = pos_lo + (x.skv - x.sq);
    // Global side: buffer descriptors over this (b, kv head)'s K and V rows,
    // each ending at the last byte of row seq_kv - 1.  The host guarantees
    // (seq_kv + 192) * row stride * 2 < 2^31, so every offset (up to two
    // tiles past the end) fits 32 bits.  (An empty key range gets an empty
    // descriptor: every load reads zero.)
    x.kbh = static_cast<const char*>(p.k.ptr) + 2 * ((PAGED ? 0 : (int64_t)x.b * p.k.sb) + (int64_t)x.kvh * p.k.sh);
    x.vbh = static_cast<const char*>(p.v.ptr) + 2 * ((PAGED ? 0 : (int64_t)x.b * p.v.sb) + (int64_t)x.kvh * p.v.sh);
    const bool flat = !PAGED && dm.Skv > 0;
    x.rk = make_rsrc(x.kbh, flat ? (uint32_t)(dm.Skv - 1) * kssb + 2 * D : 0u);
    x.rv = make_rsrc(x.vbh, flat ? (uint32_t)(dm.Skv - 1) * vssb + 2 * D : 0u);
    x.table_row = PAGED ? p.block_table + (int64_t)x.b * p.table_stride : nullptr;
    return x;
  };

  int k_item = 0;
  Item it = decode(item_at(0), i, p.block_m);
  if (!PERSIST && it.pid_m * p.block_m >= it.sq) return;  // a block past this sequence's queries (variable lengths)
  // Element offset of (query row pos, head h) in q / o.
  auto row_off = [&](const Item& x, const TensorRef& tr, int pos_, int h) -> int64_t {
    return varlen ? (x.tok0 + pos_) * tr.ss + (int64_t)h * tr.sh
                  : (int64_t)x.b * tr.sb + (int64_t)h * tr.sh + (int64_t)pos_ * tr.ss;
  };

  const int lrow = lane / CPR;
  const uint32_t koff =
      (uint32_t)(lrow * kssb) + 16u * (uint32_t)((lane % CPR) ^ ST::gk((gw * ST::RPI + lrow) & 15));
  const uint32_t voff = (uint32_t)(lrow * vssb) + 16u * (uint32_t)((lane % CPR) ^ ST::sv(lrow));

  // Issue this wave's share of K or V tile `tile` (absolute index) into LDS
  // (gqa_fwd_parts.hpp).  The softmax phases use block ids read one phase
  // ahead (blk_next), so the table reads' latency is off the issue path.
  auto tile_block = [&](const Item& x, int tile) __attribute__((always_inline)) -> TileBlocks {
    return tile_blocks<D, PG>(x.table_row, p.block_shift, x.skv, tile, gw);
  };
  auto issue_tile = [&](const Item& x, char* lds, const char* head, __amdgpu_buffer_rsrc_t rsrc, uint32_t rowb,
                        uint32_t off, int64_t blk_stride, int tile, const TileBlocks& blk, bool is_k)
                        __attribute__((always_inline)) {
    issue_fwd_tile<D, PG>(lds, head, rsrc, rowb, off, blk_stride, p.block_shift, x.skv, tile, blk, is_k, gw, lane);
  };
  auto issue_k = [&](const Item& x, char* lds, int tile, const TileBlocks& blk) {
    issue_tile(x, lds, x.kbh, x.rk, kssb, koff, p.k.sb, tile, blk, true);
  };
  auto issue_v = [&](const Item& x, char* lds, int tile, const TileBlocks& blk) {
    issue_tile(x, lds, x.vbh, x.rv, vssb, voff, p.v.sb, tile, blk, false);
  };

  // LDS side: per-lane read offsets (the 32-key block, chunk and row offsets
  // of each read are immediates on top of these).  The masks are no-ops on
  // the values; they give the compiler known bounds.
  constexpr uint32_t kKMask = (ST::kTileBytes / 2 - 1) & ~15u;
  constexpr uint32_t kVMask = (ST::kTileBytes - 1) & ~7u;
  uint32_t ka[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks)
    ka[ks] = (uint32_t)(pi_key(i) * (2 * D) + 16 * ((2 * ks + hh) ^ ST::gk(pi_key(i)))) & kKMask;
  // At D = 128, K stages 1 and 2 lie above 64 KiB, out of reach of
  // ds_read's 16-bit offset field.  Their reads address from kah = ka + the
  // LDS address of stage 1, kept in registers (refreshed as opaque values in
  // every MFMA phase, so the compiler neither folds them back into ka nor
  // recomputes them): the stage and block offsets stay immediates, and the
  // reads need no VALU address arithmetic beside the other wave's softmax.
  // (At D = 64 every stage lies below 64 KiB.)
  constexpr bool kHighK = 6 * ST::kTileBytes > 65536;
  const uint32_t k1base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds1_k1;
  uint32_t kah[kHighK ? NKS : 1];
#pragma unroll
  for (int ks = 0; ks < (kHighK ? NKS : 1); ++ks) kah[ks] = ka[ks] + k1base;
  uint32_t vb[NDB];
  {
    const int q = lane >> 4, ii = lane & 15;                  // 16-lane group, lane in group
    const int rowl = 8 * (q >> 1) + (ii >> 2);                // key row addressed by this lane
    const int f = (CPR == 16) ? (ii >> 2) : ((ii >> 3) & 1);  // sv(rowl) / 4
#pragma unroll
    for (int db = 0; db < NDB; ++db)
      vb[db] = (uint32_t)(rowl * (2 * D) + 16 * (4 * (db ^ f) + 2 * (q & 1) + ((ii & 3) >> 1)) + 8 * (ii & 1)) &
               kVMask;
  }

  f32x16 acc[NDB];
  float m_run, l_run;
  const float c = dm.c;
  f32x16 sc[2];    // S^T of the current tile (MFMA phase -> softmax phase)
  u32x4 pk[2][2];  // P^T operands (softmax phase -> next MFMA phase)
  u32x4 qreg[NKS];

  auto kstage = [&](auto s3) -> char* {
    constexpr int S3 = decltype(s3)::value;
    return S3 == 0 ? lds1_k0 : (S3 == 1 ? lds1_k1 : lds1_k2);
  };
  auto vstage = [&](auto s3) -> char* {
    constexpr int S3 = decltype(s3)::value;
    return S3 == 0 ? lds0_v0 : (S3 == 1 ? lds0_v1 : lds0_v2);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using BT = std::true_type;
  using BF = std::false_type;

  // Prologue loads of item x: stage 0 = K(0), stage 1 = K(1) + V(0), and V(1)
  // of stage 2 (tile indices relative to tb), then Q.  The tile loads go
  // first: the Q loads behind them touch 32 rows per instruction and, issued
  // first, held the tile loads back by ~2 us.  An invalid row loads row 0 of
  // its sequence (always present here); it is zeroed once the loads have
  // landed, so that they are all in flight together (a select beside each load
  // made the compiler wait for every one of the eight in turn: 1.9-2.4 us per
  // launch).  Paged: returns the block(s) of the tile the first softmax phase
  // issues.  (Q in whole rows through LDS, as gqa_short.hip loads it, left
  // 2048 tokens at 42.2 us and 16384 0.6 % slower here.)
  auto prologue_q = [&](const Item& x) __attribute__((always_inline)) {
    const T* qrow = static_cast<const T*>(p.q.ptr) + row_off(x, p.q, x.valid ? x.pos : 0, x.head);
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qreg[ks] = *reinterpret_cast<const u32x4*>(qrow + 16 * ks + 8 * hh);
  };
  auto prologue_kv = [&](const Item& x) __attribute__((always_inline)) -> TileBlocks {
    TileBlocks bn = tile_block(x, x.tb);
    if (grp == 0) {
      issue_k(x, lds1_k0, x.tb, bn);
    } else {
      issue_v(x, lds0_v1, x.tb, bn);
    }
    bn = tile_block(x, x.tb + 1);
    if (grp == 0) {
      issue_k(x, lds1_k1, x.tb + 1, bn);
    } else {
      issue_v(x, lds0_v2, x.tb + 1, bn);
    }
    bn = tile_block(x, x.tb + 2);
    return bn;
  };
  TileBlocks blk_next = prologue_kv(it);
  prologue_q(it);

  // MFMA phase of tile tt: P*V of tile tt-1 and S^T of tile tt, from ring
  // slot s3 = tt % 3.
  auto mphase = [&](auto s3, auto pvc, auto sc_) {
    constexpr bool DO_PV = decltype(pvc)::value;
    constexpr bool DO_S = decltype(sc_)::value;
    constexpr int NPV = DO_PV ? 4 * NDB : 0;
    constexpr int NS = DO_S ? 2 * NKS : 0;
    const char* ck = kstage(s3);
    const char* cv = vstage(s3);
    // Issue priority: the MFMA-phase wave of a SIMD first (its MFMA stream is
    // the matrix core's only work), the softmax wave in the gaps (~+2 %).
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(3);
    __builtin_amdgcn_sched_barrier(0);
    u32x4 opv[NPV > 0 ? NPV : 1];
    u32x4 opk[NS > 0 ? NS : 1];
    if constexpr (DO_PV) {
#pragma unroll
      for (int j = 0; j < NPV; ++j) {
        const int mb = j / (2 * NDB), kk = (j / NDB) & 1, db = j % NDB;
        const int ro = (32 * mb + 16 * kk) * (2 * D);
        const u32x2 lo = ld_tr(cv + vb[db] + ro);
        const u32x2 hi = ld_tr(cv + vb[db] + ro + 4 * (2 * D));
        opv[j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
    }
    if constexpr (DO_S) {
      if constexpr (decltype(s3)::value == 0 || !kHighK) {
#pragma unroll
        for (int j = 0; j < NS; ++j) opk[j] = *reinterpret_cast<const u32x4*>(ck + (j & 1) * 32 * (2 * D) + ka[j >> 1]);
      } else {
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) asm volatile("" : "+v"(kah[ks]));
#pragma unroll
        for (int j = 0; j < NS; ++j)
          opk[j] = *reinterpret_cast<const u32x4*>(ck + (j & 1) * 32 * (2 * D) + (kah[j >> 1] - k1base));
      }
    }
    if constexpr (DO_PV) {
#pragma unroll
      for (int j = 0; j < NPV; ++j) {
        const int mb = j / (2 * NDB), kk = (j / NDB) & 1, db = j % NDB;
        acc[db] = E::mfma(opv[j], pk[mb][kk], acc[db]);
      }
    }
    if constexpr (DO_S) {
      sc[0] = f32x16{};
      sc[1] = f32x16{};
#pragma unroll
      for (int j = 0; j < NS; ++j) sc[j & 1] = E::mfma(opk[j], qreg[j >> 1], sc[j & 1]);
    }
    mphase_prefetch<NPV, NPV + NS, PF, 0>();
    mphase_pipe<NPV, NPV + NS, PF, 0>();
    if constexpr (DO_S) {
      pin(sc[0]);
      pin(sc[1]);
    }
#pragma unroll
    for (int db = 0; db < NDB; ++db) pin(acc[db]);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
    phase_barrier();
  };

  // Softmax phase of tile tt (ring slot tt % 3; tt counts from tb).  First
  // issues this wave's share of the loads two tiles ahead (group A: K(tt+2)
  // into stage tt+2; group B: V(tt+2) into stage tt+3), last waits for the
  // loads it issued one softmax phase earlier.
  auto vphase = [&](auto s3, int tt, auto first_c) {
    constexpr int S3 = decltype(s3)::value;
    constexpr bool FIRST = decltype(first_c)::value;  // the item's first tile: nothing to keep or rescale
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    __builtin_amdgcn_sched_barrier(0);
    const int ta = it.tb + tt;  // absolute tile index
    if (grp == 0) {
      issue_k(it, kstage(std::integral_constant<int, (S3 + 2) % 3>{}), ta + 2, blk_next);
    } else {
      issue_v(it, vstage(s3), ta + 2, blk_next);
    }
    blk_next = tile_block(it, ta + 3);
    const int key0 = ta * ST::kKeys;
    const bool need_mask = (key0 + ST::kKeys > it.skv) || (dm.causal && key0 + ST::kKeys - 1 > it.qpos_lo);
    if (need_mask) mask_tile(sc, it.vis - key0);
    // Exponentials against the current reference; the exact pass when a
    // row has none yet or a lane's partial sum leaves the bound (not
    // `> kRescaleSum`: NaN and inf sums take the exact pass too).
    float rs0 = 0.f, rs1 = 0.f;
    bool keep = false;
    if constexpr (!FIRST) keep = __builtin_amdgcn_ballot_w64(m_run == -__builtin_inff()) == 0;
    if (keep) {
      const float nmc = -m_run * c;
      rs0 = softmax_exp<DT>(sc[0], nmc, c, pk[0]);
      rs1 = softmax_exp<DT>(sc[1], nmc, c, pk[1]);
      keep = __builtin_amdgcn_ballot_w64(!(rs0 + rs1 <= kRescaleSum)) == 0;
    }
    if (!keep) {
      float nmc;
      if constexpr (FIRST) {
        f32x16 none[1] = {f32x16{}};
        nmc = softmax_rebase<1>(sc, m_run, l_run, none, c);
      } else {
        nmc = softmax_rebase<NDB>(sc, m_run, l_run, acc, c);
      }
      rs0 = softmax_exp<DT>(sc[0], nmc, c, pk[0]);
      rs1 = softmax_exp<DT>(sc[1], nmc, c, pk[1]);
    }
    l_run += rs0 + rs1;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) pin(pk[mb][kk]);
#pragma unroll
    for (int db = 0; db < NDB; ++db) pin(acc[db]);
    pin(l_run);
    pin(m_run);
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(ST::NI));  // all but this phase's loads
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
    phase_barrier();
  };

  for (;;) {
#pragma unroll
    for (int db = 0; db < NDB; ++db) acc[db] = f32x16{};
    m_run = -__builtin_inff();
    l_run = 0.f;
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // the prologue loads
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) pin(qreg[ks]);
    if (__builtin_amdgcn_ballot_w64(!it.valid) != 0) {
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) qreg[ks] = it.valid ? qreg[ks] : u32x4{0u, 0u, 0u, 0u};
    }
    phase_barrier();
    if (grp == 1) phase_barrier();  // group B runs one phase behind

    const int ntiles = it.ntiles;
    if (ntiles > 0) {
      mphase(I0{}, BF{}, BT{});
      vphase(I0{}, 0, BT{});
      int tt = 1;
      for (; tt + 3 <= ntiles; tt += 3) {
        mphase(I1{}, BT{}, BT{});
        vphase(I1{}, tt, BF{});
        mphase(I2{}, BT{}, BT{});
        vphase(I2{}, tt + 1, BF{});
        mphase(I0{}, BT{}, BT{});
        vphase(I0{}, tt + 2, BF{});
      }
      if (tt < ntiles) {
        mphase(I1{}, BT{}, BT{});
        vphase(I1{}, tt, BF{});
        ++tt;
        if (tt < ntiles) {
          mphase(I2{}, BT{}, BT{});
          vphase(I2{}, tt, BF{});
          ++tt;
        }
      }
      const int s3 = tt % 3;
      if (s3 == 0) mphase(I0{}, BT{}, BF{});
      else if (s3 == 1) mphase(I1{}, BT{}, BF{});
      else mphase(I2{}, BT{}, BF{});
    } else {
      phase_barrier();
    }
    if (grp == 0) phase_barrier();  // both groups pass the same number of barriers
    // No LDS-DMA load (of a tile past the end) may still be writing when the
    // stages are reused (by the next item, or for the output below), nor
    // when the workgroup exits.
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    __syncthreads();

    int* sched = nullptr;
    if constexpr (PERSIST) sched = s_sched;
    const bool dyn = sched != nullptr;
    int w_next = PERSIST && !dyn ? item_at(k_item + 1) : -1;
    // Dynamic schedule: thread 0 claims a ticket of this XCD's queue as the
    // epilogue begins; it is resolved after the output stores, which hide
    // the atomic's round trip.
    const int xq = (int)(__builtin_amdgcn_s_getreg((31 << 11) | 20) & 7);  // HW_REG_XCC_ID
    int ticket = 0;
    if (dyn && t == 0) ticket = __hip_atomic_fetch_add(&sched[xq], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // One workgroup per item: this item's parameters and the lane ids again,
    // from the item index, block_m and a zero laundered through SGPRs (the
    // lane id through v_mbcnt): kept from the start, the values read only
    // here would stay live across the whole tile loop (at D = 64, in
    // scratch).  The persistent kernel keeps them (and measured 35-60 %
    // slower on short key-split prefills when re-deriving them).
    int w_cur = item_at(k_item), zero = 0, bm = p.block_m;
    if constexpr (!PERSIST) asm volatile("" : "+s"(w_cur), "+s"(zero), "+s"(bm));
    // The output rows' places are worked out here, not hoisted out of the
    // item loop (where they delayed the first loads).
    int wave_e = wave;
    asm volatile("" : "+s"(wave_e));
    const int lane_e =
        PERSIST ? lane : (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, (unsigned)zero));
    const int t_e = wave * 64 + lane_e, i_e = lane_e & 31, hh_e = lane_e >> 5;
    const Item ie = PERSIST ? it : decode(w_cur, i_e, bm);

    // Split query block: publish this half's state (reference max, lane
    // partial row sum, accumulators in groups of four, lane-major so each lane
    // of the other item reads back exactly its own row with 16-byte loads, all
    // requested before the first is used); the item that completes the
    // block's counter merges the other half into its registers and writes o.
    // The counter is read first: when the other half has already published
    // (counter 1), this item is the last one and skips publishing its own.
    // Otherwise it publishes, then counts itself in; whichever item's
    // increment finds 1 merges.  Every increment follows its item's completed
    // stores, so a counter of 1 means the other state is readable.
    bool write_out = true;
    if (!chunked && ie.part >= 0) {
      constexpr int PF_ = kFwdPartFloats(D);
      constexpr int NA = NDB * 16;  // accumulators per lane
      constexpr uint32_t kQuad = kFwdThreads * 16;  // bytes of one group of four
      const int slot = ie.bh * p.n_split + (p.n_mblk - 1 - ie.pid_m);
      float* mine = p.part_ws + ((int64_t)slot * 2 + ie.part) * PF_;
      const float* other = p.part_ws + ((int64_t)slot * 2 + (1 - ie.part)) * PF_;
      if (t_e == 0) s_last = __hip_atomic_load(&p.part_cnt[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 1;
      __syncthreads();
      bool last = s_last;
      if (!last) {
        const __amdgpu_buffer_rsrc_t rm = make_rsrc(mine, NDB * 4 * kQuad);
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            store_coherent4(rm, 16u * t_e, (db * 4 + j) * kQuad,
                            f32x4{acc[db][4 * j], acc[db][4 * j + 1], acc[db][4 * j + 2], acc[db][4 * j + 3]});
        store_coherent(mine + NA * kFwdThreads + t_e, m_run);
        store_coherent(mine + (NA + 1) * kFwdThreads + t_e, l_run);
        __builtin_amdgcn_s_waitcnt(0);  // this thread's stores are done
        __syncthreads();
        if (t_e == 0) s_last = __hip_atomic_fetch_add(&p.part_cnt[slot], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 1;
        __syncthreads();
        last = s_last;
      }
      __syncthreads();  // every wave has read s_last before the next item's writes it
      if (last) {
        // Both halves have arrived: leave the counter zero for the next call.
        if (t_e == 0) __hip_atomic_store(&p.part_cnt[slot], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // The merge is written in terms of the lower (0) and upper (1) half,
        // not of this item and the other one, so the rounding (fma
        // contraction included) does not depend on which half finished
        // last: repeated calls give identical outputs.
        const bool lo = ie.part == 0;
        const __amdgpu_buffer_rsrc_t ro = make_rsrc(other, NDB * 4 * kQuad);
        const float m_o = load_coherent(other + NA * kFwdThreads + t_e);
        const float l_o = load_coherent(other + (NA + 1) * kFwdThreads + t_e);
        f32x4 xo[NDB * 4];
#pragma unroll
        for (int j = 0; j < NDB * 4; ++j) xo[j] = load_coherent4(ro, 16u * t_e, j * kQuad);
        __builtin_amdgcn_sched_barrier(0);
        const float m0 = lo ? m_run : m_o, m1 = lo ? m_o : m_run;
        const float mm = fmaxf(m0, m1);
        const float mu = (mm == -__builtin_inff()) ? 0.f : mm;
        const float a0 = fast_exp2((m0 - mu) * c), a1 = fast_exp2((m1 - mu) * c);
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const float x_o = xo[db * 4 + (v >> 2)][v & 3];
            const float x0 = lo ? acc[db][v] : x_o, x1 = lo ? x_o : acc[db][v];
            acc[db][v] = __builtin_fmaf(x0, a0, x1 * a1);
          }
        const float l0 = lo ? l_run : l_o, l1 = lo ? l_o : l_run;
        l_run = __builtin_fmaf(l0, a0, l1 * a1);
        m_run = mm;
      }
      write_out = last;
    }

    if constexpr (chunked) {
      // Key chunk: the partial state of this lane's row, as the split-KV
      // first pass stores it (m = m_ref * c in log2 units, relative to which
      // l and acc are kept; -inf with l = 0 for a row that saw no key in
      // this chunk; 0 for a sequence without keys, which the combine turns
      // into a zero row).  Lane (i, hh) holds dims 32 db + 8 j + 4 hh + 0..3
      // of its row in acc[db][4 j .. 4 j + 3].
      const float l_tot = xhalf_sum(l_run);
      if (ie.valid) {
        const int chunk = ie.tb / p.kv_chunk_tiles;
        const int64_t row = (((int64_t)ie.b * dm.Hq + ie.head) * dm.Sq + ie.pos) * p.kv_splits + chunk;
        float* wa = p.ws_acc + row * D + 4 * hh_e;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            *reinterpret_cast<f32x4*>(wa + 32 * db + 8 * j) =
                f32x4{acc[db][4 * j], acc[db][4 * j + 1], acc[db][4 * j + 2], acc[db][4 * j + 3]};
        if (hh_e == 0) {
          p.ws_m[row] = ie.skv == 0 ? 0.f : m_run * c;
          p.ws_l[row] = l_tot;
        }
      }
    } else if (write_out) {
      // Epilogue: o = acc / l (0/0 = NaN for a row whose keys are all
      // masked, as the reference's acc / l_i at gqa_fwd.py:106).  A sequence
      // with no keys at all gives zero rows instead: tests/reference.py:33-34
      // takes the softmax over an empty key axis and multiplies it with an
      // empty V.  Optional LSE side output: ln sum_k exp(s_k * D^-0.5) =
      // (m_ref * c + log2 l) * ln 2 (l is relative to the reference point
      // m_ref); -inf for a row with no visible key.
      const float l_tot = xhalf_sum(l_run);
      const float inv = ie.skv == 0 ? 0.f : 1.0f / l_tot;
      if (p.lse != nullptr && ie.valid && hh_e == 0) {
        // (B, Hq, Sq), or (tokens, Hq) with variable lengths.
        const int64_t li = varlen ? (ie.tok0 + ie.pos) * dm.Hq + ie.head
                                  : ((int64_t)ie.b * dm.Hq + ie.head) * dm.Sq + ie.pos;
        p.lse[li] = (m_run * c + __log2f(l_tot)) * kLn2;
      }
      {
        // The wave's 32 x D output tile goes through LDS (row-major, 16-byte
        // chunks XOR-swizzled by row; two waves per former K/V stage), so that
        // it leaves as whole rows: each store instruction writes 64 lanes x 16
        // bytes covering RPI complete rows, where storing straight from the
        // O^T accumulators would write 16 bytes into each of 32 rows per
        // instruction.
        constexpr int CPR16 = 2 * D / 16;  // 16-byte chunks per row
        constexpr int RPI = 64 / CPR16;    // rows per store instruction
        const int sw = wave >> 1;
        char* ot = (sw == 0 ? lds1_k0 : sw == 1 ? lds1_k1 : sw == 2 ? lds1_k2 : lds0_v0) + (wave & 1) * (32 * 2 * D);
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            u32x2 x;
            x[0] = E::pack2(acc[db][4 * j] * inv, acc[db][4 * j + 1] * inv);
            x[1] = E::pack2(acc[db][4 * j + 2] * inv, acc[db][4 * j + 3] * inv);
            const int ch = (4 * db + j) ^ (i_e & (CPR16 - 1));
            *reinterpret_cast<u32x2*>(ot + i_e * (2 * D) + ch * 16 + 8 * hh_e) = x;
          }
        __builtin_amdgcn_s_waitcnt(kLgkm0);  // this wave's LDS writes before its reads
        const int cc = lane_e % CPR16, r0 = lane_e / CPR16;
        if ((bm & 31) == 0) {
          // The wave's 32 rows are consecutive positions of one head: one row
          // address, advanced by RPI rows per store.
          const int g2 = (int)(__umul24(wave_e * 32, p.bm_mul) >> 16);
          const int pos2 = ie.pid_m * bm + (wave_e * 32 - g2 * bm) + r0;
          T* orow = static_cast<T*>(const_cast<void*>(p.o.ptr)) + row_off(ie, p.o, pos2, ie.kvh * dm.G + g2) + 8 * cc;
          const int left = g2 < dm.G ? ie.sq - pos2 : 0;  // rows from this one on
#pragma unroll
          for (int ri = 0; ri < 32 / RPI; ++ri) {
            const int rr = RPI * ri + r0;  // row of the tile
            const u32x4 x = *reinterpret_cast<const u32x4*>(ot + rr * (2 * D) + ((cc ^ (rr & (CPR16 - 1))) * 16));
            if (RPI * ri < left) *reinterpret_cast<u32x4*>(orow + (int64_t)(RPI * ri) * p.o.ss) = x;
          }
        } else {
#pragma unroll 1
          for (int ri = 0; ri < 32 / RPI; ++ri) {
            const int rr = RPI * ri + r0;
            const u32x4 x = *reinterpret_cast<const u32x4*>(ot + rr * (2 * D) + ((cc ^ (rr & (CPR16 - 1))) * 16));
            const int r2 = wave_e * 32 + rr;
            const int g2 = (int)(__umul24(r2, p.bm_mul) >> 16), pos2 = ie.pid_m * bm + (r2 - g2 * bm);
            if (g2 < dm.G && pos2 < ie.sq) {
              T* orow = static_cast<T*>(const_cast<void*>(p.o.ptr)) + row_off(ie, p.o, pos2, ie.kvh * dm.G + g2);
              *reinterpret_cast<u32x4*>(orow + 8 * cc) = x;
            }
          }
        }
      }
    }
    if (dyn) {
      if (wave == 0) {
        int lo, n, S;
        xrange(xq, lo, n, S);
        int w = __builtin_amdgcn_readfirstlane(S + ticket < n ? lo + S + ticket : -1);
        // This XCD's queue is empty: lanes 1-7 read the other queues'
        // counters at once; the first one with items left is claimed (a
        // failed claim means that queue has just run out: counters only
        // grow, so at most 7 rounds).
        for (int round = 0; round < 8 && w < 0; ++round) {
          const int y = (xq + lane) & 7;
          int ly, ny, Sy;
          xrange(y, ly, ny, Sy);
          int left = 0;
          if (lane >= 1 && lane < 8 && Sy < ny)
            left = ny - Sy - __hip_atomic_load(&sched[y], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const uint64_t has = __builtin_amdgcn_ballot_w64(left > 0);
          if (has == 0) break;  // every queue is empty
          const int d = __builtin_ffsll((long long)has) - 1;
          const int yc = (xq + d) & 7;
          int lc, nc, Sc;
          xrange(yc, lc, nc, Sc);
          int tk = 0;
          if (lane == 0) tk = __hip_atomic_fetch_add(&sched[yc], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          tk = __builtin_amdgcn_readfirstlane(tk);
          if (Sc + tk < nc) w = lc + Sc + tk;
        }
        if (w < 0 && lane == 0) {
          // No work left: count out, in two levels so that the workgroups
          // ending together do not all queue on one counter: the S
          // workgroups of group g = blockIdx % 8, then the groups.  The
          // last workgroup out has seen every other workgroup's claims
          // complete: it clears the counters.
          const int g = blockIdx.x & 7;
          int lg, ng, Sg;
          xrange(g, lg, ng, Sg);
          const int dg = __hip_atomic_fetch_add(&sched[8 + g], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if (dg == Sg - 1) {
            const int groups = min(n_wg, 8);
            const int dt = __hip_atomic_fetch_add(&sched[16], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (dt == groups - 1)
              for (int z = 0; z < 17; ++z) __hip_atomic_store(&sched[z], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
        }
        if (lane == 0) s_next = w;
      }
      __syncthreads();
      w_next = s_next;
    }
    if (!PERSIST || w_next < 0) break;
    // Persistent: the next item's first tiles (once every wave's output has
    // left the stages) and Q, loaded while the output stores drain.
    __syncthreads();
    it = decode(w_next, i, p.block_m);
    blk_next = prologue_kv(it);
    prologue_q(it);
    ++k_item;
  }
}

template <int DT, int D, int PG>
static hipError_t launch_fwd_t(FwdParams p, hipStream_t stream) {
  const int per_bh = p.kv_splits > 0 ? p.n_mblk * p.kv_splits : p.n_mblk + p.n_split;
  const int total = per_bh * p.dm.Hkv * p.dm.B;
  if (total <= 0) return hipSuccess;
  const int cus = device_cu_count();
  const bool fixed_lists = p.kv_splits == 0 && total < kFwdDynMinItemsPerWg * std::max(cus, 1);
  // (item_of has the figures.)  Contiguous without a mask: only the split
  // blocks, whose count is chosen for this order (dispatch.py
  // FWD_SPLIT_MAX_ROUNDS).
  if (p.kv_splits > 0)
    set_item_order(p, per_bh, PG > 0 && D == 128, kDealPairs(D));
  else if (PG == 0 && !p.dm.causal)
    set_item_order(p, per_bh, p.n_split > 0, p.dm.B * p.dm.Hkv);
  else
    set_item_order(p, per_bh, (PG > 0 && D == 128) || (total > cus && (PG > 0 || D == 64 || fixed_lists)),
                   kDealPairs(D));
  p.div_mblk = make_fast_div((uint32_t)p.n_mblk);
  p.div_hkv = make_fast_div((uint32_t)p.dm.Hkv);
  p.bm_mul = (65536u + (uint32_t)p.block_m - 1) / (uint32_t)p.block_m;
  int grid = total;
  if (PG == 0 && D == 128) {
    grid = cus > 0 ? std::min(total, cus) : total;
    p.n_wg = grid;
    // The dynamic schedule pays for its claims (atomic round trips of ~2 us,
    // and a tail of them as the last workgroups finish) only with many
    // items per workgroup: measured -0.5 to -1.1 % at 8 (16K-token
    // prefill), +1 to +3 % at 2-4 and +25 % at 1-2 (key-split short
    // prefill); below 8 the static snake schedule runs.
    if (total < kFwdDynMinItemsPerWg * grid) p.sched = nullptr;
  } else {
    p.sched = nullptr;
  }
  if (p.kv_splits > 0)
    hipLaunchKernelGGL((gqa_fwd_kernel<DT, D, PG, true>), dim3(grid), dim3(kFwdThreads), 0, stream, p);
  else
    hipLaunchKernelGGL((gqa_fwd_kernel<DT, D, PG>), dim3(grid), dim3(kFwdThreads), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_fwd(const FwdParams& p, int dtype, hipStream_t stream) {
  if (dtype == 0)
    return p.dm.D == 128 ? launch_fwd_t<0, 128, 0>(p, stream) : launch_fwd_t<0, 64, 0>(p, stream);
  return p.dm.D == 128 ? launch_fwd_t<1, 128, 0>(p, stream) : launch_fwd_t<1, 64, 0>(p, stream);
}

template <int PG>
static hipError_t launch_paged_fwd_t(const FwdParams& p, int dtype, hipStream_t stream) {
  if (dtype == 0)
    return p.dm.D == 128 ? launch_fwd_t<0, 128, PG>(p, stream) : launch_fwd_t<0, 64, PG>(p, stream);
  return p.dm.D == 128 ? launch_fwd_t<1, 128, PG>(p, stream) : launch_fwd_t<1, 64, PG>(p, stream);
}

// Requires block_size >= 512 / D, the rows of one LDS-DMA instruction
// (pages of >= 64 keys hold whole tiles, of 16-32 keys whole 16-row wave
// shares of a tile, smaller ones whole instructions).  The 16-32-key form at
// D = 64 derives its K offsets by an XOR of bit 5 and so takes row strides
// of a multiple of 64 bytes; other strides take the per-instruction form,
// which serves any page of >= 8 keys there.
hipError_t launch_paged_fwd(const FwdParams& p, int dtype, hipStream_t stream) {
  if ((1 << p.block_shift) < 512 / p.dm.D) return hipErrorInvalidValue;
  if (p.block_shift >= 6) return launch_paged_fwd_t<1>(p, dtype, stream);
  const bool medium = p.block_shift >= 4 && (p.dm.D != 64 || (2 * p.k.ss) % 64 == 0);
  return medium ? launch_paged_fwd_t<3>(p, dtype, stream) : launch_paged_fwd_t<2>(p, dtype, stream);
}

}  // namespace gqa
