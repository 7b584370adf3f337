// gqa_short.hip — single-pass forward of short calls: few query blocks, or
// blocks of few keys, where the chain of tiles of one block and the start and
// end of a workgroup, not the matrix cores, set the run time.
//
// As gqa_fwd.hip (group-packed rows, transposed tiles, lazily rescaled online
// softmax, MFMA phases of one wave group beside softmax phases of the other),
// but a workgroup takes 128 packed rows instead of 256 and its two groups of
// four waves split the KEYS: group g computes rows 0-127 over tiles 2 j + g,
// with its own online softmax, and the two states are merged in LDS at the end
// (as the split-KV combine merges two splits).  Twice the workgroups, half the
// tiles one after another; a tile still costs a wave the same instructions, so
// the matrix rate of a full GPU is the same, less the merge and twice the LDS
// traffic from L2.
//
// What bounds it: 5 us from launch to the first product (launch, kernel
// arguments, first loads), ~1.1 us per step of two tiles, and ~1.5 us for the
// merge and the output.
//
// Each group streams its own K and V tiles through two LDS stages each (128
// KiB for both groups at head_dim 128, one workgroup per CU): the softmax
// phase of step j, whose barriers on both sides have every wave of the group
// done with K(j) and V(j-1), refills K's stage with K(j+2) and V's with V(j+1)
// and waits for the loads issued one softmax phase earlier.
#include <algorithm>
#include <type_traits>

#include "gqa_common.hpp"
#include "gqa_fwd_parts.hpp"
#include "gqa_lds.hpp"
#include "gqa_params.hpp"

namespace gqa {

template <int DT, int D, int PG>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gqa_short_kernel(FwdParams p) {
  using E = Elem<DT>;
  using T = typename E::T;
  using ST = FwdStage<D>;
  constexpr int CPR = ST::CPR;
  constexpr bool PAGED = PG != 0;
  constexpr int NDB = D / 32;  // 32-wide d blocks of O^T
  constexpr int NKS = D / 16;  // k-steps of S^T
  constexpr int PF = 6;        // MFMA slots of LDS-read lookahead
  constexpr int TB = ST::kTileBytes;
  // One array per stage of K and of V, the two groups' tiles side by side:
  // the compiler can then tell the LDS-DMA targets from the stages being
  // read.  V below 64 KiB, where a transposing read's address fits its offset
  // field; K addressed from per-lane register bases (kah).  The compiler lays
  // kernel LDS variables out in name order.
  __shared__ __attribute__((aligned(1024))) char lds0_v0[2 * TB];
  __shared__ __attribute__((aligned(1024))) char lds0_v1[2 * TB];
  __shared__ __attribute__((aligned(1024))) char lds1_k0[2 * TB];
  __shared__ __attribute__((aligned(1024))) char lds1_k1[2 * TB];

  const Dims& dm = p.dm;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6) & 7;
  const int grp = wave >> 2, gw = wave & 3;
  const int i = lane & 31, hh = lane >> 5;
  const bool varlen = p.q_len != nullptr;

  // Work item: one query block of one (b, kv head), heavy (late) blocks first
  // under causal; every XCD gets a contiguous range of items.
  const int w = xcd_remap(blockIdx.x, p.n_mblk * dm.Hkv * dm.B);
  int bh, mrank;
  item_of(p, w, p.n_mblk, bh, mrank);
  const int pid_m = dm.causal ? p.n_mblk - 1 - mrank : mrank;
  const int b = fast_div(bh, p.div_hkv.mul, p.div_hkv.shift), kvh = bh - b * dm.Hkv;
  const int skv = PAGED ? min(max(load_uniform(p.seq_lens + b), 0), dm.Skv) : dm.Skv;
  const int sq = varlen ? min(max(load_uniform(p.q_len + b), 0), dm.Sq) : dm.Sq;
  const int64_t tok0 = varlen ? (int64_t)load_uniform(p.q_start + b) : 0;
  const int pos_lo = pid_m * p.block_m;
  if (pos_lo >= sq) return;  // a block past this sequence's queries

  // This lane's query row (the same in both groups).
  const int r = gw * 32 + i;
  const int g = (int)(__umul24(r, p.bm_mul) >> 16);
  const int pos = pos_lo + r - g * p.block_m;
  const bool valid = g < dm.G && pos < sq;
  const int head = kvh * dm.G + (g < dm.G ? g : 0);
  const int qpos_lo = pos_lo + (skv - sq);
  // The keys this row sees, as mask_tile counts them.
  const int vis = (dm.causal ? min(skv, pos + (skv - sq) + 1) : skv) - 8 * hh;

  // Tiles of the block (its last visible key); loads end with them, so a
  // tile past an odd count reads zeros and is masked.
  const int pos_hi = min(pos_lo + p.block_m, sq) - 1;
  const int kv_end = dm.causal ? max(min(skv, pos_hi + (skv - sq) + 1), 0) : skv;
  const int ntiles = (kv_end + ST::kKeys - 1) / ST::kKeys;
  const int steps = (ntiles + 1) >> 1;
  const int rows_ld = min(skv, ntiles * ST::kKeys);

  const uint32_t kssb = (uint32_t)(2 * p.k.ss), vssb = (uint32_t)(2 * p.v.ss);
  const char* kbh = static_cast<const char*>(p.k.ptr) + 2 * ((PAGED ? 0 : (int64_t)b * p.k.sb) + (int64_t)kvh * p.k.sh);
  const char* vbh = static_cast<const char*>(p.v.ptr) + 2 * ((PAGED ? 0 : (int64_t)b * p.v.sb) + (int64_t)kvh * p.v.sh);
  const bool flat = !PAGED && rows_ld > 0;
  const __amdgpu_buffer_rsrc_t rk = make_rsrc(kbh, flat ? (uint32_t)(rows_ld - 1) * kssb + 2 * D : 0u);
  const __amdgpu_buffer_rsrc_t rv = make_rsrc(vbh, flat ? (uint32_t)(rows_ld - 1) * vssb + 2 * D : 0u);
  const int* table_row = PAGED ? p.block_table + (int64_t)b * p.table_stride : nullptr;
  const int lrow = lane / CPR;
  const uint32_t koff =
      (uint32_t)(lrow * kssb) + 16u * (uint32_t)((lane % CPR) ^ ST::gk((gw * ST::RPI + lrow) & 15));
  const uint32_t voff = (uint32_t)(lrow * vssb) + 16u * (uint32_t)((lane % CPR) ^ ST::sv(lrow));
  using Blocks = FwdTileBlocks<D, PG>;
  auto ids = [&](int j) __attribute__((always_inline)) -> Blocks {  // block(s) of this group's tile j
    return tile_blocks<D, PG>(table_row, p.block_shift, rows_ld, 2 * j + grp, gw);
  };
  auto issue_k = [&](char* stage, int j, const Blocks& blk) __attribute__((always_inline)) {
    issue_fwd_tile<D, PG>(stage + grp * TB, kbh, rk, kssb, koff, p.k.sb, p.block_shift, rows_ld, 2 * j + grp, blk, true,
                          gw, lane);
  };
  auto issue_v = [&](char* stage, int j, const Blocks& blk) __attribute__((always_inline)) {
    issue_fwd_tile<D, PG>(stage + grp * TB, vbh, rv, vssb, voff, p.v.sb, p.block_shift, rows_ld, 2 * j + grp, blk,
                          false, gw, lane);
  };

  // Loads in the order of their first use: K(0) and Q, K(1), V(0).  Q's 128
  // rows go through LDS (V's second stage, first written after every wave has
  // read its rows) in whole rows, 16 per wave: loaded straight into the
  // operand registers, each of a wave's eight instructions touched 32 rows, in
  // both groups, and issuing them took the second group 1.9 us (64 tokens: 9.9
  // -> 8.9 us).  An invalid row loads the block's first row and is zeroed when
  // it has landed.  16-byte chunk ch of row r lies at chunk ch ^ qsw(r): 16
  // lanes reading one chunk of 16 rows hit 16 distinct bank groups.
  auto qsw = [](int row) { return CPR == 16 ? row & 15 : (row >> 1) & 7; };
  Blocks id_v = ids(0), id_k = ids(1);  // of the next V and K tiles to load
  issue_k(lds1_k0, 0, id_v);
  {
    typedef __attribute__((address_space(3))) void lds_void;
    typedef const __attribute__((address_space(1))) void glb_void;
    const T* qblk = static_cast<const T*>(p.q.ptr) + (int64_t)(kvh * dm.G) * p.q.sh +
                    (varlen ? (tok0 + pos_lo) * p.q.ss : (int64_t)b * p.q.sb + (int64_t)pos_lo * p.q.ss);
    auto put = [&](int n, int64_t off) __attribute__((always_inline)) {
      const int row = 16 * wave + n * ST::RPI + lrow;
      __builtin_amdgcn_global_load_lds((glb_void*)(uintptr_t)(qblk + off + 8 * ((lane % CPR) ^ qsw(row))),
                                       (lds_void*)(lds0_v1 + (16 * wave + n * ST::RPI) * (2 * D)), 16, 0, 0);
    };
    if ((p.block_m & 15) == 0) {  // this wave's 16 rows: consecutive positions of one head
      const int rg = (int)(__umul24(16 * wave, p.bm_mul) >> 16), rm = 16 * wave - rg * p.block_m + lrow;
      const int64_t off = (int64_t)rg * p.q.sh + (int64_t)rm * p.q.ss;
      const int left = rg < dm.G ? sq - (pos_lo + rm) : 0;
#pragma unroll
      for (int n = 0; n < 16 / ST::RPI; ++n) put(n, n * ST::RPI < left ? off + (int64_t)(n * ST::RPI) * p.q.ss : 0);
    } else {
#pragma unroll 1
      for (int n = 0; n < 16 / ST::RPI; ++n) {
        const int row = 16 * wave + n * ST::RPI + lrow;
        const int rg = (int)(__umul24(row, p.bm_mul) >> 16), rm = row - rg * p.block_m;
        put(n, rg < dm.G && pos_lo + rm < sq ? (int64_t)rg * p.q.sh + (int64_t)rm * p.q.ss : 0);
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  issue_k(lds1_k1, 1, id_k);
  issue_v(lds0_v0, 0, id_v);
  id_v = id_k;
  id_k = ids(2);

  // LDS read offsets, with the group's half of a stage array and (K) the LDS
  // address of stage 0 in the register: every read is a register plus an
  // immediate.  (The masks are no-ops on the values; they give the compiler
  // known bounds.)
  const uint32_t k0base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds1_k0;
  uint32_t kah[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks)
    kah[ks] = k0base + (uint32_t)(grp * TB) +
              ((uint32_t)(pi_key(i) * (2 * D) + 16 * ((2 * ks + hh) ^ ST::gk(pi_key(i)))) & ((TB / 2 - 1) & ~15u));
  uint32_t vb[NDB];
  {
    const int q = lane >> 4, ii = lane & 15;
    const int rowl = 8 * (q >> 1) + (ii >> 2);
    const int f = (CPR == 16) ? (ii >> 2) : ((ii >> 3) & 1);  // sv(rowl) / 4
#pragma unroll
    for (int db = 0; db < NDB; ++db)
      vb[db] = (uint32_t)(grp * TB) +
               ((uint32_t)(rowl * (2 * D) + 16 * (4 * (db ^ f) + 2 * (q & 1) + ((ii & 3) >> 1)) + 8 * (ii & 1)) &
                ((TB - 1) & ~7u));
  }

  f32x16 acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = f32x16{};
  float m_run = -__builtin_inff(), l_run = 0.f;
  const float c = dm.c;
  f32x16 sc[2];    // S^T of the current tile (MFMA phase -> softmax phase)
  u32x4 pk[2][2];  // P^T operands (softmax phase -> next MFMA phase)
  u32x4 qreg[NKS];

  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using BT = std::true_type;
  using BF = std::false_type;

  // MFMA phase of step j (j even: PAR = 0): P*V of this group's previous tile
  // (V stage 1 - PAR) and S^T of its current one (K stage PAR).
  auto mphase = [&](auto par, auto pvc, auto sc_) __attribute__((always_inline)) {
    constexpr int PAR = decltype(par)::value;
    constexpr bool DO_PV = decltype(pvc)::value;
    constexpr bool DO_S = decltype(sc_)::value;
    constexpr int NPV = DO_PV ? 4 * NDB : 0;
    constexpr int NS = DO_S ? 2 * NKS : 0;
    const char* ck = PAR == 0 ? lds1_k0 : lds1_k1;
    const char* cv = PAR == 0 ? lds0_v1 : lds0_v0;
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
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) asm volatile("" : "+v"(kah[ks]));
#pragma unroll
      for (int j = 0; j < NS; ++j)
        opk[j] = *reinterpret_cast<const u32x4*>(ck + (j & 1) * 32 * (2 * D) + (kah[j >> 1] - k0base));
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

  // Softmax phase of step j: refills K's stage (K(j+2)) and V's other one
  // (V(j+1)), last waits for the loads issued one softmax phase earlier.
  auto vphase = [&](auto par, int j, auto first_c) __attribute__((always_inline)) {
    constexpr int PAR = decltype(par)::value;
    constexpr bool FIRST = decltype(first_c)::value;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    __builtin_amdgcn_sched_barrier(0);
    issue_k(PAR == 0 ? lds1_k0 : lds1_k1, j + 2, id_k);
    issue_v(PAR == 0 ? lds0_v1 : lds0_v0, j + 1, id_v);
    id_v = id_k;
    id_k = ids(j + 3);
    const int key0 = (2 * j + grp) * ST::kKeys;
    const bool need_mask = (key0 + ST::kKeys > skv) || (dm.causal && key0 + ST::kKeys - 1 > qpos_lo);
    if (need_mask) mask_tile(sc, vis - key0);
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
      if constexpr (FIRST) {  // (nothing to rescale yet)
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
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(2 * ST::NI));
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
    phase_barrier();
  };

  __builtin_amdgcn_s_waitcnt(vmcnt_imm(2 * ST::NI));  // K(0) and Q
  phase_barrier();
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks)
    qreg[ks] = *reinterpret_cast<const u32x4*>(lds0_v1 + r * (2 * D) + 16 * ((2 * ks + hh) ^ qsw(r)));
  if (__builtin_amdgcn_ballot_w64(!valid) != 0) {
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qreg[ks] = valid ? qreg[ks] : u32x4{0u, 0u, 0u, 0u};
  }
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) pin(qreg[ks]);
  if (grp == 1) phase_barrier();  // group B runs one phase behind
  if (steps > 0) {
    mphase(I0{}, BF{}, BT{});
    vphase(I0{}, 0, BT{});
    int j = 1;
    for (; j + 2 <= steps; j += 2) {
      mphase(I1{}, BT{}, BT{});
      vphase(I1{}, j, BF{});
      mphase(I0{}, BT{}, BT{});
      vphase(I0{}, j + 1, BF{});
    }
    if (j < steps) {
      mphase(I1{}, BT{}, BT{});
      vphase(I1{}, j, BF{});
      mphase(I0{}, BT{}, BF{});
    } else {
      mphase(I1{}, BT{}, BF{});
    }
  } else {
    phase_barrier();
  }
  if (grp == 0) phase_barrier();  // both groups pass the same number of barriers
  // No LDS-DMA load may still be writing when the stages are reused.
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  __syncthreads();

  // Merge: each group hands the other half of its accumulators (the 32-wide d
  // blocks of the other's half) and its row statistics through LDS, and
  // merges its own half.  Written in terms of group 0 and group 1, so both
  // groups compute the same statistics.  A group that saw no key (m = -inf, l
  // = 0, acc = 0) adds nothing; a row without any keeps l = 0.
  constexpr int HDB = NDB / 2;
  // (K's stages hold the accumulators, [wave of the group][4 HDB][64], group
  // 0's in the first; V's second stage the statistics, [wave][2][64].)
  static_assert(4 * 4 * HDB * 64 * 16 <= 2 * TB && 8 * 128 * 4 <= 2 * TB && kShortRows * 2 * D <= 2 * TB, "LDS reuse");
  f32x4* xmine = reinterpret_cast<f32x4*>(grp == 0 ? lds1_k0 : lds1_k1) + gw * 4 * HDB * 64 + lane;
  const f32x4* xother = reinterpret_cast<const f32x4*>(grp == 0 ? lds1_k1 : lds1_k0) + gw * 4 * HDB * 64 + lane;
  float* xml = reinterpret_cast<float*>(lds0_v1);
#pragma unroll
  for (int d = 0; d < HDB; ++d)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 a;
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = grp == 0 ? acc[HDB + d][4 * j + e] : acc[d][4 * j + e];
      xmine[(d * 4 + j) * 64] = a;
    }
  xml[wave * 128 + lane] = m_run;
  xml[wave * 128 + 64 + lane] = l_run;
  __syncthreads();
  const int other = wave ^ 4;
  const float m_o = xml[other * 128 + lane], l_o = xml[other * 128 + 64 + lane];
  const float m0 = grp == 0 ? m_run : m_o, m1 = grp == 0 ? m_o : m_run;
  const float mm = fmaxf(m0, m1);
  const float mu = (mm == -__builtin_inff()) ? 0.f : mm;
  const float a0 = fast_exp2((m0 - mu) * c), a1 = fast_exp2((m1 - mu) * c);
  const float l0 = grp == 0 ? l_run : l_o, l1 = grp == 0 ? l_o : l_run;
  const float l_tot = xhalf_sum(__builtin_fmaf(l0, a0, l1 * a1));
  const float inv = skv == 0 ? 0.f : 1.0f / l_tot;  // (a sequence without keys: zero rows)
  if (p.lse != nullptr && valid && grp == 0 && hh == 0) {
    const int64_t li = varlen ? (tok0 + pos) * dm.Hq + head : ((int64_t)b * dm.Hq + head) * dm.Sq + pos;
    p.lse[li] = (mm * c + __log2f(l_tot)) * kLn2;
  }
  // The output block goes through LDS (row-major, 16-byte chunks XOR-swizzled
  // by row), so that it leaves as whole rows.
  constexpr int CPR16 = 2 * D / 16, RPI = 64 / CPR16;
  char* ot = lds0_v0;
#pragma unroll
  for (int d = 0; d < HDB; ++d)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 xo = xother[(d * 4 + j) * 64];
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x0 = grp == 0 ? acc[d][4 * j + e] : xo[e], x1 = grp == 0 ? xo[e] : acc[HDB + d][4 * j + e];
        y[e] = __builtin_fmaf(x0, a0, x1 * a1) * inv;
      }
      u32x2 x;
      x[0] = E::pack2(y[0], y[1]);
      x[1] = E::pack2(y[2], y[3]);
      const int ch = (4 * (grp * HDB + d) + j) ^ (i & (CPR16 - 1));
      *reinterpret_cast<u32x2*>(ot + r * (2 * D) + ch * 16 + 8 * hh) = x;
    }
  __syncthreads();
  const int cc = lane % CPR16;
#pragma unroll
  for (int ri = 0; ri < 16 / RPI; ++ri) {
    const int rr = wave * 16 + RPI * ri + lane / CPR16;
    const u32x4 x = *reinterpret_cast<const u32x4*>(ot + rr * (2 * D) + ((cc ^ (rr & (CPR16 - 1))) * 16));
    const int g2 = (int)(__umul24(rr, p.bm_mul) >> 16), pos2 = pos_lo + rr - g2 * p.block_m;
    if (g2 < dm.G && pos2 < sq) {
      T* orow = static_cast<T*>(const_cast<void*>(p.o.ptr)) + (int64_t)(kvh * dm.G + g2) * p.o.sh +
                (varlen ? (tok0 + pos2) * p.o.ss : (int64_t)b * p.o.sb + (int64_t)pos2 * p.o.ss);
      *reinterpret_cast<u32x4*>(orow + 8 * cc) = x;
    }
  }
}

template <int DT, int D, int PG>
static hipError_t launch_short_t(FwdParams p, hipStream_t stream) {
  const int64_t total = (int64_t)p.n_mblk * p.dm.Hkv * p.dm.B;
  if (total <= 0) return hipSuccess;
  set_item_order(p, p.n_mblk, PG > 0 || D == 64 || total > device_cu_count(), kDealPairs(D));
  p.div_hkv = make_fast_div((uint32_t)p.dm.Hkv);
  p.bm_mul = (65536u + (uint32_t)p.block_m - 1) / (uint32_t)p.block_m;
  hipLaunchKernelGGL((gqa_short_kernel<DT, D, PG>), dim3((unsigned)total), dim3(kFwdThreads), 0, stream, p);
  return hipGetLastError();
}

template <int PG>
static hipError_t launch_short_pg(const FwdParams& p, int dtype, hipStream_t stream) {
  if (dtype == 0)
    return p.dm.D == 128 ? launch_short_t<0, 128, PG>(p, stream) : launch_short_t<0, 64, PG>(p, stream);
  return p.dm.D == 128 ? launch_short_t<1, 128, PG>(p, stream) : launch_short_t<1, 64, PG>(p, stream);
}

// p.block_m = kShortRows / G, p.n_mblk accordingly; paged as launch_paged_fwd.
hipError_t launch_short(const FwdParams& p, int dtype, hipStream_t stream) {
  if (p.block_table == nullptr) return launch_short_pg<0>(p, dtype, stream);
  if ((1 << p.block_shift) < 512 / p.dm.D) return hipErrorInvalidValue;
  if (p.block_shift >= 6) return launch_short_pg<1>(p, dtype, stream);
  const bool medium = p.block_shift >= 4 && (p.dm.D != 64 || (2 * p.k.ss) % 64 == 0);
  return medium ? launch_short_pg<3>(p, dtype, stream) : launch_short_pg<2>(p, dtype, stream);
}

}  // namespace gqa
