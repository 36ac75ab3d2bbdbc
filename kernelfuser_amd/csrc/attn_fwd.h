#pragma once
// The general attention kernel (attn_fwd_kernel): any D in {128, 256} and GQA
// ratio.  One workgroup = 4 waves = 128 query rows, 32 rows a wave, of one head
// or shared between two or four heads of a GQA group; 16 KiB K and V tiles (64
// keys at D = 128, 32 at D = 256), one barrier per tile.  attn_fwd128.hip and
// attn_fwd256.hip instantiate it, with NaN semantics (pack_rows).
//
// Each wave is one instruction stream in which every MFMA has its share of the
// other work beside it: iteration u issues GEMM1 of key block u+1 and GEMM2 of
// block u (32 keys each) back to back, and between them the exponentials of
// both blocks, the LDS reads of MFMAs to come and the next tiles' copies, at
// fixed slots.  With the phases one after the other (GEMM1, softmax, GEMM2) a
// wave kept its matrix core busy half of the time, and at D = 256, one wave per
// SIMD, nothing filled the rest: 2010 cycles per 32-key tile for 1024 of MFMA.
// Now 1400 at D = 256 (B=2 S=2048 Hq=16 factored: 92.6 -> 79-82 us with the
// preparation launch) and 1530 for 1024 at D = 128 with two workgroups on the
// CU, 1830 alone (2.0k before; B=1 S=2048 Hq=32: 49.5 -> 47 us).
//
// What bounds it now: with the loop's matrix cores ~70% busy the GPU's power
// management lowers the clock (B=2 S=2048 factored 2.34 -> 2.01 GHz, B=1 S=2048
// at D = 128 1.92); leaving out the exponentials, the copies, or half of the LDS
// reads of a D = 256 iteration takes 9%, 11% and 0% off its cycles.  Short
// sequences are bound by what surrounds the loop: per workgroup and 8 tiles
// (16-18k cycles at D = 128) 13k cycles of norm + RoPE prologue (prepared Q 4.5k),
// 2.5-3k to the first tile's maximum, 2.7k of epilogue; at D = 256 and 16 tiles
// (22-23k) 21k (9k), 2-3k and 5k.
#include <cstdio>
#include <string>
#include <type_traits>

#include "attn_common.h"
#include "attn_mfma.h"
#include "attn_split.h"

namespace kfmi {
namespace {

// Slot of the first operation of element e of a key block's 16 (see the
// schedule in the kernel).
template <int D>
constexpr int f_slot(int e) {
  return D == 128 ? 10 + 7 * e / 8 : 20 + 2 * e;
}

template <int D, int BN, bool CAUSAL, int PRO, int ST, bool FK>
__global__ __launch_bounds__(256, (D == 128 ? 2 : 1)) void attn_fwd_kernel(AttnParams p) {
  static_assert(!FK && BN * D == 8192, "16 KiB tiles; mode 'full' has its own kernel");
  constexpr int BM = 128, RB = 2 * D;
  constexpr int TILE = BN * RB;         // 16 KiB
  constexpr int LPW = TILE / 1024 / 4;  // copies per wave per tile (4)
  constexpr int NC = D / 16, NDB = D / 32, NK16 = BN / 16;
  constexpr int SUB = BN / 32;  // 32-key blocks per tile
  // Rings of R K and R V tiles: tile t is in buffer (t - t0) % R.  D = 128 runs
  // two workgroups per CU with 64 KiB each, D = 256 one with 128 KiB.
  constexpr int R = D == 128 ? 2 : 4;
  constexpr int VRING = R * TILE;
  // D = 256: O (128 registers) and Q (64) in AGPRs, everything else in VGPRs.
  // D = 128: everything fits in the 256 VGPRs of a wave.
  constexpr bool ACC = D == 256;

  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * R * TILE];

  // Every argument the decoding below needs, requested together: left to
  // themselves the loads sit in the branches that use them, each a round trip
  // (eight layers of Gemma-3-4B S=1024 240 -> 233 us, Qwen3-0.6B S=128 87.8 ->
  // 87.0).
  asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.out), "s"(p.S), "s"(p.units), "s"(p.groups), "s"(p.hpw_log),
               "s"(p.n_qblocks), "s"(p.xcd_remap), "s"(p.slot2), "s"(p.n_items), "s"(p.head_major));
  asm volatile("" ::"s"(p.by_units.mul), "s"(p.by_units.shift), "s"(p.by_units.mask), "s"(p.by_groups.mul),
               "s"(p.by_groups.shift), "s"(p.by_groups.mask), "s"(p.by_hkv.mul), "s"(p.by_hkv.shift),
               "s"(p.by_hkv.mask), "s"(p.Hq), "s"(p.Hkv), "s"(p.stamps));
  clock_stamp<false>(p.stamps);
  // Two-slot pairing (slot2 > 0): the second slot holds the short causal
  // blocks, whose workgroups have slack; they start about 12k cycles late, so
  // the long blocks of the first slot, which set the kernel's end, stage their
  // tables, Q rows and first tiles without that traffic.  (s_sleep n waits
  // about 64n cycles.)
  if (CAUSAL && D == 128 && p.slot2 > 0 && (int)blockIdx.x >= p.slot2) {
    __builtin_amdgcn_s_sleep(96);
    __builtin_amdgcn_s_sleep(96);
  }
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;   // half-wave: selects the k-group of the MFMA operands
  const int lr = lane & 31;  // query row of this lane within the wave
  const int64_t S = p.S;

  // ---- work item: heaviest query blocks (or split halves) first, over all heads
  // or (head_major) within a KV head's turn; KV heads pinned to an XCD ----
  const int bid = blockIdx.x;
  int rank, kq, hg;
  if (p.head_major) {
    const int j = bid >> 3;
    kq = p.by_kv_wgs.div(j);
    const int rem = j - kq * (p.groups * p.n_qblocks);
    rank = p.by_groups.div(rem);
    hg = rem - rank * p.groups;
  } else {
    rank = p.by_units.div(bid);
    const int r = bid - rank * p.units;
    const int jj = p.xcd_remap ? r >> 3 : r;
    kq = p.by_groups.div(jj);
    hg = jj - kq * p.groups;
  }
  int qb, t0 = 0, t1 = -1, sid = -1;
  if (D == 256 && p.n_items > 0) {
    qb = p.it_qb[rank];
    t0 = p.it_t0[rank];
    t1 = p.it_t1[rank];
    sid = p.it_sid[rank];
  } else if (CAUSAL && D == 128 && p.slot2 > 0 && bid >= p.slot2) {
    qb = p.by_units.div(bid - p.slot2);
  } else {
    qb = CAUSAL ? p.n_qblocks - 1 - rank : rank;
  }
  // Head group hg of KV head kg (batch and KV head).  Workgroups are dispatched
  // round-robin over the 8 XCDs (bid % 8): with xcd_remap KV head kg runs on XCD
  // kg % 8, so the query heads that read the same K/V share one L2.
  const int kg = p.xcd_remap ? (bid & 7) + 8 * kq : kq;
  const int b = p.by_hkv.div(kg), kvh = kg - b * p.Hkv;
  // this wave's head of the group and its block of 32 rows
  const int wl = 2 - p.hpw_log;
  const int rb = w & ((1 << wl) - 1);
  const int h = (((kvh * p.groups + hg) << p.hpw_log) + (w >> wl));
  const int rows = BM >> p.hpw_log;  // query rows per head
  const int64_t qoff = ((int64_t)b * p.Hq + h) * S;
  const int64_t kvoff = (int64_t)kg * S;

  const uint32_t head_bytes = (uint32_t)(S * RB);
  const i32x4_t krs = buffer_rsrc(p.k + kvoff * D, head_bytes);
  const i32x4_t vrs = buffer_rsrc(p.v + kvoff * D, head_bytes);
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char *)smem);
  uint32_t kvo[LPW], vvo[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    kvo[i] = copy_lane_offset<D>(w * LPW + i, lane, false);
    vvo[i] = copy_lane_offset<D>(w * LPW + i, lane, true);
  }

  const int q0 = qb * rows + rb * 32;
  const int qrow = q0 + lr;

  // ---- KV tile range [t0, nT) of this work item, [u0, nUw) of this wave ----
  const int64_t kv_end = CAUSAL ? ((int64_t)(qb + 1) * rows < S ? (int64_t)(qb + 1) * rows : S) : S;
  const int nT = t1 >= 0 ? t1 : (int)((kv_end + BN - 1) / BN);
  const int64_t wave_end = CAUSAL ? ((int64_t)q0 + 32 < S ? (int64_t)q0 + 32 : S) : S;
  // the loop runs over blocks u of 32 keys (tile u / SUB): this wave's end, and
  // the first that needs masks (it reaches past the wave's first row, when
  // causal, or past S)
  const int u0 = SUB * t0;
  const int nUw0 = q0 < S ? (int)((wave_end + 31) / 32) : 0;
  const int nUw = nUw0 < SUB * nT ? nUw0 : SUB * nT;
  const int u_mask = CAUSAL && (int64_t)q0 + 32 <= S ? q0 / 32 : (int)(S / 32);

  // Copies of tile t; past the item's last tile the offset lies past every
  // head, so the copy moves no data and the count of copies in flight stays
  // the same on every iteration.
  auto tile_off = [&](int t) -> uint32_t { return t < nT ? (uint32_t)t * TILE : 0xffffc000u; };
  auto copy_k1 = [&](int t, int buf, int i) {
    copy16_to_lds(krs, lds0 + buf * TILE + (w * LPW + i) * 1024, kvo[i] + tile_off(t));
  };
  auto copy_v1 = [&](int t, int buf, int i) {
    copy16_to_lds(vrs, lds0 + VRING + buf * TILE + (w * LPW + i) * 1024, vvo[i] + tile_off(t));
  };
  auto copy_k = [&](int t, int buf) {
#pragma unroll
    for (int i = 0; i < LPW; ++i) copy_k1(t, buf, i);
  };
  auto copy_v = [&](int t, int buf) {
#pragma unroll
    for (int i = 0; i < LPW; ++i) copy_v1(t, buf, i);
  };
  auto first_copies = [&]() {
    copy_k(t0, 0);
    copy_k(t0 + 1, 1);
    copy_v(t0, 0);
  };

  uint32_t kra[8], vra[4];
  lds_read_offsets<D>(lane, kra, vra);

  // ---- Q prologue ----
  bf16x8_t qreg[NC];
  float cl;
  if constexpr (PRO == PRO_NORM_ROPE) {
    // The rotary-table rows of the workgroup's positions are first staged in K/V
    // buffers with coalesced copies (the K tiles' chunk swizzle, so kra addresses
    // the lane's chunks) instead of loads that each touch 32 rows.
    const i32x4_t crs = buffer_rsrc(p.cos, (uint32_t)(S * RB));
    const i32x4_t srs = buffer_rsrc(p.sin, (uint32_t)(S * RB));
    const int ncp = rows * RB / 4096;  // 1 KiB copies per wave per table
    auto stage = [&](int cos0, int sin0) {
      for (int i = 0; i < ncp; ++i) {
        const int j = ncp * w + i;
        const uint32_t voff = copy_lane_offset<D>(j, lane, false) + (uint32_t)qb * (uint32_t)(rows * RB);
        copy16_to_lds(crs, lds0 + cos0 + j * 1024, voff);
        copy16_to_lds(srs, lds0 + sin0 + j * 1024, voff);
      }
      StagedTables tab;
      tab.cos = smem + cos0 + rb * 32 * RB;
      tab.sin = smem + sin0 + rb * 32 * RB;
      tab.off = kra;
      return tab;
    };
    if constexpr (D == 128) {
      // 128 or 64 positions: in the buffers of the first tiles, whose copies are
      // issued once every wave holds its rows in registers (they land while the
      // prologue computes); 32 positions: in V buffer 1, which no first copy
      // writes.
      const bool apart = p.hpw_log == 2;
      const int cos0 = apart ? VRING + TILE : 0;
      const StagedTables tab = stage(cos0, cos0 + rows * RB);
      q_prologue<D, PRO, ST, false, true>(p, qoff, qrow, qrow < S, g, qreg, cl, tab, [&]() {
        if (!apart) __syncthreads();  // every wave's table reads have completed
        first_copies();
      });
    } else if (p.hpw_log == 1) {
      // 64 positions: cos in K buffers 2 and 3, sin in V buffers 2 and 3
      const StagedTables tab = stage(2 * TILE, VRING + 2 * TILE);
      first_copies();
      q_prologue<D, PRO, ST, false, true>(p, qoff, qrow, qrow < S, g, qreg, cl, tab);
    } else {
      first_copies();
      q_prologue<D, PRO, ST>(p, qoff, qrow, qrow < S, g, qreg, cl);
    }
  } else if constexpr (PRO == PRO_NORM) {
    first_copies();
    q_prologue<D, PRO, ST>(p, qoff, qrow, qrow < S, g, qreg, cl);
  }
  f32x16_t o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) o[db] = f32x16_t{};
  if constexpr (PRO == PRO_NONE || PRO == PRO_FACTORED_READ || PRO == PRO_FACTORED_CALC) {
    QRows<D, PRO, ST> q;
    if constexpr (R == 4) {
      // Q rows come through LDS, like K: a load straight into the operand layout
      // touches 32 rows and takes the CU's address unit ~64 cycles, a copy of
      // two whole rows 16 (start to Q in registers: 4.9k -> 2.5k cycles).  The
      // wave's 32 rows go to a buffer that no tile needs yet, with the K tiles'
      // chunk swizzle; rows at or past S arrive as zeros.
      const int qbuf = (w & 1) + (w & 2 ? 6 : 2);  // K buffers 2 and 3, V buffers 2 and 3
      const i32x4_t qrs = buffer_rsrc(p.q + qoff * D, head_bytes);
#pragma unroll
      for (int i = 0; i < 16; ++i)
        copy16_to_lds(qrs, lds0 + qbuf * TILE + i * 1024, copy_lane_offset<D>(i, lane, false) + (uint32_t)q0 * RB);
      if constexpr (PRO == PRO_FACTORED_READ) q.load_inv(p, qoff, qrow);
      first_copies();
      pin_acc<ACC>(o);
      asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
#pragma unroll
      for (int c = 0; c < NC; ++c)
        q.raw[c] = *reinterpret_cast<const u32x4_t *>(smem + qbuf * TILE + kra[c & 7] + (c >> 3) * 256);
    } else {
      q.load(p, qoff, qrow, g);
      first_copies();
      pin_acc<ACC>(o);
    }
    q.finish(p, qoff, qrow, g, qreg, cl);
  } else {
    pin_acc<ACC>(o);
  }
  pin_acc<ACC>(qreg);
  // the V ring may start past what an LDS read's immediate offset reaches: its
  // base is part of the address registers
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    vra[e] += lds0 + VRING;
    asm volatile("" : "+v"(vra[e]));
  }

  // Schedule.  Iteration u issues GEMM1 of block u+1 (N1 slots of one MFMA) and
  // GEMM2 of block u (N2 slots) as one stream, with the probabilities, the LDS
  // reads (eight slots ahead of their MFMA) and the copies between them.
  //
  // Copies: set t is the eight copies a wave issues between the barriers of
  // tiles t and t+1: the first C0 right after barrier t, the others spread over
  // the following iteration's MFMAs (each copy occupies the CU's address unit
  // for 16 cycles).
  //   R = 4: set t = K(t+4) into the buffer of K(t) and V(t+3) into that of
  //          V(t-1).  Barrier t (at slot BS of the tile's last block) waits for
  //          set t-2 (K(t+2), V(t+1)); every read of the buffers that set t
  //          refills has been consumed.
  //   R = 2: set t = K(t+3) into the buffer of K(t+1) and V(t+2) into that of
  //          V(t).  Barrier t waits for set t-1 (K(t+2), V(t+1)), and for the
  //          wave's LDS reads: of V(t), and of the second half of K(t+1), which
  //          are issued ahead of it.
  constexpr int N1 = NC, N2 = 2 * NDB, NS = N1 + N2;
  constexpr int BS = R == 4 ? 16 : 14, C0 = R == 4 ? 4 : 2;
  auto set_copy = [&](int t, int pb, int c) {  // copy c of set t; pb = (t - t0) % R
    if constexpr (R == 4) {
      if (c < 4) copy_k1(t + 4, pb, c);
      else copy_v1(t + 3, (pb + 3) % R, c - 4);
    } else {
      if (c < 4) copy_k1(t + 3, (pb + 1) % R, c);
      else copy_v1(t + 2, pb, c - 4);
    }
  };
  auto barrier = [] {
    if constexpr (R == 4) asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

  float m_run = -INFINITY, nm = 0.f;
  float l_run = 0.f, ls[4];  // this lane's share of the row sum: whole tiles, and the chains of the present one
  f32x16_t sa, sb;
  bf16x8_t pb[2], kop[8];
  float x[16], pe[16];

  auto kread = [&](int buf, int sub, auto cc) {  // K operand of chunk c of a block
    constexpr int C = decltype(cc)::value;
    return *reinterpret_cast<const bf16x8_t *>(smem + buf * TILE + sub * 32 * RB + kra[C & 7] + (C >> 3) * 256);
  };
  auto vread = [&](int buf, int sub, auto ii, auto hh) {  // half of the V operand of GEMM2 slot i of a block
    constexpr int I = decltype(ii)::value, C2 = I / NDB, DB = I % NDB, HH = decltype(hh)::value;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_i16x4_t *)(uintptr_t)(vra[DB & 3] +
                                   (uint32_t)(buf * TILE + (32 * sub + 16 * C2) * RB + (DB >> 2) * 256 + HH * 8 * RB)));
  };
  auto vop = [](const i16x4_t &lo, const i16x4_t &hi) {
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  auto mask = [&](f32x16_t &s, int u) {
    const int last = (int)(S - 1);
    const int lim = (CAUSAL ? (qrow < last ? qrow : last) : last) - u * 32 - 4 * g;
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (8 * (i >> 2) + (i & 3) > lim) s[i] = -INFINITY;
  };
  auto pack_pair = [](bf16x8_t &d, auto ii, float v0, float v1) {
    constexpr int I = decltype(ii)::value;
    u32x4_t w4 = __builtin_bit_cast(u32x4_t, d);
    w4[I] = pack_bf16x2(v0, v1);
    d = __builtin_bit_cast(bf16x8_t, w4);
  };

  // The probabilities of a block are computed element by element (register e
  // of the scores; registers 0-7 and 8-15 are its two 16-key steps, in the
  // order of the GEMM2 operands) over T, the slot counted from the start of the
  // iteration that makes the scores (T >= NS: the next iteration, whose GEMM2
  // consumes them): FMA at F, exp2 at F+1, row sum at F+2, BF16 pack of a pair
  // two slots after its second FMA.  The first FMA comes three MFMAs after the
  // scores' last one; a pack comes after the last GEMM2 MFMA that reads the
  // previous block's operand, and slots before the first that reads its own.
  // A tile's row sum is made in four chains and added to l_run once, after its
  // last block (SB), as Softmax::step does: a sweep rounds S / BN + 10 times, where
  // chains over the whole range would round S / 4 times.  The last iteration of
  // a sweep makes probabilities of a block that is not there: no iteration adds
  // that tile's sum, or (second block of a tile) they are masked to zero.
  constexpr int FIRST_F = f_slot<D>(0);
  static_assert(FIRST_F >= N1 + 2 && f_slot<D>(1) + 2 >= N1 + NDB, "scores complete; first operand free");
  static_assert(f_slot<D>(7) + 2 < NS + N1 - 2 && f_slot<D>(15) + 2 < NS + N1 + NDB - 2, "packed before use");
  static_assert(f_slot<D>(15) + 2 - NS < f_slot<D>(0) + 2, "a block's sum ends before the next one's begins");
  auto valu = [&](auto TT, auto sbc, const f32x16_t &s) {
    constexpr int T = decltype(TT)::value, SB = decltype(sbc)::value;
    static_for<0, 16>([&](auto ee) {
      constexpr int e = decltype(ee)::value, F = f_slot<D>(e);
      if constexpr (T == F + 2) {
        if constexpr (SB == 0 && e < 4) ls[e] = pe[e];
        else ls[e & 3] += pe[e];
        if constexpr (SB == SUB - 1 && e == 15) l_run += (ls[0] + ls[1]) + (ls[2] + ls[3]);
        if constexpr (e % 2 == 1) pack_pair(pb[e / 8], std::integral_constant<int, (e % 8) / 2>{}, pe[e - 1], pe[e]);
      }
      if constexpr (T == F + 1) pe[e] = __builtin_amdgcn_exp2f(x[e]);
      if constexpr (T == F) x[e] = __builtin_fmaf(s[e], cl, nm);
    });
  };
  // Pins what lives across a branch after slot T (an empty asm that rewrites
  // it): no later pass may sink its computation past the branch.
  auto pin_valu = [&](auto TT) {
    constexpr int T = decltype(TT)::value;
    static_for<0, 16>([&](auto ee) {
      constexpr int e = decltype(ee)::value, F = f_slot<D>(e), PK = f_slot<D>(e | 1) + 2;
      if constexpr (T == F) pin_reg(x[e]);
      if constexpr (T > F && T < PK) pin_reg(pe[e]);
    });
  };

  // Iteration u = (tile t, block SB of it); PB = (t - t0) % R.  MADE: the scores
  // of block u+1 are there already, masked (the first tile's second block).
  auto full = [&](auto pbc, auto sbc, auto made, int t, f32x16_t &cur, f32x16_t &nxt) __attribute__((always_inline)) {
    constexpr int PB = decltype(pbc)::value, SB = decltype(sbc)::value;
    constexpr bool MADE = decltype(made)::value;
    constexpr bool LAST = SB == SUB - 1;                      // the tile's last block: its barrier
    constexpr int K1B = SB + 1 < SUB ? PB : (PB + 1) % R;     // K of block u+1
    constexpr int K1S = (SB + 1) % SUB;
    constexpr int K2B = (PB + (SB + 2) / SUB) % R, K2S = SB % SUB;  // K of block u+2
    static_assert((SB + 2) % SUB == K2S, "block u + 2");
    const int u = SUB * t + SB;
    bf16x8_t kop2[8];
    i16x4_t vlo[8], vhi[8];
    static_for<0, NS>([&](auto mm) {
      constexpr int m = decltype(mm)::value;
      if constexpr (m == FIRST_F) {
        pin_valu(std::integral_constant<int, m - 1>{});
        pin_valu(std::integral_constant<int, NS + m - 1>{});
        pin_reg(l_run);
        if constexpr (!LAST) {
#pragma unroll
          for (int j = 0; j < 4; ++j) pin_reg(ls[j]);
        }
        pin_reg(pb[1]);
        if constexpr (!MADE) {
          if (u + 1 >= u_mask && (!LAST || u + 1 < nUw)) {
            mfma_settle(nxt);
            mask(nxt, u + 1);
          }
        }
      }
      if constexpr (LAST && m == BS) barrier();
      // ---- MFMA ----
      if constexpr (m < N1) {
        if constexpr (MADE) {
          if constexpr (m == N1 - 1) valu_settle(pb[0]);  // no MFMA since it was packed
        } else if constexpr (m == 0) mfma_s_zero<ACC>(nxt, kop[0], qreg[0]);
        else mfma_s<ACC>(nxt, m < 8 ? kop[m % 8] : kop2[m % 8], qreg[m]);
      } else {
        constexpr int i = m - N1;
        mfma_o<ACC>(o[i % NDB], vop(vlo[i % 8], vhi[i % 8]), pb[i / NDB]);
      }
      // ---- probabilities ----
      valu(std::integral_constant<int, NS + m>{}, sbc, cur);
      valu(mm, std::integral_constant<int, K1S>{}, nxt);
      // ---- LDS reads ----
      if constexpr (N1 == 16 && m < 8) kop2[m] = kread(K1B, K1S, std::integral_constant<int, 8 + m>{});
      if constexpr (m >= N1 - 8 && m < N1 + N2 - 8) {
        constexpr int i = m - (N1 - 8);
        vlo[i % 8] = vread(PB, SB, std::integral_constant<int, i>{}, std::integral_constant<int, 0>{});
        vhi[i % 8] = vread(PB, SB, std::integral_constant<int, i>{}, std::integral_constant<int, 1>{});
      }
      if constexpr (R == 2 && LAST) {  // ahead of the barrier
        if constexpr (m >= 8 && m < 12) {
          constexpr int c = 2 * (m - 8);
          kop[c] = kread(K2B, K2S, std::integral_constant<int, c>{});
          kop[c + 1] = kread(K2B, K2S, std::integral_constant<int, c + 1>{});
        }
      } else if constexpr (m >= NS - 8) {
        kop[m - (NS - 8)] = kread(K2B, K2S, std::integral_constant<int, m - (NS - 8)>{});
      }
      // ---- copies ----
      if constexpr (R == 4) {
        if constexpr (m % 4 == 1 && m < 16) set_copy(t - 1, (PB + R - 1) % R, C0 + m / 4);
        if constexpr (m % 4 == 1 && m > 16) set_copy(t, PB, (m - 16) / 4);
      } else {
        if constexpr (SB == 0 && m % 2 == 1 && m < 12) set_copy(t - 1, (PB + R - 1) % R, C0 + m / 2);
        if constexpr (LAST && m >= 14) set_copy(t, PB, m - 14);
      }
      if constexpr (m == NS - 1) {
        pin_valu(mm);
        pin_reg(l_run);
#pragma unroll
        for (int j = 0; j < 4; ++j) pin_reg(ls[j]);
        pin_reg(pb[0]);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  // Tile t, buffers PB: the wave's blocks, or what keeps it in step with the others.
  auto tile_step = [&](auto pbc, auto first, int t) __attribute__((always_inline)) {
    constexpr int PB = decltype(pbc)::value;
    using NO = std::false_type;
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    auto rest = [&] {
#pragma unroll
      for (int c = C0; c < 8; ++c) set_copy(t - 1, (PB + R - 1) % R, c);
    };
    auto meet = [&] {
      barrier();
#pragma unroll
      for (int c = 0; c < C0; ++c) set_copy(t, PB, c);
    };
    if constexpr (SUB == 2) {
      if (2 * t < nUw) full(pbc, I0{}, first, t, sa, sb);
      else rest();
      if (2 * t + 1 < nUw) full(pbc, I1{}, NO{}, t, sb, sa);
      else meet();
    } else {
      if (t < nUw) {
        if constexpr (PB % 2 == 0) full(pbc, I0{}, NO{}, t, sa, sb);
        else full(pbc, I0{}, NO{}, t, sb, sa);
      } else {
        rest();
        meet();
      }
    }
  };

  // ---- lean sweep: the first tile's maximum is every row's shift, later blocks
  // take p = exp2(logit - shift) and never rescale.  At D = 128 both of the tile's
  // blocks are multiplied first: the maximum of 64 keys rounds P less than that
  // of 32 (error against 64 bits 0.02-0.7% smaller over 20 shapes), for 0.5% of
  // B=32 S=509 and 0.8% of eight layers of Qwen3-0.6B S=128. ----
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // K(t0), K(t0+1), V(t0); every wave has its Q
  if constexpr (R == 4) {
    copy_k(t0 + 2, 2);
    copy_v(t0 + 1, 1);
#pragma unroll
    for (int c = 0; c < C0; ++c) set_copy(t0 - 1, 3, c);
  }
  if (u0 < nUw) {
    bf16x8_t kf[NC];
    static_for<0, NC>([&](auto cc) { kf[decltype(cc)::value] = kread(0, 0, cc); });
    static_for<0, NC>([&](auto cc) {
      constexpr int c = decltype(cc)::value;
      if constexpr (c == 0) mfma_s_zero<ACC>(sa, kf[0], qreg[0]);
      else mfma_s<ACC>(sa, kf[c], qreg[c]);
    });
    static_for<0, 8>([&](auto cc) { kop[decltype(cc)::value] = kread(SUB == 2 ? 0 : 1, SUB - 1, cc); });
  }
  if constexpr (R == 2) {  // every wave has read K(t0)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int c = 0; c < C0; ++c) set_copy(t0 - 1, 1, c);
  }
  if (u0 < nUw) {
    mfma_settle(sa);
    if (u0 >= u_mask) mask(sa, u0);
    float mt[8];
    static_for<0, 8>([&](auto cc) {
      constexpr int c = decltype(cc)::value;
      if constexpr (SUB == 2 && c == 0) mfma_s_zero<ACC>(sb, kop[0], qreg[0]);
      else if constexpr (SUB == 2) mfma_s<ACC>(sb, kop[c], qreg[c]);
      mt[c] = fmaxf(sa[c], sa[8 + c]);
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (SUB == 2) {
      mfma_settle(sb);
      if (u0 + 1 >= u_mask) mask(sb, u0 + 1);  // all of it where the wave has one block
#pragma unroll
      for (int i = 0; i < 8; ++i) mt[i] = fmaxf(mt[i], fmaxf(sb[i], sb[8 + i]));
    }
#pragma unroll
    for (int n = 4; n > 0; n /= 2)
#pragma unroll
      for (int i = 0; i < n; ++i) mt[i] = fmaxf(mt[i], mt[i + n]);
    m_run = max_halves(mt[0]) * cl;
    nm = -m_run;
    static_for<0, NS>([&](auto mm) { valu(mm, std::integral_constant<int, 0>{}, sa); });  // what the slots of iteration u0 - 1 would have computed
  }
  if constexpr (SUB == 2) {
    int t = t0;
    tile_step(std::integral_constant<int, 0>{}, std::true_type{}, t);
    if (++t < nT)
      for (;;) {
        tile_step(std::integral_constant<int, 1>{}, std::false_type{}, t);
        if (++t >= nT) break;
        tile_step(std::integral_constant<int, 0>{}, std::false_type{}, t);
        if (++t >= nT) break;
      }
  } else {
    for (int t = t0;;) {
      tile_step(std::integral_constant<int, 0>{}, std::false_type{}, t);
      if (++t >= nT) break;
      tile_step(std::integral_constant<int, 1>{}, std::false_type{}, t);
      if (++t >= nT) break;
      tile_step(std::integral_constant<int, 2 % R>{}, std::false_type{}, t);
      if (++t >= nT) break;
      tile_step(std::integral_constant<int, 3 % R>{}, std::false_type{}, t);
      if (++t >= nT) break;
    }
  }
  mfma_settle_acc<ACC>(o);
  wait_copies();  // no copy may land in the buffers from here on
  if (SUB == 2 && (nUw & 1)) l_run += (ls[0] + ls[1]) + (ls[2] + ls[3]);  // ended within a tile
  u32x2_t words[D / 8];
  // A shift per row is exact as long as no row sum comes near overflow (each
  // lane's share below 2^64; a finite share alone would not do, as two of them
  // can add up to inf) and no accumulator overflows; otherwise the workgroup
  // redoes the item with the exact online softmax.  The halves of a split item
  // are added at the larger of their shifts: accumulators below 2^126 leave room
  // for that, and a half whose factor flushes to zero (shift 126 or more below)
  // weighs less than 2^-60 of the other.
  bool bad = sum_too_large(l_run);
  if (D != 256 || sid < 0) bad |= pack_rows(o, __fdiv_rn(1.0f, sum_halves(l_run)), words);
  else bad |= any_not_finite<0x7e800000u>(o);
  if (__syncthreads_or(bad)) {
    Softmax<D, BN, CAUSAL> sm;
#pragma unroll
    for (int db = 0; db < NDB; ++db) o[db] = f32x16_t{};
    pin_acc<ACC>(o);
    for (int t = t0; t < nT; ++t) {
      copy_k(t, t & 1);
      copy_v(t, t & 1);
      wait_copies();
      __syncthreads();
      if (SUB * t < nUw) {
        const unsigned char *kt = smem + (t & 1) * TILE;
        f32x16_t s[SUB];
        static_for<0, 16>([&](auto mm) {
          constexpr int m = decltype(mm)::value, kb = m / NC, c = m % NC;
          const bf16x8_t a = *reinterpret_cast<const bf16x8_t *>(kt + kb * 32 * RB + kra[c & 7] + (c >> 3) * 256);
          if constexpr (c == 0) mfma_s_zero<ACC>(s[kb], a, qreg[c]);
          else mfma_s<ACC>(s[kb], a, qreg[c]);
        });
#pragma unroll
        for (int kb = 0; kb < SUB; ++kb) mfma_settle(s[kb]);
        bf16x8_t px[NK16];
        sm.step(s, t, q0, qrow, S, g, cl, o, px);
        pin_acc<ACC>(o);
#pragma unroll
        for (int c2 = 0; c2 < NK16; ++c2) valu_settle(px[c2]);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int c2 = i / NDB, db = i % NDB;
          const uint32_t base = vra[db & 3] + (uint32_t)((t & 1) * TILE + 16 * c2 * RB + (db >> 2) * 256);
          const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t *)(uintptr_t)base);
          const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t *)(uintptr_t)(base + 8 * RB));
          mfma_o<ACC>(o[db], vop(lo, hi), px[c2]);
        }
        mfma_settle_acc<ACC>(o);
      }
    }
    l_run = sm.l_run;
    m_run = sm.m_run;
    if (D != 256 || sid < 0) pack_rows(o, __fdiv_rn(1.0f, sum_halves(l_run)), words);
    __syncthreads();  // the buffers become the epilogue's staging tiles
  }

  unsigned char *tile = smem + w * (32 * RB);
  if (D != 256 || sid < 0) store_packed<D>(tile, p.out + qoff * D, S, q0, lane, words);
  else if constexpr (D == 256)
    split_finish<D>(p, tile, sid * (p.B * p.Hq) + (b * p.Hq + h), t0 > 0 ? 1 : 0, qoff, q0, tid, lane, m_run, l_run, o);
  clock_stamp<true>(p.stamps);
}

template <int D, bool CAUSAL, int PRO, int ST>
hipError_t launch_fwd_t(const AttnParams &p, int blocks, hipStream_t s) {
  constexpr int BN = 8192 / D;
  hipLaunchKernelGGL((attn_fwd_kernel<D, BN, CAUSAL, PRO, ST, false>), dim3(blocks), dim3(256), 0, s, p);
  static const std::string name = [] {
    char b[96];
    snprintf(b, sizeof(b), "attn_fwd_kernel<%d, %d, %s, %d, %d, false>", D, BN, tf(CAUSAL), PRO, ST);
    return std::string(b);
  }();
  launch_log_add(reinterpret_cast<const void *>(&attn_fwd_kernel<D, BN, CAUSAL, PRO, ST, false>), name.c_str(), blocks,
                 256);
  return hipGetLastError();
}

template <int D, bool CAUSAL>
hipError_t launch_fwd_c(const AttnParams &p, int pro, int st, int blocks, hipStream_t s) {
  switch (pro) {
    case PRO_NONE: return launch_fwd_t<D, CAUSAL, PRO_NONE, ST_FP32>(p, blocks, s);
    case PRO_FACTORED_READ: return launch_fwd_t<D, CAUSAL, PRO_FACTORED_READ, ST_FP32>(p, blocks, s);
    case PRO_FACTORED_CALC: return launch_fwd_t<D, CAUSAL, PRO_FACTORED_CALC, ST_FP32>(p, blocks, s);
    case PRO_NORM:
      if (st == ST_HF) return launch_fwd_t<D, CAUSAL, PRO_NORM, ST_HF>(p, blocks, s);
      if (st == ST_LEGACY) return launch_fwd_t<D, CAUSAL, PRO_NORM, ST_LEGACY>(p, blocks, s);
      return launch_fwd_t<D, CAUSAL, PRO_NORM, ST_FP32>(p, blocks, s);
    case PRO_NORM_ROPE:
      if (st == ST_HF) return launch_fwd_t<D, CAUSAL, PRO_NORM_ROPE, ST_HF>(p, blocks, s);
      if (st == ST_LEGACY) return launch_fwd_t<D, CAUSAL, PRO_NORM_ROPE, ST_LEGACY>(p, blocks, s);
      return launch_fwd_t<D, CAUSAL, PRO_NORM_ROPE, ST_FP32>(p, blocks, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace
}  // namespace kfmi
