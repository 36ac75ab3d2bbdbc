// The dispatch of launch_attention over the attention kernels, and the general
// kernel's mode 'full' (K normalised tile by tile).  Counterpart of the
// reference's attention_v2_kernel (src/e1_rope_publication_v1.py:608-649) and
// factored_attention_kernel (src/e1_qk_publication_v3.py:612-638).  The
// arithmetic the kernels share (Q prologue, online softmax, MFMA operand
// layouts, LDS staging, epilogue) is in attn_common.h; the general kernel's
// other modes are in attn_fwd.h, the ping-pong kernel in attn_pp.hip, the
// wide-wave kernel in attn_wide.hip.
#include <math.h>

#include <atomic>

#include <cstdio>
#include <string>

#include "attn_common.h"
#include "attn_split.h"

namespace kfmi {
namespace {

// ---------------------------------------------------------------------------
// Mode 'full': K arrives raw and every tile gets the K prologue (FK).  One head,
// 4 waves x 32 rows, GEMM1 of tile t+1 issued ahead of the softmax and GEMM2 of
// tile t, exact online softmax.
// ---------------------------------------------------------------------------
// (FK tells it from the other forms in the name that launch records carry.)
template <int D, int BN, bool CAUSAL, int PRO, int ST, bool FK>
__global__ __launch_bounds__(256, (D == 128 ? 2 : 1)) void attn_fwd_kernel(AttnParams p) {
  static_assert(FK && (PRO == PRO_NORM || PRO == PRO_NORM_ROPE), "the other forms: attn_fwd.h");
  constexpr int BM = 128;            // query rows per workgroup (4 waves x 32)
  constexpr int RB = 2 * D;          // bytes per K/V row
  constexpr int TILE = BN * RB;      // bytes per K or V tile
  constexpr int NINST = TILE / 1024; // 1 KiB copies per tile
  constexpr int LPW = NINST / 4;     // copies per wave per tile
  constexpr int NC = D / 16, NKB = BN / 32, NK16 = BN / 16, NDB = D / 32;
  constexpr int K0 = 0, K1 = TILE, V0 = 2 * TILE, V1 = 3 * TILE;
  static_assert(TILE == 16384 && LPW * 4 == NINST, "tiles are 16 KiB, 4 copies per wave");

  __shared__ __attribute__((aligned(1024))) unsigned char smem[4 * TILE];

  clock_stamp<false>(p.stamps);
  // Two-slot pairing (slot2 > 0): the short causal blocks of the second slot
  // start about 12k cycles late (s_sleep n waits about 64n cycles), so the long
  // blocks of the first, which set the kernel's end, load without that traffic.
  if (CAUSAL && p.slot2 > 0 && (int)blockIdx.x >= p.slot2) {
    __builtin_amdgcn_s_sleep(96);
    __builtin_amdgcn_s_sleep(96);
  }
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;   // half-wave: selects k-group of the MFMA operands
  const int lr = lane & 31;  // query row of this lane within the wave
  const int64_t S = p.S;

  // ---- work item: heaviest query blocks (or split halves) first; KV groups
  // pinned to an XCD ----
  const int nbh = p.B * p.Hq;
  const int bid = blockIdx.x;
  const int rank = bid / nbh;
  const int r = bid - rank * nbh;
  int qb, t0 = 0, t1 = -1, sid = -1;
  if (p.n_items > 0) {
    qb = p.it_qb[rank];
    t0 = p.it_t0[rank];
    t1 = p.it_t1[rank];
    sid = p.it_sid[rank];
  } else if (CAUSAL && p.slot2 > 0 && bid >= p.slot2) {
    qb = (bid - p.slot2) / nbh;
  } else {
    qb = CAUSAL ? p.n_qblocks - 1 - rank : rank;
  }
  const int G = p.Hq / p.Hkv;
  int b, h;
  if (p.xcd_remap) {
    // Workgroups are dispatched round-robin over the 8 XCDs (bid % 8).  Map
    // KV group kg to XCD kg % 8 so the G query heads that read the same K/V
    // share one L2.
    const int xcd = r & 7, jj = r >> 3;
    const int kg = xcd + 8 * (jj / G);
    b = kg / p.Hkv;
    h = (kg - b * p.Hkv) * G + jj % G;
  } else {
    b = r / p.Hq;
    h = r - b * p.Hq;
  }
  const int kvh = h / G;
  const int64_t qoff = ((int64_t)b * p.Hq + h) * S;
  const int64_t kvoff = ((int64_t)b * p.Hkv + kvh) * S;

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
  auto copy_k = [&](int t, int buf) {
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const int inst = w * LPW + i;
      copy16_to_lds(krs, lds0 + buf + inst * 1024, kvo[i] + (uint32_t)(t * TILE));
    }
  };
  auto copy_v = [&](int t, int buf) {
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const int inst = w * LPW + i;
      copy16_to_lds(vrs, lds0 + buf + inst * 1024, vvo[i] + (uint32_t)(t * TILE));
    }
  };

  const int q0 = qb * BM + w * 32;
  const int qrow = q0 + lr;
  const bool qvalid = qrow < S;

  // ---- KV tile range [t0, nT) of this work item ----
  const int64_t kv_end = CAUSAL ? ((int64_t)(qb + 1) * BM < S ? (int64_t)(qb + 1) * BM : S) : S;
  const int nT = t1 >= 0 ? t1 : (int)((kv_end + BN - 1) / BN);
  const int64_t wave_end = CAUSAL ? ((int64_t)q0 + 32 < S ? (int64_t)q0 + 32 : S) : S;
  const int nTw0 = q0 < S ? (int)((wave_end + BN - 1) / BN) : 0;  // tiles with any unmasked key
  const int nTw = nTw0 < nT ? nTw0 : nT;

  uint32_t kra[8], vra[4];
  lds_read_offsets<D>(lane, kra, vra);

  auto first_copies = [&]() {
    copy_k(t0, K0);
    copy_v(t0, V0);
    if (t0 + 1 < nT) copy_k(t0 + 1, K1);
  };
  // Start the first copies before the prologue's own global loads.
  first_copies();
  bf16x8_t qreg[NC];
  float cl;
  q_prologue<D, PRO, ST>(p, qoff, qrow, qvalid, g, qreg, cl);

  f32x16_t o[NDB];
  Softmax<D, BN, CAUSAL> sm;

  // Pipeline (one barrier per KV tile): iteration t issues the copies of
  // K(t+2) and V(t+1), then GEMM1 of tile t+1 and the softmax + GEMM2 of tile
  // t; each copy has a full iteration to land.  PAR = t % 2 selects buffers.
  auto iteration = [&](auto par, int t, f32x16_t (&cur)[NKB], f32x16_t (&nxt)[NKB]) {
    constexpr int PAR = decltype(par)::value;
    constexpr int KNEXT = PAR ? K0 : K1;   // holds K(t+1)
    constexpr int KFREE = PAR ? K1 : K0;   // held K(t), read in the previous iteration
    constexpr int VCUR = PAR ? V1 : V0;    // holds V(t)
    constexpr int VFREE = PAR ? V0 : V1;   // held V(t-1)
    wait_copies();
    __syncthreads();
    if (t + 2 < nT) copy_k(t + 2, KFREE);
    if (t + 1 < nT) copy_v(t + 1, VFREE);
    if (t + 1 < nTw) {
      gemm1_fused_k<D, BN, ST, PRO == PRO_NORM_ROPE>(smem, KNEXT, kra, qreg, nxt, p, (t + 1) * BN, g, lr);
    }
    if (t < nTw) {
      bf16x8_t pb[NK16];
      sm.step(cur, t, q0, qrow, S, g, cl, o, pb);
      gemm2<D, BN>(smem, VCUR, vra, pb, o);
    }
  };
#pragma unroll
  for (int db = 0; db < NDB; ++db) o[db] = f32x16_t{};
  f32x16_t sa[NKB], sb[NKB];
  wait_copies();
  __syncthreads();
  if (t0 < nTw) gemm1_fused_k<D, BN, ST, PRO == PRO_NORM_ROPE>(smem, K0, kra, qreg, sa, p, t0 * BN, g, lr);
  // the first iteration stands by itself: with it in the loop D = 256 ran 1-3%
  // slower (S=1024 171.0 vs 166.8 us, S=200 51.0 vs 47.2, Hq=16 and 8, RoPE)
  iteration(std::integral_constant<int, 0>{}, t0, sa, sb);
  for (int t = t0 + 1; t < nT;) {
    iteration(std::integral_constant<int, 1>{}, t, sb, sa);
    if (++t >= nT) break;
    iteration(std::integral_constant<int, 0>{}, t, sa, sb);
    ++t;
  }

  // direct stores (the kernel runs at the register limit); the host plans
  // splits for D = 256 only (plan_split)
  if (D != 256 || sid < 0) store_rows<D>(p.out + qoff * D, qrow, qvalid, g, sm.l_run, o);
  else
    split_finish<D>(p, smem + w * (32 * 2 * D), sid * nbh + (b * p.Hq + h), t0 > 0 ? 1 : 0, qoff, q0, tid, lane, sm.m_run,
                    sm.l_run, o);
  clock_stamp<true>(p.stamps);
}

template <int D, int BN, bool CAUSAL, int PRO, int ST, bool FK>
const char *fwd_name() {
  static const std::string n = [] {
    char b[96];
    snprintf(b, sizeof(b), "attn_fwd_kernel<%d, %d, %s, %d, %d, %s>", D, BN, tf(CAUSAL), PRO, ST, tf(FK));
    return std::string(b);
  }();
  return n.c_str();
}
template <int D, int BN, bool CAUSAL, int PRO, int ST>
hipError_t launch_t(const AttnParams &p, int kind, int blocks, hipStream_t s) {
  if constexpr (PRO == PRO_NORM || PRO == PRO_NORM_ROPE) {
    if (p.gk) {  // mode 'full': general kernel with the per-tile K prologue
      hipLaunchKernelGGL((attn_fwd_kernel<D, BN, CAUSAL, PRO, ST, true>), dim3(blocks), dim3(256), 0, s, p);
      launch_log_add(reinterpret_cast<const void *>(&attn_fwd_kernel<D, BN, CAUSAL, PRO, ST, true>),
                     fwd_name<D, BN, CAUSAL, PRO, ST, true>(), blocks, 256);
      return hipGetLastError();
    }
  }
  if constexpr (D == 128) {
    if (kind == KFMI_KERNEL_WIDE) return launch_wide(p, CAUSAL, PRO, ST, blocks, s);
    if (kind == KFMI_KERNEL_PINGPONG) return launch_pp(p, CAUSAL, PRO, ST, blocks, s);
  }
  if constexpr (D == 256) return launch_fwd256(p, CAUSAL, PRO, ST, blocks, s);
  else return launch_fwd128(p, CAUSAL, PRO, ST, blocks, s);
}

template <int D, int BN, bool CAUSAL>
hipError_t dispatch_pro(const AttnParams &p, int pro, int st, int kind, int blocks, hipStream_t s) {
  switch (pro) {
    case PRO_NONE: return launch_t<D, BN, CAUSAL, PRO_NONE, ST_FP32>(p, kind, blocks, s);
    case PRO_FACTORED_READ: return launch_t<D, BN, CAUSAL, PRO_FACTORED_READ, ST_FP32>(p, kind, blocks, s);
    case PRO_FACTORED_CALC: return launch_t<D, BN, CAUSAL, PRO_FACTORED_CALC, ST_FP32>(p, kind, blocks, s);
    case PRO_NORM:
      if (st == ST_HF) return launch_t<D, BN, CAUSAL, PRO_NORM, ST_HF>(p, kind, blocks, s);
      if (st == ST_LEGACY) return launch_t<D, BN, CAUSAL, PRO_NORM, ST_LEGACY>(p, kind, blocks, s);
      return launch_t<D, BN, CAUSAL, PRO_NORM, ST_FP32>(p, kind, blocks, s);
    case PRO_NORM_ROPE:
      if (st == ST_HF) return launch_t<D, BN, CAUSAL, PRO_NORM_ROPE, ST_HF>(p, kind, blocks, s);
      if (st == ST_LEGACY) return launch_t<D, BN, CAUSAL, PRO_NORM_ROPE, ST_LEGACY>(p, kind, blocks, s);
      return launch_t<D, BN, CAUSAL, PRO_NORM_ROPE, ST_FP32>(p, kind, blocks, s);
  }
  return hipErrorInvalidValue;
}

// Compute units of the current device (256 on MI355X), cached per device;
// 256 when no device can be queried.  Scheduling only: results never depend
// on it.
int64_t device_cus() {
  static std::atomic<int> cached[64];  // 0: not queried yet (host threads may race; every writer stores the same value)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int v = cached[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    int n = 0;
    v = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
    cached[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

struct PpGrid {
  int hpg;
  int64_t n_qblocks, npairs, items, units;
  bool xcd_remap, persistent;
};

// Geometry of the ping-pong kernel's grid: items of hpg Q heads per wave
// group (two heads x 128 rows for hpg 1, four heads x 64 rows for hpg 2),
// and whether the persistent long/short pairing applies (causal, the pairs
// of every (long, short) item fill all CUs equally, XCD-remapped heads).
PpGrid pp_grid(int64_t B, int64_t Hq, int64_t Hkv, int64_t S, bool causal, int hpg, int64_t cus) {
  PpGrid g;
  const int64_t G = Hq / Hkv;
  g.hpg = hpg;
  g.n_qblocks = (S + 128 / hpg - 1) / (128 / hpg);
  g.npairs = B * Hkv * (G / (2 * hpg));
  g.xcd_remap = (B * Hkv) % 8 == 0 && g.npairs % 8 == 0;
  g.items = g.n_qblocks * g.npairs;
  g.units = g.npairs * ((g.n_qblocks + 1) / 2);
  g.persistent = causal && g.xcd_remap && cus % 8 == 0 && g.units % cus == 0;
  return g;
}

int pp_heads_for(int64_t Hq, int64_t Hkv) {
  const int t = thread_tuning().pp_heads;
  return t ? t : (Hq / Hkv) % 4 == 0 ? 2 : 1;
}

}  // namespace

// Kernel choice by shape, from measurements on MI355X (both sides timed in
// turn, mode 'query', FP32 / HF style).  The ping-pong kernel needs D = 128 and
// an even GQA ratio and runs one 512-thread workgroup per CU; the general
// kernel's two 4-wave workgroups per CU hide each other's Q prologues, so the
// ping-pong kernel is ahead only where its items fill whole rounds of CUs:
// - below 16 query blocks of 128 rows the general kernel runs (B=8 S=1024 95.9 /
//   99.4 vs 97.1 / 102.2 us, B=4 S=1536 94.3 / 96.9 vs 98.2 / 102.9), except
//   causal grids whose persistent pairs give every CU exactly one (long, short)
//   unit (B=4 S=1000 52.2 / 52.8 vs 51.7 / 53.6) of enough tiles to pay for
//   their prologues: B=32 S=128 (one unit of 3 tiles per CU) ran 35.6 vs 37.7
//   us, so at least 8 blocks;
// - from 16 blocks on, non-causal: when the item count is a multiple of the CU
//   count (S=2048 69.6 / 70.6 vs 68.8 / 71.8 us, S=8192 902 / 901 vs 865 / 900);
//   S=3072, 1.5 rounds, 144 / 146 vs 155 / 163;
// - causal: when the persistent pairing applies (S=4096 136.6 / 138.2 vs 129.8 /
//   135.2 us, Qwen3-0.6B S=8192 256.7 / 257.1 vs 238.4 / 246.6; Qwen3-8B S=2048,
//   half the CUs paired, 47.4 / 47.4 vs 55.4 / 57.4), and from 24 blocks also
//   with 1.5 items per CU or more.  The ping-pong kernel leads on unpaired grids
//   of 1.6 to 2 items per CU (S=3328 99.4 / 101.7 vs 97.5 / 100.9, S=3500 109.2 /
//   110.4 vs 105.0 / 109.0, S=3840 124.7 / 127.1 vs 120.5 / 125.4); at 1.5 it trails
//   by 2-4% (S=3072 90.2 / 89.8 vs 92.4 / 92.5, Hq=32 Hkv=16 S=2945 84.5 / 86.2 vs
//   86.5 / 89.7), which the choice published for S=3072 keeps, and on unpaired
//   grids beyond 2 mostly too, which no rule here tells apart yet (S=4500 161.5 /
//   162.6 vs 169.9 / 177.4, S=5000 192 / 194 vs 204 / 212, S=7000 355 / 357 vs 354 /
//   366; B=2 S=3072 156.1 / 156.6 vs 163.9 / 168.4; Hq=64 S=5000 367 / 370 vs 369 /
//   385).  Below 1.5, little fills a CU whose short item has ended and the longest
//   items set the time: Qwen3-0.6B S=3072 (192 items on 256 CUs) 59.5 / 60.4 vs
//   71.8 / 75.8 us, S=4096 (256) 83.7 / 84.0 vs 97.2 / 101.4, S=4500 (288) 100.9 /
//   101.2 vs 112.2 / 117.0; Hq=16 Hkv=4 S=5000 (316) 117.1 / 117.9 vs 126.2 /
//   131.6; heads in plain order (Hq=8 Hkv=2 S=8000, 250) 147 / 148 vs 172 / 180.
// The wide kernel runs only when the tuning overrides ask for it: one wave per
// SIMD issues the softmax's VALU work and the MFMA stream by itself, and it
// measures 5-12% slower than the ping-pong kernel from S=3072 on.
int attention_kernel_by_shape(int64_t B, int64_t Hq, int64_t Hkv, int64_t S, int64_t D, bool causal) {
  const int64_t G = Hq / Hkv;
  const int64_t qb128 = (S + 127) / 128;
  if (D != 128 || G % 2 != 0) return KFMI_KERNEL_GENERAL;
  const int64_t cus = device_cus();
  const PpGrid g = pp_grid(B, Hq, Hkv, S, causal, pp_heads_for(Hq, Hkv), cus);
  if (causal && qb128 >= 24) return 2 * g.items >= 3 * cus ? KFMI_KERNEL_PINGPONG : KFMI_KERNEL_GENERAL;
  const bool paired = causal && g.persistent && thread_tuning().persistent != 1;
  if (qb128 < 16) return paired && g.units == cus && qb128 >= 8 ? KFMI_KERNEL_PINGPONG : KFMI_KERNEL_GENERAL;
  const bool fills = causal ? paired : g.items % cus == 0;
  return fills ? KFMI_KERNEL_PINGPONG : KFMI_KERNEL_GENERAL;
}

const char *attention_tuning_error(int64_t Hq, int64_t Hkv, int64_t D, bool full) {
  const kfmi_tuning &t = thread_tuning();
  const int64_t G = Hq / Hkv;
  const int k = full ? KFMI_KERNEL_GENERAL : t.attn_kernel;
  if (k == KFMI_KERNEL_PINGPONG && (D != 128 || G % 2 != 0))
    return "the ping-pong kernel needs D == 128 and an even Hq/Hkv";
  if (k == KFMI_KERNEL_WIDE && (D != 128 || G % 4 != 0))
    return "the wide kernel needs D == 128 and Hq/Hkv divisible by 4";
  // wherever the ping-pong kernel may run (forced, or chosen by shape)
  const bool pp_possible = k == KFMI_KERNEL_PINGPONG || (k == KFMI_KERNEL_AUTO && D == 128 && G % 2 == 0);
  if (t.pp_heads == 2 && G % 4 != 0 && pp_possible)
    return "four heads per ping-pong item need Hq/Hkv divisible by 4";
  return nullptr;
}

int attention_kernel(int64_t B, int64_t Hq, int64_t Hkv, int64_t S, int64_t D, bool causal, bool full) {
  if (full) return KFMI_KERNEL_GENERAL;
  const int k = thread_tuning().attn_kernel;
  return k != KFMI_KERNEL_AUTO ? k : attention_kernel_by_shape(B, Hq, Hkv, S, D, causal);
}

// Whether mode 'query' prepares Q with K in its first launch (into `out`, which
// the attention launch then reads as prepared Q and overwrites, block by block)
// instead of in the attention prologue.  On a grid of few workgroups the
// prologue's arithmetic is on the critical path of one wave per SIMD (10k cycles
// with RoPE at D = 128, 17k at D = 256), while the preparation launch spreads it
// over every CU; on larger grids the extra pass over Q costs more.  Measured,
// graph-replayed, prologue against preparation, hf and fp32 style:
//   RoPE, D = 128:  16 workgroups (Hq=16 S=128) causal 13.2 vs 11.1 us, 12.6 vs
//     10.9, not causal 12.8 vs 10.7, 11.9 vs 10.4; 64 (Hq=32 S=256) 14.7 vs 13.7,
//     14.0 vs 13.7, not causal 14.5 vs 13.4, 13.6 vs 13.1; 128 (S=512) 18.6 vs
//     18.8, 17.7 vs 18.2, not causal 18.5 vs 18.8, 17.5 vs 18.0;
//   RoPE, D = 256, causal:  16 (Hq=16 S=128) 19.2 vs 14.1, 17.9 vs 13.9; 128 (B=8)
//     22.5 vs 20.0, 21.0 vs 19.7; 160 (S=1280) 45.8 vs 44.2, 44.7 vs 43.9;
//   not causal, whose workgroups are all as long as the longest:  128 (S=1024)
//     40.3 vs 38.6, 37.9 vs 37.2; 144 (S=1152) 42.4 vs 40.7, 40.9 vs 41.4; 160
//     46.2 vs 47.2, 44.6 vs 46.0;
//   no RoPE, D = 128: 32 workgroups causal 11.6 vs 11.0, 11.3 vs 11.0, not causal
//     11.1 vs 10.7, 10.7 vs 10.6; 64: 13.6 vs 13.5, 13.2 vs 13.4, not causal 13.1
//     vs 13.1, 12.7 vs 12.9; D = 256: 64 workgroups 27.3 vs 26.0, 26.5 vs 25.7, not
//     causal 24.3 vs 23.0, 23.3 vs 22.3; 96: 31.4 vs 31.1, 30.0 vs 30.4, not
//     causal 30.4 vs 30.4, 28.8 vs 29.6.
bool query_prepares_q(int64_t B, int64_t Hq, int64_t Hkv, int64_t S, int64_t D, bool causal, bool rope) {
  if (attention_kernel(B, Hq, Hkv, S, D, causal, false) != KFMI_KERNEL_GENERAL) return false;
  const int64_t wgs = B * Hq * ((S + 127) / 128), cus = device_cus();
  if (D == 128) return wgs <= (rope ? cus / 4 : cus / 8);
  return wgs <= (!rope ? cus / 4 : causal ? cus * 5 / 8 : cus / 2);
}

}  // namespace kfmi

namespace kfmi {

namespace {


// Split-KV plan for the general kernel at D = 256, which runs one workgroup
// per CU: with fewer work items than CUs, longest-first ordering cannot
// balance a causal grid (the heaviest query block alone sets the time, and
// no co-resident workgroup fills the gap).  Blocks with more key tiles than
// half the maximum are then split into two halves of their key range (the
// second holds the diagonal), and all items are listed longest first.
// Measured (attention alone, causal, split against unsplit): Gemma-3-4B S=2048
// 33.6 vs 45.6 us, S=1024 22.2 vs 26.1, S=512 17.3 vs 16.6; a merge costs about
// 4.5 us, so blocks of up to 8 key tiles stay whole (S=256 14.2 vs 11.6 us),
// except in mode 'full', whose tiles cost several times as much (S=200 Hq=8 71.0
// vs 51.0 us with RoPE, 39.1 vs 31.8 without).
// A grid that already fills every CU (Gemma-3-12B S=2048, 256 workgroups) loses
// by splitting, so the plan needs fewer query blocks than CUs (Gemma-3-12B
// S=1536, 192 blocks: 36.8 vs 37.8 us).  At D = 128 two workgroups share each
// CU and one already keeps it nearly busy, so the extra prologues of a split
// cost more than the balance gains.

// Workspace layout: a counter region of the same size for every shape (one
// 4-byte arrival counter per split (block, head) pair, at most
// SPLIT_MAX_PAIRS; a plan has fewer than B*Hq*nqb < CUs pairs), then the
// partial results.  Because no shape's partials ever land in the counter
// region and every launch leaves the counters it used at zero, a workspace
// zero-filled once stays valid for any sequence of shapes launched on it.
constexpr int64_t SPLIT_MAX_PAIRS = 1024;
constexpr int64_t SPLIT_COUNTER_BYTES = SPLIT_MAX_PAIRS * 4;

struct SplitPlan {
  int n_items = 0, n_split = 0;
  int16_t qb[MAX_SPLIT_ITEMS], t0[MAX_SPLIT_ITEMS], t1[MAX_SPLIT_ITEMS], sid[MAX_SPLIT_ITEMS];
};

bool plan_split(int64_t B, int64_t Hq, int64_t S, int64_t D, bool causal, bool full, int64_t cus, SplitPlan &pl) {
  const int64_t BM = 128, BN = D == 128 ? 64 : 32;
  const int64_t nqb = (S + BM - 1) / BM;
  if (D != 256 || !causal || nqb < 2 || B * Hq * nqb >= cus) return false;
  auto tiles = [&](int64_t qb) { return ((qb + 1) * BM < S ? (qb + 1) * BM : S) + BN - 1; };
  const int64_t t_max = tiles(nqb - 1) / BN;
  if (t_max <= 8 && !full) return false;
  const int64_t half = (t_max + 1) / 2;
  struct Item { int qb, t0, t1, sid; };
  Item items[MAX_SPLIT_ITEMS];
  int n = 0, n_split = 0;
  for (int64_t qb = 0; qb < nqb; ++qb) {
    const int nt = (int)(tiles(qb) / BN);
    if (nt > half) {
      if (n + 2 > MAX_SPLIT_ITEMS) return false;
      const int mid = (nt + 1) / 2;
      items[n++] = {(int)qb, 0, mid, n_split};
      items[n++] = {(int)qb, mid, nt, n_split};
      ++n_split;
    } else {
      if (n + 1 > MAX_SPLIT_ITEMS) return false;
      items[n++] = {(int)qb, 0, nt, -1};
    }
  }
  if (n_split == 0 || n_split * B * Hq > SPLIT_MAX_PAIRS) return false;
  // longest first (insertion sort: n <= 128)
  for (int i = 1; i < n; ++i)
    for (int j = i; j > 0 && items[j].t1 - items[j].t0 > items[j - 1].t1 - items[j - 1].t0; --j) {
      const Item t = items[j]; items[j] = items[j - 1]; items[j - 1] = t;
    }
  pl.n_items = n;
  pl.n_split = n_split;
  for (int i = 0; i < n; ++i) {
    pl.qb[i] = (int16_t)items[i].qb; pl.t0[i] = (int16_t)items[i].t0;
    pl.t1[i] = (int16_t)items[i].t1; pl.sid[i] = (int16_t)items[i].sid;
  }
  return true;
}

int64_t split_partial_bytes(int64_t pairs, int64_t D) { return pairs * 2 * (D / 2 + 2) * 256 * 4; }

}  // namespace

int64_t attention_workspace_bytes(int64_t B, int64_t Hq, int64_t Hkv, int64_t S, int64_t D, bool causal, bool full) {
  SplitPlan pl;
  if (!plan_split(B, Hq, S, D, causal, full, device_cus(), pl)) return 0;
  const int64_t pairs = (int64_t)pl.n_split * B * Hq;
  return SPLIT_COUNTER_BYTES + split_partial_bytes(pairs, D);
}

int64_t attention_workspace_counter_bytes(int64_t B, int64_t Hq, int64_t Hkv, int64_t S, int64_t D, bool causal,
                                          bool full) {
  SplitPlan pl;
  if (!plan_split(B, Hq, S, D, causal, full, device_cus(), pl)) return 0;
  return SPLIT_COUNTER_BYTES;
}

namespace {

// Q heads of one GQA group that a workgroup of the general kernel takes (log2):
// as many as divide the group, up to four at D = 128 and two at D = 256, each
// with its share of the 128 query rows.  With fewer positions the workgroup
// stages fewer rotary-table rows (at D = 256 that is what lets it stage them at
// all), no wave idles while a neighbour runs key blocks past its own diagonal,
// and the causal grid is finer: Gemma-3-12B B=8 S=512 57.4 -> 53.0 us,
// Qwen3-8B B=1 S=2048 47.3 -> 46.8, B=8 S=512 not causal 52.3 -> 51.3.  Without
// tables to stage, grids of up to one workgroup per CU lose 1-2% (eight layers
// of Qwen3-0.6B S=128 88.8 vs 89.7 us) and keep one head.
int heads_per_workgroup_log(int64_t G, int64_t D, bool rope, int64_t wgs, int64_t cus) {
  if (!rope && wgs <= cus) return 0;
  if (D == 128 && G % 4 == 0) return 2;
  return G % 2 == 0 ? 1 : 0;
}
// Grids of at least this many workgroups per CU list the query blocks of one KV
// head after the other (longest first within the head), so that the workgroups
// running at one time share few heads' K and V in each L2; below, all heads'
// longest blocks come first, for balance.  Qwen3-8B B=32 S=509 (16 per CU) 162
// -> 152 us, B=29 S=239 not causal 68.6 -> 61.5; Gemma-3-12B B=8 S=512 (2 per
// CU) would go from 49.9 to 56.5.
constexpr int64_t HEAD_MAJOR_WGS_PER_CU = 4;

}  // namespace

hipError_t launch_attention(const AttnArgs &a, hipStream_t stream) {
  constexpr double LOG2E = 1.4426950408889634;
  AttnParams p;
  p.n_items = 0;
  p.pp_units = 0;
  p.pp_hpg = 1;
  p.slot2 = 0;
  p.counters = nullptr;
  p.partials = nullptr;
  p.stamps = nullptr;
  p.q = a.q; p.k = a.k; p.v = a.v; p.gq = a.gq; p.cos = a.cos; p.sin = a.sin;
  p.gk = a.gk;
  p.out = a.out; p.inv = a.inv;
  p.vt = nullptr;
  p.S = a.S;
  p.B = (int)a.B; p.Hq = (int)a.Hq; p.Hkv = (int)a.Hkv;
  p.eps = a.eps;
  const bool factored = a.prologue == PRO_FACTORED_READ || a.prologue == PRO_FACTORED_CALC;
  // rope:636 SCALE*log2e; qk:621 D**-.5*log2e (both formed in double, then FP32)
  p.c_scale = (float)((factored ? 1.0 / sqrt((double)a.D) : a.scale) * LOG2E);
  const int BM = 128;
  p.n_qblocks = (int)((a.S + BM - 1) / BM);
  const kfmi_tuning &tun = thread_tuning();
  const int kind = attention_kernel(a.B, a.Hq, a.Hkv, a.S, a.D, a.causal, a.gk != nullptr);
  if (kind == KFMI_KERNEL_PINGPONG && a.vt && a.S % 8 == 0) p.vt = a.vt;  // V^T rows must be 16-byte aligned
  int blocks, n_split = 0;
  if (kind == KFMI_KERNEL_PINGPONG || kind == KFMI_KERNEL_WIDE) {
    // items of hpg Q heads per wave group: the wide kernel's four heads x 64
    // rows, or the ping-pong kernel's two heads x 128 rows (hpg 1) or four x
    // 64 (hpg 2)
    const int64_t cus = device_cus();
    const PpGrid g = pp_grid(a.B, a.Hq, a.Hkv, a.S, a.causal, kind == KFMI_KERNEL_WIDE ? 2 : pp_heads_for(a.Hq, a.Hkv),
                             cus);
    p.pp_hpg = g.hpg;
    p.n_qblocks = (int)g.n_qblocks;
    p.xcd_remap = g.xcd_remap ? 1 : 0;
    blocks = (int)g.items;
    // persistent mode when the (long, short) pairs fill every CU equally
    if (g.persistent && tun.persistent != 1) {
      p.pp_units = (int)g.units;
      blocks = (int)cus;
    }
  } else {
    const int nbh = p.B * p.Hq;
    p.xcd_remap = (p.B * p.Hkv) % 8 == 0 ? 1 : 0;
    blocks = p.n_qblocks * nbh;
    SplitPlan pl;
    if (a.work && tun.split != 1 && plan_split(a.B, a.Hq, a.S, a.D, a.causal, a.gk != nullptr, device_cus(), pl)) {
      const int64_t pairs = (int64_t)pl.n_split * nbh;
      if (a.work_bytes >= SPLIT_COUNTER_BYTES + split_partial_bytes(pairs, a.D)) {
        n_split = pl.n_split;
        p.n_items = pl.n_items;
        for (int i = 0; i < pl.n_items; ++i) {
          p.it_qb[i] = pl.qb[i]; p.it_t0[i] = pl.t0[i]; p.it_t1[i] = pl.t1[i]; p.it_sid[i] = pl.sid[i];
        }
        p.counters = (int *)a.work;
        p.partials = (float *)((char *)a.work + SPLIT_COUNTER_BYTES);
        blocks = pl.n_items * nbh;
      }
    }
    p.hpw_log = a.gk || p.n_items > 0 ? 0 : heads_per_workgroup_log(a.Hq / a.Hkv, a.D, a.prologue == PRO_NORM_ROPE, blocks, device_cus());
    p.groups = (int)(a.Hq / a.Hkv) >> p.hpw_log;
    p.units = p.B * p.Hkv * p.groups;
    if (p.n_items == 0) {
      const int64_t rows = 128 >> p.hpw_log;
      p.n_qblocks = (int)((a.S + rows - 1) / rows);
      blocks = p.n_qblocks * p.units;
    }
    p.by_units = FastDiv::of((uint32_t)p.units);
    p.by_groups = FastDiv::of((uint32_t)p.groups);
    p.by_hkv = FastDiv::of((uint32_t)a.Hkv);
    p.by_kv_wgs = FastDiv::of((uint32_t)(p.groups * p.n_qblocks));
    p.head_major = a.gk == nullptr && p.n_items == 0 && p.xcd_remap && blocks >= HEAD_MAJOR_WGS_PER_CU * device_cus() ? 1 : 0;
    // D = 128, causal, all workgroups resident in one round of two per CU:
    // pair each CU's long block with a short one (the heads stay the same,
    // as bid and bid + cus map to the same heads when cus % units == 0)
    const int64_t cus = device_cus();
    if (a.causal && a.D == 128 && p.n_items == 0 && cus % p.units == 0 && blocks > cus && blocks <= 2 * cus)
      p.slot2 = (int)cus;
  }
  if (tun.clock_stamps) {
    void *st = nullptr;
    const hipError_t se = clock_stamp_buffer(&st);
    if (se != hipSuccess) return se;
    p.stamps = (unsigned long long *)st;
    clock_stamps_recorded(blocks);
  }
  hipError_t e;
  if (a.D == 128) {
    e = a.causal ? dispatch_pro<128, 64, true>(p, a.prologue, a.style, kind, blocks, stream)
                 : dispatch_pro<128, 64, false>(p, a.prologue, a.style, kind, blocks, stream);
  } else {
    e = a.causal ? dispatch_pro<256, 32, true>(p, a.prologue, a.style, KFMI_KERNEL_GENERAL, blocks, stream)
                 : dispatch_pro<256, 32, false>(p, a.prologue, a.style, KFMI_KERNEL_GENERAL, blocks, stream);
  }
  if (kind == KFMI_KERNEL_PINGPONG || kind == KFMI_KERNEL_WIDE)
    launch_log_plan("hpg=%d persistent=%d xcd=%d", p.pp_hpg, p.pp_units > 0 ? 1 : 0, p.xcd_remap);
  else
    launch_log_plan("split=%d pair=%d xcd=%d heads=%d", n_split, p.slot2 > 0 ? 1 : 0, p.xcd_remap, 1 << p.hpw_log);
  return e;
}

}  // namespace kfmi
