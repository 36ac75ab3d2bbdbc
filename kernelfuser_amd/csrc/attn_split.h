#pragma once
// The end of a split-KV work item at D = 256 (attn_fwd.h, and mode 'full' in
// attention.hip).
#include "attn_common.h"

namespace kfmi {
namespace {

// One half of a split query block: publish the partial state (O relative to
// m_run, the lane's row-sum share, m_run); the half that finishes second reads
// the other's, merges and stores, and re-arms the counter.  Slot layout
// (floats): O quad q of thread tid at [(q * 256 + tid) * 4], m_run at
// [NQ * 1024 + tid], l_run after it.
//
// The slots are written and read with agent-coherent accesses (cache
// policy SC1, what the compiler gives agent-scope atomic accesses on
// gfx950): a store that has completed (vmcnt) is visible to SC1 loads on
// any XCD.  That orders the handover through the counter without the L2
// writeback and invalidate that a device-scope fence costs.
//
// `pair` is the (split block, head) pair, `part` 0 or 1, `tile` the wave's
// staging tile of 32 rows in LDS.
template <int D>
__device__ __forceinline__ void split_finish(const AttnParams &p, unsigned char *tile, int pair, int part, int64_t qoff,
                                             int q0, int tid, int lane, float m_run, float l_run,
                                             f32x16_t (&o)[D / 32]) {
  constexpr int NQ = D / 32 * 4;
  constexpr int SLOT = (NQ * 4 + 2) * 256;  // floats
  constexpr int SC1 = 16;
  pair = __builtin_amdgcn_readfirstlane(pair);  // wave-uniform: keeps the descriptors in SGPRs
  const auto mine =
      __builtin_amdgcn_make_buffer_rsrc(p.partials + (int64_t)(2 * pair + part) * SLOT, 0, SLOT * 4, 0x00020000);
  const auto other =
      __builtin_amdgcn_make_buffer_rsrc(p.partials + (int64_t)(2 * pair + 1 - part) * SLOT, 0, SLOT * 4, 0x00020000);
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const f32x4_t v = {o[q / 4][(q % 4) * 4], o[q / 4][(q % 4) * 4 + 1], o[q / 4][(q % 4) * 4 + 2],
                       o[q / 4][(q % 4) * 4 + 3]};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), mine, tid * 16, q * 4096, SC1);
  }
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, m_run), mine, (NQ * 1024 + tid) * 4, 0, SC1);
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, l_run), mine, (NQ * 1024 + 256 + tid) * 4, 0,
                                        SC1);
  wait_copies();  // every store of this thread has completed
  __syncthreads();
  __shared__ int arrived_before;
  if (tid == 0) {
    // Release/acquire at agent scope around the arrival counter (the
    // memory model's own mapping: L2 writeback before, invalidate after), so
    // the handover is ordered even where the SC1 accesses alone would not
    // be; one thread per workgroup, after the barrier that follows every
    // thread's completed stores.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    arrived_before = atomicAdd(p.counters + pair, 1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
  if (arrived_before == 0) return;  // the other half merges
  // Merge in fixed (first half, second half) operand order, whichever half
  // runs it, with explicit fmaf, so the result does not depend on timing.
  const float mo = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(other, (NQ * 1024 + tid) * 4, 0, SC1));
  const float lo =
      __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(other, (NQ * 1024 + 256 + tid) * 4, 0, SC1));
  // Every load of a half is issued before the first is waited for (they miss
  // every cache): left to itself the compiler loads and merges one quad at a
  // time, 32 round trips.  Gemma-3-4B, B=1 causal, attention alone: S=1024
  // 30.2 -> 22.2 us, S=2048 40.8 -> 33.6 us.
  constexpr int NB = 16;  // quads in flight
  float a0 = 0.f, a1 = 0.f;
#pragma unroll
  for (int b0 = 0; b0 < NQ; b0 += NB) {
    u32x4_t v[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) v[q] = __builtin_amdgcn_raw_buffer_load_b128(other, tid * 16, (b0 + q) * 4096, SC1);
    __builtin_amdgcn_sched_barrier(0);
    if (b0 == 0) {
      const float m0 = part == 0 ? m_run : mo, m1 = part == 0 ? mo : m_run;
      const float m = fmaxf(m0, m1);
      // rows past S may hold -inf maxima in both halves; they are not stored
      a0 = m0 == m ? 1.0f : __builtin_amdgcn_exp2f(m0 - m);
      a1 = m1 == m ? 1.0f : __builtin_amdgcn_exp2f(m1 - m);
    }
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const f32x4_t vq = __builtin_bit_cast(f32x4_t, v[q]);
      const int n = b0 + q;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float r = o[n / 4][(n % 4) * 4 + k];
        const float x0 = part == 0 ? r : vq[k], x1 = part == 0 ? vq[k] : r;
        o[n / 4][(n % 4) * 4 + k] = fmaf(x0, a0, x1 * a1);
      }
    }
  }
  const float l0 = part == 0 ? l_run : lo, l1 = part == 0 ? lo : l_run;
  __syncthreads();
  store_rows_lds<D>(tile, p.out + qoff * D, q0, p.S, lane, fmaf(l0, a0, l1 * a1), o);
  if (tid == 0) atomicExch(p.counters + pair, 0);
}

}  // namespace
}  // namespace kfmi
