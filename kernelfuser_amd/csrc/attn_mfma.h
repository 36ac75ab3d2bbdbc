#pragma once
// v_mfma_f32_32x32x16_bf16 as inline assembly, so that each operand sits in
// the register file its kernel needs: scores in VGPRs (the VALU reads them),
// O and the Q operands in AGPRs.  (With the builtin the compiler puts every
// accumulator of a kernel in one file.)  The compiler does not know that these
// are MFMAs, so the kernels keep their dependency distances themselves.  For
// this MFMA on gfx950 the compiler's own hazard rules are: none for an
// accumulation chain on one register, 2 wait states from a VALU write to an
// MFMA operand read, 12 from an MFMA result to any other instruction that
// reads it (and an MFMA source register may be overwritten right after
// issue).  The loops consume an MFMA result only after further MFMAs have
// been issued, and feed VALU results to MFMAs slots later; everywhere else an
// explicit wait (mfma_settle, s_nop) pads the gap, on operands that tie the
// waiting to the registers concerned.
#include <type_traits>

#include "attn_common.h"

namespace kfmi {
namespace {

__device__ __forceinline__ void mfma_v(f32x16_t &d, const bf16x8_t &a, const bf16x8_t &b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "a"(b));
}
__device__ __forceinline__ void mfma_v_from(f32x16_t &d, const bf16x8_t &a, const bf16x8_t &b, const f32x16_t &c) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %3" : "=&v"(d) : "v"(a), "a"(b), "v"(c));
}
__device__ __forceinline__ void mfma_v_zero(f32x16_t &d, const bf16x8_t &a, const bf16x8_t &b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "a"(b));
}
__device__ __forceinline__ void mfma_a(f32x16_t &d, const bf16x8_t &a, const bf16x8_t &b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(d) : "v"(a), "v"(b));
}
// The same with every operand in VGPRs (ACC = false): a kernel whose registers
// all fit there moves nothing between the files.
template <bool ACC>
__device__ __forceinline__ void mfma_s(f32x16_t &d, const bf16x8_t &a, const bf16x8_t &b) {  // scores
  if constexpr (ACC) mfma_v(d, a, b);
  else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
}
template <bool ACC>
__device__ __forceinline__ void mfma_s_zero(f32x16_t &d, const bf16x8_t &a, const bf16x8_t &b) {
  if constexpr (ACC) mfma_v_zero(d, a, b);
  else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
}
template <bool ACC>
__device__ __forceinline__ void mfma_o(f32x16_t &d, const bf16x8_t &a, const bf16x8_t &b) {  // O
  if constexpr (ACC) mfma_a(d, a, b);
  else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
}
// 16 wait states after the last MFMA writing these registers, before any
// other instruction reads them.
__device__ __forceinline__ void mfma_settle(f32x16_t &s) { asm volatile("s_nop 7\n\ts_nop 7" : "+v"(s)); }
__device__ __forceinline__ void mfma_settle(f32x16_t (&s)[2][2]) {
  asm volatile("s_nop 7\n\ts_nop 7" : "+v"(s[0][0]), "+v"(s[0][1]), "+v"(s[1][0]), "+v"(s[1][1]));
}
template <bool ACC = true, int N>
__device__ __forceinline__ void mfma_settle_acc(f32x16_t (&o)[N]) {
  if constexpr (ACC) {
    asm volatile("s_nop 7\n\ts_nop 7" : "+a"(o[0]));
#pragma unroll
    for (int i = 1; i < N; ++i) asm volatile("" : "+a"(o[i]));
  } else {
    asm volatile("s_nop 7\n\ts_nop 7" : "+v"(o[0]));
#pragma unroll
    for (int i = 1; i < N; ++i) asm volatile("" : "+v"(o[i]));
  }
}
// Pins values into AGPRs (VGPRs for ACC = false; the copies the compiler makes
// land before this point), then 2 wait states so that an MFMA may read them next.
template <bool ACC = true, typename T, int N>
__device__ __forceinline__ void pin_acc(T (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if constexpr (ACC) asm volatile("" : "+a"(x[i]));
    else asm volatile("" : "+v"(x[i]));
  }
  asm volatile("s_nop 1");
}
// 2 wait states after VALU writes of an MFMA operand.
template <typename T>
__device__ __forceinline__ void valu_settle(T &x) {
  asm volatile("s_nop 1" : "+v"(x));
}

// An empty asm that rewrites a value: no later pass may move its computation
// past this point.
template <typename T>
__device__ __forceinline__ void pin_reg(T &x) {
  asm volatile("" : "+v"(x));
}

template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// The Q prologue of q_prologue (attn_common.h) for rows that are not normalised,
// in two halves, so that a kernel puts other work into the loads' round trip.
// Rows at or past S load the last row: every load is unconditional and in
// bounds, and what those rows compute is never stored.
template <int D, int PRO, int ST>
struct QRows {
  static constexpr int NC = D / 16;
  static_assert(PRO == PRO_NONE || PRO == PRO_FACTORED_READ || PRO == PRO_FACTORED_CALC, "no norm: q_prologue");
  u32x4_t raw[NC];
  float inv_in;

  __device__ __forceinline__ void load_inv(const AttnParams &p, int64_t qoff, int qrow) {
    inv_in = p.inv[qoff + (qrow < p.S ? qrow : (int)p.S - 1)];
  }
  __device__ __forceinline__ void load(const AttnParams &p, int64_t qoff, int qrow, int g) {
    const int row = qrow < p.S ? qrow : (int)p.S - 1;
    const uint16_t *q = p.q + (qoff + row) * D + 8 * g;
#pragma unroll
    for (int c = 0; c < NC; ++c) raw[c] = ld16(q + 16 * c);
    if constexpr (PRO == PRO_FACTORED_READ) load_inv(p, qoff, qrow);
  }

  // GEMM1 B operands and the lane's logit multiplier.
  __device__ __forceinline__ void finish(const AttnParams &p, int64_t qoff, int qrow, int g, bf16x8_t (&qreg)[NC],
                                         float &cl) const {
    cl = p.c_scale;
#pragma unroll
    for (int c = 0; c < NC; ++c) qreg[c] = as_bf16x8(raw[c]);
    if constexpr (PRO == PRO_FACTORED_READ) cl = inv_in * p.c_scale;  // qk:621
    if constexpr (PRO == PRO_FACTORED_CALC) {
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        float x[8];
        unpack8(raw[c], x);
#pragma unroll
        for (int j = 0; j < 8; ++j) ss = __fmaf_rn(x[j], x[j], ss);
      }
      ss = sum_halves(ss);
      const float inv = rsqrt_rn(ss * (1.0f / D) + p.eps);
      if (p.inv != nullptr && g == 0 && qrow < p.S) p.inv[qoff + qrow] = inv;  // qk:597-601
      cl = inv * p.c_scale;                                                   // qk:621
    }
  }
};

// The epilogue in two halves, for kernels that check O for overflow: pack_rows
// normalises and rounds O into the words of the lane's query row and returns
// whether any accumulator is inf or NaN (v_maximum3 keeps a NaN); store_packed
// writes the wave's 32 rows as store_rows_lds does, with the row guard left to
// the range check of a descriptor over the wave's rows below S.
template <int NDB>
__device__ __forceinline__ bool pack_rows(const f32x16_t (&o)[NDB], float rl, u32x2_t (&w)[4 * NDB]) {
  float m[2] = {0.f, 0.f};
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const float a = o[db][4 * q4], b = o[db][4 * q4 + 1], c = o[db][4 * q4 + 2], d = o[db][4 * q4 + 3];
      m[0] = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m[0], __builtin_fabsf(a)), __builtin_fabsf(b));
      m[1] = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m[1], __builtin_fabsf(c)), __builtin_fabsf(d));
      w[4 * db + q4][0] = pack_bf16x2(a * rl, b * rl);
      w[4 * db + q4][1] = pack_bf16x2(c * rl, d * rl);
    }
  return not_finite(__builtin_elementwise_maximum(m[0], m[1]));
}
template <int D>
__device__ __forceinline__ void store_packed(unsigned char *tile, uint16_t *out, int64_t S, int q0, int lane,
                                             const u32x2_t (&w)[D / 8]) {
  constexpr int RB = 2 * D, CPR = D / 8, RPI = 64 / CPR;
  const int lr = lane & 31, g = lane >> 5;
#pragma unroll
  for (int k = 0; k < CPR; ++k)  // 16-byte chunk k of the row: columns 8k + 4g ..
    *reinterpret_cast<u32x2_t *>(tile + lr * RB + ((k ^ (lr % CPR)) << 4) + 8 * g) = w[k];
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  const int c = lane % CPR, rr = lane / CPR;
  u32x4_t x[32 / RPI];
#pragma unroll
  for (int i = 0; i < 32 / RPI; ++i) {
    const int r = i * RPI + rr;
    x[i] = *reinterpret_cast<const u32x4_t *>(tile + r * RB + ((c ^ (r % CPR)) << 4));
  }
  const int64_t left = S - q0;
  const int rows = left < 0 ? 0 : left < 32 ? (int)left : 32;
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(out + (int64_t)q0 * D, 0, rows * RB, 0x00020000);
#pragma unroll
  for (int i = 0; i < 32 / RPI; ++i)
    __builtin_amdgcn_raw_buffer_store_b128(x[i], rsrc, rr * RB + 16 * c + i * (RPI * RB), 0, 0);
}

}  // namespace
}  // namespace kfmi
