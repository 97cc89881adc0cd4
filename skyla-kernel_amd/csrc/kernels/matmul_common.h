// What the prefill matmul tiles share (matmul.hip, matmul_ring.hip): the push words, raw weight
// stages and their scales, and the loads that write LDS themselves.
#pragma once
#include "common.h"

namespace {

struct MatmulPush {  // 13 words (graph.rs:27-32, graph/moe.rs:26-40)
  uint32_t o0, o1, o2, o3, x_off, y_off, n_in, n_out, x_stride, y_stride, table_off, list_off,
      x_div;
};

SK_DEV f16x2 splat(f16 v) {
  f16x2 r = {v, v};
  return r;
}

// Raw weight bytes of one row for one 256-k stage, held by each lane.
template <int TYPE>
struct WStage;

template <>
struct WStage<1> {  // Q4_K: 128 B qs + 16 B header
  uint4 qs[8];
  uint4 hd;
};
template <>
struct WStage<2> {  // Q6_K: ql 128 B, qh 64 B, 16 scales, d
  uint4 ql[8];
  uint4 qh[4];
  uint4 sc;
  uint32_t d;
};
template <>
struct WStage<0> {  // Q8_0: 8 blocks of 32 quants + 8 scales
  uint4 q[16];
  uint32_t d[8];
};

// Scale (and negated min) of lane half hh at step t, as f16 pairs.  The f32 products
// d*sc and dmin*m are the reference's d0 / min0 (quant.rs:60-61), rounded once to f16.
template <int TYPE>
SK_DEV void step_scale(const WStage<TYPE> &s, int t, uint32_t hh, f16x2 &scale, f16x2 &negmin) {
  if constexpr (TYPE == 1) {
    const uint32_t j = 2 * (t >> 2) + hh;
    uint32_t sc, m;
    q4k_scale_min(j, s.hd.y, s.hd.z, s.hd.w, sc, m);
    const float d = f16_bits_to_f32(s.hd.x & 0xffffu);
    const float dmin = f16_bits_to_f32(s.hd.x >> 16);
    // high nibbles arrive as 16q: fold the 1/16 into the scale
    const float sc_f = d * (float)sc * (hh ? 0.0625f : 1.0f);
    scale = splat((f16)sc_f);
    negmin = splat((f16)(-(dmin * (float)m)));
  } else if constexpr (TYPE == 2) {
    const int hf = t >> 3, g = (t >> 1) & 3;
    const uint32_t k = 8 * hf + (t & 1) + 2 * g;
    const uint32_t wv = k < 4 ? s.sc.x : (k < 8 ? s.sc.y : (k < 12 ? s.sc.z : s.sc.w));
    const int sc = (int)(int8_t)((wv >> (8 * (k & 3))) & 255u);
    const float d = f16_bits_to_f32(s.d);
    scale = splat((f16)(d * (float)sc * (g >= 2 ? 0.0625f : 1.0f)));
    negmin = splat((f16)0.0f);
  } else {
    scale = splat(__builtin_bit_cast(f16, (uint16_t)s.d[t >> 1]));
    negmin = splat((f16)0.0f);
  }
}

// f16 range guard: rows reaching |x| = tm are held as x 2^-e, e putting tm below 2^15.
SK_DEV int range_exp(float tm) {
  return tm >= 32768.0f ? (int)((__builtin_bit_cast(uint32_t, tm) >> 23) & 255u) - 127 - 14 : 0;
}
// The same for each E_RUN values of a row (Q8_0 rows, whose tile rescales its sums between runs:
// one exponent for a row would flush what lies 2^29 below its largest).  v: four values per lane,
// 32 lanes a run.
constexpr uint32_t E_RUN = 128;
SK_DEV int run_exp(const float4 &v) {
  float m = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
#pragma unroll
  for (int d = 16; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
  return range_exp(m);
}

// 16 B unit slot swizzle of a direct-to-LDS row (128 B rows, 8 units): distinct banks for 16
// consecutive rows in a 256 B bank line and for 8 in a 128 B one
SK_DEV uint32_t dl_swz(uint32_t r) { return (r & 7u) ^ ((r >> 3) & 1u); }
typedef __attribute__((address_space(3))) void dl_lds;
// vmcnt(N), the other counters unconstrained (gfx9 s_waitcnt encoding).  The empty statement keeps
// the reads of what the loads wrote behind the wait: where a wave reads its own loads alone no
// barrier stands between them, and the builtin by itself claims no effect on memory.
template <int N>
SK_DEV void dl_wait_vm() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
  asm volatile("" ::: "memory");
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Buffer resource words over [base, base + bytes) (as buf_res builds them: stride 0, raw
// 32-bit data), for the loads below, which take it as an SGPR quad.
SK_DEV u32x4 dl_res(const void *base, uint64_t bytes) {
  const uint64_t a = (uint64_t)base;
  u32x4 r = {(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, (uint32_t)(bytes < 0xffffffffull ? bytes : 0xffffffffull),
             0x00020000u};
  return r;
}
// One 16 B-per-lane buffer load into LDS: lane l's 16 B land at byte lds + 16 l (wave-
// uniform lds, in M0); a load past the resource's end writes zeros.  Written as assembly on
// purpose: with the compiler's own form of this load, every later LDS read waits until all
// such loads in flight are done (the compiler cannot tell which LDS bytes they write),
// which serialises the double buffering; here the explicit waits of dl_stage order each
// buffer's loads before its reads, and the compiler's own waits (it does not count these
// loads) can only wait longer than needed, never less.
// (m0 is declared clobbered; the compiler warns that it reserves m0, which these kernels
// use for nothing else)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
SK_DEV void dl_load16(const u32x4 &res, uint32_t lds, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(lds), "v"(voff), "s"(res), "s"(soff)
               : "memory", "m0");
}
#pragma clang diagnostic pop
SK_DEV uint32_t lds_addr(const void *p) { return (uint32_t)(uintptr_t)(dl_lds *)p; }

}  // namespace
