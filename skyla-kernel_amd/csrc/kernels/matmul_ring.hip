// Dense prefill matmul on f16 rows: a tile with a ring of activation chunks and an explicit
// instruction order.
//
// Workgroup: WR waves over rows times WK groups of them over K; a wave owns 32 rows and all
// 32 NB tokens of the tile, so each dequantised weight fragment feeds NB MFMAs.  K groups take
// consecutive runs of super-blocks and their sums meet in LDS, neighbours first; the splits of a
// launch meet in global memory, in order.  K in two parts gives the same bits either way, and so
// do quarters and two splits of halves; four splits add up in another order.
//
// Operands go from global memory straight into LDS (dl_load16), 64 k at a time:
//   activations  f16 rows of x_half_rows, 128 B per token and chunk, 16 B units XOR-swizzled
//                (dl_swz), shared by the WR waves of a K group
//   weights      private to the wave that owns the rows (no barrier orders them)
//     Q4_K  32 B of qs per row and chunk at 32 r, headers 16 B per row and super-block
//     Q6_K  per 128 k: ql 64 B at 64 r (units ^ (r >> 2) & 3), qh 32 B (units ^ (r >> 3) & 1);
//           scales 16 B, and the 16 B around the row's d, per super-block
//     Q8_0  64 B of quants per row and chunk at 64 r (units ^ (r >> 2) & 3); the two 16 B pieces
//           that hold the row's eight d (2 B-aligned), per 256 k
// Exponents (|x| reaching 2^15): rows of K-quant matrices have one each, by which the sums are
// scaled at the end.  Rows of Q8_0 matrices have one per 128 values (x_half_rows's e_off): a tile
// that holds such a row (e[t] nonzero) keeps its sums in units of the current run's, rescaled
// between the runs by powers of two.  (One exponent a row flushed what lay 2^29 below the row's
// largest; the runs' cost 0.3 us of a launch that has none.)
// Chunk c + DX - 1 is requested in the second half of chunk c; the one wait and barrier of a
// chunk stand in its middle: after them chunk c + 1 is in LDS, so the last step's MFMAs run
// with the first fragments of the next chunk on their way, and the buffer of chunk c - 1 is
// free.  Chunks past the last are requested through a resource of no bytes (zeros, no memory
// access), so every wait counts the same loads.
//
// What bounds a wave is the order of its instructions: it issues one per 4 cycles, an MFMA
// holds the matrix unit for 32, and a chunk (16 MFMAs at NB = 4) takes about 60 vector, 25
// LDS and 40 scalar instructions more.  Left to itself the compiler put a step's
// dequantisation after its MFMAs and the chunk's loads in one run; here each MFMA is followed
// by one LDS read and a few of the next step's vector instructions (a scheduling barrier
// after each group, the values pinned so that they are not moved to their use).  Gate and up
// of Qwen3-8B at M = 128 (24576 rows, n_in 4096, weights from HBM), us a launch: the eight-wave
// 128 x 128 tile 60.1 (429 TFLOP/s), its four-wave form 50.9, this tile without the order 56.6,
// with it 37.3 (690 TFLOP/s) on a ring of four chunks; 41 on five to seven, 48 on three.  Timing copies put the rest at 0.45 us
// a chunk against 0.26 of MFMAs, plus 8 us a launch for its start, first loads and stores.
// Seven Q8_0 products of a Qwen3-0.6B layer at M = 200: 458 -> 75 us (they had 8 to 48
// workgroups, each summing all of K).
#include "matmul_common.h"

namespace {

template <int N>
struct IC {
  static constexpr int v = N;
};

template <int TYPE>
struct RingW;  // DMA instructions (1 KiB each) of a wave's weight buffer and of its scales per super-block
template <>
struct RingW<1> {
  static constexpr int WI = 1, HI = 1;
};
template <>
struct RingW<2> {
  static constexpr int WI = 3, HI = 1;
};
template <>
struct RingW<0> {
  static constexpr int WI = 2, HI = 1;
};
// weight buffers of a wave: one per chunk in the ring (Q6_K: per 128 k)
template <int TYPE, int DX>
constexpr int ring_nw() { return TYPE == 2 ? DX / 2 + 1 : DX; }
template <int TYPE, int WR, int WK, int NB, int DX>
constexpr uint32_t ring_lds() {
  const uint32_t x = WK * DX * NB * 4096u;
  const uint32_t w = WR * WK * 1024u * (ring_nw<TYPE, DX>() * RingW<TYPE>::WI + 2u * RingW<TYPE>::HI);
  const uint32_t red = WK > 1 ? WR * WK * NB * 4096u : 0u;  // the K groups' sums, after the loop
  return x + w > red ? x + w : red;
}
// does chunk c (mod 4) bring weights (Q6_K: every second) / the next super-block's scales?
template <int TYPE>
constexpr int ring_wi(int c) { return TYPE == 2 && (c & 1) ? 0 : RingW<TYPE>::WI; }
// loads of a wave in flight behind chunk c + 1 at the wait of chunk c: chunks c + 2 .. c + DX - 2
template <int TYPE>
constexpr int ring_fly(int c, int dx, int xi) {
  int n = 0;
  for (int i = 2; i <= dx - 2; i++) n += xi + ring_wi<TYPE>(c + i) + (((c + i) & 3) == 3 ? RingW<TYPE>::HI : 0);
  return n;
}
#define RING_PIN4(d) asm volatile("" : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]))

template <int TYPE, int ACCUM, int WR, int WK, int NB, int DX>
SK_DEV void matmul_ring(unsigned char *smem, const uint4 *__restrict__ w, const uint16_t *__restrict__ wd, const f16 *x,
                        float *y, const MatmulPush &p, uint32_t row0, uint32_t col0, uint32_t n_tok, uint32_t st0,
                        uint32_t st1, float *part, uint32_t *count, uint32_t S, uint32_t sp) {
  using RW = RingW<TYPE>;
  constexpr uint32_t XB = NB * 4096u, WB = RW::WI * 1024u, HB = RW::HI * 1024u, NW = ring_nw<TYPE, DX>();
  constexpr int XI = 4 * NB / WR;  // activation DMA instructions per wave and chunk
  static_assert(XI * WR == 4 * NB, "the waves share the activation loads evenly");
  static_assert(WK == 1 || WK == 2 || WK == 4, "the order of the K groups' sum");
  const uint32_t tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t wr = wave % WR, wk = wave / WR;
  // this K group's super-blocks; every group runs the loop as often as the longest
  const uint32_t n_all = st1 - st0;
  const uint32_t s_lo = st0 + wk * n_all / WK, n_st = st0 + (wk + 1) * n_all / WK - s_lo;
  const uint32_t n_max = (n_all + WK - 1) / WK, n_chunk = 4 * n_st;

  unsigned char *const xg = smem + wk * DX * XB;
  unsigned char *const wg = smem + WK * DX * XB + wave * (NW * WB + 2u * HB);
  unsigned char *const hg = wg + NW * WB;
  const uint32_t xg_a = lds_addr(xg), wg_a = lds_addr(wg), hg_a = lds_addr(hg);

  const uint32_t supers = p.n_in >> 8, blocks = p.n_in >> 5;
  const uint32_t rowb = row0 + wr * 32, rlast = p.n_out - 1;
  // (w and wd are two views of one buffer: the runtime launches this tile only then)
  const u32x4 xres = dl_res(x, 0x7fffffffull), wres = dl_res(w, 0xffffffffull);
  // activation rows of this lane: token 8 (WR i + wr) + lane / 8, its swizzled 16 B unit
  // (tokens past the tile's: an offset past the resource, zeros)
  uint32_t xo[XI], xk[TYPE == 0 ? XI : 1];
#pragma unroll
  for (int i = 0; i < XI; i++) {
    const uint32_t tok = 8 * (WR * i + wr) + (lane >> 3), u = (lane & 7) ^ dl_swz(tok);
    xo[i] = tok < n_tok ? 2u * (p.x_off + (col0 + tok) * p.x_stride + 8u * u) : 0x80000000u;
    if constexpr (TYPE == 0) xk[i] = 8 * u;
  }
  uint32_t wo[RW::WI], ho, hd2 = 0, wu = 0;
  const uint32_t dlast = TYPE == 0 ? (2u * (p.o1 + p.n_out * blocks) - 1) & ~15u : 0u;
  auto R = [&](uint32_t r) { return min(rowb + r, rlast); };
  if constexpr (TYPE == 1) {
    wo[0] = 16u * (p.o0 + R(lane >> 1) * supers * 8 + (lane & 1));
    ho = 16u * (p.o1 + R(l32) * supers);
  } else if constexpr (TYPE == 2) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const uint32_t r = 16 * i + (lane >> 2);
      wo[i] = 16u * (p.o0 + R(r) * supers * 8 + ((lane & 3) ^ ((r >> 2) & 3)));
    }
    const uint32_t r = lane >> 1;
    wo[2] = 16u * (p.o1 + R(r) * supers * 4 + ((lane & 1) ^ ((r >> 3) & 1)));
    // lanes 0..31 the scales of row l32, lanes 32..63 the 16 B that hold its d
    hd2 = 2u * (p.o3 + R(l32) * supers);
    ho = hh ? hd2 : 16u * (p.o2 + R(l32) * supers);
  } else {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const uint32_t r = 16 * i + (lane >> 2);
      wo[i] = 16u * (p.o0 + R(r) * (p.n_in >> 4) + ((lane & 3) ^ ((r >> 2) & 3)));
    }
    wu = 16u * ((lane & 3) ^ ((lane >> 4) & 3));  // this lane's k inside a chunk
    ho = 2u * (p.o1 + R(l32) * blocks);
  }

  // one of a chunk's loads: XI of activations, then the weights, then (chunk 3 of a super-block)
  // the next super-block's scales; `on` 0xffffffff, or 0 past the last chunk
  // (the resource's words are wave-uniform; readfirstlane keeps them in SGPRs, as the load takes them)
  auto masked = [](const u32x4 &r, uint32_t on) -> u32x4 {
    u32x4 v = {(uint32_t)__builtin_amdgcn_readfirstlane(r.x), (uint32_t)__builtin_amdgcn_readfirstlane(r.y),
               (uint32_t)__builtin_amdgcn_readfirstlane(r.z & on), (uint32_t)__builtin_amdgcn_readfirstlane(r.w)};
    return v;
  };
  auto dma_x = [&](uint32_t c, uint32_t buf, int i, uint32_t on) {
    const u32x4 r = masked(xres, on);
    const uint32_t k = 256u * s_lo + 64u * c, l = xg_a + buf * XB + (WR * i + wr) * 1024u;
    if constexpr (TYPE == 0)  // columns past the row's end read zeros
      dl_load16(r, l, k + xk[i] < p.n_in ? xo[i] + 2u * k : 0x80000000u, 0);
    else
      dl_load16(r, l, xo[i], 2u * k);
  };
  auto dma_w = [&](uint32_t c, uint32_t buf, int i, uint32_t on) {
    const u32x4 r = masked(wres, on);
    const uint32_t st = s_lo + (c >> 2), l = wg_a + buf * WB + i * 1024u;
    if constexpr (TYPE == 1) {
      dl_load16(r, l, wo[0], 128u * st + 32u * (c & 3));
    } else if constexpr (TYPE == 2) {
      dl_load16(r, l, wo[i], i < 2 ? 128u * st + 32u * (c & 3) : 64u * st + 16u * (c & 3));
    } else {  // past the row's end the activations and d are zero: any bytes of the row will do
      const uint32_t k = 256u * s_lo + 64u * c;
      dl_load16(r, l, k + wu < p.n_in ? wo[i] + k : wo[i], 0);
    }
  };
  auto dma_h = [&](uint32_t st, uint32_t on) {
    const u32x4 r = masked(wres, on);
    const uint32_t l = hg_a + (st & 1) * HB;
    if constexpr (TYPE == 1)
      dl_load16(r, l, ho, 16u * st);
    else if constexpr (TYPE == 2)
      dl_load16(r, l, hh ? (ho + 2u * st) & ~15u : ho + 16u * st, 0);
    else  // the second piece of the matrix's last row may lie past its d: then the last one again
      dl_load16(r, l, min(((ho + 16u * st) & ~15u) + 16u * hh, dlast), 0);
  };
  // all ones for a chunk of the range, zero past it (arithmetic, not a select: the compiler put
  // a select into a vector register)
  auto live = [&](uint32_t c) { return (uint32_t)((int32_t)(c - n_chunk) >> 31); };
  // weight buffer of chunk c
  auto wbuf = [&](uint32_t c, uint32_t xbuf) { return TYPE == 2 ? (c >> 1) % NW : xbuf; };

  // Q8_0: the rows' e[t], in the buffer that chunk DX - 1 fills after them
  const unsigned char *const xe = xg + (DX - 1) * XB;
  if constexpr (TYPE == 0)
    dl_load16(masked(xres, ~0u), xg_a + (DX - 1) * XB, lane < 32 ? 4u * col0 + 16u * lane : 0x80000000u, 0);
  // ---- prologue: the first scales, chunks 0 .. DX - 2
  dma_h(s_lo, live(0));
#pragma unroll
  for (int c = 0; c < DX - 1; c++) {
#pragma unroll
    for (int i = 0; i < XI; i++) dma_x(c, c, i, live(c));
#pragma unroll
    for (int i = 0; i < ring_wi<TYPE>(c); i++) dma_w(c, TYPE == 2 ? c >> 1 : c, i, live(c));
    if ((c & 3) == 3) dma_h(s_lo + 1, live(c + 1));
  }
  dl_wait_vm<ring_fly<TYPE>(-1, DX + 1, XI)>();
  __syncthreads();

  f32x16 acc[NB];
#pragma unroll
  for (int j = 0; j < NB; j++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[j][i] = 0.0f;

  // does a row of this tile have exponents?
  bool big = false;
  if constexpr (TYPE == 0) {
    uint32_t f = lane < n_tok ? *(const uint32_t *)(xe + 4 * lane) : 0u;
    if constexpr (NB > 2) f |= 64 + lane < n_tok ? *(const uint32_t *)(xe + 256 + 4 * lane) : 0u;
    big = __ballot(f != 0) != 0;
  }
  // the sums from units of run `from` of 128 values to those of run `to` (past the last run: 1)
  auto rescale = [&](uint32_t from, uint32_t to) {
    const uint32_t ne = (p.n_in + E_RUN - 1) / E_RUN;
    const int *e = (const int *)x, *er = e + p.table_off;
    // lane l finds the change of tokens l and 64 + l, and takes its sums' from their lanes
    int d[NB > 2 ? 2 : 1];
#pragma unroll
    for (int h = 0; h < (NB > 2 ? 2 : 1); h++) {
      const uint32_t tok = 64 * h + lane, at = (col0 + tok) * ne;
      d[h] = 0;
      if (tok < n_tok && e[col0 + tok] != 0) d[h] = (from < ne ? er[at + from] : 0) - (to < ne ? er[at + to] : 0);
    }
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
      for (int i = 0; i < 16; i++)
        acc[j][i] = __builtin_ldexpf(
            acc[j][i], __builtin_amdgcn_ds_bpermute(4 * (4 * hh + (32 * (j & 1) + 8 * (i >> 2) + (i & 3))), d[j >> 1]));
  };

  // ---- scales: hd of the current super-block; sc / nm of the next step to dequantise
  uint4 hd;
  uint32_t hdd = 0;  // Q6_K: the row's d
  auto load_h = [&](uint32_t st) {
    const unsigned char *h = hg + (st & 1) * HB;
    if constexpr (TYPE != 0) hd = *(const uint4 *)(h + 16u * l32);
    if constexpr (TYPE == 2) hdd = *(const uint16_t *)(h + 512u + 16u * l32 + ((hd2 + 2u * st) & 15u));
  };
  // (scale, -min) of step t (0..15) of the super-block hd holds, or of super-block st (Q8_0)
  auto scale_of = [&](uint32_t st, int t, f16x2 &sc, f16x2 &nm) {
    if constexpr (TYPE == 1) {
      WStage<1> s;
      s.hd = hd;
      step_scale<1>(s, t, hh, sc, nm);
    } else if constexpr (TYPE == 2) {
      WStage<2> s;
      s.sc = hd;
      s.d = hdd;
      step_scale<2>(s, t, hh, sc, nm);
    } else {
      const uint32_t pos = (ho & 15u) + (uint32_t)(t & ~1);
      const uint16_t d = *(const uint16_t *)(hg + (st & 1) * HB + 16u * l32 + (pos & 15u) + 512u * (pos >> 4));
      sc = splat(__builtin_bit_cast(f16, (uint16_t)(8 * st + (t >> 1) < blocks ? d : 0)));
    }
    uint32_t a = as_u32(sc);
    asm volatile("" : "+v"(a));
    sc = as_f16x2(a);
    if constexpr (TYPE == 1) {
      uint32_t b = as_u32(nm);
      asm volatile("" : "+v"(b));
      nm = as_f16x2(b);
    }
  };

  // ---- raw quants: Q4_K one read per pair of steps (raw4[step / 2]), others one (two) per step
  uint4 raw4[2];
  uint2 rl[2], rh[2];
  auto load_raw = [&](const unsigned char *wb, int ts) {
    if constexpr (TYPE == 1) {
      raw4[ts >> 1] = *(const uint4 *)(wb + 32u * l32 + 16u * (ts >> 1));
    } else {
      rl[ts & 1] = *(const uint2 *)(wb + 64u * l32 + 16u * (ts ^ ((l32 >> 2) & 3)) + 8u * hh);
      if constexpr (TYPE == 2)
        rh[ts & 1] = *(const uint2 *)(wb + 2048u + 32u * l32 + 16u * ((ts & 1) ^ ((l32 >> 3) & 1)) + 8u * hh);
    }
  };
  // dequantisation of step t in three phases (masks, offset, scale), four pairs each
  const uint32_t mask = hh ? 0x00f000f0u : 0x000f000fu;
  auto deq = [&](int phase, int t, f16x2 sc, f16x2 nm, uint32_t(&d)[4]) {
    constexpr uint32_t M = 0x64006400u;
    const int g = (t >> 1) & 3;  // Q6_K quant group
    if (phase == 0) {
      if constexpr (TYPE == 1) {
        const uint4 r = raw4[(t >> 1) & 1];
        const uint32_t a = (t & 1) ? r.z : r.x, b = (t & 1) ? r.w : r.y;
        d[0] = (a & mask) | M;
        d[1] = ((a >> 8) & mask) | M;
        d[2] = (b & mask) | M;
        d[3] = ((b >> 8) & mask) | M;
      } else if constexpr (TYPE == 2) {
        const uint2 l = rl[t & 1], h = rh[t & 1];
        const uint32_t lm = g >= 2 ? 0x00f000f0u : 0x000f000fu, hm = g >= 2 ? 0x03000300u : 0x00300030u;
        const int hs = 4 - 2 * (g & 1);
        auto q6 = [&](uint32_t lv, uint32_t hv) -> uint32_t { return (lv & lm) | M | ((hv << hs) & hm); };
        d[0] = q6(l.x, h.x);
        d[1] = q6(l.x >> 8, h.x >> 8);
        d[2] = q6(l.y, h.y);
        d[3] = q6(l.y >> 8, h.y >> 8);
      } else {
        const uint32_t a = rl[t & 1].x ^ 0x80808080u, b = rl[t & 1].y ^ 0x80808080u;
        d[0] = (a & 0x00ff00ffu) | M;
        d[1] = ((a >> 8) & 0x00ff00ffu) | M;
        d[2] = (b & 0x00ff00ffu) | M;
        d[3] = ((b >> 8) & 0x00ff00ffu) | M;
      }
    } else if (phase == 1) {
      const f16x2 off = splat((f16)(TYPE == 1 ? -1024.0f : TYPE == 2 ? (g >= 2 ? -1536.0f : -1056.0f) : -1152.0f));
#pragma unroll
      for (int q = 0; q < 4; q++) d[q] = as_u32(as_f16x2(d[q]) + off);
    } else {
#pragma unroll
      for (int q = 0; q < 4; q++)
        d[q] = as_u32(TYPE == 1 ? __builtin_elementwise_fma(as_f16x2(d[q]), sc, nm) : as_f16x2(d[q]) * sc);
    }
    RING_PIN4(d);
  };

  // activation fragment addresses of the four steps of a chunk
  uint32_t xa[4];
#pragma unroll
  for (int t = 0; t < 4; t++) xa[t] = l32 * 128u + 16u * ((TYPE == 1 ? 4 * hh + t : 2 * t + hh) ^ dl_swz(l32));
  f16x8 xf[2][NB];
  uint32_t wf[2][4];
  f16x2 sc, nm = splat((f16)0.0f), scn, nmn = nm;
  load_h(s_lo);
  load_raw(wg, 0);
  if constexpr (TYPE != 1) load_raw(wg, 1);
  scale_of(s_lo, 0, sc, nm);
  scn = sc;
  nmn = nm;
#pragma unroll
  for (int j = 0; j < NB; j++) xf[0][j] = *(const f16x8 *)(xg + xa[0] + j * 4096u);
#pragma unroll
  for (int ph = 0; ph < 3; ph++) deq(ph, 0, sc, nm, wf[0]);
  if constexpr (TYPE == 2) scale_of(s_lo, 1, sc, nm);

  uint32_t bc = 0;  // activation buffer of the current chunk
  for (uint32_t s = 0; s < n_max; s++) {
    if (s < n_st) {
      auto chunk = [&](auto C4) {
        constexpr int c4 = decltype(C4)::v;
        const uint32_t c = 4 * s + c4, bn = bc + 1 == DX ? 0 : bc + 1, bf = bc == 0 ? DX - 1 : bc - 1;
        const unsigned char *xc = xg + bc * XB, *xn = xg + bn * XB;
        const unsigned char *wc = wg + wbuf(c, bc) * WB, *wn = wg + wbuf(c + 1, bn) * WB;
        const uint32_t cl = c + DX - 1, on = live(cl), onh = live(cl + 1);
        auto step = [&](auto TS) {
          constexpr int ts = decltype(TS)::v, nt = (ts + 1) & 3;
          constexpr int tn = (4 * c4 + ts + 1) & 15;  // the next step in its super-block
          const uint32_t sn = s_lo + s + (4 * c4 + ts + 1 > 15);
          uint32_t d[4];
          typedef uint32_t frag4 __attribute__((ext_vector_type(4)));
          const frag4 wc4 = {wf[ts & 1][0], wf[ts & 1][1], wf[ts & 1][2], wf[ts & 1][3]};
          const f16x8 wcur = __builtin_bit_cast(f16x8, wc4);
#pragma unroll
          for (int j = 0; j < NB; j++) {
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[ts & 1][j], wcur, acc[j], 0, 0, 0);
            xf[nt & 1][j] = *(const f16x8 *)((ts == 3 ? xn : xc) + xa[nt] + j * 4096u);
            if (j == 0) {
              // raw quants two steps ahead
              if (TYPE != 1 || (ts & 1) == 0) load_raw(ts < 2 ? wc : wn, (ts + 2) & 3);
              // the next super-block's scales, after the last use of this one's
              if (c4 == 3 && ts == (TYPE == 1 ? 0 : 2)) load_h(s_lo + s + 1);
            }
            if (j == 0) deq(0, tn, sc, nm, d);
            if (j == NB / 4) deq(1, tn, sc, nm, d);
            if (j == NB / 2) deq(2, tn, sc, nm, d);
            if (j == NB - 1) {
#pragma unroll
              for (int q = 0; q < 4; q++) wf[nt & 1][q] = d[q];
              // scales: Q4_K the next chunk's at step 1, Q6_K two steps ahead, Q8_0 the next pair's
              constexpr int t2 = (4 * c4 + ts + 2) & 15;
              if (TYPE == 1 && ts == 1) scale_of(sn, (4 * c4 + 4) & 15, scn, nmn);
              if (TYPE == 1 && ts == 2) sc = scn, nm = nmn;
              if (TYPE == 2) scale_of(sn, t2, sc, nm);
              if (TYPE == 0 && (ts & 1) == 0) scale_of(s_lo + s + (4 * c4 + ts + 2 > 15), t2, sc, nm);
            }
            if (ts >= 2) {
              constexpr int NI = XI + ring_wi<TYPE>(c4 + DX - 1), slot = 2 * NB;
#pragma unroll
              for (int i = 0; i < NI; i++)
                if (i * slot / NI == (ts - 2) * NB + j) {
                  if (i < XI)
                    dma_x(cl, bf, i, on);
                  else
                    dma_w(cl, wbuf(cl, bf), i - XI, on);
                }
              if (ts == 3 && j == NB - 1 && ((c4 + DX - 1) & 3) == 3) dma_h(s_lo + (cl >> 2) + 1, onh);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        };
        step(IC<0>{});
        step(IC<1>{});
        dl_wait_vm<ring_fly<TYPE>(c4, DX, XI)>();
        if constexpr (WR > 1) __syncthreads();
        step(IC<2>{});
        step(IC<3>{});
        bc = bn;
      };
      if (TYPE == 0 && __builtin_expect(big, 0)) rescale(2 * (s_lo + s) - 1, 2 * (s_lo + s));
      chunk(IC<0>{});
      chunk(IC<1>{});
      if (TYPE == 0 && __builtin_expect(big, 0)) rescale(2 * (s_lo + s), 2 * (s_lo + s) + 1);
      chunk(IC<2>{});
      chunk(IC<3>{});
    } else if constexpr (WR > 1) {
#pragma unroll
      for (int i = 0; i < 4; i++) __syncthreads();
    }
  }
  dl_wait_vm<0>();  // no load may write LDS after this
  if (TYPE == 0 && big && n_st != 0) rescale(2 * (s_lo + n_st) - 1, ~0u);

  // ---- the K groups' sums.  Group wk finishes token blocks [wk NBF, wk NBF + NBF); with
  // fewer blocks than groups the first NB groups take one each.
  constexpr int NBF = WK == 1 ? NB : NB >= WK ? NB / WK : 1;
  static_assert(NB < WK || NB % WK == 0, "whole token blocks per K group");
  const bool fins = WK == 1 || wk * NBF < (uint32_t)NB;
  const uint32_t tok0 = WK == 1 || !fins ? 0u : 32u * NBF * wk;
  const uint32_t row = rowb + l32;
  // (y relative to the tile's first token; offsets of tokens or rows past the tile lie past the
  // resource: loads return zero, stores are dropped)
  const BufRes yres = buf_res(y + p.y_off + (size_t)col0 * p.y_stride, 0x7fffffffull);
  auto yoff = [&](int j, int i) {
    const uint32_t tok = tok0 + 32 * j + 8 * (i >> 2) + 4 * hh + (i & 3);
    return tok < n_tok && row < p.n_out ? 4u * (tok * p.y_stride + row) : 0x80000000u;
  };
  float fin[NBF][16], old[ACCUM ? NBF : 1][16];
  int4 ex[NBF][4];  // the rows came as x * 2^-e (Q8_0: scaled back already)
#pragma unroll
  for (int j = 0; j < NBF; j++)
    if constexpr (TYPE == 0)
#pragma unroll
      for (int q = 0; q < 4; q++) ex[j][q] = make_int4(0, 0, 0, 0);
    else
#pragma unroll
    for (int q = 0; q < 4; q++) ex[j][q] = *(const int4 *)((const int *)x + col0 + tok0 + 32 * j + 8 * q + 4 * hh);
  if constexpr (ACCUM) {
    if (S == 1 && fins)
#pragma unroll
      for (int j = 0; j < NBF; j++)
#pragma unroll
        for (int i = 0; i < 16; i++)
          old[j][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(yres, yoff(j, i), 0, 0));
  }
  if constexpr (WK == 1) {
#pragma unroll
    for (int j = 0; j < NBF; j++)
#pragma unroll
      for (int i = 0; i < 16; i++) fin[j][i] = acc[j][i];
  } else {
    __syncthreads();  // every wave is done with the operand buffers
    float *red = (float *)smem;
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        *(float4 *)(red + ((wave * NB + j) * 4 + q) * 256 + 4 * lane) =
            make_float4(acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]);
    __syncthreads();
    if (fins)
#pragma unroll
      for (int j = 0; j < NBF; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          auto group = [&](int g) {
            return *(const float4 *)(red + (((g * WR + wr) * NB + wk * NBF + j) * 4 + q) * 256 + 4 * lane);
          };
          auto add = [](float4 u, float4 v) { return make_float4(u.x + v.x, u.y + v.y, u.z + v.z, u.w + v.w); };
          float4 t = add(group(0), group(1));
          if constexpr (WK == 4) t = add(t, add(group(2), group(3)));
          fin[j][4 * q] = t.x;
          fin[j][4 * q + 1] = t.y;
          fin[j][4 * q + 2] = t.z;
          fin[j][4 * q + 3] = t.w;
        }
  }

  // ---- a launch split in K: the last workgroup of the tile adds the splits in order (the
  // handoff of matmul_tile128_w)
  if (S > 1) {
    constexpr uint32_t PER = NBF * 16 * 64, PART = WR * WK * PER;
    if (fins) {
      float *mine = part + (size_t)sp * PART + wave * PER;
#pragma unroll
      for (int j = 0; j < NBF; j++)
#pragma unroll
        for (int i = 0; i < 16; i++)
          __hip_atomic_store(mine + (j * 16 + i) * 64 + lane, fin[j][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    uint32_t *last = (uint32_t *)smem;  // (the operands and the groups' sums are read)
    if (tid == 0) *last = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT) == S - 1;
    __syncthreads();
    if (!*last) return;
    if (fins) {
      if constexpr (ACCUM)
#pragma unroll
        for (int j = 0; j < NBF; j++)
#pragma unroll
          for (int i = 0; i < 16; i++)
            old[j][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(yres, yoff(j, i), 0, 0));
      float t[NBF][16];
      for (uint32_t q = 0; q < S; q++) {
        float v[NBF][16];
        const float *src = part + (size_t)q * PART + wave * PER + lane;
        if (q == sp) {
#pragma unroll
          for (int j = 0; j < NBF; j++)
#pragma unroll
            for (int i = 0; i < 16; i++) v[j][i] = fin[j][i];
        } else {
#pragma unroll
          for (int j = 0; j < NBF; j++)
#pragma unroll
            for (int i = 0; i < 16; i++)
              v[j][i] = __hip_atomic_load(src + (j * 16 + i) * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int j = 0; j < NBF; j++)
#pragma unroll
          for (int i = 0; i < 16; i++) t[j][i] = q == 0 ? v[j][i] : t[j][i] + v[j][i];
      }
#pragma unroll
      for (int j = 0; j < NBF; j++)
#pragma unroll
        for (int i = 0; i < 16; i++) fin[j][i] = t[j][i];
    }
    if (tid == 0) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  if (!fins) return;
#pragma unroll
  for (int j = 0; j < NBF; j++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int ee[4] = {ex[j][q].x, ex[j][q].y, ex[j][q].z, ex[j][q].w};
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = 4 * q + r;
        float v = __builtin_ldexpf(fin[j][i], ee[r]);
        if constexpr (ACCUM) v = old[j][i] + v;
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), yres, yoff(j, i), 0, 0);
      }
    }
}

// Workgroup (row tile, token tile, split) of a launch over up to four matrices that read the
// same rows (segments as matmul_tile128_w takes them: row tiles of segment s after those of
// s - 1).  Ids are dealt to the XCDs round-robin; consecutive ones take consecutive token
// tiles, then splits.  NB: token blocks of the grid's tiles; a tile with fewer live blocks
// runs the body that holds them.
template <int TYPE, int ACCUM, int WR, int WK, int NB, int DX>
SK_DEV void ring_entry(const uint4 *w, const uint16_t *wd, const f16 *x, float *y, const uint32_t *ctl,
                       const Segments<MatmulPush> &m, float *ws, uint32_t *cnt, uint32_t S) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[ring_lds<TYPE, WR, WK, NB, DX>()];
  constexpr uint32_t TR = 32 * WR, TT = 32 * NB;
  const uint32_t gz = gridDim.z, Z = gz / S, lin = blockIdx.x + gridDim.x * blockIdx.z;
  const uint32_t rem = lin % gz, tt = rem % Z, sp = rem / Z, kt = (lin / gz) * Z + tt;
  const uint32_t n_all = ctl[2], col0 = tt * TT;
  if (col0 >= n_all) return;
  const uint32_t n_tok = min(n_all - col0, TT);
  uint32_t rt = lin / gz;
  // field by field, the (wave-uniform) segment in an SGPR
  const uint32_t sg = __builtin_amdgcn_readfirstlane(segment_of(m, rt));
  auto pick = [&](uint32_t MatmulPush::*f) -> uint32_t {
    const uint32_t a = m.p[0].*f, b = m.p[1].*f, c = m.p[2].*f, d = m.p[3].*f;
    return sg == 0 ? a : sg == 1 ? b : sg == 2 ? c : d;
  };
  MatmulPush p = m.p[0];
  p.o0 = pick(&MatmulPush::o0);
  p.o1 = pick(&MatmulPush::o1);
  p.o2 = pick(&MatmulPush::o2);
  p.o3 = pick(&MatmulPush::o3);
  p.y_off = pick(&MatmulPush::y_off);
  p.n_out = pick(&MatmulPush::n_out);
  p.y_stride = pick(&MatmulPush::y_stride);
  rt -= sg == 0 ? 0u : sg == 1 ? m.start[1] : sg == 2 ? m.start[2] : m.start[3];
  const uint32_t n_st = (p.n_in + 255) / 256, st0 = sp * n_st / S, st1 = (sp + 1) * n_st / S;
  // a partial tile holds at most WR * WK * max(NB / WK, 1) * 1024 values
  float *part = ws + (size_t)kt * S * (WR * WK * (NB >= WK ? NB / WK : 1) * 1024);
  if constexpr (NB >= 4)
    if (n_tok > 64) {
      matmul_ring<TYPE, ACCUM, WR, WK, 4, DX>(smem, w, wd, x, y, p, rt * TR, col0, n_tok, st0, st1, part, cnt + kt, S, sp);
      return;
    }
  if constexpr (NB >= 2)
    if (n_tok > 32) {
      matmul_ring<TYPE, ACCUM, WR, WK, 2, DX>(smem, w, wd, x, y, p, rt * TR, col0, n_tok, st0, st1, part, cnt + kt, S, sp);
      return;
    }
  matmul_ring<TYPE, ACCUM, WR, WK, 1, DX>(smem, w, wd, x, y, p, rt * TR, col0, n_tok, st0, st1, part, cnt + kt, S, sp);
}

}  // namespace

// matmul_ring__TYPE_ACCUM_WR_WK_NB_DX (not engine symbols; the runtime's rule picks the shape)
#define RING(T, A, WR, WK, NB, DX, OCC)                                                                         \
  extern "C" __global__ __launch_bounds__(64 * WR * WK, OCC) void matmul_ring__##T##_##A##_##WR##_##WK##_##NB##_##DX( \
      const uint4 *w, const uint16_t *wd, const f16 *x, float *y, const uint32_t *ctl, Segments<MatmulPush> m,  \
      float *ws, uint32_t *cnt, uint32_t S) {                                                                   \
    ring_entry<T, A, WR, WK, NB, DX>(w, wd, x, y, ctl, m, ws, cnt, S);                                           \
  }
#define RING_SHAPES(T, A) \
  RING(T, A, 4, 1, 4, 4, 1) \
  RING(T, A, 4, 1, 4, 3, 2) \
  RING(T, A, 4, 2, 2, 4, 1) \
  RING(T, A, 1, 4, 2, 3, 1)
RING_SHAPES(0, 0)
RING_SHAPES(0, 1)
RING_SHAPES(1, 0)
RING_SHAPES(1, 1)
RING_SHAPES(2, 0)
RING_SHAPES(2, 1)
