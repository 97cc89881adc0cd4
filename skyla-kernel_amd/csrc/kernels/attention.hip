// The rest of the decode step around the weight matvecs, gfx950: RMSNorm, the QK-norm +
// RoPE + KV-cache write, split-K attention over the cache and its merge, and the last-row
// copy of a prefill chunk (graph.rs:48-113, 200-233; the kernels of kernels.rs:186-193).
//
// Contract (bindings, push words, grids) as the engine dispatches them:
//   rmsnorm          [W, A, C]            6 words  grid [1, tokens, 1]
//   qkv_prep         [W, A, C, KV, KV8]  16 words  grid [n_head + 2 n_kv, tokens, 1]
//   attention        [A, C, KV, KV8, KVS] 11 words grid [n_kv, n_split, tokens], 256 threads
//   attention_merge  [A, C]               6 words  grid [n_head, tokens, 1], 1024 threads
//   attention_prep   [W, A, C, KV, KV8]  17 words  grid [n_kv, n_split, 1], 256 threads:
//                    qkv_prep + attention of a single-token step
//   take_last        [A, C]               4 words  grid [ceil(n / 256), 1, 1]
// W is a weight buffer (f32 tables: norm weights, RoPE frequencies), A the f32 arena and C
// its u32 view (ctl[1] = position of the first token, ctl[2] = token count), KV the cache
// buffer as f16 (keys, f16 values, the per-32 scales of 8-bit entries) and KV8 as i8.
// Offsets are element indices of the view they index.  Heads are 128 wide (head_dim =
// n_rot = 128, no gate: the plain Qwen3 layout Engine::new accepts, engine.rs:27-39).
//
// KV layout (kv.rs): a layer's keys at kc_off + pos * kv_dim + head * 128, values likewise
// at vc_off; an 8-bit row keeps one f16 scale per 32 values at
// scales + pos * kv_dim / 32 + head * 4 + block.  An entry is quantised as
// s = max|y| over its block / 127, q = round(y / s) (qkv_prep.comp:44-65; ties to even).
#include "matmul_common.h"

namespace {

constexpr uint32_t HD = 128;     // head width
constexpr uint32_t CHUNK = 64;   // positions per attention split (arena.rs:6)
constexpr uint32_t PART = HD + 2;  // one (head, split) partial: m, l, acc[128]

struct NormPush { uint32_t x_off, w_off, y_off, n; float eps; uint32_t stride; };
struct QkvPush {
  uint32_t q_off, k_off, v_off, qn_off, kn_off, kc_off, vc_off, n_head, n_kv;
  float eps;
  uint32_t rope_off;
  float mscale;
  uint32_t q_stride, kv_stride, ks_off, vs_off;
};
struct AttnPush {
  uint32_t q_off, part_off, kc_off, vc_off, n_kv, n_split;
  float scale;
  uint32_t q_stride, part_stride, ks_off, vs_off;
};
struct MergePush { uint32_t part_off, o_off, n_split, chunk, part_stride, o_stride; };
// attention_prep: qkv_prep's and attention's words for a single-token step (17 words)
struct PrepPush {
  uint32_t q_off, k_off, v_off, qn_off, kn_off, kc_off, vc_off, n_kv;
  float eps;
  uint32_t rope_off;
  float mscale;
  uint32_t ks_off, vs_off, part_off, n_split;
  float scale;
  uint32_t part_stride;
  uint32_t cs_off;  // the step's rope pairs (rope_table) in the arena, or NO_TABLE: computed here
};
constexpr uint32_t NO_TABLE = 0xffffffffu;
// attention_prep1: attention_prep's words, then attention_merge's output offset and stride
struct PrepPush1 {
  PrepPush pp;
  uint32_t o_off, o_stride;
};
struct LastPush { uint32_t src_off, dst_off, n, stride; };

SK_DEV float wave_sum(float v) { return group_sum<64>(v); }

SK_DEV float wave_max(float v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
  return v;
}

// max |v| over the 32-lane half of the wave that holds v (one quantisation block)
SK_DEV float block_max(float v) {
  v = fabsf(v);
#pragma unroll
  for (int d = 16; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
  return v;
}

// Writes y0 (element t) and y1 (element t + 64) of one head's cache row.  With `raw`, the
// stored row also goes to LDS as the cache holds it (128 f16, or 128 i8 and the four block
// scales in `sc`), for a reader in the same workgroup.
template <int Q8>
SK_DEV void store_kv(f16 *kv, int8_t *kv8, uint32_t cache, uint32_t scales, uint32_t kv_dim, uint32_t pos,
                     uint32_t head, uint32_t t, float y0, float y1, uint32_t *raw = nullptr,
                     float *sc = nullptr) {
  const uint32_t dst = cache + pos * kv_dim + head * HD;
  if constexpr (!Q8) {
    const f16 h0 = (f16)y0, h1 = (f16)y1;
    kv[dst + t] = h0;
    kv[dst + t + 64] = h1;
    if (raw) {
      ((f16 *)raw)[t] = h0;
      ((f16 *)raw)[t + 64] = h1;
    }
  } else {
    const float s0 = block_max(y0) / 127.0f, s1 = block_max(y1) / 127.0f;
    const int8_t q0 = (int8_t)(s0 > 0.0f ? __builtin_rintf(y0 / s0) : 0.0f);
    const int8_t q1 = (int8_t)(s1 > 0.0f ? __builtin_rintf(y1 / s1) : 0.0f);
    kv8[dst + t] = q0;
    kv8[dst + t + 64] = q1;
    if ((t & 31) == 0) {
      const uint32_t sd = scales + pos * (kv_dim / 32) + head * 4 + t / 32;
      kv[sd] = (f16)s0;
      kv[sd + 2] = (f16)s1;
    }
    if (raw) {
      ((int8_t *)raw)[t] = q0;
      ((int8_t *)raw)[t + 64] = q1;
      if ((t & 31) == 0) {
        sc[t / 32] = (float)(f16)s0;
        sc[t / 32 + 2] = (float)(f16)s1;
      }
    }
  }
}

// QK-norm (rmsnorm.comp over one 128-wide head, weights at nw) and NeoX RoPE (rope.rs:60-68)
// of the pair (element t, element t + 64), one wave per head.
SK_DEV void norm_rope(const float *w, uint32_t nw, uint32_t rope_off, float eps, float mscale, uint32_t pos,
                      uint32_t t, float x0, float x1, float &y0, float &y1, const float *cs = nullptr) {
#pragma clang fp contract(off)
  const float r = 1.0f / sqrtf(wave_sum(x0 * x0 + x1 * x1) / (float)HD + eps);
  const float n0 = x0 * r * w[nw + t], n1 = x1 * r * w[nw + t + 64];
  float c, s;
  if (cs) {  // rope_table's pairs for this position: the same two products
    c = cs[2 * t];
    s = cs[2 * t + 1];
  } else {
    const float angle = (float)pos * w[rope_off + t];
    c = cosf(angle) * mscale;
    s = sinf(angle) * mscale;
  }
  y0 = n0 * c - n1 * s;
  y1 = n0 * s + n1 * c;
}

// rope_table: the (cos, sin) x mscale pairs of the step's position (ctl[1]) for the 64
// rotation frequencies, computed once per decode step into the arena for every layer's
// attention_prep -- its workgroups (one per kv head and split) would each reduce the same
// large angles otherwise.  norm_rope's expressions, so the same values.
struct RopePush { uint32_t rope_off, o_off; float mscale; };
extern "C" __global__ __launch_bounds__(64) void rope_table(const float *w, float *a, const uint32_t *ctl, RopePush p) {
#pragma clang fp contract(off)
  const uint32_t t = threadIdx.x;
  const float angle = (float)ctl[1] * w[p.rope_off + t];
  a[p.o_off + 2 * t] = cosf(angle) * p.mscale;
  a[p.o_off + 2 * t + 1] = sinf(angle) * p.mscale;
}

template <int K8, int V8>
SK_DEV void qkv_body(const float *w, float *a, const uint32_t *ctl, f16 *kv, int8_t *kv8, const QkvPush &p) {
#pragma clang fp contract(off)
  const uint32_t h = blockIdx.x, tok = blockIdx.y;
  if (tok >= ctl[2]) return;
  const uint32_t t = threadIdx.x, pos = ctl[1] + tok, kv_dim = p.n_kv * HD;
  if (h >= p.n_head + p.n_kv) {  // value head: cache it as it is
    const uint32_t vh = h - p.n_head - p.n_kv;
    const uint32_t src = p.v_off + tok * p.kv_stride + vh * HD;
    store_kv<V8>(kv, kv8, p.vc_off, p.vs_off, kv_dim, pos, vh, t, a[src + t], a[src + t + 64]);
    return;
  }
  const bool is_q = h < p.n_head;
  const uint32_t head = is_q ? h : h - p.n_head;
  const uint32_t src = (is_q ? p.q_off + tok * p.q_stride : p.k_off + tok * p.kv_stride) + head * HD;
  const uint32_t nw = is_q ? p.qn_off : p.kn_off;
  float y0, y1;
  norm_rope(w, nw, p.rope_off, p.eps, p.mscale, pos, t, a[src + t], a[src + t + 64], y0, y1);
  if (is_q) {
    a[src + t] = y0;
    a[src + t + 64] = y1;
  } else {
    store_kv<K8>(kv, kv8, p.kc_off, p.ks_off, kv_dim, pos, head, t, y0, y1);
  }
}

// Element d of cache row `pos` of head kvh.
template <int Q8>
SK_DEV float load_kv(const f16 *kv, const int8_t *kv8, uint32_t cache, uint32_t scales, uint32_t kv_dim,
                     uint32_t pos, uint32_t kvh, uint32_t d) {
  const uint32_t at = cache + pos * kv_dim + kvh * HD + d;
  if constexpr (!Q8)
    return (float)kv[at];
  else
    return (float)kv8[at] * (float)kv[scales + pos * (kv_dim / 32) + kvh * 4 + d / 32];
}

// One workgroup of four waves per (kv head, split of CHUNK positions, token); every load of
// the split is issued up front.  Scores with f16 keys run on the matrix cores: wave w
// computes the N_REP query heads (A, from LDS) against its 16 positions (B, one key row's
// 32 dims per lane group and k-step) in four v_mfma_f32_16x16x32_f16 k-steps, once with
// the heads' f16 high parts and once with their low parts (the heads scaled by a power of
// two first, so hi + lo carries each value to 2^-22 of the head's largest and the products
// with the f16 keys are exact in the f32 sums).  With 8-bit keys, thread t takes dims
// 8 (t % 16) ... of the key rows of positions t / 16 + 16 k (k < 4) and dots them with the
// heads in f32; the 16 partial dots of a row meet in a DPP sum.  The chunk's softmax numerators
// e_p = exp(s_p - m) go through LDS to the value phase, where thread t weights 8 dims
// (8 (t % 16) ...) of the value rows of positions 4 (t / 16) ... 4 (t / 16) + 3; the 16
// position groups are then summed in LDS.  The partial (m, l = sum e_p, acc = sum e_p v_p)
// goes to the part region for attention_merge; it is the same quantity as the reference's
// running (m, l, acc) over the chunk (attention.comp:83-97).  Positions past the token's
// own are masked (e = 0) and read a live row instead, so no load leaves the cache.
//
// PREP (attention_prep, single-token steps): qkv_prep folded in.  Each workgroup norms and
// rotates its own query heads from the raw q rows (one wave per head, the same arithmetic
// as qkv_prep), and the workgroup whose split holds the new position writes that
// position's key and value rows to the cache as qkv_prep would, keeping the stored bytes
// in LDS: its threads take them from there in place of the rows they loaded from the cache
// before the write (the new row and the masked slots clamped to it).
//
// DIRECT (attention_prep1, a grid of one split: every position of the step in the first 64):
// the workgroup writes the merged output itself, o = (acc + 0) / l per dim -- what
// attention_merge computes over one split (its weight is exp(0) = 1 and every other term
// adds zero), so the same bits -- and no partial; o_off / o_stride are the merge's.
template <int N_REP, int K8, int V8, bool PREP = false, bool DIRECT = false>
SK_DEV void attention_body(const float *w, float *a, const uint32_t *ctl, f16 *kv, int8_t *kv8, const AttnPush &p,
                           const PrepPush *pp, uint32_t o_off = 0, uint32_t o_stride = 0) {
  // heads per value reduction round: two keep vp at 16 KB and the workgroup near 20 KB of
  // LDS, so six share a CU (with four heads, 32 KB, LDS allowed four, and a 16k-position
  // step's 2056 workgroups took a third round of eight)
  constexpr int HG = N_REP < 2 ? N_REP : 2;
  // f16 keys: the scores on the matrix cores (MQ); 8-bit keys keep the VALU dots
  constexpr bool MQ = !K8;
  // the A operand's rows: head m % N_REP in row m (rows past the heads repeat them, and
  // their products are not used); a row pitch of 320 B (80 banks) puts the 16 distinct
  // 16 B pieces that a k-step's lanes read (four heads x four dim groups) on distinct banks
  constexpr int QP = HD + 32;
  __shared__ float qs[MQ ? 1 : N_REP][HD];
  __shared__ __attribute__((aligned(16))) f16 qh[2][MQ ? N_REP : 1][MQ ? QP : 8];
  __shared__ int qsh[MQ ? N_REP : 1];
  __shared__ __attribute__((aligned(16))) uint32_t nk[PREP ? 64 : 1], nv[PREP ? 64 : 1];
  __shared__ float nks[PREP ? 4 : 1], nvs[PREP ? 4 : 1];
  __shared__ float es[N_REP][CHUNK];
  __shared__ float wm[4][N_REP];
  __shared__ float4 vp[16][HG * HD / 4];
  __shared__ float lsh[DIRECT ? N_REP : 1];
  const uint32_t kvh = blockIdx.x, split = blockIdx.y, tok = blockIdx.z;
  const uint32_t n_pos = ctl[1] + tok + 1;
  if (tok >= ctl[2] || split * CHUNK >= n_pos) return;
  const uint32_t t = threadIdx.x, wave = t >> 6, kv_dim = p.n_kv * HD;
  const uint32_t begin = split * CHUNK, cnt = min(CHUNK, n_pos - begin);

  // keys: dims [8 kd, 8 kd + 8) of positions kg + 16 k, k < 4 (16 lanes cover a row: every
  // load instruction reads whole cache lines)
  // MQ: lane i of wave w takes position mp = 16 w + i % 16 and dims 8 (mg + 4 k), mg = i / 16:
  // its B operand of k-step k (32 dims) of v_mfma_f32_16x16x32_f16
  const uint32_t kd = t & 15, kg = t >> 4;
  const uint32_t lane = t & 63, mp = 16 * wave + (lane & 15), mg = lane >> 4;
  uint4 kr[4];
  float ksc[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    if constexpr (MQ) {
      const uint32_t kpos = begin + min(mp, cnt - 1);
      kr[k] = *(const uint4 *)(kv + p.kc_off + kpos * kv_dim + kvh * HD + 8 * (mg + 4 * k));
      ksc[k] = 1.0f;
    } else {
      const uint32_t kpos = begin + min(kg + 16 * k, cnt - 1);
      const uint2 r = *(const uint2 *)(kv8 + p.kc_off + kpos * kv_dim + kvh * HD + 8 * kd);
      kr[k] = make_uint4(r.x, r.y, 0u, 0u);
      ksc[k] = (float)kv[p.ks_off + kpos * (kv_dim / 32) + kvh * 4 + (kd >> 2)];
    }
  }
  // values: dims [8 vg, 8 vg + 8) of positions 4 vq + [0, 4)
  const uint32_t vg = t & 15, vq = t >> 4;
  uint4 vr[4];
  float vsc[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const uint32_t vpos = begin + min(4 * vq + q, cnt - 1);
    if constexpr (!V8) {
      vr[q] = *(const uint4 *)(kv + p.vc_off + vpos * kv_dim + kvh * HD + 8 * vg);
      vsc[q] = 1.0f;
    } else {
      const uint2 r = *(const uint2 *)(kv8 + p.vc_off + vpos * kv_dim + kvh * HD + 8 * vg);
      vr[q] = make_uint4(r.x, r.y, 0u, 0u);
      vsc[q] = (float)kv[p.vs_off + vpos * (kv_dim / 32) + kvh * 4 + (vg >> 2)];
    }
  }
  // the scaled query head j (this lane's dims lane and lane + 64; the caller's wave holds
  // the whole head).  MQ: as f16 hi + lo parts of v 2^sh, sh putting the head's largest
  // |v| in [2^10, 2^11): hi + lo is v 2^sh to 2^-22 of that largest value, nothing
  // overflows, and each product with an f16 key is exact in the f32 accumulation
  auto put_q = [&](uint32_t j, float v0, float v1) {
    if constexpr (MQ) {
      const float big = wave_max(fmaxf(fabsf(v0), fabsf(v1)));
      const int sh = big > 0.0f ? 11 - __builtin_amdgcn_frexp_expf(big) : 0;
      const float s0 = ldexpf(v0, sh), s1 = ldexpf(v1, sh);
      const f16 h0 = (f16)s0, h1 = (f16)s1;
      qh[0][j][lane] = h0;
      qh[0][j][lane + 64] = h1;
      qh[1][j][lane] = (f16)(s0 - (float)h0);
      qh[1][j][lane + 64] = (f16)(s1 - (float)h1);
      if (lane == 0) qsh[j] = sh;
    } else {
      qs[j][lane] = v0;
      qs[j][lane + 64] = v1;
    }
  };
  // the query heads of this kv head, scaled
  const uint32_t q_base = p.q_off + tok * p.q_stride + kvh * N_REP * HD;
  if constexpr (PREP) {
    const uint32_t pos = ctl[1];
    const float *cs = pp->cs_off != NO_TABLE ? a + pp->cs_off : nullptr;
    for (uint32_t j = wave; j < (uint32_t)N_REP; j += 4) {
      float y0, y1;
      norm_rope(w, pp->qn_off, pp->rope_off, pp->eps, pp->mscale, pos, lane, a[q_base + j * HD + lane],
                a[q_base + j * HD + lane + 64], y0, y1, cs);
      put_q(j, y0 * p.scale, y1 * p.scale);
    }
    if (pos / CHUNK == split) {
      if (wave == 0) {
        float y0, y1;
        const uint32_t src = pp->k_off + kvh * HD;
        norm_rope(w, pp->kn_off, pp->rope_off, pp->eps, pp->mscale, pos, lane, a[src + lane], a[src + lane + 64], y0,
                  y1, cs);
        store_kv<K8>(kv, kv8, p.kc_off, p.ks_off, kv_dim, pos, kvh, lane, y0, y1, nk, nks);
      } else if (wave == 1) {
        const uint32_t src = pp->v_off + kvh * HD;
        store_kv<V8>(kv, kv8, p.vc_off, p.vs_off, kv_dim, pos, kvh, lane, a[src + lane], a[src + lane + 64], nv, nvs);
      }
    }
  } else if constexpr (MQ) {
    for (uint32_t j = wave; j < (uint32_t)N_REP; j += 4)
      put_q(j, a[q_base + j * HD + lane] * p.scale, a[q_base + j * HD + lane + 64] * p.scale);
  } else {
    for (uint32_t i = t; i < N_REP * HD; i += 256) qs[i / HD][i % HD] = a[q_base + i] * p.scale;
  }
  __syncthreads();
  if constexpr (PREP) {
    if (ctl[1] / CHUNK == split) {  // the new row (pl = cnt - 1) and the masked slots clamped to it
      const uint32_t pl = cnt - 1;
      if constexpr (MQ) {
        if (mp >= pl)
#pragma unroll
          for (int k = 0; k < 4; k++) kr[k] = ((const uint4 *)nk)[mg + 4 * k];
      } else {
#pragma unroll
        for (int k = 0; k < 4; k++)
          if (kg + 16 * k >= pl) {
            const uint2 u = ((const uint2 *)nk)[kd];
            kr[k] = make_uint4(u.x, u.y, 0u, 0u);
            ksc[k] = nks[kd >> 2];
          }
      }
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (4 * vq + q >= pl) {
          if constexpr (!V8) {
            vr[q] = ((const uint4 *)nv)[vg];
          } else {
            const uint2 u = ((const uint2 *)nv)[vg];
            vr[q] = make_uint4(u.x, u.y, 0u, 0u);
            vsc[q] = nvs[vg >> 2];
          }
        }
    }
  }

  float mx[N_REP];
  if constexpr (MQ) {
    // scores on the matrix cores: A rows are the query heads (hi, then lo parts, each k-step
    // 32 dims), B columns the wave's 16 positions; lane i then holds the scores of heads
    // 4 (i / 16) + r (r < 4, those below N_REP) at position mp
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const uint32_t m = lane & (N_REP - 1);  // A row lane % 16 holds head (lane % 16) % N_REP
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const f16x8 bk = __builtin_bit_cast(f16x8, kr[k]);
#pragma unroll
      for (int part = 0; part < 2; part++)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(*(const f16x8 *)&qh[part][m][8 * (mg + 4 * k)], bk, acc, 0, 0, 0);
    }
    // heads of this lane: 4 mg + r; with at most four heads, only mg = 0 holds any
    constexpr int MGS = N_REP > 4 ? 2 : 1;
    float sr[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const uint32_t h = 4 * mg + r;
      sr[r] = -INFINITY;
      if (h < (uint32_t)N_REP && mp < cnt) sr[r] = ldexpf(acc[r], -qsh[h < (uint32_t)N_REP ? h : 0]);
      // the head's maximum over the wave's 16 positions (one DPP row)
      float v = sr[r];
      v = fmaxf(v, dpp_f<0xb1>(v));
      v = fmaxf(v, dpp_f<0x4e>(v));
      v = fmaxf(v, dpp_f<0x141>(v));
      v = fmaxf(v, dpp_f<0x140>(v));
      if ((lane & 15) == 0 && h < (uint32_t)N_REP) wm[wave][h] = v;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < N_REP; j++) mx[j] = fmaxf(fmaxf(wm[0][j], wm[1][j]), fmaxf(wm[2][j], wm[3][j]));
    if (mg < (uint32_t)MGS) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int h = MGS == 1 ? r : (mg ? 4 + r : r);
        if (h < N_REP) {
          const float mh = MGS == 1 ? mx[r < N_REP ? r : 0] : (mg ? mx[(4 + r) % N_REP] : mx[r % N_REP]);
          es[h][mp] = mp < cnt ? expf(sr[r] - mh) : 0.0f;
        }
      }
    }
    __syncthreads();
  } else {
    float sc[4][N_REP];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      float key[8];
      const uint32_t wd[2] = {kr[k].x, kr[k].y};
#pragma unroll
      for (int bb = 0; bb < 8; bb++) key[bb] = (float)(int8_t)((wd[bb >> 2] >> (8 * (bb & 3))) & 255u) * ksc[k];
#pragma unroll
      for (int j = 0; j < N_REP; j++) {
        const float4 q0 = *(const float4 *)&qs[j][8 * kd], q1 = *(const float4 *)&qs[j][8 * kd + 4];
        float s = 0.0f;
        s = __builtin_fmaf(q0.x, key[0], s);
        s = __builtin_fmaf(q0.y, key[1], s);
        s = __builtin_fmaf(q0.z, key[2], s);
        s = __builtin_fmaf(q0.w, key[3], s);
        s = __builtin_fmaf(q1.x, key[4], s);
        s = __builtin_fmaf(q1.y, key[5], s);
        s = __builtin_fmaf(q1.z, key[6], s);
        s = __builtin_fmaf(q1.w, key[7], s);
        sc[k][j] = lane_sum<16>(s);  // the row's dot, in all 16 lanes
      }
    }
    // The 16 lanes of a group hold the same 4 x N_REP scores, so the wave maximum needs only
    // the two cross-group steps, and each lane then exponentiates its own share of them.
#pragma unroll
    for (int j = 0; j < N_REP; j++) {
      float m = -INFINITY;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        if (kg + 16 * k >= cnt) sc[k][j] = -INFINITY;
        m = fmaxf(m, sc[k][j]);
      }
      m = fmaxf(m, __shfl_xor(m, 16, 64));
      m = fmaxf(m, __shfl_xor(m, 32, 64));
      if ((t & 63) == 0) wm[wave][j] = m;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < N_REP; j++) mx[j] = fmaxf(fmaxf(wm[0][j], wm[1][j]), fmaxf(wm[2][j], wm[3][j]));
    constexpr int NS = 4 * N_REP;  // scores of a lane group: (position k, head j) = (i / N_REP, i % N_REP)
#pragma unroll
    for (int i0 = 0; i0 < NS; i0 += 16) {
      const int i = i0 + (int)kd;
      if (i < NS) {
        float s = -INFINITY, m = 0.0f;
#pragma unroll
        for (int u = i0; u < (i0 + 16 < NS ? i0 + 16 : NS); u++)
          if (u == i) {
            s = sc[u / N_REP][u % N_REP];
            m = mx[u % N_REP];
          }
        const uint32_t pk = kg + 16 * (uint32_t)(i / N_REP);
        es[i % N_REP][pk] = pk < cnt ? expf(s - m) : 0.0f;
      }
    }
    __syncthreads();
  }
  // l = sum of the split's e per head: wave 0 adds the LDS rows while the others go on
  float lrow[N_REP];
  if (wave == 0) {
#pragma unroll
    for (int j = 0; j < N_REP; j++) lrow[j] = wave_sum(es[j][t]);
    if constexpr (DIRECT) {  // every thread divides by l (read after the value round's barrier)
#pragma unroll
      for (int j = 0; j < N_REP; j++)
        if (t == 0) lsh[j] = lrow[j];
    }
  }

  float v[4][8];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    if constexpr (!V8) {
      const uint32_t wd[4] = {vr[q].x, vr[q].y, vr[q].z, vr[q].w};
#pragma unroll
      for (int h = 0; h < 4; h++) {
        const f16x2 x = as_f16x2(wd[h]);
        v[q][2 * h] = (float)x.x;
        v[q][2 * h + 1] = (float)x.y;
      }
    } else {
      const uint32_t wd[2] = {vr[q].x, vr[q].y};
#pragma unroll
      for (int bb = 0; bb < 8; bb++) v[q][bb] = (float)(int8_t)((wd[bb >> 2] >> (8 * (bb & 3))) & 255u) * vsc[q];
    }
  }
  const uint32_t part_base = p.part_off + tok * p.part_stride;
#pragma unroll
  for (int h0 = 0; h0 < N_REP; h0 += HG) {
    if (h0 != 0) __syncthreads();  // the previous round's sums are read
#pragma unroll
    for (int j = 0; j < HG; j++) {
      float acc[8];
#pragma unroll
      for (int i = 0; i < 8; i++) acc[i] = 0.0f;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const float ep = es[h0 + j][4 * vq + q];
#pragma unroll
        for (int i = 0; i < 8; i++) acc[i] = __builtin_fmaf(ep, v[q][i], acc[i]);
      }
      vp[vq][(j * HD + 8 * vg) / 4] = make_float4(acc[0], acc[1], acc[2], acc[3]);
      vp[vq][(j * HD + 8 * vg) / 4 + 1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
    }
    __syncthreads();
    for (uint32_t o = t; o < HG * HD; o += 256) {
      float sum = 0.0f;
#pragma unroll
      for (int g = 0; g < 16; g++) sum += ((const float *)vp[g])[o];
      const uint32_t j = h0 + o / HD;
      if constexpr (DIRECT)
        a[o_off + tok * o_stride + (kvh * N_REP + j) * HD + o % HD] = (sum + 0.0f) / lsh[j];
      else
        a[part_base + ((kvh * N_REP + j) * p.n_split + split) * PART + 2 + o % HD] = sum;
    }
  }
  if constexpr (DIRECT) return;
  if (t < N_REP) {
    const uint32_t base = part_base + ((kvh * N_REP + t) * p.n_split + split) * PART;
    float l = 0.0f, m = 0.0f;
#pragma unroll
    for (int j = 0; j < N_REP; j++)
      if ((uint32_t)j == t) {
        m = mx[j];
        l = lrow[j];
      }
    a[base] = m;
    a[base + 1] = l;
  }
}

// attention of a batched step (attention_rows, the runtime's form of an attention grid of
// several tokens): one wave per (kv head, split of CHUNK positions, 16 query rows), the rows
// being N_REP heads of 16 / N_REP tokens.  It leaves the partials attention_body leaves.
// One workgroup per token re-read the split's key and value rows (24 to 32 KB) for N_REP
// rows and spent its time on staging, barriers and f32 FMAs; here both products run on the
// matrix cores, the rows are read once per 16 queries, and nothing passes through LDS (but in
// the rare splits taken in f32, below):
//   S^T = K Q^T   A = key rows (row: position 16 t + c, c = lane % 16; dims 8 g + 32 k,
//                 g = lane / 16), B = query rows, as loaded; a lane then holds query row c's
//                 scores at positions 16 t + 4 g + r.
//   O^T = V^T P^T B = that lane's own e values: a k-step's element j of group g is position
//                 32 s + 16 (j / 4) + 4 g + j % 4.  A = value rows of those positions, lane c
//                 holding dims 8 c + [0, 8) of each (whole rows a load); tile d takes dim
//                 8 c + d as row c, so the transposition is 8 x 8 inside a lane.
// Precision: what attention_body holds in f32 keeps its 24 bits, as three f16 parts of 11: e 2^15
// (exact from e = 2^-16 of the split's largest, below that to 2^-40) and, over 8-bit keys, the
// query rows v 2^sh (to 2^-39 of the row's largest); over f16 keys the rows are hi + lo, as put_q
// has them.  f16 keys and values and 8-bit keys are exact operands (8-bit keys' scales multiply
// each 32-dim k-step's f32 sums); 8-bit values q s are 18 bits, exact as hi + lo of q s 2^vsh while
// the scales of a block's positions lie within 2^20 of its largest.  Only the product of the last
// parts (2^-33) is left out; sums are f32.  Positions past a row's own have e = 0.  A split with
// scales further apart, or with a value or scale that is not finite, takes its values in f32
// (attention_body's arithmetic), each row over its own positions alone.
// Error against 64 bits over attention_body's on the same inputs, N(0, 1) rows at positions to
// 1517 in every precision, queries of N(0, 1), 8 times that, or spread over 2^12: 0.83 to 1.005
// (with two parts of e and of the query rows and no product of the low parts 0.93 to 1.12, and
// 0.6 us less a launch at most).
// Measured (MI355X, a launch): 128 tokens of Qwen3-8B at positions to 512, f16 keys and 8-bit
// values, 25.9 -> 12.3 us; 60 tokens of Qwen3-0.6B in f16 5.8 -> 5.7 us.  All a wave's loads
// are in flight at once, which two waves a SIMD (256 registers) hold; with one (288 to 320
// registers) and the value loads behind the scores the former ran 16.0 us.  Bound by the
// round trip and, with several waves a SIMD, by the values' conversion and the partials' writes.
template <int N_REP, int K8, int V8>
SK_DEV void attention_rows_body(float *a, const uint32_t *ctl, const f16 *kv, const int8_t *kv8, const AttnPush &p,
                                uint32_t n_grid) {
  constexpr uint32_t TT = 16 / N_REP;
  const uint32_t lane = threadIdx.x, c = lane & 15, g = lane >> 4;
  const uint32_t kvh = blockIdx.x, split = blockIdx.y, tok0 = blockIdx.z * TT, begin = split * CHUNK;
  const uint32_t pos0 = ctl[1], n_tok = min(ctl[2], n_grid), kv_dim = p.n_kv * HD;
  if (tok0 >= n_tok) return;
  const uint32_t last = min(tok0 + TT, n_tok) - 1;  // the last live token of the group
  if (begin >= pos0 + last + 1) return;
  const uint32_t live = min(CHUNK, pos0 + last + 1 - begin);
  // positions of this split that token t attends to
  auto count = [&](uint32_t t) { return pos0 + t + 1 > begin ? min(CHUNK, pos0 + t + 1 - begin) : 0u; };
  // this lane's query row (rows past the last live token repeat it and are not written)
  const uint32_t tok = min(tok0 + c / N_REP, last), j = c % N_REP, cnt = count(tok);

  uint4 kr[4][4];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const uint32_t at = p.kc_off + (begin + min(16 * t + c, live - 1)) * kv_dim + kvh * HD + 8 * g;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if constexpr (K8) {
        const uint2 r = *(const uint2 *)(kv8 + at + 32 * k);
        kr[t][k] = make_uint4(r.x, r.y, 0u, 0u);
      } else {
        kr[t][k] = *(const uint4 *)(kv + at + 32 * k);
      }
    }
  }
  float4 qv[4][2];
  const float *qrow = a + p.q_off + tok * p.q_stride + (kvh * N_REP + j) * HD + 8 * g;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    qv[k][0] = *(const float4 *)(qrow + 32 * k);
    qv[k][1] = *(const float4 *)(qrow + 32 * k + 4);
  }
  f16x4 ks[4][4];  // 8-bit keys: the four block scales of positions 16 t + 4 g + r
  if constexpr (K8)
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        ks[t][r] = *(const f16x4 *)(kv + p.ks_off + (begin + min(16 * t + 4 * g + r, live - 1)) * (kv_dim / 32) + kvh * 4);
  uint4 vr[2][8];
  f16 vs[2][8];
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const uint32_t vpos = begin + min(32 * s + 16 * (e >> 2) + 4 * g + (e & 3), live - 1);
      const uint32_t at = p.vc_off + vpos * kv_dim + kvh * HD + 8 * c;
      if constexpr (V8) {
        const uint2 r = *(const uint2 *)(kv8 + at);
        vr[s][e] = make_uint4(r.x, r.y, 0u, 0u);
        vs[s][e] = kv[p.vs_off + vpos * (kv_dim / 32) + kvh * 4 + (c >> 2)];
      } else {
        vr[s][e] = *(const uint4 *)(kv + at);
        vs[s][e] = (f16)1.0f;
      }
    }

  // every load is issued before the first product (left alone, the compiler moves the value
  // rows' below the scores: a second round trip)
  __builtin_amdgcn_sched_barrier(0);
  // the query row's hi and lo parts
  float q[4][8], big = 0.0f;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const float u[8] = {qv[k][0].x, qv[k][0].y, qv[k][0].z, qv[k][0].w, qv[k][1].x, qv[k][1].y, qv[k][1].z, qv[k][1].w};
#pragma unroll
    for (int e = 0; e < 8; e++) {
      q[k][e] = u[e] * p.scale;
      big = fmaxf(big, fabsf(q[k][e]));
    }
  }
  big = fmaxf(big, __shfl_xor(big, 16, 64));
  big = fmaxf(big, __shfl_xor(big, 32, 64));
  const int sh = big > 0.0f ? (K8 ? 15 : 11) - __builtin_amdgcn_frexp_expf(big) : 0;
  f16x8 qh[4], ql[4], qt[4];  // qt: the third part (8-bit keys)
#pragma unroll
  for (int k = 0; k < 4; k++)
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float s = ldexpf(q[k][e], sh);
      qh[k][e] = (f16)s;
      const float r = s - (float)qh[k][e];
      ql[k][e] = (f16)r;
      if constexpr (K8) qt[k][e] = (f16)(r - (float)ql[k][e]);
    }

  // two bytes picked by sel as an f16 pair: 1024 + (byte ^ 0x80), minus 1152
  auto widen = [](uint32_t hi, uint32_t lo, uint32_t sel) {
    const f16x2 off = {(f16)1152.0f, (f16)1152.0f};
    return as_u32(as_f16x2((__builtin_amdgcn_perm(hi, lo, sel) ^ 0x00800080u) | 0x64006400u) - off);
  };
  float sc[4][4], m = -INFINITY;
#pragma unroll
  for (int t = 0; t < 4; t++) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if constexpr (K8) {
        const uint32_t x = kr[t][k].x, y = kr[t][k].y;
        const uint4 w = make_uint4(widen(x, x, 0x0c010c00u), widen(x, x, 0x0c030c02u), widen(y, y, 0x0c010c00u),
                                   widen(y, y, 0x0c030c02u));
        f32x4 part = {0.0f, 0.0f, 0.0f, 0.0f};
        part = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), qt[k], part, 0, 0, 0);
        part = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), ql[k], part, 0, 0, 0);
        part = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), qh[k], part, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; r++) acc[r] = __builtin_fmaf((float)ks[t][r][k], part[r], acc[r]);
      } else {
        const f16x8 w = __builtin_bit_cast(f16x8, kr[t][k]);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, qh[k], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, ql[k], acc, 0, 0, 0);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      sc[t][r] = 16 * t + 4 * g + r < cnt ? ldexpf(acc[r], -sh) : -INFINITY;
      m = fmaxf(m, sc[t][r]);
    }
  }
  m = fmaxf(m, __shfl_xor(m, 16, 64));
  m = fmaxf(m, __shfl_xor(m, 32, 64));
  // a masked score is -inf and its e is 0 without a branch (a row without positions is not written)
  const float mu = cnt ? m : 0.0f;
  float l = 0.0f;
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      sc[t][r] = expf(sc[t][r] - mu);
      l += sc[t][r];
    }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  const bool writes = tok0 + c / N_REP <= last && cnt != 0;
  const uint32_t base = p.part_off + tok * p.part_stride + ((kvh * N_REP + j) * p.n_split + split) * PART;

  // 8-bit values: the block's largest finite scale goes to [64, 128).  odd: the split takes f32
  int vsh = 0;
  bool odd = false;
  if constexpr (V8) {
    float top = 0.0f;
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float v = fabsf((float)vs[s][e]);
        const bool fin = v < INFINITY;
        odd |= !fin;
        top = fmaxf(top, fin ? v : 0.0f);
      }
    top = fmaxf(top, __shfl_xor(top, 16, 64));
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    vsh = top > 0.0f ? 7 - __builtin_amdgcn_frexp_expf(top) : 0;
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float x = ldexpf((float)vs[s][e], vsh);
        vs[s][e] = (f16)x;
        odd |= (float)vs[s][e] != x;  // too far below the block's largest
      }
  } else {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    u16x2 top = {0, 0};
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const uint32_t u[4] = {vr[s][e].x, vr[s][e].y, vr[s][e].z, vr[s][e].w};
#pragma unroll
        for (int i = 0; i < 4; i++)
          top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, u[i] & 0x7fff7fffu));
      }
    odd = top.x >= 0x7c00 || top.y >= 0x7c00;
  }
  if (__ballot(odd)) {
    // row i's e at [position][i]; lane: dims 2 lane, 2 lane + 1 of every row
    __shared__ float es[CHUNK][16];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) es[16 * t + 4 * g + r][c] = sc[t][r];
    __syncthreads();
    float ox[16], oy[16];
#pragma unroll
    for (int i = 0; i < 16; i++) ox[i] = oy[i] = 0.0f;
    for (uint32_t n = 0; n < live; n++) {
      const uint32_t pos = begin + n, at = p.vc_off + pos * kv_dim + kvh * HD + 2 * lane;
      float vx, vy;
      if constexpr (V8) {
        const float s = (float)kv[p.vs_off + pos * (kv_dim / 32) + kvh * 4 + (lane >> 4)];
        vx = (float)kv8[at] * s;
        vy = (float)kv8[at + 1] * s;
      } else {
        vx = (float)kv[at];
        vy = (float)kv[at + 1];
      }
#pragma unroll
      for (int i = 0; i < 16; i++)
        if (n < count(tok0 + i / N_REP)) {
          ox[i] = __builtin_fmaf(es[n][i], vx, ox[i]);
          oy[i] = __builtin_fmaf(es[n][i], vy, oy[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const uint32_t tk = tok0 + i / N_REP;
      if (tk <= last && count(tk) != 0)
        *(float2 *)(a + p.part_off + tk * p.part_stride + ((kvh * N_REP + i % N_REP) * p.n_split + split) * PART + 2 +
                    2 * lane) = make_float2(ox[i], oy[i]);
    }
    if (g == 0 && writes) *(float2 *)(a + base) = make_float2(m, l);
    return;
  }
  f16x8 ph[2], pm[2], pl[2];  // e 2^15 in three parts
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int s = t >> 1, i = 4 * (t & 1) + r;
      const float x = sc[t][r] * 32768.0f;
      ph[s][i] = (f16)x;
      const float y = x - (float)ph[s][i];
      pm[s][i] = (f16)y;
      pl[s][i] = (f16)(y - (float)pm[s][i]);
    }
  auto word = [](const uint4 &u, int i) { return i == 0 ? u.x : i == 1 ? u.y : i == 2 ? u.z : u.w; };
  f32x4 o[8];
#pragma unroll
  for (int d = 0; d < 8; d++) o[d] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int d = 0; d < 8; d++) {
    f16x8 vh[2], vl[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
      if constexpr (V8) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          // q s rounded once, and what that left (exact): two packed operations a pair
          const uint32_t at = d & 3, sel = 0x0c040c00u + at * 0x00010001u;
          const f16x2 v = as_f16x2(widen(word(vr[s][e + 1], d >> 2), word(vr[s][e], d >> 2), sel));
          const f16x2 sv = {vs[s][e], vs[s][e + 1]};
          const f16x2 hi = v * sv, lo = __builtin_elementwise_fma(v, sv, -hi);
          vh[s][e] = hi.x, vh[s][e + 1] = hi.y;
          vl[s][e] = lo.x, vl[s][e + 1] = lo.y;
        }
      } else {
        const uint32_t sel = d & 1 ? 0x07060302u : 0x05040100u;
        uint32_t u[4];
#pragma unroll
        for (int e = 0; e < 4; e++)
          u[e] = __builtin_amdgcn_perm(word(vr[s][2 * e + 1], d >> 1), word(vr[s][2 * e], d >> 1), sel);
        vh[s] = __builtin_bit_cast(f16x8, make_uint4(u[0], u[1], u[2], u[3]));
      }
    }
    // the smallest products first: the sum rounds at its full size twice
    auto add = [&](const f16x8 &v, const f16x8 &e) {
      o[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, e, o[d], 0, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < 2; s++) add(vh[s], pl[s]);
    if constexpr (V8)
#pragma unroll
      for (int s = 0; s < 2; s++) add(vl[s], pm[s]);
#pragma unroll
    for (int s = 0; s < 2; s++) add(vh[s], pm[s]);
    if constexpr (V8)
#pragma unroll
      for (int s = 0; s < 2; s++) add(vl[s], ph[s]);
#pragma unroll
    for (int s = 0; s < 2; s++) add(vh[s], ph[s]);
  }
  // row 4 g + r of tile d is dim 8 (4 g + r) + d, of block g
  const int back = -15 - __shfl(vsh, (int)(4 * g), 64);
  if (!writes) return;
#pragma unroll
  for (int r = 0; r < 4; r++)
#pragma unroll
    for (int d = 0; d < 8; d += 2)
      *(float2 *)(a + base + 2 + 8 * (4 * g + r) + d) = make_float2(ldexpf(o[d][r], back), ldexpf(o[d + 1][r], back));
  if (g == 0) *(float2 *)(a + base) = make_float2(m, l);
}

}  // namespace

// rmsnorm (rmsnorm.comp; ops.rs:1-16): y = x * r * w, r = 1 / sqrt(mean(x^2) + eps), per
// token below ctl[2].  256 threads; rows of at most 4096 floats at 16-byte aligned offsets
// (every arena row and norm table) are read once as float4, all loads in flight together,
// and kept in registers for the scaling; other rows take a plain loop.  Partial sums of
// squares per wave, added in wave order.
extern "C" __global__ __launch_bounds__(256) void rmsnorm(const float *w, float *a, const uint32_t *ctl,
                                                           NormPush p) {
#pragma clang fp contract(off)
  __shared__ float part[4];
  const uint32_t tok = blockIdx.y, t = threadIdx.x;
  if (tok >= ctl[2]) return;
  const uint32_t x = p.x_off + tok * p.stride, y = p.y_off + tok * p.stride;
  if (((x | y | p.w_off | p.n) & 3u) == 0 && p.n <= 4096) {
    float4 yv[4];
    norm_row4(a + x, w + p.w_off, p.n, p.eps, yv);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t i = t + 256 * k;
      if (i < (p.n >> 2)) ((float4 *)(a + y))[i] = yv[k];
    }
    return;
  }
  float ss = 0.0f;
  for (uint32_t i = t; i < p.n; i += 256) {
    const float v = a[x + i];
    ss += v * v;
  }
  ss = wave_sum(ss);
  if ((t & 63) == 0) part[t >> 6] = ss;
  __syncthreads();
  const float total = ((part[0] + part[1]) + part[2]) + part[3];
  const float r = 1.0f / sqrtf(total / (float)p.n + p.eps);
  for (uint32_t i = t; i < p.n; i += 256) a[y + i] = a[x + i] * r * w[p.w_off + i];
}

// qkv_prep (qkv_prep.comp): per (head, token) wave, QK-norm + RoPE of the q and k heads (q
// rewritten in place, k into the cache) and the value heads copied to the cache.
// Spec [K_Q8, V_Q8, head_dim, n_rot, gated]; exported for head_dim = n_rot = 128, gated 0.
#define QKV(K8, V8)                                                                            \
  extern "C" __global__ __launch_bounds__(64) void qkv_prep__##K8##_##V8##_128_128_0(         \
      const float *w, float *a, const uint32_t *ctl, f16 *kv, int8_t *kv8, QkvPush p) {       \
    qkv_body<K8, V8>(w, a, ctl, kv, kv8, p);                                                   \
  }
QKV(0, 0)
QKV(0, 1)
QKV(1, 1)

// attention (attention.comp): spec [N_REP, CHUNK, K_Q8, V_Q8, head_dim, q_head].
// Six waves per SIMD for the forms of at most four query heads per kv head (at most 80
// VGPRs, no spill; about 20 KB of LDS, six workgroups per CU); eight heads keep their
// registers.
#define ATTN(R, K8, V8)                                                                          \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(R == 8 ? 1 : 6))) void attention__##R##_64_##K8##_##V8##_128_128(   \
      float *a, const uint32_t *ctl, const f16 *kv, const int8_t *kv8, const f16 *kvs, AttnPush p) { \
    (void)kvs;                                                                                   \
    attention_body<R, K8, V8>(nullptr, a, ctl, const_cast<f16 *>(kv), const_cast<int8_t *>(kv8), p, nullptr); \
  }                                                                                              \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(R == 8 ? 1 : 6))) void attention_prep__##R##_64_##K8##_##V8##_128_128( \
      const float *w, float *a, const uint32_t *ctl, f16 *kv, int8_t *kv8, PrepPush pp) {        \
    const AttnPush p = {pp.q_off, pp.part_off, pp.kc_off, pp.vc_off, pp.n_kv, pp.n_split,         \
                        pp.scale, 0u, pp.part_stride, pp.ks_off, pp.vs_off};                     \
    attention_body<R, K8, V8, true>(w, a, ctl, kv, kv8, p, &pp);                                 \
  }                                                                                              \
  extern "C" __global__ __launch_bounds__(256) void attention_prep1__##R##_64_##K8##_##V8##_128_128( \
      const float *w, float *a, const uint32_t *ctl, f16 *kv, int8_t *kv8, PrepPush1 q) {        \
    const PrepPush &pp = q.pp;                                                                   \
    const AttnPush p = {pp.q_off, pp.part_off, pp.kc_off, pp.vc_off, pp.n_kv, pp.n_split,         \
                        pp.scale, 0u, pp.part_stride, pp.ks_off, pp.vs_off};                     \
    attention_body<R, K8, V8, true, true>(w, a, ctl, kv, kv8, p, &pp, q.o_off, q.o_stride);      \
  }
#define ATTN_REP(K8, V8) ATTN(1, K8, V8) ATTN(2, K8, V8) ATTN(4, K8, V8) ATTN(8, K8, V8)
ATTN_REP(0, 0)
ATTN_REP(0, 1)
ATTN_REP(1, 1)

#define ATTN_ROWS(R, K8, V8)                                                                     \
  extern "C" __global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void attention_rows__##R##_64_##K8##_##V8##_128_128( \
      float *a, const uint32_t *ctl, const f16 *kv, const int8_t *kv8, const f16 *kvs, AttnPush p,  \
      uint32_t n_grid) {                                                                         \
    (void)kvs;                                                                                   \
    attention_rows_body<R, K8, V8>(a, ctl, kv, kv8, p, n_grid);                                  \
  }
#define ATTN_ROWS_REP(K8, V8) ATTN_ROWS(1, K8, V8) ATTN_ROWS(2, K8, V8) ATTN_ROWS(4, K8, V8) ATTN_ROWS(8, K8, V8)
ATTN_ROWS_REP(0, 0)
ATTN_ROWS_REP(0, 1)
ATTN_ROWS_REP(1, 1)

// attention_merge (attention_merge.comp): o = sum_s w_s acc_s / sum_s w_s l_s with
// w_s = exp(m_s - max m) over the splits that hold positions.  Spec [head_dim, gated] =
// [128, 0].  One workgroup of 1024 threads per (head, token).  Wave w takes the splits
// s = w + 16 i; lane l holds dims 2 l and 2 l + 1.  Every load of a round of 1024 splits is
// issued before any arithmetic: lane j loads (m, l) of the wave's split i = j, and each lane
// its two dims of the wave's splits, MG at a time.  A wave keeps its own running maximum
// M_w, and its sums over its splits weighted by exp(m_s - M_w); the waves then meet in LDS:
// M = max M_w, and each wave's sums are scaled by exp(M_w - M) before they are added in
// wave order.  That is the same quantity as the reference's single pass with M from the
// start, in another rounding: exp(m_s - M_w) exp(M_w - M) for exp(m_s - M).  Over a single
// split every factor is exp(0) = 1, so o = (acc + 0) / l, the bits attention_prep1 writes.
constexpr uint32_t MAX_SPLITS = 4096;  // 262144 positions; the engine's arena stays below
constexpr uint32_t MG = 24;            // a wave's splits whose loads are in flight together

extern "C" __global__ __launch_bounds__(1024) void attention_merge__128_0(float *a, const uint32_t *ctl,
                                                                           MergePush p) {
  __shared__ float wmax[16], wl[16];
  __shared__ float2 sums[16][HD / 2];
  const uint32_t h = blockIdx.x, tok = blockIdx.y, t = threadIdx.x, wave = t >> 6, lane = t & 63;
  if (tok >= ctl[2]) return;
  const uint32_t used = min(min((ctl[1] + tok + p.chunk) / p.chunk, p.n_split), MAX_SPLITS);
  const uint32_t first = p.part_off + tok * p.part_stride + h * p.n_split * PART;
  float mw = -INFINITY, lw = 0.0f, ax = 0.0f, ay = 0.0f;
  for (uint32_t base = 0; base < used; base += 1024) {
    // this pass's splits of the wave: s_i = base + wave + 16 i, i < n_i
    const uint32_t s0 = base + wave;
    const uint32_t n_i = s0 < used ? min(64u, (used - s0 + 15) / 16) : 0u;
    if (n_i == 0) break;  // wave-uniform; no later round holds a split of this wave either
    const uint32_t sj = s0 + 16 * lane;
    const bool live = lane < n_i;
    const float mj = live ? a[first + sj * PART] : -INFINITY;
    const float lj = live ? a[first + sj * PART + 1] : 0.0f;
    float2 v[MG];
#pragma unroll
    for (uint32_t i = 0; i < MG; i++)
      v[i] = i < n_i ? *(const float2 *)(a + first + (s0 + 16 * i) * PART + 2 + 2 * lane) : make_float2(0.f, 0.f);
    const float mn = fmaxf(mw, wave_max(mj));
    const float r = expf(mw - mn);  // 0 in the first round (mw = -inf)
    const float wj = expf(mj - mn);  // 0 for lanes past n_i
    lw = __builtin_fmaf(lw, r, wave_sum(wj * lj));
    ax *= r;
    ay *= r;
#pragma unroll
    for (uint32_t i = 0; i < MG; i++) {
      const float wi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wj), (int)i));
      ax = __builtin_fmaf(wi, v[i].x, ax);
      ay = __builtin_fmaf(wi, v[i].y, ay);
    }
    for (uint32_t i = MG; i < n_i; i++) {  // past MG splits of the wave in one round (long contexts)
      const float wi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wj), (int)i));
      const float2 u = *(const float2 *)(a + first + (s0 + 16 * i) * PART + 2 + 2 * lane);
      ax = __builtin_fmaf(wi, u.x, ax);
      ay = __builtin_fmaf(wi, u.y, ay);
    }
    mw = mn;
  }
  if (lane == 0) wmax[wave] = mw;
  __syncthreads();
  float big = wmax[0];
#pragma unroll
  for (int w = 1; w < 16; w++) big = fmaxf(big, wmax[w]);
  const float f = expf(mw - big);  // 0 for a wave without splits (mw = -inf)
  sums[wave][lane] = make_float2(ax * f, ay * f);
  if (lane == 0) wl[wave] = lw * f;
  __syncthreads();
  if (t < HD) {
    float o = 0.0f, total = 0.0f;
#pragma unroll
    for (int g = 0; g < 16; g++) {
      o += ((const float *)sums[g])[t];
      total += wl[g];
    }
    a[p.o_off + tok * p.o_stride + h * HD + t] = o / total;
  }
}

// attention_merge for batched steps (prefill chunks, grid [ceil(n_head / 4), tokens] by the
// runtime): one wave per (head, token), lane l the head's dims 2l and 2l + 1.  The split
// weights exp(m_s - M) are formed 64 at a time, one per lane, and broadcast by readlane (the
// split index is wave-uniform).  The same quantity as attention_merge__128_0 in another
// summation order; a prefill token has few splits, which the 1024-thread form leaves idle.
SK_DEV float2 merge_head(const float *a, const uint32_t *ctl, const MergePush &p, uint32_t h, uint32_t tok,
                         uint32_t lane) {
  const uint32_t used = min(min((ctl[1] + tok + p.chunk) / p.chunk, p.n_split), MAX_SPLITS);
  const uint32_t first = p.part_off + tok * p.part_stride + h * p.n_split * PART;
  if (used <= 16) {
    // at most 16 splits (a prefill chunk within 1024 positions): every load in flight at
    // once, then the arithmetic below in the same order (the same bits)
    float ml = -INFINITY, ll = 0.0f, vx[16], vy[16];
    if (lane < used) {
      ml = a[first + lane * PART];
      ll = a[first + lane * PART + 1];
    }
#pragma unroll
    for (uint32_t j = 0; j < 16; j++)
      if (j < used) {
        vx[j] = a[first + j * PART + 2 + 2 * lane];
        vy[j] = a[first + j * PART + 3 + 2 * lane];
      }
    const float big = wave_max(ml);
    const float wl = lane < used ? expf(ml - big) : 0.0f;
    float total = lane < used ? __builtin_fmaf(wl, ll, 0.0f) : 0.0f;
    float ox = 0.0f, oy = 0.0f;
#pragma unroll
    for (uint32_t j = 0; j < 16; j++)
      if (j < used) {
        const float wj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wl), (int)j));
        ox = __builtin_fmaf(wj, vx[j], ox);
        oy = __builtin_fmaf(wj, vy[j], oy);
      }
    total = wave_sum(total);
    return make_float2(ox / total, oy / total);
  }
  float big = -INFINITY;
  for (uint32_t s = lane; s < used; s += 64) big = fmaxf(big, a[first + s * PART]);
  big = wave_max(big);
  float total = 0.0f, ox = 0.0f, oy = 0.0f;
  for (uint32_t s0 = 0; s0 < used; s0 += 64) {
    const uint32_t s = s0 + lane;
    const float wl = s < used ? expf(a[first + s * PART] - big) : 0.0f;
    if (s < used) total = __builtin_fmaf(wl, a[first + s * PART + 1], total);
    const uint32_t n = min(used - s0, 64u);
    for (uint32_t j = 0; j < n; j++) {
      const float wj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wl), (int)j));
      const float *v = a + first + (s0 + j) * PART + 2 + 2 * lane;
      ox = __builtin_fmaf(wj, v[0], ox);
      oy = __builtin_fmaf(wj, v[1], oy);
    }
  }
  total = wave_sum(total);
  return make_float2(ox / total, oy / total);
}
extern "C" __global__ __launch_bounds__(256) void attention_merge_t__128_0(float *a, const uint32_t *ctl,
                                                                             MergePush p, uint32_t n_head,
                                                                             uint32_t n_tok) {
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint32_t h = blockIdx.x * 4 + wave, tok = blockIdx.y;
  (void)n_tok;
  if (tok >= ctl[2] || h >= n_head) return;
  const float2 v = merge_head(a, ctl, p, h, tok, lane);
  float *o = a + p.o_off + tok * p.o_stride + h * HD + 2 * lane;
  o[0] = v.x;
  o[1] = v.y;
}

// attention_merge_t with the f16 row prepass of the matmul that reads its rows (o) in the same
// launch: the f32 rows as attention_merge_t writes them, and each row's f16 values and
// exponent (or the runs' exponents) at out as x_half_rows (matmul.hip) writes them: x 2^-e in the
// order 0, 2, 1, 3 of every four, e = 0 unless the row's largest |x| reaches 2^15.  The row
// passes through LDS; sixteen waves, a head each at a time (n_head <= MHEADS).  The separate prepass read back
// what the launch before it wrote, its time mostly the launch's own.  Measured (MI355X, merge +
// prepass -> one launch): 128 tokens of 32 heads at positions to 512 5.2 + 4.8 -> 8.1 us, 60
// tokens of 16 heads in one split 4.5 + 4.3 -> 4.6 us.  Bound by a head's two dependent round
// trips (with four waves a workgroup, eight heads each, the two launches were faster, as they are
// with more heads or many splits: the runtime's merge_joins).  Grid: one workgroup per token.
constexpr uint32_t MHEADS = 32;
struct MergeHalfPush {
  MergePush m;
  uint32_t n_head, h_off, e_off;
};
extern "C" __global__ __launch_bounds__(1024) void attention_merge_half(float *a, uint32_t *out, const uint32_t *ctl,
                                                                        MergeHalfPush q) {
  __shared__ __attribute__((aligned(16))) float row[MHEADS * HD];
  __shared__ float wm[16];
  __shared__ uint32_t big[16];
  const uint32_t t = threadIdx.x, wave = t >> 6, lane = t & 63, tok = blockIdx.x;
  const MergePush &p = q.m;
  if (tok >= ctl[2]) return;
  float m = 0.0f;
  bool b = false;  // NaN counts as big, as in x_half_rows
  for (uint32_t h = wave; h < q.n_head; h += 16) {
    const float2 v = merge_head(a, ctl, p, h, tok, lane);
    *(float2 *)(a + p.o_off + tok * p.o_stride + h * HD + 2 * lane) = v;
    *(float2 *)&row[h * HD + 2 * lane] = v;
    const float mh = fmaxf(fabsf(v.x), fabsf(v.y));
    m = fmaxf(m, mh);
    b |= !(mh < 32768.0f);
  }
  m = wave_max(m);
  const uint64_t anyb = __ballot(b);
  if (lane == 0) {
    wm[wave] = m;
    big[wave] = anyb != 0;
  }
  __syncthreads();
  float tm = wm[0];
  uint32_t any = big[0];
#pragma unroll
  for (int i = 1; i < 16; i++) {
    tm = fmaxf(tm, wm[i]);
    any |= big[i];
  }
  const int e = any ? range_exp(tm) : 0;
  float sc = __builtin_ldexpf(1.0f, -e);
  const uint32_t n = q.n_head * HD;
  f16 *half = (f16 *)(out + q.h_off) + (size_t)tok * n;
  for (uint32_t k = 4 * t; k < n; k += 4096) {
    float4 v = *(const float4 *)&row[k];
    if (e && q.e_off) {  // an exponent per run of 128 values (n is a multiple of 128)
      const int er = run_exp(v);
      sc = __builtin_ldexpf(1.0f, -er);
      if ((t & 31) == 0) out[q.e_off + tok * (n / E_RUN) + k / E_RUN] = (uint32_t)er;
    }
    if (e) v = make_float4(v.x * sc, v.y * sc, v.z * sc, v.w * sc);
    *(uint2 *)(half + k) = make_uint2(as_u32(pack_f16x2(v.x, v.z)), as_u32(pack_f16x2(v.y, v.w)));
  }
  if (t == 0) out[tok] = (uint32_t)e;
}

// take_last (take_last.comp): the last token row of a chunk, for the output head.
extern "C" __global__ __launch_bounds__(256) void take_last(float *a, const uint32_t *ctl, LastPush p) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < p.n) a[p.dst_off + i] = a[p.src_off + (ctl[2] - 1) * p.stride + i];
}
