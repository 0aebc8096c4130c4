// k_attn.hip — attention over many query rows (prefill) in one pass: bf16 MFMA with f32 accumulation,
// and an all-f32 variant for a backend without the bf16 flag.
//
// The op sequence of catgrad-llm/src/models/llama.rs:95-107 (also gemma3.rs:153-186):
//   scores = matmul(q, transpose(k));  scores / sqrt(d);  + mask;  softmax;  matmul(., v)
// materialises [b, h, S, T] twice on the generic path.  Here a workgroup takes 128 (or 64) query rows of one
// (batch, head) and walks the keys 64 at a time with the running maximum / sum of the row
// (online softmax); scores and probabilities only ever exist in registers.
//
// Everything is computed transposed so that a lane owns one query for the whole kernel:
//   S^T[key, query]   = K[key, :] . Q[query, :]       A = K tile (LDS), B = Q rows (registers)
//   O^T[dim, query]  += V^T[dim, key] . P^T[key, query]  A = V^T tile (LDS), B = P^T (registers)
// In the 32x32 MFMA result layout a lane holds column (lane & 31) = its query, so the row
// statistics are in-lane reductions plus one exchange with lane ^ 32, the rescaling of O by
// exp(m_old - m_new) is a per-lane scalar, and P^T feeds the second product straight from the
// registers of the first: the key order inside each 16-key block is permuted the same way for
// both operands (a lane's eight values are keys {4h..4h+3, 8+4h..8+4h+3}, h = lane >> 5), which
// the V^T fragment mirrors with two 8-byte LDS reads.
#include <hip/hip_runtime.h>
#include <math.h>
#include "launch.hpp"
#include "dev_common.hpp"

namespace cgk {

typedef __attribute__((ext_vector_type(8))) __bf16 a_bf16x8;
typedef __attribute__((ext_vector_type(16))) float a_f32x16;

typedef __attribute__((ext_vector_type(2))) __bf16 a_bf16x2;
typedef __attribute__((ext_vector_type(2))) float a_f32x2;

// eight floats -> eight bf16 (round to nearest even: v_cvt_pk_bf16_f32, one instruction per pair)
__device__ __forceinline__ a_bf16x8 pack8(const float *v) {
  union {
    a_bf16x2 h2[4];
    a_bf16x8 h;
  } r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r.h2[i] = __builtin_convertvector((a_f32x2){v[2 * i], v[2 * i + 1]}, a_bf16x2);
  return r.h;
}

// The values of this lane and of the one 32 lanes away, the lower half's first: v_permlane32_swap_b32, two VALU cycles where
// a trip through the LDS crossbar costs a step of these kernels over a hundred.
__device__ __forceinline__ float2 both_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return make_float2(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float max_of_halves(float v) {
  const float2 p = both_halves(v);
  return fmaxf(p.x, p.y);
}
__device__ __forceinline__ float sum_of_halves(float v) {
  const float2 p = both_halves(v);
  return p.x + p.y;
}

// The classes of one query tile's key tiles (AttnPrefillDesc::tile_class), as the kernels walk them.  A row
// of up to 128 entries is read once, by the lanes of a wave, and kept as bit masks: finding the next
// live tile is then bit arithmetic, not a chain of dependent loads.
template <int BN>
struct KeyTiles {
  const uint8_t *cls;  // null: no table, every tile is visited and reads its mask values
  uint32_t cols, t;
  uint64_t live[2], zero[2];  // bit i of word w: tile 64 w + i is not dead / needs no mask values
  bool bits;
  uint32_t c0, c1;
  // asks for the row; what is asked for between here and arrived() travels with it
  __device__ __forceinline__ KeyTiles(const AttnPrefillDesc &a, uint32_t q_tile, int lane) {
    cls = a.tile_class ? a.tile_class + (size_t)q_tile * a.tile_cols : nullptr;
    cols = a.tile_cols;
    t = a.t;
    bits = cls && cols <= 128;
    c0 = c1 = 0;
    if (bits) {
      c0 = cls[min((uint32_t)lane, cols - 1)];
      c1 = cls[min((uint32_t)lane + 64, cols - 1)];
    }
  }
  __device__ __forceinline__ void arrived(int lane) {
    live[0] = live[1] = zero[0] = zero[1] = 0;
    if (bits) {
      if ((uint32_t)lane >= cols) c0 = 0;
      if ((uint32_t)lane + 64 >= cols) c1 = 0;
      live[0] = __ballot(c0 != 0);
      live[1] = __ballot(c1 != 0);
      zero[0] = __ballot(c0 == 2);
      zero[1] = __ballot(c1 == 2);
    }
  }
  // the first step at or after t0 that is not dead (>= t: none)
  __device__ __forceinline__ uint32_t next_step(uint32_t t0) const {
    if (!cls) return t0;
    uint32_t i = t0 / BN;
    if (bits) {
      if (i < 64) {
        const uint64_t m = live[0] >> i;
        if (m) return (i + (uint32_t)__builtin_ctzll(m)) * (uint32_t)BN;
        i = 64;
      }
      const uint64_t m = i < 128 ? live[1] >> (i - 64) : 0;
      return (m ? i + (uint32_t)__builtin_ctzll(m) : cols) * (uint32_t)BN;
    }
    while (i < cols && cls[i] == 0) ++i;
    return i * (uint32_t)BN;
  }
  // the n-th live step after the one at t0
  __device__ __forceinline__ uint32_t skip(uint32_t t0, int n) const {
    for (int i = 0; i < n && t0 < t; ++i) t0 = next_step(t0 + BN);
    return t0;
  }
  __device__ __forceinline__ uint32_t live_steps() const {
    if (bits) return (uint32_t)(__builtin_popcountll(live[0]) + __builtin_popcountll(live[1]));
    uint32_t n = 0;
    for (uint32_t t0 = next_step(0); t0 < t; t0 = next_step(t0 + BN)) ++n;
    return n;
  }
  // does the step at t0 read mask values (given that there is a mask)?
  __device__ __forceinline__ bool reads_mask(uint32_t t0) const {
    if (!cls || t0 >= t) return true;
    const uint32_t i = t0 / BN;
    return bits ? !(((i < 64 ? zero[0] : zero[1]) >> (i & 63)) & 1) : cls[i] != 2;
  }
};

constexpr float ATTN_MAX_SLACK = 8.0f;

// One step of the online softmax: the scores S^T of KT x 32 keys (register e of tile kt is key t0 + kt*32 + (e>>2)*8 +
// half*4 + (e&3)) become the B fragments of the second product, and the row's maximum and sum move on.  `l` sums this
// lane's keys only: the two lanes of a query meet after the last step.  Returns the factor O has to be rescaled by.
//
// Most steps of a causal or sliding-window layer read no mask and have no key past the end: there a score costs a
// maximum, one fma and an exp2 (the scale and log2 e in the factor; the scale is positive there), a sum and half a
// conversion.  One path with the tail's and the mask's selects took 541 vector instructions for 32 scores a lane; this one
// takes 110.  With it, one barrier a step and the long query tiles first: 2900 tokens of 32 heads of 64 212 -> 96 us a
// layer, 8 x 2048 of 4 heads of 256 227 -> 168, 4 x 256 of 16 heads of 128 26.6 -> 22.7, 512 of 32 heads of 64 17.0 -> 14.9.
// LATE: the mask values are asked for here, not handed in: 32 registers less across the score product, which is a third wavefront to
// a SIMD for heads of 64 (2900 tokens 97.6 -> 89.8 us, 4000 154 -> 132), and a trip to L2 in the few steps that read a mask.
template <int KT, bool LATE>
__device__ __forceinline__ float attn_softmax_step(const AttnPrefillDesc &a, a_f32x16 (&st)[KT], const float *M, const float4 (&early)[KT][4],
                                                   a_bf16x8 (&pf)[KT * 2], float &m_run, float &l_run, float inv_scale, bool plain,
                                                   bool use_mask, uint32_t t0, int half, bool mask_covers = false) {
  constexpr float LOG2E = 1.44269504f, LOWEST = -3.40282347e+38f;
  float tmax = LOWEST, alpha, psum = 0.f;
  if (plain) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int e = 0; e < 16; ++e) tmax = fmaxf(tmax, st[kt][e]);
    tmax = max_of_halves(tmax) * inv_scale;
    const float m_new = tmax > m_run + ATTN_MAX_SLACK ? tmax : m_run;
    alpha = __expf(m_run - m_new);
    m_run = m_new;
    const float c = inv_scale * LOG2E, ref = fmaxf(m_new * LOG2E, LOWEST);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int blk = 0; blk < 2; ++blk) {
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[kt][blk * 8 + i], c, -ref));
          psum += p[i];
        }
        pf[kt * 2 + blk] = pack8(p);
      }
  } else if (const bool tail = t0 + KT * 32 > a.t; use_mask && (!tail || mask_covers)) {  // (uniform)
    // (mask_covers: the keys past the end are zeros, and the mask's padded row has f32::MIN for them)
    // Mask values and no key past the end: the general form below without its selects, half of the vector instructions (us a layer,
    // causal, with and before: 32 heads of 64, 2900 tokens 87.3, 89.5; 16 heads of 128, 4 x 256 tokens 17.8, 18.5).
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4 m = LATE ? *(const float4 *)(M + min(t0 + kt * 32 + j * 8 + half * 4, a.m_len - 4)) : early[kt][j];
        const float mv[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = st[kt][j * 4 + i] * inv_scale + mv[i];
          st[kt][j * 4 + i] = v;
          tmax = fmaxf(tmax, v);
        }
      }
    tmax = max_of_halves(tmax);
    const float m_new = tmax > m_run + ATTN_MAX_SLACK ? tmax : m_run;
    alpha = __expf(m_run - m_new);
    m_run = m_new;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int blk = 0; blk < 2; ++blk) {
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          p[i] = __expf(st[kt][blk * 8 + i] - m_new);
          psum += p[i];
        }
        pf[kt * 2 + blk] = pack8(p);
      }
  } else {  // the only step with keys past the end, or a constant in the mask's place
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      float4 mask[4];
      if (use_mask) {
#pragma unroll
        for (int j = 0; j < 4; ++j) mask[j] = LATE ? *(const float4 *)(M + min(t0 + kt * 32 + j * 8 + half * 4, a.m_len - 4)) : early[kt][j];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t key = t0 + kt * 32 + j * 8 + half * 4;
        float mv[4] = {0.f, 0.f, 0.f, 0.f};
        if (use_mask) { mv[0] = mask[j].x; mv[1] = mask[j].y; mv[2] = mask[j].z; mv[3] = mask[j].w; }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = st[kt][j * 4 + i];
          if (a.has_scale) v = v * inv_scale;
          if (use_mask) v = v + mv[i];
          else if (!a.mask && a.has_mask_const) v = v + a.mask_const;
          if (tail && key + i >= a.t) v = LOWEST;  // past the end: contributes exp(..) = 0
          st[kt][j * 4 + i] = v;
          tmax = fmaxf(tmax, v);
        }
      }
    }
    tmax = max_of_halves(tmax);
    const float m_new = tmax > m_run + ATTN_MAX_SLACK ? tmax : m_run;
    alpha = __expf(m_run - m_new);
    m_run = m_new;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int blk = 0; blk < 2; ++blk) {
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const uint32_t key = t0 + kt * 32 + (blk * 2 + (i >> 2)) * 8 + half * 4 + (i & 3);
          p[i] = __expf(st[kt][blk * 8 + i] - m_new);
          if (tail && key >= a.t) p[i] = 0.f;
          psum += p[i];
        }
        pf[kt * 2 + blk] = pack8(p);
      }
  }
  l_run = l_run * alpha + psum;
  return alpha;
}

// BN keys per step.  The K / V rows of step i + 1 are in registers, asked for a step ago, while step i is computed from
// one LDS buffer, and go to the other buffer behind its first product: one barrier per step.
// NW waves of 32 queries each per workgroup (4, or 2 when that is what it takes to occupy the CUs).
// KG = 2: half of the waves share their queries with the other half and take every other live step of them, with tiles of their own;
// the partial results meet once, in LDS.  The longest query tile of a causal mask is then half as long.
// DS = 2: two waves share 32 queries, each with half of the values' dims.
// LEAN: bf16 in and out (AttnPrefillDesc::q16), for a result that only products read.
// Workgroups: the query tiles with the most keys first (a causal mask gives the last tile all of them), and the heads of a
// (batch, kv head) on one XCD, whose L2 then holds their keys and values.
// (the register budget of two waves to a SIMD keeps the accumulators of heads of 64 and 128 out of the accumulation file,
// 64 moves a step.  Heads of 64 have room for three since the mask values are asked for where they are used and the products of a
// step take turns between accumulators: 2900 tokens of 32 heads, causal, 90 us a layer where two waves and one chain after the
// other took 97, 4000 tokens 131 for 154)
#define ATTN_WAVES(n) __attribute__((amdgpu_waves_per_eu(n, n)))
template <int D, int BN, int NW, int KG = 1, int DS = 1, bool LEAN = false>
__global__ void __launch_bounds__(NW * 64) ATTN_WAVES((D == 64 && NW == 4 && (KG == 1 || BN == 32) ? 3 : 2)) attn_prefill_kernel(AttnPrefillDesc a) {
  warm_kernel_arguments<sizeof(AttnPrefillDesc)>();
  constexpr int NT = NW * 64 / KG, NQ = NW / KG / DS, QROWS = NQ * 32;  // threads of a key group; query groups, queries of the workgroup
  constexpr int KP = D + 8;              // K tile row pitch (bf16 elements)
  constexpr int VP = BN + 8;             // V^T tile row pitch
  constexpr int DT = D / 32 / DS;        // 32-row tiles of O^T of a wave
  constexpr int KT = BN / 32;            // 32-key tiles of S^T
  constexpr int KCH = BN * D / 8 / NT;   // 16-byte chunks of the K tile / of the V^T tile per thread
  constexpr int TILE = BN * KP + D * VP;
  __shared__ __attribute__((aligned(16))) uint16_t tile[KG][2][TILE];
  const int lane = threadIdx.x & 63, all_waves = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = KG == 1 ? 0 : all_waves / (NW / KG), of_group = KG == 1 ? all_waves : all_waves % (NW / KG), tid = of_group * 64 + lane;
  const int wave = DS == 1 ? of_group : of_group % NQ, dim0 = DS == 1 ? 0 : of_group / NQ * (D / DS);
  const int col = lane & 31, half = lane >> 5;
  const uint32_t n_bh = a.heads * a.b, q_tiles = (a.s + QROWS - 1) / QROWS;
  const uint32_t rank = blockIdx.x / n_bh, slot = blockIdx.x - rank * n_bh, q_tile = q_tiles - 1 - rank;
  const uint32_t bh = n_bh % 8 == 0 ? (slot % 8) * (n_bh / 8) + slot / 8 : slot;
  const uint32_t b = bh / a.heads, h = bh - b * a.heads;
  const uint32_t kvh = h / a.rep, rp = h % a.rep;
  const uint32_t query = q_tile * QROWS + wave * 32 + col;
  const bool q_ok = query < a.s;
  const uint32_t qc = q_ok ? query : a.s - 1;  // loads of lanes past the end go to a valid row
  const int64_t q_at = (int64_t)b * a.q_sb + (int64_t)h * a.q_sh + (int64_t)qc * a.q_ss;
  // K rows as bf16 (the twin of the rotated keys), V as bf16 V^T [b, kv, d, T]: both were narrowed
  // once, not once per query block
  const uint16_t *K = a.k16 + (int64_t)b * a.k_sb + (int64_t)kvh * a.k_skv + (int64_t)rp * a.k_srep;
  const uint16_t *VT = a.vt16 + ((int64_t)b * (a.heads / a.rep) + kvh) * D * (int64_t)a.vt_st;
  const float *V = a.v + (int64_t)b * a.v_sb + (int64_t)kvh * a.v_skv + (int64_t)rp * a.v_srep;
  const float *M = a.mask ? a.mask + (int64_t)b * a.m_sb + (int64_t)h * a.m_sh + (int64_t)qc * a.m_ss : nullptr;

  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  u32x4 kreg[KCH], vreg[KCH];  // the step in flight
  // All loads are unconditional so that they are issued back to back; chunks past the end are zeroed when the registers are
  // consumed.  With a class table, dead key tiles are never visited and all-zero ones need no mask values.  This thread's first
  // chunk of each tile is kept as a pointer; a step without the end of the keys in it is a scalar away from there (with every
  // index clamped and every product taken in every step, a quarter of the step's vector instructions).
  KeyTiles<BN> tiles(a, q_tile, lane);
  // this lane's query row as B fragments: k-step ks covers dims 16 ks .. 16 ks + 15, half h takes 8 (lanes past the end repeat the
  // last row; what they compute goes nowhere)
  float4 qx[LEAN ? 1 : D / 8];
  a_bf16x8 qf[D / 16];
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) {
    if constexpr (LEAN) {
      qf[ks] = *(const a_bf16x8 *)(a.q16 + q_at + ks * 16 + half * 8);
    } else {
      qx[2 * ks] = *(const float4 *)(a.q + q_at + ks * 16 + half * 8);
      qx[2 * ks + 1] = *(const float4 *)(a.q + q_at + ks * 16 + half * 8 + 4);
    }
  }
  tiles.arrived(lane);
  constexpr int KROWS = NT * 8 / D, VROWS = NT * 8 / BN;  // rows of the K tile, of the V^T tile, between a thread's chunks
  const uint32_t k_row = tid / (D / 8), k_d8 = (tid % (D / 8)) * 8, v_row = tid / (BN / 8), v_k8 = (tid % (BN / 8)) * 8;
  const char *kp = (const char *)(K + (int64_t)k_row * a.k_st + k_d8), *vp = (const char *)(VT + (int64_t)v_row * a.vt_st + v_k8);
  const int64_t k_step = a.k_st * 2, v_chunk = (int64_t)VROWS * a.vt_st * 2;
  auto fetch = [&](uint32_t at) {
    const uint32_t t0 = __builtin_amdgcn_readfirstlane(at);
    if (t0 + BN <= a.t) {
#pragma unroll
      for (int c = 0; c < KCH; ++c) kreg[c] = *(const u32x4 *)(kp + (int64_t)(t0 + c * KROWS) * k_step);
#pragma unroll
      for (int c = 0; c < KCH; ++c) vreg[c] = *(const u32x4 *)(vp + (c * v_chunk + (int64_t)t0 * 2));
      return;
    }
#pragma unroll
    for (int c = 0; c < KCH; ++c) kreg[c] = *(const u32x4 *)(K + (int64_t)min(t0 + k_row + c * KROWS, a.t - 1) * a.k_st + k_d8);
#pragma unroll
    for (int c = 0; c < KCH; ++c) vreg[c] = *(const u32x4 *)(VT + (int64_t)(v_row + c * VROWS) * a.vt_st + min(t0 + v_k8, a.vt_st - 8));
  };
  uint16_t *const k_at = &tile[kg][0][k_row * KP + k_d8], *const v_at = &tile[kg][0][BN * KP + v_row * VP + v_k8];
  auto stash = [&](int to, uint32_t at) {  // registers -> LDS: K [BN, D] and V^T [D, BN]
    const uint32_t t0 = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
    for (int c = 0; c < KCH; ++c) *(u32x4 *)(k_at + to * TILE + c * KROWS * KP) = kreg[c];  // (rows past the end repeat the last one: their scores are discarded)
    if (t0 + BN > a.t) {
      const u32x4 none = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int c = 0; c < KCH; ++c) vreg[c] = t0 + v_k8 < a.t ? vreg[c] : none;
    }
#pragma unroll
    for (int c = 0; c < KCH; ++c) *(u32x4 *)(v_at + to * TILE + c * VROWS * VP) = vreg[c];
  };
  uint32_t t0 = tiles.skip(tiles.next_step(0), kg), t_next = a.t;
  if (t0 < a.t) fetch(t0);  // (uniform)

  if constexpr (!LEAN) {
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      const float4 x0 = qx[2 * ks], x1 = qx[2 * ks + 1];
      const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
      qf[ks] = pack8(v);
    }
  }
  a_f32x16 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
  float m_run = -3.40282347e+38f, l_run = 0.f;
  const float inv_scale = a.has_scale ? 1.0f / a.scale : 1.0f;  // bf16 mode: a product, not the reference's quotient
  const bool can_be_plain = inv_scale > 0.f && (M || !a.has_mask_const);

  if (t0 < a.t) {
    stash(0, t0);
    t_next = tiles.skip(t0, KG);
    if (t_next < a.t) fetch(t_next);
  }
  __syncthreads();
  const uint32_t turns = KG > 1 ? (tiles.live_steps() + KG - 1) / KG : 0;  // (as many for every group: they share the barrier)
  for (uint32_t turn = 0, buf = 0; KG > 1 ? turn < turns : t0 < a.t; ++turn, buf ^= 1) {
    if (KG > 1 && t0 >= a.t) {  // (the last turn of an odd number of steps)
      __syncthreads();
      continue;
    }
    const uint16_t *Ks = tile[kg][buf], *Vt = Ks + BN * KP;
    const bool use_mask = M && tiles.reads_mask(t0);  // uniform
    const bool plain = can_be_plain && !use_mask && t0 + BN <= a.t;
    // The mask values of this step are asked for here and used after the score product; rows allow 16-byte loads
    // (checked by the host).  A step whose every pair is masked - possible only without a class table - needs no
    // special case: its weights exp(f32::MIN - m) are zero once any live key has been seen, and a row that never
    // sees one is rebuilt at the end.
    constexpr bool LATE = D > 64 || (D == 64 && NW == 4 && (KG == 1 || BN == 32));
    float4 mcur[KT][4];
    if (use_mask && !LATE) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int j = 0; j < 4; ++j) mcur[kt][j] = *(const float4 *)(M + min(t0 + kt * 32 + j * 8 + half * 4, a.m_len - 4));
    }
    // ---- S^T = K . Q^T
    a_f32x16 st[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int e = 0; e < 16; ++e) st[kt][e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {  // (chains of products that do not wait for each other)
        const a_bf16x8 kf = *(const a_bf16x8 *)(&Ks[(kt * 32 + col) * KP + ks * 16 + half * 8]);
        st[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], st[kt], 0, 0, 0);
      }
    const uint32_t t_cur = t0, t_after = t_next < a.t ? tiles.skip(t_next, KG) : a.t;
    if (t_next < a.t) stash(buf ^ 1, t_next);  // (everyone is past the barrier behind the last reads of that buffer)
    if (t_after < a.t) fetch(t_after);
    t0 = t_next;
    t_next = t_after;
    // ---- scale, mask, running maximum and sum; P^T as B fragments of the 16-key blocks.
    // The reference point of the exponentials only follows the maximum when that has moved by more than
    // ATTN_MAX_SLACK: the quotient O / l at the end does not depend on it, weights of up to e^slack are as
    // exact in f32 and bf16 as weights of up to 1, and O is rescaled on a few steps instead of on most.
    a_bf16x8 pf[KT * 2];
    const float alpha = attn_softmax_step<KT, LATE>(a, st, M, mcur, pf, m_run, l_run, inv_scale, plain, use_mask, t_cur, half);
    // ---- O^T = O^T * alpha + V^T . P^T
    if (__any(alpha != 1.0f)) {  // the running maximum moved for some query of this wave
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] *= alpha;
    }
#pragma unroll
    for (int blk = 0; blk < KT * 2; ++blk) {
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        // A fragment: row = dim t*32 + col, the lane's eight keys of this block in the permuted order
        const uint16_t *vr = &Vt[(dim0 + t * 32 + col) * VP + blk * 16 + half * 4];
        union {
          uint2 u[2];
          a_bf16x8 hv;
        } vf;
        vf.u[0] = *(const uint2 *)vr;
        vf.u[1] = *(const uint2 *)(vr + 8);
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.hv, pf[blk], o[t], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  l_run = sum_of_halves(l_run);
  if constexpr (KG == 2) {  // the second group's partial results, [register][lane], join the first's
    float *part = (float *)&tile[0][0][0] + of_group * (DT * 16 + 2) * 64;
    static_assert((NW / KG) * (DT * 16 + 2) * 64 * 4 <= 2 * 2 * TILE * 2, "partial results fit in the tiles");
    if (kg) {  // (everyone is past the barrier behind the last step)
      part[lane] = m_run;
      part[64 + lane] = l_run;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) part[(2 + t * 16 + e) * 64 + lane] = o[t][e];
    }
    __syncthreads();
    if (kg) return;
    const float m_w = part[lane], l_w = part[64 + lane], m_new = fmaxf(m_run, m_w);
    const float f0 = __expf(m_run - m_new), f1 = __expf(m_w - m_new);
    l_run = l_run * f0 + l_w * f1;
    m_run = m_new;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[t][e] = o[t][e] * f0 + part[(2 + t * 16 + e) * 64 + lane] * f1;
  }
  // A row whose every key is masked has all scores equal to f32::MIN on the reference path:
  // uniform weights, i.e. the mean of V.  Dead steps were skipped above, so rebuild that here.
  if (M && q_ok && m_run <= -3.0e38f) {
    l_run = (float)a.t;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
    for (uint32_t key = 0; key < a.t; ++key)
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float4 vv = *(const float4 *)(V + (int64_t)key * a.v_st + dim0 + t * 32 + j * 8 + half * 4);
          o[t][j * 4 + 0] += vv.x; o[t][j * 4 + 1] += vv.y; o[t][j * 4 + 2] += vv.z; o[t][j * 4 + 3] += vv.w;
        }
  }
  // ---- normalise and store: O^T register e of tile t is dim t*32 + (e>>2)*8 + half*4 + (e&3)
  if (q_ok) {
    const int64_t o_off = (int64_t)b * a.o_sb + (int64_t)h * a.o_sh + (int64_t)query * a.o_ss;
    float *out = LEAN ? nullptr : a.out + o_off;
    uint16_t *out16 = LEAN || a.out16 ? a.out16 + o_off : nullptr;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float4 r;
        r.x = o[t][j * 4 + 0] / l_run; r.y = o[t][j * 4 + 1] / l_run;
        r.z = o[t][j * 4 + 2] / l_run; r.w = o[t][j * 4 + 3] / l_run;
        const int dim = dim0 + t * 32 + j * 8 + half * 4;
        if (!LEAN) *(float4 *)(out + dim) = r;
        if (LEAN || out16) *(uint2 *)(out16 + dim) = bf16_pack4(r);
      }
  }
}

// Few query rows (a 512-token prompt: 256 workgroups of 64 queries, one per CU, each walking up to eight
// key tiles one memory round trip at a time): the keys are divided instead.  The NW waves of a workgroup
// all own the same 32 queries; wave w takes every NW-th live key tile into an LDS region of its own, so
// the main loop needs no workgroup barrier and the waves' memory waits overlap each other's arithmetic.
// Each wave ends with its own running maximum, sum and O^T; they meet once, in LDS, and wave 0 merges
// them (the same rescaling as between two steps of one wave).
// ONE: all keys are one step, of one wave; nothing waits for the class table, the mask values travel with the keys, and the waves that had no
// step, and their merge, are gone (us a layer, causal, 32 heads of 64: 20 tokens 7.9 -> 4.9, 37 7.9 -> 4.8, 64 7.4 -> 5.1).
template <int D, int BN, int NW, bool LEAN = false, bool ONE = false>
__global__ void __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))  // two workgroups per CU
attn_prefill_keysplit_kernel(AttnPrefillDesc a) {
  warm_kernel_arguments<sizeof(AttnPrefillDesc)>();
  constexpr int KP = D + 8;
  constexpr int VP = BN + 8;
  constexpr int DT = D / 32;
  constexpr int KT = BN / 32;
  constexpr int KCH = BN * D / 8 / 64;   // 16-byte chunks of the K tile / of the V^T tile per lane
  constexpr int REGION = BN * KP + D * VP;  // bf16 elements of one wave's tiles
  static_assert(REGION * 2 >= (DT * 16 + 2) * 64 * 4, "a wave's partial result must fit in its tile region");
  __shared__ __attribute__((aligned(16))) uint16_t lds[NW * REGION];
  __shared__ __attribute__((aligned(16))) uint16_t qs[32 * (D + 8)];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 31, half = lane >> 5;
  uint16_t *Ks = lds + wave * REGION, *Vt = Ks + BN * KP;
  const uint32_t h = blockIdx.y, b = blockIdx.z;
  const uint32_t kvh = h / a.rep, rp = h % a.rep;
  const uint32_t query = blockIdx.x * 32 + col;
  const bool q_ok = query < a.s;
  const uint32_t qc = q_ok ? query : a.s - 1;
  const uint16_t *K = a.k16 + (int64_t)b * a.k_sb + (int64_t)kvh * a.k_skv + (int64_t)rp * a.k_srep;
  const uint16_t *VT = a.vt16 + ((int64_t)b * (a.heads / a.rep) + kvh) * D * (int64_t)a.vt_st;
  const float *V = a.v + (int64_t)b * a.v_sb + (int64_t)kvh * a.v_skv + (int64_t)rp * a.v_srep;
  const float *M = a.mask ? a.mask + (int64_t)b * a.m_sb + (int64_t)h * a.m_sh + (int64_t)qc * a.m_ss : nullptr;

  KeyTiles<BN> tiles(a, blockIdx.x, lane);
  // The queries: each wave converts a quarter of the workgroup's 32 rows (16 bytes of bf16 per lane and
  // piece), the rows meet in LDS, and every wave reads its B fragments from there - a quarter of the loads
  // of every wave fetching every row.  (Rows past the end repeat the last; what they compute goes nowhere.)
  constexpr int QP = D + 8, QC = 32 * D / 8 / (NW * 64);  // row pitch (bf16 elements), pieces of a lane
  float4 qx[QC][2];
  a_bf16x8 qh[QC];
#pragma unroll
  for (int c = 0; c < QC; ++c) {
    const int ch = tid + c * NW * 64, r = ch / (D / 8), d8 = (ch % (D / 8)) * 8;
    const int64_t at = (int64_t)b * a.q_sb + (int64_t)h * a.q_sh + (int64_t)min(blockIdx.x * 32 + r, a.s - 1) * a.q_ss + d8;
    if constexpr (LEAN) {
      qh[c] = *(const a_bf16x8 *)(a.q16 + at);
    } else {
      qx[c][0] = *(const float4 *)(a.q + at);
      qx[c][1] = *(const float4 *)(a.q + at + 4);
    }
  }
  tiles.arrived(lane);
  static_assert(!ONE || NW == 1, "one step, one wave");
  auto step_mask = [&](uint32_t t0) { return M && (ONE || tiles.reads_mask(t0)); };
  uint4 kreg[KCH], vreg[KCH];
  auto fetch = [&](uint32_t t0) {
#pragma unroll
    for (int c = 0; c < KCH; ++c) {
      const int ch = lane + c * 64, key = ch / (D / 8), d8 = (ch % (D / 8)) * 8;
      kreg[c] = *(const uint4 *)(K + (int64_t)min(t0 + key, a.t - 1) * a.k_st + d8);
    }
#pragma unroll
    for (int c = 0; c < KCH; ++c) {
      const int ch = lane + c * 64, dim = ch / (BN / 8), k8 = (ch % (BN / 8)) * 8;
      vreg[c] = *(const uint4 *)(VT + (int64_t)dim * a.vt_st + min(t0 + k8, a.vt_st - 8));
    }
  };
  uint32_t t0 = ONE ? 0 : tiles.skip(tiles.next_step(0), wave);
  if (t0 < a.t) fetch(t0);
  float4 first_mask[ONE ? KT : 1][4];
  if (ONE && M) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int j = 0; j < 4; ++j) first_mask[ONE ? kt : 0][j] = *(const float4 *)(M + min(kt * 32u + j * 8 + half * 4, a.m_len - 4));
  }
#pragma unroll
  for (int c = 0; c < QC; ++c) {
    const int ch = tid + c * NW * 64, r = ch / (D / 8), d8 = (ch % (D / 8)) * 8;
    if constexpr (LEAN) {
      *(a_bf16x8 *)(&qs[r * QP + d8]) = qh[c];
    } else {
      const float v[8] = {qx[c][0].x, qx[c][0].y, qx[c][0].z, qx[c][0].w, qx[c][1].x, qx[c][1].y, qx[c][1].z, qx[c][1].w};
      *(a_bf16x8 *)(&qs[r * QP + d8]) = pack8(v);
    }
  }
  __syncthreads();
  a_bf16x8 qf[D / 16];
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) qf[ks] = *(const a_bf16x8 *)(&qs[col * QP + ks * 16 + half * 8]);
  a_f32x16 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
  float m_run = -3.40282347e+38f, l_run = 0.f;
  const float inv_scale = a.has_scale ? 1.0f / a.scale : 1.0f;

  const bool can_be_plain = inv_scale > 0.f && (M || !a.has_mask_const);

  while (t0 < a.t) {
    const uint32_t t_next = ONE ? a.t : tiles.skip(t0, NW);
    const bool use_mask = step_mask(t0);  // uniform over the wave
    const bool tail = t0 + BN > a.t;
    const uint32_t t_cur = t0;
    t0 = t_next;
    // The mask values of this step are asked for here and used after the score product.  (A step whose
    // every pair is masked - possible only without a class table - needs no special case: its terms
    // carry the weight exp(f32::MIN - m), which is zero once any live key has been seen, and a row
    // that never sees one is rebuilt at the end.)
    float4 mcur[KT][4];
    if (use_mask) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int j = 0; j < 4; ++j) mcur[kt][j] = ONE ? first_mask[ONE ? kt : 0][j] : *(const float4 *)(M + min(t_cur + kt * 32 + j * 8 + half * 4, a.m_len - 4));
    }
    // registers -> this wave's LDS region.  Its LDS instructions run in program order, so the fragment
    // reads of the previous step are behind these writes and the reads below are ahead of them; the
    // fences keep the compiler from reordering across them.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int c = 0; c < KCH; ++c) {
      const int ch = lane + c * 64, key = ch / (D / 8), d8 = (ch % (D / 8)) * 8;
      *(uint4 *)(&Ks[key * KP + d8]) = (t_cur + key < a.t) ? kreg[c] : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int c = 0; c < KCH; ++c) {
      const int ch = lane + c * 64, dim = ch / (BN / 8), k8 = (ch % (BN / 8)) * 8;
      *(uint4 *)(&Vt[dim * VP + k8]) = (t_cur + k8 < a.t) ? vreg[c] : make_uint4(0u, 0u, 0u, 0u);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (t_next < a.t) fetch(t_next);  // in flight during the arithmetic below
    a_f32x16 st[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
      for (int e = 0; e < 16; ++e) st[kt][e] = 0.f;
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) {
        const a_bf16x8 kf = *(const a_bf16x8 *)(&Ks[(kt * 32 + col) * KP + ks * 16 + half * 8]);
        st[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], st[kt], 0, 0, 0);
      }
    }
    a_bf16x8 pf[KT * 2];
    const float alpha = attn_softmax_step<KT, false>(a, st, M, mcur, pf, m_run, l_run, inv_scale, can_be_plain && !use_mask && !tail, use_mask, t_cur, half, ONE && a.m_len >= BN);
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] *= alpha;
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) {
#pragma unroll
      for (int blk = 0; blk < KT * 2; ++blk) {
        const uint16_t *vr = &Vt[(t * 32 + col) * VP + blk * 16 + half * 4];
        union {
          uint2 u[2];
          a_bf16x8 hv;
        } vf;
        vf.u[0] = *(const uint2 *)vr;
        vf.u[1] = *(const uint2 *)(vr + 8);
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.hv, pf[blk], o[t], 0, 0, 0);
      }
    }
  }
  l_run = sum_of_halves(l_run);
  // ---- the waves' partial results meet: [register][lane] floats in each wave's own region
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  float *mine = (float *)(lds + wave * REGION);
  if (wave) {
    mine[lane] = m_run;
    mine[64 + lane] = l_run;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) mine[(2 + t * 16 + e) * 64 + lane] = o[t][e];
  }
  __syncthreads();
  if (wave) return;
#pragma unroll 1
  for (int w = 1; w < NW; ++w) {
    const float *other = (const float *)(lds + w * REGION);
    const float m_w = other[lane], l_w = other[64 + lane];
    const float m_new = fmaxf(m_run, m_w);
    const float f0 = __expf(m_run - m_new), f1 = __expf(m_w - m_new);
    l_run = l_run * f0 + l_w * f1;
    m_run = m_new;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[t][e] = o[t][e] * f0 + other[(2 + t * 16 + e) * 64 + lane] * f1;
  }
  if (M && q_ok && m_run <= -3.0e38f) {  // every key masked: uniform weights, as on the reference path
    l_run = (float)a.t;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
    for (uint32_t key = 0; key < a.t; ++key)
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float4 vv = *(const float4 *)(V + (int64_t)key * a.v_st + t * 32 + j * 8 + half * 4);
          o[t][j * 4 + 0] += vv.x; o[t][j * 4 + 1] += vv.y; o[t][j * 4 + 2] += vv.z; o[t][j * 4 + 3] += vv.w;
        }
  }
  if (q_ok) {
    const int64_t o_off = (int64_t)b * a.o_sb + (int64_t)h * a.o_sh + (int64_t)query * a.o_ss;
    float *out = LEAN ? nullptr : a.out + o_off;
    uint16_t *out16 = LEAN || a.out16 ? a.out16 + o_off : nullptr;
    const float inv_l = 1.0f / l_run;  // bf16 products: a reciprocal and a product, not 64 quotients
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float4 r;
        r.x = o[t][j * 4 + 0] * inv_l; r.y = o[t][j * 4 + 1] * inv_l;
        r.z = o[t][j * 4 + 2] * inv_l; r.w = o[t][j * 4 + 3] * inv_l;
        const int dim = t * 32 + j * 8 + half * 4;
        if (!LEAN) *(float4 *)(out + dim) = r;
        if (LEAN || out16) *(uint2 *)(out16 + dim) = bf16_pack4(r);
      }
  }
}

// The same pass with every product in f32 (v_mfma_f32_32x32x2_f32), for a backend without the bf16 flag:
// the results stay within the f32 bar of the reference's three-step sequence, and the [b, h, S, T]
// scores are still never written.  One MFMA consumes two values of the reduction axis, one per lane
// half, so
//   S^T: A = K[key kt*32 + col][dim 2 ks + half] (LDS, row pitch D + 2: 64 lanes, 64 banks),
//        B = the lane's query, dim 2 ks + half (registers);
//   O^T: B = register i of the lane's probabilities, which is key (i>>2)*8 + half*4 + (i&3) of the tile,
//        A = V[that key][dim t*32 + col] (LDS, rows as they lie in memory: no transpose).
// K and V take turns in one LDS tile: the V rows of a step are fetched while its scores are computed,
// the K rows of the next step while the V product runs.
// QLDS: the queries of the workgroup stay in LDS instead of registers (a 256-wide head would need 128
// registers per lane for them, on top of 128 for O^T).
template <bool QLDS, int D, int BN, int NW>
__global__ void __launch_bounds__(NW * 64) attn_prefill_f32_kernel(AttnPrefillDesc a) {
  constexpr int NT = NW * 64;
  constexpr int KP = D + 2;              // K tile row pitch (floats)
  constexpr int VP = D + 8;              // V tile row pitch
  constexpr int DT = D / 32;
  constexpr int KT = BN / 32;
  constexpr int CH = BN * D / 4 / NT;    // 16-byte chunks of a tile per thread
  constexpr bool AHEAD = !QLDS;          // fetch the next tile during the arithmetic (costs CH x 4 registers throughout)
  __shared__ __attribute__((aligned(16))) float tile[BN * VP];
  __shared__ __attribute__((aligned(16))) float qs[QLDS ? NW * 32 * KP : 2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 31, half = lane >> 5;
  const uint32_t h = blockIdx.y, b = blockIdx.z;
  const uint32_t kvh = h / a.rep, rp = h % a.rep;
  const uint32_t query = blockIdx.x * (NW * 32) + wave * 32 + col;
  const bool q_ok = query < a.s;
  const uint32_t qc = q_ok ? query : a.s - 1;
  const float *Q = a.q + (int64_t)b * a.q_sb + (int64_t)h * a.q_sh + (int64_t)qc * a.q_ss;
  const float *K = a.k + (int64_t)b * a.k_sb + (int64_t)kvh * a.k_skv + (int64_t)rp * a.k_srep;
  const float *V = a.v + (int64_t)b * a.v_sb + (int64_t)kvh * a.v_skv + (int64_t)rp * a.v_srep;
  const float *M = a.mask ? a.mask + (int64_t)b * a.m_sb + (int64_t)h * a.m_sh + (int64_t)qc * a.m_ss : nullptr;

  float qf[QLDS ? 1 : D / 2];
  if constexpr (QLDS) {  // the workgroup's rows, zero past the end; first read after the loop's first barrier
    const float *Q0 = a.q + (int64_t)b * a.q_sb + (int64_t)h * a.q_sh;
#pragma unroll
    for (int c = 0; c < NW * 32 * D / 4 / NT; ++c) {
      const int ch = tid + c * NT, r = ch / (D / 4), d4 = (ch % (D / 4)) * 4;
      const uint32_t row = blockIdx.x * (NW * 32) + r;
      float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
      if (row < a.s) x = *(const float4 *)(Q0 + (int64_t)row * a.q_ss + d4);
      *(float2 *)(&qs[r * KP + d4]) = make_float2(x.x, x.y);
      *(float2 *)(&qs[r * KP + d4 + 2]) = make_float2(x.z, x.w);
    }
  } else {
#pragma unroll
    for (int c = 0; c < D / 4; ++c) {  // dims 4c .. 4c+3: k-steps 2c (x, y) and 2c+1 (z, w)
      float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
      if (q_ok) x = *(const float4 *)(Q + c * 4);
      qf[2 * c] = half ? x.y : x.x;
      qf[2 * c + 1] = half ? x.w : x.z;
    }
  }
  a_f32x16 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
  float m_run = -3.40282347e+38f, l_run = 0.f;

  float4 treg[CH];
  float4 mreg[KT][4];
  KeyTiles<BN> tiles(a, blockIdx.x, lane);
  tiles.arrived(lane);
  auto next_step = [&](uint32_t t0) { return tiles.next_step(t0); };
  auto step_mask = [&](uint32_t t0) { return M && tiles.reads_mask(t0); };
  // rows of K (or V) of the step at t0 into registers; rows past the end repeat the last one and are
  // zeroed when they are written to LDS
  auto fetch_rows = [&](const float *base, int64_t row_stride, uint32_t t0) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int ch = tid + c * NT, key = ch / (D / 4), d4 = (ch % (D / 4)) * 4;
      treg[c] = *(const float4 *)(base + (int64_t)min(t0 + key, a.t - 1) * row_stride + d4);
    }
  };
  auto fetch_mask = [&](uint32_t t0) {
    if (step_mask(t0)) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          mreg[kt][j] = *(const float4 *)(M + min(t0 + kt * 32 + j * 8 + half * 4, a.m_len - 4));
    }
  };
  uint32_t t0 = next_step(0);
  if (t0 < a.t) {
    if (AHEAD) fetch_rows(K, a.k_st, t0);
    fetch_mask(t0);
  }
  for (; t0 < a.t;) {
    const uint32_t t_next = next_step(t0 + BN);
    const bool use_mask = step_mask(t0);
    const bool tail = t0 + BN > a.t;
    bool live_pair = !use_mask;
    float4 mcur[KT][4];
    if (use_mask) {
      float mmax = -3.40282347e+38f;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          mcur[kt][j] = mreg[kt][j];
          float4 mk = mcur[kt][j];
          if (tail) {
            const uint32_t key = t0 + kt * 32 + j * 8 + half * 4;
            if (key >= a.t) mk.x = -3.40282347e+38f;
            if (key + 1 >= a.t) mk.y = -3.40282347e+38f;
            if (key + 2 >= a.t) mk.z = -3.40282347e+38f;
            if (key + 3 >= a.t) mk.w = -3.40282347e+38f;
          }
          mmax = fmaxf(mmax, fmaxf(fmaxf(mk.x, mk.y), fmaxf(mk.z, mk.w)));
        }
      live_pair = q_ok && mmax > -3.0e38f;
    }
    const bool live = __syncthreads_or(live_pair);  // also: the V rows of the previous step have been read
    const uint32_t t_cur = t0;
    t0 = t_next;
    if (!live) {  // uniform
      if (t_next < a.t) {
        if (AHEAD) fetch_rows(K, a.k_st, t_next);
        fetch_mask(t_next);
      }
      continue;
    }
    if (!AHEAD) fetch_rows(K, a.k_st, t_cur);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int ch = tid + c * NT, key = ch / (D / 4), d4 = (ch % (D / 4)) * 4;
      const float4 x = (t_cur + key < a.t) ? treg[c] : make_float4(0.f, 0.f, 0.f, 0.f);
      *(float2 *)(&tile[key * KP + d4]) = make_float2(x.x, x.y);
      *(float2 *)(&tile[key * KP + d4 + 2]) = make_float2(x.z, x.w);
    }
    __syncthreads();
    if (AHEAD) fetch_rows(V, a.v_st, t_cur);  // in flight during the score product
    // ---- S^T = K . Q^T
    a_f32x16 st[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
      for (int e = 0; e < 16; ++e) st[kt][e] = 0.f;
#pragma unroll
      for (int ks = 0; ks < D / 2; ++ks) {
        float qv;
        if constexpr (QLDS) qv = qs[(wave * 32 + col) * KP + 2 * ks + half];
        else qv = qf[ks];
        st[kt] = __builtin_amdgcn_mfma_f32_32x32x2f32(tile[(kt * 32 + col) * KP + 2 * ks + half], qv, st[kt], 0, 0, 0);
        // keep the scheduler from hoisting a whole tile's LDS reads above the MFMAs (registers)
        if (ks % 16 == 15) __builtin_amdgcn_sched_barrier(0);
      }
    }
    // ---- scale, mask, running maximum.  Register e of tile kt is key t_cur + kt*32 + (e>>2)*8 + half*4 + (e&3)
    float tmax = -3.40282347e+38f;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t key = t_cur + kt * 32 + j * 8 + half * 4;
        float mv[4] = {0.f, 0.f, 0.f, 0.f};
        if (use_mask) { mv[0] = mcur[kt][j].x; mv[1] = mcur[kt][j].y; mv[2] = mcur[kt][j].z; mv[3] = mcur[kt][j].w; }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float s = st[kt][j * 4 + i];
          if (a.has_scale) s = s / a.scale;  // the reference's quotient
          if (use_mask) s = s + mv[i];
          else if (!M && a.has_mask_const) s = s + a.mask_const;
          if (tail && key + i >= a.t) s = -3.40282347e+38f;
          st[kt][j * 4 + i] = s;
          tmax = fmaxf(tmax, s);
        }
      }
    tmax = max_of_halves(tmax);
    const float m_new = fmaxf(m_run, tmax);
    const float alpha = expf(m_run - m_new);
    float psum = 0.f;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const uint32_t key = t_cur + kt * 32 + (e >> 2) * 8 + half * 4 + (e & 3);
        float p = expf(st[kt][e] - m_new);
        if (tail && key >= a.t) p = 0.f;
        st[kt][e] = p;
        psum += p;
      }
    psum = sum_of_halves(psum);
    l_run = l_run * alpha + psum;
    m_run = m_new;
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int t = 0; t < DT; ++t) {
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] *= alpha;
        __builtin_amdgcn_sched_barrier(0);  // one tile of O^T at a time through the VALU registers
      }
    }
    if (!AHEAD) fetch_rows(V, a.v_st, t_cur);
    __syncthreads();  // every wave has read its K fragments
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int ch = tid + c * NT, key = ch / (D / 4), d4 = (ch % (D / 4)) * 4;
      *(float4 *)(&tile[key * VP + d4]) = (t_cur + key < a.t) ? treg[c] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    __syncthreads();
    if (t_next < a.t) {  // in flight during the value product
      if (AHEAD) fetch_rows(K, a.k_st, t_next);
      fetch_mask(t_next);
    }
    // ---- O^T += V^T . P^T
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = kt * 32 + (i >> 2) * 8 + half * 4 + (i & 3);
          o[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(tile[key * VP + t * 32 + col], st[kt][i], o[t], 0, 0, 0);
          if (i == 15) __builtin_amdgcn_sched_barrier(0);
        }
  }
  if (M && q_ok && m_run <= -3.0e38f) {  // every key masked: uniform weights, as on the reference path
    l_run = (float)a.t;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
    for (uint32_t key = 0; key < a.t; ++key)
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float4 vv = *(const float4 *)(V + (int64_t)key * a.v_st + t * 32 + j * 8 + half * 4);
          o[t][j * 4 + 0] += vv.x; o[t][j * 4 + 1] += vv.y; o[t][j * 4 + 2] += vv.z; o[t][j * 4 + 3] += vv.w;
        }
  }
  if (q_ok) {
    float *out = a.out + (int64_t)b * a.o_sb + (int64_t)h * a.o_sh + (int64_t)query * a.o_ss;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float4 r;
        r.x = o[t][j * 4 + 0] / l_run; r.y = o[t][j * 4 + 1] / l_run;
        r.z = o[t][j * 4 + 2] / l_run; r.w = o[t][j * 4 + 3] / l_run;
        *(float4 *)(out + t * 32 + j * 8 + half * 4) = r;
      }
  }
}

// Heads of 64 under a mask whose workgroups of 128 queries would all run at once, two to a CU: the one with the most keys is then
// what the launch takes, and two key groups of 64 queries halve it.  With more of them the long tiles start first and the short
// ones fill in.  Up to one such workgroup a CU the key-split kernel's 32 queries are ahead.  us a layer, 32 heads, causal, against
// what the line keeps them from: 512 tokens 16.5 (key-split 14.2), 900 24.8 (34), 1050 25.4 (128 queries 36.7), 1500 38 (50),
// 2000 50 (61); 2900 93 (90) and 4000 154 (131) lie past it.
static bool attn_prefill_two_groups(const LaunchCtx &lc, const AttnPrefillDesc &d) {
  return !d.f32 && d.d == 64 && d.mask && (uint64_t)((d.s + 63) / 64) * d.heads * d.b > (uint64_t)lc.n_cus &&
         (uint64_t)((d.s + 127) / 128) * d.heads * d.b <= 2 * (uint64_t)lc.n_cus;
}

// Keys a step of the two groups.  32 leave registers for a third workgroup on the CU, which pays once two and a half are there for
// each: 1200 tokens 31.6 us (64 keys 29.6), 1500 38.3 (39.8), 1800 47.0 (53.6), 2000 50.7 (60.2).
static uint32_t attn_prefill_two_groups_keys(const LaunchCtx &lc, const AttnPrefillDesc &d) {
  return 2 * (uint64_t)((d.s + 63) / 64) * d.heads * d.b > 5 * (uint64_t)lc.n_cus ? 32 : 64;
}

// bf16 products, few query rows: 64-query workgroups would not give every CU two of them
static bool attn_prefill_keysplit(const LaunchCtx &lc, const AttnPrefillDesc &d) {
  return !d.f32 && d.d == 64 && (uint64_t)((d.s + 63) / 64) * d.heads * d.b < 2 * (uint64_t)lc.n_cus &&
         !attn_prefill_two_groups(lc, d);
}

bool attn_prefill_one_step(const LaunchCtx &lc, const AttnPrefillDesc &d) { return d.t <= 64 && attn_prefill_keysplit(lc, d); }

// Heads of 128 and 256: two wavefronts to 32 queries, each with half of the values' dims (both compute the scores; the accumulators of
// two waves then fit on a SIMD, and one's softmax runs under the other's products).  us a layer, heads of 128, causal, against one
// wavefront to 32 queries: 16 heads of 400 tokens 24.0 -> 18.5, 1400 61.1 -> 49.2, 4 x 256 20.5 -> 17.9.  Beyond one workgroup of 128
// queries a CU a second round of these begins and the doubled scores weigh more (causal mask, no mask, a mask without dead tiles: 16
// heads of 2048 tokens 71, 83, 121, with one wavefront 88, 88, 120; 3000 tokens 107, 193, 289 here, 110, 136, 185 there; 2 x 1100 44,
// 80, 115 and 49, 58, 77; 4 x 700 39, 58, 78 and 36, 43, 55).  Heads of 256, causal: 4 heads of 2000 tokens 75.5 -> 51.9, 8 x 1000
// 81.7 -> 61.1, 8 x 2048 152 -> 130; without a mask 369 -> 316.
static bool attn_prefill_wide(const LaunchCtx &lc, const AttnPrefillDesc &d) {
  return !d.f32 && (d.d == 256 || (d.d == 128 && (uint64_t)((d.s + 127) / 128) * d.heads * d.b <= (uint64_t)lc.n_cus));
}
// ... in two key groups of 32 or 64 queries (0: one group) while a CU has at most one such workgroup and the keys are more than a
// step: 100 tokens of 16 heads of 128 10.5 -> 9.8, 400 18.5 -> 16.7, 900 33.9 -> 27.8; 4 heads of 256, 700 tokens 40.3 -> 34.1, 2000
// 51.9 -> 44.1, 4 x 1000 45.3 -> 40.4 (64 queries; 32 in two rounds 64).
static int attn_prefill_wide_groups(const LaunchCtx &lc, const AttnPrefillDesc &d) {
  if (!attn_prefill_wide(lc, d) || d.t <= (d.d == 128 ? 64u : 32u)) return 0;
  if ((uint64_t)((d.s + 31) / 32) * d.heads * d.b <= (uint64_t)lc.n_cus) return 32;
  return (uint64_t)((d.s + 63) / 64) * d.heads * d.b <= (uint64_t)lc.n_cus ? 64 : 0;
}

static bool attn_prefill_small_tiles(const LaunchCtx &lc, const AttnPrefillDesc &d) {
  if (d.f32 && d.d == 256) return true;  // its queries live in LDS: 64 of them fit beside the K / V tile
  return (uint64_t)((d.s + 127) / 128) * d.heads * d.b < (uint64_t)lc.n_cus;  // too few workgroups of 128 queries: 64 each
}

void attn_prefill_tiling(const LaunchCtx &lc, const AttnPrefillDesc &d, uint32_t *q_rows, uint32_t *keys) {
  if (attn_prefill_keysplit(lc, d) || attn_prefill_wide_groups(lc, d) == 32) *q_rows = 32;
  else *q_rows = attn_prefill_wide(lc, d) || attn_prefill_small_tiles(lc, d) || attn_prefill_two_groups(lc, d) ? 64 : 128;
  *keys = attn_prefill_two_groups(lc, d) ? attn_prefill_two_groups_keys(lc, d) : (d.d == 256 || (d.f32 && d.d == 128)) ? 32 : 64;
}

// one workgroup per (key tile, query tile): any value above the masked level, any value that is not zero
__global__ void __launch_bounds__(256) mask_tiles_kernel(const float *mask, int64_t m_ss, uint32_t s, uint32_t t, uint32_t q_rows,
                                                         uint32_t keys, uint8_t *out) {
  __shared__ uint32_t flags;
  if (threadIdx.x == 0) flags = 0;
  __syncthreads();
  const uint32_t q0 = blockIdx.y * q_rows, k0 = blockIdx.x * keys;
  uint32_t f = 0;  // bit 0: some pair is not masked, bit 1: some value is not zero
  for (uint32_t i = threadIdx.x; i < q_rows * keys; i += 256) {
    const uint32_t q = q0 + i / keys, k = k0 + i % keys;
    if (q < s && k < t) {
      const float v = mask[(int64_t)q * m_ss + k];
      if (v > -3.0e38f) f |= 1u;
      if (v != 0.f) f |= 2u;
    }
  }
  if (f) atomicOr(&flags, f);
  __syncthreads();
  if (threadIdx.x == 0) out[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = !(flags & 1u) ? 0 : (flags & 2u) ? 1 : 2;
}

// A mask whose rows do not allow 16-byte loads (an odd number of keys), copied once to rows of `pitch` floats; past the
// last key every value is f32::MIN.
__global__ void __launch_bounds__(256) mask_pad_kernel(const float *mask, int64_t m_ss, uint32_t t, uint32_t pitch, float *out) {
  const float *row = mask + (int64_t)blockIdx.y * m_ss;
  const uint32_t c = blockIdx.x * 256 + threadIdx.x;
  if (c < pitch) out[(size_t)blockIdx.y * pitch + c] = c < t ? row[c] : -3.40282347e+38f;
}

hipError_t launch_mask_pad(const LaunchCtx &lc, const float *mask, int64_t m_ss, uint32_t s, uint32_t t, uint32_t pitch, float *out) {
  if (!s || !t) return hipSuccess;
  if (pitch < t || s > 65535) return hipErrorInvalidValue;
  CG_LAUNCH(lc, mask_pad_kernel, dim3((pitch + 255) / 256, s), 256, mask, m_ss, t, pitch, out);
  return hipGetLastError();
}

hipError_t launch_mask_tiles(const LaunchCtx &lc, const float *mask, int64_t m_ss, uint32_t s, uint32_t t, uint32_t q_rows,
                             uint32_t keys, uint8_t *out) {
  if (!s || !t) return hipSuccess;
  CG_LAUNCH(lc, mask_tiles_kernel, dim3((t + keys - 1) / keys, (s + q_rows - 1) / q_rows), 256, mask, m_ss, s, t, q_rows, keys, out);
  return hipGetLastError();
}

hipError_t launch_attn_prefill(const LaunchCtx &lc, const AttnPrefillDesc &d) {
  if (!d.b || !d.heads || !d.s) return hipSuccess;
  if (d.f32 ? !d.k : (!d.k16 || !d.vt16 || d.vt_st < d.t || d.vt_st % 8)) return hipErrorInvalidValue;
  if (d.mask && (d.m_len < d.t || d.m_len % 4)) return hipErrorInvalidValue;
  if (d.q16 ? d.f32 || !d.out16 : !d.q || !d.out) return hipErrorInvalidValue;
#define CG_ATTN(kernel, grid, block, ...)                                            \
  do {                                                                               \
    if (d.q16) CG_LAUNCH(lc, (kernel<__VA_ARGS__, true>), grid, block, d);           \
    else CG_LAUNCH(lc, (kernel<__VA_ARGS__, false>), grid, block, d);                \
  } while (0)
  if (attn_prefill_keysplit(lc, d)) {
    dim3 g32((d.s + 31) / 32, d.heads, d.b);
    if (attn_prefill_one_step(lc, d)) {
      if (d.q16) CG_LAUNCH(lc, (attn_prefill_keysplit_kernel<64, 64, 1, true, true>), g32, 64, d);
      else CG_LAUNCH(lc, (attn_prefill_keysplit_kernel<64, 64, 1, false, true>), g32, 64, d);
      return hipGetLastError();
    }
    CG_ATTN(attn_prefill_keysplit_kernel, g32, 256, 64, 64, 4);
    return hipGetLastError();
  }
  if (attn_prefill_two_groups(lc, d)) {
    const uint32_t grid = (d.s + 63) / 64 * d.heads * d.b;
    if (attn_prefill_two_groups_keys(lc, d) == 32) CG_ATTN(attn_prefill_kernel, grid, 256, 64, 32, 4, 2, 1);
    else CG_ATTN(attn_prefill_kernel, grid, 256, 64, 64, 4, 2, 1);
    return hipGetLastError();
  }
  if (attn_prefill_wide(lc, d)) {
    const int groups = attn_prefill_wide_groups(lc, d);
    const uint32_t bh = d.heads * d.b, g32 = (d.s + 31) / 32 * bh, g64 = (d.s + 63) / 64 * bh;
#define CG_ATTN_WIDE(DD, BN)                                                                        \
    if (groups == 32) CG_ATTN(attn_prefill_kernel, g32, 256, DD, BN, 4, 2, 2);           \
    else if (groups == 64) CG_ATTN(attn_prefill_kernel, g64, 512, DD, BN, 8, 2, 2);      \
    else CG_ATTN(attn_prefill_kernel, g64, 256, DD, BN, 4, 1, 2);
    if (d.d == 128) { CG_ATTN_WIDE(128, 64) }
    else { CG_ATTN_WIDE(256, 32) }
#undef CG_ATTN_WIDE
    return hipGetLastError();
  }
  const bool small = attn_prefill_small_tiles(lc, d);  // (f32 only: bf16 products of so few rows are gone by now)
  dim3 grid(small ? (d.s + 63) / 64 : (d.s + 127) / 128, d.heads, d.b);
  if (!d.f32) grid = dim3(grid.x * d.heads * d.b);
#define CG_ATTN_CASE(DD, ...)                                               \
  case DD:                                                                  \
    if (small) CG_LAUNCH(lc, (__VA_ARGS__, 2>), grid, 128, d);              \
    else CG_LAUNCH(lc, (__VA_ARGS__, 4>), grid, 256, d);                    \
    break;
  if (d.f32) {
    switch (d.d) {
      CG_ATTN_CASE(64, attn_prefill_f32_kernel<false, 64, 64)
      CG_ATTN_CASE(128, attn_prefill_f32_kernel<false, 128, 32)
      case 256: CG_LAUNCH(lc, (attn_prefill_f32_kernel<true, 256, 32, 2>), grid, 128, d); break;
      default: return hipErrorInvalidValue;
    }
  } else {
    switch (d.d) {
      case 64: CG_ATTN(attn_prefill_kernel, grid, 256, 64, 64, 4, 1, 1); break;
      case 128: CG_ATTN(attn_prefill_kernel, grid, 256, 128, 64, 4, 1, 1); break;
      default: return hipErrorInvalidValue;
    }
  }
#undef CG_ATTN_CASE
#undef CG_ATTN
  return hipGetLastError();
}

}  // namespace cgk
