// k_gemm_f32.hip — f32 products whose operands can travel to LDS as they lie.
//
// C[m, n] = sum_k A[m, k] B[k, n] in f32 (Backend::matmul, mod.rs:41; ndarray.rs:549-615): A with unit stride along k, B
// along k (a weight [N, K]) or along n, rows in whole 16-byte pieces.
//
// What bounds it: v_mfma_f32_32x32x2_f32, 64 cycles for 4096 multiply-adds - 157 TFLOP/s on the card -, and for up to 64 rows the
// stream of weights.  Everything else fits beside that if the CU is never idle, so
//   * a workgroup's tile is 32 to 256 rows, in steps of 16, by 128 columns, chosen with the number of k-slices for the fewest MFMAs
//     on the busiest CU (launch_gemm_f32): 200 rows are one tile of 208 and not two of 128;
//   * its four wavefronts have 32 columns each and all of the rows: R + 1 reads of 16 bytes from LDS feed 4 R MFMAs, and 16 rows more
//     the four of v_mfma_f32_16x16x1_4b_f32, half as long: its blocks take the lanes of B as they are - both column halves, for the
//     lower and the upper k of a group -, the same 16 rows of A four times, and the two sums over k meet at the end;
//   * NS stages of BK values of k come straight into LDS (global_load_lds_dwordx4, pieces of rows swizzled on the way so that the
//     reads meet no bank twice), NS - 1 steps ahead of their use, one barrier a step;
//   * two workgroups fit on a CU, one's stores and barriers under the other's products.
// A lane's 16 bytes of a row are four consecutive k; MFMA j of a group of eight takes element j of both operands, so the lower half
// of the wave supplies k = 8 g + j and the upper k = 8 g + 4 + j.
// Measured (weights from memory, us, slices and their sum included) against 128 x 128 tiles whose operands went through registers, or
// 32 x 32 ones: 17 x 8192 x 2048 35.3 -> 19.8, 64 53.3 -> 28.6, 200 95.6 -> 75.8, 300 167 -> 101, 700 321 -> 206; 700 x 2048 x 8192
// 312 -> 215; 6000 x 4100 x 1000, B along n, 546 -> 423; 4096 cubed 1142 -> 1015 (135 TFLOP/s; the MFMAs alone 916 at 2.3 GHz).
#include <hip/hip_runtime.h>
#include <algorithm>
#include "launch.hpp"
#include "dev_common.hpp"

namespace cgk {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ const float4 gemm_f32_zero = {0.f, 0.f, 0.f, 0.f};  // what lies past the end of k

static __device__ __forceinline__ void to_lds16(const float *from, uint32_t lds_byte) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_byte), "v"(from) : "memory", "m0");
}
template <int N> static __device__ __forceinline__ void loads_left() {
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// BKM: B has unit stride along n; its tile travels as BK rows of 128 columns.
// HALF: 16 rows more.
template <int R, int BK, int NS, bool BKM, bool HALF>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) gemm_f32_dma_kernel(GemmDesc g) {
  constexpr int CH = BK / 4, RPP = 64 / CH;                 // 16-byte pieces of a row, rows of a load of 1 KB
  constexpr int ROWS = 32 * R + (HALF ? 16 : 0), PA = ROWS / RPP, TP = PA + 128 / RPP;     // loads of a stage: A's, all
  constexpr int LPW = (TP + 3) / 4, STAGE = TP * 1024;
  extern __shared__ __attribute__((aligned(16))) float f32_smem[];
  warm_kernel_arguments<sizeof(GemmDesc)>();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5;
  const uint32_t tiles_m = (g.M + ROWS - 1) / ROWS, tiles_n = (g.N + 127) / 128;
  const uint32_t per_batch = tiles_m * tiles_n, batch = g.nb0 * g.nb1;
  // a contiguous range of tiles to each XCD, walked in groups of four tile rows (as TilePlace has it, which is no faster here: 1000 x
  // 2048 x 8192 272 us, 278 with it)
  uint32_t id = blockIdx.x;
  if (gridDim.x % 8 == 0) id = (id % 8) * (gridDim.x / 8) + id / 8;
  const uint32_t zz = id / per_batch, t = id - zz * per_batch;
  const uint32_t split = zz / batch, bz = zz - split * batch;
  const uint32_t b0 = bz / g.nb1, b1 = bz - b0 * g.nb1;
  const uint32_t first_m = t / (4 * tiles_n) * 4, gsz = min(tiles_m - first_m, 4u), tg = t % (4 * tiles_n);
  const uint32_t m0 = (first_m + tg % gsz) * ROWS, n0 = tg / gsz * 128;
  const float *A = (const float *)g.a + b0 * g.sa_b0 + b1 * g.sa_b1;
  const float *B = (const float *)g.b + b0 * g.sb_b0 + b1 * g.sb_b1;
  const uint32_t k_begin = g.splits > 1 ? min(g.K, split * g.k_per_split) : 0;
  const uint32_t k_end = g.splits > 1 ? min(g.K, k_begin + g.k_per_split) : g.K;
  const uint32_t n_steps = (k_end - k_begin + BK - 1) / BK, rem = (k_end - k_begin) % BK;

  // This wavefront's loads: consecutive pieces of the stacked [A; B] tile (the last wavefront repeats the last piece where
  // they do not divide by four).
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float *)f32_smem;
  auto piece = [&](int i) { return min(wave * LPW + i, TP - 1); };
  auto key = [](int row) { return BK == 32 ? (row >> 1) & 7 : (row >> 2) & 3; };
  auto k_in_step = [&](int i) {  // first k of this lane's 16 bytes
    const int p = piece(i), row = p * RPP + lane / CH;
    return BKM && p >= PA ? (p - PA) * 2 + lane / 32 : ((lane % CH) ^ key(row)) * 4;
  };
  const float *from[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const int p = piece(i), row = p * RPP + lane / CH;
    const int64_t k = k_begin + k_in_step(i);
    if (p < PA) from[i] = A + (int64_t)min(m0 + row, g.M - 1) * g.sam + k;
    else if (BKM) from[i] = B + k * g.sbk + min(n0 + (uint32_t)(((lane & 31) ^ (((k_in_step(i) >> 2) & 1) << 3)) * 4), g.N - 4);
    else from[i] = B + (int64_t)min(n0 + row - ROWS, g.N - 1) * g.sbn + k;
  }
  auto request = [&](uint32_t step, int stage) {
    const bool tail = rem && step + 1 == n_steps;  // (uniform)
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const float *p = from[i];
      if (tail) p = (uint32_t)k_in_step(i) < rem ? p : (const float *)&gemm_f32_zero;
      to_lds16(p, lds0 + stage * STAGE + piece(i) * 1024);
      from[i] += BKM && piece(i) >= PA ? (int64_t)BK * g.sbk : (int64_t)BK;
    }
  };

  f32x16 acc[R], last;  // (last: block b of 16 x 16 is columns 16 (b % 2) on, k in the lower or upper half of a group)
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
#pragma unroll
  for (int e = 0; e < 16; ++e) last[e] = 0.f;
  auto multiply = [&](int stage) {
    const float *As = f32_smem + stage * (STAGE / 4), *Bs = As + ROWS * BK;
    f32x4 af[2][R], lf[2], bf[2];
    auto fragments = [&](int q, int set) {
      const int at = (lane & 31) * BK + (((2 * q + half) ^ key(lane & 31)) * 4);
#pragma unroll
      for (int i = 0; i < R; ++i) af[set][i] = *(const f32x4 *)(As + i * 32 * BK + at);
      if (HALF) lf[set] = *(const f32x4 *)(As + R * 32 * BK + (lane & 15) * BK + (((2 * q + half) ^ key(lane & 15)) * 4));
      if (!BKM) {
        bf[set] = *(const f32x4 *)(Bs + wave * 32 * BK + at);
      } else {
        const int col = (wave * 32 + (lane & 31)) ^ (half << 5);
#pragma unroll
        for (int j = 0; j < 4; ++j) bf[set][j] = Bs[(8 * q + 4 * half + j) * 128 + col];
      }
    };
    fragments(0, 0);
#pragma unroll
    for (int q = 0; q < BK / 8; ++q) {
      if (q + 1 < BK / 8) fragments(q + 1, (q + 1) & 1);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int i = 0; i < R; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[q & 1][i][j], bf[q & 1][j], acc[i], 0, 0, 0);
        if (HALF) last = __builtin_amdgcn_mfma_f32_16x16x1f32(lf[q & 1][j], bf[q & 1][j], last, 0, 0, 0);
      }
    }
  };

#pragma unroll
  for (int s = 0; s < NS - 1; ++s)
    if ((uint32_t)s < n_steps) request(s, s);
  int stage = 0;
  for (uint32_t step = 0; step < n_steps; ++step) {
    // stage `step` is here (this wave's part): at most NS - 2 younger ones are on their way, or, near the end, none is waited for
    if (step + NS - 1 <= n_steps) loads_left<(NS - 2) * LPW>();
    else loads_left<0>();
    __syncthreads();  // ... and everyone's part; the stage refilled next has been read
    // (in one go: with the second workgroup's products to hide behind, spreading them over this one's gains nothing)
    if (step + NS - 1 < n_steps) request(step + NS - 1, stage == 0 ? NS - 1 : stage - 1);
    multiply(stage);
    stage = stage + 1 == NS ? 0 : stage + 1;
  }

  float *C = (g.splits > 1 ? g.workspace + (uint64_t)split * batch * g.M * g.N : g.c) + (uint64_t)bz * g.M * g.N;
  const bool act = g.act_sigmoid && g.splits <= 1;
  const uint32_t col = n0 + wave * 32 + (lane & 31), row0 = m0 + half * 4;
  float *to = C + (uint64_t)row0 * g.N + col;
  if (act) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][e] = sigmoid_ref(acc[i][e]);
  }
  if (col < g.N) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {  // accumulator element e of a lane: row (e / 4) * 8 + half * 4 + e % 4, column lane % 32
        const uint32_t r = i * 32 + (e >> 2) * 8 + (e & 3);
        if (row0 + r < g.M) to[(uint64_t)r * g.N] = acc[i][e];
      }
  }
  if (HALF) {  // element e of block b: row lane / 16 * 4 + e, column lane % 16 of the block's
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint32_t col16 = n0 + wave * 32 + b * 16 + (lane & 15), row16 = m0 + R * 32 + (lane >> 4) * 4;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = last[b * 4 + e] + last[8 + b * 4 + e];
        if (col16 < g.N && row16 + e < g.M) C[(uint64_t)(row16 + e) * g.N + col16] = act ? sigmoid_ref(v) : v;
      }
    }
  }
}

bool gemm_f32_ok(const GemmDesc &g) {
  if (g.bf16_math || g.a_stype != ST_F32 || g.b_stype != ST_F32 || g.b_index || g.M <= 8 || g.K < 32 || g.K % 4) return false;
  if (g.glu_gate || g.c16 || g.n_group || g.dual_b) return false;
  auto whole = [](const void *p, int64_t s0, int64_t s1, int64_t s2) { return (uintptr_t)p % 16 == 0 && s0 % 4 == 0 && s1 % 4 == 0 && s2 % 4 == 0; };
  if (g.sak != 1 || !whole(g.a, g.sam, g.sa_b0, g.sa_b1)) return false;
  if (g.sbk == 1) return whole(g.b, g.sbn, g.sb_b0, g.sb_b1);
  return g.sbn == 1 && g.N % 4 == 0 && g.N >= 4 && whole(g.b, g.sbk, g.sb_b0, g.sb_b1);
}

static uint32_t f32_k_per_split(uint32_t K, uint32_t splits) { return ((K + splits - 1) / splits + 63) / 64 * 64; }

// Microseconds for tiles of 16 H rows and `splits` slices of k, close enough to choose by: the busiest CU's MFMAs (16 cycles per k
// and 16 x 128 products; the factor is what such a tile takes beyond them on 4096 cubed, and a workgroup alone on its CU takes 8 %
// more), the stream of B where that is longer, what surrounds a launch, and the slices' way through memory.
static double f32_cost(const LaunchCtx &lc, const GemmDesc &g, uint32_t H, uint32_t splits) {
  static const double factor[17] = {0, 0, 1.38, 1.47, 1.21, 1.22, 1.17, 1.18, 1.15, 1.13, 1.10, 1.11, 1.12, 1.12, 1.12, 1.11, 1.10};
  const uint32_t batch = g.nb0 * g.nb1, per = splits > 1 ? f32_k_per_split(g.K, splits) : g.K;
  const uint64_t tiles = (uint64_t)((g.M + 16 * H - 1) / (16 * H)) * ((g.N + 127) / 128) * batch * splits;
  const uint64_t rounds = (tiles + lc.n_cus - 1) / lc.n_cus;
  const double products = ((double)rounds + (rounds % 2 ? 0.08 : 0)) * per * H * 16 / 2300.0 * factor[H];
  const double stream = (double)batch * g.N * g.K * 4 / 4.4e6 * (rounds > 1 ? 1.0 : (double)lc.n_cus / tiles);
  const double out = (double)batch * g.M * g.N * 4 / 4.5e6;
  return 6.0 + std::max(products, stream) + (splits > 1 ? 3.0 + (splits + 1) * out : 0);
}
// Of equal cost the fewest rows (bound by the stream of B: 17 x 8192 x 2048 on 48 rows 22.2 us, on 32 17.5).  Odd heights for up to 512
// rows (us without and with them, weights from memory: 40 x 8192 x 2048 26.6, 22.6, 72 36.4, 32.3, 100 45.1, 41.0, 200 69.6, 66.5, 400
// 126, 118; 200 x 2048 x 8192 72, 67.5; 232 x 4100 x 1000, B along n, 33.1, 28.4); beyond, some are ahead and some are not (2048 x 8192,
// 700 rows 202, 187, 600 174.5, 176.6, 1000 264, 269), and of a few k a launch is mostly what surrounds it.
static double f32_best(const LaunchCtx &lc, const GemmDesc &g, uint32_t splits, uint32_t *height) {
  double best = 1e30;
  for (uint32_t H = 16; H >= 2; --H) {
    if (H % 2 && (g.M > 512 || g.K < 256)) continue;
    if (const double us = f32_cost(lc, g, H, splits); us <= best) {
      best = us;
      *height = H;
    }
  }
  return best;
}

// No form takes less than f32_cost has it for one round of 32 rows over all of k, or over the 64 that a slice has at least.
double gemm_f32_least_us(const GemmDesc &g) {
  const double per_k = 1.08 * 32 / 2300.0 * 1.38;
  return std::min(6.0 + per_k * g.K, 9.0 + per_k * 64) * (1 - 1e-9);
}

uint32_t gemm_f32_split(const LaunchCtx &lc, const GemmDesc &g, double *us) {
  uint32_t best_splits = 1, height = 0;
  double best = 1e30;
  for (uint32_t s = 1; s <= 16 && (s == 1 || g.K / s >= 64); ++s) {
    if (s > 1 && (uint64_t)(s - 1) * f32_k_per_split(g.K, s) >= g.K) continue;  // (a last slice of nothing)
    if (const double c = f32_best(lc, g, s, &height); c < best) {
      best = c;
      best_splits = s;
    }
  }
  *us = best;
  return best_splits;
}

template <int R, int BK, int NS, bool HALF = false>
static hipError_t launch_as(const LaunchCtx &lc, const GemmDesc &g) {
  constexpr uint32_t ROWS = 32 * R + (HALF ? 16 : 0);
  const uint32_t tiles = (g.M + ROWS - 1) / ROWS * ((g.N + 127) / 128) * g.nb0 * g.nb1 * (g.splits > 1 ? g.splits : 1);
  constexpr int smem = NS * (ROWS + 128) * BK * 4;
  static bool configured = false;  // one attribute call per kernel and process
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void *)gemm_f32_dma_kernel<R, BK, NS, false, HALF>, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e == hipSuccess) e = hipFuncSetAttribute((const void *)gemm_f32_dma_kernel<R, BK, NS, true, HALF>, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) return e;
    configured = true;
  }
  if (g.sbk == 1) cg_launch(lc, gemm_f32_dma_kernel<R, BK, NS, false, HALF>, dim3(tiles), dim3(256), smem, g);
  else cg_launch(lc, gemm_f32_dma_kernel<R, BK, NS, true, HALF>, dim3(tiles), dim3(256), smem, g);
  return hipGetLastError();
}

hipError_t launch_gemm_f32(const LaunchCtx &lc, const GemmDesc &g) {
  if (!gemm_f32_ok(g) || (g.splits > 1 && g.k_per_split % 64)) return hipErrorInvalidValue;
  uint32_t height = 0;
  f32_best(lc, g, g.splits > 1 ? g.splits : 1, &height);
  // (as many stages as let two workgroups have a CU's 160 KB)
  switch (height) {
    case 2: return launch_as<1, 32, 4>(lc, g);
    case 3: return launch_as<1, 32, 3, true>(lc, g);
    case 4: return launch_as<2, 32, 3>(lc, g);
    case 5: return launch_as<2, 32, 3, true>(lc, g);
    case 6: return launch_as<3, 32, 2>(lc, g);
    case 7: return launch_as<3, 32, 2, true>(lc, g);
    case 8: return launch_as<4, 32, 2>(lc, g);
    case 9: return launch_as<4, 16, 4, true>(lc, g);
    case 10: return launch_as<5, 16, 4>(lc, g);
    case 11: return launch_as<5, 16, 4, true>(lc, g);
    case 12: return launch_as<6, 16, 4>(lc, g);
    case 13: return launch_as<6, 16, 3, true>(lc, g);
    case 14: return launch_as<7, 16, 3>(lc, g);
    case 15: return launch_as<7, 16, 3, true>(lc, g);
    default: return launch_as<8, 16, 3>(lc, g);
  }
}

}  // namespace cgk
