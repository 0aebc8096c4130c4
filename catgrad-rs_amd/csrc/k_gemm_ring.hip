// k_gemm_ring.hip — the bf16 NT product of large problems: 256 x 256 tiles, four wavefronts, one per SIMD.
//
// C[m, n] = sum_k A[m, k] B[n, k], both operands bf16 with unit stride along k, K a multiple of 64 and at least 128
// (Backend::matmul, mod.rs:41; ndarray.rs:549-615).
//
// What bounds it: the matrix cores, if nothing else of a k-step of 64 takes longer than its 2048 cycles of MFMAs (64 per
// wavefront, 32 cycles each).  A wavefront owns 128 x 128 of the tile, so a k-step reads 128 KB of fragments out of LDS
// and writes 64 KB into it (eight wavefronts of 128 x 64 read 192 KB, all that the LDS delivers in that time), and the
// CU takes in 64 KB through its one load path of 64 bytes a cycle: 1024 cycles, if the loads are spread evenly.  Issued
// in one burst at the top of a step - which is what a compiler makes of them, since it moves nothing across their inline
// assembly - each of them costs its wave 55 to 120 cycles, in which no MFMA is issued.  So the whole main loop is one
// statement of assembly with a fixed place for everything:
//   * The tile is four quadrants of 128 x 128, (A half, B half) = (0,0) (0,1) (1,1) (1,0), a phase each; in a quadrant a
//     wavefront owns 64 x 64, and a phase is 16 MFMAs in four k-slices.
//   * A unit is half an operand's tile: 128 rows x 128 bytes.  A stage is four units, LDS holds two.  Every phase reads
//     the fragments of one unit (8 reads) for the phases after it, and requests the same unit of the step after the
//     next (4 loads of 1 KB by each wavefront), into the place whose last reader was two phases ago.  A load has six
//     phases, 3072 cycles, to arrive, and there is no point at which everything is waited for.
//   * One barrier a phase: before it a wavefront has seen its own loads of the unit about to be read (a count) and the
//     reads of two phases ago (a count); so behind it the unit is there for everyone, and its predecessor's place free.
// On tiles of 256 rows the products of an element are added in the order of k, the same bits as gemm_bf16_dma_kernel's for products of
// more than 128 rows (but for its tiles of 128 x 128 and 192 x 128 with the scheduled loop); on tiles of 128, which up to 128 rows and the
// routed experts may be given with an order of their own, see KOrder.
// Tiles of 192 x 256, for gate / up and rotating products: see SPHASE1.
// Tiles of 128 x 256, for the stacked gate / up of fewer rows, for one round of plain, grouped and rotating products, and for the routed
// experts: see HPHASE0.
// Measured against 256 x 256 tiles with eight wavefronts whose loads a compiler placed, on the same box: 16384 x 1152 by 2 x 6912
// gate and up 531 -> 464 us, 2900 x 2048 by 2 x 8192 184 -> 161; 13056 x 6912 x 1152 203 -> 177, 16384 x 1152 x 1536 77 -> 67
// (100 MB of result); 6000 x 1024 x 4100 with a sigmoid 77 -> 64.  What is left is power: 8192 cubed takes 1.40 us a step on
// random operands (1.35 PFLOP/s) and 0.99 on zeros (1.96), with the same loads.  Around the loop a tile takes 0.8 us to set up,
// 1.1 for its first loads and 5.3 to store.
#include <hip/hip_runtime.h>
#include "launch.hpp"
#include <type_traits>
#include "dev_common.hpp"

namespace cgk {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

// These kernels' places in LDS are constants that start at 0, where a static __shared__ variable would lie too: no kernel that has
// one is launched.
static hipError_t whole_lds(const void *kernel, int bytes) {
  hipFuncAttributes a;
  const hipError_t e = hipFuncGetAttributes(&a, kernel);
  if (e != hipSuccess) return e;
  if (a.sharedSizeBytes) return hipErrorInvalidConfiguration;
  return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

// ---- the main loop, in pieces -------------------------------------------------------------------------
// Fragments live in v[128:255]: (half U, 32-row block r, k-slice ks) as below.  s[40:41] points at A, s[42:43] and s[44:45]
// at the two halves of B, at the step being requested; s46 is this wavefront's place in the stage being requested, s47
// counts steps.  M0 (a load's place in LDS) is set an instruction ahead of the load.
#define FR_A0_0_0 "v[128:131]"
#define FR_A0_0_1 "v[132:135]"
#define FR_A0_0_2 "v[136:139]"
#define FR_A0_0_3 "v[140:143]"
#define FR_A0_1_0 "v[144:147]"
#define FR_A0_1_1 "v[148:151]"
#define FR_A0_1_2 "v[152:155]"
#define FR_A0_1_3 "v[156:159]"
#define FR_A1_0_0 "v[160:163]"
#define FR_A1_0_1 "v[164:167]"
#define FR_A1_0_2 "v[168:171]"
#define FR_A1_0_3 "v[172:175]"
#define FR_A1_1_0 "v[176:179]"
#define FR_A1_1_1 "v[180:183]"
#define FR_A1_1_2 "v[184:187]"
#define FR_A1_1_3 "v[188:191]"
#define FR_B0_0_0 "v[192:195]"
#define FR_B0_0_1 "v[196:199]"
#define FR_B0_0_2 "v[200:203]"
#define FR_B0_0_3 "v[204:207]"
#define FR_B0_1_0 "v[208:211]"
#define FR_B0_1_1 "v[212:215]"
#define FR_B0_1_2 "v[216:219]"
#define FR_B0_1_3 "v[220:223]"
#define FR_B1_0_0 "v[224:227]"
#define FR_B1_0_1 "v[228:231]"
#define FR_B1_0_2 "v[232:235]"
#define FR_B1_0_3 "v[236:239]"
#define FR_B1_1_0 "v[240:243]"
#define FR_B1_1_1 "v[244:247]"
#define FR_B1_1_2 "v[248:251]"
#define FR_B1_1_3 "v[252:255]"
// byte offset of a 32-row block of a unit in its stage
#define AT_A0_0 "0"
#define AT_A0_1 "4096"
#define AT_B0_0 "16384"
#define AT_B0_1 "20480"
#define AT_B1_0 "32768"
#define AT_B1_1 "36864"
#define AT_A1_0 "49152"
#define AT_A1_1 "53248"
#define BASE_A0(ks) "%[ra" #ks "]"
#define BASE_A1(ks) "%[ra" #ks "]"
#define BASE_B0(ks) "%[rb" #ks "]"
#define BASE_B1(ks) "%[rb" #ks "]"
#define RD(U, r, ks) "ds_read_b128 " FR_##U##_##r##_##ks ", " BASE_##U(ks) " offset:" AT_##U##_##r "\n\t"
#define RD_UNIT(U) RD(U, 0, 0) RD(U, 1, 0) RD(U, 0, 1) RD(U, 1, 1) RD(U, 0, 2) RD(U, 1, 2) RD(U, 0, 3) RD(U, 1, 3)
#define PTR_A0 "s[40:41]"
#define PTR_A1 "s[40:41]"
#define PTR_B0 "s[42:43]"
#define PTR_B1 "s[44:45]"
// piece i (1 KB, eight rows) of unit U
#define M0_A0(i) "s_add_u32 m0, s46, " #i "*1024\n\t"
#define M0_B0(i) "s_add_u32 m0, s46, 16384+" #i "*1024\n\t"
#define M0_B1(i) "s_add_u32 m0, s46, 32768+" #i "*1024\n\t"
#define M0_A1(i) "s_add_u32 m0, s46, 49152+" #i "*1024\n\t"
#define LOAD(U, i) "global_load_lds_dwordx4 %[d" #U #i "], " PTR_##U "\n\t"
#define LOAD_AS(U, i, HINT) "global_load_lds_dwordx4 %[d" #U #i "], " PTR_##U HINT "\n\t"
#define LOAD_UNIT(U)                                                                                              \
  M0_##U(0) "s_nop 0\n\t" LOAD(U, 0) M0_##U(1) "s_nop 0\n\t" LOAD(U, 1) M0_##U(2) "s_nop 0\n\t" LOAD(U, 2) M0_##U(3) \
  "s_nop 0\n\t" LOAD(U, 3)
#define NEXT_STEP                                                                                              \
  "s_add_u32 s40, s40, 128\n\ts_addc_u32 s41, s41, 0\n\ts_add_u32 s42, s42, 128\n\ts_addc_u32 s43, s43, 0\n\t" \
  "s_add_u32 s44, s44, 128\n\ts_addc_u32 s45, s45, 0\n\t"
#define OTHER_STAGE_LOADS "s_xor_b32 s46, s46, 0x10000\n\t"
#define OTHER_STAGE_A                                                                        \
  "v_xor_b32 %[ra0], 0x10000, %[ra0]\n\tv_xor_b32 %[ra1], 0x10000, %[ra1]\n\t" \
  "v_xor_b32 %[ra2], 0x10000, %[ra2]\n\tv_xor_b32 %[ra3], 0x10000, %[ra3]\n\t"
#define OTHER_STAGE_B                                                                        \
  "v_xor_b32 %[rb0], 0x10000, %[rb0]\n\tv_xor_b32 %[rb1], 0x10000, %[rb1]\n\t" \
  "v_xor_b32 %[rb2], 0x10000, %[rb2]\n\tv_xor_b32 %[rb3], 0x10000, %[rb3]\n\t"
#define POINTERS "s_mov_b64 s[40:41], %[pa]\n\ts_mov_b64 s[42:43], %[pb0]\n\ts_mov_b64 s[44:45], %[pb1]\n\ts_mov_b32 s46, %[lds]\n\t"
// products of row block i of A half a with row block j of B half b.  The operands in this order leave the tile transposed: a
// lane holds four consecutive columns of a row of C.
#define PRODUCT(a, b, i, j, UA, UB, ks)                                                                                \
  "v_mfma_f32_32x32x16_bf16 %[c" #a #b #i #j "], " FR_##UB##_##j##_##ks ", " FR_##UA##_##i##_##ks ", %[c" #a #b #i #j \
  "]\n\t"
#define NONE ""
#define READS_BUT(n) "s_waitcnt lgkmcnt(" #n ")\n\t"
// a k-slice: its fragments (all but the six youngest reads are there), four products, two reads and one load among them
#define SLICE(a, b, UA, UB, ks, W, R1, M0, R2, L) \
  W PRODUCT(a, b, 0, 0, UA, UB, ks) R1 PRODUCT(a, b, 0, 1, UA, UB, ks) R2 M0 PRODUCT(a, b, 1, 0, UA, UB, ks) L PRODUCT(a, b, 1, 1, UA, UB, ks)
#define SYNC(v) "s_waitcnt vmcnt(" #v ") lgkmcnt(8)\n\ts_barrier\n\t"
#define ON_M(U, i) M0_##U(i)
#define ON_L(U, i) LOAD(U, i)
#define OFF_M(U, i) ""
#define OFF_L(U, i) ""
// G: ON while there is a step after the next to request.  v: this wavefront's loads that may still be under way.
#define PHASE0(G, v)                                                                            \
  SYNC(v)                                                                                           \
  SLICE(0, 0, A0, B0, 0, READS_BUT(6), RD(B1, 0, 0), G##_M(A0, 0), RD(B1, 1, 0), G##_L(A0, 0))  \
  SLICE(0, 0, A0, B0, 1, READS_BUT(6), RD(B1, 0, 1), G##_M(A0, 1), RD(B1, 1, 1), G##_L(A0, 1))  \
  SLICE(0, 0, A0, B0, 2, READS_BUT(6), RD(B1, 0, 2), G##_M(A0, 2), RD(B1, 1, 2), G##_L(A0, 2))  \
  SLICE(0, 0, A0, B0, 3, READS_BUT(6), RD(B1, 0, 3), G##_M(A0, 3), RD(B1, 1, 3), G##_L(A0, 3))
#define PHASE1(G, v)                                                                                           \
  SYNC(v)                                                                                                          \
  SLICE(0, 1, A0, B1, 0, READS_BUT(6), RD(A1, 0, 0), G##_M(B0, 0), RD(A1, 1, 0), G##_L(B0, 0))                 \
  SLICE(0, 1, A0, B1, 1, READS_BUT(6), RD(A1, 0, 1), G##_M(B0, 1), RD(A1, 1, 1), G##_L(B0, 1))                 \
  SLICE(0, 1, A0, B1, 2, READS_BUT(6), RD(A1, 0, 2), G##_M(B0, 2), RD(A1, 1, 2) OTHER_STAGE_B, G##_L(B0, 2))   \
  SLICE(0, 1, A0, B1, 3, READS_BUT(6), RD(A1, 0, 3), G##_M(B0, 3), RD(A1, 1, 3) OTHER_STAGE_A, G##_L(B0, 3))
#define PHASE2(G, v)                                                                            \
  SYNC(v)                                                                                           \
  SLICE(1, 1, A1, B1, 0, READS_BUT(6), RD(A0, 0, 0), G##_M(B1, 0), RD(A0, 1, 0), G##_L(B1, 0))  \
  SLICE(1, 1, A1, B1, 1, READS_BUT(6), RD(A0, 0, 1), G##_M(B1, 1), RD(A0, 1, 1), G##_L(B1, 1))  \
  SLICE(1, 1, A1, B1, 2, READS_BUT(6), RD(A0, 0, 2), G##_M(B1, 2), RD(A0, 1, 2), G##_L(B1, 2))  \
  SLICE(1, 1, A1, B1, 3, READS_BUT(6), RD(A0, 0, 3), G##_M(B1, 3), RD(A0, 1, 3), G##_L(B1, 3))
// (these reads replace fragments of this phase: each comes behind the products that use what it replaces)
#define PHASE3(G, v)                                                                                  \
  SYNC(v)                                                                                                 \
  SLICE(1, 0, A1, B0, 0, NONE, NONE, G##_M(A1, 0), NONE, G##_L(A1, 0))                                \
  SLICE(1, 0, A1, B0, 1, NONE, RD(B0, 0, 0), G##_M(A1, 1), RD(B0, 1, 0), G##_L(A1, 1))                \
  SLICE(1, 0, A1, B0, 2, NONE, RD(B0, 0, 1), G##_M(A1, 2), RD(B0, 1, 1), G##_L(A1, 2))                \
  SLICE(1, 0, A1, B0, 3, NONE, RD(B0, 0, 2), G##_M(A1, 3), RD(B0, 1, 2), G##_L(A1, 3)) RD(B0, 0, 3)   \
  RD(B0, 1, 3)
// the last step has nothing further to read in its second half
#define LAST_HALF                                                            \
  SLICE(1, 1, A1, B1, 0, READS_BUT(6), NONE, NONE, NONE, NONE)               \
  SLICE(1, 1, A1, B1, 1, READS_BUT(4), NONE, NONE, NONE, NONE)               \
  SLICE(1, 1, A1, B1, 2, READS_BUT(2), NONE, NONE, NONE, NONE)               \
  SLICE(1, 1, A1, B1, 3, READS_BUT(0), NONE, NONE, NONE, NONE)               \
  SLICE(1, 0, A1, B0, 0, NONE, NONE, NONE, NONE, NONE)                       \
  SLICE(1, 0, A1, B0, 1, NONE, NONE, NONE, NONE, NONE)                       \
  SLICE(1, 0, A1, B0, 2, NONE, NONE, NONE, NONE, NONE)                       \
  SLICE(1, 0, A1, B0, 3, NONE, NONE, NONE, NONE, NONE)
// steps 0 and 1 requested: 32 loads
#define FIRST_LOADS                                                                                                   \
  POINTERS LOAD_UNIT(A0) LOAD_UNIT(B0) LOAD_UNIT(B1) LOAD_UNIT(A1) NEXT_STEP OTHER_STAGE_LOADS LOAD_UNIT(A0) LOAD_UNIT(B0) \
  LOAD_UNIT(B1) LOAD_UNIT(A1)
// all n >= 2 steps (the nops: nothing behind this statement may read the accumulators before the last product is done)
#define MAIN_LOOP                                                                                                    \
  POINTERS NEXT_STEP NEXT_STEP "s_sub_u32 s47, %[n], 2\n\t"                                                              \
  "s_waitcnt vmcnt(24)\n\ts_barrier\n\t" RD_UNIT(A0) RD_UNIT(B0)                                                         \
  "s_cmp_eq_u32 s47, 0\n\ts_cbranch_scc1 2f\n\t"                                                                         \
  "1:\n\t" PHASE0(ON, 20) PHASE1(ON, 20) PHASE2(ON, 20) PHASE3(ON, 20) NEXT_STEP OTHER_STAGE_LOADS       \
  "s_sub_u32 s47, s47, 1\n\ts_cmp_lg_u32 s47, 0\n\ts_cbranch_scc1 1b\n\t"                                                \
  "2:\n\t" PHASE0(OFF, 20) PHASE1(OFF, 16) PHASE2(OFF, 12) PHASE3(OFF, 8) PHASE0(OFF, 4)             \
  PHASE1(OFF, 0) LAST_HALF "s_nop 15\n\ts_nop 7\n\t"

// ---- tiles of 192 x 256: half of A1 (its unit is 64 rows, 32 of each wavefront's row half, eight KB in two pieces 8192 bytes apart, as
// the fragments of 256 rows lie), so the phases (1,1) and (1,0) have eight products, A1 four reads a step and two loads.  For rows
// that 256 to a tile put in as many rounds: gate and up of 2100 rows by 2 x 8192, K = 2048, 149 -> 124 us, q / k / v of 2900 58.6 -> 49.9.
#define SM0_A1(i) "s_add_u32 m0, s48, 49152+" #i "*1024\n\t"
#define SSLICE(b, UB, ks, W, R1, M0, R2, L) W PRODUCT(1, b, 0, 0, A1, UB, ks) R1 M0 PRODUCT(1, b, 0, 1, A1, UB, ks) R2 L
#define SSYNC(v, r) "s_waitcnt vmcnt(" #v ") lgkmcnt(" #r ")\n\ts_barrier\n\t"
#define ON_S(x) x
#define OFF_S(x) ""
#define SPHASE1(G, v)                                                                                    \
  SSYNC(v, 8)                                                                                            \
  SLICE(0, 1, A0, B1, 0, READS_BUT(6), RD(A1, 0, 0), G##_M(B0, 0), NONE, G##_L(B0, 0))                   \
  SLICE(0, 1, A0, B1, 1, READS_BUT(5), RD(A1, 0, 1), G##_M(B0, 1), NONE, G##_L(B0, 1))                   \
  SLICE(0, 1, A0, B1, 2, READS_BUT(4), RD(A1, 0, 2), G##_M(B0, 2), OTHER_STAGE_B, G##_L(B0, 2))          \
  SLICE(0, 1, A0, B1, 3, READS_BUT(3), RD(A1, 0, 3), G##_M(B0, 3), OTHER_STAGE_A, G##_L(B0, 3))
#define SPHASE2(G, v)                                                                                    \
  SSYNC(v, 4)                                                                                            \
  SSLICE(1, B1, 0, READS_BUT(3), RD(A0, 0, 0), G##_M(B1, 0), RD(A0, 1, 0), G##_L(B1, 0))                 \
  SSLICE(1, B1, 1, READS_BUT(4), RD(A0, 0, 1), G##_M(B1, 1), RD(A0, 1, 1), G##_L(B1, 1))                 \
  SSLICE(1, B1, 2, READS_BUT(5), RD(A0, 0, 2), G##_M(B1, 2), RD(A0, 1, 2), G##_L(B1, 2))                 \
  SSLICE(1, B1, 3, READS_BUT(6), RD(A0, 0, 3), G##_M(B1, 3), RD(A0, 1, 3), G##_L(B1, 3))
#define SPHASE3(G, v)                                                                                    \
  SSYNC(v, 8)                                                                                            \
  SSLICE(0, B0, 0, NONE, NONE, G##_S(SM0_A1(0)), NONE, G##_L(A1, 0))                                     \
  SSLICE(0, B0, 1, NONE, RD(B0, 0, 0), G##_S(SM0_A1(1)), RD(B0, 1, 0), G##_L(A1, 1))                     \
  SSLICE(0, B0, 2, NONE, RD(B0, 0, 1), NONE, RD(B0, 1, 1), NONE)                                         \
  SSLICE(0, B0, 3, NONE, RD(B0, 0, 2), NONE, RD(B0, 1, 2), NONE) RD(B0, 0, 3) RD(B0, 1, 3)
#define SLAST_HALF                                                                                       \
  SSLICE(1, B1, 0, READS_BUT(3), NONE, NONE, NONE, NONE) SSLICE(1, B1, 1, READS_BUT(2), NONE, NONE, NONE, NONE) \
  SSLICE(1, B1, 2, READS_BUT(1), NONE, NONE, NONE, NONE) SSLICE(1, B1, 3, READS_BUT(0), NONE, NONE, NONE, NONE) \
  SSLICE(0, B0, 0, NONE, NONE, NONE, NONE, NONE) SSLICE(0, B0, 1, NONE, NONE, NONE, NONE, NONE)          \
  SSLICE(0, B0, 2, NONE, NONE, NONE, NONE, NONE) SSLICE(0, B0, 3, NONE, NONE, NONE, NONE, NONE)
#define SPOINTERS POINTERS "s_mov_b32 s48, %[lds1]\n\t"
#define SOTHER_STAGE_LOADS OTHER_STAGE_LOADS "s_xor_b32 s48, s48, 0x10000\n\t"
#define SSTEP_LOADS \
  LOAD_UNIT(A0) LOAD_UNIT(B0) LOAD_UNIT(B1) SM0_A1(0) "s_nop 0\n\t" LOAD(A1, 0) SM0_A1(1) "s_nop 0\n\t" LOAD(A1, 1)
// steps 0 and 1 requested: 28 loads
#define SFIRST_LOADS SPOINTERS SSTEP_LOADS NEXT_STEP SOTHER_STAGE_LOADS SSTEP_LOADS
// n >= 2 steps
#define SMAIN_LOOP                                                                                                   \
  SPOINTERS NEXT_STEP NEXT_STEP "s_sub_u32 s47, %[n], 2\n\t"                                                        \
  "s_waitcnt vmcnt(20)\n\ts_barrier\n\t" RD_UNIT(A0) RD_UNIT(B0)                                                  \
  "s_cmp_eq_u32 s47, 0\n\ts_cbranch_scc1 2f\n\t"                                                                  \
  "1:\n\t" PHASE0(ON, 16) SPHASE1(ON, 18) SPHASE2(ON, 18) SPHASE3(ON, 18) NEXT_STEP SOTHER_STAGE_LOADS            \
  "s_sub_u32 s47, s47, 1\n\ts_cmp_lg_u32 s47, 0\n\ts_cbranch_scc1 1b\n\t"                                        \
  "2:\n\t" PHASE0(OFF, 16) SPHASE1(OFF, 14) SPHASE2(OFF, 10) SPHASE3(OFF, 6) PHASE0(OFF, 2)                        \
  SPHASE1(OFF, 0) SLAST_HALF "s_nop 15\n\ts_nop 7\n\t"

// ---- tiles of 128 x 256: one unit of A, so a step is three units, two phases - (A, B0), (A, B1) - of 16 MFMAs.  LDS holds ten
// units, in the order A, B0, B1 of every step; the place of the unit 3 s + u is (3 s + u) % 10 (s48 A, s49 B0, s50 B1 of this
// step, s51 and s52 A and B0 of the next, s53 B1 of the one before).  The second phase of a step reads A and B0 of the next, the
// first B1 of this one; what they leave is requested again two phases later: A of step s + 3 in the first phase of s, B0 and B1
// in the second.  Fragments of A are replaced behind the products that use them, a slice late.  Against eight wavefronts with three
// stages: 400 rows by 2 x 5632, K = 2048, 31 -> 26.5 us, 512 by 2 x 6912, K = 1152, 21.3 -> 18; 512 by 2 x 8192, K = 2048, 38 to 40
// either way.  (Workgroups of different columns starting at different k: no change.  Loads past the L1: no change.  Four wavefronts that
// only load beside four that only multiply: 41 us a launch of twelve in a row against 41.)  What bounds it in a row of such launches is
// power: a step takes 1300 cycles, 1024 of them MFMAs, at 1.36 to 1.4 GHz; without the MFMAs 1360 at 2.1, without the loads 1210 at 1.9.
#define HRD(U, B, r, ks) "ds_read_b128 " FR_##U##_##r##_##ks ", " B " offset:" #r "*4096\n\t"
#define HFROM_A(S, ks) "v_add_u32 v126, " S ", %[ra" #ks "]\n\t"
#define HFROM_B(S, ks) "v_add_u32 v127, " S ", %[rb" #ks "]\n\t"
#define HA(r, ks) HRD(A0, "v126", r, ks)
#define HB0(r, ks) HRD(B0, "v127", r, ks)
#define HB1(r, ks) HRD(B1, "v127", r, ks)
#define HM0(i) "s_add_u32 m0, s54, " #i "*1024\n\t"
// (rows of A may be gathered: a pointer to each lane's)
#define HLOAD_A(i) "global_load_lds_dwordx4 %[ga" #i "], off\n\tv_lshl_add_u64 %[ga" #i "], %[ga" #i "], 0, s[58:59]\n\t"
#define HON(x) x
#define HOFF(x) ""
#define HSYNC(v) "s_waitcnt vmcnt(" #v ")\n\ts_barrier\n\t"
// (C: the accumulators, of a step's two phases alike)
#define HSLICE(C, b, UB, ks, W, E0, E1, E2, E3) \
  W PRODUCT(C, b, 0, 0, A0, UB, ks) E0 PRODUCT(C, b, 0, 1, A0, UB, ks) E1 PRODUCT(C, b, 1, 0, A0, UB, ks) E2 PRODUCT(C, b, 1, 1, A0, UB, ks) E3
// s[58:59]: bytes from the step being requested to the next (KOrder::advance; s55 is its place in the order); the main loop finds the
// next size out among its products
#define HSTEP_A "s_xor_b32 s40, s55, %[flip]\n\ts_add_u32 s55, s55, 1\n\t"
#define HSTEP_B "s_cmp_eq_u32 s55, %[n]\n\ts_cselect_b32 s55, 0, s55\n\t"
#define HSTEP_C "s_xor_b32 s41, s55, %[flip]\n\ts_sub_u32 s41, s41, s40\n\t"
#define HSTEP_D(lo, hi) "s_lshl_b32 " lo ", s41, 7\n\ts_ashr_i32 " hi ", s41, 31\n\t"
#define HSTEP_SIZE HSTEP_A HSTEP_B HSTEP_C HSTEP_D("s58", "s59")
#define HPHASE0(C, G, v)                                                                                                              \
  G("s_add_u32 s54, s53, %[lds]\n\t") HSYNC(v)                                                                                     \
  HFROM_A("s48", 3) HFROM_B("s50", 0)                                                                                              \
  HSLICE(C, 0, B0, 0, READS_BUT(8), HA(0, 3) G(HM0(0)), HA(1, 3) G(HLOAD_A(0)), HB1(0, 0), HB1(1, 0)) HFROM_B("s50", 1)          \
  HSLICE(C, 0, B0, 1, READS_BUT(8), HB1(0, 1) G(HM0(1)), HB1(1, 1) G(HLOAD_A(1)), "", "") HFROM_B("s50", 2)                          \
  HSLICE(C, 0, B0, 2, READS_BUT(6), HB1(0, 2) G(HM0(2)), HB1(1, 2) G(HLOAD_A(2)), "", "") HFROM_B("s50", 3)                          \
  HSLICE(C, 0, B0, 3, READS_BUT(6), HB1(0, 3) G(HM0(3)), HB1(1, 3) G(HLOAD_A(3)), "", "")
#define HPHASE1(C, G, v, HINT)                                                                                                              \
  G("s_add_u32 s54, s48, %[lds]\n\t") HSYNC(v)                                                                                     \
  HFROM_B("s52", 0)                                                                                                                \
  HSLICE(C, 1, B1, 0, READS_BUT(6), HB0(0, 0) G(HM0(0)), HB0(1, 0) G(LOAD_AS(B0, 0, HINT) HM0(1)), G(LOAD_AS(B0, 1, HINT)), G(HSTEP_A HSTEP_B)) \
  HFROM_A("s51", 0) HFROM_B("s52", 1)                                                                                              \
  HSLICE(C, 1, B1, 1, READS_BUT(6), HB0(0, 1) G(HM0(2)), HB0(1, 1) G(LOAD_AS(B0, 2, HINT) HM0(3)), HA(0, 0) G(LOAD_AS(B0, 3, HINT)), HA(1, 0) G(HSTEP_C HSTEP_D("s56", "s57")))      \
  HFROM_A("s51", 1) HFROM_B("s52", 2) G("s_add_u32 s54, s49, %[lds]\n\t")                                                          \
  HSLICE(C, 1, B1, 2, READS_BUT(8), HB0(0, 2) G(HM0(0)), HB0(1, 2) G(LOAD_AS(B1, 0, HINT) HM0(1)), HA(0, 1) G(LOAD_AS(B1, 1, HINT)), HA(1, 1))      \
  HFROM_A("s51", 2) HFROM_B("s52", 3)                                                                                              \
  HSLICE(C, 1, B1, 3, READS_BUT(10), HB0(0, 3) G(HM0(2)), HB0(1, 3) G(LOAD_AS(B1, 2, HINT) HM0(3)), HA(0, 2) G(LOAD_AS(B1, 3, HINT)), HA(1, 2))
// (the last step's second phase reads and requests nothing)
#define HLAST(C)                                                                                                    \
  HSLICE(C, 1, B1, 0, READS_BUT(6), "", "", "", "") HSLICE(C, 1, B1, 1, READS_BUT(4), "", "", "", "")                  \
  HSLICE(C, 1, B1, 2, READS_BUT(2), "", "", "", "") HSLICE(C, 1, B1, 3, READS_BUT(0), "", "", "", "")
#define HNEXT(x, y) "s_add_u32 " x ", " y ", 16384\n\ts_cmp_eq_u32 " x ", 163840\n\ts_cselect_b32 " x ", 0, " x "\n\t"
#define HNEXT_PLACES \
  "s_mov_b32 s53, s50\n\ts_mov_b32 s48, s51\n\ts_mov_b32 s49, s52\n\t" HNEXT("s50", "s52") HNEXT("s51", "s50") HNEXT("s52", "s51")
#define HLOADS_A \
  HM0(0) "s_nop 0\n\t" HLOAD_A(0) HM0(1) "s_nop 0\n\t" HLOAD_A(1) HM0(2) "s_nop 0\n\t" HLOAD_A(2) HM0(3) "s_nop 0\n\t" HLOAD_A(3)
#define HLOADS_B(U, HINT) \
  HM0(0) "s_nop 0\n\t" LOAD_AS(U, 0, HINT) HM0(1) "s_nop 0\n\t" LOAD_AS(U, 1, HINT) HM0(2) "s_nop 0\n\t" LOAD_AS(U, 2, HINT) HM0(3) "s_nop 0\n\t" LOAD_AS(U, 3, HINT)
#define HPOINTERS "s_mov_b64 s[42:43], %[pb0]\n\ts_mov_b64 s[44:45], %[pb1]\n\ts_mov_b32 s55, %[first]\n\t" HSTEP_SIZE
#define HNEXT_B "s_add_u32 s42, s42, s58\n\ts_addc_u32 s43, s43, s59\n\ts_add_u32 s44, s44, s58\n\ts_addc_u32 s45, s45, s59\n\t"
#define HNEXT_STEP HNEXT_B HSTEP_SIZE
#define HSTEP_LOADS(HINT) \
  HLOADS_A "s_add_u32 s54, s54, 16384\n\t" HLOADS_B(B0, HINT) "s_add_u32 s54, s54, 16384\n\t" HLOADS_B(B1, HINT) "s_add_u32 s54, s54, 16384\n\t"
// steps 0 to 2 requested: 36 loads
#define HFIRST_LOADS(HINT) HPOINTERS "s_mov_b32 s54, %[lds]\n\t" HSTEP_LOADS(HINT) HNEXT_STEP HSTEP_LOADS(HINT) HNEXT_STEP HSTEP_LOADS(HINT)
// n >= 3 steps
#define HMAIN_START                                                                                                              \
  HPOINTERS HNEXT_STEP HNEXT_STEP HNEXT_STEP "s_sub_u32 s47, %[n], 3\n\t"                                                          \
  "s_mov_b32 s48, 0\n\ts_movk_i32 s49, 0x4000\n\ts_mov_b32 s50, 0x8000\n\ts_mov_b32 s51, 0xC000\n\ts_mov_b32 s52, 0x10000\n\t"  \
  "s_mov_b32 s53, 0x24000\n\t" HSYNC(28)                                                                                        \
  HFROM_A("s48", 0) HFROM_B("s49", 0) HB0(0, 0) HB0(1, 0) HFROM_B("s49", 1) HB0(0, 1) HB0(1, 1) HA(0, 0) HA(1, 0)           \
  HFROM_A("s48", 1) HFROM_B("s49", 2) HB0(0, 2) HB0(1, 2) HA(0, 1) HA(1, 1)                                                 \
  HFROM_A("s48", 2) HFROM_B("s49", 3) HB0(0, 3) HB0(1, 3) HA(0, 2) HA(1, 2)                                                 \
  "s_cmp_eq_u32 s47, 0\n\ts_cbranch_scc1 2f\n\t"
#define HMAIN_STEP(C, HINT) \
  HPHASE0(C, HON, 24) HPHASE1(C, HON, 20, HINT) HNEXT_B "s_mov_b64 s[58:59], s[56:57]\n\t" HNEXT_PLACES "s_sub_u32 s47, s47, 1\n\t"
#define HMAIN_END(C0, C1, C2, HINT)                                                                                              \
  "2:\n\t" HPHASE0(C0, HOFF, 24) HPHASE1(C0, HOFF, 16, HINT) HNEXT_PLACES HPHASE0(C1, HOFF, 12) HPHASE1(C1, HOFF, 4, HINT)        \
  HNEXT_PLACES HPHASE0(C2, HOFF, 0) HLAST(C2) "s_nop 15\n\ts_nop 7\n\t"
#define HMAIN_LOOP(HINT) \
  HMAIN_START "1:\n\t" HMAIN_STEP(0, HINT) "s_cmp_lg_u32 s47, 0\n\ts_cbranch_scc1 1b\n\t" HMAIN_END(0, 0, 0, HINT)
// ... every other step in accumulators of its own (an odd number in front of the last three starts with the second of a pair)
#define HMAIN_LOOP_2(HINT)                                                                                                       \
  HMAIN_START "s_bitcmp1_b32 s47, 0\n\ts_cbranch_scc1 3f\n\t" "1:\n\t" HMAIN_STEP(1, HINT) "3:\n\t" HMAIN_STEP(0, HINT)          \
  "s_cmp_lg_u32 s47, 0\n\ts_cbranch_scc1 1b\n\t" HMAIN_END(1, 0, 1, HINT)

// ---- tiles of 256 x 288: the four quadrants and a strip X of 32 columns more, a ninth of the products with no wavefront idle: in each
// half of A a wavefront multiplies its first row block - rows wn * 32 of its 64, so that the two wavefronts of the same rows share
// them - by the strip, in the phases (0,1) and (1,1).  The strip's fragments are read in the first phase of a step and requested in the
// third; a stage's strip lies behind the two stages.  Rows of A are therefore read from two places a slice: rc is the other row block.
// A step reads 144 KB of fragments and takes in 68 KB for 72 products (128 and 64 for 64).  Bound by power like 256 x 256: 16384 x 1152 x
// 6912, one round, 229 us with the matrix cores busy 89 % of the time at the 1235 MHz that are left (256 x 256 in whole rounds, and the
// rest on smaller tiles, 274).
#define FR_X_0 "v[112:115]"
#define FR_X_1 "v[116:119]"
#define FR_X_2 "v[120:123]"
#define FR_X_3 "v[124:127]"
#define WRD(U, at, ks) "ds_read_b128 " FR_##U##_0_##ks ", %[ra" #ks "] offset:" at "\n\tds_read_b128 " FR_##U##_1_##ks ", %[rc" #ks "] offset:" at "\n\t"
#define WRD0(U, at, ks) "ds_read_b128 " FR_##U##_0_##ks ", %[ra" #ks "] offset:" at "\n\t"
#define WRD1(U, at, ks) "ds_read_b128 " FR_##U##_1_##ks ", %[rc" #ks "] offset:" at "\n\t"
#define WRDX(ks) "ds_read_b128 " FR_X_##ks ", %[rx" #ks "]\n\t"
#define WSTRIP(a, UA, ks) "v_mfma_f32_32x32x16_bf16 %[x" #a "], " FR_X_##ks ", " FR_##UA##_0_##ks ", %[x" #a "]\n\t"
#define WLOADX "global_load_lds_dwordx4 %[dX], s[50:51]\n\t"
#define WOTHER_STAGE_A OTHER_STAGE_A                                           \
  "v_xor_b32 %[rc0], 0x10000, %[rc0]\n\tv_xor_b32 %[rc1], 0x10000, %[rc1]\n\t" \
  "v_xor_b32 %[rc2], 0x10000, %[rc2]\n\tv_xor_b32 %[rc3], 0x10000, %[rc3]\n\t"
#define WOTHER_STAGE_X                                                       \
  "v_xor_b32 %[rx0], 0x1000, %[rx0]\n\tv_xor_b32 %[rx1], 0x1000, %[rx1]\n\t" \
  "v_xor_b32 %[rx2], 0x1000, %[rx2]\n\tv_xor_b32 %[rx3], 0x1000, %[rx3]\n\t"
#define WNEXT_STEP NEXT_STEP "s_add_u32 s50, s50, 128\n\ts_addc_u32 s51, s51, 0\n\t"
#define WOTHER_STAGE_LOADS OTHER_STAGE_LOADS "s_xor_b32 s48, s48, 0x1000\n\t"
#define WPOINTERS POINTERS "s_mov_b64 s[50:51], %[px]\n\ts_mov_b32 s48, %[ldsx]\n\t"
#define WSYNC(v, r) "s_waitcnt vmcnt(" #v ") lgkmcnt(" #r ")\n\ts_barrier\n\t"
#define ON_X(x) x
#define OFF_X(x) ""
#define WPHASE0(G, v)                                                                                                    \
  WSYNC(v, 8)                                                                                                            \
  SLICE(0, 0, A0, B0, 0, READS_BUT(6), RD(B1, 0, 0), G##_M(A0, 0), RD(B1, 1, 0) WRDX(0), G##_L(A0, 0))                   \
  SLICE(0, 0, A0, B0, 1, READS_BUT(7), RD(B1, 0, 1), G##_M(A0, 1), RD(B1, 1, 1) WRDX(1), G##_L(A0, 1))                   \
  SLICE(0, 0, A0, B0, 2, READS_BUT(8), RD(B1, 0, 2), G##_M(A0, 2), RD(B1, 1, 2) WRDX(2), G##_L(A0, 2))                   \
  SLICE(0, 0, A0, B0, 3, READS_BUT(9), RD(B1, 0, 3), G##_M(A0, 3), RD(B1, 1, 3) WRDX(3), G##_L(A0, 3))
#define WPHASE1(G, v)                                                                                                                    \
  WSYNC(v, 12)                                                                                                                           \
  SLICE(0, 1, A0, B1, 0, READS_BUT(9), WRD0(A1, AT_A1_0, 0), G##_M(B0, 0), WRD1(A1, AT_A1_0, 0), G##_L(B0, 0)) WSTRIP(0, A0, 0)          \
  SLICE(0, 1, A0, B1, 1, READS_BUT(8), WRD0(A1, AT_A1_0, 1), G##_M(B0, 1), WRD1(A1, AT_A1_0, 1), G##_L(B0, 1)) WSTRIP(0, A0, 1)          \
  SLICE(0, 1, A0, B1, 2, READS_BUT(7), WRD0(A1, AT_A1_0, 2), G##_M(B0, 2), WRD1(A1, AT_A1_0, 2) OTHER_STAGE_B, G##_L(B0, 2))             \
  WSTRIP(0, A0, 2) WOTHER_STAGE_X                                                                                                        \
  SLICE(0, 1, A0, B1, 3, READS_BUT(6), WRD0(A1, AT_A1_0, 3), G##_M(B0, 3), WRD1(A1, AT_A1_0, 3) WOTHER_STAGE_A, G##_L(B0, 3))            \
  WSTRIP(0, A0, 3)
#define WPHASE2(G, v)                                                                                                                    \
  WSYNC(v, 8)                                                                                                                            \
  SLICE(1, 1, A1, B1, 0, READS_BUT(6), WRD0(A0, AT_A0_0, 0), G##_M(B1, 0), WRD1(A0, AT_A0_0, 0), G##_L(B1, 0)) WSTRIP(1, A1, 0)          \
  SLICE(1, 1, A1, B1, 1, READS_BUT(6), WRD0(A0, AT_A0_0, 1), G##_M(B1, 1), WRD1(A0, AT_A0_0, 1), G##_L(B1, 1)) WSTRIP(1, A1, 1)          \
  SLICE(1, 1, A1, B1, 2, READS_BUT(6), WRD0(A0, AT_A0_0, 2), G##_M(B1, 2), WRD1(A0, AT_A0_0, 2), G##_L(B1, 2)) WSTRIP(1, A1, 2)          \
  SLICE(1, 1, A1, B1, 3, READS_BUT(6), WRD0(A0, AT_A0_0, 3), G##_M(B1, 3), WRD1(A0, AT_A0_0, 3), G##_L(B1, 3))                           \
  G##_X("s_mov_b32 m0, s48\n\t") WSTRIP(1, A1, 3) G##_X(WLOADX)
#define WPHASE3(G, v)                                                                                 \
  WSYNC(v, 8)                                                                                         \
  SLICE(1, 0, A1, B0, 0, NONE, NONE, G##_M(A1, 0), NONE, G##_L(A1, 0))                                \
  SLICE(1, 0, A1, B0, 1, NONE, RD(B0, 0, 0), G##_M(A1, 1), RD(B0, 1, 0), G##_L(A1, 1))                \
  SLICE(1, 0, A1, B0, 2, NONE, RD(B0, 0, 1), G##_M(A1, 2), RD(B0, 1, 1), G##_L(A1, 2))                \
  SLICE(1, 0, A1, B0, 3, NONE, RD(B0, 0, 2), G##_M(A1, 3), RD(B0, 1, 2), G##_L(A1, 3)) RD(B0, 0, 3)   \
  RD(B0, 1, 3)
#define WLAST_HALF                                                                            \
  SLICE(1, 1, A1, B1, 0, READS_BUT(6), NONE, NONE, NONE, NONE) WSTRIP(1, A1, 0)               \
  SLICE(1, 1, A1, B1, 1, READS_BUT(4), NONE, NONE, NONE, NONE) WSTRIP(1, A1, 1)               \
  SLICE(1, 1, A1, B1, 2, READS_BUT(2), NONE, NONE, NONE, NONE) WSTRIP(1, A1, 2)               \
  SLICE(1, 1, A1, B1, 3, READS_BUT(0), NONE, NONE, NONE, NONE) WSTRIP(1, A1, 3)               \
  SLICE(1, 0, A1, B0, 0, NONE, NONE, NONE, NONE, NONE)                                        \
  SLICE(1, 0, A1, B0, 1, NONE, NONE, NONE, NONE, NONE)                                        \
  SLICE(1, 0, A1, B0, 2, NONE, NONE, NONE, NONE, NONE)                                        \
  SLICE(1, 0, A1, B0, 3, NONE, NONE, NONE, NONE, NONE)
#define WSTEP_LOADS LOAD_UNIT(A0) LOAD_UNIT(B0) LOAD_UNIT(B1) "s_mov_b32 m0, s48\n\ts_nop 0\n\t" WLOADX LOAD_UNIT(A1)
// steps 0 and 1 requested: 34 loads
#define WFIRST_LOADS WPOINTERS WSTEP_LOADS WNEXT_STEP WOTHER_STAGE_LOADS WSTEP_LOADS
// n >= 2 steps
#define WMAIN_LOOP                                                                                                       \
  WPOINTERS WNEXT_STEP WNEXT_STEP "s_sub_u32 s47, %[n], 2\n\t"                                                           \
  "s_waitcnt vmcnt(26)\n\ts_barrier\n\t" WRD(A0, AT_A0_0, 0) WRD(A0, AT_A0_0, 1) WRD(A0, AT_A0_0, 2)                     \
  WRD(A0, AT_A0_0, 3) RD_UNIT(B0)                                                                                        \
  "s_cmp_eq_u32 s47, 0\n\ts_cbranch_scc1 2f\n\t"                                                                         \
  "1:\n\t" WPHASE0(ON, 21) WPHASE1(ON, 21) WPHASE2(ON, 21) WPHASE3(ON, 22) WNEXT_STEP WOTHER_STAGE_LOADS                 \
  "s_sub_u32 s47, s47, 1\n\ts_cmp_lg_u32 s47, 0\n\ts_cbranch_scc1 1b\n\t"                                                \
  "2:\n\t" WPHASE0(OFF, 21) WPHASE1(OFF, 17) WPHASE2(OFF, 13) WPHASE3(OFF, 9) WPHASE0(OFF, 4)                            \
  WPHASE1(OFF, 0) WLAST_HALF "s_nop 15\n\ts_nop 7\n\t"

// RING_PLAIN: C (f32) straight from the accumulators, with the biases of grouped products.  RING_SIGMOID: sigmoid(A . B)
// as the next product's operand, whole rows of c16_pitch bf16 values with zeros past the last column.  RING_SILU, RING_GELU: half the tile's B rows are gate_proj's, half up_proj's;
// act(gate) * up, 128 columns a tile, as bf16.  (GemmDesc says what each field means.)
// RING_ROPE_*: grouped q / k / v, rotated and transposed as they leave (GemmDesc::rope_role; rope_s >= 64, groups of whole tiles), for heads
// of 64, 128 and 256 columns, those with biases, and with a norm in front of the rotation.
enum { RING_PLAIN, RING_SIGMOID, RING_SILU, RING_GELU, RING_ROPE_64, RING_ROPE_64_BIAS, RING_ROPE_128, RING_ROPE_128_BIAS, RING_ROPE_256, RING_ROPE_256_NORM };
// q / k / v of an attention (GemmDesc::rope_role) out of the accumulators of a 256 x 256 tile, half of the rows at a time: every
// wavefront puts its 64 rows of both column halves into LDS - with a bias, or leaving the sums of their squares -, row r's piece of four
// columns `chunk` of a column half at place chunk ^ (r & 15).
struct RingRope {  // one group's part of a GemmDesc
  const float *cos, *sin, *bias;  // (NORM: bias is the norm's gamma)
  float *out, *c;
  uint16_t *out16;
  int64_t cs_ss;
  float n_as_float, eps, gamma_offset;
  uint32_t M, N, S;
};
__device__ __forceinline__ uint32_t ring_place(uint32_t r, uint32_t chunk) { return r * 64 + ((chunk ^ (r & 15)) << 2); }
// (IB: blocks of 32 rows that a wavefront has of the half tile, two, or one of 192 rows' second)
template <bool BIAS, bool SQUARES, int IB>
__device__ __forceinline__ void ring_half_to_lds(const f32x16 (&acc)[2][2][2], const float *bias, float *mine, float *sums) {
  const uint32_t lane = threadIdx.x & 63, half = lane >> 5;
  float ss[2] = {0.f, 0.f};
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float4 w;
        if (BIAS) __builtin_memcpy(&w, bias + b * 128 + j * 32 + q * 8 + half * 4, 16);
#pragma unroll
        for (int i = 0; i < IB; ++i) {
          const f32x16 &x = acc[b][i][j];
          float4 v = make_float4(x[q * 4], x[q * 4 + 1], x[q * 4 + 2], x[q * 4 + 3]);
          if (BIAS) { v.x += w.x; v.y += w.y; v.z += w.z; v.w += w.w; }
          if (SQUARES) ss[i] += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
          *(float4 *)(mine + b * 4096 + ring_place(i * 32 + (lane & 31), j * 8 + q * 2 + half)) = v;
        }
      }
  if (SQUARES) {
#pragma unroll
    for (int i = 0; i < IB; ++i) {
      ss[i] += __shfl_xor(ss[i], 32, 64);
      if (!half) sums[i * 32 + lane] = ss[i];
    }
  }
}

// Queries and keys, heads of HD columns, rotated with the arithmetic of rope_kernel; NORM: normed before that with rmsnorm_kernel's.  A lane
// takes a piece of the lower half of a head and its partner of the upper - in the same rows (heads of 64), from the neighbouring
// wavefront (128: each does half of the 64 rows), from the other column half (256) - and stores both.  Table rows serve both column halves
// (not heads of 256), and are on their way a group of pieces ahead: the first group's (`t`) while the tile goes to LDS.
template <int HD, int IB>
struct RingPieces {
  static constexpr uint32_t H = HD / 2, PER = HD == 64 ? 8 : 16, RPU = 64 / PER;  // pieces to half a row, rows to a unit
  static constexpr int UNITS = (HD == 256 ? 8 : 4) * IB, GROUP = 4, BS = HD == 256 ? 1 : 2;  // units of a half tile, of a group; pairs to a unit
  uint32_t row0, sq0, pos0;  // this wavefront's first row, its sequence and position
  uint32_t chunk, row_in, in_half;  // the piece of its row, the row of the first unit, the piece's column of the lower half of its head
  float4 t[GROUP][4];  // cos and sin of the lower half, of the upper
  __device__ __forceinline__ RingPieces(uint32_t first_row, uint32_t S, uint32_t wn, uint32_t lane)
      : row0(first_row), sq0(first_row / S), pos0(first_row - first_row / S * S), chunk(lane % PER), row_in(lane / PER + (HD == 128 ? wn * IB * 16 : 0)),
        in_half((HD == 256 ? wn * 64 : 0) + lane % PER * 4) {}
  __device__ __forceinline__ void tables(const RingRope &d, int u0) {
#pragma unroll
    for (int u = 0; u < GROUP; ++u) {
      const uint32_t r = row_in + (u0 + u) * RPU;
      uint32_t pos = pos0 + (row0 + r < d.M ? r : 0);
      if (pos >= d.S) pos -= d.S;
      const int64_t from = (int64_t)pos * d.cs_ss + in_half;
      t[u][0] = *(const float4 *)(d.cos + from);
      t[u][1] = *(const float4 *)(d.sin + from);
      t[u][2] = *(const float4 *)(d.cos + from + H);
      t[u][3] = *(const float4 *)(d.sin + from + H);
    }
  }
};
template <int HD, bool NORM, int IB>
__device__ __forceinline__ void ring_store_rotated(const RingRope &d, RingPieces<HD, IB> &p, uint32_t n0, float *smem, uint32_t wave, uint32_t lane) {
  typedef RingPieces<HD, IB> P;
  const uint32_t wn = wave & 1, S = d.S, heads = d.N / HD;
  const float *mine = smem + wave * 8192;
  float *sums = smem + 32768 + wave * 128;  // NORM: the sums of squares, then each row's divisor and its inverse
  float4 g_lo, g_hi;
  if (NORM) {  // (heads of 256: a row's columns are with two wavefronts)
    if (d.bias) {
      g_lo = *(const float4 *)(d.bias + p.in_half);
      g_hi = *(const float4 *)(d.bias + p.in_half + P::H);
    }
    const float sum = sums[lane] + smem[32768 + (wave ^ 1) * 128 + lane];
    __syncthreads();
    const float rms = sqrtf(sum / d.n_as_float + d.eps);
    sums[lane] = rms == INFINITY ? 0.f : rms;  // (then 1 / rms = 0, and every finite value of the row leaves as 0)
    sums[64 + lane] = 1.f / rms;
  }
#pragma unroll 1
  for (int u0 = 0; u0 < P::UNITS; u0 += P::GROUP) {
    float4 now[P::GROUP][4];
#pragma unroll
    for (int u = 0; u < P::GROUP; ++u)
#pragma unroll
      for (int k = 0; k < 4; ++k) now[u][k] = p.t[u][k];
    if (u0 + P::GROUP < P::UNITS) p.tables(d, u0 + P::GROUP);
#pragma unroll
    for (int u = 0; u < P::GROUP; ++u) {
      const uint32_t r = p.row_in + (u0 + u) * P::RPU;
#pragma unroll
      for (int b = 0; b < P::BS; ++b) {
        const float *lo = HD == 128 ? smem + (wave & ~1u) * 8192 + b * 4096 : mine + b * 4096;
        const float *hi = HD == 64 ? lo : HD == 128 ? lo + 8192 : lo + 4096;
        float4 x = *(const float4 *)(lo + ring_place(r, p.chunk)), y = *(const float4 *)(hi + ring_place(r, HD == 64 ? p.chunk + 8 : p.chunk));
        if (NORM) {
          // x / rms, rounded once: the quotient by the inverse, and what it leaves of x
          const float rms = sums[r], inv = sums[64 + r];
          auto normed = [&](float v, float w) {
            const float q = v * inv, n = fmaf(fmaf(-q, rms, v), inv, q);
            return d.bias ? n * (d.gamma_offset + w) : n;
          };
          x = make_float4(normed(x.x, g_lo.x), normed(x.y, g_lo.y), normed(x.z, g_lo.z), normed(x.w, g_lo.w));
          y = make_float4(normed(y.x, g_hi.x), normed(y.y, g_hi.y), normed(y.z, g_hi.z), normed(y.w, g_hi.w));
        }
        const float4 c0 = now[u][0], s0 = now[u][1], c1 = now[u][2], s1 = now[u][3];
        // (the compiler's choice in rope_kernel, which product is rounded on its own, written out: the same bits)
        const float4 l = make_float4(fmaf(c0.x, x.x, s0.x * -y.x), fmaf(c0.y, x.y, s0.y * -y.y), fmaf(c0.z, x.z, s0.z * -y.z), fmaf(c0.w, x.w, s0.w * -y.w));
        const float4 h = make_float4(fmaf(c1.x, y.x, s1.x * x.x), fmaf(c1.y, y.y, s1.y * x.y), fmaf(c1.z, y.z, s1.z * x.z), fmaf(c1.w, y.w, s1.w * x.w));
        if (p.row0 + r < d.M) {
          // [sequence][head][position][column]; a position past a sequence's end is the next one's
          const uint32_t head = (n0 + b * 128 + (HD == 64 ? wn * 64 : 0)) / HD, over = p.pos0 + r >= S ? 1 : 0;
          const uint64_t to = ((uint64_t)((p.sq0 + over) * heads + head) * S + (p.pos0 + r - over * S)) * HD + p.in_half;
          if (d.out) {
            *(float4 *)(d.out + to) = l;
            *(float4 *)(d.out + to + P::H) = h;
          }
          if (d.out16) {
            *(uint2 *)(d.out16 + to) = bf16_pack4(l);
            *(uint2 *)(d.out16 + to + P::H) = bf16_pack4(h);
          }
        }
      }
    }
  }
}

// Values: as they are, and as bf16 [sequence][column][position], rows of positions padded with zeros to a multiple of eight.
template <int IB>
__device__ __forceinline__ void ring_store_values(const RingRope &d, uint32_t row0, uint32_t n0, const float *mine, uint32_t wn, uint32_t lane) {
  const uint32_t S = d.S, Sp = (S + 7) & ~7u, sq0 = row0 / S, pos0 = row0 - sq0 * S;
  const uint32_t r0 = (lane >> 2) * 4, row = row0 + r0, over = pos0 + r0 >= S ? 1 : 0, sq = sq0 + over, pos = pos0 + r0 - over * S;
#pragma unroll 1
  for (uint32_t b = 0; b < 2; ++b) {
    const uint32_t col0 = n0 + b * 128 + wn * 64;  // (whole tiles: every column exists)
    const float *tile = mine + b * 4096;
#pragma unroll 4
    for (uint32_t it = 0; it < 8 * IB; ++it) {
      const uint32_t r = it * 4 + (lane >> 4);
      if (row0 + r < d.M) *(float4 *)(d.c + (uint64_t)(row0 + r) * d.N + col0 + (lane & 15) * 4) = *(const float4 *)(tile + ring_place(r, lane & 15));
    }
    // four positions of four columns to a lane
    if (IB == 1 && lane >= 32) continue;
#pragma unroll 1
    for (uint32_t it = 0; it < 4; ++it) {
      const uint32_t chunk = it * 4 + (lane & 3);
      float4 f[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) f[e] = *(const float4 *)(tile + ring_place(r0 + e, chunk));
      uint16_t *to = d.out16 + ((uint64_t)sq * d.N + col0 + chunk * 4) * Sp + pos;
      if (row + 4 <= d.M && pos % 4 == 0 && pos + 4 <= S) {
        const uint2 w[4] = {bf16_pack4(make_float4(f[0].x, f[1].x, f[2].x, f[3].x)), bf16_pack4(make_float4(f[0].y, f[1].y, f[2].y, f[3].y)),
                            bf16_pack4(make_float4(f[0].z, f[1].z, f[2].z, f[3].z)), bf16_pack4(make_float4(f[0].w, f[1].w, f[2].w, f[3].w))};
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          *(uint2 *)(to + (uint64_t)x * Sp) = w[x];
          if (pos + 4 == S && Sp > S) *(uint2 *)(to + (uint64_t)x * Sp + 4) = make_uint2(0u, 0u);
        }
      } else {  // the product's last rows, or four that straddle two sequences
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (row + e >= d.M) continue;
          const bool next = pos + e >= S;
          uint16_t *at = to + e + (next ? (uint64_t)d.N * Sp - S : 0);
          const uint2 h = bf16_pack4(f[e]);
          const uint16_t v[4] = {(uint16_t)h.x, (uint16_t)(h.x >> 16), (uint16_t)h.y, (uint16_t)(h.y >> 16)};
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            at[(uint64_t)x * Sp] = v[x];
            if (pos + e + 1 == (next ? 2 * S : S))
              for (uint32_t z = 1; z <= Sp - S; ++z) at[(uint64_t)x * Sp + z] = 0;
          }
        }
      }
    }
  }
}

// (one place that reads the accumulators: where two branches do, the compiler spills them)
template <int HD, bool BIAS, bool NORM, int AH, bool SHORT>
__device__ __forceinline__ void ring_store_attention(const RingRope d, bool values, uint32_t m0, uint32_t n0, const f32x16 (&acc)[AH][2][2][2], float *smem) {
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave >> 1, wn = wave & 1;
  float *mine = smem + wave * 8192;
  auto half_tile = [&](auto A) __attribute__((always_inline)) {
    constexpr int a = A, IB = SHORT && a ? 1 : 2;
    const uint32_t row0 = m0 + a * 128 + wm * IB * 32;
    RingPieces<HD, IB> p(row0, d.S, wn, lane);
    if (!values) p.tables(d, 0);
    if (a) __syncthreads();  // the other half has been read
    ring_half_to_lds<BIAS, NORM, IB>(acc[a], d.bias + n0 + wn * 64, mine, smem + 32768 + wave * 128);
    __syncthreads();
    if (values) ring_store_values<IB>(d, row0, n0, mine, wn, lane);
    else ring_store_rotated<HD, NORM, IB>(d, p, n0, smem, wave, lane);
  };
  half_tile(std::integral_constant<int, 0>());
  if constexpr (AH == 2) half_tile(std::integral_constant<int, 1>());
}

// AH: halves of 128 rows to a tile, two or (not RING_SIGMOID) one.  WIDE: with the strip of 32 columns (RING_SILU, RING_GELU: 16
// rows of each matrix), N % 4 == 0.  SHORT: 192 rows, the second half is 64.
template <int KIND, int AH, bool WIDE = false, bool SHORT = false>
__global__ void __launch_bounds__(256, 1) gemm_bf16_ring_kernel(GemmDesc g) {
  constexpr bool GATED = KIND == RING_SILU || KIND == RING_GELU;
  constexpr bool ROPE = KIND >= RING_ROPE_64;
  static_assert(!WIDE || (AH == 2 && KIND != RING_SIGMOID && !ROPE), "the strip's epilogues");
  constexpr uint32_t BNO = (GATED ? 128 : 256) + (WIDE ? (GATED ? 16 : 32) : 0);  // output columns of a tile
  warm_kernel_arguments<sizeof(GemmDesc)>();
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wn = wave & 1;
  constexpr uint32_t BM = SHORT ? 192 : AH * 128;
  static_assert(!SHORT || (AH == 2 && !WIDE && (GATED || (ROPE && KIND < RING_ROPE_256))), "the epilogues of 192-row tiles");
  static_assert(AH == 2 || KIND != RING_SIGMOID, "the epilogues of 128-row tiles");
  const uint32_t tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BNO - 1) / BNO;
  const TilePlace place(tiles_m, tiles_n, g.nb0, g.nb1, max(g.splits, 1u));
  const uint32_t batch = g.nb0 * g.nb1, split = place.split, bz = place.bz, b0 = place.b0, b1 = place.b1;
  const uint32_t m0 = place.tm * BM;
  uint32_t n0 = place.tn * BNO, Nl = g.N;
  const uint16_t *B = (const uint16_t *)g.b + b0 * g.sb_b0 + b1 * g.sb_b1;
  float *C = (g.splits > 1 ? g.workspace + (uint64_t)split * batch * g.M * g.N : g.c) + (uint64_t)bz * g.M * g.N;
  const float *Bias = nullptr, *Cadd = KIND == RING_PLAIN && g.c_add && g.splits <= 1 ? g.c_add + (uint64_t)bz * g.M * g.N : nullptr;
  uint32_t grp = 0;
  if ((KIND == RING_PLAIN || ROPE) && g.n_group) {  // grouped products: tiles never straddle two
    uint32_t p = 0;
    while (p + 1 < g.n_group && n0 >= g.grp_n[p]) {
      n0 -= g.grp_n[p];
      ++p;
    }
    B = (const uint16_t *)g.grp_b[p];
    C = g.grp_c[p];
    Nl = g.grp_n[p];
    Bias = g.grp_bias[p];
    grp = p;
  }
  const uint32_t k_begin = split * g.k_per_split, k_end = min(g.K, k_begin + g.k_per_split);
  const uint32_t n_steps = __builtin_amdgcn_readfirstlane((k_end - k_begin) / 64);
  // Where this lane's piece of each load comes from: byte offsets from the tile's first row (rows past the end repeat the last
  // one), the 16-byte chunk swizzled so that the fragment reads are free of bank conflicts.
  const KOrder order(AH == 1 ? g.k_rotate : 0u, place.tn + tiles_n * place.zz, n_steps);  // (tiles of 256 rows have more than 128)
  const uint32_t k_first = k_begin + order.step() * 64;
  const uint16_t *pa = (const uint16_t *)g.a + b0 * g.sa_b0 + b1 * g.sa_b1 + (int64_t)m0 * g.sam + k_first;
  const uint16_t *pb0 = B + (int64_t)n0 * g.sbn + k_first;
  const uint16_t *pb1 = GATED ? (const uint16_t *)g.dual_b + b0 * g.sb_b0 + b1 * g.sb_b1 + (int64_t)n0 * g.sbn + k_first : pb0;
  const uint32_t sa = (uint32_t)g.sam * 2, sb = (uint32_t)g.sbn * 2, last_a = g.M - 1 - m0, last_b = Nl - 1 - n0;
  uint32_t dA0[4], dA1[4], dB0[4], dB1[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t r = (wave * 4 + i) * 8 + (lane >> 3), c = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    dA0[i] = min(r, last_a) * sa + c;
    dA1[i] = min(SHORT ? 128 + (wave * 2 + i) * 8 + (lane >> 3) : r + 128, last_a) * sa + c;  // (SHORT: two pieces)
    dB0[i] = min(r, last_b) * sb + c;
    dB1[i] = GATED ? dB0[i] : min(r + 128, last_b) * sb + c;
  }
  // (the compiler may keep a uniform value in a vector register; the assembly wants scalars)
  auto scalar = [](const uint16_t *p) {
    const uint64_t v = (uint64_t)p;
    return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)v) | (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32;
  };
  const uint64_t sa0 = scalar(pa), sb0 = scalar(pb0), sb1 = scalar(pb1);
  const uint32_t lds = wave * 4096;  // (all LDS of this kernel is the stages, at offset 0: whole_lds)
  // WIDE: eight rows of the strip, behind the columns of the quadrants
  constexpr uint32_t STRIP_AT = 2 * 65536;
  const uint32_t ldsx = STRIP_AT + wave * 1024, rx_row = wave * 8 + (lane >> 3);
  const uint64_t sx = GATED && wave >= 2 ? sb1 : sb0;
  const uint32_t dX = min((GATED ? 128 : 256) + (GATED ? rx_row & 15 : rx_row), last_b) * sb + ((lane & 7) ^ ((rx_row >> 1) & 7)) * 16;
#define RING_IN_B                                                                                                         \
  [dB00] "v"(dB0[0]), [dB01] "v"(dB0[1]), [dB02] "v"(dB0[2]), [dB03] "v"(dB0[3]), [dB10] "v"(dB1[0]), [dB11] "v"(dB1[1]), \
      [dB12] "v"(dB1[2]), [dB13] "v"(dB1[3]), [pb0] "s"(sb0), [pb1] "s"(sb1), [lds] "s"(lds)
#define RING_IN                                                                                                            \
  [dA00] "v"(dA0[0]), [dA01] "v"(dA0[1]), [dA02] "v"(dA0[2]), [dA03] "v"(dA0[3]), [dA10] "v"(dA1[0]), [dA11] "v"(dA1[1]),  \
      [dA12] "v"(dA1[2]), [dA13] "v"(dA1[3]), [pa] "s"(sa0), RING_IN_B
#define RING_ORDER [first] "s"(order.at), [flip] "s"(order.flip), [n] "s"(n_steps)
#define RING_GATHERED [ga0] "+v"(ga[0]), [ga1] "+v"(ga[1]), [ga2] "+v"(ga[2]), [ga3] "+v"(ga[3])
#define RING_HALF_SCALARS "v126", "v127", "s48", "s49", "s50", "s51", "s52", "s53"
#define RING_SCALARS "s54", "s55", "s56", "s57", "s58", "s59", "s40", "s41", "s42", "s43", "s44", "s45", "s46", "s47", "m0", "scc", "memory"
#define RING_V10(d) "v" #d "0", "v" #d "1", "v" #d "2", "v" #d "3", "v" #d "4", "v" #d "5", "v" #d "6", "v" #d "7", "v" #d "8", "v" #d "9"
#define RING_FRAGMENTS                                                                                                     \
  "v128", "v129", RING_V10(13), RING_V10(14), RING_V10(15), RING_V10(16), RING_V10(17), RING_V10(18), RING_V10(19),        \
      RING_V10(20), RING_V10(21), RING_V10(22), RING_V10(23), RING_V10(24), "v250", "v251", "v252", "v253", "v254", "v255"
  uint64_t ga[4];  // AH == 1: this lane's pieces of A, a step on after every load
#pragma unroll
  for (int i = 0; i < 4; ++i) ga[i] = (uint64_t)pa + dA0[i];
#define RING_WIDE_IN [dX] "v"(dX), [px] "s"(sx), [ldsx] "s"(ldsx)
#define RING_WIDE_SCALARS "s48", "s50", "s51"
#define RING_STRIP RING_V10(11), "v120", "v121", "v122", "v123", "v124", "v125", "v126", "v127"
  // SHORT: this wavefront's place for A1 in a stage
  const uint32_t lds1 = lds - (wave & 1) * 2048;
#define RING_SHORT_IN                                                                                                      \
  [dA00] "v"(dA0[0]), [dA01] "v"(dA0[1]), [dA02] "v"(dA0[2]), [dA03] "v"(dA0[3]), [dA10] "v"(dA1[0]), [dA11] "v"(dA1[1]),  \
      [lds1] "s"(lds1), [pa] "s"(sa0), RING_IN_B
  if constexpr (WIDE) asm volatile(WFIRST_LOADS::RING_IN, RING_WIDE_IN : RING_SCALARS, RING_WIDE_SCALARS);
  else if constexpr (SHORT) asm volatile(SFIRST_LOADS::RING_SHORT_IN : RING_SCALARS, "s48");
  else if constexpr (AH == 2) asm volatile(FIRST_LOADS::RING_IN : RING_SCALARS);
  else asm volatile(HFIRST_LOADS("") : RING_GATHERED : RING_IN_B, RING_ORDER : RING_SCALARS);
  float zero;
  asm volatile("v_mov_b32 %0, 0" : "=v"(zero));  // (the accumulators are cleared behind the first loads, not in front of them)
  f32x16 acc[AH][2][2][2];  // [A half][B half][row block][column block]
#pragma unroll
  for (int q = 0; q < AH * 8; ++q)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[q >> 3][(q >> 2) & 1][(q >> 1) & 1][q & 1][e] = zero;
  f32x16 strip[2];  // WIDE: [A half]
#pragma unroll
  for (int e = 0; e < 16; ++e) strip[0][e] = strip[1][e] = zero;
  const uint32_t half = lane >> 5;
  uint32_t ra[4], rb[4], rc[4], rx[4];  // where this lane's fragments of a k-slice start in a unit
  const uint32_t first = WIDE ? wn : 0;  // (row block 0 of the accumulators is this one of the 64 rows' two)
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const uint32_t p = ((ks * 2 + half) ^ ((lane >> 1) & 7)) * 16 + (lane & 31) * 128;
    ra[ks] = wm * 8192 + first * 4096 + p;
    rc[ks] = wm * 8192 + (1 - first) * 4096 + p;
    rb[ks] = wn * 8192 + p;
    rx[ks] = STRIP_AT + p;
  }
  unsigned long long tick0 = 0, real0 = 0;  // (clock probe only: GemmDesc::clock_ticks)
  if (KIND == RING_PLAIN && g.clock_ticks) {
    tick0 = __builtin_amdgcn_s_memtime();
    real0 = __builtin_amdgcn_s_memrealtime();
  }
#define RING_ACC(a, b, i, j) [c##a##b##i##j] "+a"(acc[a][b][i][j])
#define RING_ACC0                                                                                                        \
  RING_ACC(0, 0, 0, 0), RING_ACC(0, 0, 0, 1), RING_ACC(0, 0, 1, 0), RING_ACC(0, 0, 1, 1), RING_ACC(0, 1, 0, 0),          \
      RING_ACC(0, 1, 0, 1), RING_ACC(0, 1, 1, 0), RING_ACC(0, 1, 1, 1)
#define RING_ACC1                                                                                                        \
  RING_ACC(1, 0, 0, 0), RING_ACC(1, 0, 0, 1), RING_ACC(1, 0, 1, 0), RING_ACC(1, 0, 1, 1), RING_ACC(1, 1, 0, 0),          \
      RING_ACC(1, 1, 0, 1), RING_ACC(1, 1, 1, 0), RING_ACC(1, 1, 1, 1)
#define RING_ACC_SHORT RING_ACC(1, 0, 0, 0), RING_ACC(1, 0, 0, 1), RING_ACC(1, 1, 0, 0), RING_ACC(1, 1, 0, 1)
#define RING_PLACES                                                                                                      \
  [ra0] "+v"(ra[0]), [ra1] "+v"(ra[1]), [ra2] "+v"(ra[2]), [ra3] "+v"(ra[3]), [rb0] "+v"(rb[0]), [rb1] "+v"(rb[1]),      \
      [rb2] "+v"(rb[2]), [rb3] "+v"(rb[3])
#define RING_WIDE_PLACES                                                                                                  \
  [x0] "+v"(strip[0]), [x1] "+v"(strip[1]), [rc0] "+v"(rc[0]), [rc1] "+v"(rc[1]), [rc2] "+v"(rc[2]), [rc3] "+v"(rc[3]),   \
      [rx0] "+v"(rx[0]), [rx1] "+v"(rx[1]), [rx2] "+v"(rx[2]), [rx3] "+v"(rx[3])
  if constexpr (WIDE)
    asm volatile(WMAIN_LOOP : RING_ACC0, RING_ACC1, RING_PLACES, RING_WIDE_PLACES : RING_IN, RING_WIDE_IN, [n] "s"(n_steps)
                 : RING_SCALARS, RING_WIDE_SCALARS, RING_STRIP, RING_FRAGMENTS);
  else if constexpr (SHORT)
    asm volatile(SMAIN_LOOP : RING_ACC0, RING_ACC_SHORT, RING_PLACES : RING_SHORT_IN, [n] "s"(n_steps) : RING_SCALARS, "s48", RING_FRAGMENTS);
  else if constexpr (AH == 2)
    asm volatile(MAIN_LOOP : RING_ACC0, RING_ACC1, RING_PLACES : RING_IN, [n] "s"(n_steps) : RING_SCALARS, RING_FRAGMENTS);
  else
    asm volatile(HMAIN_LOOP("") : RING_ACC0, RING_PLACES, RING_GATHERED : RING_IN_B, RING_ORDER : RING_SCALARS, RING_HALF_SCALARS, RING_FRAGMENTS);
  if (KIND == RING_PLAIN && g.clock_ticks && tid == 0) {
    atomicAdd(g.clock_ticks, __builtin_amdgcn_s_memtime() - tick0);
    atomicAdd(g.clock_ticks + 1, __builtin_amdgcn_s_memrealtime() - real0);
  }
  // The tile leaves through LDS, a quadrant at a time and each wavefront for itself: a lane holds pieces of four columns in 32
  // different rows, and stored as they are every instruction would touch 32 lines; out of LDS a store is four rows of 64
  // columns, whole lines.  (Chunks of 16 bytes swizzled by the row: no bank conflicts either way.)  A tile without edges has
  // no branch in all of this: with one per store the accumulators' 256 registers leave one at a time, 8 us a tile.
  // At an edge the sixteen pieces, and what is added to them, are on their way before the first is stored, as in the middle (one
  // after the other, and value by value, 13 us more a tile: 16 x 1000 x 1000 x 128 32 -> 19 us, 16 x 257 x 2000 x 128 30 -> 16,
  // 1500 x 20000 x 1024 90 -> 76, 6000 x 4100 x 256 and a residual 88 -> 55; biases, which took that path in every tile,
  // 6000 x 3072 x 2048 178 -> 95).
  __syncthreads();  // every wavefront has read its last fragments
  extern __shared__ __attribute__((aligned(16))) float ring_smem[];
  if constexpr (ROPE) {
    // (read here, not held through the main loop)
    auto *late = (const __attribute__((address_space(4))) GemmDesc *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(late));
    const RingRope d = {late->rope_cos[grp], late->rope_sin[grp], late->grp_bias[grp], late->rope_out[grp], late->grp_c[grp],
                        late->rope_out16[grp], late->rope_cs_ss[grp], late->rope_n_as_float, late->rope_eps, late->rope_gamma_offset,
                        late->M, late->grp_n[grp], late->rope_s};
    constexpr int HD = KIND >= RING_ROPE_256 ? 256 : KIND >= RING_ROPE_128 ? 128 : 64;
    ring_store_attention<HD, KIND == RING_ROPE_64_BIAS || KIND == RING_ROPE_128_BIAS, KIND == RING_ROPE_256_NORM, AH, SHORT>(d, late->rope_role[grp] == 2, m0, n0, acc, ring_smem);
    return;
  }
  uint16_t *C16 = g.c16 ? g.c16 + (uint64_t)bz * g.M * g.N : nullptr;
  const bool whole = m0 + BM <= g.M && n0 + BNO <= Nl;
  constexpr bool F32 = KIND == RING_PLAIN;
  const uint32_t pitch = KIND == RING_SIGMOID ? g.c16_pitch : Nl;
  uint32_t at_row[4], at_col[4], to[4];  // this lane's piece of rows 0-3, 4-7, 8-11, 12-15 of a quadrant; its bytes from the corner
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    at_row[u] = u * 4 + (lane >> 4);
    at_col[u] = ((lane & 15) ^ at_row[u]) << 2;
    to[u] = (at_row[u] * pitch + at_col[u]) * (F32 ? 4u : 2u);
  }
#pragma unroll
  for (int qd = 0; qd < (GATED ? AH : 2 * AH); ++qd) {
    const int a = GATED ? qd : qd >> 1, b = GATED ? 0 : qd & 1;
    float *tile = ring_smem + wave * 8192 + (qd & 1) * 4096;
    const int blocks = SHORT && a ? 1 : 2;  // of 32 rows (guards in loops of a fixed length: registers are not indexed)
    const uint32_t col0 = n0 + b * 128 + wn * 64, row0 = m0 + a * 128 + wm * blocks * 32;
    if (row0 >= g.M || col0 >= pitch) continue;  // (uniform: nothing of this quadrant is stored)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (i >= blocks) continue;
          const uint32_t r = (i ^ first) * 32 + (lane & 31), chunk = j * 8 + q * 2 + half;
          const f32x16 &x = acc[a][b][i][j], &u = acc[a][GATED ? 1 : b][i][j];
          float4 v = make_float4(x[q * 4], x[q * 4 + 1], x[q * 4 + 2], x[q * 4 + 3]);
          if (KIND == RING_GELU) v = make_float4(gelu_fast(v.x), gelu_fast(v.y), gelu_fast(v.z), gelu_fast(v.w));
          if (KIND == RING_SILU) v = make_float4(silu_fast(v.x), silu_fast(v.y), silu_fast(v.z), silu_fast(v.w));
          if (KIND == RING_SIGMOID) v = make_float4(sigmoid_fast(v.x), sigmoid_fast(v.y), sigmoid_fast(v.z), sigmoid_fast(v.w));
          if (GATED) { v.x *= u[q * 4]; v.y *= u[q * 4 + 1]; v.z *= u[q * 4 + 2]; v.w *= u[q * 4 + 3]; }
          *(float4 *)(tile + r * 64 + ((chunk ^ (r & 15)) << 2)) = v;
        }
    const float *from = tile + ((lane >> 4) << 6) + ((lane & 15) << 2);
    float4 out[16];
#pragma unroll
    for (int it = 0; it < 16; ++it)
      if (it < blocks * 8) out[it] = *(const float4 *)(from + it * 256);
    auto plus = [](float4 x, float4 y) { return make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w); };
    if (F32 && Bias) {  // (grouped products: columns in fours, clamped to the last)
      float4 bias[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) __builtin_memcpy(&bias[u], Bias + min(col0 + at_col[u], Nl - 4), 16);
#pragma unroll
      for (int it = 0; it < 16; ++it) out[it] = plus(out[it], bias[it & 3]);
    }
    if (whole) {
      if (F32 && Cadd) {
        const char *corner = (const char *)(Cadd + (uint64_t)row0 * Nl + col0);
        float4 add[16];
#pragma unroll
        for (int it = 0; it < 16; ++it) __builtin_memcpy(&add[it], corner + (uint64_t)(it >> 2) * 16 * pitch * 4 + to[it & 3], 16);
#pragma unroll
        for (int it = 0; it < 16; ++it) out[it] = plus(out[it], add[it]);
      }
      char *corner = F32 ? (char *)(C + (uint64_t)row0 * Nl + col0) : (char *)(C16 + (uint64_t)row0 * pitch + col0);
#pragma unroll
      for (int it = 0; it < 16; ++it) {
        if (it >= blocks * 8) continue;
        char *at = corner + (uint64_t)(it >> 2) * 16 * pitch * (F32 ? 4 : 2) + to[it & 3];
        if (F32) {
          __builtin_memcpy(at, &out[it], 16);  // (rows of any length: 4-byte aligned)
        } else {
          *(uint2 *)at = bf16_pack4(out[it]);
        }
      }
      continue;
    }
    if (F32) {
      if (Cadd) {  // (rows and columns clamped into the matrix: what is not stored is not used)
        float4 add[16];
#pragma unroll
        for (int it = 0; it < 16; ++it)
          __builtin_memcpy(&add[it], Cadd + (uint64_t)min(row0 + (it >> 2) * 16 + at_row[it & 3], g.M - 1) * Nl + min(col0 + at_col[it & 3], Nl - 4), 16);
#pragma unroll
        for (int it = 0; it < 16; ++it) out[it] = plus(out[it], add[it]);
      }
#pragma unroll
      for (int it = 0; it < 16; ++it) {
        const uint32_t row = row0 + (it >> 2) * 16 + at_row[it & 3], col = col0 + at_col[it & 3];
        if (row < g.M && col + 4 <= Nl) __builtin_memcpy(C + (uint64_t)row * Nl + col, &out[it], 16);
      }
      if (Nl % 4 && col0 + 64 > Nl) {  // the last one to three columns (a product that is not grouped)
#pragma unroll
        for (int it = 0; it < 16; ++it) {
          const uint32_t row = row0 + (it >> 2) * 16 + at_row[it & 3], col = col0 + at_col[it & 3];
          if (row < g.M && col < Nl && col + 4 > Nl) {
            float4 v = *(const float4 *)(from + it * 256);
            const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int k = 0; k < 3; ++k)
              if (col + k < Nl) C[(uint64_t)row * Nl + col + k] = Cadd ? e[k] + Cadd[(uint64_t)row * Nl + col + k] : e[k];
          }
        }
      }
    } else {  // (N % 4 == 0, or padded rows: a piece is inside or outside; zeros past the last column)
#pragma unroll
      for (int it = 0; it < 16; ++it) {
        if (it >= blocks * 8) continue;
        const uint32_t row = row0 + (it >> 2) * 16 + at_row[it & 3], col = col0 + at_col[it & 3];
        float4 v = out[it];
        v = make_float4(col < Nl ? v.x : 0.f, col + 1 < Nl ? v.y : 0.f, col + 2 < Nl ? v.z : 0.f, col + 3 < Nl ? v.w : 0.f);
        if (row < g.M && col < pitch) *(uint2 *)(C16 + (uint64_t)row * pitch + col) = bf16_pack4(v);
      }
    }
  }
  if constexpr (WIDE) {
    // The strip: 32 rows of each half of A, 32 columns (16 where it is gated: of a block's columns the first 16 are gate's, and the
    // same lane holds up's).  Rows of 128 bytes, out of LDS eight (gated: 32, sixteen) to a store.
    constexpr int CH = GATED ? 4 : 8, RPS = 64 / CH;  // pieces of four columns to a row, rows to a store
    constexpr uint32_t Q = GATED ? 2 : 4;
    float *tile = ring_smem + wave * 8192;
    const uint32_t col = n0 + (GATED ? 128 : 256) + (lane % CH) * 4;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
      for (uint32_t q = 0; q < Q; ++q) {
        const f32x16 &x = strip[a];
        float4 v = make_float4(x[q * 4], x[q * 4 + 1], x[q * 4 + 2], x[q * 4 + 3]);
        if (KIND == RING_GELU) v = make_float4(gelu_fast(v.x), gelu_fast(v.y), gelu_fast(v.z), gelu_fast(v.w));
        if (KIND == RING_SILU) v = make_float4(silu_fast(v.x), silu_fast(v.y), silu_fast(v.z), silu_fast(v.w));
        if (GATED) { v.x *= x[q * 4 + 8]; v.y *= x[q * 4 + 9]; v.z *= x[q * 4 + 10]; v.w *= x[q * 4 + 11]; }
        *(float4 *)(tile + a * 1024 + (lane & 31) * 32 + (((q * 2 + half) ^ (lane & (CH - 1))) << 2)) = v;
      }
      const uint32_t row0 = m0 + a * 128 + wm * 64 + first * 32;
#pragma unroll
      for (int it = 0; it < 32 / RPS; ++it) {
        const uint32_t r = it * RPS + lane / CH, row = row0 + r;
        float4 v = *(const float4 *)(tile + a * 1024 + r * 32 + (((lane % CH) ^ (r & (CH - 1))) << 2));
        if (row >= g.M || col >= Nl) continue;  // (N % 4 == 0: a piece is inside or outside)
        if (GATED) {
          *(uint2 *)(C16 + (uint64_t)row * pitch + col) = bf16_pack4(v);
          continue;
        }
        if (Cadd) {
          float4 add;
          __builtin_memcpy(&add, Cadd + (uint64_t)row * Nl + col, 16);
          v = make_float4(v.x + add.x, v.y + add.y, v.z + add.z, v.w + add.w);
        }
        __builtin_memcpy(C + (uint64_t)row * Nl + col, &v, 16);
      }
    }
  }
}

// ---- the routed experts of a prefill: a row tile of 128 (slot, token) pairs of one expert by 256 weight rows ------------------
// (MoeGemmDesc with route_tiles; the work and its order are those of moe_gemm_dma_kernel, which says how pairs are sorted.)
// MOE_SILU, MOE_GELU: 128 rows of gate_proj and the same of up_proj, act(gate) * up leaves as bf16; MOE_PLAIN: 256 rows of one
// matrix, f32.  Rows of A are gathered; those past the expert's last pair are some token's, and are not stored.
//
// MoeGemmDesc::dense is one more expert that all tokens pass through, tiles of the same launch: the routed ones wait for memory (68 rows
// to 256 of weights), its tiles for the matrix cores, and neither launch has a last round of its own.  60 experts of 2 x 1408 x 2048 and
// 2048 x 1408, 4 to a token, a dense one of 5632, 1024 tokens, both launches: 338 us in four launches and a sum of k-slices, 252 so; 1500
// tokens 380, 293; 660 309, 247; 2600 590, 510.
//
// Bound by the stream of weights, which the loads alone take 117 and 60 us for (692 and 346 MB; 256 workgroups that load these tiles into
// LDS and do nothing else).  What it reaches of that, without the dense expert, 140 and 76 us (before: 158 and 84):
//   * Weights that one row tile reads are loaded with the hint that they are used once, what others will read is not (60 experts, 1024
//     tokens 236 -> 216 us in both launches, the dense tiles' weights with it 277 instead of 253; 2048 tokens, two row tiles to most
//     experts, 334 and 347 with it).
//   * Results leave with that hint, whole lines at a time: 83 -> 76 us for the f32 result of 33 MB, 144 -> 140 for gate and up.
//   * What a tile needs to know comes in two trips to memory in front of its first load - the place of a row tile's pairs in the list
//     follows from the work list's entry -, and where its rows go with them: under the weights' stream a trip is 2 to 4 us.
//   * The row tiles of a crowded expert stand next to each other (2048 tokens, both launches with the dense expert 440 -> 424 us, 4096 708
//     -> 677, 1024 in crowded experts 301 -> 293; by expert and row tile before).
//   * A loop over tiles that requests the next one's first steps in front of the stores of this one: no change (217 and 216 us).
// A dense expert's down_proj is deep, and in slices of k by itself: every other step of it has accumulators of its own, so that its sums
// are no longer chains than in two slices (5632 values off by 3.24e-7 of the 64-bit sum, in one chain 4.69e-7; the same time).
enum { MOE_PLAIN, MOE_SILU, MOE_GELU };
template <int KIND>
__global__ void __launch_bounds__(256, 1) moe_ring_kernel(MoeGemmDesc g) {
  constexpr bool GATED = KIND != MOE_PLAIN;
  constexpr uint32_t BNO = GATED ? 128 : 256;
  typedef const __attribute__((address_space(4))) uint32_t *Uniform;  // (read by scalar loads: written by the launch before)
  warm_kernel_arguments<sizeof(MoeGemmDesc)>();
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wn = wave & 1;
  const uint32_t prob = GATED ? 0 : blockIdx.y, tiles_n = (g.prob[prob].N + BNO - 1) / BNO;
  // This XCD's tiles: its columns of the dense expert, all row tiles of a column one after the other, and a contiguous range of the
  // routed experts' that makes the numbers of all XCDs equal.
  const uint32_t dense_m = (g.S + 127) / 128, dense_n = (g.dense.N + BNO - 1) / BNO, xcd = blockIdx.x & 7, at = blockIdx.x >> 3;
  const uint32_t total = ((Uniform)g.route_tiles)[0] * tiles_n + dense_m * dense_n, mine = total / 8 + (xcd < total % 8);
  const uint32_t mine_dense = dense_m * (dense_n / 8 + (xcd < dense_n % 8));
  if (at >= mine) return;  // the grid is sized for the most tiles there can be, and the wider problem
  uint32_t before;  // dense tiles in front of this one
  bool dense;
  if (g.dense.K > g.K) {  // the longer tiles first
    before = min(at, mine_dense);
    dense = at < mine_dense;
  } else {  // spread evenly: what waits for the matrix cores among what waits for memory
    before = uniform_quotient(at * mine_dense, mine);
    dense = uniform_quotient((at + 1) * mine_dense, mine) > before;
  }
  const uint32_t *list = g.route_list;
  uint32_t e = 0, m0, n0, live, N = g.prob[prob].N, K = g.K;
  bool once = false;  // no other row tile reads these weights
  if (dense) {
    const uint32_t col = uniform_quotient(before, dense_m);
    m0 = (before - col * dense_m) * 128;
    n0 = (col * 8 + xcd) * BNO;
    live = min(g.S - m0, 128u);
    N = g.dense.N;
    K = g.dense.K;
  } else {
    const uint32_t t = xcd * (total / 8) + min(xcd, total % 8) - dense_m * (xcd * (dense_n / 8) + min(xcd, dense_n % 8)) + at - before;
    const uint32_t tile = uniform_quotient(t, tiles_n), entry = ((Uniform)g.route_tiles)[1 + tile], many = moe_entry_tiles(entry);
    e = moe_entry_expert(entry);
    uint32_t row = moe_entry_row(entry), col = t - tile * tiles_n;
    list += (tile - row) * 128;
    if (many > 1) {  // an expert's column tiles one after the other, all row tiles at each: they share the weights
      const uint32_t place = row * tiles_n + col;
      col = uniform_quotient(place, many);
      row = place - col * many;
    }
    n0 = col * BNO;
    m0 = row * 128;
    list += m0;
    const uint32_t pairs = ((Uniform)g.route_count)[e];
    live = min(pairs - m0, 128u);
    once = pairs <= 128;
  }
  uint32_t ent[5];  // slot << 16 | token of this lane's rows of A, and of the row it sends off
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const uint32_t r = i < 4 ? (wave * 4 + i) * 8 + (lane >> 3) : wm * 64 + lane, in_list = list[r];
    ent[i] = dense ? m0 + r : in_list;
    if (r >= live) ent[i] = 0;  // past the expert's last pair, where the list is not written: some token's row, not stored
  }
  const uint32_t n_steps = __builtin_amdgcn_readfirstlane(K / 64);
  const int64_t sbn0 = dense ? g.dense.sbn : g.prob[prob].sbn, sbn1 = dense || !GATED ? sbn0 : g.prob[1].sbn;
  // (routed experts: no flip, since the row tile that a pair lies in depends on the order in which the sort's atomics land)
  const KOrder order(dense ? 0u : g.k_rotate, e * tiles_n + n0 / BNO, n_steps, dense ? m0 / 128 + n0 / BNO : 0u);
  const uint16_t *w0 = dense ? (const uint16_t *)g.dense.w[0] : (const uint16_t *)g.prob[prob].w + (int64_t)e * g.sb_index;
  const uint16_t *w1 = dense ? (const uint16_t *)g.dense.w[1] : (const uint16_t *)g.prob[1].w + (int64_t)e * g.sb_index;
  const uint16_t *pb0 = w0 + (int64_t)n0 * sbn0 + order.step() * 64, *pb1 = GATED ? w1 + (int64_t)n0 * sbn1 + order.step() * 64 : pb0;
  const uint32_t sb = (uint32_t)sbn0 * 2, sb1 = (uint32_t)sbn1 * 2, last_b = N - 1 - n0;
  const uint16_t *rows = dense ? g.dense.a16 : g.slot[0].a16;
  const int64_t row_pitch = dense ? g.dense.a_bs : g.slot[0].a_bs;
  uint64_t ga[4];
  uint32_t dB0[4], dB1[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t r = (wave * 4 + i) * 8 + (lane >> 3), c = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    ga[i] = (uint64_t)(rows + (ent[i] >> 16) * g.a_slot + (ent[i] & 0xFFFFu) * row_pitch) + order.step() * 128 + c;
    dB0[i] = min(r, last_b) * sb + c;
    dB1[i] = GATED ? min(r, last_b) * sb1 + c : min(r + 128, last_b) * sb + c;
  }
  auto scalar = [](const uint16_t *p) {
    const uint64_t v = (uint64_t)p;
    return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)v) | (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32;
  };
  const uint64_t s_b0 = scalar(pb0), s_b1 = scalar(pb1);
  const uint32_t lds = wave * 4096;  // (as above)
#define MOE_IN                                                                                                            \
  [dB00] "v"(dB0[0]), [dB01] "v"(dB0[1]), [dB02] "v"(dB0[2]), [dB03] "v"(dB0[3]), [dB10] "v"(dB1[0]), [dB11] "v"(dB1[1]), \
      [dB12] "v"(dB1[2]), [dB13] "v"(dB1[3]), [pb0] "s"(s_b0), [pb1] "s"(s_b1), [lds] "s"(lds)
  if (once) asm volatile(HFIRST_LOADS(" nt") : RING_GATHERED : MOE_IN, RING_ORDER : RING_SCALARS);
  else asm volatile(HFIRST_LOADS("") : RING_GATHERED : MOE_IN, RING_ORDER : RING_SCALARS);
  const uint64_t out = (uint64_t)(GATED ? (void *)(dense ? g.dense.h16 : g.slot[0].h16) : (void *)(dense ? g.dense.c : g.slot[0].c[prob]));
  const uint64_t base = out + ((ent[4] >> 16) * g.out_slot + (ent[4] & 0xFFFFu) * (uint64_t)N) * (GATED ? 2 : 4);
  float zero;
  asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
  f32x16 acc[GATED ? 1 : 2][2][2][2];  // [0, or every other step's][B half][row block][column block]
#pragma unroll
  for (int q = 0; q < 8; ++q)
#pragma unroll
    for (int k = 0; k < 16; ++k) acc[0][q >> 2][(q >> 1) & 1][q & 1][k] = zero;
  const uint32_t half = lane >> 5;
  uint32_t ra[4], rb[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const uint32_t p = ((ks * 2 + half) ^ ((lane >> 1) & 7)) * 16 + (lane & 31) * 128;
    ra[ks] = wm * 8192 + p;
    rb[ks] = wn * 8192 + p;
  }
  if (once) {
    asm volatile(HMAIN_LOOP(" nt") : RING_ACC0, RING_PLACES, RING_GATHERED : MOE_IN, RING_ORDER : RING_SCALARS, RING_HALF_SCALARS, RING_FRAGMENTS);
  } else if (!GATED && dense) {
    if constexpr (!GATED) {
#pragma unroll
      for (int q = 0; q < 8; ++q)
#pragma unroll
        for (int k = 0; k < 16; ++k) acc[1][q >> 2][(q >> 1) & 1][q & 1][k] = zero;
      asm volatile(HMAIN_LOOP_2("") : RING_ACC0, RING_ACC1, RING_PLACES, RING_GATHERED : MOE_IN, RING_ORDER : RING_SCALARS, RING_HALF_SCALARS, RING_FRAGMENTS);
#pragma unroll
      for (int q = 0; q < 8; ++q)
#pragma unroll
        for (int k = 0; k < 16; ++k) acc[0][q >> 2][(q >> 1) & 1][q & 1][k] += acc[1][q >> 2][(q >> 1) & 1][q & 1][k];
    }
  } else {
    asm volatile(HMAIN_LOOP("") : RING_ACC0, RING_PLACES, RING_GATHERED : MOE_IN, RING_ORDER : RING_SCALARS, RING_HALF_SCALARS, RING_FRAGMENTS);
  }
  // Rows back to their slot and token, through 4 KB of LDS of each wavefront's own: 32 rows of 64 bf16 or of 32 f32 values at a time, of
  // which eight lanes store a line.  A lane knows where the row of its number goes, and hands that to the eight.
  __syncthreads();  // every wavefront has read its last fragments
  extern __shared__ __attribute__((aligned(16))) float ring_smem[];
  float *stage = ring_smem + wave * 1024;
  const uint32_t my_rows = live > wm * 64u ? live - wm * 64u : 0u, piece = (lane & 7) ^ (lane >> 3);
  const int base_lo = (int)base, base_hi = (int)(base >> 32);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint64_t to[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int r = i * 32 + it * 8 + (lane >> 3);
      to[it] = (uint64_t)(uint32_t)__shfl(base_lo, r, 64) | (uint64_t)(uint32_t)__shfl(base_hi, r, 64) << 32;
    }
    if constexpr (GATED) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t r = lane & 31, chunk = j * 8 + q * 2 + half;  // four columns
          const f32x16 &x = acc[0][0][i][j], &u = acc[0][1][i][j];
          float4 v = make_float4(x[q * 4], x[q * 4 + 1], x[q * 4 + 2], x[q * 4 + 3]);
          if (KIND == MOE_GELU) v = make_float4(gelu_fast(v.x), gelu_fast(v.y), gelu_fast(v.z), gelu_fast(v.w));
          if (KIND == MOE_SILU) v = make_float4(silu_fast(v.x), silu_fast(v.y), silu_fast(v.z), silu_fast(v.w));
          v.x *= u[q * 4]; v.y *= u[q * 4 + 1]; v.z *= u[q * 4 + 2]; v.w *= u[q * 4 + 3];
          *(uint2 *)((char *)stage + r * 128 + ((chunk ^ ((r & 7) << 1)) << 3)) = bf16_pack4(v);
        }
      const uint32_t col = n0 + wn * 64 + (lane & 7) * 8;
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const u32x4 v = *(const u32x4 *)((const char *)stage + (it * 8 + (lane >> 3)) * 128 + piece * 16);
        if (i * 32 + it * 8 + (lane >> 3) < my_rows && col < N)  // (N % 8 == 0: a piece is inside or outside)
          __builtin_nontemporal_store(v, (u32x4 *)((uint16_t *)to[it] + col));
      }
    } else {
#pragma unroll
      for (int b = 0; b < 4; ++b) {  // column half, block of 32 columns
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x16 &x = acc[0][b >> 1][i][b & 1];
          *(float4 *)(stage + (lane & 31) * 32 + (((q * 2 + half) ^ (lane & 7)) << 2)) = make_float4(x[q * 4], x[q * 4 + 1], x[q * 4 + 2], x[q * 4 + 3]);
        }
        const uint32_t col = n0 + (b >> 1) * 128 + wn * 64 + (b & 1) * 32 + (lane & 7) * 4;
#pragma unroll
        for (int it = 0; it < 4; ++it) {
          const f32x4 v = *(const f32x4 *)(stage + (it * 8 + (lane >> 3)) * 32 + piece * 4);
          if (i * 32 + it * 8 + (lane >> 3) < my_rows && col < N) __builtin_nontemporal_store(v, (f32x4 *)((float *)to[it] + col));
        }
      }
    }
  }
}

// what lies between the rows and between the results of consecutive slots, in values
static bool moe_slot_pitches(const MoeGemmDesc &g, int64_t *a, int64_t *out) {
  const int64_t ob = g.fuse_glu ? 2 : 4;
  auto out_of = [&](uint32_t s, uint32_t p) { return g.fuse_glu ? (int64_t)(intptr_t)g.slot[s].h16 : (int64_t)(intptr_t)g.slot[s].c[p]; };
  const int64_t ab = g.n_slot > 1 ? (int64_t)(intptr_t)g.slot[1].a16 - (int64_t)(intptr_t)g.slot[0].a16 : 0, cb = g.n_slot > 1 ? out_of(1, 0) - out_of(0, 0) : 0;
  for (uint32_t s = 0; s < g.n_slot; ++s) {
    if ((int64_t)(intptr_t)g.slot[s].a16 != (int64_t)(intptr_t)g.slot[0].a16 + s * ab || g.slot[s].a_bs != g.slot[0].a_bs) return false;
    for (uint32_t p = 0; p < (g.fuse_glu ? 1 : g.n_prob); ++p)
      if (out_of(s, p) != out_of(0, p) + s * cb) return false;
  }
  *a = ab / 2;
  *out = cb / ob;
  return ab % 2 == 0 && cb % ob == 0;
}

// (32-bit byte offsets within a tile's weight rows, three k-steps; otherwise what moe_gemm_pipelined_ok asks)
bool moe_ring_ok(const MoeGemmDesc &g) {
  // With few pairs to an expert most of a tile's products are padding, and they cost what they cost here, where eight wavefronts
  // wait for weights either way (a whole prefill of 60 experts, 4 to a token: 17 pairs to an expert 7.85 -> 8.55 ms, 34 9.49 ->
  // 9.77, 40 9.73 -> 9.82; 47 10.9 -> 10.3, 73 13.8 -> 12.4).
  if ((uint64_t)g.S * g.n_slot < 44 * (uint64_t)g.n_expert) return false;
  int64_t a, out;
  if (!moe_gemm_pipelined_ok(g) || g.planes || g.K < 192 || !moe_slot_pitches(g, &a, &out)) return false;
  for (uint32_t p = 0; p < g.n_prob; ++p)
    if (g.prob[p].sbn < 0 || g.prob[p].sbn > (1 << 22)) return false;
  return g.fuse_glu ? g.n_prob == 2 && g.prob[0].N == g.prob[1].N : true;
}

// The dense expert's tiles are dealt to the XCDs by whole columns, and the others even that out: there have to be enough of those (eight
// columns' worth), and few enough of all for the products of their numbers.
// Up to 3072 tokens: beyond, the routed experts' tiles wait for the matrix cores too, and 256 x 256 tiles are as fast for the dense one (24 layers
// of 60 experts of 2 x 1408 x 2048 and 2048 x 1408, 4 to a token, a dense one of 5632, ms with it in launches of its own and in these: 660 tokens
// 8.26, 7.52; 1024 10.5, 9.73; 1400 11.8, 10.96; 2048 15.3, 14.6; 2600 18.6, 18.2; 4096 24.9, 24.7; 6144 39.6, 39.6; 8192 48.3, 48.9; 16384 93.8
// either way).
bool moe_dense_ok(const MoeGemmDesc &g) {
  const auto &d = g.dense;
  const uint64_t bno = g.fuse_glu ? 128 : 256, rows = (g.S + 127) / 128, cols = (d.N + bno - 1) / bno, tiles_n = (g.prob[0].N + bno - 1) / bno;
  const uint64_t fewest = ((uint64_t)g.S * g.n_slot + 127) / 128 * tiles_n, most = moe_route_max_tiles(g) * tiles_n + rows * cols;
  if (!d.N || !moe_ring_ok(g) || g.S > 3072 || (!g.fuse_glu && g.n_prob != 1) || fewest < 8 * rows || most / 8 >= 65535 || rows * (cols / 8 + 1) >= 65535) return false;
  return d.N % 8 == 0 && d.K % 64 == 0 && d.K >= 192 && d.a16 && (uintptr_t)d.a16 % 16 == 0 && d.a_bs % 8 == 0 && (uintptr_t)d.w[0] % 16 == 0 &&
         (!g.fuse_glu || (uintptr_t)d.w[1] % 16 == 0) && d.sbn % 8 == 0 && d.sbn >= 0 && d.sbn <= (1 << 22) &&
         (g.fuse_glu ? d.h16 && (uintptr_t)d.h16 % 16 == 0 : d.c && (uintptr_t)d.c % 16 == 0);
}

template <int KIND>
static hipError_t launch_moe_ring_as(const LaunchCtx &lc, const MoeGemmDesc &g, dim3 grid) {
  constexpr int smem = 10 * 16384;
  static bool configured = false;  // one attribute call per kernel and process
  if (!configured) {
    const hipError_t e = whole_lds((const void *)moe_ring_kernel<KIND>, smem);
    if (e != hipSuccess) return e;
    configured = true;
  }
  cg_launch(lc, moe_ring_kernel<KIND>, grid, dim3(256), smem, g);
  return hipGetLastError();
}

hipError_t launch_moe_ring(const LaunchCtx &lc, const MoeGemmDesc &given) {
  MoeGemmDesc g = given;
  if (!moe_ring_ok(g) || (g.dense.N && !moe_dense_ok(g)) || !moe_slot_pitches(g, &g.a_slot, &g.out_slot)) return hipErrorInvalidValue;
  uint32_t max_n = 0;
  for (uint32_t p = 0; p < g.n_prob; ++p) max_n = g.prob[p].N > max_n ? g.prob[p].N : max_n;
  const uint32_t bno = g.fuse_glu ? 128 : 256;
  const uint32_t most = (max_n + bno - 1) / bno * moe_route_max_tiles(g) + (g.S + 127) / 128 * ((g.dense.N + bno - 1) / bno);
  const dim3 grid((most + 7) / 8 * 8, g.fuse_glu ? 1 : g.n_prob, 1);
  if (g.fuse_glu) return g.fuse_glu == PRO_GEGLU ? launch_moe_ring_as<MOE_GELU>(lc, g, grid) : launch_moe_ring_as<MOE_SILU>(lc, g, grid);
  return launch_moe_ring_as<MOE_PLAIN>(lc, g, grid);
}

// q / k / v that rotate as they leave: groups of whole tiles (so whole heads), all with a bias or none, all that rotate normed or none
// (heads of 256, no bias), sequences no shorter than the 64 rows that a wavefront stores at a time.
static bool gemm_ring_rope_ok(const GemmDesc &g) {
  if (!g.n_group || g.splits > 1 || g.rope_s < 64 || (g.rope_hd != 64 && g.rope_hd != 128 && g.rope_hd != 256)) return false;
  bool norm = false, plain = false;
  for (uint32_t p = 0; p < g.n_group; ++p) {
    if (!g.rope_role[p] || g.grp_n[p] % 256) return false;
    if (g.rope_role[p] != 3 && g.grp_bias[p] && g.rope_hd == 256) return false;
    if (g.rope_hd != 256 && !g.grp_bias[p] != !g.grp_bias[0]) return false;
    norm = norm || g.rope_role[p] == 3;
    plain = plain || g.rope_role[p] == 1;
  }
  return !norm || (!plain && g.rope_hd == 256);
}

// Operands whose rows lie within 32-bit byte offsets of a tile's first row, two k-steps at least to each slice.
bool gemm_ring_ok(const GemmDesc &g) {
  const uint32_t splits = g.splits > 1 ? g.splits : 1, last = splits > 1 ? g.K - (splits - 1) * g.k_per_split : g.K;
  if (splits > 1 && ((uint64_t)(splits - 1) * g.k_per_split >= g.K || g.k_per_split % 64 || g.k_per_split < 128)) return false;
  return g.sak == 1 && g.sbk == 1 && last % 64 == 0 && last >= 128 && g.sam >= 0 && g.sbn >= 0 && g.sam <= (1 << 22) &&
         g.sbn <= (1 << 22) && (!g.rope_s || gemm_ring_rope_ok(g)) && !g.glu_gate && (!g.act_sigmoid || splits > 1 || g.c16_pitch) &&
         (!g.dual_b || (g.c16 && !g.c));
}

template <int KIND, int AH = 2, bool WIDE = false, bool SHORT = false>
static hipError_t launch_ring_as(const LaunchCtx &lc, const GemmDesc &g, uint32_t grid) {
  constexpr int smem = AH == 2 ? 2 * 65536 + (WIDE ? 2 * 4096 : 0) + (KIND >= RING_ROPE_64 ? 4 * 128 * 4 : 0) : 10 * 16384;  // (ring_store_rotated: sums of squares)
  static bool configured = false;  // one attribute call per kernel and process
  if (!configured) {
    const hipError_t e = whole_lds((const void *)gemm_bf16_ring_kernel<KIND, AH, WIDE, SHORT>, smem);
    if (e != hipSuccess) return e;
    configured = true;
  }
  cg_launch(lc, gemm_bf16_ring_kernel<KIND, AH, WIDE, SHORT>, dim3(grid), dim3(256), smem, g);
  return hipGetLastError();
}

template <int AH>
static hipError_t launch_ring_rope(const LaunchCtx &lc, const GemmDesc &g, uint32_t grid) {
  const bool bias = g.grp_bias[0] != nullptr, norm = g.rope_role[0] == 3 || g.rope_role[1] == 3 || g.rope_role[2] == 3;
  if (g.rope_hd == 256) return norm ? launch_ring_as<RING_ROPE_256_NORM, AH>(lc, g, grid) : launch_ring_as<RING_ROPE_256, AH>(lc, g, grid);
  if (g.rope_hd == 128) return bias ? launch_ring_as<RING_ROPE_128_BIAS, AH>(lc, g, grid) : launch_ring_as<RING_ROPE_128, AH>(lc, g, grid);
  return bias ? launch_ring_as<RING_ROPE_64_BIAS, AH>(lc, g, grid) : launch_ring_as<RING_ROPE_64, AH>(lc, g, grid);
}

bool gemm_ring_192_ok(const GemmDesc &g) {
  return gemm_ring_ok(g) && g.splits <= 1 && !g.act_sigmoid && (g.dual_b || (g.rope_s && g.rope_hd != 256));
}

hipError_t launch_gemm_ring(const LaunchCtx &lc, const GemmDesc &g, RingTile tile) {
  if (!gemm_ring_ok(g)) return hipErrorInvalidValue;
  if (tile == RING_128 && (g.act_sigmoid || g.splits > 1 || g.K < 192)) return hipErrorInvalidValue;
  if (tile == RING_192 && !gemm_ring_192_ok(g)) return hipErrorInvalidValue;
  if (tile == RING_288 && (g.N % 4 || g.n_group || g.act_sigmoid || g.rope_s)) return hipErrorInvalidValue;
  const uint32_t bm = tile == RING_128 ? 128 : tile == RING_192 ? 192 : 256, bn = tile == RING_288 ? 288 : 256, bno = g.dual_b ? bn / 2 : bn;
  const uint64_t tiles = (uint64_t)((g.M + bm - 1) / bm) * ((g.N + bno - 1) / bno) * g.nb0 * g.nb1 * (g.splits > 1 ? g.splits : 1);
  if (tiles > 0x7FFFFFFFull) return hipErrorInvalidValue;
  const uint32_t grid = (uint32_t)tiles;
  if (tile == RING_192) {
    if (g.dual_b) return g.glu_kind ? launch_ring_as<RING_GELU, 2, false, true>(lc, g, grid) : launch_ring_as<RING_SILU, 2, false, true>(lc, g, grid);
    const bool bias = g.grp_bias[0] != nullptr;
    if (g.rope_hd == 128)
      return bias ? launch_ring_as<RING_ROPE_128_BIAS, 2, false, true>(lc, g, grid) : launch_ring_as<RING_ROPE_128, 2, false, true>(lc, g, grid);
    return bias ? launch_ring_as<RING_ROPE_64_BIAS, 2, false, true>(lc, g, grid) : launch_ring_as<RING_ROPE_64, 2, false, true>(lc, g, grid);
  }
  if (tile == RING_128) {
    if (g.rope_s) return launch_ring_rope<1>(lc, g, grid);
    if (!g.dual_b) return launch_ring_as<RING_PLAIN, 1>(lc, g, grid);
    return g.glu_kind ? launch_ring_as<RING_GELU, 1>(lc, g, grid) : launch_ring_as<RING_SILU, 1>(lc, g, grid);
  }
  if (tile == RING_288) {
    if (!g.dual_b) return launch_ring_as<RING_PLAIN, 2, true>(lc, g, grid);
    return g.glu_kind ? launch_ring_as<RING_GELU, 2, true>(lc, g, grid) : launch_ring_as<RING_SILU, 2, true>(lc, g, grid);
  }
  if (g.rope_s) return launch_ring_rope<2>(lc, g, grid);
  if (g.dual_b) return g.glu_kind ? launch_ring_as<RING_GELU>(lc, g, grid) : launch_ring_as<RING_SILU>(lc, g, grid);
  if (g.act_sigmoid && g.splits <= 1) return launch_ring_as<RING_SIGMOID>(lc, g, grid);
  return launch_ring_as<RING_PLAIN>(lc, g, grid);
}

}  // namespace cgk
