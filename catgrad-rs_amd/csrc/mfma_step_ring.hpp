// mfma_step_ring.hpp — the main loop of the direct-to-LDS bf16 GEMM on four wavefronts, for tiles of 128 x 128 and 192 x 128, as
// one statement of assembly.
//
// These tiles hold one workgroup to a CU (few tiles, or an odd number of rows) and are bound by what the CU takes in and by how
// long a load is under way, so as many stages as LDS holds are in flight and the loads are spread over a step (see
// k_gemm_ring.hip for what a burst of them costs).  A wavefront owns RA x RB blocks of 32 x 32; a k-step of 64 is four slices of
// RA * RB MFMAs.  The fragments of a slice are read, for the next step, among the MFMAs of the slice behind it, into the
// registers that slice has just freed, so one set of them is enough; the loads of step s + NS - 1 go out among slices 1 to 3,
// into the stage that step s - 1 has left.  One barrier a step, between slices 0 and 1: before it a wavefront has seen its own
// loads of step s + 1 (a count of younger ones may be under way), behind it that stage is there for everyone.
// Registers: fragments in v[144:223], addresses of a slice's reads in v142 / v143; s46 and s50 are this wavefront's places for
// loads of A and B in the stage being requested, s47 counts steps, s48 is the stage being read, s[44:45] a step's bytes.
#pragma once

#define SR_A_0_0 "v[144:147]"
#define SR_A_0_1 "v[148:151]"
#define SR_A_0_2 "v[152:155]"
#define SR_A_0_3 "v[156:159]"
#define SR_A_1_0 "v[160:163]"
#define SR_A_1_1 "v[164:167]"
#define SR_A_1_2 "v[168:171]"
#define SR_A_1_3 "v[172:175]"
#define SR_A_2_0 "v[176:179]"
#define SR_A_2_1 "v[180:183]"
#define SR_A_2_2 "v[184:187]"
#define SR_A_2_3 "v[188:191]"
#define SR_B_0_0 "v[192:195]"
#define SR_B_0_1 "v[196:199]"
#define SR_B_0_2 "v[200:203]"
#define SR_B_0_3 "v[204:207]"
#define SR_B_1_0 "v[208:211]"
#define SR_B_1_1 "v[212:215]"
#define SR_B_1_2 "v[216:219]"
#define SR_B_1_3 "v[220:223]"
#define SR_RDA(i, k) "ds_read_b128 " SR_A_##i##_##k ", v142 offset:" #i "*4096\n\t"
#define SR_RDB(j, k) "ds_read_b128 " SR_B_##j##_##k ", v143 offset:" #j "*4096\n\t"
#define SR_FROM(k) "v_add_u32 v142, s48, %[ra" #k "]\n\tv_add_u32 v143, s48, %[rb" #k "]\n\t"
#define SR_P(i, j, k) "v_mfma_f32_32x32x16_bf16 %[c" #i #j "], " SR_A_##i##_##k ", " SR_B_##j##_##k ", %[c" #i #j "]\n\t"
#define SR_W(n) "s_waitcnt lgkmcnt(" #n ")\n\t"
#define SR_SYNC(v) "s_waitcnt vmcnt(" #v ")\n\ts_barrier\n\t"
// a load: its place first (an MFMA comes between), then the load and its pointer's step
#define SR_MA(i) "s_add_u32 m0, s46, " #i "*1024\n\t"
#define SR_MB(i) "s_add_u32 m0, s50, " #i "*1024\n\t"
#define SR_LA(i) "global_load_lds_dwordx4 %[ga" #i "], off\n\tv_lshl_add_u64 %[ga" #i "], %[ga" #i "], 0, s[44:45]\n\t"
#define SR_LB(i) "global_load_lds_dwordx4 %[gb" #i "], off\n\tv_lshl_add_u64 %[gb" #i "], %[gb" #i "], 0, s[44:45]\n\t"
#define SR_NEXT_READ "s_add_u32 s48, s48, %[stage]\n\ts_cmp_eq_u32 s48, %[all]\n\ts_cselect_b32 s48, 0, s48\n\t"
// bytes from the step being requested to the next (KOrder; a product of up to 128 rows is on 128 x 128, so the others go straight on)
#define SR_STEP_SIZE "s_sub_u32 s51, s51, 1\n\ts_cmp_eq_u32 s51, 0\n\ts_cselect_b32 s44, %[back], 128\n\ts_cselect_b32 s45, -1, 0\n\t"
#define SR_STEP_22 SR_STEP_SIZE
#define SR_STEP_32 ""
#define SR_FIRST_STEP_22 "s_mov_b32 s51, %[wrap]\n\t" SR_STEP_SIZE
#define SR_FIRST_STEP_32 "s_movk_i32 s44, 128\n\ts_mov_b32 s45, 0\n\t"
#define SR_NEXT_LOAD                                                                                                     \
  "s_add_u32 s46, s46, %[stage]\n\ts_cmp_eq_u32 s46, %[limit]\n\ts_cselect_b32 s46, %[la], s46\n\ts_add_u32 s50, s46, " \
  "%[ab]\n\t"
#define SR_S22(k, e0, e1, e2, e3) SR_P(0, 0, k) e0 SR_P(0, 1, k) e1 SR_P(1, 0, k) e2 SR_P(1, 1, k) e3
#define SR_S32(k, e0, e1, e2, e3, e4, e5) SR_S22(k, e0, e1, e2, e3) SR_P(2, 0, k) e4 SR_P(2, 1, k) e5
#define SR_ON(x) x
#define SR_OFF(x) ""
// 128 x 128 (four reads a slice, 4 + 4 loads a step) and 192 x 128 (five, 6 + 4).  D: loads on or off
#define SR_HEAD_22 SR_W(8) SR_FROM(3) SR_S22(0, SR_RDA(0, 3), SR_RDA(1, 3), SR_RDB(0, 3), SR_RDB(1, 3)) SR_NEXT_READ
#define SR_REST_22(D, v)                                                                                                       \
  SR_SYNC(v)                                                                                                                      \
  SR_W(8) SR_FROM(0) SR_S22(1, SR_RDA(0, 0) D(SR_MA(0)), SR_RDA(1, 0) D(SR_LA(0) SR_MA(1)), SR_RDB(0, 0) D(SR_LA(1) SR_MA(2)), \
                            SR_RDB(1, 0) D(SR_LA(2)))                                                                             \
  SR_W(8) SR_FROM(1) SR_S22(2, SR_RDA(0, 1) D(SR_MA(3)), SR_RDA(1, 1) D(SR_LA(3) SR_MB(0)), SR_RDB(0, 1) D(SR_LB(0) SR_MB(1)), \
                            SR_RDB(1, 1) D(SR_LB(1)))                                                                             \
  SR_W(8) SR_FROM(2) SR_S22(3, SR_RDA(0, 2) D(SR_MB(2)), SR_RDA(1, 2) D(SR_LB(2) SR_MB(3)), SR_RDB(0, 2) D(SR_LB(3)), SR_RDB(1, 2))
#define SR_LAST_22 \
  SR_W(8) SR_S22(1, "", "", "", "") SR_W(4) SR_S22(2, "", "", "", "") SR_W(0) SR_S22(3, "", "", "", "")
#define SR_FIRST_22                                                                                               \
  SR_FROM(0) SR_RDA(0, 0) SR_RDA(1, 0) SR_RDB(0, 0) SR_RDB(1, 0) SR_FROM(1) SR_RDA(0, 1) SR_RDA(1, 1) SR_RDB(0, 1) \
  SR_RDB(1, 1) SR_FROM(2) SR_RDA(0, 2) SR_RDA(1, 2) SR_RDB(0, 2) SR_RDB(1, 2)
#define SR_HEAD_32 \
  SR_W(10) SR_FROM(3) SR_S32(0, SR_RDA(0, 3), SR_RDA(1, 3), SR_RDA(2, 3), SR_RDB(0, 3), SR_RDB(1, 3), "") SR_NEXT_READ
#define SR_REST_32(D, v)                                                                                                         \
  SR_SYNC(v)                                                                                                                        \
  SR_W(10) SR_FROM(0) SR_S32(1, SR_RDA(0, 0) D(SR_MA(0)), SR_RDA(1, 0) D(SR_LA(0) SR_MA(1)), SR_RDA(2, 0) D(SR_LA(1) SR_MA(2)),  \
                             SR_RDB(0, 0) D(SR_LA(2) SR_MA(3)), SR_RDB(1, 0) D(SR_LA(3)), "")                                       \
  SR_W(10) SR_FROM(1) SR_S32(2, SR_RDA(0, 1) D(SR_MA(4)), SR_RDA(1, 1) D(SR_LA(4) SR_MA(5)), SR_RDA(2, 1) D(SR_LA(5) SR_MB(0)),  \
                             SR_RDB(0, 1) D(SR_LB(0)), SR_RDB(1, 1), "")                                                            \
  SR_W(10) SR_FROM(2) SR_S32(3, SR_RDA(0, 2) D(SR_MB(1)), SR_RDA(1, 2) D(SR_LB(1) SR_MB(2)), SR_RDA(2, 2) D(SR_LB(2) SR_MB(3)),  \
                             SR_RDB(0, 2) D(SR_LB(3)), SR_RDB(1, 2), "")
#define SR_LAST_32                                    \
  SR_W(10) SR_S32(1, "", "", "", "", "", "")          \
  SR_W(5) SR_S32(2, "", "", "", "", "", "") SR_W(0) SR_S32(3, "", "", "", "", "", "")
#define SR_FIRST_32                                                                                                           \
  SR_FROM(0) SR_RDA(0, 0) SR_RDA(1, 0) SR_RDA(2, 0) SR_RDB(0, 0) SR_RDB(1, 0) SR_FROM(1) SR_RDA(0, 1) SR_RDA(1, 1) SR_RDA(2, 1) \
  SR_RDB(0, 1) SR_RDB(1, 1) SR_FROM(2) SR_RDA(0, 2) SR_RDA(1, 2) SR_RDA(2, 2) SR_RDB(0, 2) SR_RDB(1, 2)
// n >= NS - 1 steps, NS - 1 of them requested already: v0 counts the loads of NS - 2 steps, v those of NS - 3; TAIL: the NS - 2
// steps before the last, which request nothing
#define SR_LOOP(R, v0, v, TAIL)                                                                                             \
  SR_FIRST_STEP_##R "s_mov_b32 s46, %[first]\n\ts_add_u32 s50, s46, %[ab]\n\ts_mov_b32 s48, 0\n\t"    \
  "s_sub_u32 s47, %[n], %[held]\n\t" SR_SYNC(v0) SR_FIRST_##R "s_cmp_eq_u32 s47, 0\n\ts_cbranch_scc1 2f\n\t"                   \
  "1:\n\t" SR_HEAD_##R SR_REST_##R(SR_ON, v) SR_NEXT_LOAD SR_STEP_##R                                                                \
  "s_sub_u32 s47, s47, 1\n\ts_cmp_lg_u32 s47, 0\n\ts_cbranch_scc1 1b\n\t"                                                      \
  "2:\n\t" TAIL SR_HEAD_##R SR_LAST_##R "s_nop 15\n\ts_nop 7\n\t"
#define SR_QUIET(R, v) SR_HEAD_##R SR_REST_##R(SR_OFF, v)
#define SR_LOOP_22 SR_LOOP(22, 24, 16, SR_QUIET(22, 16) SR_QUIET(22, 8) SR_QUIET(22, 0))
#define SR_LOOP_32 SR_LOOP(32, 20, 10, SR_QUIET(32, 10) SR_QUIET(32, 0))
#define SR_V10(d) "v" #d "0", "v" #d "1", "v" #d "2", "v" #d "3", "v" #d "4", "v" #d "5", "v" #d "6", "v" #d "7", "v" #d "8", "v" #d "9"
#define SR_CLOBBERS                                                                                                            \
  "v142", "v143", "v144", "v145", "v146", "v147", "v148", "v149", SR_V10(15), SR_V10(16), SR_V10(17), SR_V10(18), SR_V10(19),  \
      SR_V10(20), SR_V10(21), "v220", "v221", "v222", "v223", "s44", "s45", "s46", "s47", "s48", "s50", "s51", "m0", "scc", "memory"
