/*
 * amd_matmul_plan.h -- what the host's rules in libamd_matmul.so pick for a launch, without one: no device and no handle is
 * needed, nothing is launched or kept.  For tools that name a launch's kernel and for tests of the rules; no counterpart in
 * the reference.  Sizes and operand conventions are those of amd_matmul.h; cu_count: compute units of the device (256).
 */
#ifndef AMD_MATMUL_PLAN_H
#define AMD_MATMUL_PLAN_H

#include "dataflow_amd.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Tiles of an aligned problem that is not split along K: the direct kernel's, or BIG: the persistent kernels */
enum { AMD_MATMUL_TILE_64x32, AMD_MATMUL_TILE_64x64, AMD_MATMUL_TILE_64x128, AMD_MATMUL_TILE_128x128, AMD_MATMUL_TILE_128x128_PAIR, AMD_MATMUL_TILE_BIG };
/* has_c: D also takes C (beta is not 0) */
int amd_matmul_planned_tile(int M, int K, int N, int has_c, int cu_count);

/* Parts into which the matmul op splits K of an aligned problem with a workspace of that size (1: not split) */
int amd_matmul_planned_splits(int to_trans_a, int to_trans_b, int M, int K, int N, int has_c, uint64_t workspace_bytes, int cu_count);

/* Tilings of the token rows that a ragged-N launch without C goes out on where it runs on the persistent kernels: the sum of
 * one or two of these bits (D 16-byte aligned); with two, the device picks one from the group sizes */
enum { AMD_MATMUL_ROWS_288 = 1, AMD_MATMUL_ROWS_384 = 2, AMD_MATMUL_ROWS_224 = 4, AMD_MATMUL_ROWS_192 = 8 };
int amd_matmul_planned_tilings(int M, int K, int N, int num_groups, int cu_count);

/* 1: one problem without C and with to_trans_b == 0, not split along K, runs on tiles of 256 x 384, 0: on 256 x 256 or a smaller tile */
int amd_matmul_planned_wide(int M, int K, int N, int cu_count);

/* 1: two k-major operands, that is to_trans_a == 0 and to_trans_b == 1, run on the four-wave kernel that takes them in slices (FOUR_WAVES_384 of
 * amd_matmul.h), 0: on the eight-wave kernel or on a smaller tile.  num_groups: of a ragged-K launch, K then being the rows of all groups together; 0:
 * one problem, not split along K.  Aligned operands, C and D; a kernel named with amd_matmul_select_kernel counts. */
int amd_matmul_planned_sliced(int M, int K, int N, int num_groups, int has_c, int cu_count);

#ifdef __cplusplus
}
#endif

#endif
