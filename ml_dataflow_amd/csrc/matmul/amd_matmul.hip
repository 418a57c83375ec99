/*
 * amd_matmul.hip -- bf16 GEMM family for gfx950 behind the reference's external matmul op.
 *
 *   amd_matmul           the "default_matmul" op: replaces cublas_matmul
 *                        (backends/nvidia/src/ops/src/external/matmul_helper/src/matmul_helper.c:774-946)
 *   amd_grouped_matmul   one launch for all experts of a ragged group (an addition: the reference loops
 *                        over experts on the host, dataflow_transformer.c:2848-2940, 3460-3641, 4101-4148)
 *
 * Semantics (column-major BLAS view, matmul_helper.c:345-425):  D[M,N] = alpha*op(A)[M,K]*op(B)[K,N] + beta*C.
 * Read as row-major arrays: A is [M][K] (to_trans_a=1) or [K][M]; B is [N][K] (to_trans_b=0) or [K][N];
 * C and D are [N][M].  bf16 in and out, fp32 accumulation on the matrix cores, one rounding to bf16.
 *
 * The kernels live in gemm_kernel.h (eight waves), gemm_w4_kernel.h (four waves) and gemm_typed_kernel.h (element
 * types beside all-bf16); this file decodes the op arguments, checks them on the host and picks a kernel: the
 * direct-to-LDS kernels when every operand is 16-byte aligned with a contiguous extent that is a multiple of 8
 * elements, or a workspace holds padded copies of those that are not (pad_operands), the register-staged kernel otherwise; large
 * ragged-N launches without a C operand run on one of four tilings (ragged_n_tilings).
 */
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "dataflow_amd.h"
#include "dataflow_amd_ops.h"
#include "amd_matmul.h"
#include "amd_matmul_plan.h"
#include "gemm_kernel.h"
#include "gemm_w4_kernel.h"
#include "gemm_typed_kernel.h"
#include "route_kernel.h"

/* ------------------------------------------------------------------ host side */

struct MatmulExtra {
	int cu_count;
	int lds_optin;
};

/* Scratch of amd_matmul_no_alloc: the fp32 partial sums of a split along K, which amd_matmul keeps in the caller's
 * workspace.  64 MiB hold every split that plan_split makes on 256 compute units (four work-groups each, 64 KiB of sums per work-group), so
 * the call splits as the op does with any workspace that is large enough.  A file-scope device array: every GPU the library runs on holds
 * its own copy at its own address until the process ends.  In host code the name is only a handle for hipGetSymbolAddress; the address of
 * each device's copy is looked up once per device in amd_matmul_init and everything below uses that pointer. */
#define AMD_MATMUL_SCRATCH_BYTES (64u << 20)
#define AMD_MATMUL_MAX_DEVICES 64
static __device__ __align__(256) unsigned char scratch[AMD_MATMUL_SCRATCH_BYTES];
static void * scratch_of_device[AMD_MATMUL_MAX_DEVICES];

static int check_launch(void) {
	hipError_t e = hipGetLastError();
	if (e != hipSuccess) {
		fprintf(stderr, "Error: gemm kernel launch failed: %s...\n", hipGetErrorString(e));
		return -1;
	}
	return 0;
}

/* register-staged kernel: dynamic LDS, two stages */
template <int BM, int BN, int WAVES_M, int WAVES_N, bool PK, bool QK, int MODE>
static int launch_staged(const GemmParams & p, long grid, hipStream_t stream) {
	constexpr int threads = WAVES_M * WAVES_N * 64;
	constexpr size_t lds_bytes = 2 * (BM + BN) * BK * sizeof(bf16_t);
	auto kernel = gemm_bf16_staged_kernel<BM, BN, WAVES_M, WAVES_N, PK, QK, MODE>;
	static bool attr_done = false;
	if (lds_bytes > 65536 && !attr_done) {
		hipError_t e = hipFuncSetAttribute((const void *) kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds_bytes);
		if (e != hipSuccess) {
			fprintf(stderr, "Error: could not raise dynamic LDS limit to %zu bytes: %s...\n", lds_bytes, hipGetErrorString(e));
			return -1;
		}
		attr_done = true;
	}
	hipLaunchKernelGGL(kernel, dim3((unsigned int) grid), dim3(threads), lds_bytes, stream, p);
	return check_launch();
}

/* direct-to-LDS kernel: static LDS */
template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, bool PK, bool QK, int MODE, int GATHER = GATHER_NONE, bool SWIGLU = false, bool ONCE = false>
static int launch_direct_tile(const GemmParams & p, long grid, hipStream_t stream) {
	constexpr int threads = WAVES_M * WAVES_N * 64;
	hipLaunchKernelGGL((gemm_bf16_direct_kernel<BM, BN, WAVES_M, WAVES_N, PK, QK, MODE, GATHER, STAGES, SWIGLU, ONCE>), dim3((unsigned int) ((grid + 7) & ~7L)), dim3(threads), 0, stream, p);
	return check_launch();
}

static long tiles_of(long extent, long tile) { return (extent + tile - 1) / tile; }

/* The work-group tiles of the direct kernel, and which of them a problem runs on (BIG: the persistent kernels instead).
 *
 * A problem with few tiles takes as long as one work-group needs for its k-tiles, and what a k-tile costs one work-group
 * grows much more slowly than its tile: measured on problems of 88 to 512 tiles, K of 1024-4096 (microseconds per k-tile
 * and work-group with the compute units sharing the load) 64 x 32: 0.20-0.28, 64 x 64: 0.21-0.31, 64 x 128: 0.29-0.44,
 * 128 x 128 with three stages and eight waves: 0.47-0.66, two of them with two stages on one compute unit: 0.50 each (0.56
 * alone), the persistent 256 x 256: 1.1-1.4.  So the cheapest tile is the one with the least (rounds of tiles over the
 * compute units) x (cost of a k-tile), small tiles while they still fit one round and larger ones behind that.  1408 x
 * 2048 x 256 takes 10 us on 64 x 64 tiles (29 on 128 x 128 with one k-tile in flight, which this replaced), 4096 x 4096 x
 * 512 31 us on 64 x 128 (55), 4096 x 4096 x 2048 66 us on pairs of 128 x 128 (92 on the persistent kernel).  The
 * costs are in hundredths of a microsecond.  A single problem's rounds are charged what writing their tiles of D takes (store), the
 * persistent kernel's also the read of C (the other kernels' is hidden behind their neighbours' k-tiles), and the launch of that
 * kernel 2 us; a partial last round of it 60 % of a whole one plus the rest by its share (270 tiles of 256 x 256, 3840 x 3328 x 4582,
 * take 104 us, in pairs of 128 x 128 146).  Without the bytes of C and D a K of one or two k-tiles went to whatever tile has the fewest
 * rounds: the router's input gradient, 2048 x 32 x 3001 with C, to 96 work-groups of 256 x 256 in 13.3 us, where pairs of 128 x 128 take 9.1
 * (4096 x 64 x 8192 31.4 and 27.5, 4096 x 64 x 65536 194 and 271, the other way round).  Over 544 products of 64-4096 columns,
 * 16-65536 tokens, K 8-16384 the choice is 0.8 % behind the best of all tiles, at a flat half a microsecond a round it was 3.5 %.
 * BIG's cost and its read of C are those of the eight-wave kernel, also where the problem then runs on 256 x 384 tiles or on the sliced kernel, which
 * reads C under the multiplies (3776 x 1000 x 4032 with C 38 us on eight waves, 34 on that one): there the choice leans to the smaller tiles.
 * Ragged launches have no term per tile: with caches that hold nothing of the operands the choice is 0.0 % behind the best of all
 * tiles over 60 ragged-K launches of 4-1500 rows per group, and 2.4 % over 120 ragged-N launches of 4-400. */
enum { TILE_64x32 = AMD_MATMUL_TILE_64x32, TILE_64x64 = AMD_MATMUL_TILE_64x64, TILE_64x128 = AMD_MATMUL_TILE_64x128, TILE_128x128 = AMD_MATMUL_TILE_128x128,
	TILE_128x128_PAIR = AMD_MATMUL_TILE_128x128_PAIR, TILE_BIG = AMD_MATMUL_TILE_BIG, NUM_TILES };
static const struct { int bm, bn, cost, store; } TILES[NUM_TILES] = {{64, 32, 21, 40}, {64, 64, 25, 60}, {64, 128, 36, 90}, {128, 128, 58, 110}, {128, 128, 50, 110}, {256, 256, 130, 100}};
#define TILE_BIG_READ_C_COST 320
#define TILE_BIG_LAUNCH_COST 200
#define TILE_PAIR_COST_ALONE 62      /* of a k-tile of the pair's tile where it has the compute unit to itself, or its lines come from HBM */

/* tiles of the launch for tile `which`.  Ragged N: the group sizes are on the device; a group of the mean size has on
 * average half a tile more than its rows fill, and at least one */
static long tiles_in_launch(int which, int mode, const GemmParams & p) {
	const long tm = tiles_of(p.M, TILES[which].bm), bn = TILES[which].bn;
	if (mode == MODE_SINGLE) {
		return tm * tiles_of(p.N, bn);
	}
	if (mode == MODE_RAGGED_K) {
		return tm * tiles_of(p.N, bn) * p.num_groups;
	}
	const long filled = p.N < p.num_groups ? p.N : p.num_groups;
	const long tn = p.N / bn + filled / 2;
	return tm * (tn > filled ? tn : filled);
}

/* upper bound for the grid */
static long grid_of(int which, int mode, const GemmParams & p) {
	if (mode != MODE_RAGGED_N) {
		return tiles_in_launch(which, mode, p);
	}
	return tiles_of(p.M, TILES[which].bm) * ((long) p.N / TILES[which].bn + (p.N < p.num_groups ? p.N : p.num_groups));
}

static long tile_cost(int which, int mode, const GemmParams & p, long cu_count) {
	const long tiles = tiles_in_launch(which, mode, p);
	const bool alone = which == TILE_128x128_PAIR && (tiles <= cu_count || mode == MODE_RAGGED_N);
	const long cost = alone ? TILE_PAIR_COST_ALONE : TILES[which].cost;
	if (mode != MODE_SINGLE) {
		return tiles_of(tiles, cu_count) * cost;
	}
	const bool big = which == TILE_BIG;
	const long round = tiles_of(p.K, BK) * cost + TILES[which].store + (big && p.C ? TILE_BIG_READ_C_COST : 0);
	const long full = tiles / cu_count, left = tiles % cu_count;
	if (big && full > 0) {
		return TILE_BIG_LAUNCH_COST + full * round + (left ? round * (3 * cu_count + 2 * left) / (5 * cu_count) : 0);
	}
	return (big ? TILE_BIG_LAUNCH_COST : 0) + (full + (left ? 1 : 0)) * round;
}

/* the cheapest tile; `cost`: what it costs (single problems: hundredths of a microsecond) */
static int choose_tile(int mode, const GemmParams & p, long cu_count, bool persistent_ok = true, long * cost = NULL) {
	const bool big_ok = persistent_ok && p.M >= 256 && (mode == MODE_RAGGED_N || p.N >= 256);
	int best = TILE_64x32;
	long best_cost = 0;
	for (int which = 0; which < NUM_TILES; which++) {
		if (which == TILE_BIG && !big_ok) {
			continue;
		}
		const long c = tile_cost(which, mode, p, cu_count);
		if (which == 0 || c < best_cost) {
			best = which;
			best_cost = c;
		}
	}
	if (cost) {
		*cost = best_cost;
	}
	return best;
}

extern "C" int amd_matmul_planned_tile(int M, int K, int N, int has_c, int cu_count) {
	GemmParams p;
	memset(&p, 0, sizeof(p));
	p.M = M; p.K = K; p.N = N;
	p.C = has_c ? (const bf16_t *) scratch_of_device : NULL;      /* any address: the rules look at whether there is one */
	return choose_tile(MODE_SINGLE, p, cu_count);
}

/* Few rows per group: a launch is bound by the weights of the groups that have any, and where these have one tile of rows each line of the
 * weights is read by one work-group.  Such lines are loaded non-temporally: rows of 8 KiB, 128 bytes at a time, stream at 6.0-6.6 TB/s
 * so and at 5.3 with plain loads (whole arrays in order: 7.1 and 6.25).  Forwards, us: 16 tokens, 64 experts, top 8, 4096 x 1024 258 -> 229; 50 tokens, 42 experts,
 * 3584 x 1600 287 -> 253; 4 tokens, 43 experts, 1792 x 1216 61 -> 55.  A group with more tiles of rows keeps plain loads (712 tokens dealt to 35 experts by a Zipf
 * router, non-temporal throughout: 104 -> 118), and so do launches whose weights are few enough to be found in the 256 MiB memory-side cache
 * (7 tokens, 55 experts, top 2, 512 x 1472, over three sets of weights: 32.4 -> 33.7; over fourteen 37.8 -> 34.5).
 * The line is drawn for a program whose layers together have more weights than the cache holds.  Forwards of 16 tokens over many layers and over one
 * in a loop, us: 16 experts, 2048 x 1024 (192 MiB in all, 128 in the launch) 61.4 -> 55.0 and 46.0 -> 52.9, 24 (288 and 192) 75.9 -> 68.3 and 68.6 -> 67.2, 32 (384 and 256)
 * 89.7 -> 81.0 and 89.2 -> 79.4; 32 experts, 1024 x 1024 52.4 -> 47.2 and 42.9 -> 45.0; 64 tokens, 32, 2048 x 768 79.5 -> 72.2 and 67.3 -> 72.1.  So a single layer of 72 to
 * some 290 MiB that is run again and again loses 5-15 % by it, and from there on nothing is found in the cache either way.
 * It is another instance of the kernel, with a copy of the loop for each kind of load: a choice between two copies that no group of a launch needs cost it
 * about 1 % (900 tokens, 8 experts, top 2, 1024 x 1024 51.8 -> 52.4, 1624, 23, 2, 3328 x 512 137.7 -> 138.8).  So it is taken only where the mean group has no
 * more rows than a tile, and no more than 96: over sets of weights beyond the cache, even and Zipf routers, 27 drawn forwards with fewer rows 0.88-1.00 of the time without (two of 14
 * and 24 tokens, whose few experts stay in the cache, 1.05), 17 with more than a tile 1.00; between 96 and 128 rows it is 0.96-1.03 (1259 tokens, 61 experts, top 5,
 * 3712 x 1152 416 -> 428, 1540, 16, 1, 1792 x 1280 103 -> 99).  Training steps of one layer, whose backward finds in the cache what plain loads of the
 * forward leave there: 36 drawn ones 0.93-1.03, 0.972 in the mean; above 1.01 only where weights of 290-450 MiB meet 64-110 rows an expert (608 tokens, 41, 5,
 * 2304 x 832 450 -> 460). */
#define STREAM_WEIGHTS_BYTES (48u << 20)
#define STREAM_WEIGHTS_MOST_ROWS 96
static bool streams_weights(const GemmParams & p, int tile_rows) {
	const long filled = p.N < p.num_groups ? p.N : p.num_groups, rows = tile_rows < STREAM_WEIGHTS_MOST_ROWS ? tile_rows : STREAM_WEIGHTS_MOST_ROWS;
	return p.N <= rows * filled && (uint64_t) filled * (uint64_t) p.M * (uint64_t) p.K * 2u > STREAM_WEIGHTS_BYTES;
}

/* one tile of the direct kernel, with or without them */
template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, bool PK, bool QK, int MODE, int GATHER, bool SWIGLU>
static int launch_direct_either(const GemmParams & p, long grid, hipStream_t stream) {
	if constexpr (MODE == MODE_RAGGED_N) {
		if (streams_weights(p, BN)) {
			return launch_direct_tile<BM, BN, WAVES_M, WAVES_N, STAGES, PK, QK, MODE, GATHER, SWIGLU, true>(p, grid, stream);
		}
	}
	return launch_direct_tile<BM, BN, WAVES_M, WAVES_N, STAGES, PK, QK, MODE, GATHER, SWIGLU>(p, grid, stream);
}

/* the direct kernel on one of its tiles */
template <bool PK, bool QK, int MODE, int GATHER = GATHER_NONE, bool SWIGLU = false>
static int launch_direct(const GemmParams & p, int which, hipStream_t stream, int problems = 1) {
	const long grid = grid_of(which, MODE, p) * problems;
	switch (which) {
		case TILE_64x32: return launch_direct_either<64, 32, 2, 2, 4, PK, QK, MODE, GATHER, SWIGLU>(p, grid, stream);
		case TILE_64x64: return launch_direct_either<64, 64, 2, 2, 4, PK, QK, MODE, GATHER, SWIGLU>(p, grid, stream);
		case TILE_64x128: return launch_direct_either<64, 128, 2, 2, 3, PK, QK, MODE, GATHER, SWIGLU>(p, grid, stream);
		case TILE_128x128: return launch_direct_either<128, 128, 4, 2, 3, PK, QK, MODE, GATHER, SWIGLU>(p, grid, stream);
		default: return launch_direct_either<128, 128, 4, 2, 2, PK, QK, MODE, GATHER, SWIGLU>(p, grid, stream);
	}
}

/* The partial products of a split along K, on one of the direct kernel's tiles with more than two stages */
template <bool PK, bool QK>
static int launch_split_layout(const GemmParams & p, int tile, hipStream_t stream) {
	const long grid = tiles_in_launch(tile, MODE_SINGLE, p) * p.split_k;
	switch (tile) {
		case TILE_64x32: return launch_direct_tile<64, 32, 2, 2, 4, PK, QK, MODE_SINGLE>(p, grid, stream);
		case TILE_64x64: return launch_direct_tile<64, 64, 2, 2, 4, PK, QK, MODE_SINGLE>(p, grid, stream);
		case TILE_64x128: return launch_direct_tile<64, 128, 2, 2, 3, PK, QK, MODE_SINGLE>(p, grid, stream);
		default: return launch_direct_tile<128, 128, 2, 2, 4, PK, QK, MODE_SINGLE>(p, grid, stream);
	}
}
static int launch_split(const GemmParams & p, int tile, int transa, int transb, hipStream_t stream) {
	const bool pk = !transa;
	const bool qk = transb != 0;
	if (!pk && !qk) { return launch_split_layout<false, false>(p, tile, stream); }
	if (pk && !qk) { return launch_split_layout<true, false>(p, tile, stream); }
	if (pk && qk) { return launch_split_layout<true, true>(p, tile, stream); }
	return launch_split_layout<false, true>(p, tile, stream);
}

/* streaming kernel: one persistent work-group per compute unit (LDS allows no more), a multiple of 8 so every die gets the same share */
template <int BM, int BN, int WAVES_M, int WAVES_N, bool PK, bool QK, int MODE, int GATHER = GATHER_NONE>
static int launch_stream(const GemmParams & p, long tiles_upper_bound, long cu_count, hipStream_t stream) {
	constexpr int threads = WAVES_M * WAVES_N * 64;
	long grid = cu_count & ~7L;
	if (grid < 8) {
		grid = 8;
	}
	const long need = (tiles_upper_bound + 7) & ~7L;
	if (need < grid) {
		grid = need;
	}
	hipLaunchKernelGGL((gemm_bf16_stream_kernel<BM, BN, WAVES_M, WAVES_N, PK, QK, MODE, GATHER>), dim3((unsigned int) grid), dim3(threads), 0, stream, p);
	return check_launch();
}

/* four-wave kernel (gemm_w4_kernel.h): same grid rule as the streaming kernel, 256 threads */
template <bool PK, int MODE, int GATHER = GATHER_NONE>
static int launch_w4(const GemmParams & p, long tiles_upper_bound, long cu_count, hipStream_t stream) {
	long grid = cu_count & ~7L;
	if (grid < 8) {
		grid = 8;
	}
	const long need = (tiles_upper_bound + 7) & ~7L;
	if (need < grid) {
		grid = need;
	}
	hipLaunchKernelGGL((gemm_bf16_w4_kernel<PK, MODE, GATHER>), dim3((unsigned int) grid), dim3(256), 0, stream, p);
	return check_launch();
}

/* the four symmetric waves with the 256 x 384 tile (gemm_w4_kernel.h): same grid rule */
template <bool PK, int MODE, int GATHER = GATHER_NONE>
static int launch_w4d(const GemmParams & p, long tiles_upper_bound, long cu_count, hipStream_t stream) {
	long grid = cu_count & ~7L;
	if (grid < 8) {
		grid = 8;
	}
	const long need = (tiles_upper_bound + 7) & ~7L;
	if (need < grid) {
		grid = need;
	}
	hipLaunchKernelGGL((gemm_bf16_w4d_kernel<PK, MODE, GATHER>), dim3((unsigned int) grid), dim3(256), 0, stream, p);
	return check_launch();
}

/* the four waves with k-major operands in slices (gemm_w4_kernel.h): same grid rule */
template <int MODE, int GATHER = GATHER_NONE>
static int launch_w4k(const GemmParams & p, long tiles, long cu_count, hipStream_t stream) {
	long grid = cu_count & ~7L;
	if (grid < 8) {
		grid = 8;
	}
	const long need = (tiles + 7) & ~7L;
	if (need < grid) {
		grid = need;
	}
	if (p.C && p.beta != 0.0f) {
		hipLaunchKernelGGL((gemm_bf16_w4k_kernel<true, MODE, GATHER>), dim3((unsigned int) grid), dim3(256), 0, stream, p);
	} else {
		hipLaunchKernelGGL((gemm_bf16_w4k_kernel<false, MODE, GATHER>), dim3((unsigned int) grid), dim3(256), 0, stream, p);
	}
	return check_launch();
}

/* Which persistent kernel large problems run, one of AMD_MATMUL_KERNEL_* (amd_matmul.h).  Process-wide; amd_matmul_select_kernel changes it, the
 * environment variable AMD_MATMUL_KERNEL ("auto", "8", "384" or "4") sets the initial value when the op is registered. */
static int kernel_choice = AMD_MATMUL_KERNEL_DEFAULT;

extern "C" int amd_matmul_select_kernel(int which) {
	if (which != AMD_MATMUL_KERNEL_AUTO && which != AMD_MATMUL_KERNEL_EIGHT_WAVES && which != AMD_MATMUL_KERNEL_FOUR_WAVES &&
		which != AMD_MATMUL_KERNEL_FOUR_WAVES_384) {
		fprintf(stderr, "Error: amd_matmul_select_kernel: unknown kernel %d...\n", which);
		return -1;
	}
	kernel_choice = which;
	return 0;
}

/* the four-wave kernel takes whole k-tiles in pairs from k-contiguous operands, 16-byte lines of output, no C; a wave's rows of D
 * (128 at most) stay below 2 GiB (W4_NO_COLUMN) */
static bool w4_ok(const GemmParams & p) {
	return !(p.C && p.beta != 0.0f) && (p.K % 128 == 0) && p.K <= (1 << 21) &&
		   (p.M % 8 == 0) && p.M <= (1 << 22) && ((((uintptr_t) p.D) & 15) == 0);
}

/* the sliced kernel takes and leaves 16-byte pieces of rows of C and D; a wave's 128 rows of D stay below 2 GiB (W4_NO_COLUMN), a
 * slice of either operand below 4 GiB */
static bool w4k_ok(const GemmParams & p) {
	return p.M % 8 == 0 && p.N % 8 == 0 && p.M <= (1 << 22) && p.N <= (1 << 24) && p.strideD % 8 == 0 && ((((uintptr_t) p.D) & 15) == 0) &&
		   (!(p.C && p.beta != 0.0f) || (((uintptr_t) p.C) & 15) == 0);
}

/* gathered k-rows: a row that does not exist, and a lane's column behind it, lie outside a source of this size */
static bool w4k_gather_ok(const GemmParams & p) {
	return (uint64_t) p.gather_rows * (uint64_t) p.M * 2u <= 0xFFFFF000ull;
}

/* The k-rows a tile has to have, in the mean, for the sliced kernel to be the faster one.  Its tiles have at least 8 slices of 32 k-rows
 * (5 without C), and a fixed part that two waves on a SIMD hide better; what it gains, beside the loads in flight, is the read of C.
 * Time on it over time on eight waves.
 * Ragged K, the groups' sizes on the device, 36 launches of 8-60 groups, 512-4096 x 512-4096, several rounds of tiles, even rows and rows dealt by a
 * Zipf router, most of whose groups are shorter than the mean.  With C: 320 rows a group 0.985 and 1.068 (at worst 1.07 and 1.11), 384 0.982 and
 * 1.035, 448 0.976 and 1.008, 512 0.975 and 0.990 (1.02 and 1.03), 640 0.970 and 0.966.  Without: 512 0.996 and 0.978 (1.06 and 1.02), 640 0.990
 * and 0.961 (1.03 and 1.01).  In one round or less (14 launches of 150-240 tiles): with C 512 0.938 and 1.007, without 1024 1.021 and
 * 0.975, 1536 0.984 and 0.937 (1.04 and 0.98), 2048 0.930 and 0.889.
 * One problem (14 of one round, 5 of more): with C, K 256 0.91 in one round, 0.99 (1.05) in more, 512 0.88; without, in one round 512 1.04,
 * 1024 1.017, 1536 0.998 (1.013), 2048 0.988, in more 512 0.994 (1.02), 1024 0.972.  The lines lie where neither distribution loses. */
static bool w4k_pays(int mode, const GemmParams & p, long tiles, long cu_count) {
	const bool reads_c = p.C && p.beta != 0.0f, one_round = tiles <= cu_count;
	if (mode == MODE_RAGGED_K) {
		return (long) p.K >= (reads_c ? 512L : one_round ? 2048L : 640L) * p.num_groups;
	}
	return p.K >= (reads_c ? (one_round ? 256 : 512) : one_round ? 2048 : 1024);
}

/* whether two k-major operands on the 256 x 256 tile run on it: also where a caller named FOUR_WAVES_384, whose weight gradients of few rows ran
 * on eight waves before there was another kernel for them (32 groups of 64 rows, 2048 x 1408 with C, 77 us, 89 on the sliced one) */
static bool takes_sliced(int mode, const GemmParams & p, long tiles, long cu_count) {
	return (kernel_choice == AMD_MATMUL_KERNEL_AUTO || kernel_choice == AMD_MATMUL_KERNEL_FOUR_WAVES_384) && w4k_ok(p) && w4k_pays(mode, p, tiles, cu_count);
}

/* A single problem without C, whose tiles are known here: `wide` tiles of 256 x 384 against `narrow` ones of 256 x 256 on the eight-wave kernel.  A
 * round costs the bytes of its k-tiles and a part of its own, a last round that is not full, as fewer work-groups share the card's power and
 * memory, a half (wide: seven tenths) and the rest by its share.  Over 260 problems beside the 170 of the fit, M 512-8192, K 128-4096, N 1024-32768,
 * half of them such that the prices disagree, the choice was 0.1 % behind the better one, at worst 3.6 %, when a partial round of 384 went out in whole
 * tiles.  In pieces (W4DWalk) it costs less than these prices say: over 260 drawn problems, M 512-8192, K 128-4096, N 1024-32768, the choice is 0.6 %
 * behind, in 16 of them more than 3 %, each time 256 where 384 would be the faster one with a last round that is half full or less (2432 x 3712 x 20930, 2.15
 * rounds, 322 us and 281, 5184 x 384 x 6808, 1.48, 40 and 35).  Whole rounds at the prices of the ragged launches were 1.6 % behind before that. */
static bool single_wide_is_cheaper(long wide, long narrow, long k_tiles, long cu_count) {
	const long groups = (cu_count & ~7L) < 8 ? 8 : cu_count & ~7L;
	const long wide_left = wide % groups, narrow_left = narrow % groups;
	const long wide_rounds = wide / groups * 10 * groups + (wide_left ? 7 * groups + 3 * wide_left : 0);
	const long narrow_rounds = narrow / groups * 10 * groups + (narrow_left ? 5 * groups + 5 * narrow_left : 0);
	return wide_rounds * (256 + 384) * (105 * k_tiles + 250) < narrow_rounds * (256 + 256) * (100 * k_tiles + 150);
}

/* a ragged reduction's operands have their rows packed along k (or gathered): group bases are aligned where M and N are multiples of 8 */
static bool operand_direct_ok(const void * base, bool kmajor, long rows, long K, long group_stride_elems);
static bool ragged_k_direct_ok(const GemmParams & p) {
	return operand_direct_ok(p.A, true, p.M, p.K, 0) && operand_direct_ok(p.B, true, p.N, p.K, 0) && (p.strideD % 4 == 0);
}

/* whether it runs on the sliced kernel with its k-rows gathered; `tile`: of the launch */
static bool gathers_on_sliced(const GemmParams & p, bool direct, int tile, long tiles, long cu_count) {
	return direct && tile == TILE_BIG && w4k_gather_ok(p) && takes_sliced(MODE_RAGGED_K, p, tiles, cu_count);
}

/* a caller that named one of the persistent kernels gets it wherever it has enough tiles for half the compute units */
static int tile_of_launch(int mode, const GemmParams & p, long grid_big, long cu_count) {
	const bool named = kernel_choice != AMD_MATMUL_KERNEL_AUTO && p.M >= 256 && (mode == MODE_RAGGED_N ? (long) p.N / 256 * tiles_of(p.M, 256) : p.N >= 256 ? grid_big : 0) >= 128;
	return named ? TILE_BIG : choose_tile(mode, p, cu_count);
}

/* a ragged-N launch without C on one of its tilings; grid: an upper bound on the tiles */
template <bool PK, int GATHER>
static int launch_ragged_n_tiling(int tiling, const GemmParams & p, long grid, long cu_count, hipStream_t stream) {
	switch (tiling) {
		case RAGGED_N_384: return launch_w4d<PK, MODE_RAGGED_N, GATHER>(p, grid, cu_count, stream);
		case RAGGED_N_288: return launch_stream<256, 288, 4, 2, PK, false, MODE_RAGGED_N, GATHER>(p, grid, cu_count, stream);
		case RAGGED_N_224: return launch_stream<256, 224, 4, 2, PK, false, MODE_RAGGED_N, GATHER>(p, grid, cu_count, stream);
		default: return launch_stream<256, 192, 4, 2, PK, false, MODE_RAGGED_N, GATHER>(p, grid, cu_count, stream);
	}
}

/* on every tiling of `tilings` (bits) */
static int launch_ragged_n(int tilings, const GemmParams & p, bool pk, long grid, long cu_count, hipStream_t stream) {
	GemmParams q = p;
	q.candidates = (tilings & (tilings - 1)) ? tilings : 0;
	for (int tiling = RAGGED_N_TILINGS - 1; tiling >= 0; tiling--) {
		if (!((tilings >> tiling) & 1)) {
			continue;
		}
		int r;
		if (p.gather) {
			r = pk ? launch_ragged_n_tiling<true, GATHER_Q_ROWS>(tiling, q, grid, cu_count, stream)
				   : launch_ragged_n_tiling<false, GATHER_Q_ROWS>(tiling, q, grid, cu_count, stream);
		} else {
			r = pk ? launch_ragged_n_tiling<true, GATHER_NONE>(tiling, q, grid, cu_count, stream)
				   : launch_ragged_n_tiling<false, GATHER_NONE>(tiling, q, grid, cu_count, stream);
		}
		if (r) {
			return r;
		}
	}
	return 0;
}

/* Tiles of `tile_rows` rows of all groups together, for one of the distributions that a router may deal the rows in.  EVEN: a group's
 * share near-normal with the mean's root as standard deviation.  UNEVEN: shares that fall like a power (0.9) of the group's rank, the
 * largest 4.1 times the mean.  Either is seen at twelve equally likely quantiles.  ONE: 95 % of the rows in one group, the rest even.
 * spread: standard deviation of the result. */
enum { ROWS_EVEN, ROWS_UNEVEN, ROWS_IN_ONE, ROWS_DISTRIBUTIONS };
static double expected_n_tiles(const GemmParams & p, long tile_rows, int rows_dealt, double * spread) {
	static const double NORMAL[6] = {0.104, 0.319, 0.549, 0.812, 1.150, 1.732};
	static const double SHARES[12] = {4.122, 1.855, 1.223, 0.921, 0.743, 0.624, 0.540, 0.476, 0.427, 0.387, 0.354, 0.327};
	const double rows = (double) p.N / p.num_groups, deviation = sqrt(rows);
	*spread = 0.0;
	if (rows_dealt == ROWS_IN_ONE) {
		const int others = p.num_groups - 1;
		return (double) tiles_of(lrint(0.95 * p.N), tile_rows) + (others ? (double) others * tiles_of(lrint(0.05 * p.N / others), tile_rows) : 0.0);
	}
	const bool uneven = rows_dealt == ROWS_UNEVEN;
	double sum = 0.0, squares = 0.0;
	for (int i = 0; i < 12; i++) {
		const double r = rint(uneven ? rows * SHARES[i] : rows + (i & 1 ? -1.0 : 1.0) * NORMAL[i / 2] * deviation);
		const double tiles = r > 0.0 ? (double) tiles_of((long) r, tile_rows) : 0.0;
		sum += tiles;
		squares += tiles * tiles;
	}
	const double mean = sum / 12.0, variance = squares / 12.0 - mean * mean;
	*spread = variance > 0.0 && !uneven ? sqrt(variance * p.num_groups) : 0.0;
	return mean * p.num_groups;
}

/* Rounds of those tiles over the work-groups of a launch; a few tiles more or less decide over a whole round, so half a
 * standard deviation to both sides counts a quarter each */
static double expected_rounds(const GemmParams & p, long tile_rows, int rows_dealt, long groups) {
	double spread;
	const double n_tiles = expected_n_tiles(p, tile_rows, rows_dealt, &spread);
	double rounds = 0.0;
	for (int side = -1; side <= 1; side++) {
		rounds += (side ? 0.25 : 0.5) * (double) tiles_of(tiles_of(p.M, 256) * lrint(n_tiles + 0.5 * side * spread), groups);
	}
	return rounds;
}

/* expected costs of the tilings, and the cheapest by them.  No tiling is faster than the weights arrive (STREAMED_WEIGHTS: 6 TB/s).
 * 384 is never the cheapest where its kernel does not apply, whatever `cost` says of it.  `second`: for uneven rows beside another tiling, see
 * ragged_n_tilings. */
#define WIDE_TILE_COST_SECOND(rounds, k_tiles) ((rounds) * (256 + 384) * (103 * (k_tiles) + 160))
#define STREAMED_WEIGHTS(bytes) ((bytes) / 200)
static double larger(double a, double b) { return a > b ? a : b; }
static int cheapest_tiling(const GemmParams & p, long groups, bool four_ok, int rows_dealt, bool second, double cost[RAGGED_N_TILINGS]) {
	const long k_tiles = tiles_of(p.K, BK);
	const double narrow = expected_rounds(p, 288, rows_dealt, groups), wide = expected_rounds(p, 384, rows_dealt, groups);
	const double streamed = STREAMED_WEIGHTS((double) p.num_groups * p.M * p.K * 2.0);
	const double surcharge = second ? larger(WIDE_TILE_COST_SECOND(wide, k_tiles) - WIDE_TILE_COST(wide, k_tiles), 0.0) : 0.0;
	int best = four_ok && surcharge + WIDE_TILE_COST(wide, k_tiles) < NARROW_TILE_COST(narrow, k_tiles) ? RAGGED_N_384 : RAGGED_N_288;
	cost[RAGGED_N_288] = larger(NARROW_TILE_COST(narrow, k_tiles), streamed);
	cost[RAGGED_N_384] = larger(surcharge + WIDE_TILE_COST(wide, k_tiles), streamed);
	for (int tiling = RAGGED_N_224; tiling <= RAGGED_N_192; tiling++) {
		const long rows = ragged_n_rows(tiling);
		cost[tiling] = larger(FINER_TILE_COST(expected_rounds(p, rows, rows_dealt, groups), rows, k_tiles), streamed);
		if (cost[tiling] < cost[best]) {
			best = tiling;
		}
	}
	return best;
}

/* The tilings a ragged-N launch without C goes out on, as bits: the cheapest for the group sizes that an even router gives, and a
 * second one where that one costs 5 % and 4 us more than the cheapest with UNEVEN group sizes, or 10 % and 15 us more with nearly all
 * rows IN_ONE group: of the others the one that leaves the smaller of the worst cases.  The sizes are on the device, whose
 * work-groups then agree on one of the two from the real sizes (ragged_n_choice).  A launch that loses costs 3 us, so both
 * go out only there.  Over 310 launches of the layer's kind (8-64 experts, 30-9000 rows each, K 512-4096) with even groups one launch on
 * the expected tiling took 1.9 % longer than the best of all tilings; up to three launches, among them 288 always,
 * took 4.7 %.  A first training step of 3001 tokens, 32 experts, dim 2048 934 -> 905 us, a forward of 8192 tokens 635 -> 632, one with
 * a Zipf router, whose launches take a second tiling, unchanged.  Over 341 launches whose rows lie in one, two or four of 8-64 experts to 95 % or are dealt by Zipf routers, this
 * rule was 3.4 % behind the best, without the second list 4.8 %, up to three launches 6.8 %; 17 / 41 of them were more than 3 % slower
 * than those three launches and 4 / 27 more than 8 % (1024 x 3072, 41 groups, 6205 of 6478 rows in one: 90 / 136 us, on 288 alone 87).
 * All these with tiles of 384 that took as long as full ones.  With that kernel's short tiles and pieces, which the prices do not know, over 212 launches
 * of the same ranges that reach these kernels: even rows 2.7 % behind the best tiling (at worst 18), Zipf routers 2.1 (21), 95 % in one group 2.6 (22),
 * nearly always for another tiling where 384 is the faster one by now (44 groups of 236 rows, 1024 x 3968: 130 us on 288, 110 on 384); 384
 * throughout 2.4, 2.1 and 2.3 (39, 55 and 28).
 * As a second tiling beside another one 384 is charged 4 to 8 % more from 1024 k on (its price before its epilogue was generated): at its own
 * price the up-projections of 32 groups of 512 rows, 1408 x 2048, went out on two tilings, and a grouped training step of 4096 tokens took 1405 us
 * instead of 1389.  Where 384 is the first, UNEVEN compares at its own price: 18 launches to which the surcharge added 288 take, rows
 * dealt by a Zipf router, 3 % less on 384 alone (3648 x 1792, 61 groups, 22868 rows: 385 us on both, 288 chosen, 366; 17 launches more, to which
 * neither adds it, 3-12 % less on 384 than on 288).  IN_ONE charges it always: there the narrower tile is the better one by up to
 * 45 % (2176 x 896, 26 groups, 7056 rows: 53 us with 224, 71 without). */
#define SECOND_TILING_MARGIN 121000          /* 4 us */
#define IN_ONE_TILING_MARGIN 454000          /* 15 us */
static int ragged_n_tilings(const GemmParams & p, long cu_count, bool four_ok) {
	static const struct { double share; double margin; } SECOND[ROWS_DISTRIBUTIONS] = {{0.0, 0.0}, {1.05, SECOND_TILING_MARGIN}, {1.10, IN_ONE_TILING_MARGIN}};
	long groups = cu_count & ~7L;
	groups = groups < 8 ? 8 : groups;
	double cost[ROWS_DISTRIBUTIONS][RAGGED_N_TILINGS];
	int cheapest[ROWS_DISTRIBUTIONS];
	const int first = cheapest[ROWS_EVEN] = cheapest_tiling(p, groups, four_ok, ROWS_EVEN, false, cost[ROWS_EVEN]);
	for (int dealt = ROWS_UNEVEN; dealt < ROWS_DISTRIBUTIONS; dealt++) {
		cheapest[dealt] = cheapest_tiling(p, groups, four_ok, dealt, dealt == ROWS_IN_ONE || first != RAGGED_N_384, cost[dealt]);
	}
	int second = first;
	double least = 0.0;                             /* the worst case with `first` and `second`, over the cheapest's cost */
	for (int tiling = 0; tiling < RAGGED_N_TILINGS; tiling++) {
		double worst = 0.0;
		for (int dealt = ROWS_UNEVEN; dealt < ROWS_DISTRIBUTIONS; dealt++) {
			const double best = cost[dealt][cheapest[dealt]];
			if (cost[dealt][first] < SECOND[dealt].share * best + SECOND[dealt].margin) {
				continue;
			}
			const double with = (cost[dealt][tiling] < cost[dealt][first] ? cost[dealt][tiling] : cost[dealt][first]) / best;
			worst = with > worst ? with : worst;
		}
		if (tiling != first && worst > 0.0 && (four_ok || tiling != RAGGED_N_384) && (second == first || worst < least || (worst == least && cost[ROWS_EVEN][tiling] < cost[ROWS_EVEN][second]))) {
			second = tiling;
			least = worst;
		}
	}
	return 1 << first | 1 << second;
}

extern "C" int amd_matmul_planned_tilings(int M, int K, int N, int num_groups, int cu_count) {
	GemmParams p;
	memset(&p, 0, sizeof(p));
	p.M = M; p.K = K; p.N = N;
	p.num_groups = num_groups;
	return ragged_n_tilings(p, cu_count, w4_ok(p));
}

extern "C" int amd_matmul_planned_wide(int M, int K, int N, int cu_count) {
	GemmParams p;
	memset(&p, 0, sizeof(p));
	p.M = M; p.K = K; p.N = N;
	return choose_tile(MODE_SINGLE, p, cu_count) == TILE_BIG && w4_ok(p)
		&& single_wide_is_cheaper(tiles_of(M, 256) * tiles_of(N, 384), tiles_in_launch(TILE_BIG, MODE_SINGLE, p), tiles_of(K, BK), cu_count);
}

extern "C" int amd_matmul_planned_sliced(int M, int K, int N, int num_groups, int has_c, int cu_count) {
	GemmParams p;
	memset(&p, 0, sizeof(p));
	p.M = M; p.K = K; p.N = N;
	p.num_groups = num_groups;
	p.C = has_c ? (const bf16_t *) scratch_of_device : NULL;
	p.beta = has_c ? 1.0f : 0.0f;
	const int mode = num_groups ? MODE_RAGGED_K : MODE_SINGLE;
	const long tiles = tiles_in_launch(TILE_BIG, mode, p);
	return tile_of_launch(mode, p, tiles, cu_count) == TILE_BIG && takes_sliced(mode, p, tiles, cu_count);
}

static long round_up8(long v) { return (v + 7) & ~7L; }

#define BIG_TILE 256, 256, 4, 2          /* 8 waves, wave tile 64 x 128 */
#define SMALL_TILE 128, 128, 2, 2        /* 4 waves, wave tile 64 x 64 */

/* `direct`: the operands suit the direct-to-LDS kernels.  grid_big / grid_small: work-group counts of the persistent kernel
 * and of the register-staged one; grid_wide: tiles of 192 token rows (ragged N), which bounds
 * the count of the larger ones too */
template <int MODE>
static int launch_gemm(const GemmParams & p, int transa, int transb, bool direct, long grid_big, long grid_small, long cu_count, hipStream_t stream,
					   long grid_wide = 0) {
	/* to_trans_a = 1 means A is stored [M][K] (k contiguous); to_trans_b = 1 means B is stored [K][N] (k-major) */
	const bool pk = !transa;
	const bool qk = transb != 0;
	if (grid_big <= 0 || grid_small <= 0) {
		return 0;
	}
	const int tile = tile_of_launch(MODE, p, grid_big, cu_count);
	const bool big = tile == TILE_BIG;
	const bool four_ok = direct && big && !qk && w4_ok(p);
	const bool wide_only = kernel_choice == AMD_MATMUL_KERNEL_FOUR_WAVES_384;
	const bool either = kernel_choice == AMD_MATMUL_KERNEL_AUTO;
	if (MODE == MODE_RAGGED_N && four_ok && grid_wide > 0 && wide_only) {
		return launch_ragged_n(1 << RAGGED_N_384, p, pk, grid_wide, cu_count, stream);
	}
	if (MODE == MODE_SINGLE && four_ok && p.split_k <= 1 && (wide_only || either)) {
		const long tiles = tiles_of(p.M, 256) * tiles_of(p.N, 384);
		if (wide_only || single_wide_is_cheaper(tiles, grid_big, tiles_of(p.K, BK), cu_count)) {
			if (pk) { return launch_w4d<true, MODE_SINGLE>(p, tiles, cu_count, stream); }
			return launch_w4d<false, MODE_SINGLE>(p, tiles, cu_count, stream);
		}
	}
	const bool four_one_loader = kernel_choice == AMD_MATMUL_KERNEL_FOUR_WAVES;
	if (MODE == MODE_RAGGED_N && four_ok && grid_wide > 0 && four_one_loader) {
		if (p.gather) {
			if (pk) { return launch_w4<true, MODE_RAGGED_N, GATHER_Q_ROWS>(p, grid_wide, cu_count, stream); }
			return launch_w4<false, MODE_RAGGED_N, GATHER_Q_ROWS>(p, grid_wide, cu_count, stream);
		}
		if (pk) { return launch_w4<true, MODE_RAGGED_N>(p, grid_wide, cu_count, stream); }
		return launch_w4<false, MODE_RAGGED_N>(p, grid_wide, cu_count, stream);
	}
	if (MODE == MODE_SINGLE && four_ok && p.split_k <= 1 && four_one_loader) {
		const long tiles = tiles_of(p.M, 256) * tiles_of(p.N, 288);
		if (pk) { return launch_w4<true, MODE_SINGLE>(p, tiles, cu_count, stream); }
		return launch_w4<false, MODE_SINGLE>(p, tiles, cu_count, stream);
	}
	if (MODE == MODE_RAGGED_N && direct && big && grid_wide > 0 && !qk && !(p.C && p.beta != 0.0f)) {
		/* Token rows in tiles of up to 384: a launch takes as long as its tiles are many (a k-tile step is paced by the
		 * latency of the operand stream, not by the multiplies), and a group of slightly more than a multiple of 256
		 * rows -- every second expert when the mean is such a multiple -- then needs no extra, nearly empty tile.
		 * Every element is accumulated over k in the same order as in the 256-row tiles: results are bit-identical. */
		return launch_ragged_n(either ? ragged_n_tilings(p, cu_count, four_ok) : 1 << RAGGED_N_288, p, pk, grid_wide, cu_count, stream);
	}
#define PICK(PK, QK) do { \
		if (direct) { \
			return big ? launch_stream<BIG_TILE, PK, QK, MODE>(p, grid_big, cu_count, stream) \
					   : launch_direct<PK, QK, MODE>(p, tile, stream); \
		} \
		return launch_staged<SMALL_TILE, PK, QK, MODE>(p, round_up8(grid_small), stream); \
	} while (0)
	if (MODE == MODE_RAGGED_N && p.gather) {
		/* gathered B: its rows are fetched through the row map by the loaders themselves (B is k-contiguous here) */
#define PICK_GATHER(PK) do { \
			if (direct) { \
				return big ? launch_stream<BIG_TILE, PK, false, MODE_RAGGED_N, GATHER_Q_ROWS>(p, grid_big, cu_count, stream) \
						   : launch_direct<PK, false, MODE_RAGGED_N, GATHER_Q_ROWS>(p, tile, stream); \
			} \
			return launch_staged<SMALL_TILE, PK, false, MODE_RAGGED_N>(p, round_up8(grid_small), stream); \
		} while (0)
		if (pk) { PICK_GATHER(true); }
		PICK_GATHER(false);
#undef PICK_GATHER
	}
	if (MODE == MODE_RAGGED_K && p.gather) {
		/* gathered A: the k-rows of the reduction are fetched through the row map (both operands are k-major here) */
		if (gathers_on_sliced(p, direct, tile, grid_big, cu_count)) {
			return launch_w4k<MODE_RAGGED_K, GATHER_P_KROWS>(p, grid_big, cu_count, stream);
		}
		if (direct) {
			return big ? launch_stream<BIG_TILE, true, true, MODE_RAGGED_K, GATHER_P_KROWS>(p, grid_big, cu_count, stream)
					   : launch_direct<true, true, MODE_RAGGED_K, GATHER_P_KROWS>(p, tile, stream);
		}
		return launch_staged<SMALL_TILE, true, true, MODE_RAGGED_K>(p, round_up8(grid_small), stream);
	}
	if constexpr (MODE != MODE_RAGGED_N) {
		if (pk && qk && direct && big && !p.gather && takes_sliced(MODE, p, grid_big, cu_count)) {
			return launch_w4k<MODE>(p, grid_big, cu_count, stream);
		}
	}
	if (!pk && !qk) { PICK(false, false); }
	if (pk && !qk) { PICK(true, false); }
	if (pk && qk) { PICK(true, true); }
	PICK(false, true);
#undef PICK
}

static bool aligned16(const void * ptr) { return (((uintptr_t) ptr) & 15) == 0; }

/* Can the operand (k-contiguous: rows of K elements; k-major: K rows of `rows` elements) be fetched with 16-byte
 * buffer loads?  Needs a 16-byte aligned base, a contiguous extent that is a multiple of 8 elements (so every row
 * starts aligned) and group bases that keep that alignment.  The kernels address one k-tile of one 256-row panel with
 * 32-bit offsets and everything above that with 64-bit pointers, so the operand's total size does not matter; the
 * contiguous extent itself is bounded (256 rows of K elements, or 64 k of `rows` elements, must stay below 4 GiB). */
static bool operand_direct_ok(const void * base, bool kmajor, long rows, long K, long group_stride_elems) {
	const long contiguous = kmajor ? rows : K;
	const long bound = kmajor ? (1L << 24) : (1L << 22);
	return aligned16(base) && (contiguous % 8 == 0) && (group_stride_elems % 8 == 0) && contiguous <= bound;
}

static int check_dtypes(DataflowDatatype a_dt, DataflowDatatype b_dt, DataflowDatatype c_dt, DataflowDatatype d_dt,
						DataflowDatatype compute_dt, const void * C, float beta) {
	if (a_dt != DATAFLOW_BF16 || b_dt != DATAFLOW_BF16 || d_dt != DATAFLOW_BF16) {
		fprintf(stderr, "Error: this matmul takes bf16 operands with a bf16 result; the single matmul also fp32 -> fp32, fp16 -> fp16 | fp32 and bf16 -> fp32 with fp32 accumulation and C in D's type (got A=%s B=%s D=%s)...\n",
				dataflow_datatype_as_string(a_dt), dataflow_datatype_as_string(b_dt), dataflow_datatype_as_string(d_dt));
		return -1;
	}
	if (c_dt != DATAFLOW_NONE && c_dt != DATAFLOW_BF16 && C != NULL && beta != 0.0f) {
		fprintf(stderr, "Error: this matmul implements a BF16 C only (got %s)...\n", dataflow_datatype_as_string(c_dt));
		return -1;
	}
	if (compute_dt != DATAFLOW_FP32 && compute_dt != DATAFLOW_BF16 && compute_dt != DATAFLOW_NONE) {
		fprintf(stderr, "Error: unsupported compute type %s; accumulation is always fp32...\n", dataflow_datatype_as_string(compute_dt));
		return -1;
	}
	return 0;
}

static int resolve_stream(Dataflow_Handle * handle, int stream_id, hipStream_t * stream) {
	if (stream_id == -1) {
		*stream = NULL;
		return 0;
	}
	if (stream_id < 0 || stream_id >= handle->num_streams) {
		fprintf(stderr, "Error: trying to dispatch matmul on stream id %d, but only have %d streams...\n", stream_id, handle->num_streams);
		return -1;
	}
	*stream = ((hipStream_t *) handle->streams)[stream_id];
	return 0;
}

extern "C" int amd_matmul_init(Dataflow_Handle * dataflow_handle, void * op_table_value) {
	Hip_Function * fn = (Hip_Function *) op_table_value;
	MatmulExtra * extra = (MatmulExtra *) calloc(1, sizeof(MatmulExtra));
	if (!extra) {
		fprintf(stderr, "Error: malloc failed for matmul op extra...\n");
		return -1;
	}
	const int dev = dataflow_handle->device_id;
	if (dev >= 0 && dev < AMD_MATMUL_MAX_DEVICES && !scratch_of_device[dev]) {
		void * ptr = NULL;
		hipError_t e = hipSetDevice(dev);
		if (e == hipSuccess) {
			e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
		}
		if (e != hipSuccess || !ptr) {
			fprintf(stderr, "Error: could not look up the matmul scratch on device %d: %s...\n", dev, hipGetErrorString(e));
			free(extra);
			return -1;
		}
		scratch_of_device[dev] = ptr;
	}
	Hip_Device_Info * info = (Hip_Device_Info *) dataflow_handle->device_info;
	extra->cu_count = info ? info->cu_count : 256;
	extra->lds_optin = info ? info->optin_max_lds_per_block : 65536;
	fn->op_extra = extra;
	const char * env = getenv("AMD_MATMUL_KERNEL");
	if (env && (env[0] == '4' || env[0] == '8') && env[1] == 0) {
		kernel_choice = env[0] == '4' ? AMD_MATMUL_KERNEL_FOUR_WAVES : AMD_MATMUL_KERNEL_EIGHT_WAVES;
	} else if (env && strcmp(env, "384") == 0) {
		kernel_choice = AMD_MATMUL_KERNEL_FOUR_WAVES_384;
	} else if (env && strcmp(env, "auto") == 0) {
		kernel_choice = AMD_MATMUL_KERNEL_AUTO;
	}
	return 0;
}

static long extra_cu_count(void * op_extra) {
	return op_extra ? ((MatmulExtra *) op_extra)->cu_count : 256;
}

/* amd_matmul_no_alloc's limit, part of its interface: a problem whose 128 x 128 tiles leave half of the compute units idle, with a K of
 * eight k-tiles or more, is refused where the partial sums of a split over those (a multiple of four k-tiles each) are more than 8 MiB.
 * 0: taken; otherwise that number of splits */
#define NO_ALLOC_LIMIT_BYTES (8u << 20)
static long beyond_scratch(const GemmParams & p, bool direct, long cu_count) {
	const long k_tiles = tiles_of(p.K, BK);
	const bool big = tiles_of(p.M, 256) * tiles_of(p.N, 256) >= cu_count / 2 && p.M >= 256 && p.N >= 256;
	long splits = direct && !big ? cu_count / (tiles_of(p.M, 128) * tiles_of(p.N, 128)) : 1;
	if (splits < 2 || k_tiles < 8) {
		return 0;
	}
	const long per = tiles_of(k_tiles, splits);
	splits = tiles_of(k_tiles, per < 4 ? 4 : (per + 3) & ~3L);
	return splits < 2 || (uint64_t) NO_ALLOC_LIMIT_BYTES / 4 / (uint64_t) splits >= (uint64_t) p.M * (uint64_t) p.N ? 0 : splits;
}

/* Few tiles and a long K (the router's GEMMs: up to 64 experts on one side; projections of few tokens): K split over the
 * compute units that the tiles leave idle, fp32 partial sums in `workspace` (16-byte aligned), added up by the pass behind.
 * Split where the cheapest tile and number of splits that the workspace holds cost less than the problem unsplit: the k-tiles
 * of a split at the tile's cost (the 128 x 128 tile has four waves here: 0.66), 4 us for the pass behind and its 3 TB/s over the partial
 * sums.  Over 310 problems (8-4096 columns, 16-30000 tokens, K 64-30000) it takes 2 % longer than the best of all tiles and splits; splits
 * over all idle compute units wherever there were any, on 128 x 128 tiles, took 15 % longer.  1792 x 896 x 937, us: 8.0 unsplit on
 * 64 x 128 tiles, 19.9 split in two; 2176 x 19234 x 64: 20.9 in six on 64 x 64, 67.9 unsplit.
 * The router's logits (up to 64 rows of k-contiguous weights) are charged 1 us for the pass and a quarter for each split: the layer's
 * routing adds up their partial sums in its selection, whose few work-groups wait for a split's loads behind the last ones'.  A
 * plain product of that form pays for the pass behind all the same, but has to split alike: the routing leaves the matmul's bits.  Over 63
 * of them (8, 32 and 64 columns, 16-32768 tokens, K 512-4096) that price costs 1.6 us at most (8 or 32 x 2048 x 8192, 11.0 us
 * against 9.4) and saves 1.3 at 3001 tokens; over all it is 0.6 % faster than the plain one.
 * 0: unsplit; otherwise the split in `p`, and its tile + 1. */
#define SPLIT_ROUND_COST 50                 /* the partial sums' stores, beside their bytes below */
#define SPLIT_PASS_COST 400
#define SPLIT_LOGITS_PASS_COST 100
#define SPLIT_LOGITS_COST 25
#define SPLIT_LOGITS_MAX_ROWS 64
#define SPLIT_BYTES_PER_COST 30000          /* 3 TB/s */
static int plan_split(GemmParams & p, int transa, int transb, bool direct, float * workspace, uint64_t workspace_bytes, long cu_count) {
	static const int SPLITS[] = {2, 3, 4, 6, 8, 12, 16, 24, 32, 48};
	const long k_tiles = tiles_of(p.K, BK);
	if (!direct || k_tiles < 4 || !workspace || (((uintptr_t) workspace) & 15)) {
		return 0;
	}
	const uint64_t count = (uint64_t) p.M * (uint64_t) p.N;
	const bool logits = transa && !transb && p.M <= SPLIT_LOGITS_MAX_ROWS;
	long least;
	choose_tile(MODE_SINGLE, p, cu_count, true, &least);
	int best = 0;
	for (int tile = TILE_64x32; tile <= TILE_128x128; tile++) {
		const long tiles = tiles_in_launch(tile, MODE_SINGLE, p);
		const long cost_of_k_tile = tile == TILE_128x128 ? 66 : TILES[tile].cost;
		for (int splits_wanted : SPLITS) {
			const long per = tiles_of(k_tiles, splits_wanted);
			const long splits = tiles_of(k_tiles, per);
			if (per < 2 || splits < 2 || tiles * splits > 4 * cu_count || workspace_bytes / 4 / (uint64_t) splits < count) {
				continue;
			}
			const long cost = tiles_of(tiles * splits, cu_count) * (per * cost_of_k_tile + SPLIT_ROUND_COST) + (logits ? SPLIT_LOGITS_PASS_COST + splits * SPLIT_LOGITS_COST : SPLIT_PASS_COST)
				+ (long) ((uint64_t) splits * count * 4 / SPLIT_BYTES_PER_COST);
			if (cost < least) {
				least = cost;
				best = tile + 1;
				p.split_k = (int) splits;
				p.kt_per_split = (int) per;
			}
		}
	}
	if (best) {
		p.partial = workspace;
	}
	return best;
}

extern "C" int amd_matmul_planned_splits(int to_trans_a, int to_trans_b, int M, int K, int N, int has_c, uint64_t workspace_bytes, int cu_count) {
	GemmParams p;
	memset(&p, 0, sizeof(p));
	p.M = M; p.K = K; p.N = N;
	p.C = has_c ? (const bf16_t *) scratch_of_device : NULL;
	/* an aligned workspace at no address in particular: the plan writes nothing */
	return plan_split(p, to_trans_a, to_trans_b, true, (float *) 4096, workspace_bytes, cu_count) ? p.split_k : 1;
}

/* the pass behind the partial products: D from their sums */
static int launch_split_reduce(const GemmParams & p, hipStream_t stream) {
	const uint64_t count = (uint64_t) p.M * (uint64_t) p.N;
	const long blocks = (long) ((count + 1023) / 1024);
	hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned int) (blocks < 4096 ? blocks : 4096)), dim3(256), 0, stream,
					   (const float *) p.partial, p.split_k, (long long) count, p.alpha, p.beta, p.C, p.D);
	return check_launch();
}

/* ---- operands that the 16-byte loads cannot fetch (an odd number of experts: the rows of the router's gradient) ----
 *
 * The register-staged kernel fetches such an operand element by element, 5 us per k-tile of 128 x 128, unsplit along K: the
 * router's weight gradient of 46398 tokens and 33 experts (1024 x 46398 x 33) took 3828 us, its input gradient
 * 93.  A copy with its rows padded to a multiple of 8 elements (zeros) in the caller's workspace costs a pass over that
 * operand (4-6 us here), and the copy then runs on the direct kernel, split along K where the matmul op splits.  A training step of
 * that layer (dim 1024, top 8, expert dim 640) takes 5582 us instead of 9998, one of 1132 tokens and 59 experts 717 instead of
 * 792; also where the staged kernel has one k-tile to do it takes 12 us, copy and product 10. */

__global__ void __launch_bounds__(256) pad_rows_kernel(const bf16_t * __restrict__ src, long long rows, int extent, int pitch, u32x4 * __restrict__ dst) {
	const int chunks = pitch >> 3;                       /* 16-byte chunks of a padded row */
	const long long total = rows * chunks;
	const long long stride = (long long) gridDim.x * 256;
	for (long long i = (long long) blockIdx.x * 256 + threadIdx.x; i < total; i += stride) {
		const long long r = i / chunks;
		const int c = (int) (i - r * chunks) * 8;
		const bf16_t * s = src + r * extent + c;
		uint32_t e[8];
		#pragma unroll
		for (int j = 0; j < 8; j++) {
			e[j] = c + j < extent ? (uint32_t) s[j] : 0u;
		}
		dst[i] = u32x4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
	}
}

/* Copies of the operands of `p` that need one, at the start of the workspace, which is advanced past them; `p` then
 * describes the padded problem.  1: done, 0: does not apply or does not fit (`p` as it was), -1: error. */
static int pad_operands(GemmParams & p, int transa, int transb, uint8_t *& workspace, uint64_t & workspace_bytes, hipStream_t stream) {
	if (!workspace || (((uintptr_t) workspace) & 15) || p.K < 1) {
		return 0;
	}
	const bool copy_a = !operand_direct_ok(p.A, !transa, p.M, p.K, 0), copy_b = !operand_direct_ok(p.B, transb != 0, p.N, p.K, 0);
	const long pitch_a = round_up8(transa ? p.K : p.M), pitch_b = round_up8(transb ? p.N : p.K);
	/* row lengths and K as ints, and what operand_direct_ok allows of a contiguous extent */
	if (pitch_a > (transa ? 1L << 22 : 1L << 24) || pitch_b > (transb ? 1L << 24 : 1L << 22)) {
		return 0;
	}
	const long rows_a = transa ? p.M : p.K, rows_b = transb ? p.K : p.N;
	const uint64_t bytes_a = copy_a ? (((uint64_t) rows_a * (uint64_t) pitch_a * 2u) + 255) & ~255UL : 0;
	const uint64_t bytes_b = copy_b ? (((uint64_t) rows_b * (uint64_t) pitch_b * 2u) + 255) & ~255UL : 0;
	if (workspace_bytes < bytes_a || workspace_bytes - bytes_a < bytes_b) {
		return 0;
	}
	for (int which = 0; which < 2; which++) {
		if (!(which ? copy_b : copy_a)) {
			continue;
		}
		const long rows = which ? rows_b : rows_a, pitch = which ? pitch_b : pitch_a;
		const int extent = which ? (transb ? p.N : p.K) : (transa ? p.K : p.M);
		const long blocks = tiles_of(rows * (pitch / 8), 256);
		u32x4 * dst = (u32x4 *) (workspace + (which ? bytes_a : 0));
		hipLaunchKernelGGL(pad_rows_kernel, dim3((unsigned int) (blocks < 16384 ? blocks : 16384)), dim3(256), 0, stream,
						   which ? p.B : p.A, (long long) rows, extent, (int) pitch, dst);
		if (check_launch()) {
			return -1;
		}
		(which ? p.B : p.A) = (const bf16_t *) dst;
	}
	workspace += bytes_a + bytes_b;
	workspace_bytes -= bytes_a + bytes_b;
	if (copy_a && !transa) {
		p.pitchA = (int) pitch_a;
	}
	if (copy_b && transb) {
		p.pitchB = (int) pitch_b;
	}
	if ((copy_a && transa) || (copy_b && !transb)) {
		p.k_rows = p.K;
		p.K = (int) round_up8(p.K);
	}
	return 1;
}

/* a padded problem that is not split: the direct kernel on its cheapest tile */
static int launch_padded(const GemmParams & p, int transa, int transb, long cu_count, hipStream_t stream) {
	const int tile = choose_tile(MODE_SINGLE, p, cu_count, false);
	const bool pk = !transa, qk = transb != 0;
	if (!pk && !qk) { return launch_direct<false, false, MODE_SINGLE>(p, tile, stream); }
	if (pk && !qk) { return launch_direct<true, false, MODE_SINGLE>(p, tile, stream); }
	if (pk && qk) { return launch_direct<true, true, MODE_SINGLE>(p, tile, stream); }
	return launch_direct<false, true, MODE_SINGLE>(p, tile, stream);
}

/* shared by amd_matmul and amd_matmul_no_alloc: checks, kernel choice, launch.  `workspace` (may be NULL) holds the fp32
 * partial sums of a split along K; `must_fit`: a split that the workspace cannot hold is an error (beyond_scratch) */
static int run_matmul(Dataflow_Handle * dataflow_handle, int stream_id, GemmParams & p, int transa, int transb,
					  uint8_t * workspace, uint64_t workspace_bytes, long cu_count, bool must_fit) {
	if (p.M < 0 || p.N < 0 || p.K < 0 || !p.D || ((p.M > 0 && p.N > 0 && p.K > 0) && (!p.A || !p.B))) {
		fprintf(stderr, "Error: bad matmul arguments M=%d K=%d N=%d A=%p B=%p D=%p...\n", p.M, p.K, p.N, (void *) p.A, (void *) p.B, (void *) p.D);
		return -1;
	}
	if (p.M == 0 || p.N == 0) {
		return 0;
	}
	hipStream_t stream;
	if (resolve_stream(dataflow_handle, stream_id, &stream)) {
		return -1;
	}
	if (hipSetDevice(dataflow_handle->device_id) != hipSuccess) {
		fprintf(stderr, "Error: hipSetDevice failed in matmul...\n");
		return -1;
	}
	const bool direct = operand_direct_ok(p.A, !transa, p.M, p.K, 0) && operand_direct_ok(p.B, transb != 0, p.N, p.K, 0);
	const long grid_big = tiles_of(p.M, 256) * tiles_of(p.N, 256);
	const long grid_small = tiles_of(p.M, 128) * tiles_of(p.N, 128);
	const int padded = direct ? 0 : pad_operands(p, transa, transb, workspace, workspace_bytes, stream);
	if (padded < 0) {
		return -1;
	}
	const long refused = must_fit && !padded ? beyond_scratch(p, direct, cu_count) : 0;
	if (refused) {
		fprintf(stderr, "Error: this %d x %d x %d matmul may split along K into %ld parts of %lu partial sums each, more than the %u bytes of scratch that one call may ask for; use the matmul op with a workspace...\n",
				p.M, p.K, p.N, refused, (unsigned long) p.M * (unsigned long) p.N, NO_ALLOC_LIMIT_BYTES);
		return -1;
	}
	const int split = plan_split(p, transa, transb, direct || padded, (float *) workspace, workspace_bytes, cu_count);
	if (split) {
		if (launch_split(p, split - 1, transa, transb, stream)) {
			return -1;
		}
		return launch_split_reduce(p, stream);
	}
	if (padded) {
		return launch_padded(p, transa, transb, cu_count, stream);
	}
	return launch_gemm<MODE_SINGLE>(p, transa, transb, direct, grid_big, grid_small, cu_count, stream);
}

/* Ragged K without a C operand: D_g = alpha * (sum over no rows) = 0 for a group without rows.  The GEMM kernels give such
 * a group no tile, so its zeros are written here, by work-groups that find the group empty (the others exit at once). */
__global__ void __launch_bounds__(256) zero_empty_groups_kernel(const int * __restrict__ cumsum, int num_groups, bf16_t * __restrict__ D, long long strideD, long long count) {
	const long long step = (long long) gridDim.x * 256;
	const long long first = (long long) blockIdx.x * 256 + threadIdx.x;
	for (int g = blockIdx.y; g < num_groups; g += gridDim.y) {
		const int hi = cumsum[g];
		const int lo = g ? cumsum[g - 1] : 0;
		if (hi - lo > 0) {
			continue;
		}
		bf16_t * dst = D + (long long) g * strideD;
		const long long vecs = (((uintptr_t) dst) & 15) == 0 ? count >> 3 : 0;       /* 16-byte stores where the group's base allows them */
		for (long long i = first; i < vecs; i += step) {
			reinterpret_cast<uint4 *>(dst)[i] = uint4{0u, 0u, 0u, 0u};
		}
		for (long long i = (vecs << 3) + first; i < count; i += step) {
			dst[i] = (bf16_t) 0;
		}
	}
}

/* The element types beside all-bf16 (gemm_typed_kernel.h).  Returns 0 when the combination is not one of them, 1 after a
 * launch, -1 on an error.  A and B share a type; C, where it is used, has D's type. */
static int run_typed_matmul(Dataflow_Handle * dataflow_handle, int stream_id, DataflowDatatype ab_dt, DataflowDatatype d_dt,
							int transa, int transb, int M, int K, int N, float alpha, float beta, const void * A, const void * B,
							const void * C, void * D) {
	const bool f32_f32 = ab_dt == DATAFLOW_FP32 && d_dt == DATAFLOW_FP32;
	const bool f16_f16 = ab_dt == DATAFLOW_FP16 && d_dt == DATAFLOW_FP16;
	const bool f16_f32 = ab_dt == DATAFLOW_FP16 && d_dt == DATAFLOW_FP32;
	const bool bf16_f32 = ab_dt == DATAFLOW_BF16 && d_dt == DATAFLOW_FP32;
	if (!f32_f32 && !f16_f16 && !f16_f32 && !bf16_f32) {
		return 0;
	}
	if (M < 0 || N < 0 || K < 0 || !D || ((M > 0 && N > 0 && K > 0) && (!A || !B))) {
		fprintf(stderr, "Error: bad matmul arguments M=%d K=%d N=%d A=%p B=%p D=%p...\n", M, K, N, A, B, D);
		return -1;
	}
	if (M == 0 || N == 0) {
		return 1;
	}
	hipStream_t stream;
	if (resolve_stream(dataflow_handle, stream_id, &stream)) {
		return -1;
	}
	if (hipSetDevice(dataflow_handle->device_id) != hipSuccess) {
		fprintf(stderr, "Error: hipSetDevice failed in matmul...\n");
		return -1;
	}
	const long tiles = tiles_of(M, TYPED_TILE) * tiles_of(N, TYPED_TILE);
	if (tiles > 0x7fffffffL) {
		fprintf(stderr, "Error: %d x %d is more output tiles than one launch of this matmul takes...\n", M, N);
		return -1;
	}
	TypedGemmParams t;
	t.P = A; t.Q = B; t.C = C; t.D = D;
	t.M = M; t.N = N; t.K = K;
	t.p_kmajor = !transa;
	t.q_kmajor = transb != 0;
	t.alpha = alpha; t.beta = beta;
	const dim3 grid((unsigned int) tiles), block(TYPED_THREADS);
	if (f32_f32) {
		hipLaunchKernelGGL((gemm_typed_kernel<float, float>), grid, block, 0, stream, t);
	} else if (f16_f16) {
		hipLaunchKernelGGL((gemm_typed_kernel<_Float16, _Float16>), grid, block, 0, stream, t);
	} else if (f16_f32) {
		hipLaunchKernelGGL((gemm_typed_kernel<_Float16, float>), grid, block, 0, stream, t);
	} else {
		hipLaunchKernelGGL((gemm_typed_kernel<bf16_t, float>), grid, block, 0, stream, t);
	}
	return check_launch() ? -1 : 1;
}

extern "C" int amd_matmul(Dataflow_Handle * dataflow_handle, int stream_id, Op * op, void * op_extra) {
	void ** a = op->op_args;
	DataflowDatatype a_dt = *((DataflowDatatype *) a[1]);
	DataflowDatatype b_dt = *((DataflowDatatype *) a[2]);
	DataflowDatatype c_dt = *((DataflowDatatype *) a[3]);
	DataflowDatatype d_dt = *((DataflowDatatype *) a[4]);
	DataflowDatatype compute_dt = *((DataflowDatatype *) a[5]);
	int transa = *((int *) a[6]);
	int transb = *((int *) a[7]);
	GemmParams p;
	memset(&p, 0, sizeof(p));
	p.M = *((int *) a[8]);
	p.K = *((int *) a[9]);
	p.N = *((int *) a[10]);
	p.alpha = *((float *) a[11]);
	p.beta = *((float *) a[12]);
	p.A = (const bf16_t *) *((uint64_t *) a[13]);
	p.B = (const bf16_t *) *((uint64_t *) a[14]);
	p.C = (const bf16_t *) *((uint64_t *) a[15]);
	p.D = (bf16_t *) *((uint64_t *) a[16]);
	if (c_dt == DATAFLOW_NONE || p.beta == 0.0f) {
		p.C = NULL;
	}
	if (a_dt == b_dt && !(a_dt == DATAFLOW_BF16 && d_dt == DATAFLOW_BF16)) {
		/* fp32, fp16, or bf16 with an fp32 result: fp32 accumulation only, C in D's type */
		if ((p.C == NULL || c_dt == d_dt) && (compute_dt == DATAFLOW_FP32 || compute_dt == DATAFLOW_NONE)) {
			const int r = run_typed_matmul(dataflow_handle, stream_id, a_dt, d_dt, transa, transb, p.M, p.K, p.N, p.alpha, p.beta,
										   (const void *) p.A, (const void *) p.B, (const void *) p.C, (void *) p.D);
			if (r != 0) {
				return r < 0 ? -1 : 0;
			}
		}
	}
	if (check_dtypes(a_dt, b_dt, c_dt, d_dt, compute_dt, p.C, p.beta)) {
		return -1;
	}
	const uint64_t workspace_bytes = *((uint64_t *) a[17]);
	uint8_t * workspace = (uint8_t *) *((uint64_t *) a[18]);
	return run_matmul(dataflow_handle, stream_id, p, transa, transb, workspace, workspace_bytes, extra_cu_count(op_extra), false);
}

/* Two products with the same A, both operands k-major: what amd_matmul leaves without a workspace for (A, B, C, D) and for (A, B2,
 * C2, D2), bit for bit (../layer/layer_ops.h).  On the direct kernel's tiles one launch does both. */
extern "C" int amd_matmul_twin(Dataflow_Handle * dataflow_handle, int stream_id, Op * op, void * op_extra) {
	void ** a = op->op_args;
	GemmParams p;
	memset(&p, 0, sizeof(p));
	p.M = *((int *) a[0]);
	p.K = *((int *) a[1]);
	p.N = *((int *) a[2]);
	p.beta = *((float *) a[3]);
	p.alpha = 1.0f;
	p.A = (const bf16_t *) *((uint64_t *) a[4]);
	p.B = (const bf16_t *) *((uint64_t *) a[5]);
	p.C = p.beta == 0.0f ? NULL : (const bf16_t *) *((uint64_t *) a[6]);
	p.D = (bf16_t *) *((uint64_t *) a[7]);
	GemmParams second = p;
	second.B = (const bf16_t *) *((uint64_t *) a[8]);
	second.C = p.beta == 0.0f ? NULL : (const bf16_t *) *((uint64_t *) a[9]);
	second.D = (bf16_t *) *((uint64_t *) a[10]);
	const long cu_count = extra_cu_count(op_extra);
	if (p.M >= 1 && p.K >= 1 && p.N >= 1 && p.N <= (1 << 24) && p.A && p.B && p.D && second.B && second.D && (p.C == NULL) == (second.C == NULL) && kernel_choice == AMD_MATMUL_KERNEL_AUTO
		&& operand_direct_ok(p.A, true, p.M, p.K, 0) && operand_direct_ok(p.B, true, p.N, p.K, 0) && operand_direct_ok(second.B, true, p.N, p.K, 0)) {
		GemmParams both = p;
		both.N = 2 * p.N;
		const int tile = choose_tile(MODE_SINGLE, both, cu_count);
		if (tile != TILE_BIG) {
			p.B_twin = second.B;
			p.C_twin = second.C;
			p.D_twin = second.D;
			hipStream_t stream;
			if (resolve_stream(dataflow_handle, stream_id, &stream)) {
				return -1;
			}
			if (hipSetDevice(dataflow_handle->device_id) != hipSuccess) {
				fprintf(stderr, "Error: hipSetDevice failed in the twin matmul...\n");
				return -1;
			}
			return launch_direct<true, true, MODE_SINGLE>(p, tile, stream, 2);
		}
	}
	return run_matmul(dataflow_handle, stream_id, p, 0, 1, NULL, 0, cu_count, false)
		|| run_matmul(dataflow_handle, stream_id, second, 0, 1, NULL, 0, cu_count, false) ? -1 : 0;
}

/* D = alpha * op(A) op(B) + beta * C like amd_matmul (same kernels, same split along K, bit-identical results), for
 * callers that cannot allocate: the split's partial sums go to the library's own scratch on the handle's device
 * instead of a caller's workspace, and the call makes no allocation of any kind.  BF16 operands and result, fp32
 * accumulation; C is ignored when NULL or beta == 0.  Refused with -1: see beyond_scratch.  The scratch keeps the last call's contents (nothing in it
 * has to start at zero: every partial sum is written before it is read); it is shared by every call on that device, so
 * calls that overlap on one device -- two streams, two host threads -- race on it. */
extern "C" int amd_matmul_no_alloc(Dataflow_Handle * dataflow_handle, int stream_id, int to_trans_a, int to_trans_b,
								   int M, int K, int N, float alpha, float beta, void * A, void * B, void * C, void * D) {
	if (!dataflow_handle) {
		fprintf(stderr, "Error: amd_matmul_no_alloc needs a handle...\n");
		return -1;
	}
	const int dev = dataflow_handle->device_id;
	if (dev < 0 || dev >= AMD_MATMUL_MAX_DEVICES || !scratch_of_device[dev]) {
		fprintf(stderr, "Error: amd_matmul_no_alloc on device %d before the matmul op was registered on a handle of that device...\n", dev);
		return -1;
	}
	GemmParams p;
	memset(&p, 0, sizeof(p));
	p.M = M; p.K = K; p.N = N;
	p.alpha = alpha; p.beta = beta;
	p.A = (const bf16_t *) A; p.B = (const bf16_t *) B; p.C = (beta == 0.0f) ? NULL : (const bf16_t *) C; p.D = (bf16_t *) D;
	Hip_Device_Info * info = (Hip_Device_Info *) dataflow_handle->device_info;
	return run_matmul(dataflow_handle, stream_id, p, to_trans_a, to_trans_b, (uint8_t *) scratch_of_device[dev], AMD_MATMUL_SCRATCH_BYTES,
					  info ? info->cu_count : 256, true);
}

extern "C" int amd_grouped_matmul(Dataflow_Handle * dataflow_handle, int stream_id, Op * op, void * op_extra) {
	void ** a = op->op_args;
	DataflowDatatype a_dt = *((DataflowDatatype *) a[1]);
	DataflowDatatype b_dt = *((DataflowDatatype *) a[2]);
	DataflowDatatype c_dt = *((DataflowDatatype *) a[3]);
	DataflowDatatype d_dt = *((DataflowDatatype *) a[4]);
	DataflowDatatype compute_dt = *((DataflowDatatype *) a[5]);
	int transa = *((int *) a[6]);
	int transb = *((int *) a[7]);
	int ragged = *((int *) a[8]);
	GemmParams p;
	memset(&p, 0, sizeof(p));
	p.M = *((int *) a[9]);
	p.K = *((int *) a[10]);
	p.N = *((int *) a[11]);
	p.num_groups = *((int *) a[12]);
	p.cumsum = (const int *) *((uint64_t *) a[13]);
	p.alpha = *((float *) a[14]);
	p.beta = *((float *) a[15]);
	p.A = (const bf16_t *) *((uint64_t *) a[16]);
	uint64_t strideA_bytes = *((uint64_t *) a[17]);
	p.B = (const bf16_t *) *((uint64_t *) a[18]);
	p.C = (const bf16_t *) *((uint64_t *) a[19]);
	p.D = (bf16_t *) *((uint64_t *) a[20]);
	uint64_t strideD_bytes = *((uint64_t *) a[21]);
	/* the gathered form of the op carries two more arguments: the row map and the number of rows of the gathered operand */
	if (op->op_skeleton.header.num_args == 24) {
		p.gather = (const int *) *((uint64_t *) a[22]);
		p.gather_rows = *((int *) a[23]);
		const int row_elems = ragged == AMD_GROUPED_RAGGED_N ? p.K : p.M;      /* one row of the gathered operand */
		if (!p.gather || p.gather_rows < 1 || (ragged != AMD_GROUPED_RAGGED_N && ragged != AMD_GROUPED_RAGGED_K) || row_elems < 1 ||
			(uint64_t) p.gather_rows * (uint64_t) row_elems * 2u > 0xFFFFFFFFull) {
			fprintf(stderr, "Error: bad gathered grouped matmul arguments (row map %p, %d rows of %d elements: the gathered operand must stay below 4 GiB)...\n",
					(const void *) p.gather, p.gather_rows, row_elems);
			return -1;
		}
	}
	if (c_dt == DATAFLOW_NONE || p.beta == 0.0f) {
		p.C = NULL;
	}
	if (check_dtypes(a_dt, b_dt, c_dt, d_dt, compute_dt, p.C, p.beta)) {
		return -1;
	}
	if (p.num_groups < 1 || !p.cumsum || !p.A || !p.B || !p.D || p.M < 1 || (strideA_bytes & 1) || (strideD_bytes & 1)) {
		fprintf(stderr, "Error: bad grouped matmul arguments (groups=%d M=%d K=%d N=%d)...\n", p.num_groups, p.M, p.K, p.N);
		return -1;
	}
	p.strideA = (long long) (strideA_bytes / 2);
	p.strideD = (long long) (strideD_bytes / 2);
	hipStream_t stream;
	if (resolve_stream(dataflow_handle, stream_id, &stream)) {
		return -1;
	}
	if (hipSetDevice(dataflow_handle->device_id) != hipSuccess) {
		fprintf(stderr, "Error: hipSetDevice failed in grouped matmul...\n");
		return -1;
	}
	if (ragged == AMD_GROUPED_RAGGED_N) {
		if (transb != 0 || p.K < 1 || p.N < 0) {
			fprintf(stderr, "Error: ragged-N grouped matmul needs to_trans_b == 0 and K >= 1...\n");
			return -1;
		}
		if (p.N == 0) {
			return 0;
		}
		/* A: one matrix per group at strideA; B: rows packed, so every group base is K-aligned */
		const bool direct = operand_direct_ok(p.A, !transa, p.M, p.K, p.strideA) && operand_direct_ok(p.B, false, p.N, p.K, 0);
		/* upper bound of n-tiles: every group may end in one partial tile */
		const long grid_big = tiles_of(p.M, 256) * ((long) p.N / 256 + p.num_groups);
		const long grid_small = tiles_of(p.M, 128) * ((long) p.N / 128 + p.num_groups);
		const long grid_wide = tiles_of(p.M, 256) * ((long) p.N / 192 + p.num_groups);
		return launch_gemm<MODE_RAGGED_N>(p, transa, transb, direct, grid_big, grid_small, extra_cu_count(op_extra), stream, grid_wide);
	}
	if (ragged == AMD_GROUPED_RAGGED_K) {
		if (transa != 0 || transb != 1 || p.N < 1) {
			fprintf(stderr, "Error: ragged-K grouped matmul needs to_trans_a == 0 and to_trans_b == 1...\n");
			return -1;
		}
		const bool direct = ragged_k_direct_ok(p);
		const long grid_big = tiles_of(p.M, 256) * tiles_of(p.N, 256) * p.num_groups;
		const long grid_small = tiles_of(p.M, 128) * tiles_of(p.N, 128) * p.num_groups;
		if (p.C == nullptr) {
			const long long count = (long long) p.M * p.N;
			const long long blocks = (count / 8 + 255) / 256;
			hipLaunchKernelGGL(zero_empty_groups_kernel, dim3((unsigned int) (blocks < 64 ? (blocks < 1 ? 1 : blocks) : 64), (unsigned int) (p.num_groups < 65535 ? p.num_groups : 65535)), dim3(256), 0, stream,
							   p.cumsum, p.num_groups, p.D, p.strideD, count);
			if (check_launch()) {
				return -1;
			}
		}
		return launch_gemm<MODE_RAGGED_K>(p, transa, transb, direct, grid_big, grid_small, extra_cu_count(op_extra), stream);
	}
	fprintf(stderr, "Error: unknown ragged dimension %d...\n", ragged);
	return -1;
}

/* The layer's question in front of its dW1 | dW3 (../layer/layer_ops.h), answered by the launch's own rules: 1 where the gathered form runs on
 * the sliced kernel.  Launches nothing. */
extern "C" int amd_gathers_k_rows(Dataflow_Handle * dataflow_handle, int stream_id, Op * op, void * op_extra) {
	(void) dataflow_handle; (void) stream_id;
	void ** a = op->op_args;
	GemmParams p;
	memset(&p, 0, sizeof(p));
	p.M = *((int *) a[0]);
	p.K = *((int *) a[1]);
	p.N = *((int *) a[2]);
	p.num_groups = *((int *) a[3]);
	p.A = (const bf16_t *) *((uint64_t *) a[4]);
	p.gather_rows = *((int *) a[5]);
	p.B = (const bf16_t *) *((uint64_t *) a[6]);
	p.C = (const bf16_t *) *((uint64_t *) a[7]);
	p.beta = p.C ? 1.0f : 0.0f;
	p.D = (bf16_t *) *((uint64_t *) a[8]);
	p.strideD = (long long) (*((uint64_t *) a[9]) / 2);
	if (p.M < 1 || p.N < 1 || p.num_groups < 1 || p.gather_rows < 1) {
		return 0;
	}
	const long cu_count = extra_cu_count(op_extra), tiles = tiles_in_launch(TILE_BIG, MODE_RAGGED_K, p);
	return gathers_on_sliced(p, ragged_k_direct_ok(p), tile_of_launch(MODE_RAGGED_K, p, tiles, cu_count), tiles, cu_count);
}

/* The activation behind an up-projection on kernels whose epilogue does not compute it */
__global__ void __launch_bounds__(256) up_swiglu_kernel(const bf16_t * x1, const bf16_t * x3, int row_stride, bf16_t * h, long long rows, int half) {
	const int per_row = half >> 3;
	const long long v = (long long) blockIdx.x * 256 + threadIdx.x;
	if (v < rows * per_row) {
		swiglu_strided_vector((size_t) v, (size_t) per_row, (size_t) row_stride, x1, x3, h);
	}
}
static int launch_up_swiglu(const GemmParams & p, int half, const bf16_t * x3, int row_stride, hipStream_t stream) {
	const long long vectors = (long long) p.N * (half >> 3);
	hipLaunchKernelGGL(up_swiglu_kernel, dim3((unsigned int) ((vectors + 255) / 256)), dim3(256), 0, stream, (const bf16_t *) p.D, x3, row_stride, p.h, (long long) p.N, half);
	return check_launch();
}

/* a GEMM of the up-projection as the matmul ops launch it */
static int launch_up_projection(const GemmParams & p, bool single, long cu_count, hipStream_t stream) {
	if (single) {
		return launch_gemm<MODE_SINGLE>(p, 1, 0, true, tiles_of(p.M, 256) * tiles_of(p.N, 256), tiles_of(p.M, 128) * tiles_of(p.N, 128), cu_count, stream);
	}
	return launch_gemm<MODE_RAGGED_N>(p, 1, 0, true, tiles_of(p.M, 256) * ((long) p.N / 256 + p.num_groups), tiles_of(p.M, 128) * ((long) p.N / 128 + p.num_groups),
									  cu_count, stream, tiles_of(p.M, 256) * ((long) p.N / 192 + p.num_groups));
}

/* The layer's up-projection and its activation in one op (../layer/layer_ops.h): x1 | x3 of the routed rows and h.  Few
 * rows run on the direct kernel, whose epilogue then computes h; where the GEMM is large enough for the persistent kernels the
 * activation follows in a launch of its own.  A thirteenth argument, x3: the two halves of a row go to arrays of their own,
 * on the direct kernel; without a prefix sum the rows are those of one expert, packed.  A caller that named a kernel
 * (amd_matmul_select_kernel) has the GEMMs and the activation launched as the ops this one stands in for launch them. */
extern "C" int amd_up_swiglu(Dataflow_Handle * dataflow_handle, int stream_id, Op * op, void * op_extra) {
	void ** a = op->op_args;
	GemmParams p;
	memset(&p, 0, sizeof(p));
	const int half = *((int *) a[0]);
	p.M = 2 * half;
	p.K = *((int *) a[1]);
	p.N = *((int *) a[2]);
	p.num_groups = *((int *) a[3]);
	p.cumsum = (const int *) *((uint64_t *) a[4]);
	p.A = (const bf16_t *) *((uint64_t *) a[5]);
	const uint64_t strideA_bytes = *((uint64_t *) a[6]);
	p.strideA = (long long) (strideA_bytes / 2);
	p.B = (const bf16_t *) *((uint64_t *) a[7]);
	p.gather = (const int *) *((uint64_t *) a[8]);
	p.gather_rows = *((int *) a[9]);
	p.D = (bf16_t *) *((uint64_t *) a[10]);
	p.h = (bf16_t *) *((uint64_t *) a[11]);
	p.alpha = 1.0f;
	bool aligned = aligned16(p.A) && aligned16(p.B) && aligned16(p.D) && aligned16(p.h) && (strideA_bytes & 15) == 0 && (p.K & 7) == 0 && (half & 7) == 0;
	const bool apart = op->op_skeleton.header.num_args == 13, single = apart && !p.cumsum && !p.gather && p.num_groups == 1;
	if (apart) {
		const uint64_t x3 = *((uint64_t *) a[12]);
		aligned = aligned && (x3 & 15) == 0 && x3 && x3 != (uint64_t) p.D;
		p.x3_apart = ((long long) x3 - (long long) (uint64_t) p.D) / 2;
	}
	if (half < 8 || half > (1 << 24) || p.K < 8 || p.K > (1 << 22) || p.N < 1 || p.num_groups < 1 || !p.A || !p.B || (!single && (!p.cumsum || !p.gather)) || !p.D || !p.h || !aligned
		|| p.gather_rows < 1 || (uint64_t) p.gather_rows * (uint64_t) p.K * 2u > 0xFFFFFFFFull || (uint64_t) (half + 64) * (uint64_t) p.K * 2u > 0xFFFFFFFFull) {
		fprintf(stderr, "Error: bad arguments of the up-projection op (expert dim %d, model dim %d, %d rows, %d groups)...\n", half, p.K, p.N, p.num_groups);
		return -1;
	}
	hipStream_t stream;
	if (resolve_stream(dataflow_handle, stream_id, &stream)) {
		return -1;
	}
	if (hipSetDevice(dataflow_handle->device_id) != hipSuccess) {
		fprintf(stderr, "Error: hipSetDevice failed in the up-projection op...\n");
		return -1;
	}
	const long cu_count = extra_cu_count(op_extra);
	const bool named = kernel_choice != AMD_MATMUL_KERNEL_AUTO;
	if (apart && named) {
		GemmParams one = p, three = p;
		one.M = three.M = half;
		one.x3_apart = three.x3_apart = 0;
		three.A = p.A + (long long) half * p.K;
		three.D = p.D + p.x3_apart;
		if (launch_up_projection(one, single, cu_count, stream) || launch_up_projection(three, single, cu_count, stream)) {
			return -1;
		}
		return launch_up_swiglu(p, half, three.D, half, stream);
	}
	if (single) {
		return launch_direct<false, false, MODE_SINGLE, GATHER_NONE, true>(p, choose_tile(MODE_SINGLE, p, cu_count, false), stream);
	}
	if (apart) {
		return launch_direct<false, false, MODE_RAGGED_N, GATHER_Q_ROWS, true>(p, choose_tile(MODE_RAGGED_N, p, cu_count, false), stream);
	}
	const int tile = choose_tile(MODE_RAGGED_N, p, cu_count);
	if (tile != TILE_BIG && !named) {
		return launch_direct<false, false, MODE_RAGGED_N, GATHER_Q_ROWS, true>(p, tile, stream);
	}
	if (launch_up_projection(p, false, cu_count, stream)) {
		return -1;
	}
	return launch_up_swiglu(p, half, p.D + half, 2 * half, stream);
}

/* The layer's routing in one op (../layer/layer_ops.h): router product, selection, counts, prefix sum, permutation. */
extern "C" int amd_route_tokens(Dataflow_Handle * dataflow_handle, int stream_id, Op * op, void * op_extra) {
	void ** a = op->op_args;
	RouteParams r;
	memset(&r, 0, sizeof(r));
	r.T = *((int *) a[0]);
	r.E = *((int *) a[1]);
	r.K = *((int *) a[2]);
	GemmParams p;
	memset(&p, 0, sizeof(p));
	p.M = r.E;
	p.K = *((int *) a[3]);
	p.N = r.T;
	p.B = (const bf16_t *) *((uint64_t *) a[4]);
	p.A = (const bf16_t *) *((uint64_t *) a[5]);
	p.C = (const bf16_t *) *((uint64_t *) a[6]);
	p.D = (bf16_t *) *((uint64_t *) a[7]);
	p.alpha = 1.0f;
	p.beta = p.C ? 1.0f : 0.0f;
	r.bias = p.C;
	r.x_routed = p.D;
	r.weights = (float *) *((uint64_t *) a[8]);
	r.chosen = (uint16_t *) *((uint64_t *) a[9]);
	r.expert_counts = (int *) *((uint64_t *) a[10]);
	r.expert_counts_cumsum = (int *) *((uint64_t *) a[11]);
	r.host_expert_counts = (int *) *((uint64_t *) a[12]);
	r.expert_mapping = (int *) *((uint64_t *) a[13]);
	r.token_mapping = (int *) *((uint64_t *) a[14]);
	const uint64_t workspace_bytes = *((uint64_t *) a[15]);
	uint8_t * workspace = (uint8_t *) *((uint64_t *) a[16]);

	r.counts_pitch = 16;
	while (r.counts_pitch < r.E) {
		r.counts_pitch *= 2;
	}
	const long blocks = tiles_of(r.T, ROUTE_TOKENS);
	const uint64_t counts_bytes = ((uint64_t) blocks * (uint64_t) r.counts_pitch + 255) & ~255UL;
	if (r.T < 1 || r.E < 1 || r.E > ROUTE_MAX_EXPERTS || r.K < 1 || r.K > r.E || r.K > SELECT_MAX_K || p.K < 1 || !p.A || !p.B || !p.D
		|| blocks * (r.counts_pitch / 16) > 2047L * ROUTE_MAP_THREADS || !workspace || (((uintptr_t) workspace) & 15) || workspace_bytes < counts_bytes) {
		fprintf(stderr, "Error: bad arguments of the routing op (%d tokens, %d experts, top %d, model dim %d, %lu bytes of workspace)...\n",
				r.T, r.E, r.K, p.K, (unsigned long) workspace_bytes);
		return -1;
	}
	hipStream_t stream;
	if (resolve_stream(dataflow_handle, stream_id, &stream)) {
		return -1;
	}
	if (hipSetDevice(dataflow_handle->device_id) != hipSuccess) {
		fprintf(stderr, "Error: hipSetDevice failed in the routing op...\n");
		return -1;
	}
	const long cu_count = extra_cu_count(op_extra);
	const bool direct = operand_direct_ok(p.A, false, p.M, p.K, 0) && operand_direct_ok(p.B, false, p.N, p.K, 0);
	r.counts = workspace;
	/* The product is split where the matmul op splits it, by the whole workspace: another order of the sums would be another
	 * rounding of the logits.  Selection adds up the partial sums itself if the counts fit behind them; if they do not, the
	 * sums are reduced first and the counts then overwrite them. */
	const int split = plan_split(p, 1, 0, direct, (float *) workspace, workspace_bytes, cu_count);
	if (split) {
		if (launch_split(p, split - 1, 1, 0, stream)) {
			return -1;
		}
		const uint64_t partial_bytes = ((uint64_t) p.split_k * (uint64_t) r.T * (uint64_t) r.E * sizeof(float) + 255) & ~255UL;
		if (partial_bytes <= workspace_bytes && counts_bytes <= workspace_bytes - partial_bytes) {
			r.partial = p.partial;
			r.splits = p.split_k;
			r.counts = workspace + partial_bytes;
		} else if (launch_split_reduce(p, stream)) {
			return -1;
		}
	} else if (launch_gemm<MODE_SINGLE>(p, 1, 0, direct, tiles_of(p.M, 256) * tiles_of(p.N, 256), tiles_of(p.M, 128) * tiles_of(p.N, 128), cu_count, stream)) {
		return -1;
	}
	int lanes = 1;                                      /* one slot per lane */
	while (lanes < r.K) {
		lanes *= 2;
	}
	/* Few tokens: selection and permutation in one work-group, one launch less in a chain of which nothing else is left.
	 * Its one compute unit adds up the partial sums at 20-30 GB/s a wave: bounded, so that it stays below a launch. */
	if (r.T <= ROUTE_SMALL_TOKENS && r.T * lanes <= ROUTE_SMALL_THREADS && (long) r.T * r.E * (r.splits > 1 ? r.splits : 1) <= ROUTE_SMALL_PARTIALS) {
		int threads = (r.T * lanes + WAVE - 1) / WAVE * WAVE;
		/* The logits are added up by all its waves, four experts of a token each, before the selection's have work: a wave for every 64 of
		 * those up to eight waves, and sixteen waves beyond 2048.  us, as many as the selection has and so: 32 tokens, 52 experts, top 2 8.1 and 7.0,
		 * 68, 38 and 4 14.2 and 9.7, 256, 64 and 2 17.7 and 13.7; sixteen at 68 tokens 11.0. */
		const long sums = r.T * tiles_of(r.E < ROUTE_CHUNK ? r.E : ROUTE_CHUNK, 4);
		const long wanted = sums > 2048 ? ROUTE_SMALL_THREADS : sums > 512 ? 512 : sums < 256 ? 256 : tiles_of(sums, WAVE) * WAVE;
		threads = threads < wanted ? (int) wanted : threads;
		hipLaunchKernelGGL(route_small_kernel, dim3(1), dim3((unsigned int) threads), 0, stream, r, lanes);
		return check_launch();
	}
	hipLaunchKernelGGL(route_select_kernel, dim3((unsigned int) blocks), dim3((unsigned int) (ROUTE_TOKENS * lanes < 256 ? 256 : ROUTE_TOKENS * lanes)), 0, stream, r, lanes);
	if (check_launch()) {
		return -1;
	}
	hipLaunchKernelGGL(route_map_kernel, dim3((unsigned int) tiles_of(blocks, ROUTE_MAP_WAVES)), dim3(ROUTE_MAP_THREADS), 0, stream, r, (int) blocks);
	return check_launch();
}
