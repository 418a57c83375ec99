/*
 * norm.hip -- RMS norm around the MoE layer: forward, forward from saved statistics, backward w.r.t. the
 * input and w.r.t. the scale (bf16 data, fp32 arithmetic).  Included by hip_kernels.hip after movement.hip.
 *
 * Semantics follow backends/nvidia/src/ops/src/native/src/norm/{rms_norm.cu:226-340, rms_norm_recompute.cu:63-135,
 * rms_norm_bwd_x.cu:241-393, rms_norm_bwd_w.cu:225-324, rms_norm_bwd_w_combine.cu:200-294}:
 *   r[row]   = rsqrt(mean(x^2) + eps)                    (saved in rms_vals: the reciprocal, not the rms)
 *   out      = bf16((x * r) * w)                          in this order of fp32 products
 *   bwd_x:   y = (x * r) * w (fp32, unrounded);  C = sum_i y_i * g_i;
 *            dX_i = bf16(float(dX_i) + r * (g_i * w_i - (C / n) * (x_i * r)));  X_out = bf16(y) if requested
 *   bwd_w:   dW_i = bf16(float(dW_i) + sum_rows g_i * x_i * r[row])   through per-work-group fp32 partial sums
 * Sums run over a row (or over rows) in fp32 in an order the reference leaves to its launch shape; results agree
 * within fp32 rounding of the sums.
 *
 * All kernels are bandwidth-bound: one 256-thread work-group per row (forward and bwd_x: one wave where rows are short
 * and many), 16 bytes per lane per access, the row kept
 * in registers between the reduction and the second use (rows up to 8192 elements; longer rows are read twice).
 * us, forward, bwd_x with X_out and bwd_w of 8192 x 4096 in turn, 604 MB: 113.3 -> 104.7 (5.8 TB/s): dX loaded with x and g instead of
 * behind the sum 109.6, bwd_x's results stored past the caches 106.8, bwd_w's loads in front of the sums of four rows 104.7.  bwd_x from
 * the last row to the first, for what the memory-side cache holds of x, was no faster (114.3).
 */

#include "norm_rows.h"

#define NORM_MAX_VEC 4

__device__ __forceinline__ void add_squares(u32x4 q, float & sum) {
	float f[8];
	unpack8(q, f);
	#pragma unroll
	for (int i = 0; i < 8; i++) {
		sum = __builtin_fmaf(f[i], f[i], sum);
	}
}

__device__ __forceinline__ u32x4 normed(u32x4 x, u32x4 w, float r) {
	float f[8], g[8], y[8];
	unpack8(x, f);
	unpack8(w, g);
	#pragma unroll
	for (int i = 0; i < 8; i++) {
		y[i] = (f[i] * r) * g[i];
	}
	return pack8(y);
}

/* A row of up to 1024 columns on one wave.  On a work-group such a row keeps two of its waves idle or more, and all four meet twice for a sum; here nothing
 * meets and both loads of x and w are out at once.  The vectors of a lane are those that two of the four waves would have, summed by wave and added in
 * their order: the same bits.  us, over sets of arrays beyond the caches, a work-group a row and so: 32768 x 512 26.7 and 14.4, 12000 x 1024 15.0 and 12.5,
 * 8192 x 576 10.2 and 7.0, 8192 x 1024 11.1 and 8.2.  From 2048 columns on (8192 rows 12.1 and 12.4) and with fewer rows (3000 x
 * 1600 5.6 and 6.7) rows on a work-group, which spread over more waves, are the faster ones. */
static_assert(NORM_WAVE_ROWS_PER_GROUP == ROW_WAVES, "a row to each wave of a work-group");
#define NORM_WAVE_ROW_VEC (NORM_WAVE_ROW_COLS / 8 / WAVE)
__device__ __forceinline__ void rms_norm_wave_row(int n_cols, float eps, const u32x4 * x, const u32x4 * __restrict__ w, u32x4 * o, float * rms) {
	const int nvec = n_cols >> 3, lane = threadIdx.x & (WAVE - 1);
	u32x4 keep[NORM_WAVE_ROW_VEC], scale[NORM_WAVE_ROW_VEC];
	#pragma unroll
	for (int j = 0; j < NORM_WAVE_ROW_VEC; j++) {
		if (lane + j * WAVE < nvec) {
			keep[j] = x[lane + j * WAVE];
		}
	}
	#pragma unroll
	for (int j = 0; j < NORM_WAVE_ROW_VEC; j++) {
		if (lane + j * WAVE < nvec) {
			scale[j] = w[lane + j * WAVE];
		}
	}
	/* one wait for all of them: in the branches below it would be for the stores in front as well (100000 x 256 31.5 and 28.5 us) */
	static_assert(NORM_WAVE_ROW_VEC == 2, "the vectors named here");
	asm volatile("" : "+v"(keep[0]), "+v"(keep[1]), "+v"(scale[0]), "+v"(scale[1]));
	float sum = 0.0f;
	#pragma unroll
	for (int j = 0; j < NORM_WAVE_ROW_VEC; j++) {
		if (j * WAVE < nvec) {                           /* uniform */
			float part = 0.0f;
			if (lane + j * WAVE < nvec) {
				add_squares(keep[j], part);
			}
			sum += wave_sum(part);
		}
	}
	const float r = rsqrtf(sum * (1.0f / (float) n_cols) + eps);
	if (lane == 0 && rms) {
		*rms = r;
	}
	#pragma unroll
	for (int j = 0; j < NORM_WAVE_ROW_VEC; j++) {
		if (lane + j * WAVE < nvec) {
			o[lane + j * WAVE] = normed(keep[j], scale[j], r);
		}
	}
}

/* Many long rows, one on a work-group: all loads of a lane's first four vectors are out before the first is waited for, those of w in front of the sum's
 * barriers.  The loop in the kernel below, a round trip to memory a vector twice over, stays for rows of up to 4608 columns, where it is
 * the faster one (2048 x 2048 4.8 and 5.0 us), and for fewer rows: at 2048 x 8192 this form is the faster one too (11.7 and 11.2), but the three norm
 * passes together, over arrays that just miss the memory-side cache, took 62.2 and 63.6.  us, that loop and this form: 8192 x 4672 30.9 and
 * 28.4, 20000 x 5120 75.0 and 71.7, 3000 x 7232 15.5 and 14.5, 2500 x 8192 14.4 and 14.2, 8192 x 8192 52.9 and 47.9, 32768 x 8192 185 and 183, 3000 x 10048 23.3
 * and 22.2.  62 registers: eight work-groups a compute unit, as before. */
__device__ __forceinline__ void rms_norm_unrolled_row(int n_cols, float eps, const u32x4 * x, const u32x4 * __restrict__ w, u32x4 * o, float * rms, float * scratch) {
	const int nvec = n_cols >> 3;
	u32x4 keep[NORM_MAX_VEC], scale[NORM_MAX_VEC];
	float part[1] = {0.0f};
	#pragma unroll
	for (int j = 0; j < NORM_MAX_VEC; j++) {
		const int v = threadIdx.x + j * ROW_THREADS;
		if (v < nvec) {
			keep[j] = x[v];
		}
	}
	__builtin_amdgcn_sched_barrier(0);                      /* the loads of x are out before the first is waited for */
	#pragma unroll
	for (int j = 0; j < NORM_MAX_VEC; j++) {
		if ((int) (threadIdx.x + j * ROW_THREADS) < nvec) {
			add_squares(keep[j], part[0]);
		}
	}
	#pragma unroll 1
	for (int v = threadIdx.x + NORM_MAX_VEC * ROW_THREADS; v < nvec; v += ROW_THREADS) {
		add_squares(x[v], part[0]);
	}
	#pragma unroll
	for (int j = 0; j < NORM_MAX_VEC; j++) {
		const int v = threadIdx.x + j * ROW_THREADS;
		if (v < nvec) {
			scale[j] = w[v];
		}
	}
	block_sum<1>(part, scratch);
	const float r = rsqrtf(part[0] * (1.0f / (float) n_cols) + eps);
	if (threadIdx.x == 0 && rms) {
		*rms = r;
	}
	#pragma unroll
	for (int j = 0; j < NORM_MAX_VEC; j++) {
		const int v = threadIdx.x + j * ROW_THREADS;
		if (v < nvec) {
			o[v] = normed(keep[j], scale[j], r);
		}
	}
	#pragma unroll 1
	for (int v = threadIdx.x + NORM_MAX_VEC * ROW_THREADS; v < nvec; v += ROW_THREADS) {
		o[v] = normed(x[v], w[v], r);
	}
}

/* r[row], out = bf16((x * r) * w).  Launch: grid = n_rows, block = 256.
 * Algorithmic HBM bytes: 2*n_rows*n_cols read, 2*n_rows*n_cols + 4*n_rows written (w stays in cache). */
extern "C" __global__ void __launch_bounds__(ROW_THREADS)
default_rms_norm_bf16_kernel(int n_rows, int n_cols, float eps, const bf16_t * __restrict__ rms_weight,
							 const bf16_t * __restrict__ X, bf16_t * __restrict__ out, float * __restrict__ rms_vals) {
	__shared__ float scratch[ROW_WAVES];
	const int row = blockIdx.x;
	if (row >= n_rows) {
		return;
	}
	const int nvec = n_cols >> 3;
	const u32x4 * x = (const u32x4 *) (X + (size_t) row * n_cols);
	u32x4 * o = (u32x4 *) (out + (size_t) row * n_cols);
	const u32x4 * w = (const u32x4 *) rms_weight;

	u32x4 keep[NORM_MAX_VEC];
	float part[1] = {0.0f};
	int j = 0;
	for (int v = threadIdx.x; v < nvec; v += ROW_THREADS, j++) {
		const u32x4 q = x[v];
		if (j < NORM_MAX_VEC) {
			keep[j] = q;
		}
		float f[8];
		unpack8(q, f);
		#pragma unroll
		for (int i = 0; i < 8; i++) {
			part[0] = __builtin_fmaf(f[i], f[i], part[0]);
		}
	}
	block_sum<1>(part, scratch);
	const float r = rsqrtf(part[0] * (1.0f / (float) n_cols) + eps);
	if (threadIdx.x == 0 && rms_vals) {
		rms_vals[row] = r;
	}
	j = 0;
	for (int v = threadIdx.x; v < nvec; v += ROW_THREADS, j++) {
		float f[8], g[8], y[8];
		unpack8(j < NORM_MAX_VEC ? keep[j] : x[v], f);
		unpack8(w[v], g);
		#pragma unroll
		for (int i = 0; i < 8; i++) {
			y[i] = (f[i] * r) * g[i];
		}
		o[v] = pack8(y);
	}
}

/* The two forms are kernels of their own, submitted in the place of the one above (../ops/dataflow_ops.c, norm_rows.h).  As branches of it their two tests,
 * a dozen scalar instructions in front of a row's first load, made every other launch the slower one: us, without and with them, 26970 x 1344 33.5 and
 * 34.6, 9000 x 1344 13.9 and 14.3, 8000 x 1024 11.1 and 11.5, 8192 x 4096 26.0 and 26.2, 20000 x 3072 47.0 and 47.5 (one test costs nothing, the
 * cheapest arrangement of two 0.1-2.6 %; the 62 registers of the long form cost it nothing).  Launch: block = 256, grid = a quarter of n_rows, rounded up,
 * and n_rows. */
extern "C" __global__ void __launch_bounds__(ROW_THREADS)
amd_rms_norm_wave_rows_bf16_kernel(int n_rows, int n_cols, float eps, const bf16_t * __restrict__ rms_weight,
								   const bf16_t * __restrict__ X, bf16_t * __restrict__ out, float * __restrict__ rms_vals) {
	const int row = (int) (blockIdx.x * ROW_WAVES) + __builtin_amdgcn_readfirstlane((int) (threadIdx.x / WAVE));
	if (row < n_rows) {
		rms_norm_wave_row(n_cols, eps, (const u32x4 *) (X + (size_t) row * n_cols), (const u32x4 *) rms_weight, (u32x4 *) (out + (size_t) row * n_cols),
						  rms_vals ? rms_vals + row : nullptr);
	}
}

extern "C" __global__ void __launch_bounds__(ROW_THREADS)
amd_rms_norm_long_rows_bf16_kernel(int n_rows, int n_cols, float eps, const bf16_t * __restrict__ rms_weight,
								   const bf16_t * __restrict__ X, bf16_t * __restrict__ out, float * __restrict__ rms_vals) {
	__shared__ float scratch[ROW_WAVES];
	const int row = blockIdx.x;
	if (row < n_rows) {
		rms_norm_unrolled_row(n_cols, eps, (const u32x4 *) (X + (size_t) row * n_cols), (const u32x4 *) rms_weight, (u32x4 *) (out + (size_t) row * n_cols),
							  rms_vals ? rms_vals + row : nullptr, scratch);
	}
}

/* out = bf16((x * r) * w) with r read from rms_vals.  Launch: grid = n_rows, block = 256. */
extern "C" __global__ void __launch_bounds__(ROW_THREADS)
default_rms_norm_recompute_bf16_kernel(int n_rows, int n_cols, const bf16_t * __restrict__ rms_weight,
									   const float * __restrict__ rms_vals, const bf16_t * __restrict__ X, bf16_t * __restrict__ out) {
	const int row = blockIdx.x;
	if (row >= n_rows) {
		return;
	}
	const int nvec = n_cols >> 3;
	const float r = rms_vals[row];
	const u32x4 * x = (const u32x4 *) (X + (size_t) row * n_cols);
	u32x4 * o = (u32x4 *) (out + (size_t) row * n_cols);
	const u32x4 * w = (const u32x4 *) rms_weight;
	for (int v = threadIdx.x; v < nvec; v += ROW_THREADS) {
		float f[8], g[8], y[8];
		unpack8(x[v], f);
		unpack8(w[v], g);
		#pragma unroll
		for (int i = 0; i < 8; i++) {
			y[i] = (f[i] * r) * g[i];
		}
		o[v] = pack8(y);
	}
}

/* Backward w.r.t. the input, accumulated into dX; X_out (nullable) receives the recomputed forward output.
 * Launch: grid = n_rows, block = 256.
 * Algorithmic HBM bytes: 6*n_rows*n_cols read (x, g, dX), 2*n_rows*n_cols written (+2*n_rows*n_cols for X_out).
 *
 * Two forms, by the rows.  A compute unit holds six of the work-groups (80 registers: the row's x, g and dX stay in them), 256 compute units
 * 1536.  Beyond that, MANY_ROWS, rows wait for their sums while others load: dX is loaded with x and g, behind the scale, as loads come
 * back in order and the sum would wait for dX too; results pass the caches by.  Up to 1536 rows everything is in flight at once,
 * an early load of dX has nothing to hide behind, and the next kernel finds what was stored in the memory-side cache: dX behind the sum,
 * plain stores.  us, forward, bwd_x and bwd_w in turn over one set of arrays, few-rows form and the other: 1120 x 7232 34.1 and 35.5, 1536 x
 * 6144 39.6 and 40.8, 2048 x 8192 64.1 and 62.4, 8192 x 4096 102.3 and 99.6, over eight sets 71.5 and 65.9 for 2048 x 8192, 113.0 and 104.8
 * for 8192 x 4096.  At 83 registers, five work-groups a compute unit, and with dX in front of the scale the other form took 36.2 at 1120 x 7232,
 * 79.2 at 3000 x 7232 (77.6 now).  Left: 1537 to 1792 rows, which the few-rows form alone, 67 registers, would hold at once: 2-6 % slower than there
 * when all arrays are in the caches, within 2 % when none is (from 4096 columns on). */
#define BWD_X_FEW_ROWS (6 * 256)
template <bool MANY_ROWS>
__device__ __forceinline__ void
rms_norm_bwd_x_row(int n_cols, float r, const u32x4 * __restrict__ x, const u32x4 * __restrict__ g, const u32x4 * __restrict__ w, u32x4 * d, u32x4 * xo, float * scratch) {
	const int nvec = n_cols >> 3;
	u32x4 keep_x[NORM_MAX_VEC], keep_g[NORM_MAX_VEC], keep_d[NORM_MAX_VEC];
	float part[1] = {0.0f};
	int j = 0;
	for (int v = threadIdx.x; v < nvec; v += ROW_THREADS, j++) {
		const u32x4 qx = x[v];
		const u32x4 qg = __builtin_nontemporal_load(g + v);
		const u32x4 qw = w[v];
		__builtin_amdgcn_sched_barrier(0);              /* loads come back in order: dX's behind what the sum needs */
		if (j < NORM_MAX_VEC) {
			keep_x[j] = qx;
			keep_g[j] = qg;
			if (MANY_ROWS) {
				keep_d[j] = d[v];
			}
		}
		float fx[8], fg[8], fw[8], y[8];
		unpack8(qx, fx);
		unpack8(qg, fg);
		unpack8(qw, fw);
		#pragma unroll
		for (int i = 0; i < 8; i++) {
			y[i] = (fx[i] * r) * fw[i];
			part[0] = __builtin_fmaf(y[i], fg[i], part[0]);
		}
		if (xo) {
			if (MANY_ROWS) {
				__builtin_nontemporal_store(pack8(y), xo + v);
			} else {
				xo[v] = pack8(y);
			}
		}
	}
	block_sum<1>(part, scratch);
	const float c_div_n = part[0] / (float) n_cols;
	j = 0;
	for (int v = threadIdx.x; v < nvec; v += ROW_THREADS, j++) {
		float fx[8], fg[8], fw[8], fd[8];
		unpack8(j < NORM_MAX_VEC ? keep_x[j] : x[v], fx);
		unpack8(j < NORM_MAX_VEC ? keep_g[j] : g[v], fg);
		unpack8(w[v], fw);
		unpack8(MANY_ROWS && j < NORM_MAX_VEC ? keep_d[j] : d[v], fd);
		#pragma unroll
		for (int i = 0; i < 8; i++) {
			fd[i] += r * (fg[i] * fw[i] - c_div_n * (fx[i] * r));
		}
		if (MANY_ROWS) {
			__builtin_nontemporal_store(pack8(fd), d + v);
		} else {
			d[v] = pack8(fd);
		}
	}
}

/* The same for a row on one wave, as in the forward (rms_norm_wave_row), all of its loads out at once.  us, over sets of arrays beyond the caches, a row on
 * a work-group and so: 32768 x 512 41.0 and 29.3, 12000 x 1024 24.2 and 23.3, 8192 x 576 14.8 and 11.4, 8192 x 1024 18.4 and 17.1.  The row's number is made uniform: its
 * addresses stay in scalar registers. */
__device__ __forceinline__ void
rms_norm_bwd_x_wave_row(int n_cols, float r, const u32x4 * __restrict__ x, const u32x4 * __restrict__ g, const u32x4 * __restrict__ w, u32x4 * d, u32x4 * xo) {
	const int nvec = n_cols >> 3, lane = threadIdx.x & (WAVE - 1);
	u32x4 qx[NORM_WAVE_ROW_VEC], qg[NORM_WAVE_ROW_VEC], qw[NORM_WAVE_ROW_VEC], qd[NORM_WAVE_ROW_VEC];
	#pragma unroll
	for (int j = 0; j < NORM_WAVE_ROW_VEC; j++) {
		const int v = lane + j * WAVE;
		if (v < nvec) {
			qx[j] = x[v];
			qg[j] = __builtin_nontemporal_load(g + v);
			qw[j] = w[v];
			qd[j] = d[v];
		}
	}
	float sum = 0.0f;
	#pragma unroll
	for (int j = 0; j < NORM_WAVE_ROW_VEC; j++) {
		const int v = lane + j * WAVE;
		if (j * WAVE < nvec) {                           /* uniform */
			float part = 0.0f;
			if (v < nvec) {
				float fx[8], fg[8], fw[8], y[8];
				unpack8(qx[j], fx);
				unpack8(qg[j], fg);
				unpack8(qw[j], fw);
				#pragma unroll
				for (int i = 0; i < 8; i++) {
					y[i] = (fx[i] * r) * fw[i];
					part = __builtin_fmaf(y[i], fg[i], part);
				}
				if (xo) {
					__builtin_nontemporal_store(pack8(y), xo + v);
				}
			}
			sum += wave_sum(part);
		}
	}
	const float c_div_n = sum / (float) n_cols;
	#pragma unroll
	for (int j = 0; j < NORM_WAVE_ROW_VEC; j++) {
		const int v = lane + j * WAVE;
		if (v < nvec) {
			float fx[8], fg[8], fw[8], fd[8];
			unpack8(qx[j], fx);
			unpack8(qg[j], fg);
			unpack8(qw[j], fw);
			unpack8(qd[j], fd);
			#pragma unroll
			for (int i = 0; i < 8; i++) {
				fd[i] += r * (fg[i] * fw[i] - c_div_n * (fx[i] * r));
			}
			__builtin_nontemporal_store(pack8(fd), d + v);
		}
	}
}

extern "C" __global__ void __launch_bounds__(ROW_THREADS)
default_rms_norm_bwd_x_bf16_bf16_kernel(int n_rows, int n_cols, float eps, const float * __restrict__ fwd_rms_vals,
										const bf16_t * __restrict__ rms_weight, const bf16_t * __restrict__ X_inp,
										const bf16_t * __restrict__ upstream_dX, bf16_t * dX, bf16_t * X_out) {
	__shared__ float scratch[ROW_WAVES];
	(void) eps;
	const int row = blockIdx.x;
	if (row >= n_rows) {
		return;
	}
	const float r = fwd_rms_vals[row];
	const u32x4 * x = (const u32x4 *) (X_inp + (size_t) row * n_cols);
	const u32x4 * g = (const u32x4 *) (upstream_dX + (size_t) row * n_cols);
	const u32x4 * w = (const u32x4 *) rms_weight;
	u32x4 * d = (u32x4 *) (dX + (size_t) row * n_cols);
	u32x4 * xo = X_out ? (u32x4 *) (X_out + (size_t) row * n_cols) : nullptr;
	if (n_rows > BWD_X_FEW_ROWS) {
		rms_norm_bwd_x_row<true>(n_cols, r, x, g, w, d, xo, scratch);
	} else {
		rms_norm_bwd_x_row<false>(n_cols, r, x, g, w, d, xo, scratch);
	}
}

/* a row on a wave, in a kernel of its own, as in the forward; launch: grid = a quarter of n_rows, block = 256 */
extern "C" __global__ void __launch_bounds__(ROW_THREADS)
amd_rms_norm_bwd_x_wave_rows_bf16_bf16_kernel(int n_rows, int n_cols, const float * __restrict__ fwd_rms_vals,
											  const bf16_t * __restrict__ rms_weight, const bf16_t * __restrict__ X_inp,
											  const bf16_t * __restrict__ upstream_dX, bf16_t * dX, bf16_t * X_out) {
	const int row = (int) (blockIdx.x * ROW_WAVES) + __builtin_amdgcn_readfirstlane((int) (threadIdx.x / WAVE));
	if (row < n_rows) {
		const size_t at = (size_t) row * n_cols;
		rms_norm_bwd_x_wave_row(n_cols, fwd_rms_vals[row], (const u32x4 *) (X_inp + at), (const u32x4 *) (upstream_dX + at), (const u32x4 *) rms_weight,
								(u32x4 *) (dX + at), X_out ? (u32x4 *) (X_out + at) : nullptr);
	}
}

/* Backward w.r.t. the scale, first half: work-group b sums g * x * r over its share of the rows (a contiguous
 * range, as in the reference) into dW_workspace[b][n_cols] (fp32) and records the number of work-groups.
 * Launch: grid x <= n_rows (chosen so that the workspace holds grid.x * n_cols floats), grid y = column slabs of
 * 2048, block = 256: every thread owns 8 columns and walks down its work-group's rows, four at a time: left to itself the compiler keeps
 * two or three loads in flight (30 registers) and not eight.  Eight rows at a time take the same 104.7 us in the sequence above.
 * Algorithmic HBM bytes: 4*n_rows*n_cols read, 4*grid*n_cols written. */
#define BWD_W_ROWS 4
/* From this row length on the rows go one by one, by the loop that the compiler leaves two or three loads in flight: us alone, one by one
 * and in fours, 8192 x 4480 33.4 and 31.7, 16384 x 4544 55.8 and 54.9, 16384 x 4608 56.2 and 55.7 (from memory 56.1 and 56.7), 16384 x 5120 58.7
 * and 62.1, 32768 x 6144 127 and 137, 32768 x 8192 166 and 185. */
#define BWD_W_FOURS_COLS 4608
extern "C" __global__ void __launch_bounds__(ROW_THREADS)
default_rms_norm_bwd_w_bf16_bf16_kernel(int n_rows, int n_cols, float eps, const float * __restrict__ fwd_rms_vals,
										const bf16_t * __restrict__ X_inp, const bf16_t * __restrict__ upstream_dX,
										float * __restrict__ dW_workspace, int * __restrict__ ret_num_blocks_launched) {
	(void) eps;
	if (blockIdx.x == 0 && threadIdx.x == 0) {
		*ret_num_blocks_launched = (int) gridDim.x;
	}
	const int b = blockIdx.x;
	int rows = n_rows / (int) gridDim.x;
	const int extra = n_rows % (int) gridDim.x;
	int first;
	if (b < extra) {
		rows += 1;
		first = b * rows;
	} else {
		first = b * rows + extra;
	}
	const int nvec = n_cols >> 3;
	typedef float f32x4 __attribute__((ext_vector_type(4)));
	const int v = blockIdx.y * ROW_THREADS + threadIdx.x;   /* one 8-column vector per thread, column slabs along grid y */
	if (v >= nvec) {
		return;
	}
	float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
	const u32x4 * x = (const u32x4 *) (X_inp + (size_t) first * n_cols) + v;
	const u32x4 * g = (const u32x4 *) (upstream_dX + (size_t) first * n_cols) + v;
	int i = 0;
	for (; n_cols < BWD_W_FOURS_COLS && i + BWD_W_ROWS <= rows; i += BWD_W_ROWS) {
		u32x4 qx[BWD_W_ROWS], qg[BWD_W_ROWS];
		float r[BWD_W_ROWS];
		#pragma unroll
		for (int k = 0; k < BWD_W_ROWS; k++) {
			qx[k] = __builtin_nontemporal_load(x + (size_t) (i + k) * nvec);
			qg[k] = __builtin_nontemporal_load(g + (size_t) (i + k) * nvec);
			r[k] = fwd_rms_vals[first + i + k];
		}
		__builtin_amdgcn_sched_barrier(0);              /* the loads stay in front of the sums */
		#pragma unroll
		for (int k = 0; k < BWD_W_ROWS; k++) {
			float fx[8], fg[8];
			unpack8(qx[k], fx);
			unpack8(qg[k], fg);
			#pragma unroll
			for (int e = 0; e < 8; e++) {
				acc[e] += (fg[e] * fx[e]) * r[k];
			}
		}
	}
	#pragma unroll 8
	for (; i < rows; i++) {
		const float r = fwd_rms_vals[first + i];
		float fx[8], fg[8];
		unpack8(__builtin_nontemporal_load(x + (size_t) i * nvec), fx);
		unpack8(__builtin_nontemporal_load(g + (size_t) i * nvec), fg);
		#pragma unroll
		for (int e = 0; e < 8; e++) {
			acc[e] += (fg[e] * fx[e]) * r;
		}
	}
	f32x4 * dst = (f32x4 *) (dW_workspace + (size_t) b * n_cols + (size_t) v * 8);
	dst[0] = f32x4{acc[0], acc[1], acc[2], acc[3]};
	dst[1] = f32x4{acc[4], acc[5], acc[6], acc[7]};
}

/* Second half: dW_i = bf16(float(dW_i) + sum over the recorded work-groups of dW_workspace[b][i]).
 * Launch: grid = ceil(model_dim / 64), block = 1024: a work-group owns 64 columns, each of its 16 waves sums a
 * sixteenth of the partial rows (lanes along the columns, so reads are contiguous; the loads of a wave are
 * independent of each other), then the waves are added.  The kernel is latency-bound: a few dependent rounds. */
#define COMBINE_WAVES 16
extern "C" __global__ void __launch_bounds__(COMBINE_WAVES * WAVE)
default_rms_norm_bwd_w_combine_bf16_kernel(const int * __restrict__ num_orig_blocks_launched, int model_dim,
										   const float * __restrict__ dW_workspace, bf16_t * dW) {
	__shared__ float partial[COMBINE_WAVES][WAVE];
	const int lane = threadIdx.x & (WAVE - 1);
	const int wave = threadIdx.x / WAVE;
	const int col = blockIdx.x * WAVE + lane;
	const int nb = *num_orig_blocks_launched;
	float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
	if (col < model_dim) {
		int b = wave;
		for (; b + 3 * COMBINE_WAVES < nb; b += 4 * COMBINE_WAVES) {
			s0 += dW_workspace[(size_t) b * model_dim + col];
			s1 += dW_workspace[(size_t) (b + COMBINE_WAVES) * model_dim + col];
			s2 += dW_workspace[(size_t) (b + 2 * COMBINE_WAVES) * model_dim + col];
			s3 += dW_workspace[(size_t) (b + 3 * COMBINE_WAVES) * model_dim + col];
		}
		for (; b < nb; b += COMBINE_WAVES) {
			s0 += dW_workspace[(size_t) b * model_dim + col];
		}
	}
	partial[wave][lane] = (s0 + s1) + (s2 + s3);
	__syncthreads();
	if (wave == 0 && col < model_dim) {
		float t = bf16_to_f32(dW[col]);
		#pragma unroll
		for (int w = 0; w < COMBINE_WAVES; w++) {
			t += partial[w][lane];
		}
		dW[col] = f32_to_bf16(t);
	}
}

/* Both halves in one launch, for few rows: a work-group owns 64 columns and all rows.  Each of its 128 groups of eight lanes
 * takes every 128th row (128 contiguous bytes a row), the sums of the groups are added through the LDS and on to dW.  The two
 * launches it replaces are bound by their submission, 3.7 us each, and the second by its 512 partial rows; this one by the
 * load path of a compute unit, which each row takes 256 bytes through: 4.0 us up to 768 rows (7.4-11.6 before), 4.7 at 1024 x
 * 2048 (9.2).  More rows are left to the two launches, which spread them over all compute units.
 * Launch: grid = ceil(n_cols / 64), block = 1024.
 * `blocks`: what the two-launch form records as its number of work-groups, recorded here for callers that read it. */
#define FEW_ROWS_LANES 128
extern "C" __global__ void __launch_bounds__(FEW_ROWS_LANES * 8)
amd_rms_norm_bwd_w_few_rows_bf16_bf16_kernel(int n_rows, int n_cols, const float * __restrict__ fwd_rms_vals, const bf16_t * __restrict__ X_inp,
											 const bf16_t * __restrict__ upstream_dX, bf16_t * dW, int blocks, int * __restrict__ ret_num_blocks_launched) {
	__shared__ float partial[FEW_ROWS_LANES][WAVE + 1];
	__shared__ float wave_sum[COMBINE_WAVES][WAVE];
	static_assert(FEW_ROWS_LANES * 8 == COMBINE_WAVES * WAVE, "sixteen waves add up the partial sums");
	if (blockIdx.x == 0 && threadIdx.x == 0) {
		*ret_num_blocks_launched = blocks;
	}
	const int row_lane = threadIdx.x >> 3;
	const int nvec = n_cols >> 3;
	const int v = blockIdx.x * 8 + (threadIdx.x & 7);
	float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
	if (v < nvec) {
		#pragma unroll 4
		for (int row = row_lane; row < n_rows; row += FEW_ROWS_LANES) {
			const size_t off = (size_t) row * n_cols;
			const float r = fwd_rms_vals[row];
			float fx[8], fg[8];
			unpack8(((const u32x4 *) (X_inp + off))[v], fx);
			unpack8(((const u32x4 *) (upstream_dX + off))[v], fg);
			#pragma unroll
			for (int e = 0; e < 8; e++) {
				acc[e] += (fg[e] * fx[e]) * r;
			}
		}
	}
	#pragma unroll
	for (int e = 0; e < 8; e++) {
		partial[row_lane][(threadIdx.x & 7) * 8 + e] = acc[e];
	}
	__syncthreads();
	const int lane = threadIdx.x & (WAVE - 1);
	const int wave = threadIdx.x / WAVE;
	float sum = 0.0f;
	#pragma unroll
	for (int i = 0; i < FEW_ROWS_LANES / COMBINE_WAVES; i++) {
		sum += partial[wave * (FEW_ROWS_LANES / COMBINE_WAVES) + i][lane];
	}
	wave_sum[wave][lane] = sum;
	__syncthreads();
	const int col = blockIdx.x * WAVE + lane;
	if (wave == 0 && col < n_cols) {
		float t = bf16_to_f32(dW[col]);
		#pragma unroll
		for (int w = 0; w < COMBINE_WAVES; w++) {
			t += wave_sum[w][lane];
		}
		dW[col] = f32_to_bf16(t);
	}
}
