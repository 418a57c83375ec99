/*
 * route_kernel.h -- the layer's routing between the router's matrix product and the expert GEMMs, for gfx950: top-k
 * selection, per-expert counts, their prefix sum and the dispatch permutation (see amd_route_tokens in amd_matmul.hip).
 *
 * Same results, bit for bit, as the ops it stands in for (router matmul, fill, select_experts, build_expert_mapping:
 * dataflow_transformer.c:2710-2784).  Those are five or six launches of 3-25 us each, none of which moves enough bytes
 * to matter: what they cost is the chain of launches, a device-wide ticket behind atomics, and a pass of every work-group
 * over all chosen ids.  Here the selection takes the split-K partial sums of the router product directly (no reduction
 * pass), leaves one byte per expert and block of 32 tokens instead of adding to device-wide counters (nothing to clear,
 * no ticket), and the mapping kernel gets totals and its own starting positions from those bytes.
 *
 * Behind the router product, kernel times: T 8192, E 32, K 4: 42 -> 21 us (reduction, fill, selection and mapping before);
 * T 65536, E 64, K 8: 163 -> 53; T 256, E 8, K 2: 25 -> 7, in one launch; T 16, E 64, K 8: 34 -> 12.
 */
#ifndef ROUTE_KERNEL_H
#define ROUTE_KERNEL_H

#include "../kernels/select_walk.h"

#define ROUTE_TOKENS 32                     /* tokens per selection block: a count fits a byte */
#define ROUTE_CHUNK 64                      /* experts staged in LDS per pass */
#define ROUTE_ROW_DWORDS (ROUTE_CHUNK / 2 + 1)
#define ROUTE_MAX_EXPERTS 512
#define ROUTE_SMALL_TOKENS 256              /* single-work-group form: at most this many tokens ... */
#define ROUTE_SMALL_THREADS 1024            /* ... and tokens x lanes */
#define ROUTE_SMALL_PARTIALS (1 << 16)      /* ... and partial sums to add up (floats) */
#define ROUTE_MAP_THREADS 256
#define ROUTE_MAP_WAVES (ROUTE_MAP_THREADS / WAVE)
#define ROUTE_MAP_AHEAD 4                   /* 64-entry steps whose ids are fetched up front: all of a block for K <= 8 */

struct RouteParams {
	int T, E, K;
	int counts_pitch;                       /* bytes per block of `counts`: the power of two >= max(E, 16) */
	const float * partial;                  /* [splits][T][E] partial sums of the router product; NULL: the logits are in x_routed */
	int splits;
	const bf16_t * bias;                    /* [T][E], or NULL */
	bf16_t * x_routed;                      /* [T][E] logits */
	float * weights;                        /* [T][K] */
	uint16_t * chosen;                      /* [T][K] */
	uint8_t * counts;                       /* [blocks of ROUTE_TOKENS tokens][counts_pitch] rows per expert */
	int * expert_counts;                    /* [E + 1]; the last entry is select_experts' ticket: its number of work-groups */
	int * expert_counts_cumsum;             /* [E] inclusive */
	int * host_expert_counts;               /* [E] device-visible host memory */
	int * expert_mapping;                   /* [T * K] */
	int * token_mapping;                    /* [T][K] */
};

/* Logits of tokens [t0, t0 + tokens) x experts [c0, c0 + ROUTE_CHUNK) as sort keys into `tile` (ROUTE_ROW_DWORDS dwords per
 * token, two keys each; the partner of an odd last expert is -inf).  With partial sums: the logit is bf16(sum over the
 * splits, in their order, + bias), what the split product's reduction pass writes, and is stored to x_routed on the way.
 * A lane adds up four experts each of AHEAD tokens, SPLITS loads apiece in flight: the chain of loads behind each other,
 * not their bytes, is what this takes (16 loads one after the other: 12 us for 16 tokens). */
template <int AHEAD, int SPLITS>
__device__ __forceinline__ void route_stage_quads(const RouteParams & p, uint32_t * __restrict__ tile, int t0, int quads, int items, int c0) {
	const long long count = (long long) p.T * p.E;
	const bool whole = (p.E & 3) == 0;                   /* then a quad is whole, and aligned in the partial sums */
	const bool whole_logits = whole && (((uintptr_t) p.x_routed) & 7) == 0;
	const float * __restrict__ partial = p.partial;
	for (int i0 = threadIdx.x; i0 < items; i0 += AHEAD * (int) blockDim.x) {
		long long at[AHEAD];
		float sum[AHEAD][4];
		#pragma unroll
		for (int u = 0; u < AHEAD; u++) {
			const int i = min(i0 + u * (int) blockDim.x, items - 1);
			const int r = i / quads;
			at[u] = (long long) (t0 + r) * p.E + c0 + 4 * (i - r * quads);
			sum[u][0] = sum[u][1] = sum[u][2] = sum[u][3] = 0.0f;
		}
		if (partial && whole) {
			for (int s0 = 0; s0 < p.splits; s0 += SPLITS) {
				f32x4_t q[SPLITS][AHEAD];
				#pragma unroll
				for (int s = 0; s < SPLITS; s++) {
					#pragma unroll
					for (int u = 0; u < AHEAD; u++) {
						q[s][u] = *((const f32x4_t *) (partial + (long long) min(s0 + s, p.splits - 1) * count + at[u]));
					}
				}
				#pragma unroll
				for (int s = 0; s < SPLITS; s++) {
					if (s0 + s < p.splits) {
						#pragma unroll
						for (int u = 0; u < AHEAD; u++) {
							sum[u][0] += q[s][u].x;
							sum[u][1] += q[s][u].y;
							sum[u][2] += q[s][u].z;
							sum[u][3] += q[s][u].w;
						}
					}
				}
			}
		} else if (partial) {
			/* rows that are no whole quads: element loads, as many in flight (55 experts, 80 tokens: 19 us one split behind the other) */
			const long long last = (long long) p.splits * count - 1;
			for (int s0 = 0; s0 < p.splits; s0 += SPLITS) {
				float q[SPLITS][AHEAD][4];
				#pragma unroll
				for (int s = 0; s < SPLITS; s++) {
					#pragma unroll
					for (int u = 0; u < AHEAD; u++) {
						#pragma unroll
						for (int j = 0; j < 4; j++) {
							q[s][u][j] = partial[min((long long) min(s0 + s, p.splits - 1) * count + at[u] + j, last)];      /* past the row's end: not used */
						}
					}
				}
				#pragma unroll
				for (int s = 0; s < SPLITS; s++) {
					if (s0 + s < p.splits) {
						#pragma unroll
						for (int u = 0; u < AHEAD; u++) {
							#pragma unroll
							for (int j = 0; j < 4; j++) {
								sum[u][j] += q[s][u][j];
							}
						}
					}
				}
			}
		}
		#pragma unroll
		for (int u = 0; u < AHEAD; u++) {
			const int i = i0 + u * (int) blockDim.x;
			if (i < items) {
				const int r = i / quads, c = 4 * (i - r * quads);
				uint32_t bits[4];
				#pragma unroll
				for (int j = 0; j < 4; j++) {
					bits[j] = 0xFF80u;
					if (c0 + c + j < p.E) {
						if (partial) {
							float v = sum[u][j];
							if (p.bias) {
								v += bf16_to_f32(p.bias[at[u] + j]);
							}
							bits[j] = f32_to_bf16(v);
						} else {
							bits[j] = p.x_routed[at[u] + j];
						}
					}
				}
				const uint32_t lo = bits[0] | (bits[1] << 16), hi = bits[2] | (bits[3] << 16);
				if (partial) {
					if (whole_logits) {
						*((u32x2 *) (p.x_routed + at[u])) = u32x2{lo, hi};
					} else {
						#pragma unroll
						for (int j = 0; j < 4; j++) {
							if (c0 + c + j < p.E) {
								p.x_routed[at[u] + j] = (bf16_t) bits[j];
							}
						}
					}
				}
				tile[r * ROUTE_ROW_DWORDS + c / 2] = sort_key_pair(lo);
				tile[r * ROUTE_ROW_DWORDS + c / 2 + 1] = sort_key_pair(hi);
			}
		}
	}
}

__device__ __forceinline__ void route_stage(const RouteParams & p, uint32_t * tile, int t0, int tokens, int c0) {
	const int quads = (min(ROUTE_CHUNK, p.E - c0) + 3) >> 2;
	const int items = min(tokens, p.T - t0) * quads;
	if (items <= (int) blockDim.x) {
		route_stage_quads<1, 8>(p, tile, t0, quads, items, c0);
	} else if (items <= 2 * (int) blockDim.x) {
		route_stage_quads<2, 4>(p, tile, t0, quads, items, c0);
	} else {
		route_stage_quads<4, 2>(p, tile, t0, quads, items, c0);
	}
}

/* selection for the work-group's tokens (one group of LANES lanes each); returns this lane's expert */
template <int LANES>
__device__ __forceinline__ int route_select(const RouteParams & p, uint32_t * tile, int t0, int tokens) {
	const int group = threadIdx.x / LANES;
	const int slot = threadIdx.x % LANES;
	SelectSlot<LANES> mine(slot, p.K);
	for (int c0 = 0; c0 < p.E; c0 += ROUTE_CHUNK) {
		__syncthreads();
		route_stage(p, tile, t0, tokens, c0);
		__syncthreads();
		if (group < tokens && t0 + group < p.T) {
			mine.walk(tile + group * ROUTE_ROW_DWORDS, c0, min(ROUTE_CHUNK, p.E - c0));
		}
	}
	const int t = t0 + group;
	if (group >= tokens || t >= p.T) {
		return 0xFFFF;
	}
	return mine.finish((size_t) t * p.K, p.weights, p.chosen);
}

#define ROUTE_SELECT(lanes_, tile_, t0_, tokens_) \
	((lanes_) == 1 ? route_select<1>(p, tile_, t0_, tokens_) : (lanes_) == 2 ? route_select<2>(p, tile_, t0_, tokens_) : \
	 (lanes_) == 4 ? route_select<4>(p, tile_, t0_, tokens_) : (lanes_) == 8 ? route_select<8>(p, tile_, t0_, tokens_) : \
	 (lanes_) == 16 ? route_select<16>(p, tile_, t0_, tokens_) : route_select<32>(p, tile_, t0_, tokens_))

/* One block of 32 tokens: logits, selection, the block's count per expert.
 * Launch: grid = ceil(T / 32), block = max(256, 32 * lanes) with lanes the power of two >= K. */
__global__ void __launch_bounds__(ROUTE_TOKENS * SELECT_MAX_K) route_select_kernel(RouteParams p, int lanes) {
	__shared__ uint32_t tile[ROUTE_TOKENS * ROUTE_ROW_DWORDS];
	__shared__ int hist[ROUTE_MAX_EXPERTS];
	for (int e = threadIdx.x; e < p.counts_pitch; e += blockDim.x) {
		hist[e] = 0;
	}
	const int e = ROUTE_SELECT(lanes, tile, (int) blockIdx.x * ROUTE_TOKENS, ROUTE_TOKENS);   /* its barriers order the clear */
	if (e < p.E) {
		atomicAdd(&hist[e], 1);
	}
	__syncthreads();
	uint32_t * dst = (uint32_t *) (p.counts + (size_t) blockIdx.x * p.counts_pitch);
	for (int v = threadIdx.x; v < p.counts_pitch / 4; v += blockDim.x) {
		dst[v] = (uint32_t) hist[4 * v] | ((uint32_t) hist[4 * v + 1] << 8) | ((uint32_t) hist[4 * v + 2] << 16) | ((uint32_t) hist[4 * v + 3] << 24);
	}
}

/* Exclusive scan of counts[0..E) by the first wave into starts[]; `publish`: also the layer's count arrays. */
__device__ __forceinline__ void route_scan(const RouteParams & p, const int * counts, int * starts, bool publish, int tickets) {
	const int lane = threadIdx.x & (WAVE - 1);
	int carry = 0;
	for (int base = 0; base < p.E; base += WAVE) {
		const int e = base + lane;
		const int c = e < p.E ? counts[e] : 0;
		int incl = c;
		#pragma unroll
		for (int off = 1; off < WAVE; off <<= 1) {
			const int up = __shfl_up(incl, off, WAVE);
			if (lane >= off) {
				incl += up;
			}
		}
		if (e < p.E) {
			starts[e] = carry + incl - c;
			if (publish) {
				p.expert_counts[e] = c;
				p.expert_counts_cumsum[e] = carry + incl;
				p.host_expert_counts[e] = c;
			}
		}
		carry += __shfl(incl, WAVE - 1, WAVE);
	}
	if (publish && lane == 0) {
		p.expert_counts[p.E] = tickets;
	}
}

/* the lanes of this wave that hold expert e (the same for all lanes that agree in every bit of the id) */
__device__ __forceinline__ uint64_t route_same(int e, int id_bits) {
	uint64_t same = ~0ULL;
	for (int bit = 0; bit < id_bits; bit++) {
		const bool set = (e >> bit) & 1;
		const uint64_t with_bit = __ballot(set);
		same &= set ? with_bit : ~with_bit;
	}
	return same;
}

/* The permutation, stable in the tokens.  Wave w of work-group b maps selection block 4 b + w: its entries of expert e
 * start behind all entries of the experts in front, those of e in the blocks in front, and are ranked with ballots.
 * Every work-group reads all blocks' counts (64 bytes per 32 tokens for 64 experts), sixteen experts per lane and load.
 * Launch: grid = ceil(blocks / 4), block = 256. */
__global__ void __launch_bounds__(ROUTE_MAP_THREADS) route_map_kernel(RouteParams p, int blocks) {
	__shared__ int tot[ROUTE_MAX_EXPERTS];
	__shared__ int pre[ROUTE_MAX_EXPERTS];
	__shared__ int starts[ROUTE_MAX_EXPERTS];
	__shared__ int run[ROUTE_MAP_WAVES][ROUTE_MAX_EXPERTS];
	const int lane = threadIdx.x & (WAVE - 1);
	const int wave = threadIdx.x / WAVE;
	const int first = blockIdx.x * ROUTE_MAP_WAVES;
	/* everything this work-group reads is asked for before the first use: its own entries, its own blocks' counts, and (in
	 * the loop below) all blocks' counts */
	const long long lo = (long long) (first + wave) * ROUTE_TOKENS * p.K;
	const long long hi = min(lo + (long long) ROUTE_TOKENS * p.K, (long long) p.T * p.K);
	int ids[ROUTE_MAP_AHEAD];
	#pragma unroll
	for (int u = 0; u < ROUTE_MAP_AHEAD; u++) {
		const long long i = lo + u * WAVE + lane;
		ids[u] = i < hi ? (int) p.chosen[i] : p.E;
	}
	int own[2][ROUTE_MAP_WAVES];                                  /* experts tid and tid + 256 */
	#pragma unroll
	for (int h = 0; h < 2; h++) {
		const int e = (int) threadIdx.x + h * ROUTE_MAP_THREADS;
		#pragma unroll
		for (int w = 0; w < ROUTE_MAP_WAVES; w++) {
			own[h][w] = e < p.E && first + w < blocks ? (int) p.counts[(size_t) (first + w) * p.counts_pitch + e] : 0;
		}
	}
	for (int e = threadIdx.x; e < p.counts_pitch; e += ROUTE_MAP_THREADS) {
		tot[e] = 0;
		pre[e] = 0;
	}
	__syncthreads();
	{
		const int cols = p.counts_pitch / 16;                      /* a power of two of at most 32: a lane stays in one column */
		const u32x4 * src = (const u32x4 *) p.counts;
		const int vecs = blocks * cols, vecs_pre = min(first, blocks) * cols;
		/* Four byte counters per dword, added up as pairs of 16-bit fields: at most 65535 / 32 blocks per lane (checked on the
		 * host).  [0]: blocks in front of this work-group's, [1]: all of them. */
		uint32_t even[2][4] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}}, odd[2][4] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}};
		#pragma unroll 4
		for (int v = threadIdx.x; v < vecs; v += ROUTE_MAP_THREADS) {
			const u32x4 q = src[v];
			const uint32_t w[4] = {q.x, q.y, q.z, q.w};
			const uint32_t front = v < vecs_pre ? 0x00FF00FFu : 0u;
			#pragma unroll
			for (int i = 0; i < 4; i++) {
				even[0][i] += w[i] & front;
				odd[0][i] += (w[i] >> 8) & front;
				even[1][i] += w[i] & 0x00FF00FFu;
				odd[1][i] += (w[i] >> 8) & 0x00FF00FFu;
			}
		}
		const int col = (int) threadIdx.x & (cols - 1);
		#pragma unroll
		for (int i = 0; i < 16; i++) {
			const int d = i >> 2, shift = (i & 2) * 8;
			int a = (int) ((((i & 1) ? odd[0][d] : even[0][d]) >> shift) & 0xFFFFu);
			int b = (int) ((((i & 1) ? odd[1][d] : even[1][d]) >> shift) & 0xFFFFu);
			for (int off = cols; off < WAVE; off <<= 1) {
				a += __shfl_xor(a, off, WAVE);
				b += __shfl_xor(b, off, WAVE);
			}
			if (lane < cols) {
				atomicAdd(&pre[col * 16 + i], a);
				atomicAdd(&tot[col * 16 + i], b);
			}
		}
	}
	__syncthreads();
	if (wave == 0) {
		route_scan(p, tot, starts, blockIdx.x == 0, blocks);
	}
	__syncthreads();
	#pragma unroll
	for (int h = 0; h < 2; h++) {
		const int e = (int) threadIdx.x + h * ROUTE_MAP_THREADS;
		if (e < p.E) {
			int at = starts[e] + pre[e];
			#pragma unroll
			for (int w = 0; w < ROUTE_MAP_WAVES; w++) {
				run[w][e] = at;
				at += own[h][w];
			}
		}
	}
	__syncthreads();

	int * my_run = run[wave];
	const int id_bits = 32 - __clz(p.E);
	for (long long i0 = lo; i0 < hi; i0 += WAVE) {
		const long long i = i0 + lane;
		const int u = (int) ((i0 - lo) / WAVE);
		int e = p.E;
		if (u < ROUTE_MAP_AHEAD) {
			#pragma unroll
			for (int j = 0; j < ROUTE_MAP_AHEAD; j++) {
				e = j == u ? ids[j] : e;
			}
		} else {
			e = i < hi ? (int) p.chosen[i] : p.E;
		}
		const bool valid = e < p.E;
		e = valid ? e : p.E;                                         /* takes part as an id no expert has */
		const uint64_t same = route_same(e, id_bits);
		const int start = valid ? my_run[e] : 0;
		const int rank = __popcll(same & lanemask_lt());
		/* all lanes have read their position before the first lane of each expert moves it on */
		if (valid && rank == 0) {
			my_run[e] = start + __popcll(same);
		}
		if (valid) {
			p.expert_mapping[start + rank] = (int) (i / p.K);
			p.token_mapping[i] = start + rank;
		}
	}
}

/* Selection and permutation of few tokens in one work-group: T * lanes <= 1024, T <= 256.
 * Launch: grid = 1, block = T * lanes rounded up to whole waves, or more waves where there are more sums to add up. */
__global__ void __launch_bounds__(ROUTE_SMALL_THREADS) route_small_kernel(RouteParams p, int lanes) {
	__shared__ uint32_t tile[ROUTE_SMALL_TOKENS * ROUTE_ROW_DWORDS];
	__shared__ uint16_t ids[ROUTE_SMALL_THREADS];
	__shared__ int tot[ROUTE_MAX_EXPERTS];
	__shared__ int starts[ROUTE_MAX_EXPERTS];
	__shared__ uint8_t in_wave[ROUTE_SMALL_THREADS / WAVE][ROUTE_MAX_EXPERTS];      /* entries of a wave per expert, at most 64 */
	const int lane = threadIdx.x & (WAVE - 1);
	const int wave = threadIdx.x / WAVE;
	for (int e = threadIdx.x; e < p.E; e += blockDim.x) {
		tot[e] = 0;
	}
	for (int i = threadIdx.x; i < (int) sizeof(in_wave) / 4; i += blockDim.x) {
		((uint32_t *) in_wave)[i] = 0u;
	}
	const int chose = ROUTE_SELECT(lanes, tile, 0, p.T);
	/* the routed entries in order, one per thread from here on: entry i = token * K + slot (at most T * lanes of them) */
	const int slot = (int) threadIdx.x % lanes, token = (int) threadIdx.x / lanes;
	if (slot < p.K && token < p.T) {
		ids[token * p.K + slot] = (uint16_t) chose;
	}
	if (chose < p.E) {
		atomicAdd(&tot[chose], 1);
	}
	__syncthreads();
	if (wave == 0) {
		route_scan(p, tot, starts, true, (p.T + ROUTE_TOKENS - 1) / ROUTE_TOKENS);
	}
	const int i = threadIdx.x;
	int e = i < p.T * p.K ? (int) ids[i] : p.E;
	const bool valid = e < p.E;
	e = valid ? e : p.E;
	const uint64_t same = route_same(e, 32 - __clz(p.E));
	const int rank = __popcll(same & lanemask_lt());
	if (valid && rank == 0) {
		in_wave[wave][e] = (uint8_t) __popcll(same);
	}
	__syncthreads();
	if (valid) {
		int at = starts[e] + rank;
		for (int w = 0; w < wave; w++) {
			at += in_wave[w][e];
		}
		p.expert_mapping[at] = i / p.K;
		p.token_mapping[i] = at;
	}
}

#endif
