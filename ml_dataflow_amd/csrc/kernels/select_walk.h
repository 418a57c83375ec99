/*
 * select_walk.h -- top-k selection over bf16 logits for gfx950: the walk over a token's experts, one slot per lane, shared
 * by the select_experts op (routing.hip) and the layer's routing kernels (../matmul/route_kernel.h).
 */
#ifndef SELECT_WALK_H
#define SELECT_WALK_H

#include "moe_common.h"

#define SELECT_MAX_K 32

/* The reference keeps K (value, expert) slots per token and walks the experts in ascending order
 * (select_experts.cu:417-468): an expert enters only if its logit is STRICTLY greater than the current
 * minimum slot, it takes that slot's place, and the new minimum is the smallest value with ties going to
 * the slot that holds the LARGER expert id (among never-filled slots, which all hold -inf / 0xFFFF, the
 * lowest slot).  The slot order is part of the result.
 *
 * Here a group of LANES lanes replays exactly that walk for one token with ONE SLOT PER LANE: every lane sees
 * the same logit, the lane whose slot is the current minimum takes it, and the new minimum is found with
 * log2(LANES) cross-lane steps instead of a serial pass over K slots.  The walk itself stays sequential in
 * the experts, as the result depends on their order: its length is 64 dependent steps for 64 experts whatever the
 * token count, so a step is kept to a handful of instructions.  Lanes beyond K hold the largest key and never win. */

/* The walk compares and moves one 32-bit key per slot instead of a (value, expert) pair:
 *   high half: the logit's bf16 bits made monotonic (sort_key16: a larger value is a larger number; -0 counts as +0, as
 *              it does in a float comparison; a NaN becomes 0, below -inf, so it never enters, as no float comparison
 *              with a NaN holds)
 *   low half:  0xFFFF - expert id, so that among equal values the larger id is the smaller key; a never-filled slot
 *              holds (-inf, slot number): the lowest such slot is the minimum, and nothing displaces it but a real
 *              entry, since a logit of -inf is not strictly greater than -inf and never enters.
 * The minimum slot of the reference's rule is then the smallest key, one v_min_u32 per cross-lane step. */
#define KEY16_NEG_INF 0x007Fu
__device__ __forceinline__ uint32_t sort_key16(uint32_t bits) {
	const uint32_t mag = bits & 0x7FFFu;
	if (mag > 0x7F80u) {
		return 0u;
	}
	if (mag == 0u) {
		return 0x8000u;
	}
	return (bits & 0x8000u) ? (bits ^ 0xFFFFu) : (bits | 0x8000u);
}
__device__ __forceinline__ float sort_key16_value(uint32_t key) {
	const uint32_t bits = (key & 0x8000u) ? (key & 0x7FFFu) : (key ^ 0xFFFFu);
	return __uint_as_float(bits << 16);
}

/* lane i <-> lane i ^ 1, i ^ 2 (inside quads), 7 - i (inside 8), 15 - i (inside 16): after the steps before it each
 * mirror pairs a lane with one from the other half, which is all a reduction needs */
template <int CTRL>
__device__ __forceinline__ uint32_t key_min_step(uint32_t key) {
	/* every lane has a partner; with the identity of min in its place the compiler folds the move into the minimum */
	const uint32_t other = (uint32_t) __builtin_amdgcn_update_dpp(-1, (int) key, CTRL, 0xF, 0xF, false);
	return min(key, other);
}

__device__ __forceinline__ uint32_t sort_key_pair(uint32_t pair) {
	return sort_key16(pair & 0xFFFFu) | (sort_key16(pair >> 16) << 16);
}

/* One slot of one token's walk: lane `slot` of the group of LANES lanes that share the token. */
template <int LANES>
struct SelectSlot {
	uint32_t key;                                          /* this lane's slot */
	uint32_t min_key;                                      /* the smallest slot of the group: the same in every lane */
	uint32_t max_key16;                                    /* largest value that entered: the first expert to have it always enters */
	int slot, K;
	bool live;

	__device__ __forceinline__ SelectSlot(int slot_, int K_) : slot(slot_), K(K_), live(slot_ < K_) {
		key = live ? ((KEY16_NEG_INF << 16) | (uint32_t) slot) : 0xFFFFFFFFu;     /* lanes beyond K are never the minimum */
		min_key = KEY16_NEG_INF << 16;                        /* slot 0's key */
		max_key16 = KEY16_NEG_INF;
	}

	/* experts [c0, c0 + count) in order; `row`: their sort keys, two per dword (an odd count's last partner is -inf and
	 * never enters).  A step is a chain: which lane holds the smallest key, the larger of that key and the expert's, the smallest
	 * again.  What does not depend on the step before is kept out of it: the expert's key is 0 where its logit can never enter, so
	 * that one unsigned maximum is the rule above, and the largest value that entered is the largest there is.  16 tokens, 64 experts,
	 * top 8 in one work-group: 8.9 -> 8.3 us; 65536 tokens, selection and mapping: 42.3 -> 39.9.  Keys read four pairs ahead: no faster. */
	__device__ __forceinline__ void walk(const uint32_t * row, int c0, int count) {
		for (int j = 0; j < count; j += 2) {
			const uint32_t pair = row[j >> 1];
			step(pair & 0xFFFFu, c0 + j);
			step(pair >> 16, c0 + j + 1);
		}
	}

	__device__ __forceinline__ void step(uint32_t k16, int expert) {
		const uint32_t entry = k16 > KEY16_NEG_INF ? (k16 << 16) | (0xFFFFu - (uint32_t) expert) : 0u;
		max_key16 = max(max_key16, k16);
		key = key == min_key ? max(key, entry) : key;
		min_key = key;
		if (LANES > 1) { min_key = key_min_step<0xB1>(min_key); }
		if (LANES > 2) { min_key = key_min_step<0x4E>(min_key); }
		if (LANES > 4) { min_key = key_min_step<0x141>(min_key); }
		if (LANES > 8) { min_key = key_min_step<0x140>(min_key); }
		if (LANES > 16) { min_key = min(min_key, (uint32_t) __shfl_xor((int) min_key, 16, WAVE)); }
	}

	/* softmax over the K slots, summed in slot order; the reference subtracts the max in bf16 before expf
	 * (select_experts.cu:480,488).  Writes slot `slot` of the token whose slots start at `first`; returns its expert
	 * (0xFFFF for a slot that was never filled or does not exist). */
	__device__ __forceinline__ int finish(size_t first, float * __restrict__ weights, uint16_t * __restrict__ chosen) const {
		const bool filled = live && (key >> 16) != KEY16_NEG_INF;
		const float val = filled ? sort_key16_value(key >> 16) : -INFINITY;
		const int idx = filled ? (int) (0xFFFFu - (key & 0xFFFFu)) : 0xFFFF;
		const float max_val = sort_key16_value(max_key16);
		const float ex = live ? expf(bf16_to_f32(f32_to_bf16(val - max_val))) : 0.0f;
		float sum = 0.0f;
		const int base = (threadIdx.x & (WAVE - 1)) - slot;
		for (int k = 0; k < K; k++) {
			sum += __shfl(ex, base + k, WAVE);
		}
		if (live) {
			weights[first + slot] = ex / sum;
			chosen[first + slot] = (uint16_t) idx;
		}
		return idx;
	}
};

#endif
