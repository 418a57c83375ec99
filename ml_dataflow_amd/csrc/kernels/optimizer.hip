/*
 * optimizer.hip -- AdamW step on bf16 parameters, gradients and moments (fp32 arithmetic).
 * Included by hip_kernels.hip after movement.hip.
 *
 * Semantics of backends/nvidia/src/ops/src/native/src/optimizer/adamw_step.cu:6-65, element by element:
 *   m = beta1 * mean + (1 - beta1) * g;        v = beta2 * var + (1 - beta2) * g * g
 *   m_hat = m / (1 - beta1^step);              v_hat = v / (1 - beta2^step)
 *   param = bf16(param - lr * (m_hat / (sqrt(v_hat) + eps) + weight_decay * param));  mean = bf16(m);  var = bf16(v)
 * Bandwidth-bound: 8 bytes read and 6 written per element.  Each lane handles 8 consecutive elements (16-byte
 * accesses) when the four arrays are 16-byte aligned, single elements otherwise and for the tail.
 */

__device__ __forceinline__ void adamw_element(float & p, float g, float & m, float & v, float lr, float beta1, float beta2,
											  float weight_decay, float epsilon, float corr1, float corr2) {
	const float m_t = beta1 * m + (1.0f - beta1) * g;
	const float v_t = beta2 * v + (1.0f - beta2) * g * g;
	const float m_hat = m_t / corr1;
	const float v_hat = v_t / corr2;
	p = p - lr * (m_hat / (sqrtf(v_hat) + epsilon) + weight_decay * p);
	m = m_t;
	v = v_t;
}

/* One 16-byte vector of each array: read, updated, written, past the caches both ways. */
__device__ __forceinline__ void adamw_vector(uint64_t i, u32x4 * param, const u32x4 * grad, u32x4 * mean, u32x4 * var, float lr, float beta1, float beta2,
											 float weight_decay, float epsilon, float corr1, float corr2) {
	float p[8], g[8], m[8], v[8];
	unpack8(__builtin_nontemporal_load(param + i), p);
	unpack8(__builtin_nontemporal_load(grad + i), g);
	unpack8(__builtin_nontemporal_load(mean + i), m);
	unpack8(__builtin_nontemporal_load(var + i), v);
	#pragma unroll
	for (int e = 0; e < 8; e++) {
		adamw_element(p[e], g[e], m[e], v[e], lr, beta1, beta2, weight_decay, epsilon, corr1, corr2);
	}
	__builtin_nontemporal_store(pack8(p), param + i);
	__builtin_nontemporal_store(pack8(m), mean + i);
	__builtin_nontemporal_store(pack8(v), var + i);
}

/* Launch: grid = ceil(num_els / 2048), block = 256: one vector per lane (the loops only take the tail, an unaligned
 * call, or what lies beyond the 2^32 lanes of the largest launch).
 * A lane's first vector stands in front of the loop: there the four loads are issued together; inside the loop the
 * compiler waits for each before it issues the next, four memory round trips in a row.
 * Every array is accessed non-temporally at every size, in one form: with a plain and a non-temporal form behind a
 * branch on the size, the compiler merges the two and drops the hint.  Each step passes over all four arrays once, and a
 * training step passes over far more than the 256 MiB memory-side cache in between.
 * Measured, us per launch: each load behind the one before / issued together / and non-temporal, with arrays that were
 * not touched by the last launches: 1 M elements 8.0 / 7.1 / 6.0; 8 M 27.6 / 25.3 / 24.1; 34 M 95 / 87 / 83; 277 M 693 /
 * 670 / 641 (6.0 TB/s); 805 M 2005 / 1969 / 1884.  Launched over and over on the same arrays: the same order or no
 * difference, but for 17 to 34 M elements, which the cache holds and plain accesses serve 1-6 % faster (25 M: 68.6 /
 * 59.2 / 61.0). */
extern "C" __global__ void __launch_bounds__(256)
default_adamw_step_bf16_bf16_bf16_bf16_kernel(uint64_t num_els, int step_num, float lr, float beta1, float beta2, float weight_decay,
											  float epsilon, bf16_t * param, const bf16_t * grad, bf16_t * mean, bf16_t * var) {
	const float corr1 = 1.0f - powf(beta1, (float) step_num);
	const float corr2 = 1.0f - powf(beta2, (float) step_num);
	const uint64_t tid = (uint64_t) blockIdx.x * 256 + threadIdx.x;
	const uint64_t nthreads = (uint64_t) gridDim.x * 256;
	const bool aligned = ((((uintptr_t) param) | ((uintptr_t) grad) | ((uintptr_t) mean) | ((uintptr_t) var)) & 15) == 0;
	const uint64_t nvec = aligned ? (num_els >> 3) : 0;
	u32x4 * const p4 = (u32x4 *) param, * const m4 = (u32x4 *) mean, * const v4 = (u32x4 *) var;
	const u32x4 * const g4 = (const u32x4 *) grad;
	if (tid < nvec) {
		adamw_vector(tid, p4, g4, m4, v4, lr, beta1, beta2, weight_decay, epsilon, corr1, corr2);
		for (uint64_t i = tid + nthreads; i < nvec; i += nthreads) {
			adamw_vector(i, p4, g4, m4, v4, lr, beta1, beta2, weight_decay, epsilon, corr1, corr2);
		}
	}
	for (uint64_t i = (nvec << 3) + tid; i < num_els; i += nthreads) {
		float p = bf16_to_f32(param[i]), m = bf16_to_f32(mean[i]), v = bf16_to_f32(var[i]);
		adamw_element(p, bf16_to_f32(grad[i]), m, v, lr, beta1, beta2, weight_decay, epsilon, corr1, corr2);
		param[i] = f32_to_bf16(p);
		mean[i] = f32_to_bf16(m);
		var[i] = f32_to_bf16(v);
	}
}
