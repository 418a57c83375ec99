/* layer_ops.c -- skeletons and submission of the layer driver's own ops (see layer_ops.h) */
#include "layer_ops.h"
#include "../ops/skeletons.h"
#include "../ops/stand_in.h"
#include "dataflow_amd_ops.h"

#include <stdio.h>

static int submit(Dataflow_Handle * handle, Op * op, int stream_id, const char * what) {
	if ((handle->submit_op)(handle, op, stream_id)) {
		fprintf(stderr, "Error: failed to submit %s op...\n", what);
		return -1;
	}
	return 0;
}

void layer_set_route_tokens_skeleton(Op_Skeleton * skeleton) {
	const DataflowDatatype t[17] = {DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_BF16, DATAFLOW_BF16,
									DATAFLOW_BF16, DATAFLOW_BF16, DATAFLOW_FP32, DATAFLOW_UINT16, DATAFLOW_INT, DATAFLOW_INT, DATAFLOW_INT, DATAFLOW_INT,
									DATAFLOW_INT, DATAFLOW_UINT64_SCALAR, DATAFLOW_VOID};
	dataflow_fill_skeleton(skeleton, "amd_route_tokens", DATAFLOW_BF16, DATAFLOW_NONE, 17, t);
}

static void route_tokens_stood_in(Op_Skeleton skeletons[3]) {
	dataflow_set_matmul_skeleton(&skeletons[0]);
	dataflow_set_default_select_experts_skeleton(&skeletons[1], DATAFLOW_BF16);
	dataflow_set_default_build_expert_mapping_skeleton(&skeletons[2]);
}

int layer_bind_route_tokens(Dataflow_Handle * handle) {
	Op_Skeleton skeleton, of[3];
	layer_set_route_tokens_skeleton(&skeleton);
	route_tokens_stood_in(of);
	return stand_in_bind(handle, &skeleton, of, 3);
}

int layer_has_route_tokens(Dataflow_Handle * handle) {
	Op_Skeleton skeleton, of[3];
	layer_set_route_tokens_skeleton(&skeleton);
	route_tokens_stood_in(of);
	return stand_in_usable(handle, &skeleton, of, 3);
}

void layer_set_up_swiglu_skeleton(Op_Skeleton * skeleton) {
	const DataflowDatatype t[12] = {DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_INT, DATAFLOW_BF16,
									DATAFLOW_UINT64_SCALAR, DATAFLOW_BF16, DATAFLOW_INT, DATAFLOW_INT_SCALAR, DATAFLOW_BF16, DATAFLOW_BF16};
	dataflow_fill_skeleton(skeleton, "amd_up_swiglu", DATAFLOW_BF16, DATAFLOW_NONE, 12, t);
}

static void up_swiglu_stood_in(Op_Skeleton skeletons[2]) {
	dataflow_set_amd_grouped_matmul_gathered_skeleton(&skeletons[0]);
	dataflow_set_amd_swiglu_strided_skeleton(&skeletons[1], DATAFLOW_BF16);
}

int layer_bind_up_swiglu(Dataflow_Handle * handle) {
	Op_Skeleton skeleton, of[2];
	layer_set_up_swiglu_skeleton(&skeleton);
	up_swiglu_stood_in(of);
	return stand_in_bind(handle, &skeleton, of, 2);
}

int layer_has_up_swiglu(Dataflow_Handle * handle) {
	Op_Skeleton skeleton, of[2];
	layer_set_up_swiglu_skeleton(&skeleton);
	up_swiglu_stood_in(of);
	return stand_in_usable(handle, &skeleton, of, 2);
}

int layer_submit_up_swiglu(Dataflow_Handle * handle, int stream_id, int expert_dim, int model_dim, int num_rows, int num_experts,
							 int * expert_counts_cumsum, void * w13, uint64_t expert_stride_bytes, void * X, int * expert_mapping, int num_tokens,
							 void * x13, void * h) {
	Op op;
	layer_set_up_swiglu_skeleton(&op.op_skeleton);
	void ** a = op.op_args;
	a[0] = &expert_dim; a[1] = &model_dim; a[2] = &num_rows; a[3] = &num_experts; a[4] = &expert_counts_cumsum; a[5] = &w13; a[6] = &expert_stride_bytes;
	a[7] = &X; a[8] = &expert_mapping; a[9] = &num_tokens; a[10] = &x13; a[11] = &h;
	return submit(handle, &op, stream_id, "up projection and swiglu");
}

void layer_set_up_swiglu_apart_skeleton(Op_Skeleton * skeleton, int which) {
	const DataflowDatatype t[13] = {DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_INT, DATAFLOW_BF16,
									DATAFLOW_UINT64_SCALAR, DATAFLOW_BF16, DATAFLOW_INT, DATAFLOW_INT_SCALAR, DATAFLOW_BF16, DATAFLOW_BF16, DATAFLOW_BF16};
	dataflow_fill_skeleton(skeleton, which == LAYER_UP_SWIGLU_EXPERT ? "amd_up_swiglu_expert" : "amd_up_swiglu_grouped", DATAFLOW_BF16, DATAFLOW_NONE, 13, t);
}

static int up_swiglu_apart_stood_in(Op_Skeleton skeletons[3], int which) {
	dataflow_set_default_swiglu_skeleton(&skeletons[0], DATAFLOW_BF16);
	if (which == LAYER_UP_SWIGLU_EXPERT) {
		dataflow_set_matmul_skeleton(&skeletons[1]);
		return 2;
	}
	dataflow_set_amd_grouped_matmul_skeleton(&skeletons[1]);
	dataflow_set_default_prepare_experts_skeleton(&skeletons[2], DATAFLOW_BF16, DATAFLOW_BF16);
	return 3;
}

int layer_bind_up_swiglu_apart(Dataflow_Handle * handle, int which) {
	Op_Skeleton skeleton, of[3];
	layer_set_up_swiglu_apart_skeleton(&skeleton, which);
	return stand_in_bind(handle, &skeleton, of, up_swiglu_apart_stood_in(of, which));
}

int layer_has_up_swiglu_apart(Dataflow_Handle * handle, int which) {
	Op_Skeleton skeleton, of[3];
	layer_set_up_swiglu_apart_skeleton(&skeleton, which);
	return stand_in_usable(handle, &skeleton, of, up_swiglu_apart_stood_in(of, which));
}

int layer_submit_up_swiglu_apart(Dataflow_Handle * handle, int stream_id, int which, int expert_dim, int model_dim, int num_rows, int num_experts,
							 int * expert_counts_cumsum, void * w13, uint64_t expert_stride_bytes, void * X, int * expert_mapping, int num_tokens,
							 void * x1, void * x3, void * h) {
	Op op;
	layer_set_up_swiglu_apart_skeleton(&op.op_skeleton, which);
	void ** a = op.op_args;
	a[0] = &expert_dim; a[1] = &model_dim; a[2] = &num_rows; a[3] = &num_experts; a[4] = &expert_counts_cumsum; a[5] = &w13; a[6] = &expert_stride_bytes;
	a[7] = &X; a[8] = &expert_mapping; a[9] = &num_tokens; a[10] = &x1; a[11] = &h; a[12] = &x3;
	return submit(handle, &op, stream_id, "up projections and swiglu");
}

void layer_set_matmul_twin_skeleton(Op_Skeleton * skeleton) {
	const DataflowDatatype t[11] = {DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_FP32_SCALAR, DATAFLOW_BF16, DATAFLOW_BF16, DATAFLOW_BF16,
									DATAFLOW_BF16, DATAFLOW_BF16, DATAFLOW_BF16, DATAFLOW_BF16};
	dataflow_fill_skeleton(skeleton, "amd_matmul_twin", DATAFLOW_BF16, DATAFLOW_NONE, 11, t);
}

int layer_bind_matmul_twin(Dataflow_Handle * handle) {
	Op_Skeleton skeleton, of;
	layer_set_matmul_twin_skeleton(&skeleton);
	dataflow_set_matmul_skeleton(&of);
	return stand_in_bind(handle, &skeleton, &of, 1);
}

int layer_has_matmul_twin(Dataflow_Handle * handle) {
	Op_Skeleton skeleton, of;
	layer_set_matmul_twin_skeleton(&skeleton);
	dataflow_set_matmul_skeleton(&of);
	return stand_in_usable(handle, &skeleton, &of, 1);
}

int layer_submit_matmul_twin(Dataflow_Handle * handle, int stream_id, int M, int K, int N, float beta, void * A,
							 void * B1, void * C1, void * D1, void * B2, void * C2, void * D2) {
	Op op;
	layer_set_matmul_twin_skeleton(&op.op_skeleton);
	void ** a = op.op_args;
	a[0] = &M; a[1] = &K; a[2] = &N; a[3] = &beta; a[4] = &A; a[5] = &B1; a[6] = &C1; a[7] = &D1; a[8] = &B2; a[9] = &C2; a[10] = &D2;
	return submit(handle, &op, stream_id, "twin matmul");
}

void layer_set_gathers_k_rows_skeleton(Op_Skeleton * skeleton) {
	const DataflowDatatype t[10] = {DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_INT_SCALAR, DATAFLOW_BF16, DATAFLOW_INT_SCALAR, DATAFLOW_BF16,
									DATAFLOW_BF16, DATAFLOW_BF16, DATAFLOW_UINT64_SCALAR};
	dataflow_fill_skeleton(skeleton, "amd_gathers_k_rows", DATAFLOW_BF16, DATAFLOW_NONE, 10, t);
}

static void gathers_k_rows_stood_in(Op_Skeleton skeletons[3]) {
	dataflow_set_amd_grouped_matmul_gathered_skeleton(&skeletons[0]);
	dataflow_set_amd_grouped_matmul_skeleton(&skeletons[1]);
	dataflow_set_default_prepare_experts_skeleton(&skeletons[2], DATAFLOW_BF16, DATAFLOW_BF16);
}

int layer_bind_gathers_k_rows(Dataflow_Handle * handle) {
	Op_Skeleton skeleton, of[3];
	layer_set_gathers_k_rows_skeleton(&skeleton);
	gathers_k_rows_stood_in(of);
	return stand_in_bind(handle, &skeleton, of, 3);
}

int layer_gathers_k_rows(Dataflow_Handle * handle, int model_dim, int num_rows, int stacked_dim, int num_experts, void * X, int num_tokens,
						 void * dx13, int accumulate, void * dw13, uint64_t expert_stride_bytes) {
	Op op;
	Op_Skeleton of[3];
	layer_set_gathers_k_rows_skeleton(&op.op_skeleton);
	gathers_k_rows_stood_in(of);
	void * C = accumulate ? dw13 : NULL;
	void ** a = op.op_args;
	a[0] = &model_dim; a[1] = &num_rows; a[2] = &stacked_dim; a[3] = &num_experts; a[4] = &X; a[5] = &num_tokens; a[6] = &dx13; a[7] = &C; a[8] = &dw13;
	a[9] = &expert_stride_bytes;
	return stand_in_ask(handle, &op, of, 3);
}

int layer_submit_route_tokens(Dataflow_Handle * handle, int stream_id, int num_tokens, int num_experts, int top_k, int model_dim,
							  void * X, void * w_router, void * logit_bias, void * x_routed, float * token_expert_weights,
							  uint16_t * chosen_experts, int * expert_counts, int * expert_counts_cumsum, int * host_expert_counts,
							  int * expert_mapping, int * token_mapping, uint64_t workspace_bytes, void * workspace) {
	Op op;
	layer_set_route_tokens_skeleton(&op.op_skeleton);
	void ** a = op.op_args;
	a[0] = &num_tokens; a[1] = &num_experts; a[2] = &top_k; a[3] = &model_dim;
	a[4] = &X; a[5] = &w_router; a[6] = &logit_bias; a[7] = &x_routed; a[8] = &token_expert_weights; a[9] = &chosen_experts;
	a[10] = &expert_counts; a[11] = &expert_counts_cumsum; a[12] = &host_expert_counts; a[13] = &expert_mapping; a[14] = &token_mapping;
	a[15] = &workspace_bytes; a[16] = &workspace;
	return submit(handle, &op, stream_id, "route tokens");
}
