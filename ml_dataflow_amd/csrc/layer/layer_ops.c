/* layer_ops.c -- skeletons and submission of the layer driver's own ops (see layer_ops.h) */
#include "layer_ops.h"
#include "../ops/skeletons.h"
#include "dataflow_amd_ops.h"

#include <stdio.h>
#include <string.h>

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

static Hip_Function * registered(Dataflow_Handle * handle, Op_Skeleton * skeleton) {
	Hip_Function * fn = NULL;
	return dataflow_find_table(&handle->op_table, skeleton->identifier.fingerprint, false, (void **) &fn) >= 0 ? fn : NULL;
}

/* the implementations in the table of the ops that routing consists of; 0 where one is not there */
static int routing_implementations(Dataflow_Handle * handle, const void * implementations[HIP_MAX_STOOD_IN]) {
	Op_Skeleton skeletons[HIP_MAX_STOOD_IN];
	dataflow_set_matmul_skeleton(&skeletons[0]);
	dataflow_set_default_select_experts_skeleton(&skeletons[1], DATAFLOW_BF16);
	dataflow_set_default_build_expert_mapping_skeleton(&skeletons[2]);
	for (int i = 0; i < HIP_MAX_STOOD_IN; i++) {
		const Hip_Function * fn = registered(handle, &skeletons[i]);
		implementations[i] = !fn ? NULL : fn->is_native ? fn->function_handle : (const void *) fn->hip_external_func;
		if (!implementations[i]) {
			return 0;
		}
	}
	return 1;
}

int layer_bind_route_tokens(Dataflow_Handle * handle) {
	Op_Skeleton skeleton;
	layer_set_route_tokens_skeleton(&skeleton);
	Hip_Function * fn = registered(handle, &skeleton);
	return fn && routing_implementations(handle, fn->stands_in_for) ? 0 : -1;
}

int layer_has_route_tokens(Dataflow_Handle * handle) {
	Op_Skeleton skeleton;
	layer_set_route_tokens_skeleton(&skeleton);
	const Hip_Function * fn = registered(handle, &skeleton);
	const void * now[HIP_MAX_STOOD_IN];
	return fn && routing_implementations(handle, now) && memcmp(now, fn->stands_in_for, sizeof(now)) == 0;
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
