/*
 * layer_ops.h -- ops that only the layer driver (moe_layer.c) submits: fused forms of parts of its op sequence.  They go
 * through the handle's op table like every other op, but are no part of the operator interface: no caller beside the
 * layer has their inputs in the form they take.
 */
#ifndef LAYER_OPS_H
#define LAYER_OPS_H

#include "dataflow_amd.h"

#define LAYER_OPS_HIDDEN __attribute__((visibility("hidden")))

/* Router product, selection, counts, prefix sum and dispatch permutation: what dataflow_submit_matmul (logits = X Wr^T +
 * bias), clearing the count arrays, dataflow_submit_default_select_experts and dataflow_submit_default_build_expert_mapping
 * leave, bit for bit, from at most four launches (../matmul/route_kernel.h).
 * Up to 512 experts and 32 slots; the workspace (16-byte aligned) has at least LAYER_ROUTE_WORKSPACE bytes.  The router
 * product is split along its K where the matmul would split it with that workspace. */
#define LAYER_ROUTE_MAX_EXPERTS 512
#define LAYER_ROUTE_WORKSPACE(tokens, experts) (((uint64_t) (tokens) + 31) / 32 * (2 * (uint64_t) (experts) + 16) + 256)
LAYER_OPS_HIDDEN void layer_set_route_tokens_skeleton(Op_Skeleton * skeleton);
/* stands in for matmul, select_experts and build_expert_mapping (../ops/stand_in.h); _bind goes behind its registration */
LAYER_OPS_HIDDEN int layer_bind_route_tokens(Dataflow_Handle * handle);
LAYER_OPS_HIDDEN int layer_has_route_tokens(Dataflow_Handle * handle);
LAYER_OPS_HIDDEN int layer_submit_route_tokens(Dataflow_Handle * handle, int stream_id, int num_tokens, int num_experts, int top_k, int model_dim,
								void * X, void * w_router, void * logit_bias, void * x_routed, float * token_expert_weights,
								uint16_t * chosen_experts, int * expert_counts, int * expert_counts_cumsum, int * host_expert_counts,
								int * expert_mapping, int * token_mapping, uint64_t workspace_bytes, void * workspace);

#endif
