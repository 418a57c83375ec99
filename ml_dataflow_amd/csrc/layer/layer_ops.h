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

/* The up-projections of the fused schedule and their activation: what dataflow_submit_amd_grouped_matmul_gathered (x1 | x3 of routed row
 * r side by side, from row expert_mapping[r] of X) and dataflow_submit_amd_swiglu_strided leave, bit for bit.  All pointers
 * 16-byte aligned; X and one expert's w1 below 4 GiB.  Stands in for those two.
 * Submitted for up to LAYER_UP_SWIGLU_VALUES values of x1 | x3: there the GEMM may run on tiles whose epilogue can compute the
 * activation, one launch less in a chain of six that launches are most of (forwards, us: 256 tokens, dim 512
 * 28.6 -> 26.6; 16 tokens, 64 experts, dim 4096 264.6 -> 258.8; 885 tokens over 34 experts, dims 3904 / 1984 392 -> 385).
 * Where it runs on the persistent kernels, which have no room for it, the activation is a second launch of the op; beyond the
 * limit they nearly always are the cheaper ones. */
#define LAYER_UP_SWIGLU_VALUES (1u << 25)
/* The same with x1 and x3 as arrays of their own, for weights that lie behind each other (w3 at w1 + expert_dim * model_dim), always on
 * the tiles whose epilogue computes the activation.
 * Of the grouped schedule, where it stands in for prepare_experts, the two grouped matmuls, which run on two streams that meet
 * before and behind them (12 us each), and swiglu: up to 2^36 multiplies, beyond which the persistent kernels gain more than
 * that (training steps, us: 1908 tokens, top 4, dims 2048 / 640 587 -> 552, 1326, top 3, 3392 / 1792 1616 -> 1580, 1445, top 2,
 * 2112 / 640 391 -> 378; at 1.5 times the limit, 1913, top 5, 3264 / 1664, 1740 -> 1758).
 * Of one expert's packed rows in the per-expert schedule, for the two matmuls and swiglu, up to LAYER_UP_SWIGLU_EXPERT_VALUES: a chain
 * of four launches per expert becomes two (16 experts of 256 rows, dims 2048 / 1408 1314 -> 1228; 60 of 570, 2624 / 1536
 * 7256 -> 6777). */
#define LAYER_UP_SWIGLU_EXPERT_VALUES (1u << 23)
#define LAYER_UP_SWIGLU_GROUPED_MULTIPLIES (1ull << 36)
enum { LAYER_UP_SWIGLU_GROUPED, LAYER_UP_SWIGLU_EXPERT };
LAYER_OPS_HIDDEN void layer_set_up_swiglu_apart_skeleton(Op_Skeleton * skeleton, int which);
LAYER_OPS_HIDDEN int layer_bind_up_swiglu_apart(Dataflow_Handle * handle, int which);
LAYER_OPS_HIDDEN int layer_has_up_swiglu_apart(Dataflow_Handle * handle, int which);
/* _EXPERT: num_experts 1, no prefix sum, no mapping, num_tokens = num_rows */
LAYER_OPS_HIDDEN int layer_submit_up_swiglu_apart(Dataflow_Handle * handle, int stream_id, int which, int expert_dim, int model_dim, int num_rows, int num_experts,
							 int * expert_counts_cumsum, void * w13, uint64_t expert_stride_bytes, void * X, int * expert_mapping, int num_tokens,
							 void * x1, void * x3, void * h);
LAYER_OPS_HIDDEN void layer_set_up_swiglu_skeleton(Op_Skeleton * skeleton);
LAYER_OPS_HIDDEN int layer_bind_up_swiglu(Dataflow_Handle * handle);
LAYER_OPS_HIDDEN int layer_has_up_swiglu(Dataflow_Handle * handle);
LAYER_OPS_HIDDEN int layer_submit_up_swiglu(Dataflow_Handle * handle, int stream_id, int expert_dim, int model_dim, int num_rows, int num_experts,
							 int * expert_counts_cumsum, void * w13, uint64_t expert_stride_bytes, void * X, int * expert_mapping, int num_tokens,
							 void * x13, void * h);

/* An expert's dW1 and dW3 of the per-expert schedule, which differ in B, C and D: what two dataflow_submit_matmul without a
 * workspace leave, bit for bit; stands in for the matmul.  One launch where the two together run on the direct kernel's tiles, which
 * an expert's few hundred rows leave half of the compute units without (training steps, us: 16 experts of 256 rows, dims 2048 /
 * 1408 1232 -> 1188, 60 of 570, 2624 / 1536 6773 -> 6435); two where they are large enough for the persistent one. */
LAYER_OPS_HIDDEN void layer_set_matmul_twin_skeleton(Op_Skeleton * skeleton);
LAYER_OPS_HIDDEN int layer_bind_matmul_twin(Dataflow_Handle * handle);
LAYER_OPS_HIDDEN int layer_has_matmul_twin(Dataflow_Handle * handle);
LAYER_OPS_HIDDEN int layer_submit_matmul_twin(Dataflow_Handle * handle, int stream_id, int M, int K, int N, float beta, void * A,
							 void * B1, void * C1, void * D1, void * B2, void * C2, void * D2);

/* dW1 | dW3 of the fused schedule: would the gathered grouped matmul over the rows of X run on the kernel that makes up for the copy it saves
 * (the sliced one)?  Asked of the library that launches it, with the launch's operands; nothing runs on the device.  dw, if C is read: accumulate.
 * 0 where it, the grouped matmul or prepare_experts, which the copy + packed form consists of, is not the one of registration. */
LAYER_OPS_HIDDEN void layer_set_gathers_k_rows_skeleton(Op_Skeleton * skeleton);
LAYER_OPS_HIDDEN int layer_bind_gathers_k_rows(Dataflow_Handle * handle);
LAYER_OPS_HIDDEN int layer_gathers_k_rows(Dataflow_Handle * handle, int model_dim, int num_rows, int stacked_dim, int num_experts, void * X, int num_tokens,
							 void * dx13, int accumulate, void * dw13, uint64_t expert_stride_bytes);

#endif
