/*
 * stand_in.h -- ops that stand in for a sequence of others: what a submit wrapper or the layer driver would submit as
 * several ops, in one.  They are in the handle's table like every other op, but no part of the operator interface.  Such an op is used
 * only where it is what the ops it stands in for would do: where the table holds it and, under each of those, the
 * implementation that stood there when it was registered.  A program that registers the ops one by one, or puts its own in
 * the place of one of those, has its ops submitted one by one.
 */
#ifndef STAND_IN_H
#define STAND_IN_H

#include "dataflow_amd.h"

/* notes, in the table's entry of `op`, what implements the `n` ops of `of` (at most HIP_MAX_STOOD_IN); -1 where one is missing */
__attribute__((visibility("hidden"))) int stand_in_bind(Dataflow_Handle * handle, Op_Skeleton * op, Op_Skeleton * of, int n);
/* may `op` be submitted in their place? */
__attribute__((visibility("hidden"))) int stand_in_usable(Dataflow_Handle * handle, Op_Skeleton * op, Op_Skeleton * of, int n);
/* asks an external op that answers on the host (what it returns) instead of launching anything; 0 where it may not be used in their place */
__attribute__((visibility("hidden"))) int stand_in_ask(Dataflow_Handle * handle, Op * op, Op_Skeleton * of, int n);

#endif
