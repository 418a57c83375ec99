/* stand_in.c -- see stand_in.h */
#include "stand_in.h"

static Hip_Function * registered(Dataflow_Handle * handle, Op_Skeleton * skeleton) {
	Hip_Function * fn = NULL;
	return dataflow_find_table(&handle->op_table, skeleton->identifier.fingerprint, false, (void **) &fn) >= 0 ? fn : NULL;
}

/* what implements the op in the table; NULL where it is not there */
static const void * implementation(Dataflow_Handle * handle, Op_Skeleton * skeleton) {
	const Hip_Function * fn = registered(handle, skeleton);
	return !fn ? NULL : fn->is_native ? fn->function_handle : (const void *) fn->hip_external_func;
}

int stand_in_bind(Dataflow_Handle * handle, Op_Skeleton * op, Op_Skeleton * of, int n) {
	Hip_Function * fn = registered(handle, op);
	if (!fn || n > HIP_MAX_STOOD_IN) {
		return -1;
	}
	for (int i = 0; i < n; i++) {
		fn->stands_in_for[i] = implementation(handle, &of[i]);
		if (!fn->stands_in_for[i]) {
			return -1;
		}
	}
	return 0;
}

int stand_in_usable(Dataflow_Handle * handle, Op_Skeleton * op, Op_Skeleton * of, int n) {
	const Hip_Function * fn = registered(handle, op);
	for (int i = 0; fn && i < n; i++) {
		const void * now = implementation(handle, &of[i]);
		if (!now || now != fn->stands_in_for[i]) {
			return 0;
		}
	}
	return fn != NULL;
}

int stand_in_ask(Dataflow_Handle * handle, Op * op, Op_Skeleton * of, int n) {
	const Hip_Function * fn = registered(handle, &op->op_skeleton);
	return fn && fn->hip_external_func && stand_in_usable(handle, &op->op_skeleton, of, n) ? (fn->hip_external_func)(handle, -1, op, fn->op_extra) : 0;
}
