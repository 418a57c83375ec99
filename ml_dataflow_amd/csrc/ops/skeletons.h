/* skeletons.h -- filling of op skeletons, shared by the operator interface (dataflow_ops.c) and the layer's own ops */
#ifndef SKELETONS_H
#define SKELETONS_H

#include "dataflow_amd.h"

/* nickname "<base>[_<dt0>[_<dt1>]]", argument tags, fingerprint; `base` has to be a string literal */
__attribute__((visibility("hidden"))) void dataflow_fill_skeleton(Op_Skeleton * skeleton, const char * base, DataflowDatatype dt0, DataflowDatatype dt1,
																  int num_args, const DataflowDatatype * arg_dtypes);

/* rms_norm_bwd_w and its combine for few rows, in one launch (dataflow_submit_default_rms_norm_bwd_w submits it) */
__attribute__((visibility("hidden"))) void dataflow_set_amd_rms_norm_bwd_w_few_rows_skeleton(Op_Skeleton * skeleton);
__attribute__((visibility("hidden"))) int dataflow_bind_amd_rms_norm_bwd_w_few_rows(Dataflow_Handle * handle);

/* the norm over short rows, one on a wave, and over long ones (dataflow_submit_default_rms_norm and its bwd_x submit them, kernels/norm_rows.h) */
enum { NORM_FORM_WAVE_ROWS, NORM_FORM_LONG_ROWS, NORM_FORM_BWD_X_WAVE_ROWS, NORM_FORMS };
__attribute__((visibility("hidden"))) void dataflow_set_amd_rms_norm_form_skeleton(Op_Skeleton * skeleton, int form);
__attribute__((visibility("hidden"))) int dataflow_bind_amd_rms_norm_form(Dataflow_Handle * handle, int form);

#endif
