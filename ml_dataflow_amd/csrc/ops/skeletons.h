/* skeletons.h -- filling of op skeletons, shared by the operator interface (dataflow_ops.c) and the layer's own ops */
#ifndef SKELETONS_H
#define SKELETONS_H

#include "dataflow_amd.h"

/* nickname "<base>[_<dt0>[_<dt1>]]", argument tags, fingerprint; `base` has to be a string literal */
__attribute__((visibility("hidden"))) void dataflow_fill_skeleton(Op_Skeleton * skeleton, const char * base, DataflowDatatype dt0, DataflowDatatype dt1,
																  int num_args, const DataflowDatatype * arg_dtypes);

#endif
