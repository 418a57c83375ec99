/*
 * norm_rows.h -- where the RMS norm's forward and bwd_x run on kernels with one row on a wave and four on a work-group, and the forward on one
 * with all loads of a long row out at once (norm.hip, where both sides are measured): for the submit wrappers, which choose, the
 * launch configurations and the kernels.
 */
#ifndef NORM_ROWS_H
#define NORM_ROWS_H

#define NORM_WAVE_ROW_COLS 1024
#define NORM_WAVE_ROW_LEAST_ROWS 8192
#define NORM_WAVE_ROWS_PER_GROUP 4
#define NORM_ROWS_ON_WAVES(n_rows, n_cols) ((n_cols) <= NORM_WAVE_ROW_COLS && (n_rows) >= NORM_WAVE_ROW_LEAST_ROWS)

#define NORM_UNROLLED_COLS 4608
#define NORM_UNROLLED_LEAST_ROWS 2500
#define NORM_LONG_ROWS(n_rows, n_cols) ((n_cols) > NORM_UNROLLED_COLS && (n_rows) >= NORM_UNROLLED_LEAST_ROWS)

#endif
