/*
 * norm_rows.h -- which launches of the RMS norm's forward and bwd_x have one row on a wave and four on a work-group, the others one on a
 * work-group: for the kernels (norm.hip, where both sides are measured) and the host's grid (launch_config.c), which have to agree.
 */
#ifndef NORM_ROWS_H
#define NORM_ROWS_H

#define NORM_WAVE_ROW_COLS 1024
#define NORM_WAVE_ROW_LEAST_ROWS 8192
#define NORM_WAVE_ROWS_PER_GROUP 4
#define NORM_ROWS_ON_WAVES(n_rows, n_cols) ((n_cols) <= NORM_WAVE_ROW_COLS && (n_rows) >= NORM_WAVE_ROW_LEAST_ROWS)

#endif
