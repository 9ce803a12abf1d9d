// Output coordinates of a strided layer in two launches, for callers of this repository (rules.hip).
#pragma once
#include <stdint.h>

#include "../../include/sphconv_hip.h"

#ifdef __cplusplus
extern "C" {
#endif
/* 64-bit words of the cells a count adds to: device memory, zeros before the call and, once *total has been written, after. */
int sph_outcoords2_cell_words(void);
/* int32 entries of the scratch the two calls share (16-byte aligned), or 0 for a geometry that sph_outcoords_count and _fill serve. */
int sph_outcoords2_scratch_ints(const sph_geom *g);
/* The row count, to *total (pinned host memory), as the kernel's last store. */
int sph_outcoords2_count(const int32_t *z_idx, const int32_t *z_ptr, int in_rows, const sph_geom *g, int32_t *scratch, uint64_t *cells,
                         int32_t *total, void *stream);
/* oz_ptr, and at most out_rows rows of oz_idx and row_cols (may be null). */
int sph_outcoords2_fill(const sph_geom *g, const int32_t *scratch, int32_t *oz_ptr, int32_t *oz_idx, int out_rows, int32_t *row_cols,
                        void *stream);
#ifdef __cplusplus
}
#endif
