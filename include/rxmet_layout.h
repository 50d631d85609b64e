/*
 * rxmet_layout.h — layers whose hidden size is not a multiple of the kernels' unit tile.
 *
 * The quantised recurrences work on whole tiles of 16 units.  A layer of another size runs with
 * its weights, biases, initial states and output gradients widened to whole tiles by zeros, and
 * its outputs and gradients narrowed again; rxmet_block_copy does either for all tensors of a
 * call in one launch.
 */
#ifndef RXMET_LAYOUT_H
#define RXMET_LAYOUT_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/*
 * One tensor: dst [outer, rows_dst, groups, cols_dst] from src [outer, rows_src, groups,
 * cols_src], both row-major fp32, not overlapping.  Elements that src does not have are zero,
 * elements that dst does not have are dropped.
 */
typedef struct rxmet_block_job {
  const float *src;
  float *dst;
  int64_t outer;
  int32_t rows_src, rows_dst, groups, cols_src, cols_dst, reserved; /* reserved: 0 */
} rxmet_block_job;

enum { RXMET_BLOCK_JOBS = 16 };

/* All jobs (1 <= n <= RXMET_BLOCK_JOBS) in one launch; jobs with an empty dst are allowed. */
int rxmet_block_copy(int32_t n, const rxmet_block_job *jobs, void *stream);

#ifdef __cplusplus
}
#endif

#endif
