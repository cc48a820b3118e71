/* hq_internal.h - helpers shared by the library's C and HIP sources (not part of the ABI). */
#ifndef HQ_INTERNAL_H
#define HQ_INTERNAL_H

#include <stddef.h>
#include <stdint.h>

#include "hq.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Records a message for hq_last_error() and returns -1. */
int hq_internal_fail(const char *fmt, ...) __attribute__((format(printf, 1, 2)));

/* Values and bytes per block of a ggml block type hq_mat_upload accepts: 0, or -1 for other types. */
int hq_internal_block_shape(int ggml_type, uint32_t *values, uint32_t *bytes);
/* The accepted block types, for messages ("Q8_0 = 8, ..."). */
const char *hq_internal_supported_types(void);

/* Whether hq_gemm_swiglu on M <= 64 rows of a pair matrix of 2 * rows rows is one small-tile kernel (else hq_gemm's kernel
 * and a pass over its product); no device is touched. */
int hq_internal_swiglu_small(int ggml_type, int M, uint32_t rows, uint32_t K, int n_cu);

/* Tokens of the backend's layer-loop pass, for activations of bytes_per_token. */
int hq_internal_pass_tokens(size_t max_seq, size_t bytes_per_token, size_t free_bytes);

/* The rows of n matrices of one type and width (Hugging Face order, one after the other) as one resident matrix. */
int hq_internal_upload_cat(const hq_wmat_t *const *w, int n, int device, hq_mat **out);

#ifdef __cplusplus
}
#endif
#endif
