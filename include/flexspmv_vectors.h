/* C interface of the vector updates of a conjugate-gradient iteration around a fused y = A p, p . y launch on
 * MI355X (gfx950).
 *
 * One library (libflexspmv_vectors.so) exports every symbol below.  All data pointers are device pointers valid on
 * the current device, all calls are asynchronous on the given hipStream_t, and none of them allocates.  The scalars
 * (r . r, p . A p) stay in device memory, so an iteration needs no word from the GPU on the host.
 *
 * The reference leaves these updates to torch (its Poisson model runs under EASIER's CG solver,
 * test_modules/utils.py:74-85): eight element-wise kernels and a library dot product per iteration.
 */
#ifndef FLEXSPMV_VECTORS_H_
#define FLEXSPMV_VECTORS_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define FLEXSPMV_VECTORS_ABI_VERSION 2

/* Return codes (negative); positive values are hipError_t codes passed through unchanged. */
enum flexspmv_vectors_status {
  FLEXSPMV_VECTORS_OK = 0,
  FLEXSPMV_VECTORS_ERR_BAD_ARGUMENT = -1 /* NULL pointer, n < 1, value width not 4 or 8 */
};

/* Values the partials of flexspmv_cg_step take (value_bytes each), whatever n is. */
#define FLEXSPMV_CG_MAX_PARTIALS 2048

/* r -= alpha ap with alpha = rr / pap (both one value), and what the blocks add to the new r . r.
 * value_bytes: 4 (float) or 8 (double).  r: updated in place; ap: read; partials: FLEXSPMV_CG_MAX_PARTIALS values,
 * filled as far as flexspmv_cg_direction with the same n reads them.  No array may overlap another. */
int flexspmv_cg_step(void* r, const void* ap, const void* rr, const void* pap, int64_t n, int value_bytes, void* partials,
                     void* stream);

/* x += alpha p with the same alpha (x: updated in place), rr_new = sum of the partials (in a fixed order) and
 * p_next = r + (rr_new / rr) p.  p_next may be p; rr_new must not be rr or pap; no other arrays may overlap. */
int flexspmv_cg_direction(void* x, void* p_next, const void* p, const void* r, const void* rr, const void* pap,
                          void* rr_new, const void* partials, int64_t n, int value_bytes, void* stream);

/* Message of the last failed call on this thread ("" if none). */
const char* flexspmv_vectors_last_error(void);

/* FLEXSPMV_VECTORS_ABI_VERSION the library was built against. */
int flexspmv_vectors_abi_version(void);

#ifdef __cplusplus
}
#endif
#endif /* FLEXSPMV_VECTORS_H_ */
