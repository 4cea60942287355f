/* Entry points beside leniax_amd.h that let a caller keep a workspace or pass a scalar by value; the same
 * conventions (status codes, streams, empty batches). */
#ifndef LENIAX_AMD_EXT_H
#define LENIAX_AMD_EXT_H

#include "leniax_amd.h"

#ifdef __cplusplus
extern "C" {
#endif

/* lx_potential_direct_adjoint with a workspace of lx_potential_direct_adjoint_size bytes for the kernel side's partial
 * sums, which then runs on the matrix cores over tiles of the worlds (without one, and for few cells and taps:
 * one workgroup per kernel tap over all worlds).  Deterministic: the partial sums are added in a fixed order. */
int lx_potential_direct_adjoint_size(const lx_rule* rule, int64_t B, int32_t kh, int32_t kw, size_t* bytes);
int lx_potential_direct_adjoint_work(const lx_rule* rule, const float* state_d, int64_t B, const float* kern_d,
                                     int32_t kh, int32_t kw, const float* dpot_d, float* dstate_d,
                                     float* dkern_d, void* work_d, void* stream);

/* lx_update with one dt for every world, by value (no device scalar to fill first). */
int lx_update_dt(const lx_rule* rule, const float* state_d, int64_t B, const void* K_half_d, int64_t k_bstride,
                 const float* gf_d, int64_t gf_bstride, const float* w_d, int64_t w_bstride, float dt,
                 float* state_out_d, float* field_d, float* potential_d, void* work_d, void* stream);

#ifdef __cplusplus
}
#endif

#endif
