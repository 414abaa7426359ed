/* optim_internal.h -- entry points of libchurten_optim.so for the operator
 * library (torch_ops.cpp), beside the public ones of include/churten_optim.h. */
#ifndef CHURTEN_OPTIM_INTERNAL_H
#define CHURTEN_OPTIM_INTERNAL_H

#include <stddef.h>
#include <stdint.h>

#include "../../include/churten_optim.h"

#ifdef __cplusplus
extern "C" {
#endif

/* The workspace size from which a *_ws call on R replicas can run as a single
 * launch ("One launch per call" in optim_drivers.h); 0 where it cannot. */
size_t ts_single_launch_bytes(int64_t R);

/* ts_sgd_step and ts_sgd_step_segments with a workspace, as the other
 * optimizers' *_ws forms. SGD has no constants to precompute, so these are for
 * the single launch alone. */
int ts_sgd_step_ws(const ts_rt_buf* bufs, ts_dtype dtype, void* state_steps, const void* lr,
                   const void* momentum, const void* dampening, const void* weight_decay,
                   const uint8_t* active_mask, int64_t R, int64_t T, uint32_t flags,
                   void* out_zero, void* workspace, size_t workspace_bytes, void* stream);
int ts_sgd_step_segments_ws(const ts_rt_buf* bufs, const ts_segment* grads, int n_grads,
                            ts_dtype dtype, void* state_steps, const void* lr,
                            const void* momentum, const void* dampening,
                            const void* weight_decay, const uint8_t* active_mask, int64_t R,
                            int64_t T, uint32_t flags, void* out_zero, void* workspace,
                            size_t workspace_bytes, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* CHURTEN_OPTIM_INTERNAL_H */
