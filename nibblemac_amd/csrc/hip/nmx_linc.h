/* The DeltaNet kernels of prefill chunks (nmx_linc.hip); not part of the ABI. */
#ifndef NMX_LINC_H
#define NMX_LINC_H

#include "nmx_internal.h"

/* whether lin_rulec_k takes the (validated) recurrence */
bool nmx_lin_rulec_ok(const nmx_lin_args &a);
int nmx_lin_rulec(nmx_ctx *ctx, const nmx_lin_args &a);
/* conv, norms and gates into p's buffers, then the recurrence over them (a.qkv = p.out, a.decay =
 * p.decay, a.beta = p.beta); p.conv_k = 4, no xin, more than 8 tokens; validated by the caller */
int nmx_lin_mixc(nmx_ctx *ctx, const nmx_lin_pre_args &p, const nmx_lin_args &a);

#endif
