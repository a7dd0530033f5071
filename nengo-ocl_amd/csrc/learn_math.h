// Element of a weight-update rule, shared by the rules' own kernel and the launch that multiplies by
// the matrix they change.
#pragma once

#include "nhip_common.h"

// One element of a rule's change.  Products and sums are rounded one by one in the order the
// expressions are written in clra_nonlinearities.py:2130-2131 (BCM: aux = theta of the row),
// :2237-2238 (Oja: the weight) and :2349-2350 (Voja: the encoder), left to right.
template <int RULE>
__device__ __forceinline__ float learn_element(float alpha, float beta, float learn, float scale,
                                               float x, float y, float aux) {
    if (RULE == NHIP_RULE_BCM)
        return __fmul_rn(__fmul_rn(__fmul_rn(alpha, y), __fsub_rn(y, aux)), x);
    if (RULE == NHIP_RULE_OJA)
        return __fmul_rn(__fmul_rn(alpha, y),
                         __fsub_rn(x, __fmul_rn(__fmul_rn(beta, aux), y)));
    return __fmul_rn(__fmul_rn(__fmul_rn(alpha, learn), y),
                     __fsub_rn(__fmul_rn(scale, x), aux));
}
