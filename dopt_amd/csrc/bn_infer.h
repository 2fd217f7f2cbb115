// What the kernels of inference batch norm take (bn.hip, bn_copies.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace dopt {

struct InferArgs {
    const float4 *x;         // the operand, or null: [splits] copies of it at `partial`, to be added, and `addend` per channel
    const float4 *partial;
    const float *addend;
    int splits;
    unsigned n4, C, inner4, units, upr, W;   // quads; channels; quads of a row; units in all and of a row; pixels of an image row
    double eps;
    const float *scale, *bias, *mean, *var;
    float4 *y;               // either may be null
    float *pooled;
    int relu;
};

// bn_copies.hip: a small launch whose operand is many copies.
int bn_infer_copies(const InferArgs &g);

}  // namespace dopt
