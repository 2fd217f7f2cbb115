// Inference batch norm of small tensors that a convolution left as many partial copies.  A file, and so a code object, of its own: in
// that of bn.hip it took the large kernels there, which were not changed, 1.3% of their time ([128, 64, 32, 32], ten layer operations one
// after the other 128.6 us, 130.1 so).
#include "bn_infer.h"
#include "common.h"
#include "pool2x2.h"

using namespace dopt;

namespace {

constexpr unsigned kBlock = 256;

// The sum of a value's copies, sixteen of them in flight, added in ascending order.
__device__ inline float4 infer_copies(const InferArgs &g, unsigned i)
{
    float4 acc = g.partial[i];
    const int last = g.splits - 1;
    for (int s = 1; s <= last; s += 16) {
        float4 v[16];
#pragma unroll
        for (int j = 0; j < 16; j++) v[j] = g.partial[(size_t)min(s + j, last) * g.n4 + i];
#pragma unroll
        for (int j = 0; j < 16; j++)
            if (s + j <= last) acc = make_float4(acc.x + v[j].x, acc.y + v[j].y, acc.z + v[j].z, acc.w + v[j].w);
    }
    return acc;
}

// bn_infer_k (bn.hip; units, arithmetic and order are its) for a small launch behind many copies, which is bound by what it waits for
// one after the other: the copies are on their way before the coefficients are made, sixteen at once.  VGG-16 on one image, 13
// such launches of up to sixteen copies: 191 us with bn_infer_k, 180 with this one.
template <bool kPool>
__global__ __launch_bounds__(kBlock) void bn_infer_copies_k(InferArgs g)
{
    __shared__ float4 coef[kBlock + 1];   // mean, scale * rstd, bias; what is added to the copies
    const unsigned begin = blockIdx.x * kBlock, end = min(begin + kBlock, g.units);
    const unsigned row0 = begin / g.upr, rows = (end - 1) / g.upr - row0 + 1;
    const unsigned i = begin + threadIdx.x, row = min(i, end - 1) / g.upr, j = i - row * g.upr;
    const bool two = kPool && g.W != 2;   // a pooled unit is one quad, a window, or the quads of two
    unsigned q = i, step = 0;
    float4 v0, v1;
    if (i < end) {
        if (kPool && !two) q = row * g.inner4 + j;
        if (two) {
            const unsigned W4 = g.W / 4, p = j / W4;
            q = row * g.inner4 + 2 * p * W4 + (j - p * W4);
            step = W4;
            v1 = infer_copies(g, q + W4);
        }
        v0 = infer_copies(g, q);
    }
    for (unsigned r = threadIdx.x; r < rows; r += kBlock) {
        const unsigned c = (row0 + r) % g.C;
        const double rstd = 1.0 / sqrt((double)g.var[c] + g.eps);
        coef[r] = make_float4(g.mean[c], (float)((double)g.scale[c] * rstd), g.bias[c], g.addend ? g.addend[c] : 0.0f);
    }
    __syncthreads();
    if (i >= end) return;
    const float4 k = coef[row - row0];
    auto one = [&](float v) {
        if (g.addend) v += k.w;
        const float r = k.y * (v - k.x) + k.z;
        return g.relu && r < 0.0f ? 0.0f : r;
    };
    auto value = [&](float4 v) { return make_float4(one(v.x), one(v.y), one(v.z), one(v.w)); };
    const float4 a = value(v0);
    if (!kPool || g.y) g.y[q] = a;
    if (kPool && !two) g.pooled[i] = pool2x2(a.x, a.y, a.z, a.w);
    if (two) {
        const float4 b = value(v1);
        if (g.y) g.y[q + step] = b;
        ((float2 *)g.pooled)[i] = make_float2(pool2x2(a.x, a.y, b.x, b.y), pool2x2(a.z, a.w, b.z, b.w));
    }
}

}  // namespace

namespace dopt {

int bn_infer_copies(const InferArgs &g)
{
    const dim3 grid((g.units + kBlock - 1) / kBlock);
    if (g.pooled) hipLaunchKernelGGL(bn_infer_copies_k<true>, grid, dim3(kBlock), 0, stream(), g);
    else hipLaunchKernelGGL(bn_infer_copies_k<false>, grid, dim3(kBlock), 0, stream(), g);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

}  // namespace dopt
