// fp32 MFMA tile engine shared by the SGEMM and the implicit-GEMM convolution kernels.
//
// A workgroup of WM x WN wavefronts owns a BM x BN output tile; each wavefront owns a
// (BM/WM) x (BN/WN) sub-tile held as MI x NI accumulators of v_mfma_f32_32x32x2_f32 (16 VGPRs
// each).  Operand slabs of BK reduction steps are staged in LDS k-major -- As[k][m], Bs[k][n] --
// so that the fragment a lane feeds to the matrix core (A: row = lane % 32, k = lane / 32; B:
// col = lane % 32, k = lane / 32) is one conflict-free ds_read_b32.  LDS is double buffered: the
// next slab is fetched from global memory into registers while the current one is multiplied,
// then written to the other buffer, so each slab costs one barrier.
#pragma once

#include <hip/hip_runtime.h>

namespace dopt {

typedef float v16f __attribute__((ext_vector_type(16)));

template <int BM_, int BN_, int WM_, int WN_>
struct Tile {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_;
    static constexpr int THREADS = 64 * WM * WN;
    static constexpr int MI = BM / WM / 32, NI = BN / WN / 32;  // 32x32 accumulators per wavefront
    static constexpr int LDA = BM + 4, LDB = BN + 4;             // LDS row strides (floats), 16-byte aligned rows
};

// Multiplies one LDS slab into the wavefront's accumulators.
//   As, Bs : slab bases;  a_off/b_off : the wavefront's first row / column inside the block tile.
// Software pipelined: the fragments of step ks+1 are requested from LDS before the MFMAs of step
// ks are issued, so the LDS latency hides behind the matrix work.
template <int BK, int LDA, int LDB, int MI, int NI>
__device__ inline void mma_slab(const float *As, const float *Bs, int a_off, int b_off, v16f (&acc)[MI][NI], int lane)
{
    const int kh = lane >> 5, l32 = lane & 31;
    const float *ap = As + kh * LDA + a_off + l32;
    const float *bp = Bs + kh * LDB + b_off + l32;
    float a[MI], b[NI];
#pragma unroll
    for (int i = 0; i < MI; i++) a[i] = ap[32 * i];
#pragma unroll
    for (int j = 0; j < NI; j++) b[j] = bp[32 * j];
#pragma unroll
    for (int ks = 0; ks < BK / 2; ++ks) {
        float na[MI], nb[NI];
#pragma unroll
        for (int i = 0; i < MI; i++) na[i] = ks + 1 < BK / 2 ? ap[(2 * ks + 2) * LDA + 32 * i] : 0.0f;
#pragma unroll
        for (int j = 0; j < NI; j++) nb[j] = ks + 1 < BK / 2 ? bp[(2 * ks + 2) * LDB + 32 * j] : 0.0f;
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < MI; i++) a[i] = na[i];
#pragma unroll
        for (int j = 0; j < NI; j++) b[j] = nb[j];
    }
}


// Compile-time loop: f(StepTag<I>{}) for I = 0 .. N-1, so that the body can use I in constant
// expressions (register-array indices, `if constexpr`).
template <int I>
struct StepTag {
    static constexpr int value = I;
};

template <int I, int N, class F>
__device__ inline void static_for(F &&f)
{
    if constexpr (I < N) {
        f(StepTag<I>{});
        static_for<I + 1, N>(f);
    }
}

template <int MI, int NI>
__device__ inline void zero_acc(v16f (&acc)[MI][NI])
{
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
}

// ---------------------------------------------------------------------------------------------------------------------
// fp32 products on the bf16 matrix instructions.
//
// v_mfma_f32_32x32x16_bf16 multiplies 16 reduction steps in half the cycles that v_mfma_f32_32x32x2_f32 takes for two
// (measured on this chip: 1770 against 124 TFLOP/s), so six of them per sixteen steps still run at 2.4 times the fp32
// rate.  An fp32 value of ordinary size is the exact sum of three bf16 values: h = bf16(a), m = bf16(a - h), l = bf16(a - h - m),
// each rounded to nearest; 24 significand bits are three times 8, so nothing is left over (Henry, Tang and Heinecke,
// "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", 2019).  bf16 has the exponents
// of fp32 but not its small steps: the parts of a value below 2^-110 would fall under the smallest bf16 number.  So operands
// are multiplied by 2^24 (kSplitUp) on their way to the split, which makes every nonzero part of every fp32 value a normal
// bf16 number, and sums by 2^-48 (kSplitDown); both are exact, and no other bit changes.
// Of the nine products of two such sums the six largest are taken; the three left out (m.l, l.m, l.l) are together at most 2^-24 of |a.b|, what ONE
// fp32 rounding of the product may be off by, and 2^-28 of it on average.  Every product of two bf16 values is exact
// in fp32, and all sums are fp32.  Against float64 the result is not less accurate than the fp32 instruction's, because
// it is rounded less often; with the large products and the small rest in accumulators of their own, where registers
// allow, it is three times as accurate (relative 2-norm of the error over normally distributed operands of 64 / 512 /
// 4096 terms: 5.0e-8 / 1.3e-7 / 3.8e-7, the fp32 instruction 1.4e-7 / 4.0e-7 / 1.2e-6, one accumulator for all six
// 1.1e-7 / 3.4e-7 / 9.8e-7).
//
// The split of an infinity, or of a value that is one after the multiplication (2^104 and more), holds NaNs, and a sum of 2^80
// and more overflows.  Kernels that use it look at their finished accumulators and form a tile that is not finite a second time
// with the fp32 instruction, so such operands and sums give what they always gave.
//
// The instruction adds the eight products of a lane half's eight slots in one go, whatever their order (measured: no
// permutation of the eight changes a bit).  So the six products of FOUR reduction steps fill the eight slots of three
// instructions in pairs that stay what they are when the two operands change places,
//     (h, m) . (h, m)      (h, m) . (m, h)      (l, h) . (h, l)
// and a product and its transpose computed as B^T A^T have the same bits.
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

constexpr float kSplitUp = 0x1p24f, kSplitDown = 0x1p-48f;

// Two values' h, m and l parts, each pair packed into one word (first value in the low half): 11 VALU instructions.
__device__ __forceinline__ void split_pair(float a, float b, unsigned &h, unsigned &m, unsigned &l)
{
    const v2f x = {a, b};
    h = __builtin_bit_cast(unsigned, __builtin_convertvector(x, v2bf));
    const v2f r = {a - __builtin_bit_cast(float, h << 16), b - __builtin_bit_cast(float, h & 0xffff0000u)};
    m = __builtin_bit_cast(unsigned, __builtin_convertvector(r, v2bf));
    const v2f s = {r.x - __builtin_bit_cast(float, m << 16), r.y - __builtin_bit_cast(float, m & 0xffff0000u)};
    l = __builtin_bit_cast(unsigned, __builtin_convertvector(s, v2bf));
}

// Four reduction steps of one row: their h parts in hm.x, .y, their m parts in hm.z, .w, their l parts in l.
__device__ __forceinline__ void split_quad(float4 q, v4u &hm, uint2 &l)
{
    unsigned h0, h1, m0, m1;
    split_pair(q.x, q.y, h0, m0, l.x);
    split_pair(q.z, q.w, h1, m1, l.y);
    hm = v4u{h0, h1, m0, m1};
}

__device__ __forceinline__ v16f mfma_bf16(v4u a, v4u b, v16f c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

// The finished sums: of the h.h products and of the five small ones.
template <int MI, int NI>
__device__ __forceinline__ void add_acc(v16f (&acc)[MI][NI], const v16f (&low)[MI][NI])
{
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = (acc[i][j][v] + low[i][j][v]) * kSplitDown;
}

// Ends a chain of sums: what it holds goes to `sum`, and the next one begins.
template <int MI, int NI>
__device__ __forceinline__ void move_acc(v16f (&sum)[MI][NI], v16f (&acc)[MI][NI])
{
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                sum[i][j][v] += acc[i][j][v];
                acc[i][j][v] = 0.0f;
            }
}

// Whether this lane's accumulators hold an infinity or a NaN: x * 0 is 0 for finite x only.
template <int MI, int NI>
__device__ __forceinline__ int not_finite(const v16f (&acc)[MI][NI])
{
    float probe = 0.0f;
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) probe = __builtin_fmaf(acc[i][j][v], 0.0f, probe);
    return probe != 0.0f;
}

// The sums of a tile that was formed twice: the first time's where they are finite, so that a finite value does not depend on
// what else lies in its tile.
template <int MI, int NI>
__device__ __forceinline__ void keep_finite(v16f (&acc)[MI][NI], const v16f (&again)[MI][NI])
{
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = acc[i][j][v] * 0.0f == 0.0f ? acc[i][j][v] : again[i][j][v];
}

// Row of accumulator register v of a 32x32 tile for this lane; the column is lane % 32.
__device__ inline int acc_row(int v, int lane) { return 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3); }

// Workgroup ids are handed to the 8 XCDs round-robin and each XCD has its own L2.  Remap so that
// every XCD works on one contiguous range of logical ids: work items that share an operand
// (adjacent logical ids) then hit the same L2.  Returns false for the padding ids past `total`.
__device__ inline bool xcd_remap(unsigned bid, unsigned total, unsigned *logical)
{
    const unsigned per = (total + 7u) / 8u;
    const unsigned l = (bid & 7u) * per + (bid >> 3);
    *logical = l;
    return l < total;
}

inline unsigned xcd_grid(unsigned total) { return ((total + 7u) / 8u) * 8u; }

// Buffer-resource loads: the hardware range check returns 0 for an offset at or past the end of
// the buffer, so a masked element is loaded from kOobOffset instead of being branched around.
// That keeps the gather loops branch-free (one basic block the scheduler can interleave with the
// MFMAs) and the address arithmetic 32-bit.  Valid byte offsets must stay below 2^31, and a masked
// lane must carry exactly kOobOffset: the wave-uniform offset is added to it without wrapping.
constexpr unsigned kOobOffset = 0x80000000u;

__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void *base, size_t bytes)
{
    const size_t clamped = bytes < 0x7fffffffu ? bytes : 0x7fffffffu;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)clamped, 0x00020000);
}

// voffset: per-lane byte offset (VGPR); soffset: wave-uniform byte offset (SGPR).
__device__ inline float buffer_load_f32(__amdgpu_buffer_rsrc_t r, unsigned voffset, unsigned soffset)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)voffset, (int)soffset, 0));
}

__device__ inline float4 buffer_load_f32x4(__amdgpu_buffer_rsrc_t r, unsigned voffset, unsigned soffset)
{
    // Keep the builtin's own vector type: converting it to an ext_vector_type first makes the
    // compiler load a single dword and splat it.
    auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)voffset, (int)soffset, 0);
    static_assert(sizeof(v) == sizeof(float4), "b128 load must yield 16 bytes");
    return __builtin_bit_cast(float4, v);
}

__device__ inline float2 buffer_load_f32x2(__amdgpu_buffer_rsrc_t r, unsigned voffset, unsigned soffset)
{
    auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)voffset, (int)soffset, 0);
    static_assert(sizeof(v) == sizeof(float2), "b64 load must yield 8 bytes");
    return __builtin_bit_cast(float2, v);
}

}  // namespace dopt
