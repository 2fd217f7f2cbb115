// Convolution forward, backward-data and backward-filter as implicit GEMMs on matrix instructions: most kernels on the bf16 one
// with each fp32 value split into three parts (mfma_core.h), the 2 x 2-image kernels on the fp32 one.
// Replaces cudnnConvolutionForward / BackwardData / BackwardFilter as called at
// cuda/source/dopt/cuda/nnet/cudnn7.d:154, :199, :244.  The reference configures cuDNN with
// CUDNN_CONVOLUTION (cudnn7.d:87), i.e. a TRUE convolution: the filter is flipped,
//     y[n,k,p,q] = sum_{c,r,s} x[n,c,p*sy-ph+r, q*sx-pw+s] * w[k,c,R-1-r,S-1-s]
// (pinned by the known-answer test at core/source/dopt/core/ops/nnet.d:270-293).  Writing
// r' = R-1-r, s' = S-1-s the filter is read in plain memory order and the flip moves onto the
// input offset: x[n,c,p*sy-ph+(R-1-r'), q*sx-pw+(S-1-s')].
//
// Forward and backward-data share one "gather" kernel:
//     out[n,m,oh,ow] = sum_{tap,ci} Wp[tap,ci][m] * in[n,ci,ih(oh,tap),iw(ow,tap)]
// GEMM view: M = output channels of the op, columns = output pixels (n,oh,ow), reduction =
// (tap, ci) with ci padded to a multiple of 16 so that a 16-deep slab has ONE tap: the input
// offset and the bounds mask are then uniform over the slab, and a lane's loads for successive
// channels differ by a wave-uniform offset.  Wp is the filter re-packed once per call as its bf16 parts, in the order
// the tile has in LDS, so the A tile goes global -> LDS with 128-bit accesses.
//
// Backward-filter is a GEMM with M = K (output channels), columns = (r', s', c) tap-major with c
// padded to 16, reduction = output pixels (n,p,q); both operands are gathered with lanes along
// the pixel index (contiguous in memory).  A second kernel sums the reduction splits and permutes
// the columns back to [K][C][R][S].
//
// All gathers go through buffer-resource loads whose range check supplies the zero padding, so
// the inner loops are branch-free.  Layers with few output tiles split the reduction; partial
// tiles go to the workspace and are summed in a fixed order -- no float atomics, so results are
// reproducible.
#include <algorithm>
#include <utility>
#include <vector>

#include "common.h"
#include "mfma_core.h"

namespace {

using namespace dopt;

constexpr int BK = 16;

// Filters packed as bf16 parts.  A value whose parts are no numbers (2^103 and more, infinities, NaNs) has this NaN for its h part
// and its bits as they are in the other two.
constexpr unsigned short kPackedRaw = 0x7fff;

// Two neighbouring channels' parts, each pair one word.
__device__ __forceinline__ void split_packed(float a, float b, unsigned &h, unsigned &m, unsigned &l)
{
    split_pair(a * kSplitUp, b * kSplitUp, h, m, l);
    const unsigned bits[2] = {__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b)};
    constexpr unsigned kTop = 0x73000000u;   // 2^103
    if (__any(max(bits[0] & 0x7fffffffu, bits[1] & 0x7fffffffu) >= kTop)) {
#pragma unroll
        for (int v = 0; v < 2; v++) {
            const unsigned shift = 16 * v, keep = 0xffff0000u >> shift;
            if ((bits[v] & 0x7fffffffu) < kTop) continue;
            h = (h & keep) | (unsigned)kPackedRaw << shift;
            m = (m & keep) | bits[v] >> 16 << shift;
            l = (l & keep) | (bits[v] & 0xffffu) << shift;
        }
    }
}

// The fp32 value e of a fragment's eight.
__device__ __forceinline__ float packed_value(const v4u (&f)[3], int e)
{
    unsigned q[3];
#pragma unroll
    for (int t = 0; t < 3; t++) q[t] = e & 1 ? f[t][e / 2] >> 16 : f[t][e / 2] & 0xffffu;
    auto val = [&](int t) { return __builtin_bit_cast(float, q[t] << 16); };
    return q[0] == kPackedRaw ? __builtin_bit_cast(float, q[1] << 16 | q[2]) : (val(0) + val(1) + val(2)) * (1.0f / kSplitUp);
}

// ------------------------------------------------------------------------------------ gather

struct GatherConv {
    const float *in;   // gathered operand [N, Cin, IH, IW]
    const float *wp;   // packed filter [16-channel chunk][tap][Mp / 4][3 parts][2 halves][4 rows][8 channels], bf16
    float *out;        // [N, Mout, OH, OW], or `splits` partial copies of it
    int N, Cin, IH, IW, Mout, OH, OW, R, S;
    int padH, padW, strideH, strideW;
    int CinPad, Mp, ncols;
    int mtiles, ntiles, slabs_total, slabs_per_split, splits;
    size_t out_elems, in_bytes;
    // where output pixel (oh, ow) of this problem lands: row oh * out_sy + out_oy, column ow * out_sx +
    // out_ox of a plane of out_plane elements and out_OW columns (the whole tensor, or every
    // stride-th pixel of it when a strided backward-data pass is run class by class)
    int out_plane, out_OW, out_sy, out_sx, out_oy, out_ox;
};

// The products run on the bf16 matrix instruction (mfma_core.h).  The filter is packed as bf16 parts; an input value is split
// once, when it is stored in LDS.  (Split by every wavefront that reads a value, splitting took 700 vector cycles of a slab beside
// 384 to 768 matrix cycles.)  LDS holds both operands as [part][half][row][8 channels], so a fragment of one part is one
// 128-bit read and neighbouring lanes' reads are neighbours.  A stage is SL slabs; under the matrix instructions of one the next is
// split and stored and the one after it is loaded, each piece pinned to a step, and the workgroup meets once per stage.  Split
// behind the products instead, with every wavefront at the same place: 5 x 5 layers below 101 and 69 us, now 75 and 58.
// 50 images of 48 x 45 x 39, 100 filters of 5 x 5 at stride 2: forward 103 -> 58 us, backward-data 95 -> 75 (with a last stage that
// only multiplies 9 -> 7 us for 2 images of 19 x 46 x 14, as before); 64 -> 64 channels of 3 x 3
// on 64 images of 33 x 31 46 -> 37 us; Wide-ResNet-28-10's two strided 3 x 3 layers backward 270 -> 240 us.  A stage of a
// 64 x 256 tile takes 1.7 us of which 0.9 are matrix time at the rate of a large product; it reads 144 KB of fragments from LDS.
// A chain of sums ends after eight slabs and is added to `sum`: the error grows with the root of a chain's length, and with few
// cuts of the reduction a chain was the whole of it.  Drawn layers (3 to 640 channels, filters of 1, 3 and 5) are 0.8 times as far off float64
// as when it was cut for twice as many workgroups, at most 1.15 times, without the chains up to 1.8 times.  160 -> 320 channels,
// stride 2: 8.5e-8 forward and 8.4e-8 backward-data, without 1.7e-7 both (the fp32 instruction: 2.1e-7, 5.3e-7).  It costs
// 1 to 2 % of the time; four stages in a row, so that nothing is decided within, instead of a test per stage, 3 %.
// Stages of one slab (SL = 1) are for short reductions (see gather_launch): no chains, and registers for two workgroups
// per CU, of which one stores its results or loads its first stage while the other multiplies.
// kBwd: backward-data, of unit stride.
// L: the workgroup's item among the problem's (split, tile) pairs, tile fastest.
template <class T, int SL>
struct GatherLds {
    static constexpr int PA = T::BM + 4, PB = T::BN;   // rows of a part's half (four more: a chunk's parts go to different banks)
    static constexpr int A = SL * 6 * PA * 4, STAGE = A + SL * 6 * PB * 4;   // floats
    static constexpr size_t BYTES = 2 * STAGE * sizeof(float);
};

template <class T, int SL, bool kBwd>
__device__ __forceinline__ void conv_gather_body(const GatherConv &p, unsigned L)
{
    constexpr int BM = T::BM, BN = T::BN, THREADS = T::THREADS, MI = T::MI, NI = T::NI;
    constexpr int CHUNKS = SL * BM * 6;                      // 16-byte pieces of a stage's filter tile
    constexpr int NA = (CHUNKS + THREADS - 1) / THREADS;     // ... of each thread
    constexpr int CPT = 16 * BN / THREADS;                   // channels of a slab that a thread gathers for its pixel
    constexpr int PA = GatherLds<T, SL>::PA, PB = GatherLds<T, SL>::PB, STAGE = GatherLds<T, SL>::STAGE, BOFF = GatherLds<T, SL>::A;
    static_assert((CPT == 4 || CPT == 8) && SL <= 2, "half a piece of LDS or a whole one; two sets of fragments");
    extern __shared__ __attribute__((aligned(16))) float lds[];

    const unsigned tiles = (unsigned)(p.mtiles * p.ntiles);
    const int split = (int)(L / tiles);
    const unsigned tile = L - (unsigned)split * tiles;
    const int mt = (int)(tile % (unsigned)p.mtiles), nt = (int)(tile / (unsigned)p.mtiles);
    const int m0 = mt * BM, n0 = nt * BN;
    const int slab_begin = split * p.slabs_per_split;
    const int slab_end = min(slab_begin + p.slabs_per_split, p.slabs_total);

    const int tid = threadIdx.x, lane = tid & 63, kh = lane >> 5, l32 = lane & 31;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = w / T::WN, wn = w % T::WN;

    const __amdgpu_buffer_rsrc_t rin = make_rsrc(p.in, p.in_bytes);

    // A: this thread's pieces of the stage's filter tile, which lies in memory as one run of 96 bytes a row per slab
    const unsigned a_rows = (unsigned)min(BM, p.Mp - m0);   // rows past the packed ones are zeros (range check)
    unsigned a_voff[NA];
    int a_lds[NA];
#pragma unroll
    for (int i = 0; i < NA; i++) {
        const int f = i * THREADS + tid, sl = f / (BM * 6), g = f - sl * (BM * 6);
        const int block = g / 24, half_part = g / 4 % 6, row = block * 4 + g % 4;
        a_voff[i] = (unsigned)g * 16u;
        a_lds[i] = ((sl * 6 + half_part) * PA + row) * 4;
    }

    // B: the output pixel this thread gathers for, CPT channels of a slab from c0 on
    const int bcol = tid % BN, c0 = w * 64 / BN * CPT;
    const int pix = n0 + bcol;
    const int pix_oob = p.ncols - 1 - pix;  // negative past the last pixel
    const int OHW = p.OH * p.OW;
    const int n_img = pix / OHW, pq = pix - n_img * OHW;
    const int oh = pq / p.OW, ow = pq - oh * p.OW;
    const int chan_stride = p.IH * p.IW;
    const int pix_base = (n_img * p.Cin + c0) * chan_stride;  // element offset of (n, channel c0, 0, 0)
    const int row_limit = p.Cin - c0;                          // channels ci0 + i >= row_limit are padding
    const int b_lds = BOFF + (c0 / 8 * PB + bcol) * 4 + c0 % 8 / 2;

    // running position in the reduction, advanced slab by slab without divisions: all taps of sixteen channels, then the next
    // sixteen, so that a tap finds most of its pixels where the one before left them in the L1
    int slab, ci0, tr, ts;
    auto rewind = [&]() {
        slab = slab_begin;
        const int taps = p.R * p.S, chunk = slab_begin / taps, tap = slab_begin - chunk * taps;
        ci0 = chunk * BK;
        tr = tap / p.S;
        ts = tap - tr * p.S;
    };

    float4 areg[NA];
    float breg[SL][CPT];
    auto load_a = [&](int first) {   // the filter's pieces of the stage that begins with slab `first`
#pragma unroll
        for (int i = 0; i < NA; i++) {
            // (the packed filter may be larger than a buffer resource reaches: a resource per slab; which slab of the stage
            // is the same for a whole wavefront)
            const int sl = SL == 1 ? 0 : (i * THREADS + w * 64) / (BM * 6);
            const bool have = first + sl < slab_end && (CHUNKS % THREADS == 0 || i * THREADS + w * 64 < CHUNKS);
            const __amdgpu_buffer_rsrc_t rwp = make_rsrc(p.wp + ((size_t)(have ? first + sl : 0) * p.Mp + m0) * 24, have ? (size_t)a_rows * 96 : 0);
            areg[i] = buffer_load_f32x4(rwp, a_voff[i], 0);
        }
    };
    auto pixel = [&]() {   // byte offset of this thread's input pixel for the slab at the running position, or kOobOffset
        int ih, iw, bad = pix_oob | (slab_end - 1 - slab);
        if constexpr (!kBwd) {
            ih = oh * p.strideH - p.padH + (p.R - 1 - tr);
            iw = ow * p.strideW - p.padW + (p.S - 1 - ts);
        } else {
            ih = oh + p.padH - (p.R - 1 - tr);
            iw = ow + p.padW - (p.S - 1 - ts);
        }
        bad |= ih | (p.IH - 1 - ih) | iw | (p.IW - 1 - iw);  // sign bit set: outside the input
        return bad < 0 ? kOobOffset : (unsigned)(pix_base + ih * p.IW + iw) * 4u;
    };
    auto next_slab = [&]() {
        ++slab;
        if (++ts == p.S) {
            ts = 0;
            if (++tr == p.R) {
                tr = 0;
                ci0 += BK;
            }
        }
    };
    // Channels past the last one are read as they lie (another image's, or zeros past the tensor): their filter values are zeros.
    // Where that makes a NaN of an infinity the sums are formed again without them: masked.  (Left out at once, by a select per
    // load, they cost 6 % of the 5 x 5 layers' time; by one per load of the last sixteen channels 3 %.)
    auto load_b = [&](int sl, int i, unsigned voff, auto masked_tag) {
        if (decltype(masked_tag)::value) voff = ci0 + i < row_limit ? voff : kOobOffset;
        breg[sl][i] = buffer_load_f32(rin, voff, (unsigned)((ci0 + i) * chan_stride) * 4u);
    };
    auto store_a = [&](float *buf) {
#pragma unroll
        for (int i = 0; i < NA; i++)
            if (CHUNKS % THREADS == 0 || i * THREADS + tid < CHUNKS) *(float4 *)(buf + a_lds[i]) = areg[i];
    };
    constexpr int PAIRS = CPT / 2;   // of a slab: four make a 16-byte piece per part, two half of one
    unsigned q[3][PAIRS];
    auto split_b = [&](int sl, int e) {
        split_pair(breg[sl][2 * e] * kSplitUp, breg[sl][2 * e + 1] * kSplitUp, q[0][e], q[1][e], q[2][e]);
    };
    auto store_b = [&](float *buf, int sl) {
#pragma unroll
        for (int t = 0; t < 3; t++) {
            float *const o = buf + b_lds + (sl * 6 + t * 2) * PB * 4;
            if constexpr (PAIRS == 4) *(v4u *)o = v4u{q[t][0], q[t][1], q[t][2], q[t][3]};
            else *(uint2 *)o = make_uint2(q[t][0], q[t][1]);
        }
    };

    v16f acc[MI][NI], low[MI][NI], sum[MI][NI];
    const int a_frag = (kh * PA + wm * (BM / T::WM) + l32) * 4, b_frag = BOFF + (kh * PB + wn * (BN / T::WN) + l32) * 4;
    v4u a[2][MI][3], b[2][NI][3];
    auto fragments = [&](const float *buf, int sl) {
#pragma unroll
        for (int t = 0; t < 3; t++) {
#pragma unroll
            for (int i = 0; i < MI; i++) a[sl & 1][i][t] = *(const v4u *)(buf + a_frag + ((sl * 6 + t * 2) * PA + 32 * i) * 4);
#pragma unroll
            for (int j = 0; j < NI; j++) b[sl & 1][j][t] = *(const v4u *)(buf + b_frag + ((sl * 6 + t * 2) * PB + 32 * j) * 4);
        }
    };
    // Under the matrix instructions of a stage the next one, which is in registers, is split and stored, and the one after
    // it is loaded: a slab's values as soon as the slab before in those registers is stored.
    // The last stage has only its products: with few slabs a block would wait for loads of nothing.
    auto stage = [&](const float *cur, float *nxt, auto more_tag, auto masked_tag) {
        constexpr bool more = decltype(more_tag)::value != 0;
        fragments(cur, 0);
        unsigned voff = 0;
        static_for<0, SL>([&](auto sl_tag) {
            constexpr int sl = decltype(sl_tag)::value;
            static_for<0, 6>([&](auto tag) {
                constexpr int s = decltype(tag)::value;
                if constexpr (s == 0 && sl + 1 < SL) fragments(cur, sl + 1);
                if constexpr (more && s < PAIRS) split_b(sl, s);
                if constexpr (more && s == 0 && sl == 0) {
                    store_a(nxt);
                    load_a(slab);
                }
                if constexpr (more && s == PAIRS) {
                    store_b(nxt, sl);
                    voff = pixel();
                }
                if constexpr (more && s == PAIRS + 1) {
#pragma unroll
                    for (int i = 0; i < CPT; i++) load_b(sl, i, voff, masked_tag);
                    next_slab();
                }
                // smallest products first: l.h, h.l, m.m, m.h, h.m, h.h
                constexpr int qa = s == 0 ? 2 : s == 2 || s == 3 ? 1 : 0, qb = s == 1 ? 2 : s == 2 || s == 4 ? 1 : 0;
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int j = 0; j < NI; j++) {
                        v16f &c = s < 5 ? low[i][j] : acc[i][j];
                        c = mfma_bf16(a[sl & 1][i][qa], b[sl & 1][j][qb], c);
                    }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        if constexpr (more) __syncthreads();
    };
    auto load_stage = [&](auto masked_tag) {   // all of it at once
        load_a(slab);
#pragma unroll
        for (int sl = 0; sl < SL; sl++) {
            const unsigned voff = pixel();
#pragma unroll
            for (int i = 0; i < CPT; i++) load_b(sl, i, voff, masked_tag);
            next_slab();
        }
    };
    const int stages = (slab_end - slab_begin + SL - 1) / SL;
    auto sums = [&](auto masked_tag) {   // (masked or not: the same order)
        zero_acc(acc);
        zero_acc(low);
        zero_acc(sum);
        rewind();
        load_stage(masked_tag);
        store_a(lds);
#pragma unroll
        for (int sl = 0; sl < SL; sl++) {
#pragma unroll
            for (int e = 0; e < PAIRS; e++) split_b(sl, e);
            store_b(lds, sl);
        }
        if (stages > 1) load_stage(masked_tag);
        __syncthreads();
        int st = 0;
        if constexpr (SL > 1) for (; st + 4 <= stages - 1; st += 4) {
            static_for<0, 4>([&](auto tag) {
                constexpr int cur = decltype(tag)::value % 2;
                stage(lds + cur * STAGE, lds + (1 - cur) * STAGE, StepTag<1>{}, masked_tag);
            });
            move_acc(sum, acc);
        }
        for (; st < stages - 1; ++st) stage(lds + (st & 1) * STAGE, lds + (~st & 1) * STAGE, StepTag<1>{}, masked_tag);
        stage(lds + ((stages - 1) & 1) * STAGE, nullptr, StepTag<0>{}, masked_tag);
        move_acc(sum, acc);
        add_acc(sum, low);
    };
    sums(StepTag<0>{});
    int again = __syncthreads_or(not_finite(sum));
    if (again && p.CinPad != p.Cin) {
        sums(StepTag<1>{});
        again = __syncthreads_or(not_finite(sum));
    }

    // the parts of an infinity hold NaNs: a tile that is not finite is formed again with the fp32 instruction, a stage at a time,
    // for its values that are not finite
    if (again) {
        zero_acc(low);
        rewind();
#pragma unroll 1
        for (int st = 0; st < stages; ++st) {
            load_stage(StepTag<1>{});
            __syncthreads();
            store_a(lds);
            // B here: [half][pixel][8 channels]
#pragma unroll
            for (int sl = 0; sl < SL; sl++)
#pragma unroll
                for (int i = 0; i < CPT; i += 4)
                    *(float4 *)(lds + BOFF + sl * 6 * PB * 4 + (((c0 + i) / 8 * PB + bcol) * 8 + (c0 + i) % 8)) =
                        make_float4(breg[sl][i], breg[sl][i + 1], breg[sl][i + 2], breg[sl][i + 3]);
            __syncthreads();
#pragma unroll 1
            for (int sl = 0; sl < SL; sl++)
#pragma unroll
                for (int i = 0; i < MI; i++) {
                    v4u f[3];
#pragma unroll
                    for (int t = 0; t < 3; t++) f[t] = *(const v4u *)(lds + a_frag + ((sl * 6 + t * 2) * PA + 32 * i) * 4);
#pragma unroll
                    for (int j = 0; j < NI; j++) {
                        const float *const src = lds + BOFF + sl * 6 * PB * 4 + (kh * PB + wn * (BN / T::WN) + 32 * j + l32) * 8;
                        const float4 b0 = *(const float4 *)src, b1 = *(const float4 *)(src + 4);
                        const float b8[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
                        for (int e = 0; e < 8; e++)
                            low[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(packed_value(f, e), b8[e], low[i][j], 0, 0, 0);
                    }
                }
        }
        keep_finite(sum, low);
    }

    float *outp = p.out + (size_t)split * p.out_elems;
#pragma unroll
    for (int j = 0; j < NI; j++) {
        const int col = n0 + wn * (BN / T::WN) + j * 32 + l32;
        if (col >= p.ncols) continue;
        const int n2 = col / OHW, pq2 = col - n2 * OHW;
        const int oh2 = pq2 / p.OW, ow2 = pq2 - oh2 * p.OW;
        float *base = outp + (size_t)n2 * p.Mout * p.out_plane + (size_t)(oh2 * p.out_sy + p.out_oy) * p.out_OW +
                      ow2 * p.out_sx + p.out_ox;
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int m = m0 + wm * (BM / T::WM) + i * 32 + acc_row(v, lane);
                if (m < p.Mout) base[(size_t)m * p.out_plane] = sum[i][j][v];
            }
    }
}

template <class T, int SL, bool kBwd>
__global__ __launch_bounds__(T::THREADS, SL > 1 ? 2 : 4) void conv_gather_k(GatherConv p)
{
    // 1-D grid over (split, tile), tile fastest: the blocks an XCD receives work on neighbouring
    // tiles of the same slice of the reduction, whatever the ratio of tiles to splits
    unsigned L;
    if (!xcd_remap(blockIdx.x, (unsigned)(p.mtiles * p.ntiles) * (unsigned)p.splits, &L)) return;
    conv_gather_body<T, SL, kBwd>(p, L);
}

// Up to nine problems that do not depend on each other in ONE launch (the residue classes of a strided backward-data
// pass - four at stride 2, nine at stride 3: same operands, different sub-filters, interleaved output pixels).  Every workgroup runs conv_gather_body on one
// tile of one problem, so each problem's values are those of a launch of its own; what changes is that the chip is not
// drained and refilled between problems that each fill only part of it.  An XCD takes the same share of every problem
// (its tiles of a problem are neighbours, as in a single launch), longest problem first.
constexpr int kGatherJobs = 9;
struct GatherGroup {
    GatherConv g[kGatherJobs];
    unsigned per[kGatherJobs];   // workgroups of problem j on each XCD: ceil(tiles * splits / 8)
    int n;
};

template <class T, int SL, bool kBwd>
__global__ __launch_bounds__(T::THREADS, 2) void conv_gather_group_k(GatherGroup gg)
{
    const unsigned xcd = blockIdx.x & 7u;
    unsigned i = blockIdx.x >> 3;
    int j = 0;
    while (j < gg.n - 1 && i >= gg.per[j]) {
        i -= gg.per[j];
        j++;
    }
    const unsigned L = xcd * gg.per[j] + i;
    if (i >= gg.per[j] || L >= (unsigned)(gg.g[j].mtiles * gg.g[j].ntiles) * (unsigned)gg.g[j].splits) return;
    conv_gather_body<T, SL, kBwd>(gg.g[j], L);
}

// ------------------------------------------------------------------------------------ patch (3x3, unit stride)
//
// Forward and backward-data of 3x3 unit-stride convolutions.  The gathered operand is not
// re-fetched per filter tap: for a chunk of 16 input channels the block loads the input patch
// under its pixel tile ONCE -- the tile's rows plus a one-pixel halo, zero-filled outside the
// image by the buffer range check -- and the nine taps read it at nine offsets.  LDS holds the patch by channel half and
// position, so that a lane's pixel operands for a whole 16-channel slab are 128-bit LDS reads; the packed filter,
// wp[slab][part][m][16 channels], has the same shape per row, and a lane's filter operands are 128-bit
// loads straight from it.  Lane half kh (= lane / 32) multiplies channels kh*8 .. kh*8+7 of the chunk.

struct PatchConv {
    const float *in;   // gathered operand [N, Cin, IH, IW]
    const float *wp;   // packed filter [chunks][9][3 parts][Mp][16], bf16 (Winograd: 16 positions in the place of 9 taps)
    float *out;        // [N, Mout, OH, OW], or `splits` partial copies of it
    const float *bias; // optional [Mout], added to the finished sums (by the split reduction when there is one)
    int N, Cin, IH, IW, Mout, OH, OW;
    int PT, PL;        // input row / column of patch position (0,0) is (oh0 - PT, -PL)
    int flip;          // 1: tap (tr,ts) reads patch offset (2-tr, 2-ts); 0: (tr, ts)
    int nimg, rows;    // images per pixel tile; output rows of each image in the tile
    int PR, PC, psz;   // patch rows and columns per image; patch positions per tile = nimg*PR*PC
    unsigned magic_img, magic_pc;  // floor(2^32/d)+1 for d = PR*PC, PC (exact for x*d < 2^32)
    unsigned magic_tpi, magic_tcn;            // Winograd: the same for the 2 x 2 tiles of one image in the pixel tile, and of one row
    int Mp;            // rows of one packed filter slab (Mout rounded up to the tile height)
    int ncols, mtiles, ntiles, chunks_total, chunks_per_split, splits;
    size_t out_elems, in_bytes;
};

__device__ inline unsigned fast_div(unsigned x, unsigned magic) { return __umulhi(x, magic); }

// The products run on the bf16 matrix instruction (mfma_core.h).  A patch value is split once, when it is stored, and its parts
// serve all nine taps of all rows, so splitting is a tenth of the loop.  The filter's parts are packed; its fragments go from
// memory straight into the registers the matrix cores read: the packed layout is the fragment layout (a wavefront fetches 32
// rows x 32 bytes, 1 KB contiguous, per part; wavefronts of a tile row fetch the same lines, all but one from the L1), two
// taps ahead.  Only the patch goes through LDS, double buffered: [part][channel half][position][8 channels], a lane's fragment
// of one part is one 128-bit read and neighbouring lanes' reads are neighbours.  The workgroup meets once per 16-channel chunk.
// The h.h products have an accumulator of their own, the five small ones another.
// Batch 128 on 32 x 32 images, the fp32 instruction -> this: 160 -> 16 channels 172 -> 54 us (tiles of 32 rows instead of 64: half
// of that), 16 -> 160 78 -> 52, 32 -> 32 43 -> 19.  48 -> 48 channels: 40 us, of which 25 are matrix time at the rate that a large
// product reaches; the rest is the first patch and the last stores of a workgroup (half as large tiles, two workgroups per CU: 41).
template <class T, int NS, bool kCFull>
__device__ __forceinline__ void conv_patch_body(const PatchConv &p, const unsigned block_id)
{
    constexpr int BM = T::BM, BN = T::BN, THREADS = T::THREADS, MI = T::MI, NI = T::NI;
    constexpr int TAPS = 9, CH = 16;
    constexpr int AHEAD = 2, RING = AHEAD + 1;   // filter fragments on their way
    static_assert(MI == 1 && TAPS % RING == 0, "two taps of one row group ahead; the ring slot of a tap follows from its number");
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int area = p.psz + 1;              // one spare position absorbs the stores of unused slots
    const int pstride = area * 24;           // floats of one patch buffer: 3 parts x 2 halves x 4 words a position
    float *const Bp0 = lds;                  // [2][pstride]

    unsigned L;
    const unsigned tiles = (unsigned)(p.mtiles * p.ntiles);
    if (!xcd_remap(block_id, tiles * (unsigned)p.splits, &L)) return;
    const int split = (int)(L / tiles);
    const unsigned tile = L - (unsigned)split * tiles;
    const int mt = (int)(tile % (unsigned)p.mtiles), nt = (int)(tile / (unsigned)p.mtiles);
    const int m0 = mt * BM, n0 = nt * BN;
    const int cb = split * p.chunks_per_split;
    const int ce = min(cb + p.chunks_per_split, p.chunks_total);

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = w / T::WN, wn = w % T::WN;
    const int kh = lane >> 5, l32 = lane & 31;
    const int OHW = p.OH * p.OW;
    const int chan_stride = p.IH * p.IW;

    const __amdgpu_buffer_rsrc_t rin = make_rsrc(p.in, p.in_bytes);

    // ---- patch slots of this thread: eight channels (one half of the chunk) of one position each
    const int n_first = n0 / OHW, oh0 = (n0 - n_first * OHW) / p.OW;
    unsigned p_voff[NS];   // byte offset of the slot's first channel inside chunk 0, or kOobOffset
    int p_lds[NS];         // float offset inside a patch buffer
    int p_left[NS];        // channels from the slot's first one to the last (only read when the last chunk is ragged)
#pragma unroll
    for (int i = 0; i < NS; i++) {
        const int e = i * THREADS + tid, half = e >= 2 * p.psz ? 2 : e >= p.psz ? 1 : 0;
        const unsigned pos = (unsigned)(half == 2 ? 0 : e - half * p.psz);
        const unsigned img = fast_div(pos, p.magic_img);
        const unsigned rem = pos - img * (unsigned)(p.PR * p.PC);
        const unsigned pr = fast_div(rem, p.magic_pc);
        const unsigned pc = rem - pr * (unsigned)p.PC;
        const int n = n_first + (int)img, ih = oh0 + (int)pr - p.PT, iw = (int)pc - p.PL;
        const int bad = (1 - half) | (p.N - 1 - n) | ih | (p.IH - 1 - ih) | iw | (p.IW - 1 - iw);
        p_voff[i] = bad < 0 ? kOobOffset : (unsigned)(((n * p.Cin + half * 8) * p.IH + ih) * p.IW + iw) * 4u;
        p_lds[i] = half == 2 ? p.psz * 4 : (half * area + (int)pos) * 4;
        p_left[i] = p.Cin - half * 8;
    }
    float preg[NS][8];
    auto patch_load = [&](int i, int c, int chunk) {
        unsigned voff = p_voff[i];
        if (!kCFull) voff = chunk * CH + c < p_left[i] ? voff : kOobOffset;
        preg[i][c] = buffer_load_f32(rin, voff, (unsigned)((chunk * CH + c) * chan_stride) * 4u);
    };
    auto patch_store = [&](int i, float *buf, const unsigned (&q)[3][4]) {
#pragma unroll
        for (int t = 0; t < 3; t++) *(v4u *)(buf + p_lds[i] + t * 2 * area * 4) = v4u{q[t][0], q[t][1], q[t][2], q[t][3]};
    };
    auto patch_split = [&](int i, int e, unsigned (&q)[3][4]) {
        split_pair(preg[i][2 * e] * kSplitUp, preg[i][2 * e + 1] * kSplitUp, q[0][e], q[1][e], q[2][e]);
    };

    // ---- filter fragments: this lane's 8 channels (kh * 8 ..) of row l32 of each 32-row group: [chunk][tap][part][row][16]
    const unsigned part_bytes = (unsigned)p.Mp * CH * 2u, slab_bytes = 3u * part_bytes;
    const unsigned fa_voff = (unsigned)((m0 + wm * (BM / T::WM) + l32) * CH + kh * 8) * 2u;   // m0 + row < Mp always
    v4u fa_ring[RING][MI][3];
    // (the packed filter may be larger than a buffer resource reaches: a resource per chunk)
    auto fa_rsrc = [&](int chunk) { return make_rsrc((const char *)p.wp + (size_t)chunk * TAPS * slab_bytes, (size_t)TAPS * slab_bytes); };
    auto fa_load = [&](int slot, __amdgpu_buffer_rsrc_t rwp, int tap) {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int t = 0; t < 3; t++)
                fa_ring[slot][i][t] = __builtin_bit_cast(v4u, buffer_load_f32x4(rwp, fa_voff + (unsigned)(i * 32 * CH) * 2u,
                                                                               (unsigned)tap * slab_bytes + t * part_bytes));
    };
    int b_pos[NI];  // this lane's pixel and channel half in the area of a part, in positions, tap offset (0,0)
#pragma unroll
    for (int j = 0; j < NI; j++) {
        const int q = wn * (BN / T::WN) + j * 32 + l32;  // pixel inside the tile
        const int img = q / (p.rows * p.OW), r = q / p.OW - img * p.rows, col = q % p.OW;
        b_pos[j] = kh * area + (img * p.PR + r) * p.PC + col;
    }
    auto tap_offset = [&](int t) { return p.flip ? (2 - t / 3) * p.PC + (2 - t % 3) : t / 3 * p.PC + t % 3; };

    v16f acc[MI][NI], low[MI][NI];
    zero_acc(acc);
    zero_acc(low);

    // prologue: the first patch and the first filter slabs
#pragma unroll
    for (int i = 0; i < NS; i++)
#pragma unroll
        for (int c = 0; c < 8; c++) patch_load(i, c, cb);
#pragma unroll
    for (int t = 0; t < AHEAD; t++) fa_load(t, fa_rsrc(cb), t);
#pragma unroll
    for (int i = 0; i < NS; i++) {
        unsigned q[3][4];
#pragma unroll
        for (int e = 0; e < 4; e++) patch_split(i, e, q);
        patch_store(i, Bp0, q);
    }
    __syncthreads();

    v4u fb[NI][3];
    auto fb_load = [&](int part, const float *bp, int t) {
        const int off = part * 2 * area + tap_offset(t);
#pragma unroll
        for (int j = 0; j < NI; j++) fb[j][part] = *(const v4u *)(bp + (off + b_pos[j]) * 4);
    };
    fb_load(2, Bp0, 0);
    fb_load(1, Bp0, 0);

    // The next patch is loaded during taps 0 .. 3 of a chunk and split and stored during taps 5 .. 7; the workgroup meets in
    // tap 8, behind the last reads of the patch being multiplied.
    constexpr int PER = NS * 2;   // loads of a tap
    static_assert(NS <= 3, "a slot per tap 5 .. 7");
    auto chunk_products = [&](int chunk, const float *bp_cur, float *bp_nxt) {
        const __amdgpu_buffer_rsrc_t rw_now = fa_rsrc(chunk), rw_next = fa_rsrc(chunk + 1 < ce ? chunk + 1 : chunk);   // (after the last chunk: loaded, not used)
        unsigned q[3][4];
#pragma unroll
        for (int j = 0; j < NI; j++) asm volatile("" : "+v"(b_pos[j]));   // (or the fifty-four addresses of a chunk are kept in registers)
        static_for<0, TAPS>([&](auto ttag) {
            constexpr int t = decltype(ttag)::value;
            constexpr int slot = t % RING;
            // the pixel part that is used last is read first again: l after its one product, m after its two, h at the tap's start
            static_for<0, 6>([&](auto stag) {
                constexpr int ks = decltype(stag)::value;
                constexpr int qb = ks == 0 ? 2 : ks <= 2 ? 1 : 0;
                constexpr int qa = ks == 0 ? 0 : ks == 1 ? 1 : ks == 2 ? 0 : ks == 3 ? 2 : ks == 4 ? 1 : 0;
                // side work of this step, pinned to it
                if constexpr (ks == 0) {
                    fa_load((t + AHEAD) % RING, t + AHEAD < TAPS ? rw_now : rw_next, (t + AHEAD) % TAPS);
                    fb_load(0, bp_cur, t);
                    if constexpr (t == TAPS - 1) __syncthreads();
                }
                if constexpr (ks == 1) fb_load(2, t == TAPS - 1 ? bp_nxt : bp_cur, (t + 1) % TAPS);
                if constexpr (ks == 3) fb_load(1, t == TAPS - 1 ? bp_nxt : bp_cur, (t + 1) % TAPS);
                if constexpr (t < 4) {
#pragma unroll
                    for (int i = ks * PER / 6; i < (ks + 1) * PER / 6; i++) patch_load((t * PER + i) / 8, (t * PER + i) % 8, chunk + 1);
                }
                if constexpr (t >= 5 && t - 5 < NS) {
                    if constexpr (ks < 4) patch_split(t - 5, ks, q);
                    if constexpr (ks == 4) patch_store(t - 5, bp_nxt, q);
                }
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int j = 0; j < NI; j++) {
                        v16f &c = ks < 5 ? low[i][j] : acc[i][j];
                        c = mfma_bf16(fa_ring[slot][i][qa], fb[j][qb], c);
                    }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
    };
    for (int chunk = cb; chunk < ce; ++chunk) {
        float *const bp_cur = Bp0 + ((chunk - cb) & 1) * pstride;
        float *const bp_nxt = Bp0 + ((chunk - cb + 1) & 1) * pstride;
        chunk_products(chunk, bp_cur, bp_nxt);
    }
    add_acc(acc, low);

    // the parts of an infinity hold NaNs: a tile that is not finite is formed again with the fp32 instruction, one chunk after the
    // other, for its values that are not finite (a word per wavefront: in a backward pair the workgroup's surplus wavefronts have
    // ended)
    __syncthreads();
    {
        const int mine = __any(not_finite(acc));
        if (lane == 0) ((int *)lds)[w] = mine;
        __syncthreads();
        int bad = 0;
#pragma unroll
        for (int i = 0; i < THREADS / 64; i++) bad |= ((const int *)lds)[i];
        if (bad) {
            zero_acc(low);
#pragma unroll 1
            for (int chunk = cb; chunk < ce; chunk++) {
                __syncthreads();
#pragma unroll
                for (int i = 0; i < NS; i++) {   // patch here: [half][position][8 channels]
#pragma unroll
                    for (int c = 0; c < 8; c++) patch_load(i, c, chunk);
                    *(float4 *)(Bp0 + p_lds[i] * 2) = make_float4(preg[i][0], preg[i][1], preg[i][2], preg[i][3]);
                    *(float4 *)(Bp0 + p_lds[i] * 2 + 4) = make_float4(preg[i][4], preg[i][5], preg[i][6], preg[i][7]);
                }
                __syncthreads();
                const __amdgpu_buffer_rsrc_t rw = fa_rsrc(chunk);
#pragma unroll 1
                for (int t = 0; t < TAPS; t++) {
                    fa_load(0, rw, t);
                    const int off = tap_offset(t);
                    float b8[NI][8];
#pragma unroll
                    for (int j = 0; j < NI; j++) {
                        const float4 b0 = *(const float4 *)(Bp0 + (off + b_pos[j]) * 8), b1 = *(const float4 *)(Bp0 + (off + b_pos[j]) * 8 + 4);
                        b8[j][0] = b0.x; b8[j][1] = b0.y; b8[j][2] = b0.z; b8[j][3] = b0.w;
                        b8[j][4] = b1.x; b8[j][5] = b1.y; b8[j][6] = b1.z; b8[j][7] = b1.w;
                    }
#pragma unroll
                    for (int i = 0; i < MI; i++)
#pragma unroll
                        for (int e = 0; e < 8; e++) {
                            const float a = packed_value(fa_ring[0][i], e);
#pragma unroll
                            for (int j = 0; j < NI; j++) low[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b8[j][e], low[i][j], 0, 0, 0);
                        }
                }
            }
            keep_finite(acc, low);
        }
    }

    float *outp = p.out + (size_t)split * p.out_elems;
    const bool add_bias = p.bias != nullptr && p.splits == 1;
#pragma unroll
    for (int j = 0; j < NI; j++) {
        const int col = n0 + wn * (BN / T::WN) + j * 32 + l32;
        if (col >= p.ncols) continue;
        const int n2 = col / OHW, pq2 = col - n2 * OHW;
        float *base = outp + (size_t)n2 * p.Mout * OHW + pq2;
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int m = m0 + wm * (BM / T::WM) + i * 32 + acc_row(v, lane);
                if (m < p.Mout) base[(size_t)m * OHW] = add_bias ? acc[i][j][v] + p.bias[m] : acc[i][j][v];
            }
    }
}

// (two wavefronts per SIMD: as one workgroup of eight, or two of four)
template <class T, int NS, bool kCFull>
__global__ __launch_bounds__(T::THREADS, 2) void conv_patch_k(PatchConv p)
{
    conv_patch_body<T, NS, kCFull>(p, blockIdx.x);
}

// ------------------------------------------------------------------------------------ Winograd F(2x2, 3x3)
//
// The same layers (3x3, unit stride, pad 1, even image sides, whole 16-channel chunks) with 16 instead of 36
// multiplications per 2x2 output pixels (Lavin & Gray): Y = At [ (G g Gt) . (Bt d B) ] A, the element-wise product summed
// over the channels - sixteen independent [rows x channels] . [channels x tiles] products, one per position xi of the
// 4x4 transformed tile.
//
// A workgroup owns 128 rows x 32 tiles (the 128 pixels of the direct kernel's column tile: whole image rows or whole
// images, so the input under them is the same rectangle with the same zero halo) or 64 rows x 64 tiles.
// Per 16-channel chunk: the raw patch goes to LDS position-major (a thread owns one position and stores its channels
// as 128-bit pieces); all 512 threads transform it - thread (i, tile, four channels) forms row i of Bt d B for its tile
// from eight 128-bit reads, splits the sixteen values into their three bf16 parts (mfma_core.h) and writes them to
// V[xi][part][channel half][tile].  The products run on the bf16 matrix instruction: per position and 32 tiles three
// 128-bit reads of V (one step ahead) and three 128-bit loads of the packed filter's parts U[chunk][xi][part][row]
// straight into operand registers (three positions ahead) feed six instructions into the position's own accumulator
// (128 accumulator registers per wavefront, two wavefronts per SIMD).  128 rows: a wavefront takes 32 rows, 32 tiles and
// eight positions; 64 rows: 32 rows, all 64 tiles and the four positions of one row i, so that a filter fragment serves
// two steps (32 tiles and eight positions each, every fragment was loaded by two wavefronts: 160 channels on 32 x 32
// images 259 us instead of 227).  With 32 tiles, patch and V are double-buffered and the next chunk's transform runs under
// this chunk's matrix instructions; every piece of side work is pinned to a matrix step (sched_barrier), or the
// scheduler sinks the prefetches to their first use.
//
// At the end a lane holds M[xi][row][tile] for its positions, complete rows i of the 4x4 grid: it applies A along j in
// registers (z[i][b]) and the wavefronts that share an output meet in LDS: y[a][b] = (At z)[a][b].  With 128 rows one of
// a pair adds the other's share of the four outputs; with 64 rows all four leave their z and finish a quarter of the
// outputs each.  Output, split reductions and bias are those of the direct kernel.
//
// What bounds it (batch 128 with packing, the fp32 instruction -> this): 640 -> 640 channels on 8 x 8 images, batch 512,
// 828 -> 627 us; 160 -> 160 on 32 x 32 318 -> 227; 128 -> 128 on 16 x 16, batch 256, 83 -> 66.  A chunk takes 2.9 us per
// workgroup (fp32: 4.6 .. 5.0), of which 1.8 are matrix time at the rate a product of large matrices reaches.  No single
// cost is left: filter fragments that hit the L1 would take 10 % off (they are 192 KB per chunk, 26 bytes per cycle from
// the L2), no transform 8 %, no patch 6 %, no V reads 3 %; with 64 rows, whose single V is transformed between two
// barriers, no transform 19 %.  64-row tiles in the place of 128-row tiles: 721 us for the first of the layers above.
// floats of the exchange area: 128 rows: four wavefront pairs x 64 values per lane; 64 rows: eight wavefronts x 64 values
constexpr int wino_xchg(int bm) { return (bm == 128 ? 4 : 8) * 64 * 64; }

// WK x TH: WK groups of 32 rows, TH groups of 32 tiles: 4 x 1 (128 rows x 32 tiles = 128 pixels) for layers with whole
// 128-row tiles, 2 x 2 (64 rows x 64 tiles = 256 pixels) for 64-row layers.
template <int NPMAX, int WK, int TH>
__global__ __launch_bounds__(512, 1) void conv_wino_k(PatchConv p)
{
    static_assert(WK * TH == 4 && NPMAX == 16, "eight wavefronts, sixteen channels per chunk");
    constexpr int BM = 32 * WK, BN = 128 * TH, TT = 32 * TH, CH = 16, LDP = 20;
    // V in words: [16 positions][part h, m, l][channel half][tile][8 channels as 4 words] - a lane's fragment of one part is
    // one 128-bit read and neighbouring lanes' reads are neighbours
    constexpr int VP = 8 * TT, VX = 3 * VP, VSZ = 16 * VX;
    // 32 tiles per workgroup: V and the raw patch are double-buffered, the transform of the next chunk runs under this
    // chunk's matrix instructions and the workgroup meets once per chunk.  64 tiles: one V (96 KB), transformed between
    // two barriers.
    constexpr bool DB = TH == 1;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int raw_floats = ((p.psz + 1) * LDP + 3) / 4 * 4;   // one spare position absorbs the stores of idle threads
    float *const raw0 = lds;
    float *const V0 = lds + (DB ? 2 : 1) * raw_floats;          // (x 2)

    unsigned L;
    const unsigned tiles = (unsigned)(p.mtiles * p.ntiles);
    if (!xcd_remap(blockIdx.x, tiles * (unsigned)p.splits, &L)) return;
    const int split = (int)(L / tiles);
    const unsigned tile = L - (unsigned)split * tiles;
    const int mt = (int)(tile % (unsigned)p.mtiles), nt = (int)(tile / (unsigned)p.mtiles);
    const int m0 = mt * BM, n0 = nt * BN;
    const int cb = split * p.chunks_per_split;
    const int ce = min(cb + p.chunks_per_split, p.chunks_total);
    const int nch = ce - cb;
    // The bf16 instruction rounds down below its guard bits; partial sums of alternating sign take that out of their total.
    const float up = split & 1 ? -kSplitUp : kSplitUp, down = split & 1 ? -kSplitDown : kSplitDown;

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wavefront-uniform, and known to be: it enters scalar load offsets
    // a wavefront multiplies its rows with XP positions from xb on, the tiles 32 at a time
    constexpr int XP = 8 / TH;
    const int wi = TH == 1 ? w & 1 : w >> 1, wk = TH == 1 ? w >> 1 : w & 1, xb = wi * XP;
    const int kh = lane >> 5, l32 = lane & 31;
    const int OHW = p.OH * p.OW;
    const int chan_stride = p.IH * p.IW;
    const __amdgpu_buffer_rsrc_t rin = make_rsrc(p.in, p.in_bytes);

    // ---- the patch: a thread owns ONE position and loads `nslots` of the chunk's channels of it, so its sixteen
    // addresses are one per-lane offset plus a wavefront-uniform channel offset (sixteen separate offsets and LDS
    // addresses would hold 32 registers).  Up to 256 positions: wavefronts 4..7 take channels 8..15 of the same positions.
    const int n_first = n0 / OHW, oh0 = (n0 - n_first * OHW) / p.OW;
    const int nslots = p.psz <= 256 ? 8 : 16;
    const int pos = p.psz <= 256 ? (tid & 255) : tid;
    const int cbase = p.psz <= 256 ? (w >> 2) * 8 : 0;
    unsigned p_voff;
    int p_lds;
    {
        const unsigned ps = (unsigned)min(pos, p.psz - 1);
        const unsigned img = fast_div(ps, p.magic_img);
        const unsigned rem = ps - img * (unsigned)(p.PR * p.PC);
        const unsigned pr = fast_div(rem, p.magic_pc);
        const unsigned pc = rem - pr * (unsigned)p.PC;
        const int n = n_first + (int)img, ih = oh0 + (int)pr - p.PT, iw = (int)pc - p.PL;
        const int bad = (p.psz - 1 - pos) | (p.N - 1 - n) | ih | (p.IH - 1 - ih) | iw | (p.IW - 1 - iw);
        p_voff = bad < 0 ? kOobOffset : (unsigned)((n * p.Cin * p.IH + ih) * p.IW + iw) * 4u;
        p_lds = (min(pos, p.psz) * LDP + cbase) * 4;
    }
    float preg[NPMAX];
    auto patch_load = [&](int i, int chunk) {
        if (i < nslots) preg[i] = buffer_load_f32(rin, p_voff, (unsigned)((chunk * CH + cbase + i) * chan_stride) * 4u);
    };
    auto patch_store = [&](int g, float *rawb) {   // channels 4 g .. 4 g + 3 of the position: one 128-bit store
        if (4 * g < nslots)
            *(float4 *)((char *)rawb + p_lds + g * 16) =
                make_float4(preg[4 * g] * up, preg[4 * g + 1] * up, preg[4 * g + 2] * up, preg[4 * g + 3] * up);
    };

    // ---- the transform items of this thread (TH of them): row ti of Bt d B for tile tau, channels 4 cq .. 4 cq + 3
    const int tcn = p.OW >> 1, tpi = (p.rows >> 1) * tcn;          // tiles per row of tiles, per image of the pixel tile
    auto tile_at = [&](int tau, int &img, int &r2, int &c2) {
        img = (int)fast_div((unsigned)tau, p.magic_tpi);
        const int tl = tau - img * tpi;
        r2 = (int)fast_div((unsigned)tl, p.magic_tcn);
        c2 = tl - r2 * tcn;
    };
    // Bt = [1 0 -1 0; 0 1 1 0; 0 -1 1 0; 0 1 0 -1]: row ti is d[ra] + sg * d[rb]
    int t_a[TH], t_b[TH], t_out[TH];
    float sg[TH];
#pragma unroll
    for (int u = 0; u < TH; u++) {
        // (two of the four channel quads on neighbouring lanes, the other two a multiple of 64 lanes on: neither the reads of
        // the patch nor the 64-bit writes of the parts meet in a bank)
        const int item = u * 512 + tid, ti = item / (TT * 4), tau_t = (item >> 1) % TT, cqh = (item / (TT * 2)) & 1;
        const int cq = 2 * cqh + (item & 1);
        int img, r2, c2;
        tile_at(tau_t, img, r2, c2);
        const int t_in = ((img * p.PR + 2 * r2) * p.PC + 2 * c2) * LDP + cq * 4;
        const int ra = ti == 0 ? 0 : ti == 2 ? 2 : 1, rb = ti == 0 ? 2 : ti == 1 ? 2 : ti == 2 ? 1 : 3;
        t_a[u] = t_in + ra * p.PC * LDP;
        t_b[u] = t_in + rb * p.PC * LDP;
        t_out[u] = ti * 4 * VX + cqh * (4 * TT) + tau_t * 4 + (item & 1) * 2;
        sg[u] = ti == 1 ? 1.0f : -1.0f;
    }
    float4 tt[TH][4];
    auto transform_read = [&](int b, const float *rawb) {       // column b of the thread's row of Bt d
#pragma unroll
        for (int u = 0; u < TH; u++) {
            const float4 da = *(const float4 *)(rawb + t_a[u] + b * LDP), db = *(const float4 *)(rawb + t_b[u] + b * LDP);
            // sg is +-1: the fused form rounds once, like the sum or difference it stands for
            tt[u][b] = make_float4(__builtin_fmaf(sg[u], db.x, da.x), __builtin_fmaf(sg[u], db.y, da.y),
                                   __builtin_fmaf(sg[u], db.z, da.z), __builtin_fmaf(sg[u], db.w, da.w));
        }
    };
    auto transform_write = [&](float *Vb, int j) {               // ... times B, position j of the row, split into its parts
#pragma unroll
        for (int u = 0; u < TH; u++) {
            const float4 x = tt[u][j == 0 ? 0 : j == 2 ? 2 : 1], y = tt[u][j < 2 ? 2 : j == 2 ? 1 : 3];
            const float s = j == 1 ? 1.0f : -1.0f;
            uint2 h, m, l;
            split_pair(__builtin_fmaf(s, y.x, x.x), __builtin_fmaf(s, y.y, x.y), h.x, m.x, l.x);
            split_pair(__builtin_fmaf(s, y.z, x.z), __builtin_fmaf(s, y.w, x.w), h.y, m.y, l.y);
            float *const o = Vb + t_out[u] + j * VX;
            *(uint2 *)o = h;
            *(uint2 *)(o + VP) = m;
            *(uint2 *)(o + 2 * VP) = l;
        }
    };

    // ---- transformed-filter fragments: this lane's 8 channels (kh * 8 ..) of row m0 + 32 wk + l32
    // [chunk][position][part][row][16 channels]
    const unsigned part_bytes = (unsigned)p.Mp * CH * 2u, slab_bytes = 3u * part_bytes;
    const unsigned fa_voff = (unsigned)((m0 + wk * 32 + l32) * CH + kh * 8) * 2u;
    v4u fa_ring[4][3];
    // (the packed filter may be larger than a buffer resource reaches: a resource per chunk)
    auto fa_rsrc = [&](int chunk) { return make_rsrc((const char *)p.wp + (size_t)chunk * 16 * slab_bytes, (size_t)16 * slab_bytes); };
    auto fa_load = [&](auto slot_tag, __amdgpu_buffer_rsrc_t rwp, int xi) {
        constexpr int slot = decltype(slot_tag)::value;
#pragma unroll
        for (int q = 0; q < 3; q++)
            fa_ring[slot][q] = __builtin_bit_cast(v4u, buffer_load_f32x4(rwp, fa_voff, (unsigned)xi * slab_bytes + q * part_bytes));
    };
    const int b_frag = xb * VX + kh * (4 * TT) + l32 * 4;   // position xb, this lane's tile and channels
    v4u fb_next[3];
    auto fb_load = [&](const float *Vb, int x) {   // step x: position x / TH, tiles 32 (x % TH) ..
#pragma unroll
        for (int q = 0; q < 3; q++) fb_next[q] = *(const v4u *)(Vb + b_frag + x / TH * VX + q * VP + x % TH * 128);
    };

    v16f acc[8];
#pragma unroll
    for (int x = 0; x < 8; x++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[x][v] = 0.0f;

    // prologue: the first patch (and, double-buffered, the second: both in flight together), the first transform, the
    // first three filter fragments
#pragma unroll
    for (int i = 0; i < NPMAX; i++) patch_load(i, cb);
    if constexpr (DB) {
        float second[NPMAX];
#pragma unroll
        for (int i = 0; i < NPMAX; i++)
            // (no branch: what is done to the values would move into it, and each load be waited for there)
            second[i] = buffer_load_f32(rin, i < nslots && nch > 1 ? p_voff : kOobOffset,
                                        (unsigned)(((nch > 1 ? cb + 1 : cb) * CH + cbase + (i < nslots ? i : 0)) * chan_stride) * 4u);
        fa_load(StepTag<0>{}, fa_rsrc(cb), xb);
        fa_load(StepTag<1>{}, fa_rsrc(cb), xb + 1);
        fa_load(StepTag<2>{}, fa_rsrc(cb), xb + 2);
#pragma unroll
        for (int g = 0; g < NPMAX / 4; g++) patch_store(g, raw0);
#pragma unroll
        for (int g = 0; g < NPMAX / 4; g++)
            if (4 * g < nslots)
                *(float4 *)((char *)(raw0 + raw_floats) + p_lds + g * 16) =
                    make_float4(second[4 * g] * up, second[4 * g + 1] * up, second[4 * g + 2] * up,
                                second[4 * g + 3] * up);
    } else {
        fa_load(StepTag<0>{}, fa_rsrc(cb), xb);
        fa_load(StepTag<1>{}, fa_rsrc(cb), xb + 1);
        fa_load(StepTag<2>{}, fa_rsrc(cb), xb + 2);
#pragma unroll
        for (int g = 0; g < NPMAX / 4; g++) patch_store(g, raw0);
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 4; b++) transform_read(b, raw0);
#pragma unroll
    for (int b = 0; b < 4; b++) transform_write(V0, b);
    __syncthreads();

    constexpr int PER = NPMAX / 4;
    fb_load(V0, 0);
    for (int it = 0; it < nch; ++it) {
        const int chunk = cb + it;
        // double-buffered: V of this chunk, raw patch and V of the next one, raw patch of the one after (into the buffer
        // this chunk's patch left when it was transformed)
        const float *const Vc = V0 + (DB ? (it & 1) * VSZ : 0);
        float *const Vn = V0 + (DB ? ((it + 1) & 1) * VSZ : 0);
        const float *const rawn = raw0 + (DB ? ((it + 1) & 1) * raw_floats : 0);
        float *const raww = raw0 + (DB ? (it & 1) * raw_floats : 0);
        const int ahead = DB ? 2 : 1;
        const bool more = it + 1 < nch, fetch = it + ahead < nch;
        const __amdgpu_buffer_rsrc_t rw_now = fa_rsrc(chunk), rw_next = fa_rsrc(more ? chunk + 1 : chunk);   // (after the last chunk: loaded, not used)
        static_for<0, 8>([&](auto xtag) {
            constexpr int xl = decltype(xtag)::value;
            const v4u fb[3] = {fb_next[0], fb_next[1], fb_next[2]};
            constexpr int xp = xl / TH;
            const v4u fa[3] = {fa_ring[xp % 4][0], fa_ring[xp % 4][1], fa_ring[xp % 4][2]};
            static_for<0, 6>([&](auto stag) {
                constexpr int ks = decltype(stag)::value;
                // side work of this step, pinned to it: left to itself the scheduler sinks every load to its first use
                if constexpr (ks == 0 && xl % TH == 0) {
                    // the filter fragments three positions ahead (into the slot of the position before this one)
                    fa_load(StepTag<(xp + 3) % 4>{}, xp + 3 < XP ? rw_now : rw_next, xb + (xp + 3) % XP);
                }
                if constexpr (ks == 1 && xl < 7) fb_load(Vc, xl + 1);   // this lane's tile at the next position
                // the patch `ahead` chunks on: loads during positions 0..3, LDS stores during 4..7
                if constexpr (xl < 4 && ks >= 2 && ks < 2 + PER) {
                    if (fetch) patch_load(xl * PER + ks - 2, chunk + ahead);
                }
                if constexpr (xl >= 4 && ks == 2) {
                    if (fetch) patch_store(xl - 4, raww);
                }
                if constexpr (DB && ks == 4) {       // the next chunk's transform: a column per position, then a product each
                    if (more) {
                        if constexpr (xl < 4) transform_read(xl, rawn);
                        if constexpr (xl >= 4) transform_write(Vn, xl - 4);
                    }
                }
                // smallest products first: l.h, h.l, m.m, m.h, h.m, h.h
                constexpr int qa = ks == 0 ? 2 : ks == 2 || ks == 3 ? 1 : 0, qb = ks == 1 ? 2 : ks == 2 || ks == 4 ? 1 : 0;
                acc[xl] = mfma_bf16(fa[qa], fb[qb], acc[xl]);
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        __syncthreads();              // every wavefront is done with V of this chunk; the next patch is in place
        if constexpr (!DB) {
            if (more) {
#pragma unroll
                for (int b = 0; b < 4; b++) transform_read(b, raw0);
#pragma unroll
                for (int b = 0; b < 4; b++) transform_write(V0, b);
            }
            __syncthreads();
        }
        fb_load(Vn, 0);
    }

    // ---- inverse transform.  This wavefront's rows of the 4x4 grid are i = 2 wi, 2 wi + 1; acc[4 il + j] = M[i][j].
    // At = [1 1 1 0; 0 1 -1 -1]:  z[i][0] = m0 + m1 + m2, z[i][1] = m1 - m2 - m3, then the same over i.
    float *const xchg = lds;          // [wavefront pair][accumulator row][lane][4]: the main loop's LDS is free now
    float *outp = p.out + (size_t)split * p.out_elems;
    const bool add_bias = p.bias != nullptr && p.splits == 1;
    // the four outputs of accumulator row v of tiles 32 t ..; y: index 2 a + b
    float scale = down, probe = 0.0f;   // probe: NaN once anything is not finite, x * 0 is 0 for finite x only
    auto store = [&](int t, int v, const float (&sum)[4]) {
        float y[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            probe = __builtin_fmaf(sum[q], 0.0f, probe);
            y[q] = sum[q] * scale;
        }
        int img, r2, c2;
        tile_at(t * 32 + l32, img, r2, c2);
        const int n = n_first + img, m = m0 + wk * 32 + acc_row(v, lane);
        if (n >= p.N || m >= p.Mout) return;
        if (add_bias) {
            const float bias = p.bias[m];
#pragma unroll
            for (int q = 0; q < 4; q++) y[q] += bias;
        }
        float *o = outp + ((size_t)n * p.Mout + m) * OHW + (oh0 + 2 * r2) * p.OW + 2 * c2;
        *(float2 *)o = make_float2(y[0], y[1]);
        *(float2 *)(o + p.OW) = make_float2(y[2], y[3]);
    };
    for (int pass = 0;; pass++) {
        if constexpr (TH == 1) {
            float part[16][4];            // per accumulator row v: this wavefront's share of y[a][b], index 2 a + b
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const float za0 = (acc[0][v] + acc[1][v]) + acc[2][v], za1 = (acc[1][v] - acc[2][v]) - acc[3][v];
                const float zb0 = (acc[4][v] + acc[5][v]) + acc[6][v], zb1 = (acc[5][v] - acc[6][v]) - acc[7][v];
                if (wi == 0) {            // rows 0, 1: y[0] += z0 + z1, y[1] += z1
                    part[v][0] = za0 + zb0; part[v][1] = za1 + zb1; part[v][2] = zb0; part[v][3] = zb1;
                } else {                  // rows 2, 3: y[0] += z2, y[1] += -z2 - z3
                    part[v][0] = za0; part[v][1] = za1; part[v][2] = -za0 - zb0; part[v][3] = -za1 - zb1;
                }
            }
            if (wi == 1) {   // a lane's four shares of one accumulator row are one 128-bit store
#pragma unroll
                for (int v = 0; v < 16; v++)
                    *(float4 *)(xchg + ((wk * 16 + v) * 64 + lane) * 4) = make_float4(part[v][0], part[v][1], part[v][2], part[v][3]);
            }
            __syncthreads();
            if (wi == 0) {
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const float4 other = *(const float4 *)(xchg + ((wk * 16 + v) * 64 + lane) * 4);
                    const float y[4] = {part[v][0] + other.x, part[v][1] + other.y, part[v][2] + other.z, part[v][3] + other.w};
                    store(0, v, y);
                }
            }
        } else {
            // a wavefront holds one row i of the grid: all four put their z in LDS, each finishes eight accumulator rows
#pragma unroll
            for (int t = 0; t < TH; t++)
#pragma unroll
                for (int v = 0; v < 16; v++)
                    *(float2 *)(xchg + (((wk * 4 + wi) * 32 + t * 16 + v) * 64 + lane) * 2) =
                        make_float2((acc[t][v] + acc[2 + t][v]) + acc[4 + t][v], (acc[2 + t][v] - acc[4 + t][v]) - acc[6 + t][v]);
            __syncthreads();
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int tv = wi * 8 + e;
                float2 z[4];
#pragma unroll
                for (int i = 0; i < 4; i++) z[i] = *(const float2 *)(xchg + (((wk * 4 + i) * 32 + tv) * 64 + lane) * 2);
                const float y[4] = {(z[0].x + z[1].x) + z[2].x, (z[0].y + z[1].y) + z[2].y, z[1].x + (-z[2].x - z[3].x), z[1].y + (-z[2].y - z[3].y)};
                store(tv >> 4, tv & 15, y);
            }
        }
        if (pass == 1) break;
        // the parts of an infinity hold NaNs: a tile that is not finite is formed again with the fp32 instruction, one chunk and
        // one position after the other (each wavefront's word lies behind the exchange area)
        int *const bad = (int *)(lds + wino_xchg(BM));
        const int mine = __any(probe != 0.0f);
        if (lane == 0) bad[w] = mine;
        __syncthreads();
        const int4 bad0 = *(const int4 *)bad, bad1 = *(const int4 *)(bad + 4);
        if (((bad0.x | bad0.y | bad0.z | bad0.w) | (bad1.x | bad1.y | bad1.z | bad1.w)) == 0) break;
        constexpr int LDV = 20;   // V here: [16 positions][tile][16 channels (+ 4 pad)]
#pragma unroll
        for (int x = 0; x < 8; x++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[x][v] = 0.0f;
#pragma unroll 1
        for (int chunk = cb; chunk < ce; chunk++) {
#pragma unroll
            for (int i = 0; i < NPMAX; i++) patch_load(i, chunk);
#pragma unroll
            for (int g = 0; g < NPMAX / 4; g++)
                if (4 * g < nslots)
                    *(float4 *)((char *)raw0 + p_lds + g * 16) = make_float4(preg[4 * g], preg[4 * g + 1], preg[4 * g + 2], preg[4 * g + 3]);
            __syncthreads();
#pragma unroll
            for (int b = 0; b < 4; b++) transform_read(b, raw0);
#pragma unroll
            for (int u = 0; u < TH; u++) {
                const int item = u * 512 + tid, ti = item / (TT * 4), tau_t = (item >> 1) % TT, cq = 2 * ((item / (TT * 2)) & 1) + (item & 1);
                float *const o = V0 + (ti * 4 * TT + tau_t) * LDV + cq * 4;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float4 x = tt[u][j == 0 ? 0 : j == 2 ? 2 : 1], y = tt[u][j < 2 ? 2 : j == 2 ? 1 : 3];
                    const float s = j == 1 ? 1.0f : -1.0f;
                    *(float4 *)(o + j * TT * LDV) = make_float4(__builtin_fmaf(s, y.x, x.x), __builtin_fmaf(s, y.y, x.y),
                                                               __builtin_fmaf(s, y.z, x.z), __builtin_fmaf(s, y.w, x.w));
                }
            }
            __syncthreads();
            const __amdgpu_buffer_rsrc_t rw = fa_rsrc(chunk);
            static_for<0, 8>([&](auto xtag) {
                constexpr int xl = decltype(xtag)::value;
                fa_load(StepTag<0>{}, rw, xb + xl / TH);
                const float *const src = V0 + ((xb + xl / TH) * TT + xl % TH * 32 + l32) * LDV + kh * 8;
                const float4 b0 = *(const float4 *)src, b1 = *(const float4 *)(src + 4);
                const float b8[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float a = packed_value(fa_ring[0], e);
                    acc[xl] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b8[e], acc[xl], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        }
        __syncthreads();
        scale = 1.0f;
    }
}

// The transformed filter of the Winograd kernel, multiplied by kSplitUp and split into its bf16 parts q = h, m, l:
// U[(((chunk*16 + xi)*3 + q)*Mp + m)*16 + j] = (G g Gt)[xi] for row m and channel chunk*16 + j, where g is the filter as the kernel applies it to the patch: g[r][s] multiplies patch offset
// (r, s), i.e. the stored taps read backwards when the operation is a true convolution (`flip`).  Staged like
// pack_tile (16 rows of one chunk); G = [1 0 0; .5 .5 .5; .5 -.5 .5; 0 0 1].
template <bool kBwd>
__device__ __forceinline__ void wino_pack_tile(int M, int Cred, int Mp, size_t sm, size_t sc, int flip, const float *w, float *wp,
                                               int chunk, int m0, float *stage)
{
    constexpr int PITCH = kBwd ? 148 : 145;
    float v[9];
#pragma unroll
    for (int i = 0; i < 9; i++) {
        const int f = i * 256 + threadIdx.x;
        const int run = f / 144, r = f - run * 144;
        bool ok;
        size_t src;
        if (!kBwd) {
            ok = m0 + run < M && chunk * 16 + r / 9 < Cred;
            src = (size_t)(m0 + run) * sm + (size_t)chunk * 16 * sc + r;
        } else {
            ok = chunk * 16 + run < Cred && m0 + r / 9 < M;
            src = (size_t)(chunk * 16 + run) * sc + (size_t)m0 * sm + r;
        }
        v[i] = ok ? w[src] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < 9; i++) {
        const int f = i * 256 + threadIdx.x;
        stage[(f / 144) * PITCH + f % 144] = v[i];
    }
    __syncthreads();
    // one (row, channel) pair per thread: 16 x 16 pairs, sixteen values each
    {
        const int j = threadIdx.x & 15, ml = threadIdx.x >> 4;
        const float *s = !kBwd ? stage + ml * PITCH + j * 9 : stage + j * PITCH + ml * 9;
        float g[3][3];
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) g[r][c] = flip ? s[(2 - r) * 3 + (2 - c)] : s[r * 3 + c];
        float h[4][3];   // G g
#pragma unroll
        for (int c = 0; c < 3; c++) {
            h[0][c] = g[0][c];
            h[1][c] = ((g[0][c] + g[1][c]) + g[2][c]) * 0.5f;
            h[2][c] = ((g[0][c] - g[1][c]) + g[2][c]) * 0.5f;
            h[3][c] = g[2][c];
        }
        // neighbouring channels share a word: the even channel's thread writes the positions of columns 0 and 2, the odd
        // one's those of columns 1 and 3, each with its neighbour's values
        const bool odd = j & 1;
        const size_t part = (size_t)Mp * 8;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float u[4] = {h[r][0], ((h[r][0] + h[r][1]) + h[r][2]) * 0.5f, ((h[r][0] - h[r][1]) + h[r][2]) * 0.5f, h[r][2]};
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                const float other = __shfl_xor(odd ? u[e] : u[e + 1], 1);
                unsigned ph, pm, pl;
                const float a = odd ? other : u[e], b = odd ? u[e + 1] : other;
                split_packed(a, b, ph, pm, pl);
                unsigned *dst = (unsigned *)wp + ((((size_t)chunk * 16 + r * 4 + e + odd) * 3) * Mp + m0 + ml) * 8 + (j >> 1);
                dst[0] = ph;
                dst[part] = pm;
                dst[2 * part] = pl;
            }
        }
    }
}

// Packed filter of the patch kernel: wp[(((chunk*9 + tap)*3 + part)*Mp + m)*16 + j], the bf16 parts of w[m*sm + (chunk*16+j)*sc + tap]
// times kSplitUp (zero where m >= M or the channel is past the end).  Forward: m = output channel k (sm = C*9,
// sc = 9); backward-data: m = input channel c (sm = 9, sc = C*9), reduction over k.
// A block transposes 16 rows of one chunk through LDS.  Its source is 16 contiguous runs of 144
// floats (forward: one per row, its 16 channels x 9 taps; backward: one per reduction channel,
// its 16 rows x 9 taps), copied to LDS as they lie -- all nine loads of a thread in flight at
// once; the scattered side of the transposition is the LDS read, whose strides spread the lanes
// over the banks.
template <bool kBwd>
__device__ __forceinline__ void pack_tile(int M, int Cred, int Mp, size_t sm, size_t sc, const float *w, float *wp,
                                          int chunk, int m0, float *stage)
{
    constexpr int PITCH = kBwd ? 148 : 145;  // floats between runs in LDS
    float v[9];
#pragma unroll
    for (int i = 0; i < 9; i++) {
        const int f = i * 256 + threadIdx.x;
        const int run = f / 144, r = f - run * 144;
        bool ok;
        size_t src;
        if (!kBwd) {  // run = row m0 + run, r = (channel, tap)
            ok = m0 + run < M && chunk * 16 + r / 9 < Cred;
            src = (size_t)(m0 + run) * sm + (size_t)chunk * 16 * sc + r;
        } else {      // run = reduction channel chunk*16 + run, r = (row, tap)
            ok = chunk * 16 + run < Cred && m0 + r / 9 < M;
            src = (size_t)(chunk * 16 + run) * sc + (size_t)m0 * sm + r;
        }
        v[i] = ok ? w[src] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < 9; i++) {
        const int f = i * 256 + threadIdx.x;
        stage[(f / 144) * PITCH + f % 144] = v[i];
    }
    __syncthreads();
    // four channels of one row and tap per thread and pass
    for (int o = threadIdx.x; o < 9 * 16 * 4; o += 256) {
        const int j4 = o & 3, ml = (o >> 2) & 15, tap = o >> 6;
        float4 q;
        if (!kBwd) {
            const float *s = stage + ml * PITCH + (j4 * 4) * 9 + tap;
            q = make_float4(s[0], s[9], s[18], s[27]);
        } else {
            const float *s = stage + (j4 * 4) * PITCH + ml * 9 + tap;
            q = make_float4(s[0], s[PITCH], s[2 * PITCH], s[3 * PITCH]);
        }
        uint2 part[3];
        split_packed(q.x, q.y, part[0].x, part[1].x, part[2].x);
        split_packed(q.z, q.w, part[0].y, part[1].y, part[2].y);
        uint2 *dst = (uint2 *)wp + ((((size_t)chunk * 9 + tap) * 3) * Mp + m0 + ml) * 4 + j4;
#pragma unroll
        for (int t = 0; t < 3; t++) dst[(size_t)t * Mp * 4] = part[t];
    }
}

template <bool kBwd>
__global__ __launch_bounds__(256) void pack_patch_k(int M, int Cred, int Mp, size_t sm, size_t sc, int wino, int flip,
                                                     const float *w, float *wp)
{
    __shared__ float stage[16 * 148];
    if (wino) wino_pack_tile<kBwd>(M, Cred, Mp, sm, sc, flip, w, wp, blockIdx.y, blockIdx.x * 16, stage);
    else pack_tile<kBwd>(M, Cred, Mp, sm, sc, w, wp, blockIdx.y, blockIdx.x * 16, stage);
}

// The filters of many layers in one launch (a training step packs each filter twice, once per
// direction, and most of those launches are far too small to fill the chip on their own).
constexpr int kPackJobs = 32;
struct PackJob {
    const float *w;
    float *wp;
    int M, Cred, Mp, bwd;
    int wino, flip;                  // wino: the Winograd kernel's transformed filter (16 positions per chunk instead of 9 taps)
    unsigned sm, sc;
    unsigned first_block, mblocks;   // blocks [first_block, next job's first_block): (chunk, row block) pairs
};
struct PackBatch {
    PackJob job[kPackJobs];
    int njobs;
};

__global__ __launch_bounds__(256) void pack_batch_k(PackBatch b)
{
    __shared__ float stage[16 * 148];
    int j = 0;
    while (j + 1 < b.njobs && blockIdx.x >= b.job[j + 1].first_block) j++;
    const PackJob &q = b.job[j];
    const unsigned local = blockIdx.x - q.first_block;
    const int chunk = (int)(local / q.mblocks), m0 = (int)(local % q.mblocks) * 16;
    if (q.wino) {
        if (q.bwd) wino_pack_tile<true>(q.M, q.Cred, q.Mp, q.sm, q.sc, q.flip, q.w, q.wp, chunk, m0, stage);
        else wino_pack_tile<false>(q.M, q.Cred, q.Mp, q.sm, q.sc, q.flip, q.w, q.wp, chunk, m0, stage);
    } else if (q.bwd) pack_tile<true>(q.M, q.Cred, q.Mp, q.sm, q.sc, q.w, q.wp, chunk, m0, stage);
    else pack_tile<false>(q.M, q.Cred, q.Mp, q.sm, q.sc, q.w, q.wp, chunk, m0, stage);
}

// ------------------------------------------------------------------------------------ backward-filter

struct FilterGrad {
    const float *dy;  // [N, K, P, Q]
    const float *x;   // [N, C, H, W]
    float *out;       // `splits` partial copies of [K][taps * Cp] (tap-major columns)
    int N, C, H, W, K, P, Q, R, S;
    int padH, padW, strideH, strideW;
    int Cp;           // C rounded up to 16: a 16-column group never straddles two taps
    int ncols;        // taps * Cp
    int npix;         // N*P*Q
    int mtiles, ntiles, slabs_total, slabs_per_split, splits;
    size_t out_elems, dy_bytes, x_bytes;
};

// Products, LDS and stages as in conv_gather_body; here both operands are split when they are stored.  A lane loads one pixel of a
// stage's 32, lane and lane + 32 neighbouring ones: v_permlane32_swap gives either lane both pixels of one of two rows, and a
// pair of pixels is a word of each part.  (Split in every wavefront that read a
// value: 64 -> 64 channels of 3 x 3 on 64 images of 33 x 31 72 us, now 57; 5 x 5 at stride 2, 48 -> 100 on 50 images of 45 x 39, 80 -> 78; the
// strided layers of Wide-ResNet-28-10 410 + 355 + 76 -> 357 + 353 + 68.  What bounds those now are the gathered loads of x.)
// TPT = number of column groups of a tile that may belong to different taps (BN / gcd(BN, Cp)):
// the input displacement and the bounds test are per group, not per element.
template <class T, int TPT>
__global__ __launch_bounds__(T::THREADS, 2) void conv_wgrad_k(FilterGrad p)
{
    constexpr int BM = T::BM, BN = T::BN, MI = T::MI, NI = T::NI, SL = 2;
    static_assert(T::THREADS == 512, "lanes run along 32 pixels, 16 rows per pass");
    constexpr int NA = BM / 16, NB = BN / 16;  // scalar loads per thread
    constexpr int GSZ = NB / TPT;              // loads per tap group
    static_assert(GSZ * TPT == NB && NA % 2 == 0 && NB % 2 == 0, "TPT must divide the loads per thread");
    constexpr int PA = BM + 4, PB = BN + 4, BOFF = SL * 6 * PA * 4, STAGE = BOFF + SL * 6 * PB * 4;   // as GatherLds
    extern __shared__ __attribute__((aligned(16))) float lds[];

    unsigned L;
    const unsigned tiles = (unsigned)(p.mtiles * p.ntiles);
    if (!xcd_remap(blockIdx.x, tiles * (unsigned)p.splits, &L)) return;
    const int split = (int)(L / tiles);
    const unsigned tile = L - (unsigned)split * tiles;
    const int mt = (int)(tile % (unsigned)p.mtiles), nt = (int)(tile / (unsigned)p.mtiles);
    const int m0 = mt * BM, n0 = nt * BN;
    const int slab_begin = split * p.slabs_per_split;
    const int slab_end = min(slab_begin + p.slabs_per_split, p.slabs_total);

    const int tid = threadIdx.x, lane = tid & 63, kh = lane >> 5, l32 = lane & 31;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = w / T::WN, wn = w % T::WN;
    // this lane's pixel of the stage, and its first tile row / column (others are multiples of 16 further on)
    const int px = 2 * (lane & 15) + kh, r0 = 2 * w + ((lane >> 4) & 1);
    const int PQ = p.P * p.Q, HW = p.H * p.W;

    const __amdgpu_buffer_rsrc_t rdy = make_rsrc(p.dy, p.dy_bytes);
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, p.x_bytes);
    // (rows past K and columns past C are read as they lie, or as zeros past the tensor: their sums are not used)

    // wave-uniform description of each tap group of this tile
    int g_dr[TPT], g_ds[TPT], g_disp[TPT], g_c0[TPT];
#pragma unroll
    for (int g = 0; g < TPT; g++) {
        const int nn = n0 + 16 * GSZ * g;
        if (nn < p.ncols) {
            const int tap = nn / p.Cp;
            const int tr = tap / p.S, ts = tap - tr * p.S;
            g_c0[g] = nn - tap * p.Cp;
            g_dr[g] = p.R - 1 - tr - p.padH;
            g_ds[g] = p.S - 1 - ts - p.padW;
        } else {
            g_c0[g] = 0;
            g_dr[g] = -(1 << 28);  // fails every bounds test
            g_ds[g] = 0;
        }
        g_disp[g] = g_dr[g] * p.W + g_ds[g];
    }

    float areg[NA], breg[NB];
    int slab;                       // first slab of the stage that is loaded next
    int ih0, iw0, x_pix, oob_pix;   // of that stage's pixel
    auto load_a = [&]() {           // and where the pixel lies
        const int kk = slab * BK + px;
        oob_pix = min(p.npix, slab_end * BK) - 1 - kk;  // negative past the last pixel
        const int n = kk / PQ, pq = kk - n * PQ;
        const int ph = pq / p.Q, qw = pq - ph * p.Q;
        const unsigned voff = oob_pix < 0 ? kOobOffset : (unsigned)((n * p.K + m0 + r0) * PQ + pq) * 4u;
#pragma unroll
        for (int i = 0; i < NA; i++) areg[i] = buffer_load_f32(rdy, voff, (unsigned)(16 * i * PQ) * 4u);
        ih0 = ph * p.strideH;
        iw0 = qw * p.strideW;
        x_pix = (n * p.C + r0) * HW + ih0 * p.W + iw0;  // element offset of (n, channel r0, ih0, iw0)
        slab += SL;
    };
    auto load_b = [&]() {
#pragma unroll
        for (int g = 0; g < TPT; g++) {
            const int ih = ih0 + g_dr[g], iw = iw0 + g_ds[g];
            const int bad = ih | (p.H - 1 - ih) | iw | (p.W - 1 - iw) | oob_pix;  // sign bit: outside
            const unsigned voff = bad < 0 ? kOobOffset : (unsigned)(x_pix + g_disp[g]) * 4u;
#pragma unroll
            for (int ii = 0; ii < GSZ; ii++)
                breg[g * GSZ + ii] = buffer_load_f32(rx, voff, (unsigned)((g_c0[g] + 16 * ii) * HW) * 4u);
        }
    };
    // rows (or columns) r0 + 32 e and r0 + 32 e + 16: after the swap lanes 0 .. 31 hold both pixels of the first, the others of the second
    const int half = (lane & 15) / 4;   // eight pixels: slab half / 2, half of the slab half % 2
    const int w_lds = half / 2 * 6, w_half = half % 2, w_row = r0 + 16 * kh, w_word = lane & 3;
    auto store = [&](float v0, float v1, int e, float *operand, int pitch) {
        const auto both = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v0 * kSplitUp), __builtin_bit_cast(unsigned, v1 * kSplitUp), false, false);
        unsigned q[3];
        const unsigned even = both[0], odd = both[1];   // (a bit cast of a vector's element takes its first one)
        split_pair(__builtin_bit_cast(float, even), __builtin_bit_cast(float, odd), q[0], q[1], q[2]);
#pragma unroll
        for (int t = 0; t < 3; t++) ((unsigned *)operand)[((w_lds + t * 2 + w_half) * pitch + w_row + 32 * e) * 4 + w_word] = q[t];
    };
    auto store_pair = [&](float *buf, int e) {   // pair e of A's and then of B's
        if (e < NA / 2) store(areg[2 * e], areg[2 * e + 1], e, buf, PA);
        else store(breg[2 * e - NA], breg[2 * e - NA + 1], e - NA / 2, buf + BOFF, PB);
    };

    // Chains of sixteen slabs (see conv_gather_body), in pairs of stages, whose places in LDS are then fixed: 5 x 5 at
    // stride 2, 48 -> 100 on 50 images of 45 x 39, 75 -> 72 us.  0.83 times as far off float64 as when the reduction was cut for twice
    // as many workgroups, without the chains 1.1 and up to 1.5 times.  Tiles of 64 rows run as two workgroups per CU, which leaves no registers for a second accumulator.
    constexpr bool kChains = BM > 64;
    v16f acc[MI][NI], low[MI][NI], sum[MI][NI];
    zero_acc(acc);
    zero_acc(low);
    zero_acc(sum);
    const int a_frag = (kh * PA + wm * (BM / T::WM) + l32) * 4, b_frag = BOFF + (kh * PB + wn * (BN / T::WN) + l32) * 4;
    v4u a[2][MI][3], b[2][NI][3];
    auto fragments = [&](const float *buf, int sl) {
#pragma unroll
        for (int t = 0; t < 3; t++) {
#pragma unroll
            for (int i = 0; i < MI; i++) a[sl][i][t] = *(const v4u *)(buf + a_frag + ((sl * 6 + t * 2) * PA + 32 * i) * 4);
#pragma unroll
            for (int j = 0; j < NI; j++) b[sl][j][t] = *(const v4u *)(buf + b_frag + ((sl * 6 + t * 2) * PB + 32 * j) * 4);
        }
    };
    constexpr int PAIRS = (NA + NB) / 2;
    static_assert(PAIRS <= 10, "a pair per step, the loads behind them");
    slab = slab_begin;
    load_a();
    load_b();
#pragma unroll
    for (int e = 0; e < PAIRS; e++) store_pair(lds, e);
    const int stages = (slab_end - slab_begin + SL - 1) / SL;
    if (stages > 1) {
        load_a();
        load_b();
    }
    __syncthreads();
    auto stage = [&](const float *cur, float *nxt, auto more_tag) {
        constexpr bool more = decltype(more_tag)::value != 0;
        fragments(cur, 0);
        static_for<0, 6 * SL>([&](auto tag) {
            constexpr int step = decltype(tag)::value, sl = step / 6, s = step % 6;
            if constexpr (step == 0) fragments(cur, 1);
            if constexpr (more && step < PAIRS) store_pair(nxt, step);
            if constexpr (more && step == NA / 2) load_a();   // (the registers' last values have just been stored)
            if constexpr (more && step == PAIRS) load_b();
            // smallest products first: l.h, h.l, m.m, m.h, h.m, h.h
            constexpr int qa = s == 0 ? 2 : s == 2 || s == 3 ? 1 : 0, qb = s == 1 ? 2 : s == 2 || s == 4 ? 1 : 0;
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NI; j++) {
                    v16f &c = s < 5 ? low[i][j] : acc[i][j];
                    c = mfma_bf16(a[sl][i][qa], b[sl][j][qb], c);
                }
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (more) __syncthreads();
    };
    int st = 0;
    if constexpr (kChains) {
        while (st + 8 <= stages - 1) {
#pragma unroll 1
            for (int pair = 0; pair < 4; pair++, st += 2) {
                stage(lds, lds + STAGE, StepTag<1>{});
                stage(lds + STAGE, lds, StepTag<1>{});
            }
            move_acc(sum, acc);
        }
    }
    for (; st < stages - 1; ++st) stage(lds + (st & 1) * STAGE, lds + (~st & 1) * STAGE, StepTag<1>{});
    stage(lds + ((stages - 1) & 1) * STAGE, nullptr, StepTag<0>{});
    move_acc(sum, acc);
    add_acc(sum, low);

    // the parts of an infinity hold NaNs: a tile that is not finite is formed again with the fp32 instruction, a stage at a time
    if (__syncthreads_or(not_finite(sum))) {
        zero_acc(sum);
        slab = slab_begin;
#pragma unroll 1
        for (int st = 0; st < stages; ++st) {
            load_a();
            load_b();
            __syncthreads();
            // here [slab][half][row][8 pixels]
            const int at = px / 16 * 2 + px / 8 % 2;
#pragma unroll
            for (int i = 0; i < NA; i++) lds[(at * PA + r0 + 16 * i) * 8 + px % 8] = areg[i];
#pragma unroll
            for (int i = 0; i < NB; i++) lds[BOFF + (at * PB + r0 + 16 * i) * 8 + px % 8] = breg[i];
            __syncthreads();
#pragma unroll 1
            for (int sl = 0; sl < SL; sl++)
#pragma unroll 1
                for (int e = 0; e < 8; e++)
#pragma unroll
                    for (int i = 0; i < MI; i++)
#pragma unroll
                        for (int j = 0; j < NI; j++)
                            sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(lds[((sl * 2 + kh) * PA + wm * (BM / T::WM) + l32 + 32 * i) * 8 + e],
                                                                              lds[BOFF + ((sl * 2 + kh) * PB + wn * (BN / T::WN) + l32 + 32 * j) * 8 + e],
                                                                              sum[i][j], 0, 0, 0);
        }
    }

    float *outp = p.out + (size_t)split * p.out_elems;
#pragma unroll
    for (int j = 0; j < T::NI; j++) {
        const int col = n0 + wn * (BN / T::WN) + j * 32 + (lane & 31);
        if (col >= p.ncols) continue;
#pragma unroll
        for (int i = 0; i < T::MI; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int m = m0 + wm * (BM / T::WM) + i * 32 + acc_row(v, lane);
                if (m < p.K) outp[(size_t)m * p.ncols + col] = sum[i][j][v];
            }
    }
}

// dw[k][c][tap] = sum_s partial[s][k][tap*Cp + c], summed in a fixed order (reproducible).
// Block (k, chunk of `ch` channels): 64 element lanes x 4 split lanes.  Wavefront sl folds the
// splits s = sl, sl+4, ... of every element with four independent chains (the split count reaches
// the hundreds for the wide early layers, one dependent chain per element would be latency
// bound); the four wavefront sums are then added in order, and the chunk is written out
// contiguously in [c][tap] order.
__global__ __launch_bounds__(256) void wgrad_reduce_k(int K, int C, int Cp, int taps, int ch, int splits,
                                                       size_t split_stride, const float *partial, float *dw)
{
    extern __shared__ float lds[];  // part[4][ch*taps] then stage[ch*taps]
    const int k = blockIdx.x, c0 = blockIdx.y * ch;
    const int nc = min(ch, C - c0);
    const int nelem = nc * taps, cap = ch * taps;
    float *part = lds, *stage = lds + 4 * cap;
    const int el = threadIdx.x & 63, sl = threadIdx.x >> 6;
    const float *src = partial + (size_t)k * taps * Cp + c0;
    for (int i = el; i < nelem; i += 64) {
        const int t = i / nc, c = i - t * nc;
        const float *q = src + (size_t)t * Cp + c;
        float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
        int sp = sl;
        for (; sp + 12 < splits; sp += 16) {
            a0 += q[(size_t)sp * split_stride];
            a1 += q[(size_t)(sp + 4) * split_stride];
            a2 += q[(size_t)(sp + 8) * split_stride];
            a3 += q[(size_t)(sp + 12) * split_stride];
        }
        for (; sp < splits; sp += 4) a0 += q[(size_t)sp * split_stride];
        part[sl * cap + i] = (a0 + a1) + (a2 + a3);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nelem; i += 256) {
        const int t = i / nc, c = i - t * nc;
        stage[c * taps + t] = (part[i] + part[cap + i]) + (part[2 * cap + i] + part[3 * cap + i]);
    }
    __syncthreads();
    float *dst = dw + ((size_t)k * C + c0) * taps;
    for (int i = threadIdx.x; i < nelem; i += 256) dst[i] = stage[i];
}

// Quad i of a result of n values that may start anywhere and end inside a quad.
__device__ __forceinline__ void store_loose(float *out, size_t n, size_t i, float4 v)
{
    const float q[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (4 * i + e < n) out[4 * i + e] = q[e];
}

// The same for small filters of many copies, where K blocks a chunk leave the chip idle and a thread goes through its copies several
// times: a block takes 64 of a row's elements in the copies' order and sixteen split lanes (lane sl: copies sl, sl + 16 .., four
// chains), whose sums are added in order, all in float64 (with sixteen roundings in a row the error was 1.1 times wgrad_reduce_k's).
// Results are written a word at a time.  The five such layers of a WRN-10-2 step on 64 images 9.3 -> 5 us each, 100 x 48 x 25 values
// 10.1 -> 7.4.
__global__ __launch_bounds__(1024) void wgrad_reduce_small_k(int C, int Cp, int taps, int splits, size_t split_stride, const float *partial, float *dw)
{
    __shared__ double part[16][64];
    const int k = blockIdx.x, el = threadIdx.x & 63, sl = threadIdx.x >> 6, i = blockIdx.y * 64 + el;
    const int t = i / C, c = i - t * C;
    if (t < taps) {
        const float *const q = partial + ((size_t)k * taps + t) * Cp + c;
        double a0 = 0, a1 = 0, a2 = 0, a3 = 0;
        int sp = sl;
        for (; sp + 48 < splits; sp += 64) {
            const float v0 = q[(size_t)sp * split_stride], v1 = q[(size_t)(sp + 16) * split_stride];
            const float v2 = q[(size_t)(sp + 32) * split_stride], v3 = q[(size_t)(sp + 48) * split_stride];
            a0 += v0, a1 += v1, a2 += v2, a3 += v3;
        }
        // up to three more, together
        const int last = splits - 1;
        const float v0 = q[(size_t)min(sp, last) * split_stride], v1 = q[(size_t)min(sp + 16, last) * split_stride], v2 = q[(size_t)min(sp + 32, last) * split_stride];
        if (sp <= last) a0 += v0;
        if (sp + 16 <= last) a1 += v1;
        if (sp + 32 <= last) a2 += v2;
        part[sl][el] = (a0 + a1) + (a2 + a3);
    }
    __syncthreads();
    if (sl == 0 && t < taps) {
        double sum = part[0][el];
#pragma unroll
        for (int s = 1; s < 16; s++) sum += part[s][el];
        dw[((size_t)k * C + c) * taps + t] = (float)sum;
    }
}

// out[i] = sum over s of partial[s * stride + i], in a fixed order: split lane sl of a block folds
// the splits s = sl, sl + SL, ... (four independent chains, then ((a0+a1)+(a2+a3))), and the SL
// lane sums are added in lane order.  256 threads = (256 / SL) float4 columns x SL split lanes; SL
// is chosen by the host so that small outputs with hundreds of splits still fill the machine.
template <int SL, bool kLoose = false>
__global__ __launch_bounds__(256) void split_sum_k(size_t n4, int splits, size_t stride4, const float4 *partial,
                                                    float4 *out, size_t n = 0)
{
    constexpr int EL = 256 / SL;
    __shared__ float4 part[SL][EL];
    const int el = threadIdx.x % EL, sl = threadIdx.x / EL;
    const size_t i = (size_t)blockIdx.x * EL + el;
    float4 a0 = make_float4(0.f, 0.f, 0.f, 0.f), a1 = a0, a2 = a0, a3 = a0;
    if (i < n4) {
        const float4 *q = partial + i;
        int sp = sl;
        for (; sp + 3 * SL < splits; sp += 4 * SL) {
            const float4 v0 = q[(size_t)sp * stride4], v1 = q[(size_t)(sp + SL) * stride4];
            const float4 v2 = q[(size_t)(sp + 2 * SL) * stride4], v3 = q[(size_t)(sp + 3 * SL) * stride4];
            a0.x += v0.x; a0.y += v0.y; a0.z += v0.z; a0.w += v0.w;
            a1.x += v1.x; a1.y += v1.y; a1.z += v1.z; a1.w += v1.w;
            a2.x += v2.x; a2.y += v2.y; a2.z += v2.z; a2.w += v2.w;
            a3.x += v3.x; a3.y += v3.y; a3.z += v3.z; a3.w += v3.w;
        }
        for (; sp < splits; sp += SL) {
            const float4 v0 = q[(size_t)sp * stride4];
            a0.x += v0.x; a0.y += v0.y; a0.z += v0.z; a0.w += v0.w;
        }
    }
    part[sl][el] = make_float4((a0.x + a1.x) + (a2.x + a3.x), (a0.y + a1.y) + (a2.y + a3.y),
                               (a0.z + a1.z) + (a2.z + a3.z), (a0.w + a1.w) + (a2.w + a3.w));
    __syncthreads();
    if (sl == 0 && i < n4) {
        float4 r = part[0][el];
#pragma unroll
        for (int k = 1; k < SL; k++) {
            const float4 v = part[k][el];
            r.x += v.x; r.y += v.y; r.z += v.z; r.w += v.w;
        }
        if constexpr (kLoose) store_loose((float *)out, n, i, r);
        else out[i] = r;
    }
}

// ------------------------------------------------------------------------------------ backward-filter, 3x3 patch
//
// Filter gradient of 3x3, unit-stride, pad-1 convolutions:
//   dw[k][c][2-r][2-s] = sum over (n, p, q) of dy[n][k][p][q] * x[n][c][p-1+r][q-1+s].
// The reduction runs over pixels.  A block owns BM output channels x BC input channels x all nine
// taps (BM x BC = 128 x 32, 64 x 64, or 160 x 32 for layers of 160 channels, which the other two would pad by
// a fifth and more) and walks the pixels in chunks of 64.  Per chunk it stages dy[BM][64] and ONE zero-haloed
// patch of x for its BC channels in LDS; the nine taps read that patch at nine offsets, so x is
// fetched once, not nine times.  The twelve wavefronts are (32 rows of k) x (32 channels) x
// (tap row r): a wavefront keeps the three taps s = 0..2 of its tap row in three 32x32
// accumulators.  A lane's operands for a 16-pixel slab are pixels kh*8 .. kh*8+7 of the slab
// (kh = lane / 32): two 128-bit reads of dy, and for x a window that serves all three taps by
// register selection.  The products run on the bf16 matrix instruction, each operand split into three parts
// (mfma_core.h).
//
// Geometry of a 64-pixel chunk (kGeo):
//   0  rows of 8, 16, 32 or 64 pixels: G = 64/W full rows of one image.  Patch rows have pitch W+8
//      with pixel q at column q+4, so interior quads are 16-byte aligned; a lane's window is two
//      aligned quads plus the two edge columns.  The halo rows above and below are fetched (or
//      masked at the image border); the halo columns are cleared once and never written.
//   1  4x4 images: four whole images.  Same column layout (pitch 12); a lane's 8 pixels are two
//      rows, each one aligned quad plus two edge columns.  All halo cells stay zero.
//   2  2x2 images: sixteen whole images, each a 4x4 cell block with the image in the middle; a
//      lane's 8 pixels are two images, and one aligned quad per (image, row) holds every column
//      the three taps need.

struct WgradPatch {
    const float *dy;  // [N, K, H, W]
    const float *x;   // [N, C, H, W]
    float *out;       // dw [K][C][3][3], or `splits` partial copies of it `split_stride` floats apart
    size_t split_stride;
    int N, C, K, H, W;
    int G, bands;         // geometry 0: output rows per chunk (G*W = 64), chunks per image; else 1
    int imgs;             // images per chunk (1, 4 or 16)
    int ppitch, cstride;  // patch row pitch; floats per channel (128-bit reads by 32 channels hit every bank once)
    int quads_row;        // W / 4 (geometry 0)
    int mtiles, ctiles, chunks_total, chunks_per_split, splits;
    size_t dy_bytes, x_bytes;
};

template <int WM, int WC, int kGeo, bool kPre>
__device__ __forceinline__ void conv_wgrad_patch_body(const WgradPatch &p, const unsigned block_id)
{
    constexpr int BM = 32 * WM, BC = 32 * WC, THREADS = 64 * 3 * WM * WC, NPIX = 64, APITCH = NPIX + 4;
    constexpr int NAQ = (BM * NPIX / 4 + THREADS - 1) / THREADS;  // float4 slots of dy per thread
    // float4 slots of x per thread: geometry 0 up to 32*4*8 (W = 32) or 32*3*16 (W = 64) quads per 32
    // channels; geometries 1, 2 have 16 quads per channel
    constexpr int NBQ = kGeo == 0 ? (WC == 1 ? 2 : 3) : (BC * 16 + THREADS - 1) / THREADS;
    static_assert(WM * WC == 4 || WM * WC == 5, "twelve or fifteen wavefronts: 4 or 5 (row, channel) groups x 3 tap rows");
    extern __shared__ __attribute__((aligned(16))) float lds[];
    // first column of a patch row; pitch of the rows of a 4 x 4 image, and its distance to the next image
    constexpr int COL0 = kPre && kGeo == 0 ? 8 : 4, RP1 = kPre ? 8 : 12, IP1 = kPre ? 40 : 72;
    const int bsize = BC * p.cstride;
    const int bstride = kPre ? bsize / 2 * 3 : bsize;           // floats of a patch buffer: three 16-bit parts a value
    float *const A0 = lds;                                      // [2][BM * APITCH]
    float *const B0 = lds + 2 * BM * APITCH - (kPre ? 4 : 0);   // [2][bstride] (the pad of the last row before it is not used)
    float *const dummy = B0 + 2 * bstride;                      // 4 floats absorbing the stores of unused slots

    unsigned L;
    const unsigned tiles = (unsigned)(p.mtiles * p.ctiles);
    if (!xcd_remap(block_id, tiles * (unsigned)p.splits, &L)) return;
    const int split = (int)(L / tiles);
    const unsigned tile = L - (unsigned)split * tiles;
    const int mt = (int)(tile % (unsigned)p.mtiles), ct = (int)(tile / (unsigned)p.mtiles);
    const int k0 = mt * BM, c0 = ct * BC;
    const int cb = split * p.chunks_per_split;
    const int ce = min(cb + p.chunks_per_split, p.chunks_total);
    // The sum over the chunks is formed in kPasses parts of alternating sign, the first of which waits in `out` (see the products below).
    constexpr bool kLow = WM * WC == 4;
    constexpr int kPasses = kLow ? 1 : 2;
    int from = cb, to = kPasses == 1 ? ce : (cb + ce + 1) / 2;
    float up = kSplitUp;   // its sign alternates

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int kh = lane >> 5, l32 = lane & 31;
    const int dr = w % 3, grp = w / 3;
    const int wm = grp / WC, wc = grp % WC;
    const int HW = p.H * p.W;

    const __amdgpu_buffer_rsrc_t rdy = make_rsrc(p.dy, p.dy_bytes);
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, p.x_bytes);

    // ---- load slots.  dy: quad `quad` of row `row` is pixels 4*quad .. 4*quad+3 of the chunk, which
    // lie in image quad / qpi of the chunk (qpi = quads of one image inside a chunk).  Slot i of a thread is the quad AROWS i
    // rows below its first one, so one offset and one LDS place serve all of them.
    constexpr int AROWS = THREADS / 16;
    const int qpi = kGeo == 0 ? 16 : HW / 4;
    const int a_row = tid / 16, a_quad = tid % 16;
    const unsigned a_voff = (unsigned)((a_quad / qpi * p.K + k0 + a_row) * HW + a_quad % qpi * 4) * 4u;
    const int a_lds = a_row * APITCH + a_quad * 4;
    const int a_rows = min(BM, p.K - k0);
    unsigned b_voff[NBQ];
    int b_lds[NBQ];   // index of the value inside a patch buffer (a multiple of four) or -1; geometry 0: + 1 = top halo row, + 2 = bottom halo row
#pragma unroll
    for (int i = 0; i < NBQ; i++) {
        const int b = i * THREADS + tid;
        if (kGeo == 0) {
            const int quads_ch = (p.G + 2) * p.quads_row;
            const int c = b / quads_ch, rem = b - c * quads_ch;
            const int pr = rem / p.quads_row, quad = rem - pr * p.quads_row;
            const bool ok = c < BC && c0 + c < p.C;
            // row p0 - 1 + pr of channel c0 + c; p0 and the image are added per chunk
            b_voff[i] = ok ? (unsigned)(((c0 + c) * p.H + pr) * p.W + quad * 4) * 4u : kOobOffset;
            b_lds[i] = c < BC ? c * p.cstride + pr * p.ppitch + COL0 + quad * 4 + (pr == 0 ? 1 : pr == p.G + 1 ? 2 : 0) : -1;
        } else if (kGeo == 1) {
            const int c = b / 16, j = (b / 4) % 4, row = b % 4;  // image j of the chunk, image row `row`
            const bool ok = c < BC && c0 + c < p.C;
            b_voff[i] = ok ? (unsigned)((j * p.C + c0 + c) * 16 + row * 4) * 4u : kOobOffset;
            b_lds[i] = c < BC ? c * p.cstride + j * IP1 + (row + 1) * RP1 + COL0 : -1;
        } else {
            const int c = b / 16, j = b % 16;  // the whole 2x2 image j is one quad
            const bool ok = c < BC && c0 + c < p.C;
            b_voff[i] = ok ? (unsigned)((j * p.C + c0 + c) * 4) * 4u : kOobOffset;
            b_lds[i] = c < BC ? c * p.cstride + j * 16 + 5 : -1;  // cell (1,1) of the 4x4 block
        }
    }
    float4 areg[NAQ], breg[NBQ];
    // position of the chunk being FETCHED: first image and, for geometry 0, the band of rows
    int n_img, band;
    auto fetch = [&]() {
        const int p0 = band * p.G;
        const unsigned a_soff = (unsigned)(n_img * p.K * HW + p0 * p.W) * 4u;
#pragma unroll
        for (int i = 0; i < NAQ; i++)
            areg[i] = buffer_load_f32x4(rdy, a_row + AROWS * i < a_rows ? a_voff + (unsigned)(AROWS * i * HW) * 4u : kOobOffset, a_soff);
        if (kGeo == 0) {
            // x row p0 - 1 + pr.  Offsets handed to a buffer load must not go negative: the "- 1" row
            // is taken off the wave-uniform part, except for the very first chunk of the tensor, where
            // it is taken off the per-lane part (whose top halo row, the only one it could underflow,
            // is masked)
            const int kill = (band == 0 ? 1 : 0) | (band == p.bands - 1 ? 2 : 0);
            const bool first = n_img == 0 && band == 0;
            const unsigned roww = (unsigned)p.W * 4u;
            const unsigned b_soff = (unsigned)(n_img * p.C * HW + p0 * p.W) * 4u - (first ? 0u : roww);
#pragma unroll
            for (int i = 0; i < NBQ; i++) {
                const bool dead = (b_lds[i] & kill) != 0 || b_voff[i] == kOobOffset;
                breg[i] = buffer_load_f32x4(rx, dead ? kOobOffset : b_voff[i] - (first ? roww : 0u), b_soff);
            }
            if (++band == p.bands) {
                band = 0;
                ++n_img;
            }
        } else {
            const unsigned b_soff = (unsigned)(n_img * p.C * HW) * 4u;
#pragma unroll
            for (int i = 0; i < NBQ; i++) breg[i] = buffer_load_f32x4(rx, b_voff[i], b_soff);
            n_img += p.imgs;
        }
    };
    auto stash = [&](int buf, auto exact_tag) {
        constexpr bool exact = decltype(exact_tag)::value != 0;
        float *A = A0 + buf * (BM * APITCH), *B = B0 + buf * bstride;
#pragma unroll
        for (int i = 0; i < NAQ; i++) {
            const float4 v = areg[i];
            const float by = kLow ? kSplitUp : up;
            *(float4 *)(AROWS * (i + 1) <= BM || a_row + AROWS * i < BM ? A + a_lds + AROWS * i * APITCH : dummy) =
                exact ? v : make_float4(v.x * by, v.y * by, v.z * by, v.w * by);
        }
#pragma unroll
        for (int i = 0; i < NBQ; i++) {
            const float4 v = exact ? breg[i] : make_float4(breg[i].x * kSplitUp, breg[i].y * kSplitUp, breg[i].z * kSplitUp, breg[i].w * kSplitUp);
            if constexpr (kPre && !exact) {
                uint2 q3[3];
                split_pair(v.x, v.y, q3[0].x, q3[1].x, q3[2].x);
                split_pair(v.z, v.w, q3[0].y, q3[1].y, q3[2].y);
#pragma unroll
                for (int t = 0; t < 3; t++) *(uint2 *)(b_lds[i] >= 0 ? B + t * (bsize / 2) + (b_lds[i] & ~3) / 2 : dummy) = q3[t];
            } else if constexpr (kGeo != 2) {
                *(float4 *)(b_lds[i] >= 0 ? B + (b_lds[i] & ~3) : dummy) = v;
            } else {
                float *q = b_lds[i] >= 0 ? B + b_lds[i] : dummy;  // rows 1 and 2 of the cell block, columns 1..2
                const int down = b_lds[i] >= 0 ? 4 : 0;
                q[0] = v.x;
                q[1] = v.y;
                q[down] = v.z;
                q[down + 1] = v.w;
            }
        }
    };

    // ---- fragment addresses
    const int a_frag = (wm * 32 + l32) * APITCH + kh * 8;
    // index inside a patch buffer: of slab 0, and how far the other slabs are from it (the same for all lanes)
    const int runs_row = p.W / 8;
    const int b_frag = kGeo == 0 ? (wc * 32 + l32) * p.cstride + (dr + (runs_row == 1 ? kh : 0)) * p.ppitch + (runs_row == 1 ? 0 : kh * 8) + COL0
                     : kGeo == 1 ? (wc * 32 + l32) * p.cstride + (2 * kh + dr) * RP1 + COL0     // image s, image rows 2kh and 2kh+1
                                 : (wc * 32 + l32) * p.cstride + 2 * kh * 16 + dr * 4;          // images 4s+2kh and 4s+2kh+1
    // geometry 0: slab s covers the 8-pixel runs 2s (kh = 0) and 2s+1 (kh = 1) of the chunk
    auto b_step = [&](int s) { return kGeo == 0 ? 2 * s / runs_row * p.ppitch + 2 * s % runs_row * 8 : kGeo == 1 ? s * IP1 : s * 64; };

    v16f acc[3], low[kLow ? 3 : 1];
    typedef __attribute__((address_space(3))) float lds_float_t;
    // Fetching runs one chunk ahead, or two, and also past the end of this block's range: those loads are
    // range-checked and their data lands in the LDS buffer that is not read again.
    // Two chunks ahead a chunk is stored at the beginning of the one before it, and the wavefronts of a SIMD, which have
    // drifted apart behind the barrier by then, store under each other's matrix instructions; one ahead, at its end, they all
    // store at once.  It takes registers: not with fifteen wavefronts.
    constexpr bool kEarly = kPre && kLow;
    struct Frag {
        float4 a_lo, a_hi, q[4];
        float e[4];
    };
    auto read_frag = [&](int buf, int s_, auto parts_tag) {
        constexpr bool parts = decltype(parts_tag)::value != 0;   // dy alone
        Frag f;
        const float *A = A0 + buf * (BM * APITCH) + a_frag;
        // float4 indexing keeps the 16-byte alignment of the patch reads visible to the compiler
        const float4 *bq = (const float4 *)B0 + (buf * bstride + b_frag + b_step(s_)) / 4;
        // The edge-column reads are volatile so that the compiler does not fuse a whole window
        // into one run starting at the unaligned edge (it would then read it in 2-dword pieces).
        const volatile lds_float_t *be = (const volatile lds_float_t *)bq;
        f.a_lo = *(const float4 *)(A + s_ * 16);
        f.a_hi = *(const float4 *)(A + s_ * 16 + 4);
        if constexpr (parts) return f;
        if constexpr (kGeo == 0) {
            f.q[0] = bq[0]; f.q[1] = bq[1];
            f.e[0] = be[-1]; f.e[1] = be[8];
        } else if constexpr (kGeo == 1) {
            f.q[0] = bq[0]; f.q[1] = bq[RP1 / 4];
            f.e[0] = be[-1]; f.e[1] = be[4]; f.e[2] = be[RP1 - 1]; f.e[3] = be[RP1 + 4];
        } else {
            // (image, row) quads: image 0 rows 0, 1 then image 1 rows 0, 1
            f.q[0] = bq[0]; f.q[1] = bq[1]; f.q[2] = bq[4]; f.q[3] = bq[5];
        }
        return f;
    };
    auto products_fp32 = [&](const Frag &f) {
        const float a8[8] = {f.a_lo.x, f.a_lo.y, f.a_lo.z, f.a_lo.w, f.a_hi.x, f.a_hi.y, f.a_hi.z, f.a_hi.w};
        if constexpr (kGeo == 0) {
            const float4 b_lo = f.q[0], b_hi = f.q[1];
            const float win[10] = {f.e[0], b_lo.x, b_lo.y, b_lo.z, b_lo.w, b_hi.x, b_hi.y, b_hi.z, b_hi.w, f.e[1]};
#pragma unroll
            for (int ks = 0; ks < 8; ks++)
#pragma unroll
                for (int ds = 0; ds < 3; ds++)
                    acc[ds] = __builtin_amdgcn_mfma_f32_32x32x2f32(a8[ks], win[ks + ds], acc[ds], 0, 0, 0);
        } else if constexpr (kGeo == 1) {
            const float4 r0 = f.q[0], r1 = f.q[1];
            const float w0[6] = {f.e[0], r0.x, r0.y, r0.z, r0.w, f.e[1]};
            const float w1[6] = {f.e[2], r1.x, r1.y, r1.z, r1.w, f.e[3]};
#pragma unroll
            for (int ks = 0; ks < 8; ks++)
#pragma unroll
                for (int ds = 0; ds < 3; ds++)
                    acc[ds] = __builtin_amdgcn_mfma_f32_32x32x2f32(a8[ks], ks < 4 ? w0[ks + ds] : w1[ks - 4 + ds],
                                                                   acc[ds], 0, 0, 0);
        } else {
            // pixel (row, col) of tap column ds reads element col + ds of the quad of patch row row + dr
            const float4 q00 = f.q[0], q01 = f.q[1], q10 = f.q[2], q11 = f.q[3];
            const float win[4][4] = {{q00.x, q00.y, q00.z, q00.w}, {q01.x, q01.y, q01.z, q01.w},
                                     {q10.x, q10.y, q10.z, q10.w}, {q11.x, q11.y, q11.z, q11.w}};
#pragma unroll
            for (int ks = 0; ks < 8; ks++)
#pragma unroll
                for (int ds = 0; ds < 3; ds++)
                    acc[ds] = __builtin_amdgcn_mfma_f32_32x32x2f32(a8[ks], win[ks / 2][(ks & 1) + ds], acc[ds], 0, 0, 0);
        }
    };
    // The same sixteen pixels on the bf16 matrix instructions (eighteen of 32 cycles for twenty-four of 64): dy's fragments are
    // split in registers (mfma_core.h); x, which twelve wavefronts read, when it is stored (kPre), in pairs of pixels that are tap
    // column 1's operands as they are; those of columns 0 and 2 are their neighbouring halves with the edge pixels.  320 -> 320
    // channels on 16 x 16, batch 128: both split in registers 296 us, x when stored 289, stored at the beginning of a chunk 278;
    // 640 -> 640 on 8 x 8 305, 296, 279; of them 205 us are matrix time at the rate of a large product.  (Reading the fragments one step
    // ahead, as the fp32 form did, needs 30 more registers than there are.)
    // The instruction rounds down what lies below its guard bits.  That is the same way in every block, so no sum over blocks
    // removes it, and the five small products of a slab suffer it most: with all six in one accumulator 77 % of the error was a
    // common offset, and it was 1.25 to 1.7 times the fp32 instruction's.  So twelve wavefronts keep the small products in an
    // accumulator of their own (which fits since a thread's dy slots share an offset and the slabs' places are scalars); fifteen
    // have no registers for it and add the chunks in two halves of opposite sign instead, whose offsets cancel.
    // 128 images of 320 -> 320 channels, 16 x 16: fp32 450 us, one accumulator 292, this 296; 160 -> 160, 32 x 32: 486, 302, 327.
    // Error against float64 (one half of x zero): 64 -> 64 channels, 32 x 32, 2.8e-7 / 4.8e-7 / 1.3e-7; 160 -> 160, 32 x 32,
    // 6.4e-7 / 1.07e-6 / 5.2e-7; 640 -> 640, 8 x 8, batch 256, 6.7e-7 / 8.4e-7 / 2.6e-7.
    constexpr int NW = kPre ? 6 : kGeo == 0 ? 5 : kGeo == 1 ? 6 : 8;   // pairs of pixels
    v4u ap[3];
    unsigned q[3][NW];
    auto split_frag = [&](const Frag &f) {
        {
            uint2 l0, l1;
            v4u hm0, hm1;
            split_quad(f.a_lo, hm0, l0);
            split_quad(f.a_hi, hm1, l1);
            ap[0] = v4u{hm0.x, hm0.y, hm1.x, hm1.y};
            ap[1] = v4u{hm0.z, hm0.w, hm1.z, hm1.w};
            ap[2] = v4u{l0.x, l0.y, l1.x, l1.y};
        }
        if constexpr (kPre) return;
        static_for<0, kGeo == 2 ? 4 : 2>([&](auto itag) {
            constexpr int i = decltype(itag)::value;
            split_pair(f.q[i].x, f.q[i].y, q[0][2 * i], q[1][2 * i], q[2][2 * i]);
            split_pair(f.q[i].z, f.q[i].w, q[0][2 * i + 1], q[1][2 * i + 1], q[2][2 * i + 1]);
        });
        if constexpr (kGeo != 2) split_pair(f.e[0], f.e[1], q[0][4], q[1][4], q[2][4]);
        if constexpr (kGeo == 1) split_pair(f.e[2], f.e[3], q[0][NW - 1], q[1][NW - 1], q[2][NW - 1]);
    };
    auto read_parts = [&](int buf, int s_) {   // the x window's pairs where they were split when stored
        const unsigned *const first = (const unsigned *)B0 + buf * bstride + (b_frag + b_step(s_)) / 2;
#pragma unroll
        for (int t = 0; t < 3; t++) {
            const unsigned *const w = first + t * (bsize / 2);
            if constexpr (kGeo == 0) {
                const v4u m = *(const v4u *)w;
                q[t][0] = m.x; q[t][1] = m.y; q[t][2] = m.z; q[t][3] = m.w;
                q[t][4] = w[-1]; q[t][NW - 1] = w[4];
            } else {
                const uint2 r0 = *(const uint2 *)w, r1 = *(const uint2 *)(w + RP1 / 2);
                q[t][0] = r0.x; q[t][1] = r0.y; q[t][2] = r1.x; q[t][3] = r1.y;
            }
        }
    };
    auto products_split = [&]() {
        auto mid = [](unsigned hi, unsigned lo) { return __builtin_amdgcn_alignbit(hi, lo, 16); };             // (lo.1, hi.0)
        auto left = [](unsigned e, unsigned w) { return __builtin_amdgcn_perm(w, e, 0x05040100u); };            // (e.0, w.0)
        auto right = [](unsigned w, unsigned e) { return __builtin_amdgcn_perm(e, w, 0x07060302u); };           // (w.1, e.1)
        static_for<0, 3>([&](auto ptag) {
            constexpr int part = 2 - decltype(ptag)::value;
            const unsigned *const w = q[part];
            v4u b[3];
            if constexpr (kPre && kGeo == 0) {   // (the edge words hold two pixels of which one is the window's)
                const unsigned m0 = mid(w[1], w[0]), m1 = mid(w[2], w[1]), m2 = mid(w[3], w[2]);
                b[0] = v4u{mid(w[0], w[4]), m0, m1, m2};
                b[1] = v4u{w[0], w[1], w[2], w[3]};
                b[2] = v4u{m0, m1, m2, mid(w[NW - 1], w[3])};
            } else if constexpr (kPre) {         // (what is left and right of a 4 x 4 image's row is zero)
                const unsigned m0 = mid(w[1], w[0]), m1 = mid(w[3], w[2]);
                b[0] = v4u{w[0] << 16, m0, w[2] << 16, m1};
                b[1] = v4u{w[0], w[1], w[2], w[3]};
                b[2] = v4u{m0, w[1] >> 16, m1, w[3] >> 16};
            } else if constexpr (kGeo == 0) {
                const unsigned m0 = mid(w[1], w[0]), m1 = mid(w[2], w[1]), m2 = mid(w[3], w[2]);
                b[0] = v4u{left(w[4], w[0]), m0, m1, m2};
                b[1] = v4u{w[0], w[1], w[2], w[3]};
                b[2] = v4u{m0, m1, m2, right(w[3], w[4])};
            } else if constexpr (kGeo == 1) {
                const unsigned m0 = mid(w[1], w[0]), m1 = mid(w[3], w[2]);
                b[0] = v4u{left(w[4], w[0]), m0, left(w[NW - 1], w[2]), m1};
                b[1] = v4u{w[0], w[1], w[2], w[3]};
                b[2] = v4u{m0, right(w[1], w[4]), m1, right(w[3], w[NW - 1])};
            } else {
                b[0] = v4u{w[0], w[2], w[4], w[NW - 2]};
                b[1] = v4u{mid(w[1], w[0]), mid(w[3], w[2]), mid(w[5 % NW], w[4]), mid(w[NW - 1], w[NW - 2])};
                b[2] = v4u{w[1], w[3], w[5 % NW], w[NW - 1]};
            }
            static_for<0, 3 - part>([&](auto atag) {   // x's l with dy's h; m with m, h; h with l, m, h
                constexpr int pa = 2 - part - decltype(atag)::value;
#pragma unroll
                for (int ds = 0; ds < 3; ds++) {
                    v16f &c = kLow && part + pa > 0 ? low[kLow ? ds : 0] : acc[ds];
                    c = mfma_bf16(ap[pa], b[ds], c);
                }
            });
        });
    };
    auto run = [&](auto exact_tag) {
        constexpr bool exact = decltype(exact_tag)::value != 0;
        n_img = kGeo == 0 ? from / p.bands : from * p.imgs;
        band = kGeo == 0 ? from - n_img * p.bands : 0;
#pragma unroll
        for (int t = 0; t < 3; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[t][v] = low[kLow ? t : 0][v] = 0.0f;
        // halo cells are not written by the loop
        for (int i = tid; i < 2 * bstride; i += THREADS) B0[i] = 0.0f;
        fetch();
        __syncthreads();
        stash(0, exact_tag);
        if (kEarly) fetch();
        __syncthreads();
        int cur = 0;
        for (int chunk = from; chunk < to; ++chunk) {
            static_for<0, 4>([&](auto stag) {
                constexpr int s = decltype(stag)::value;
                if constexpr (!kEarly && s == 0) fetch();
                if constexpr (exact) {
                    products_fp32(read_frag(cur, s, StepTag<0>{}));
                } else {
                    if constexpr (kPre) read_parts(cur, s);
                    split_frag(read_frag(cur, s, StepTag<kPre>{}));
                    products_split();
                }
                if constexpr (s == (kEarly ? 0 : 3)) stash(cur ^ 1, exact_tag);
                if constexpr (kEarly && s == 1) fetch();
            });
            __syncthreads();
            cur ^= 1;
        }
        if (exact) return;
#pragma unroll
        for (int t = 0; t < 3; t++)
#pragma unroll
            for (int v = 0; v < 16; v++)
                acc[t][v] = kLow ? (acc[t][v] + low[kLow ? t : 0][v]) * kSplitDown : acc[t][v] * (up * (kSplitDown / kSplitUp));
    };
    for (int pass = 0;; pass++) {
        run(StepTag<0>{});
        {
            // the parts of an infinity hold NaNs: a tile that is not finite is formed again with the fp32 instruction
            float probe = 0.0f;
#pragma unroll
            for (int t = 0; t < 3; t++)
#pragma unroll
                for (int v = 0; v < 16; v++) probe = __builtin_fmaf(acc[t][v], 0.0f, probe);
            volatile int *const again = (volatile int *)dummy;
            if (tid == 0) *again = 0;
            __syncthreads();
            if (probe != 0.0f) *again = 1;
            __syncthreads();
            const bool redo = *again != 0;
            __syncthreads();   // (forming it again may store there)
            if (redo) run(StepTag<1>{});
        }

        // Epilogue: the accumulators leave through LDS so that every output row -- the BC*9 values
        // [c][tap] of one k, contiguous in dw's own layout -- is written as one run.  One group of 32
        // rows (the wavefronts with the same wm) is staged at a time.  out = dw itself when there is one
        // split, else this split's partial copy (same layout, summed afterwards in split order).
        __syncthreads();  // all fragment reads of the last chunk are done: LDS is free
        constexpr int RP = BC * 9 + 1;  // staging row pitch (odd: the 4-row stride between lane halves spreads over banks)
        float *outp = p.out + (size_t)split * p.split_stride;
        const int ncv = min(BC, p.C - c0) * 9;  // valid floats of a staged row
        for (int g = 0; g < WM; g++) {
            if (wm == g) {
#pragma unroll
                for (int ds = 0; ds < 3; ds++) {
                    const int t = (2 - dr) * 3 + (2 - ds);
#pragma unroll
                    for (int v = 0; v < 16; v++) lds[acc_row(v, lane) * RP + (wc * 32 + l32) * 9 + t] = acc[ds][v];
                }
            }
            __syncthreads();
            for (int r = w; r < 32; r += 3 * WM * WC) {  // one wavefront per row
                const int k = k0 + g * 32 + r;
                if (k >= p.K) continue;
                float *dst = outp + ((size_t)k * p.C + c0) * 9;
                for (int j = lane; j < ncv; j += 64) dst[j] = pass == 0 ? lds[r * RP + j] : dst[j] + lds[r * RP + j];
            }
            __syncthreads();
        }
        if (pass + 1 == kPasses || to == ce) break;
        from = to;
        to = ce;
        up = -up;
    }
}

template <int WM, int WC, int kGeo, bool kPre>
__global__ __launch_bounds__(64 * 3 * WM * WC, 1) void conv_wgrad_patch_k(WgradPatch p)
{
    conv_wgrad_patch_body<WM, WC, kGeo, kPre>(p, blockIdx.x);
}

// Backward-data and filter gradient of one layer in ONE launch: both read dy and nothing of each other.
// The first `grid_a` workgroups run the backward-data tiles, the rest the filter-gradient tiles; workgroups are
// dispatched in id order, so a compute unit that has finished its backward-data tile starts a filter-gradient
// tile at once instead of idling until the slowest tile of the launch is done and the next launch has ramped up.
// Launched with the filter gradient's 768 threads: the wavefronts a backward-data workgroup does not need end
// at once (a barrier waits for the surviving wavefronts only).
template <class T, int NS, int WM, int WC, int kGeo>
__global__ __launch_bounds__(768, 1) void conv_bwd_pair_k(PatchConv a, WgradPatch b, unsigned grid_a)
{
    if (blockIdx.x < grid_a) {
        if (threadIdx.x >= (unsigned)T::THREADS) return;
        conv_patch_body<T, NS, true>(a, blockIdx.x);
    } else {
        conv_wgrad_patch_body<WM, WC, kGeo, true>(b, blockIdx.x - grid_a);
    }
}

// ------------------------------------------------------------------------------------ helpers

// out[i] = sum_s partial[s][i], s ascending; plus bias[channel of i] when a bias is given
// (channel = (i / inner) % C for an [N, C, inner] output).
// kS > 0: exactly kS splits, all loads issued before the first add.  kLoose: the result's n values are no whole quads, or not on
// the 16-byte grid.
template <int kS, bool kLoose = false>
__global__ __launch_bounds__(256) void splitk_reduce_k(size_t n4, int splits, const float4 *partial, float4 *out,
                                                        const float *bias, unsigned C, unsigned inner, size_t n = 0)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) {
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (kS > 0) {
            float4 v[kS];
#pragma unroll
            for (int s = 0; s < kS; s++) v[s] = partial[(size_t)s * n4 + i];
            acc = v[0];
#pragma unroll
            for (int s = 1; s < kS; s++) {
                acc.x += v[s].x;
                acc.y += v[s].y;
                acc.z += v[s].z;
                acc.w += v[s].w;
            }
        } else {
            // Rounds of four loads in flight (indices clamped to the last split, surplus values
            // dropped); the adds stay in ascending split order.
            const int last = splits - 1;
            for (int s = 0; s < splits; s += 4) {
                const float4 v0 = partial[(size_t)s * n4 + i];
                const float4 v1 = partial[(size_t)min(s + 1, last) * n4 + i];
                const float4 v2 = partial[(size_t)min(s + 2, last) * n4 + i];
                const float4 v3 = partial[(size_t)min(s + 3, last) * n4 + i];
                const bool h1 = s + 1 <= last, h2 = s + 2 <= last, h3 = s + 3 <= last;
                if (s == 0) acc = v0;   // not 0 + v0: the sum of negative zeros stays a negative zero
                else acc = make_float4(acc.x + v0.x, acc.y + v0.y, acc.z + v0.z, acc.w + v0.w);
                if (h1) acc = make_float4(acc.x + v1.x, acc.y + v1.y, acc.z + v1.z, acc.w + v1.w);
                if (h2) acc = make_float4(acc.x + v2.x, acc.y + v2.y, acc.z + v2.z, acc.w + v2.w);
                if (h3) acc = make_float4(acc.x + v3.x, acc.y + v3.y, acc.z + v3.z, acc.w + v3.w);
            }
        }
        if (bias) {
            const size_t e = i * 4;
            acc.x += bias[(e / inner) % C];
            acc.y += bias[((e + 1) / inner) % C];
            acc.z += bias[((e + 2) / inner) % C];
            acc.w += bias[((e + 3) / inner) % C];
        }
        if constexpr (kLoose) store_loose((float *)out, n, i, acc);
        else out[i] = acc;
    }
}

// The same for the general kernels, whose reductions are cut into up to sixty-four parts: added in float64 and rounded once (one fp32
// rounding per part was most of the error: 66 -> 13 channels, 3 x 3, one image of 23 x 7, 1.3e-7 off float64, so 3.8e-8, in one
// part 7e-8; the time is that of the copies' bytes).  kLoose: the result's n values are no whole quads, or not on the 16-byte grid.
template <bool kLoose>
__global__ __launch_bounds__(256) void splitk_exact_k(size_t n4, int splits, const float4 *partial, float4 *out, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) {
        double x = 0, y = 0, z = 0, w = 0;
        const int last = splits - 1;
        for (int s = 0; s < splits; s += 8) {   // eight loads in flight (indices clamped to the last part, surplus values dropped)
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = partial[(size_t)min(s + u, last) * n4 + i];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                if (s + u > last) continue;
                if (s + u == 0) {   // not 0 + v: the sum of negative zeros stays a negative zero
                    x = v[0].x, y = v[0].y, z = v[0].z, w = v[0].w;
                } else {
                    x += v[u].x, y += v[u].y, z += v[u].z, w += v[u].w;
                }
            }
        }
        const float4 sum = make_float4((float)x, (float)y, (float)z, (float)w);
        if constexpr (kLoose) store_loose((float *)out, n, i, sum);
        else out[i] = sum;
    }
}

// The general kernels' packed filters (GatherConv::wp) from w[K][C][R][S]: of the whole filter (one class with R2 = R, S2 = S, no
// stride) or of the sub-filters that the residue classes of a strided backward-data pass multiply.  Forward: rows = K, reduction
// over C; backward: rows = C, reduction over K.  Rows up to Mp and channels up to a multiple of 16 are written, zeros where the
// filter has none.  A block takes 16 rows and 8 channels: they are contiguous runs in w (forward a run per row, backward one per
// channel), staged through LDS; then a thread splits eight values of one row and tap and writes a 16-byte piece per part.
struct SubFilter {
    float *wp;            // packed copy of this class
    int R2, S2, r0, s0;   // tap rows / columns of the class and its first tap offsets
};
struct SubFilters {
    SubFilter f[kGatherJobs];
    int n;
};
template <bool kBwd>
__global__ __launch_bounds__(256) void pack_gather_k(int M, int Cred, int Mp, int R, int S, int sH, int sW, size_t sm, size_t sc,
                                                      const float *w, SubFilters subs, unsigned begin)
{
    extern __shared__ float stage[];
    const unsigned mblocks = (unsigned)(Mp + 15) / 16;
    const unsigned block = begin + blockIdx.x;
    const int RS = R * S, m0 = (int)(block % mblocks) * 16, c0 = (int)(block / mblocks) * 8;
    const int len = (kBwd ? 16 : 8) * RS, pitch = len + 1;   // of a run; backward: channel c0 + run, rows m0 ..; forward: row m0 + run, channels c0 ..
    for (int i = threadIdx.x; i < (kBwd ? 8 : 16) * len; i += 256) {
        const int run = i / len, r = i - run * len;
        const int m = m0 + (kBwd ? r / RS : run), c = c0 + (kBwd ? run : r / RS);
        stage[run * pitch + r] = m < M && c < Cred ? w[(size_t)m * sm + (size_t)c * sc + r % RS] : 0.0f;
    }
    __syncthreads();
    for (int j = 0; j < subs.n; j++) {
        const SubFilter f = subs.f[j];
        for (int i = threadIdx.x; i < 16 * f.R2 * f.S2; i += 256) {
            const int t = i / 16, ml = i % 16, tr = t / f.S2, ts = t - tr * f.S2;
            // stored tap (tr, ts) stands for offsets r = r0 + (R2 - 1 - tr) * sH, s likewise, and the element
            // that multiplies offset (r, s) is the flipped one (see subfilter_k)
            const int r = f.r0 + (f.R2 - 1 - tr) * sH, s = f.s0 + (f.S2 - 1 - ts) * sW;
            const float *const src = stage + (kBwd ? ml * RS : ml * pitch) + (R - 1 - r) * S + (S - 1 - s);
            unsigned q[3][4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int step = kBwd ? pitch : RS;
                split_packed(src[2 * e * step], src[(2 * e + 1) * step], q[0][e], q[1][e], q[2][e]);
            }
            const int m = m0 + ml;
            if (m >= Mp) continue;
            v4u *const dst = (v4u *)f.wp + ((size_t)(c0 / 16 * (f.R2 * f.S2) + t) * Mp + m / 4 * 4) * 6 + c0 / 8 % 2 * 4 + m % 4;
#pragma unroll
            for (int part = 0; part < 3; part++) dst[part * 8] = v4u{q[part][0], q[part][1], q[part][2], q[part][3]};
        }
    }
}

int launch_pack_gather(bool bwd, int K, int C, int R, int S, int sH, int sW, int Mp, const float *w, const SubFilters &subs)
{
    const int M = bwd ? C : K, Cred = bwd ? K : C, chunks = (Cred + BK - 1) / BK, RS = R * S;
    const size_t sm = bwd ? (size_t)RS : (size_t)C * RS, sc = bwd ? (size_t)C * RS : (size_t)RS;
    const size_t blocks = (size_t)((Mp + 15) / 16) * (size_t)(2 * chunks);   // (filters have less than 2^29 values: below 2^27)
    const size_t lds = (bwd ? (size_t)8 * (16 * RS + 1) : (size_t)16 * (8 * RS + 1)) * sizeof(float);   // at most 33 KB: 64 taps
    for (size_t begin = 0; begin < blocks; begin += kLaunchBlocks) {
        const dim3 grid((unsigned)std::min(blocks - begin, kLaunchBlocks));
        if (bwd) hipLaunchKernelGGL(pack_gather_k<true>, grid, dim3(256), lds, stream(), M, Cred, Mp, R, S, sH, sW, sm, sc, w, subs, (unsigned)begin);
        else hipLaunchKernelGGL(pack_gather_k<false>, grid, dim3(256), lds, stream(), M, Cred, Mp, R, S, sH, sW, sm, sc, w, subs, (unsigned)begin);
        DOPT_LAUNCH_CHECK();
    }
    return DOPT_HIP_OK;
}

int round_up(int v, int to) { return (v + to - 1) / to * to; }

// DOPT_HIP_NO_TALL=1 keeps the 160-row tiles out (for A/B measurements); read once.
bool no_tall_tiles()
{
    static const bool off = std::getenv("DOPT_HIP_NO_TALL") != nullptr;
    return off;
}

int check_desc(const dopt_hip_conv_desc *d, size_t *P, size_t *Q, const char *who)
{
    DOPT_REQUIRE(d != nullptr, "%s: descriptor is null", who);
    DOPT_REQUIRE(d->strideH > 0 && d->strideW > 0, "%s: stride must be positive", who);
    DOPT_REQUIRE(d->N && d->C && d->H && d->W && d->K && d->R && d->S, "%s: empty tensor", who);
    DOPT_REQUIRE(d->H + 2 * d->padH >= d->R && d->W + 2 * d->padW >= d->S, "%s: filter larger than padded input", who);
    DOPT_REQUIRE(d->R * d->S <= 64, "%s: filters above 64 taps are not supported", who);
    *P = (d->H + 2 * d->padH - d->R) / d->strideH + 1;  // core/ops/nnet.d:71-87
    *Q = (d->W + 2 * d->padW - d->S) / d->strideW + 1;
    const size_t lim = (size_t)1 << 29;  // byte offsets of valid elements stay below 2^31
    DOPT_REQUIRE(d->N * d->C * d->H * d->W < lim && d->N * d->K * *P * *Q < lim && d->K * d->C * d->R * d->S < lim,
                 "%s: tensors of 2^29 elements or more are not supported", who);
    return DOPT_HIP_OK;
}

// Floats from one partial copy of a general kernel's result, or of a filter gradient, to the next.
size_t copy_stride(size_t elems) { return (elems + 3) / 4 * 4; }

int launch_splitk_exact(size_t elems, int splits, const float *partial, float *out)
{
    const size_t n4 = copy_stride(elems) / 4;
    const dim3 grid((unsigned)std::min(ceil_div(n4, (size_t)256), (size_t)num_cus() * 8));
    if (elems % 4 != 0 || !aligned16(out))
        hipLaunchKernelGGL(splitk_exact_k<true>, grid, dim3(256), 0, stream(), n4, splits, (const float4 *)partial, (float4 *)out, elems);
    else
        hipLaunchKernelGGL(splitk_exact_k<false>, grid, dim3(256), 0, stream(), n4, splits, (const float4 *)partial, (float4 *)out, elems);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

int launch_splitk_reduce(size_t elems, int splits, const float *partial, float *out, const float *bias = nullptr,
                         unsigned C = 1, unsigned inner = 1)
{
    // float4 passes: the partial copies are whole quads (copy_stride) and start on 256-byte boundaries of the workspace
    const size_t n4 = copy_stride(elems) / 4;
    size_t blocks = ceil_div(n4, (size_t)256);
    size_t cap = (size_t)num_cus() * 8;
    const dim3 grid((unsigned)(blocks > cap ? cap : (blocks < 1 ? 1 : blocks)));
    const float4 *p4 = (const float4 *)partial;
    float4 *o4 = (float4 *)out;
    if (elems % 4 != 0 || !aligned16(out)) {   // (the same order)
        hipLaunchKernelGGL((splitk_reduce_k<0, true>), grid, dim3(256), 0, stream(), n4, splits, p4, o4, bias, C, inner, elems);
        DOPT_LAUNCH_CHECK();
        return DOPT_HIP_OK;
    }
    switch (splits) {
    case 2: hipLaunchKernelGGL(splitk_reduce_k<2>, grid, dim3(256), 0, stream(), n4, splits, p4, o4, bias, C, inner, elems); break;
    case 3: hipLaunchKernelGGL(splitk_reduce_k<3>, grid, dim3(256), 0, stream(), n4, splits, p4, o4, bias, C, inner, elems); break;
    case 4: hipLaunchKernelGGL(splitk_reduce_k<4>, grid, dim3(256), 0, stream(), n4, splits, p4, o4, bias, C, inner, elems); break;
    default: hipLaunchKernelGGL(splitk_reduce_k<0>, grid, dim3(256), 0, stream(), n4, splits, p4, o4, bias, C, inner, elems); break;
    }
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

// Eight wavefronts of 32 x 64, one workgroup per CU.  (Four of 64 x 64, two workgroups per CU, hid their loads as well but had
// twice the values to split per wavefront: 5 x 5 layers backward-data 104 against 101 us before the splitting was overlapped.)
// Up to 32 output channels: 64 rows would multiply as many zeros (3 x 3, 108 images of 16 x 57, 11 -> 16 channels: 27 -> 21 us; 418 -> 28, 222
// of 10 x 35, 174 -> 142).
using GatherNarrow = Tile<32, 256, 1, 8>;
using GatherWide = Tile<64, 256, 2, 4>;     // few output channels, many pixels
using GatherSquare = Tile<128, 128, 4, 2>;

unsigned div_magic(unsigned d) { return (unsigned)((((unsigned long long)1 << 32) / d) + 1); }

// Tiles of the direct 3 x 3 kernel.
using PatchNarrow = Tile<32, 256, 1, 4>;    // up to 32 output channels: 64 rows would multiply as many zeros
using PatchWide = Tile<64, 256, 2, 4>;
using PatchDeep = Tile<128, 128, 4, 2>;
using PatchTall = Tile<160, 128, 5, 2>;     // 160 output channels (and 480, ...)

template <class T, int NS>
int launch_patch(const PatchConv &pc, bool c_full, dim3 grid, size_t lds_bytes)
{
    // above 64 KB of dynamic LDS a kernel has to be told once
    static bool raised[2] = {false, false};
    if (!raised[c_full]) {
        const void *fn = c_full ? (const void *)conv_patch_k<T, NS, true> : (const void *)conv_patch_k<T, NS, false>;
        DOPT_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        raised[c_full] = true;
    }
    if (c_full) hipLaunchKernelGGL((conv_patch_k<T, NS, true>), grid, dim3(T::THREADS), lds_bytes, stream(), pc);
    else hipLaunchKernelGGL((conv_patch_k<T, NS, false>), grid, dim3(T::THREADS), lds_bytes, stream(), pc);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

// 3x3 unit-stride layers whose pixel tiles are whole rows of one image or whole images.
// Returns DOPT_HIP_OK with *done = false when the layer does not fit this path.
// What the patch kernel needs to know about one convolution, without any pointer: which tile
// shape runs it and how its filter is packed.  `ok` is false when the generic kernel takes the shape.
struct PatchSetup {
    bool ok;
    PatchConv pc;
    int shape;            // 0 wide, 1 narrow, 2 deep, 3 tall, 4 Winograd (BM 128: 128 rows x 32 tiles of 2x2 pixels, BM 64: 64 rows x 64 tiles)
    int BM, BN, blocks_wanted, tiles;
    int positions;        // of a patch, at most (the load slots of some tiles hold more: wider patches are the general kernels')
    size_t lds_bytes, wp_elems;
};

template <bool kBwd>
PatchSetup patch_setup_as(const dopt_hip_conv_desc *d, size_t P, size_t Q, bool allow_tall, int wino = 0);   // wino: rows of a Winograd tile, 0 none

// DOPT_HIP_NO_WINO=1 keeps the Winograd kernel out (for A/B measurements); read once.
bool no_wino()
{
    static const bool off = std::getenv("DOPT_HIP_NO_WINO") != nullptr;
    return off;
}

// (a layer the 160-row tiles do not take - its pixel tile does not fit their patch - is tried with the other heights)
template <bool kBwd>
PatchSetup patch_setup(const dopt_hip_conv_desc *d, size_t P, size_t Q)
{
    if (!no_wino()) {
        // 128-row tiles first: measured faster than 64-row tiles on every layer that has both (they read the input once
        // per 128 rows and transform it once)
        const PatchSetup v = patch_setup_as<kBwd>(d, P, Q, false, 128);
        if (v.ok) return v;
        const PatchSetup v2 = patch_setup_as<kBwd>(d, P, Q, false, 64);
        if (v2.ok) return v2;
    }
    const PatchSetup u = patch_setup_as<kBwd>(d, P, Q, true);
    return u.ok ? u : patch_setup_as<kBwd>(d, P, Q, false);
}

template <bool kBwd>
PatchSetup patch_setup_as(const dopt_hip_conv_desc *d, size_t P, size_t Q, bool allow_tall, int wino)
{
    PatchSetup u{};
    if (d->R != 3 || d->S != 3 || d->strideH != 1 || d->strideW != 1 || d->padH > 2 || d->padW > 2) return u;
    PatchConv &pc = u.pc;
    pc.N = (int)d->N;
    if (!kBwd) {
        pc.Cin = (int)d->C; pc.IH = (int)d->H; pc.IW = (int)d->W;
        pc.Mout = (int)d->K; pc.OH = (int)P; pc.OW = (int)Q;
        pc.PT = (int)d->padH; pc.PL = (int)d->padW; pc.flip = 1;
    } else {
        pc.Cin = (int)d->K; pc.IH = (int)P; pc.IW = (int)Q;
        pc.Mout = (int)d->C; pc.OH = (int)d->H; pc.OW = (int)d->W;
        pc.PT = 2 - (int)d->padH; pc.PL = 2 - (int)d->padW; pc.flip = 0;
    }
    pc.ncols = pc.N * pc.OH * pc.OW;
    // 160-row tiles where they pad no more than both other heights (160 channels: 160 rows, not 192 or 256; 320 and 640
    // channels: two and four such tiles - on 8 x 8 images 640 channels are then exactly 256 tiles, one per compute unit
    // with no split of the reduction, where 128-row tiles gave 320 and a four-way split); 64-row tiles for up to 64 output
    // channels, and wherever 128-row tiles would pad more
    const int up64 = (pc.Mout + 63) / 64 * 64, up128 = (pc.Mout + 127) / 128 * 128, up160 = (pc.Mout + 159) / 160 * 160;
    // (only where they still give every compute unit a tile: 480 channels on 8 x 8 images are 192 such tiles, and ran slower)
    const long tall_tiles = (long)(up160 / 160) * ((pc.ncols + 127) / 128);
    if (wino) {
        // whole 16-channel chunks of a deep reduction, pad 1, 2 x 2 tiles
        if (d->padH != 1 || d->padW != 1 || pc.Cin % 16 != 0 || pc.Cin < 64 || pc.OH % 2 != 0 || pc.OW % 2 != 0 || pc.OH < 4 ||
            pc.OW < 4)
            return u;
        // whole tiles of rows, or 64-row tiles padded by no more than a fifth (160 rows as 192: still 1.9 times fewer
        // matrix instructions than the direct kernels execute)
        if (pc.Mout % wino != 0 && !(wino == 64 && pc.Mout > 64 && up64 * 5 <= pc.Mout * 6)) return u;
        // whole 128-row tiles of 32 tiles (128 pixels), or whole 64-row tiles of 64 tiles (256 pixels)
        u.shape = 4; u.BM = wino; u.BN = u.BM == 128 ? 128 : 256;
        u.blocks_wanted = num_cus(); u.positions = 512;
    } else if (allow_tall && pc.Mout > 64 && up160 <= up64 && up160 <= up128 && tall_tiles >= num_cus() &&
        !no_tall_tiles()) {
        u.shape = 3; u.BM = 160; u.BN = 128; u.blocks_wanted = num_cus(); u.positions = 256;
    } else if (pc.Mout <= 32) {   // (16 -> 16 channels on 32 x 32 images, batch 64: 18 us with 64 rows in fp32, 10 us)
        u.shape = 1; u.BM = 32; u.BN = 256; u.blocks_wanted = 2 * num_cus(); u.positions = 384;
    } else if (pc.Mout <= 64 || up64 < up128) {
        u.shape = 0; u.BM = 64; u.BN = 256; u.blocks_wanted = num_cus(); u.positions = 384;
    } else {
        u.shape = 2; u.BM = 128; u.BN = 128; u.blocks_wanted = num_cus(); u.positions = 512;
    }
    const int BM = u.BM, BN = u.BN;
    // pixel tile = `rows` full rows of one image, or `nimg` whole images
    if (BN % pc.OW != 0) return u;
    const int tile_rows = BN / pc.OW;
    if (tile_rows <= pc.OH) {
        if (pc.OH % tile_rows != 0) return u;
        pc.nimg = 1; pc.rows = tile_rows;
    } else {
        if (tile_rows % pc.OH != 0) return u;
        pc.nimg = tile_rows / pc.OH; pc.rows = pc.OH;
    }
    pc.PR = pc.rows + 2; pc.PC = pc.OW + 2;
    pc.psz = pc.nimg * pc.PR * pc.PC;
    if (pc.psz > u.positions) return u;
    u.lds_bytes = (size_t)2 * (pc.psz + 1) * 24 * sizeof(float);
    if (wino) {
        if (pc.rows % 2 != 0) return u;   // a pixel tile is whole 2 x 2 tiles
        pc.magic_tpi = div_magic((unsigned)(pc.rows / 2 * (pc.OW / 2)));
        pc.magic_tcn = div_magic((unsigned)(pc.OW / 2));
        const size_t buffers = u.BM == 128 ? 2 : 1;   // 32 tiles: raw patch and V are double-buffered
        const size_t floats = buffers * ((size_t)(((pc.psz + 1) * 20 + 3) / 4 * 4) + (size_t)16 * (u.BN / 4) * 24);
        u.lds_bytes = std::max(floats, (size_t)wino_xchg(u.BM) + 8) * sizeof(float);
    }
    if (u.lds_bytes > 160 * 1024) return u;
    pc.magic_img = div_magic((unsigned)(pc.PR * pc.PC));
    pc.magic_pc = div_magic((unsigned)pc.PC);
    pc.mtiles = (pc.Mout + BM - 1) / BM;
    pc.ntiles = (pc.ncols + BN - 1) / BN;
    pc.Mp = pc.mtiles * BM;
    pc.chunks_total = (pc.Cin + 15) / 16;
    pc.out_elems = (size_t)pc.ncols * pc.Mout;
    u.tiles = pc.mtiles * pc.ntiles;
    u.wp_elems = (size_t)pc.chunks_total * (wino ? 16 : 9) * 24 * pc.Mp;   // three 16-bit parts a value
    // (few rows of very many channels, from 2 GiB at four bytes a value and 64 rows on, stay the general kernels', as they were
    // when the copy was one of fp32 values and reached by 32-bit offsets; not measured against the direct kernel since)
    if (!wino && (size_t)pc.chunks_total * 9 * 64 * std::max(pc.Mp, 64) > 0x7fffffffu) return u;
    u.ok = true;
    return u;
}

template <bool kBwd>
PackJob pack_job(const dopt_hip_conv_desc *d, const PatchSetup &u, const float *w, float *wp)
{
    const unsigned C9 = (unsigned)(d->C * 9);
    PackJob j{};
    j.w = w; j.wp = wp;
    j.M = u.pc.Mout; j.Cred = u.pc.Cin; j.Mp = u.pc.Mp; j.bwd = kBwd;
    j.wino = u.shape == 4; j.flip = u.pc.flip;
    j.sm = kBwd ? 9u : C9;
    j.sc = kBwd ? C9 : 9u;
    j.mblocks = (unsigned)(u.pc.Mp / 16);
    return j;
}

// How many ways to split the channel chunks of a patch convolution over blocks.  `slots` blocks run
// at once (one or two per CU); the blocks of a launch run in ceil(blocks / slots) rounds and a round
// lasts as long as one block, so 320 tiles on 256 slots cost two full rounds - unless the reduction
// is split four ways, which makes 1280 quarter-length blocks in exactly five rounds.  The estimate,
// in microseconds: rounds x (chunks per block x time per chunk + a fixed prologue/epilogue) plus,
// when split, writing and re-reading the partial tiles.  The split with the lowest estimate wins;
// ties go to the smaller one.
int patch_splits(int tiles, int chunks, int slots, int BM, int BN, size_t out_elems, bool wino)
{
    // what one CU sustains in these main loops (direct: 0.47 in fp32.  With 0.47 here, and 0.33 in place of kGatherRate, the half-width
    // VGG-16 step is 0.4 % and that of Wide-ResNet-10-2 2.4 % longer, Wide-ResNet-28-10's and the 5 x 5 layers' the same)
    const double cu_tflops = wino ? 0.47 : 0.8;
    const double per_cu = (double)slots / num_cus();                 // blocks sharing a CU
    // 16 channels x 9 taps.  The Winograd kernel takes a third of that for a chunk, but adds all six parts of a product in one
    // accumulator: with its own time here it would be cut less and be further off than the fp32 instruction, which was cut by
    // this estimate (320 channels on 16 x 16 images, error against float64: fp32 2.9e-7, uncut 4.2e-7, cut in two 2.5e-7; batch
    // 128 216 and 219 us; 160 on 32 x 32 2.5e-7, 2.9e-7, 2.1e-7, and the same time).
    const double t_chunk = 2.0 * BM * BN * 144 / (cu_tflops * 1e6 / per_cu);
    int best = 1;
    double best_cost = 0.0;
    for (int sp = 1; sp <= chunks && sp <= 64; sp++) {
        const int per_block = (chunks + sp - 1) / sp;
        if (sp > 1 && (chunks + per_block - 1) / per_block != sp) continue;   // would leave an empty split
        const double rounds = (double)(((long long)tiles * sp + slots - 1) / slots);
        double cost = rounds * (per_block * t_chunk + 6.0);
        if (sp > 1) cost += 3.0 + (sp + 1.0) * out_elems * 4.0 / 4.5e6;       // partial tiles at ~4.5 TB/s
        if (sp == 1 || cost < best_cost * 0.97) {                    // a larger split must pay for itself clearly
            best = sp;
            best_cost = cost;
        }
    }
    return best;
}

// The same estimate for the general kernels, whose unit is a slab of 16 reduction steps, at the rate that one CU sustains (0.33 on the
// fp32 instruction; measured above).
constexpr double kGatherRate = 0.6;
// sum_us: what the launch that adds the parts takes beside their bytes, where there would be none without a cut.
int gather_splits(int tiles, int slabs, int slots, int BM, int BN, size_t out_elems, double cu_tflops, int cap, double sum_us)
{
    const double per_cu = (double)slots / num_cus();
    const double t_slab = 2.0 * BM * BN * 16 / (cu_tflops * 1e6 / per_cu);
    int best = 1;
    double best_cost = 0.0;
    for (int sp = 1; sp <= slabs && sp <= cap; sp++) {
        const int per_block = (slabs + sp - 1) / sp;
        if (sp > 1 && (slabs + per_block - 1) / per_block != sp) continue;
        const double rounds = (double)(((long long)tiles * sp + slots - 1) / slots);
        double cost = rounds * (per_block * t_slab + 6.0);
        if (sp > 1) cost += sum_us + (sp + 1.0) * out_elems * 4.0 / 4.5e6;
        if (sp == 1 || cost < best_cost * 0.97) {
            best = sp;
            best_cost = cost;
        }
    }
    return best;
}

// Fills in how a patch convolution splits its channel chunks over blocks; returns the number of splits.
int patch_decide_splits(PatchSetup *u, const float *out)
{
    PatchConv &pc = u->pc;
    int splits = patch_splits(u->tiles, pc.chunks_total, u->blocks_wanted, u->BM, u->BN, pc.out_elems, u->shape == 4);
    if (pc.out_elems % 4 != 0 || !aligned16(out)) splits = 1;
    pc.chunks_per_split = (pc.chunks_total + splits - 1) / splits;
    splits = (pc.chunks_total + pc.chunks_per_split - 1) / pc.chunks_per_split;
    pc.splits = splits;
    return splits;
}

// `prepacked`: the filter already in the kernel's layout (dopt_hip_conv_pack_batch), or null to
// pack it here first.
// Device time of one kernel family alone (an entry point may also run split sums and packing): while the probe is on,
// every launch of the family - 1: the one-launch backward pairs (conv_bwd_pair_k), 2: the Winograd kernel
// (conv_wino_k) - is bracketed by two events on the stream it is launched on.
struct PairProbe {
    int on = 0;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> events;   // kept for the process's lifetime, reused
    size_t used = 0;
    double flops = 0.0, bytes = 0.0;
};
PairProbe g_pair_probe;

int probe_begin(PairProbe &probe)
{
    if (probe.used == probe.events.size()) {
        hipEvent_t e0, e1;
        DOPT_HIP_CHECK(hipEventCreate(&e0));
        DOPT_HIP_CHECK(hipEventCreate(&e1));
        probe.events.push_back({e0, e1});
    }
    DOPT_HIP_CHECK(hipEventRecord(probe.events[probe.used].first, stream()));
    return DOPT_HIP_OK;
}

// The launch of a filled-in patch setup: the tile shape picks the instance.
int dispatch_patch(const PatchSetup &u, int splits)
{
    const PatchConv &pc = u.pc;
    const dim3 grid(xcd_grid((unsigned)(u.tiles * splits)));
    const bool c_full = pc.Cin % 16 == 0;
    if (u.shape == 0) return launch_patch<PatchWide, 2>(pc, c_full, grid, u.lds_bytes);
    if (u.shape == 3) return launch_patch<PatchTall, 2>(pc, c_full, grid, u.lds_bytes);
    if (u.shape == 1) return launch_patch<PatchNarrow, 3>(pc, c_full, grid, u.lds_bytes);
    if (u.shape == 4) {
        static bool raised = false;
        if (!raised) {
            DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)conv_wino_k<16, 4, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
            DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)conv_wino_k<16, 2, 2>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
            raised = true;
        }
        PairProbe &probe = g_pair_probe;
        const bool probing = probe.on == 2 && u.BM == 128 && !capturing();   // the 128-row instantiation only: one kernel, one average
        if (probing)
            if (int rc = probe_begin(probe)) return rc;
        if (u.BM == 128) hipLaunchKernelGGL((conv_wino_k<16, 4, 1>), grid, dim3(512), u.lds_bytes, stream(), pc);
        else hipLaunchKernelGGL((conv_wino_k<16, 2, 2>), grid, dim3(512), u.lds_bytes, stream(), pc);
        DOPT_LAUNCH_CHECK();
        if (probing) {
            DOPT_HIP_CHECK(hipEventRecord(probe.events[probe.used++].second, stream()));
            // the direct algorithm's count (what the layer is, whatever the kernel multiplies): 2 N K C 9 P Q
            probe.flops += 2.0 * (double)pc.ncols * pc.Mout * pc.Cin * 9.0;
            probe.bytes += 4.0 * ((double)pc.N * pc.Cin * pc.IH * pc.IW + (double)pc.ncols * pc.Mout + (double)pc.Mout * pc.Cin * 9.0);
        }
        return DOPT_HIP_OK;
    }
    return launch_patch<PatchDeep, 2>(pc, c_full, grid, u.lds_bytes);
}

template <bool kBwd>
int run_patch(const dopt_hip_conv_desc *d, size_t P, size_t Q, const float *in, const float *w, const float *bias,
              float *out, bool *done, const float *prepacked = nullptr, dopt_hip_split_sum *open = nullptr)
{
    *done = false;
    PatchSetup u = patch_setup<kBwd>(d, P, Q);
    if (!u.ok) return DOPT_HIP_OK;
    PatchConv &pc = u.pc;
    const int splits = patch_decide_splits(&u, out);

    const size_t wp_bytes = prepacked ? 0 : (u.wp_elems * sizeof(float) + 255) / 256 * 256;
    const size_t part_bytes = splits > 1 ? (size_t)splits * pc.out_elems * sizeof(float) : 0;
    char *ws = wp_bytes + part_bytes > 0 ? (char *)workspace(wp_bytes + part_bytes) : nullptr;
    if (wp_bytes + part_bytes > 0 && !ws) return DOPT_HIP_ERR_OOM;
    float *partial = (float *)(ws + wp_bytes);
    if (!prepacked) {
        const PackJob j = pack_job<kBwd>(d, u, w, (float *)ws);
        const dim3 pgrid(j.mblocks, (unsigned)pc.chunks_total);
        if (!kBwd) hipLaunchKernelGGL(pack_patch_k<false>, pgrid, dim3(256), 0, stream(), j.M, j.Cred, j.Mp, (size_t)j.sm,
                                      (size_t)j.sc, j.wino, j.flip, w, j.wp);
        else hipLaunchKernelGGL(pack_patch_k<true>, pgrid, dim3(256), 0, stream(), j.M, j.Cred, j.Mp, (size_t)j.sm,
                                (size_t)j.sc, j.wino, j.flip, w, j.wp);
        DOPT_LAUNCH_CHECK();
        prepacked = j.wp;
    }
    pc.in = in;
    pc.wp = prepacked;
    pc.bias = bias;
    pc.in_bytes = (size_t)pc.N * pc.Cin * pc.IH * pc.IW * sizeof(float);
    pc.out = splits > 1 ? partial : out;
    if (int rc = dispatch_patch(u, splits)) return rc;
    *done = true;
    if (splits > 1 && open) {   // the caller's next call adds the copies
        open->partial = partial;
        open->splits = splits;
        open->elems = pc.out_elems;
        open->C = (size_t)pc.Mout;
        open->inner = (size_t)pc.OH * pc.OW;
        open->bias = bias;
        open->value = out;
        open_split_set(partial);
        return DOPT_HIP_OK;
    }
    if (splits > 1)
        return launch_splitk_reduce(pc.out_elems, splits, partial, out, bias, (unsigned)pc.Mout, (unsigned)(pc.OH * pc.OW));
    return DOPT_HIP_OK;
}

// ---- 2 x 2 images -------------------------------------------------------------------------------
// On a 2 x 2 image with pad 1 every output pixel sees every input pixel, each through exactly one
// tap, and the five taps that fall on padding contribute nothing.  The convolution is then a plain
// product of the batch, flattened [N, C*4], with a [C*4, K*4] matrix built from the filter:
//     Wd[(c, iy, ix)][(k, oy, ox)] = w[k][c][2 - (iy - oy + 1)][2 - (ix - ox + 1)]
// (the flipped filter, core/source/dopt/core/ops/nnet.d:270-293) - 4/9 of the multiplications of
// the nine-tap form.  NCHW needs no rearranging on either side, forward is x * Wd and backward-data
// is dy * Wd^T, so one copy of Wd serves both directions.
__global__ __launch_bounds__(256) void pack_2x2_k(unsigned C, unsigned K, const float *w, float4 *wd)
{
    // A block takes 8 output channels x 64 input channels.  It reads their filter planes as eight
    // contiguous runs of 64 x 9 floats, and after a pass through LDS writes, for each of the 256
    // (input channel, input pixel) rows, the eight quads of its output channels: one full 128-byte line.
    __shared__ float stage[8][64 * 9 + 1];
    const unsigned k0 = blockIdx.x * 8, c0 = blockIdx.y * 64;
    const unsigned nk = min(8u, K - k0), nc = min(64u, C - c0);
    float v[18];   // 8 * 64 * 9 / 256 loads per thread, all issued before the first is used (clamped, not branched)
#pragma unroll
    for (int u = 0; u < 18; u++) {
        const unsigned i = threadIdx.x + 256 * u, kk = i / (64 * 9), r = i - kk * (64 * 9);
        v[u] = w[((size_t)(k0 + min(kk, nk - 1)) * C + c0) * 9 + min(r, nc * 9 - 1)];
    }
#pragma unroll
    for (int u = 0; u < 18; u++) {
        const unsigned i = threadIdx.x + 256 * u, kk = i / (64 * 9), r = i - kk * (64 * 9);
        stage[kk][r] = v[u];   // rows and channels past the end are never read back
    }
    __syncthreads();
    for (unsigned i = threadIdx.x; i < 64 * 4 * 8; i += 256) {
        const unsigned kk = i & 7, row = i >> 3, cc = row >> 2, iy = (row >> 1) & 1, ix = row & 1;
        if (kk >= nk || cc >= nc) continue;
        // input pixel (iy, ix), output pixel (oy, ox): tap (1 - iy + oy, 1 - ix + ox)
        const float *f = &stage[kk][cc * 9 + (1 - iy) * 3 + (1 - ix)];
        wd[((size_t)(c0 + cc) * 4 + iy * 2 + ix) * K + k0 + kk] = make_float4(f[0], f[1], f[3], f[4]);
    }
}

bool dense2x2_takes(const dopt_hip_conv_desc *d)
{
    return d->R == 3 && d->S == 3 && d->strideH == 1 && d->strideW == 1 && d->padH == 1 && d->padW == 1 && d->H == 2 &&
           d->W == 2 && d->C * 4 < ((size_t)1 << 30) && d->K * 4 < ((size_t)1 << 30);
}

size_t dense2x2_elems(const dopt_hip_conv_desc *d) { return (size_t)16 * d->C * d->K; }

int dense2x2_pack(const dopt_hip_conv_desc *d, const float *w, float *wd)
{
    hipLaunchKernelGGL(pack_2x2_k, dim3((unsigned)ceil_div(d->K, (size_t)8), (unsigned)ceil_div(d->C, (size_t)64)), dim3(256), 0,
                       stream(), (unsigned)d->C, (unsigned)d->K, w, (float4 *)wd);   // pool and plan buffers are 256-byte aligned
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

// `wd`: the matrix already built, or null to build it from `w` in the workspace first
template <bool kBwd>
int run_dense2x2(const dopt_hip_conv_desc *d, const float *in, const float *w, const float *wd, const float *bias,
                 float *out)
{
    void *mine = nullptr;   // from the pool, not the workspace: the product below may use the workspace itself
    if (!wd) {
        if (int rc = scratch_alloc(&mine, dense2x2_elems(d) * sizeof(float))) return rc;
        if (int rc = dense2x2_pack(d, w, (float *)mine)) {
            dopt_hip_free(mine);
            return rc;
        }
        wd = (const float *)mine;
    }
    bool biased = false;
    int rc;
    if (!kBwd) {
        rc = sgemm_bias(0, 0, d->N, 4 * d->K, 4 * d->C, in, wd, out, bias, 2, &biased);
        if (!rc && bias && !biased) rc = dopt_hip_bias_fwd(d->N, d->K, 4, out, bias, out);
    } else {
        rc = sgemm_bias(0, 1, d->N, 4 * d->C, 4 * d->K, in, wd, out, nullptr, 0, &biased);
    }
    if (mine) dopt_hip_free(mine);   // back to the pool; whoever gets it next queues behind the product
    return rc;
}

// ---- 2 x 2 images, straight from the filter ----------------------------------------------------
// The product above needs the 16 MB matrix made first, and its 32 x 32-output blocks read their operands
// with a handful of loads in flight per wavefront (one cache line per lane and step), which is what
// bounds them.  This kernel keeps that decomposition - a block owns 32 images x 8 output channels x 4
// pixels over the WHOLE reduction, so nothing is split and no partial copies are left for a reader
// (whose 16-byte pieces per image and channel would be re-read once per copy) - but reads the taps from
// the filter as it lies (no Wd) and streams both operands through LDS in bulk:
//   * the eight wavefronts split the reduction channels (64 consecutive channels each, R % 64 == 0) and
//     never share data, so each runs a pipeline of its own with no workgroup barrier: per step of 8
//     channels it loads 32 images x 128 bytes of the batch (whole cache lines) and 8 runs of 8 x 9 taps,
//     three steps ahead, passes them through a wavefront-private LDS tile and multiplies;
//   * a batch row is read back as one 128-bit LDS read per eight reduction steps (lane half h takes
//     steps 8g + 4h .. 8g + 4h + 3 on both operands), the four taps a lane needs per (channel, pixel
//     pair) as four 4-byte reads: tap = {4,3,1,0}[input pixel] + {0,1,3,4}[output pixel] (see Wd above);
//   * the eight partial 32 x 32 tiles are added through LDS in wavefront order (+ bias).
// Forward (kBwd = false): in = x [N][C*4], columns (k, output pixel), a filter run = one output channel's
// 8 reduction channels x 9 taps; backward-data: in = dy [N][K*4], columns (c, input pixel), a run = one
// reduction channel k, its 8 output channels c x 9 taps.
struct Direct2x2 {
    const float *in;    // [N][R*4]
    const float *w;     // [K][C][3][3]
    const float *bias;  // [O] or null (forward)
    float *out;         // [N][O*4]
    int N, R, O, C;     // images, reduction channels, output channels, the filter's input channels (its pitch is C*9)
};

constexpr int kD2Rows = 32, kD2Chans = 8, kD2Step = 8, kD2Waves = 8, kD2Depth = 3;
constexpr int kD2APitch = kD2Step * 4 + 4;   // 36 floats: 128-bit reads of 32 rows touch every bank once
constexpr int kD2WPitch = kD2Step * 9 + 5;   // 77 floats per run of 8 x 9 taps
constexpr int kD2WaveLds = 2 * (kD2Rows * kD2APitch + 8 * kD2WPitch);   // floats per wavefront, double buffered
constexpr size_t kD2Lds = (size_t)kD2Waves * kD2WaveLds * sizeof(float);
static_assert(kD2Waves * kD2WaveLds >= kD2Waves * 32 * 33, "the partial tiles reuse the staging area");

template <bool kBwd>
__global__ __launch_bounds__(64 * kD2Waves) void conv2x2_direct_k(Direct2x2 p)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l32 = lane & 31, kh = lane >> 5;
    const int o0 = blockIdx.x * kD2Chans, n0 = blockIdx.y * kD2Rows;
    const int per_wave = p.R / kD2Waves, steps = per_wave / kD2Step, c_first = w * per_wave;
    float *const mine = lds + w * kD2WaveLds;

    // this lane's pieces of a step: 4 quads of the batch (row = idx / 8, quad idx % 8) and up to 3 of the taps
    // (run = idx / 18, quad idx % 18)
    const float *a_src[4];
    bool a_ok[4];
    int a_dst[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int idx = lane + 64 * i, row = idx >> 3, q = idx & 7;
        a_ok[i] = n0 + row < p.N;
        a_src[i] = p.in + ((size_t)(a_ok[i] ? n0 + row : 0) * p.R + c_first) * 4 + 4 * q;
        a_dst[i] = row * kD2APitch + 4 * q;
    }
    const float *w_src[3];
    bool w_ok[3];
    int w_dst[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const int idx = lane + 64 * i, run = min(idx / 18, 7), q = idx - (idx / 18) * 18;
        w_ok[i] = idx < 8 * 18;
        // forward: run = output channel, its 8 reduction channels of the step; backward: run = reduction channel of the
        // step, the block's 8 output channels
        w_src[i] = kBwd ? p.w + ((size_t)(c_first + run) * p.C + o0) * 9 + 4 * q : p.w + ((size_t)(o0 + run) * p.C + c_first) * 9 + 4 * q;
        w_dst[i] = run * kD2WPitch + 4 * q;
    }
    const size_t w_step = kBwd ? (size_t)kD2Step * p.C * 9 : (size_t)kD2Step * 9;   // floats between steps
    float4 ra[kD2Depth][4], rw[kD2Depth][3];
    auto load = [&](int slot, int s) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            ra[slot][i] = a_ok[i] ? *(const float4 *)(a_src[i] + (size_t)s * kD2Step * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int i = 0; i < 3; i++)
            rw[slot][i] = w_ok[i] ? *(const float4 *)(w_src[i] + (size_t)s * w_step) : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    auto store = [&](int slot, float *buf) {
        float *As = buf, *Ws = buf + kD2Rows * kD2APitch;
#pragma unroll
        for (int i = 0; i < 4; i++) *(float4 *)&As[a_dst[i]] = ra[slot][i];
#pragma unroll
        for (int i = 0; i < 3; i++)
            if (w_ok[i]) {
                float *dst = &Ws[w_dst[i]];
                dst[0] = rw[slot][i].x; dst[1] = rw[slot][i].y; dst[2] = rw[slot][i].z; dst[3] = rw[slot][i].w;
            }
    };

    const int pix = l32 & 3, oc = l32 >> 2;   // the column: output channel inside the block, and its pixel
    const int lane_tap = kBwd ? (pix == 0 ? 4 : pix == 1 ? 3 : pix == 2 ? 1 : 0) : (pix == 0 ? 0 : pix == 1 ? 1 : pix == 2 ? 3 : 4);
    const int a_frag = l32 * kD2APitch + 4 * kh;
    const int b_frag = kD2Rows * kD2APitch + (kBwd ? kh * kD2WPitch + oc * 9 + lane_tap : oc * kD2WPitch + kh * 9 + lane_tap);
    // two accumulators (even and odd channel pairs), so that consecutive matrix instructions do not wait for each other
    v16f acc0, acc1;
#pragma unroll
    for (int v = 0; v < 16; v++) acc0[v] = acc1[v] = 0.0f;

#pragma unroll
    for (int d = 0; d < kD2Depth; d++)
        if (d < steps) load(d, d);
    // steps in groups of kD2Depth so that the register slots are compile-time indices
    for (int s0 = 0; s0 < steps; s0 += kD2Depth) {
#pragma unroll
        for (int d = 0; d < kD2Depth; d++) {
            const int s = s0 + d;
            if (s < steps) {
                float *buf = mine + (s & 1) * (kD2WaveLds / 2);
                store(d, buf);
                __builtin_amdgcn_wave_barrier();   // the tile is read by other lanes of this wavefront: keep the order
                if (s + kD2Depth < steps) load(d, s + kD2Depth);
#pragma unroll
                for (int g = 0; g < 4; g++) {   // reduction steps 8g .. 8g + 7 of the tile: channels 2g (lane half 0), 2g + 1
                    const float4 a = *(const float4 *)(buf + a_frag + 8 * g);
                    const float *src = buf + b_frag + (kBwd ? 2 * g * kD2WPitch : 2 * g * 9);
                    float b0, b1, b2, b3;
                    if (kBwd) { b0 = src[0]; b1 = src[1]; b2 = src[3]; b3 = src[4]; }
                    else { b0 = src[4]; b1 = src[3]; b2 = src[1]; b3 = src[0]; }
                    if (g & 1) {
                        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b0, acc1, 0, 0, 0);
                        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b1, acc1, 0, 0, 0);
                        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b2, acc1, 0, 0, 0);
                        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b3, acc1, 0, 0, 0);
                    } else {
                        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b0, acc0, 0, 0, 0);
                        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b1, acc0, 0, 0, 0);
                        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b2, acc0, 0, 0, 0);
                        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b3, acc0, 0, 0, 0);
                    }
                }
            }
        }
    }

    // ---- the eight partial tiles, added in wavefront order
    __syncthreads();   // every wavefront is done with its staging tiles
    float *red = lds;  // [8][32 * 33]
#pragma unroll
    for (int v = 0; v < 16; v++) red[w * (32 * 33) + acc_row(v, lane) * 33 + l32] = acc0[v] + acc1[v];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int idx = tid + i * 64 * kD2Waves, rr = idx >> 5, cc = idx & 31;
        float sum = red[rr * 33 + cc];
#pragma unroll
        for (int k = 1; k < kD2Waves; k++) sum += red[k * (32 * 33) + rr * 33 + cc];
        if (p.bias) sum += p.bias[o0 + (cc >> 2)];
        if (n0 + rr < p.N) p.out[(size_t)(n0 + rr) * p.O * 4 + o0 * 4 + cc] = sum;
    }
}

bool direct2x2_takes(const dopt_hip_conv_desc *d)
{
    return dense2x2_takes(d) && d->C % 64 == 0 && d->K % 64 == 0 && d->N * d->C * 4 < ((size_t)1 << 31) &&
           d->N * d->K * 4 < ((size_t)1 << 31) && d->K * d->C * 9 < ((size_t)1 << 31) && ceil_div(d->N, (size_t)kD2Rows) < 65536;
}

// *done = false: not this kernel's shape (or operands it cannot read as quads).
template <bool kBwd>
int run_direct2x2(const dopt_hip_conv_desc *d, const float *in, const float *w, const float *bias, float *out, bool *done)
{
    *done = false;
    if (!direct2x2_takes(d) || !aligned16(in) || !aligned16(w) || !aligned16(out)) return DOPT_HIP_OK;
    Direct2x2 p{};
    p.in = in;
    p.w = w;
    p.bias = bias;
    p.out = out;
    p.N = (int)d->N;
    p.R = (int)(kBwd ? d->K : d->C);
    p.O = (int)(kBwd ? d->C : d->K);
    p.C = (int)d->C;
    static bool raised[2] = {false, false};
    if (!raised[kBwd]) {
        DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)conv2x2_direct_k<kBwd>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)kD2Lds));
        raised[kBwd] = true;
    }
    // column tiles fastest: the blocks an XCD receives share an eighth of the filter and all of the batch
    const dim3 grid((unsigned)(p.O / kD2Chans), (unsigned)ceil_div(d->N, (size_t)kD2Rows));
    hipLaunchKernelGGL(conv2x2_direct_k<kBwd>, grid, dim3(64 * kD2Waves), kD2Lds, stream(), p);
    DOPT_LAUNCH_CHECK();
    *done = true;
    return DOPT_HIP_OK;
}

// Filter gradient of the same layers: dWd = x^T * dy, [4C, N] x [N, 4K], is the gradient of the matrix
// above; every filter tap collects the (input pixel, output pixel) pairs that read it - one pair for
// a corner tap, two for an edge tap, four for the centre - in a fixed order.
__global__ __launch_bounds__(256) void fold_2x2_k(unsigned C, unsigned K, const float4 *dwd, float *dw)
{
    const size_t total = (size_t)C * K;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const unsigned k = (unsigned)(i % K), c = (unsigned)(i / K);
        float q[4][4];   // [input pixel iy*2+ix][output pixel oy*2+ox]
#pragma unroll
        for (int pin = 0; pin < 4; pin++) {
            const float4 v = dwd[((size_t)c * 4 + pin) * K + k];
            q[pin][0] = v.x; q[pin][1] = v.y; q[pin][2] = v.z; q[pin][3] = v.w;
        }
        float *out = dw + ((size_t)k * C + c) * 9;
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int b = 0; b < 3; b++) {
                float sum = 0.0f;   // pairs with 1 - iy + oy == a and 1 - ix + ox == b
#pragma unroll
                for (int iy = 0; iy < 2; iy++)
#pragma unroll
                    for (int ix = 0; ix < 2; ix++) {
                        const int oy = a - 1 + iy, ox = b - 1 + ix;
                        if (oy >= 0 && oy < 2 && ox >= 0 && ox < 2) sum += q[iy * 2 + ix][oy * 2 + ox];
                    }
                out[a * 3 + b] = sum;
            }
    }
}

int run_dense2x2_wgrad(const dopt_hip_conv_desc *d, const float *dy, const float *x, float *dw)
{
    int rc = DOPT_HIP_OK;
    if (sgemm_fold2x2(d->C, d->K, d->N, x, dy, dw, &rc)) return rc;   // product and fold in one kernel
    void *dwd = nullptr;
    if ((rc = scratch_alloc(&dwd, dense2x2_elems(d) * sizeof(float)))) return rc;
    bool biased = false;
    rc = sgemm_bias(1, 0, 4 * d->C, 4 * d->K, d->N, x, dy, (float *)dwd, nullptr, 0, &biased);
    if (!rc) {
        const size_t blocks = ceil_div(d->C * d->K, (size_t)256);
        const size_t cap = (size_t)num_cus() * 16;
        hipLaunchKernelGGL(fold_2x2_k, dim3((unsigned)(blocks > cap ? cap : blocks)), dim3(256), 0, stream(), (unsigned)d->C,
                           (unsigned)d->K, (const float4 *)dwd, dw);
        if (hipGetLastError() != hipSuccess) rc = fail(DOPT_HIP_ERR_RUNTIME, "convolution: fold launch failed");
    }
    dopt_hip_free(dwd);
    return rc;
}

// ---- few output pixels: one image through a network ----------------------------------------------
// Forward of up to 64 output pixels.  The filter is most of what such a layer moves and nothing of it is used more than 64 times, so it
// is read once, as it lies: a row of it, [C][R][S], is the reduction in order, four steps of which a lane loads as 16 bytes whatever
// their alignment, and the fp32 matrix instruction takes (32 rows, two steps).  A workgroup owns 32 rows, all pixels and a part
// of the reduction, its eight wavefronts an eighth of that each.  The input under the part's channels lies in LDS with a halo of
// zeros; a step's offset in it is read from a table.  Bound by launch and latency: 8.9 MB read (256 and 512 -> 512 channels, 3 x 3, 16 and 4 pixels,
// on average) in 7.9 us are 1.1 TB/s, the CUs have work during 44 % of the cycles counted around a launch, the matrix cores during 10.
// VGG-16 on one image, 261 us, now 191: its nine layers on 8 x 8, 4 x 4 and 2 x 2 images 7 to 9 us each (Winograd 9 to 11 and 17 to pack
// their filters, conv2x2_direct_k 15).
struct FewConv {
    const float *x, *w, *bias;
    float *out;                     // [N][K][P][Q], or `cuts` copies of it, out_elems apart
    int N, C, H, W, K, R, S, padH, padW, strideH, strideW, P, Q;
    int PR, PC, depth;              // extents of an image with its halo; steps of the reduction per part
    size_t out_elems, w_bytes, x_bytes;
};
constexpr int kFewPixels = 64, kFewWaves = 8, kFewDepthMax = 1024;

template <int NP>   // groups of 32 pixels
__global__ __launch_bounds__(64 * kFewWaves) void conv_few_k(FewConv p)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float *const red = lds;                                        // [wavefront][group][32][33]
    int *const offs = (int *)(lds + kFewWaves * NP * 32 * 33);     // of the part's steps, a multiple of eight
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int taps = p.R * p.S, total = p.C * taps, m0 = blockIdx.x * 32;
    const int k0 = (int)blockIdx.y * p.depth, k1 = min(total, k0 + p.depth), steps = (k1 - k0 + 7) / 8 * 8;
    float *const patch = (float *)(offs + (p.depth + 7) / 8 * 8);
    const int c0 = k0 / taps, chans = (k1 - 1) / taps - c0 + 1, plane = p.PR * p.PC, chan = p.N * plane;

    const int slice = (steps / 8 + kFewWaves - 1) / kFewWaves * 8, kb = k0 + wave * slice, ke = min(k1, kb + slice);
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(p.w, p.w_bytes);
    const unsigned row = m0 + l32 < p.K ? (unsigned)(m0 + l32) * (unsigned)total * 4u : kOobOffset;
    constexpr int DEPTH = 4;   // steps of eight in flight
    float4 a[DEPTH];
    auto load = [&](int k) { return buffer_load_f32x4(rw, k < ke ? row + (unsigned)k * 4u : kOobOffset, 0); };
#pragma unroll
    for (int j = 0; j < DEPTH; j++) a[j] = load(kb + 8 * j + 4 * half);

    for (int i = tid; i < steps; i += 64 * kFewWaves) {
        const int k = k0 + i, c = k / taps, t = k - c * taps, r = t / p.S, s = t - r * p.S;
        offs[i] = k < k1 ? (c - c0) * chan + (p.R - 1 - r) * p.PC + (p.S - 1 - s) : 0;   // a true convolution
    }
    // a thread takes one place of every few channels: where it lies is found once
    const int span = min(chan, 64 * kFewWaves), together = 64 * kFewWaves / span, first = tid / span;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, p.x_bytes);
    for (int e = first < together ? tid - first * span : chan; e < chan; e += span) {
        const int n = e / plane, f = e - n * plane, fr = f / p.PC, ih = fr - p.padH, iw = f - fr * p.PC - p.padW;
        const bool in = ih >= 0 && ih < p.H && iw >= 0 && iw < p.W;
        const unsigned hw4 = (unsigned)(p.H * p.W) * 4u, from = (unsigned)(((n * p.C + c0) * p.H + ih) * p.W + iw) * 4u;
#pragma unroll 8
        for (int c = first; c < chans; c += together)
            patch[c * chan + e] = buffer_load_f32(rx, in ? from + (unsigned)c * hw4 : kOobOffset, 0);
    }
    __syncthreads();

    int base[NP];
    v16f acc[NP];
#pragma unroll
    for (int g = 0; g < NP; g++) {
        const int px = min(32 * g + l32, p.N * p.P * p.Q - 1), n = px / (p.P * p.Q), pq = px - n * p.P * p.Q, oh = pq / p.Q, ow = pq - oh * p.Q;
        base[g] = n * plane + oh * p.strideH * p.PC + ow * p.strideW;
#pragma unroll
        for (int v = 0; v < 16; v++) acc[g][v] = 0.0f;
    }
    for (int k = kb; k < ke; k += 8 * DEPTH) {
#pragma unroll
        for (int j = 0; j < DEPTH; j++) {
            const int kk = k + 8 * j + 4 * half;
            const float av[4] = {a[j].x, a[j].y, a[j].z, a[j].w};
            const int4 at = *(const int4 *)(offs + min(kk - k0, steps - 4));
            const int o[4] = {at.x, at.y, at.z, at.w};
            float in[NP][4];
#pragma unroll
            for (int g = 0; g < NP; g++)
#pragma unroll
                for (int e = 0; e < 4; e++) in[g][e] = patch[o[e] + base[g]];
            // what lies past the end counts as zero on both sides
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int g = 0; g < NP; g++)
                    acc[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(kk + e < ke ? av[e] : 0.0f, kk + e < ke ? in[g][e] : 0.0f, acc[g], 0, 0, 0);
            a[j] = load(kk + 8 * DEPTH);
            __builtin_amdgcn_sched_barrier(0);   // each refill stays behind its own step
        }
    }
#pragma unroll
    for (int g = 0; g < NP; g++)
#pragma unroll
        for (int v = 0; v < 16; v++) red[((wave * NP + g) * 32 + acc_row(v, lane)) * 33 + l32] = acc[g][v];
    __syncthreads();
    float *const out = p.out + (size_t)blockIdx.y * p.out_elems;
#pragma unroll
    for (int i = 0; i < 2 * NP; i++) {
        const int idx = tid + i * 64 * kFewWaves, r = idx / (32 * NP), px = idx % (32 * NP);
        const float *const from = red + ((px >> 5) * 32 + r) * 33 + (px & 31);
        float sum = from[0];
#pragma unroll
        for (int w = 1; w < kFewWaves; w++) sum += from[w * NP * 32 * 33];
        if (m0 + r < p.K && px < p.N * p.P * p.Q) {
            const int n = px / (p.P * p.Q), pq = px - n * p.P * p.Q;
            if (p.bias) sum += p.bias[m0 + r];
            out[((size_t)n * p.K + m0 + r) * (p.P * p.Q) + pq] = sum;
        }
    }
}

struct FewSetup {
    bool ok = false;
    FewConv f{};
    int cuts = 1;
    size_t elems = 0, lds_bytes = 0;
};
// Against the kernels that run without it (transposed bf16 tiles, Winograd with its packing, a copy of the filter in rows and general
// tiles): 512 -> 512 channels on 4 x 4 34 us, now 12; 640 -> 640 on 8 x 8 36, now 17; 320 -> 640 at stride 2 to 8 x 8 32, now 15;
// 100 -> 201 on 7 x 9 48, now 11; 256 -> 32 on 4 x 4 20, now 9; 400 -> 300 on one pixel 15, now 8.
// The kernels of 2 x 2 images keep more than 32 pixels (512 -> 512 of 16 images: 14 us, 17 here), conv2x2_direct_k fewer than 384
// input channels too (320 -> 320 of 8 images: 9.9 us, 10.7 here; 512 -> 512 of 8 images 14.0, 12.8 here, of one 13.8, 11.3 here).  Filters of
// 2^27 values and more keep the kernels that are checked at such sizes (5120 -> 512 on 4 x 4, 94 MB, 117 us, now 39).
FewSetup few_setup(const dopt_hip_conv_desc *d, size_t P, size_t Q)
{
    FewSetup u;
    const size_t pixels = d->N * P * Q, total = d->C * d->R * d->S;
    if (pixels > (size_t)kFewPixels || total < 256 || d->K < 32 || d->K * total >= (size_t)1 << 27 ||
        d->N * d->C * d->H * d->W * sizeof(float) >= (size_t)kOobOffset)
        return u;
    if ((dense2x2_takes(d) && pixels > 32) || (direct2x2_takes(d) && d->C < 384)) return u;
    const size_t PR = d->H + 2 * d->padH, PC = d->W + 2 * d->padW, taps = d->R * d->S;
    const size_t tiles = ceil_div(d->K, (size_t)32);
    size_t cuts = std::min({std::max((size_t)num_cus() / tiles, (size_t)1), total / 64, (size_t)16});
    cuts = std::max(cuts, ceil_div(total, (size_t)kFewDepthMax));
    const size_t depth = ceil_div(ceil_div(total, cuts), (size_t)8) * 8;
    cuts = ceil_div(total, depth);
    const size_t groups = pixels > 32 ? 2 : 1, chans = std::min((depth + taps - 2) / taps + 1, d->C);
    u.lds_bytes = (kFewWaves * groups * 32 * 33 + depth + chans * d->N * PR * PC) * sizeof(float);
    if (u.lds_bytes > 150 * 1024 || cuts > 64) return u;
    FewConv &f = u.f;
    f.N = (int)d->N; f.C = (int)d->C; f.H = (int)d->H; f.W = (int)d->W; f.K = (int)d->K; f.R = (int)d->R; f.S = (int)d->S;
    f.padH = (int)d->padH; f.padW = (int)d->padW; f.strideH = (int)d->strideH; f.strideW = (int)d->strideW;
    f.P = (int)P; f.Q = (int)Q; f.PR = (int)PR; f.PC = (int)PC; f.depth = (int)depth;
    u.elems = pixels * d->K;
    f.out_elems = copy_stride(u.elems);
    f.w_bytes = d->K * total * sizeof(float);
    f.x_bytes = d->N * d->C * d->H * d->W * sizeof(float);
    u.cuts = (int)cuts;
    u.ok = true;
    return u;
}

// `open` as in run_patch.
int run_few(const dopt_hip_conv_desc *d, size_t P, size_t Q, const float *x, const float *w, const float *bias, float *y, bool *done,
            dopt_hip_split_sum *open = nullptr)
{
    *done = false;
    FewSetup u = few_setup(d, P, Q);
    if (!u.ok) return DOPT_HIP_OK;
    FewConv &f = u.f;
    float *partial = nullptr;
    if (u.cuts > 1 && !(partial = (float *)workspace((size_t)u.cuts * f.out_elems * sizeof(float)))) return DOPT_HIP_ERR_OOM;
    f.x = x;
    f.w = w;
    f.bias = u.cuts == 1 ? bias : nullptr;
    f.out = u.cuts > 1 ? partial : y;
    const dim3 grid((unsigned)ceil_div(d->K, (size_t)32), (unsigned)u.cuts), block(64 * kFewWaves);
    const bool two = d->N * P * Q > 32;
    static bool raised = false;   // above 64 KB of dynamic LDS a kernel has to be told once
    if (!raised) {
        DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)conv_few_k<1>, hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024));
        DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)conv_few_k<2>, hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024));
        raised = true;
    }
    if (two) hipLaunchKernelGGL(conv_few_k<2>, grid, block, u.lds_bytes, stream(), f);
    else hipLaunchKernelGGL(conv_few_k<1>, grid, block, u.lds_bytes, stream(), f);
    DOPT_LAUNCH_CHECK();
    *done = true;
    if (u.cuts == 1) return DOPT_HIP_OK;
    if (open && u.elems % 4 == 0 && aligned16(y)) {   // the caller's next call adds the copies
        open->partial = partial;
        open->splits = u.cuts;
        open->elems = u.elems;
        open->C = d->K;
        open->inner = P * Q;
        open->bias = bias;
        open->value = y;
        open_split_set(partial);
        return DOPT_HIP_OK;
    }
    // in the order in which a later call adds the open copies, wherever the result lies
    return launch_splitk_reduce(u.elems, u.cuts, partial, y, bias, (unsigned)d->K, (unsigned)(P * Q));
}

template <class T, int SL, auto kKernel, class Args>
int launch_gather_kernel(const Args &args, dim3 grid)
{
    constexpr size_t lds = GatherLds<T, SL>::BYTES;
    if constexpr (lds > 64 * 1024) {   // a kernel has to be told once
        static bool raised = false;
        if (!raised) {
            DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)kKernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            raised = true;
        }
    }
    hipLaunchKernelGGL(kKernel, grid, dim3(T::THREADS), lds, stream(), args);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

template <class T, int SL>
int launch_gather(bool bwd, const GatherConv &g, dim3 grid)
{
    return bwd ? launch_gather_kernel<T, SL, conv_gather_k<T, SL, true>>(g, grid) : launch_gather_kernel<T, SL, conv_gather_k<T, SL, false>>(g, grid);
}

// Packs the filter w[K][C][g.R * g.S] and runs conv_gather_k on a problem whose geometry the caller
// has filled in (dimensions, padding, stride, output placement).
int gather_launch(GatherConv g, bool bwd, int K, int C, const float *in, const float *w, float *out)
{
    const int taps = g.R * g.S;
    g.CinPad = round_up(g.Cin, BK);
    g.Mp = round_up(g.Mout, 4);
    g.ncols = g.N * g.OH * g.OW;
    g.slabs_total = taps * g.CinPad / BK;
    g.out_elems = (size_t)g.ncols * g.Mout;
    const bool dense = g.out_sy == 1 && g.out_sx == 1 && g.out_plane == g.OH * g.OW;

    // tile shape: 64-row tiles for <= 64 output channels and wherever 128-row tiles would pad more;
    // otherwise 128x128
    const bool narrow = g.Mout <= 32, wide = !narrow && (g.Mout <= 64 || (g.Mout + 63) / 64 * 64 < (g.Mout + 127) / 128 * 128);
    const int BM = narrow ? 32 : wide ? 64 : 128, BN = narrow || wide ? 256 : 128;
    g.mtiles = (g.Mout + BM - 1) / BM;
    g.ntiles = (g.ncols + BN - 1) / BN;
    const int tiles = g.mtiles * g.ntiles;
    // (tiles of 32 rows are cut as those of 64: staging is most of a slab there, and longer chains would be further off)
    int splits = gather_splits(tiles, g.slabs_total, num_cus(), std::max(BM, 64), BN, g.out_elems, kGatherRate, 64, 4.5);
    if (!dense) splits = 1;   // (the copies would be whole tensors)
    const size_t elems = g.out_elems;
    g.out_elems = copy_stride(elems);
    g.slabs_per_split = (g.slabs_total + splits - 1) / splits;
    splits = (g.slabs_total + g.slabs_per_split - 1) / g.slabs_per_split;  // no empty split
    g.splits = splits;

    if ((size_t)BK * g.Mp * sizeof(float) > 0x7fffffffu)
        return fail(DOPT_HIP_ERR_UNSUPPORTED, "convolution: more than 2^25 output channels are not supported");
    const size_t wp_bytes = ((size_t)g.slabs_total * g.Mp * 96 + 255) / 256 * 256;
    const size_t part_bytes = splits > 1 ? (size_t)splits * g.out_elems * sizeof(float) : 0;
    char *ws = (char *)workspace(wp_bytes + part_bytes);
    if (!ws) return DOPT_HIP_ERR_OOM;
    float *wp = (float *)ws;
    float *partial = (float *)(ws + wp_bytes);
    SubFilters subs{};
    subs.n = 1;
    subs.f[0] = SubFilter{wp, g.R, g.S, 0, 0};
    if (int rc = launch_pack_gather(bwd, K, C, g.R, g.S, 1, 1, g.Mp, w, subs)) return rc;

    g.in = in;
    g.wp = wp;
    g.in_bytes = (size_t)g.N * g.Cin * g.IH * g.IW * sizeof(float);
    g.out = splits > 1 ? partial : out;
    dim3 grid(xcd_grid((unsigned)(tiles * splits)));
    // Short reductions that are not cut: in stages of one slab, two workgroups per CU, where there are two tiles per CU, or more than
    // one and a second slab would be half of the work.  1 x 1 on 128 images of 32 x 32, stages of two slabs -> of one: 16 -> 160 channels
    // 37 -> 28 us, 112 -> 160 63 -> 53; 145 images of 29 x 25, 15 -> 7, 411 tiles, 14 -> 12; but 64 of 32 x 32, 16 -> 32, 256 tiles, 7.4 -> 8.7, and
    // 3 x 3 on 64 of 33 x 31, 16 -> 32, 256 tiles of nine slabs, 17 -> 19.  Beyond nine slabs only from four tiles per CU on, where reductions
    // were not cut before either: without chains the error is that of the whole reduction (320 -> 320 196 -> 191 us, 480 -> 320, thirty
    // slabs, 275 -> 266; but 42 -> 592, 3 x 3, 515 tiles of 27 slabs, 1.3 times as far off).
    const int cus = num_cus();
    const bool brief = splits == 1 && g.slabs_total <= (tiles >= 4 * cus ? 32 : tiles >= 2 * cus ? 9 : tiles > cus ? 3 : 0);
    if (narrow) {
        if (int rc = brief ? launch_gather<GatherNarrow, 1>(bwd, g, grid) : launch_gather<GatherNarrow, 2>(bwd, g, grid)) return rc;
    } else if (int rc = brief ? (wide ? launch_gather<GatherWide, 1>(bwd, g, grid) : launch_gather<GatherSquare, 1>(bwd, g, grid))
                       : (wide ? launch_gather<GatherWide, 2>(bwd, g, grid) : launch_gather<GatherSquare, 2>(bwd, g, grid)))
        return rc;
    if (splits > 1) return launch_splitk_exact(elems, splits, partial, out);
    return DOPT_HIP_OK;
}

// ---- backward-data with a stride, one residue class of output pixels at a time -------------------
// dx[n, c, h, w] = sum over k, r, s with (h + padH - r) and (w + padW - s) multiples of the stride of
// dy[n, k, (h + padH - r) / sH, (w + padW - s) / sW] * w[k, c, R - 1 - r, S - 1 - s] (the flipped filter).  Which taps qualify depends only
// on (h mod sH, w mod sW).  Taking all pixels together multiplies every pixel
// by every tap and masks three quarters of the products of a stride-2 3x3 layer; taking the pixels
// of one class (a, b) = (h mod sH, w mod sW) at a time, only its taps r = r0, r0 + sH, ... and s = s0,
// s0 + sW, ... are multiplied, and the class is a UNIT-stride problem on the grid (i, j) = (h / sH, w / sW):
//     dy row = i + (a + padH - r0) / sH - t   for its t-th tap row,
// i.e. backward-data of a filter with ceil((R - r0) / sH) rows, padding (a + padH - r0) / sH and rows
// stored in reverse order of r.  The sub-filter is copied out of w, the kernel's output placement
// scatters the class back into dx.
__global__ __launch_bounds__(256) void subfilter_k(int KC, int R, int S, int R2, int S2, int r0, int s0, int sH, int sW,
                                                    const float *w, float *sub)
{
    const int total = KC * R2 * S2;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const int kc = i / (R2 * S2), t = i - kc * (R2 * S2), tr = t / S2, ts = t - tr * S2;
        // stored row tr of the sub-filter stands for tap offset r = r0 + (R2 - 1 - tr) * sH, and the filter
        // element that multiplies offset r is the flipped one, w[.., R - 1 - r, S - 1 - s]
        const int r = r0 + (R2 - 1 - tr) * sH, sc = s0 + (S2 - 1 - ts) * sW;
        sub[i] = w[(size_t)kc * (R * S) + (R - 1 - r) * S + (S - 1 - sc)];
    }
}

int run_bwd_strided(const dopt_hip_conv_desc *d, size_t P, size_t Q, const float *dy, const float *w, float *dx)
{
    const int sH = (int)d->strideH, sW = (int)d->strideW, R = (int)d->R, S = (int)d->S;
    const int H = (int)d->H, W = (int)d->W, padH = (int)d->padH, padW = (int)d->padW;
    struct Cls { int n, first, taps, pad; };   // pixels of the class along one axis, its first tap, tap count, padding
    auto cls = [](int a, int extent, int stride, int pad, int filt) {
        Cls c{};
        c.n = a < extent ? (extent - a + stride - 1) / stride : 0;
        c.first = (a + pad) % stride;
        c.taps = c.first < filt ? (filt - c.first + stride - 1) / stride : 0;
        c.pad = (a + pad - c.first) / stride;
        return c;
    };
    bool gaps = false;   // classes no tap reaches: those pixels of dx are zero
    for (int a = 0; a < sH; a++) gaps = gaps || (cls(a, H, sH, padH, R).n > 0 && cls(a, H, sH, padH, R).taps == 0);
    for (int b = 0; b < sW; b++) gaps = gaps || (cls(b, W, sW, padW, S).n > 0 && cls(b, W, sW, padW, S).taps == 0);
    if (gaps)
        if (int rc = dopt_hip_memset(dx, 0, d->N * d->C * d->H * d->W * sizeof(float))) return rc;
    // Two to nine classes with work (a 3 x 3 filter at stride 2 has four: 1, 2, 2 and 4 taps): one launch packs all
    // their sub-filters and one launch multiplies all of them, instead of three dependent launches per class.
    struct Job { Cls ch, cw; int a, b; };
    Job jobs[kGatherJobs];
    int njobs = 0;
    bool fits = true;
    for (int a = 0; a < sH; a++)
        for (int b = 0; b < sW; b++) {
            const Cls ch = cls(a, H, sH, padH, R), cw = cls(b, W, sW, padW, S);
            if (ch.n == 0 || cw.n == 0 || ch.taps == 0 || cw.taps == 0) continue;
            if (njobs == kGatherJobs) { fits = false; continue; }
            jobs[njobs++] = Job{ch, cw, a, b};
        }
    if (fits && njobs >= 2) {
        for (int i = 1; i < njobs; i++)   // most taps first (insertion sort, stable)
            for (int j = i; j > 0 && jobs[j].ch.taps * jobs[j].cw.taps > jobs[j - 1].ch.taps * jobs[j - 1].cw.taps; j--)
                std::swap(jobs[j], jobs[j - 1]);
        const int K = (int)d->K, C = (int)d->C;
        const int KPad = round_up(K, BK), Mp = round_up(C, 4);
        if ((size_t)BK * Mp * sizeof(float) > 0x7fffffffu)
            return fail(DOPT_HIP_ERR_UNSUPPORTED, "convolution: more than 2^25 output channels are not supported");
        // The classes' reductions are cut into the same number of parts, each a partial copy of the whole of dx: where a handful of
        // tiles would be as many workgroups of a long chain (47 images of 4 x 11, 300 channels to 5: 61 us, now 13 with the sum).
        const bool narrow = C <= 32, wide = !narrow && (C <= 64 || (C + 63) / 64 * 64 < (C + 127) / 128 * 128);
        const int BM = narrow ? 32 : wide ? 64 : 128, BN = narrow || wide ? 256 : 128;
        const size_t elems = d->N * d->C * d->H * d->W;
        int splits = 1;
        if (!gaps) {   // (a copy has no value where no tap reaches)
            const double t_slab = 2.0 * std::max(BM, 64) * BN * 16 / (kGatherRate * 1e6);
            double best = 0;
            for (int sp = 1; sp <= 32; sp++) {
                double total = 0, longest = 0;
                bool full = true;
                for (int j = 0; j < njobs; j++) {
                    const int slabs = jobs[j].ch.taps * jobs[j].cw.taps * KPad / BK, per = (slabs + sp - 1) / sp;
                    const double tiles = ceil_div((size_t)C, (size_t)BM) * ceil_div((size_t)d->N * jobs[j].ch.n * jobs[j].cw.n, (size_t)BN);
                    full = full && (sp - 1) * per < slabs;
                    total += tiles * sp * (per * t_slab + 6.0);
                    longest = std::max(longest, per * t_slab + 6.0);
                }
                if (!full) continue;
                const double cost = std::max(total / num_cus(), longest) + (sp > 1 ? 4.5 + (sp + 1.0) * elems * 4.0 / 4.5e6 : 0.0);
                if (sp == 1 || cost < best * 0.9) {
                    splits = sp;
                    best = cost;
                }
            }
        }
        size_t wp_off[kGatherJobs + 1] = {0};
        for (int j = 0; j < njobs; j++) {
            const size_t slabs = (size_t)jobs[j].ch.taps * jobs[j].cw.taps * KPad / BK;
            wp_off[j + 1] = wp_off[j] + (slabs * Mp * 96 + 255) / 256 * 256;
        }
        char *ws = (char *)workspace(wp_off[njobs] + (splits > 1 ? (size_t)splits * copy_stride(elems) * sizeof(float) : 0));
        if (!ws) return DOPT_HIP_ERR_OOM;
        float *const partial = (float *)(ws + wp_off[njobs]);
        SubFilters subs{};
        GatherGroup gg{};
        subs.n = gg.n = njobs;
        unsigned blocks = 0;
        for (int j = 0; j < njobs; j++) {
            const Job &jb = jobs[j];
            subs.f[j] = SubFilter{(float *)(ws + wp_off[j]), jb.ch.taps, jb.cw.taps, jb.ch.first, jb.cw.first};
            GatherConv &g = gg.g[j];
            g.N = (int)d->N;
            g.R = jb.ch.taps; g.S = jb.cw.taps;
            g.padH = jb.ch.pad; g.padW = jb.cw.pad;
            g.strideH = g.strideW = 1;
            g.Cin = K; g.IH = (int)P; g.IW = (int)Q;
            g.Mout = C; g.OH = jb.ch.n; g.OW = jb.cw.n;
            g.out_plane = H * W; g.out_OW = W;
            g.out_sy = sH; g.out_sx = sW; g.out_oy = jb.a; g.out_ox = jb.b;
            g.CinPad = KPad;
            g.Mp = Mp;
            g.ncols = g.N * g.OH * g.OW;
            g.slabs_total = g.R * g.S * KPad / BK;
            g.slabs_per_split = (g.slabs_total + splits - 1) / splits;
            g.splits = splits;
            g.out_elems = copy_stride(elems);
            g.mtiles = (g.Mout + BM - 1) / BM;
            g.ntiles = (g.ncols + BN - 1) / BN;
            g.in = dy;
            g.wp = subs.f[j].wp;
            g.out = splits > 1 ? partial : dx;
            g.in_bytes = (size_t)g.N * g.Cin * g.IH * g.IW * sizeof(float);
            gg.per[j] = ((unsigned)(g.mtiles * g.ntiles * splits) + 7u) / 8u;
            blocks += 8u * gg.per[j];
        }
        if (int rc = launch_pack_gather(true, K, C, R, S, sH, sW, Mp, w, subs)) return rc;
        if (int rc = narrow ? launch_gather_kernel<GatherNarrow, 2, conv_gather_group_k<GatherNarrow, 2, true>>(gg, blocks)
                   : wide ? launch_gather_kernel<GatherWide, 2, conv_gather_group_k<GatherWide, 2, true>>(gg, blocks)
                          : launch_gather_kernel<GatherSquare, 2, conv_gather_group_k<GatherSquare, 2, true>>(gg, blocks))
            return rc;
        if (splits > 1) return launch_splitk_exact(elems, splits, partial, dx);
        return DOPT_HIP_OK;
    }
    void *sub = nullptr;
    if (int rc = scratch_alloc(&sub, d->K * d->C * d->R * d->S * sizeof(float))) return rc;
    int rc = DOPT_HIP_OK;
    for (int a = 0; a < sH && !rc; a++)
        for (int b = 0; b < sW && !rc; b++) {
            const Cls ch = cls(a, H, sH, padH, R), cw = cls(b, W, sW, padW, S);
            if (ch.n == 0 || cw.n == 0 || ch.taps == 0 || cw.taps == 0) continue;
            const int KC = (int)(d->K * d->C);
            hipLaunchKernelGGL(subfilter_k, dim3((unsigned)ceil_div((size_t)KC * ch.taps * cw.taps, (size_t)256)), dim3(256), 0,
                               stream(), KC, R, S, ch.taps, cw.taps, ch.first, cw.first, sH, sW, w, (float *)sub);
            if (hipGetLastError() != hipSuccess) {
                rc = fail(DOPT_HIP_ERR_RUNTIME, "convolution: sub-filter launch failed");
                break;
            }
            GatherConv g{};
            g.N = (int)d->N;
            g.R = ch.taps; g.S = cw.taps;
            g.padH = ch.pad; g.padW = cw.pad;
            g.strideH = g.strideW = 1;
            g.Cin = (int)d->K; g.IH = (int)P; g.IW = (int)Q;
            g.Mout = (int)d->C; g.OH = ch.n; g.OW = cw.n;
            g.out_plane = H * W; g.out_OW = W;
            g.out_sy = sH; g.out_sx = sW; g.out_oy = a; g.out_ox = b;
            rc = gather_launch(g, true, (int)d->K, (int)d->C, dy, (const float *)sub, dx);
        }
    dopt_hip_free(sub);
    return rc;
}

// Shared host driver of forward (kBwd = false) and backward-data (kBwd = true).
template <bool kBwd>
int run_gather(const dopt_hip_conv_desc *d, size_t P, size_t Q, const float *in, const float *w, float *out,
               const float *bias = nullptr)
{
    if (!kBwd) {
        bool done = false;
        if (int rc = conv_smallc_fwd(d, in, w, bias, out, &done)) return rc;
        if (done) return DOPT_HIP_OK;
        if (int rc = run_few(d, P, Q, in, w, bias, out, &done)) return rc;
        if (done) return DOPT_HIP_OK;
    }
    if (dense2x2_takes(d)) {
        bool done = false;
        if (int rc = run_direct2x2<kBwd>(d, in, w, bias, out, &done)) return rc;
        if (done) return DOPT_HIP_OK;
        return run_dense2x2<kBwd>(d, in, w, nullptr, bias, out);
    }
    {
        bool done = false;
        if (int rc = run_patch<kBwd>(d, P, Q, in, w, bias, out, &done)) return rc;
        if (done) return DOPT_HIP_OK;
    }
    if (bias) {  // the generic kernel has no fused bias: add it in place afterwards
        if (int rc = run_gather<kBwd>(d, P, Q, in, w, out, nullptr)) return rc;
        return dopt_hip_bias_fwd(d->N, kBwd ? d->C : d->K, kBwd ? d->H * d->W : P * Q, out, bias, out);
    }
    if (kBwd && (d->strideH > 1 || d->strideW > 1)) return run_bwd_strided(d, P, Q, in, w, out);
    GatherConv g{};
    g.N = (int)d->N;
    g.R = (int)d->R;
    g.S = (int)d->S;
    g.padH = (int)d->padH;
    g.padW = (int)d->padW;
    g.strideH = (int)d->strideH;
    g.strideW = (int)d->strideW;
    if (!kBwd) {
        g.Cin = (int)d->C; g.IH = (int)d->H; g.IW = (int)d->W;
        g.Mout = (int)d->K; g.OH = (int)P; g.OW = (int)Q;
    } else {
        g.Cin = (int)d->K; g.IH = (int)P; g.IW = (int)Q;
        g.Mout = (int)d->C; g.OH = (int)d->H; g.OW = (int)d->W;
    }
    g.out_plane = g.OH * g.OW;
    g.out_OW = g.OW;
    g.out_sy = g.out_sx = 1;
    return gather_launch(g, kBwd, (int)d->K, (int)d->C, in, w, out);
}

template <int WM, int WC, int kGeo, bool kPre = kGeo != 2>
int launch_wgrad_patch(const WgradPatch &wp, dim3 grid, size_t lds_bytes)
{
    static bool raised = false;
    if (!raised) {
        DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)conv_wgrad_patch_k<WM, WC, kGeo, kPre>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        raised = true;
    }
    hipLaunchKernelGGL((conv_wgrad_patch_k<WM, WC, kGeo, kPre>), grid, dim3(64 * 3 * WM * WC), lds_bytes, stream(), wp);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

template <class T, int TPT>
int launch_wgrad(const FilterGrad &f, dim3 grid)
{
    constexpr size_t lds = (size_t)2 * 2 * 6 * (T::BM + 4 + T::BN + 4) * 16;
    static bool raised = false;
    if (!raised) {   // above 64 KB of dynamic LDS a kernel has to be told once
        DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)conv_wgrad_k<T, TPT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        raised = true;
    }
    hipLaunchKernelGGL((conv_wgrad_k<T, TPT>), grid, dim3(T::THREADS), lds, stream(), f);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

int launch_wgrad_reduce(int K, int C, int Cp, int taps, int splits, size_t out_elems, const float *partial, float *dw)
{
    // few elements of many copies (fewer than sixteen: lanes with nothing to add; more values fill the chip either way)
    if (splits >= 16 && (size_t)K * C * taps <= (size_t)1 << 17) {
        hipLaunchKernelGGL(wgrad_reduce_small_k, dim3((unsigned)K, (unsigned)ceil_div((size_t)C * taps, (size_t)64)), dim3(1024), 0, stream(), C, Cp, taps, splits,
                           out_elems, partial, dw);
        DOPT_LAUNCH_CHECK();
        return DOPT_HIP_OK;
    }
    // 64-channel chunks when that still leaves >= 1024 workgroups and the LDS staging stays small
    const int ch = ((size_t)K * ((C + 63) / 64) >= 1024 && taps <= 16) ? 64 : 16;
    dim3 rgrid((unsigned)K, (unsigned)((C + ch - 1) / ch));
    hipLaunchKernelGGL(wgrad_reduce_k, rgrid, dim3(256), (size_t)5 * ch * taps * sizeof(float), stream(), K, C, Cp, taps,
                       ch, splits, out_elems, partial, dw);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

// What run_wgrad_patch decides before it touches memory: ok = false when the shape is not this path's
// (3x3, unit stride, pad 1; rows of 8 / 16 / 32 / 64 pixels, or 4x4 or 2x2 images).
struct WgradSetup {
    bool ok;
    WgradPatch wp;
    bool tall;            // 128 rows x 32 channels per block
    bool pre;             // x is split when it is stored
    bool quads;           // the result is whole quads on the 16-byte grid (else its partial copies are added here, never left open)
    int rows;             // output channels per block: 128 (tall), 160 (x 32 channels) or 64 (x 64 channels)
    int geo, tiles, splits;
    size_t out_elems, lds_bytes;
};

WgradSetup wgrad_patch_setup(const dopt_hip_conv_desc *d, const float *dw)
{
    WgradSetup u{};
    if (d->R != 3 || d->S != 3 || d->strideH != 1 || d->strideW != 1 || d->padH != 1 || d->padW != 1) return u;
    if (d->C < 16) return u;  // a 32-channel fragment would be mostly padding
    const int W = (int)d->W, H = (int)d->H;
    WgradPatch &wp = u.wp;
    int geo;
    if (W == 8 || W == 16 || W == 32 || W == 64) {
        geo = 0;
        wp.G = 64 / W;
        if (H % wp.G != 0) return u;
        wp.bands = H / wp.G;
        wp.imgs = 1;
        wp.ppitch = W + 8;
        wp.cstride = (wp.G + 2) * wp.ppitch;
        wp.chunks_total = (int)d->N * wp.bands;
    } else if ((W == 4 && H == 4) || (W == 2 && H == 2)) {
        geo = W == 4 ? 1 : 2;
        wp.G = H;
        wp.bands = 1;
        wp.imgs = 64 / (H * W);
        if (d->N % wp.imgs != 0) return u;
        wp.ppitch = geo == 1 ? 12 : 4;
        wp.cstride = geo == 1 ? 4 * 72 : 16 * 16;
        wp.chunks_total = (int)d->N / wp.imgs;
    } else {
        return u;
    }
    // 128 rows x 32 channels, or 64 x 64 when that pads the output channels less (160 -> 192, not 256)
    // ... or 160 x 32 where that pads them less than both (160 channels: 160 rows, not 192 or 256)
    const int up64 = (int)((d->K + 63) / 64 * 64), up128 = (int)((d->K + 127) / 128 * 128), up160 = (int)((d->K + 159) / 160 * 160);
    // (by a tenth at least: 480 channels are 512 rows of the 64-row tiles, and ran no faster as 3 x 160)
    // (320 and 640 channels, which the other heights do not pad either, ran slower this way: measured)
    const bool rows160 = d->K > 64 && up160 * 11 < up64 * 10 && up160 * 11 < up128 * 10 && !no_tall_tiles();
    const bool tall = !rows160 && d->K >= 128 && up128 <= up64;
    if (!tall && !rows160 && W == 64) return u;
    const int BM = rows160 ? 160 : tall ? 128 : 64, BC = BM == 64 ? 64 : 32;
    // x is split when it is stored: not with 2 x 2 images, whose values are single 16-bit ones, nor where the parts of 160 rows
    // and of rows of 64 pixels do not fit the LDS together
    const bool pre = geo != 2 && !(rows160 && W == 64);
    // 128-bit reads by 32 channels at these strides touch every LDS bank once: an odd number of 16-byte pieces (with parts, of
    // 16-bit values; one piece at least behind the last row, which holds its right edge)
    if (pre) wp.cstride = geo == 0 ? ((wp.G + 2) * wp.ppitch / 8 + 1 | 1) * 8 : 21 * 8;
    else while (wp.cstride % 8 != 4) wp.cstride += 4;
    wp.N = (int)d->N; wp.C = (int)d->C; wp.K = (int)d->K; wp.H = H; wp.W = W;
    wp.quads_row = W / 4;
    wp.mtiles = (wp.K + BM - 1) / BM;
    wp.ctiles = (wp.C + BC - 1) / BC;
    wp.dy_bytes = (size_t)wp.N * wp.K * H * W * sizeof(float);
    wp.x_bytes = (size_t)wp.N * wp.C * H * W * sizeof(float);
    const size_t out_elems = (size_t)wp.K * wp.C * 9;
    const int tiles = wp.mtiles * wp.ctiles;
    // one block per CU: never a grid slightly above the CU count (a second, nearly empty round)
    // Splits of the pixel chunks: one block per CU runs at a time, the launch takes ceil(blocks / CUs)
    // rounds of one block's duration.  Estimate (microseconds) per candidate: rounds x (chunks per
    // block x time per chunk + a fixed set-up and epilogue) + writing and re-reading the partial
    // filters; 100 tiles are better served by 5 splits (500 blocks, two nearly full rounds) than by
    // 2 (200 blocks on 256 CUs).
    int splits = 1;
    {
        const int max_by_depth = wp.chunks_total / 2 > 0 ? wp.chunks_total / 2 : 1;  // two chunks amortise the set-up
        // (0.45 TFLOP/s per CU was the fp32 instruction's loop, this one sustains 0.8; with 0.7 here the layers of VGG-16 and
        // Wide-ResNet-28-10 at batch 128 are cut the same)
        const double t_chunk = 2.0 * BM * BC * 9 * 64 / 0.45e6;
        double best = 0.0;
        for (int sp = 1; sp <= max_by_depth && sp <= 512; sp++) {
            const int per_block = (wp.chunks_total + sp - 1) / sp;
            if (sp > 1 && (wp.chunks_total + per_block - 1) / per_block != sp) continue;
            const double rounds = (double)(((long long)tiles * sp + num_cus() - 1) / num_cus());
            double cost = rounds * (per_block * t_chunk + 8.0);
            if (sp > 1) cost += 3.0 + 2.0 * sp * out_elems * 4.0 / 4.5e6;
            if (sp == 1 || cost < best * 0.97) {
                splits = sp;
                best = cost;
            }
        }
    }
    u.quads = out_elems % 4 == 0 && aligned16(dw);
    // 64-row tiles on 4 x 4 images: few workgroups of a long set-up unless the layer or the batch is large, and one without a split
    // (16 images, 64 -> 64 channels: 20 us, the general kernel 10; 140, 62 -> 27: 135 and 18; 128, 128 -> 48: 21 and 18; but 256, 16 -> 16:
    // 18 and 26; 512, 64 -> 64: 25 and 29; 128, 320 -> 320: 41 and 59; 192 -> 192, nine tiles, 8 to 128 images: within a tenth)
    if (geo == 1 && BM == 64 && (!u.quads || (tiles < 8 && d->N < 256))) return u;
    wp.chunks_per_split = (wp.chunks_total + splits - 1) / splits;
    splits = (wp.chunks_total + wp.chunks_per_split - 1) / wp.chunks_per_split;
    wp.splits = splits;
    const size_t lds_main = ((size_t)2 * BM * 68 + (pre ? (size_t)3 * BC * wp.cstride : (size_t)2 * BC * wp.cstride + 4)) * sizeof(float);
    const size_t lds_epi = (size_t)32 * (BC * 9 + 1) * sizeof(float);
    u.lds_bytes = lds_main > lds_epi ? lds_main : lds_epi;
    if (u.lds_bytes > 160 * 1024) return u;
    wp.split_stride = copy_stride(out_elems);
    u.tall = tall; u.pre = pre; u.rows = BM; u.geo = geo; u.tiles = tiles; u.splits = splits; u.out_elems = out_elems;
    u.ok = true;
    return u;
}

// Split lanes of the pass that adds a filter gradient's partial copies: enough blocks for small filters with
// hundreds of splits means more split lanes per block.
int wgrad_sum_lanes(size_t n4) { return n4 >= (size_t)64 * 512 ? 4 : 16; }

// out = `splits` partial copies of n4 quads added in the order `lanes` fixes (split_sum_k)
int launch_split_sum(size_t n4, int splits, int lanes, const float *partial, float *out)
{
    if (lanes == 4)
        hipLaunchKernelGGL(split_sum_k<4>, dim3((unsigned)ceil_div(n4, (size_t)64)), dim3(256), 0, stream(), n4, splits, n4,
                           (const float4 *)partial, (float4 *)out);
    else if (lanes == 16)
        hipLaunchKernelGGL(split_sum_k<16>, dim3((unsigned)ceil_div(n4, (size_t)16)), dim3(256), 0, stream(), n4, splits, n4,
                           (const float4 *)partial, (float4 *)out);
    else
        return fail(DOPT_HIP_ERR_INVALID, "split sum: %d lanes (4 or 16)", lanes);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

// dw = the partial filters added in split order
int wgrad_split_sum(const WgradSetup &u, const float *partial, float *dw)
{
    const size_t n4 = u.wp.split_stride / 4;
    if (!u.quads) {
        const bool few = wgrad_sum_lanes(n4) == 16;
        const dim3 grid((unsigned)ceil_div(n4, (size_t)(few ? 16 : 64)));
        if (few) hipLaunchKernelGGL((split_sum_k<16, true>), grid, dim3(256), 0, stream(), n4, u.splits, n4, (const float4 *)partial, (float4 *)dw, u.out_elems);
        else hipLaunchKernelGGL((split_sum_k<4, true>), grid, dim3(256), 0, stream(), n4, u.splits, n4, (const float4 *)partial, (float4 *)dw, u.out_elems);
        DOPT_LAUNCH_CHECK();
        return DOPT_HIP_OK;
    }
    return launch_split_sum(n4, u.splits, wgrad_sum_lanes(n4), partial, dw);
}

// The launch of a filled-in filter-gradient setup: tile height and pixel geometry pick the instance.
int dispatch_wgrad_patch(const WgradSetup &u)
{
    const WgradPatch &wp = u.wp;
    const dim3 grid(xcd_grid((unsigned)(u.tiles * u.splits)));
    const int geo = u.geo;
    if (u.rows == 160 && geo == 0 && !u.pre) return launch_wgrad_patch<5, 1, 0, false>(wp, grid, u.lds_bytes);
    if (u.rows == 160) return geo == 0 ? launch_wgrad_patch<5, 1, 0>(wp, grid, u.lds_bytes)
                            : geo == 1 ? launch_wgrad_patch<5, 1, 1>(wp, grid, u.lds_bytes)
                                       : launch_wgrad_patch<5, 1, 2>(wp, grid, u.lds_bytes);
    if (u.tall) return geo == 0 ? launch_wgrad_patch<4, 1, 0>(wp, grid, u.lds_bytes)
                     : geo == 1 ? launch_wgrad_patch<4, 1, 1>(wp, grid, u.lds_bytes)
                                : launch_wgrad_patch<4, 1, 2>(wp, grid, u.lds_bytes);
    return geo == 0 ? launch_wgrad_patch<2, 2, 0>(wp, grid, u.lds_bytes)
         : geo == 1 ? launch_wgrad_patch<2, 2, 1>(wp, grid, u.lds_bytes)
                    : launch_wgrad_patch<2, 2, 2>(wp, grid, u.lds_bytes);
}

int run_wgrad_patch(const dopt_hip_conv_desc *d, const float *dy, const float *x, float *dw, bool *done)
{
    *done = false;
    WgradSetup u = wgrad_patch_setup(d, dw);
    if (!u.ok) return DOPT_HIP_OK;
    WgradPatch &wp = u.wp;
    float *partial = nullptr;
    if (u.splits > 1) {
        partial = (float *)workspace((size_t)u.splits * wp.split_stride * sizeof(float));
        if (!partial) return DOPT_HIP_ERR_OOM;
    }
    wp.dy = dy; wp.x = x;
    wp.out = u.splits > 1 ? partial : dw;
    if (int rc = dispatch_wgrad_patch(u)) return rc;
    *done = true;
    if (u.splits > 1) return wgrad_split_sum(u, partial, dw);
    return DOPT_HIP_OK;
}

// Backward-data (on a packed filter) and filter gradient of one 3x3 layer as one launch (conv_bwd_pair_k).
// *done = false: one of the two is not a patch-kernel shape, or a combination that is not built; the
// caller runs them one after the other.  `open` as in run_patch.
template <class T, int NS, int WM, int WC, int kGeo>
int launch_bwd_pair(const PatchConv &pc, const WgradPatch &wp, unsigned grid_a, unsigned grid_b, size_t lds_bytes)
{
    static bool raised = false;
    if (!raised) {
        DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)conv_bwd_pair_k<T, NS, WM, WC, kGeo>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        raised = true;
    }
    hipLaunchKernelGGL((conv_bwd_pair_k<T, NS, WM, WC, kGeo>), dim3(grid_a + grid_b), dim3(768), lds_bytes, stream(), pc,
                       wp, grid_a);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}


int run_bwd_pair(const dopt_hip_conv_desc *d, size_t P, size_t Q, const float *dy, const float *prepacked, const float *x,
                 float *dx, float *dw, dopt_hip_split_sum *open, dopt_hip_split_sum *open_dw, bool *done)
{
    *done = false;
    PatchSetup a = patch_setup<true>(d, P, Q);
    WgradSetup b = wgrad_patch_setup(d, dw);
    if (!a.ok || !b.ok || !prepacked || a.pc.Cin % 16 != 0) return DOPT_HIP_OK;
    // The combinations that are built: 128 x 128 backward-data tiles on eight wavefronts, one workgroup per CU
    // (the 64 x 256 and 32 x 256 tiles of layers with up to 64 input channels are not built), with 128 x 32 filter-gradient tiles on
    // rows of 8 .. 64 pixels or on 4 x 4 images.
    // (a layer the Winograd kernel takes has its filter packed for that kernel: shape 4, not a pair)
    // (only where the launch needs it: with two rounds of backward-data tiles and more the two run one after the other, which
    // took as long or 1 % less: 64 images of 100 x 32 x 32, 128 filters, 350 and 348 us for the whole step; 256 of 200 x 16 x 16, 384, 1460 and 1450)
    const bool few = a.shape == 2 && a.tiles < 2 * num_cus();
    const int combo = few && b.tall && b.geo == 0 ? 0 : few && b.tall && b.geo == 1 ? 1 : -1;
    // A layer whose backward-data is the Winograd kernel on 128-row tiles: two launches, each as it would run alone, but out of ONE
    // workspace request, so that both results can stay open for the launch behind them - the filter gradient's split
    // sum rides in the batch-norm gradient there instead of being a launch of its own.  (The same for the 64-row layers
    // was measured and does not pay: they are followed by the multi-block batch norm, whose workgroups fill every CU,
    // so the riders only start when those have finished - 20 us per layer instead of the 7.6 us of the separate sum.)
    const bool two = combo < 0 && a.shape == 4 && a.BM == 128 && open_dw != nullptr && b.splits > 1 && b.quads;
    if (combo < 0 && !two) return DOPT_HIP_OK;
    PatchConv &pc = a.pc;
    WgradPatch &wp = b.wp;
    const int splits_a = patch_decide_splits(&a, dx);
    const size_t part_a = splits_a > 1 ? ((size_t)splits_a * pc.out_elems * sizeof(float) + 255) / 256 * 256 : 0;
    const size_t part_b = b.splits > 1 ? (size_t)b.splits * wp.split_stride * sizeof(float) : 0;
    char *ws = part_a + part_b > 0 ? (char *)workspace(part_a + part_b) : nullptr;
    if (part_a + part_b > 0 && !ws) return DOPT_HIP_ERR_OOM;
    float *partial_a = (float *)ws, *partial_b = (float *)(ws + part_a);
    pc.in = dy;
    pc.wp = prepacked;
    pc.bias = nullptr;
    pc.in_bytes = (size_t)pc.N * pc.Cin * pc.IH * pc.IW * sizeof(float);
    pc.out = splits_a > 1 ? partial_a : dx;
    wp.dy = dy; wp.x = x;
    wp.out = b.splits > 1 ? partial_b : dw;
    const unsigned grid_a = xcd_grid((unsigned)(a.tiles * splits_a)), grid_b = xcd_grid((unsigned)(b.tiles * b.splits));
    const size_t lds_bytes = a.lds_bytes > b.lds_bytes ? a.lds_bytes : b.lds_bytes;
    PairProbe &probe = g_pair_probe;
    const bool probing = probe.on == 1 && !capturing() && !two;
    if (probing)
        if (int rc2 = probe_begin(probe)) return rc2;
    int rc;
    if (two) {
        rc = dispatch_wgrad_patch(b);
        if (!rc) rc = dispatch_patch(a, splits_a);
    } else if (combo == 0) rc = launch_bwd_pair<PatchDeep, 2, 4, 1, 0>(pc, wp, grid_a, grid_b, lds_bytes);
    else rc = launch_bwd_pair<PatchDeep, 2, 4, 1, 1>(pc, wp, grid_a, grid_b, lds_bytes);
    if (rc) return rc;
    if (probing) {
        DOPT_HIP_CHECK(hipEventRecord(probe.events[probe.used++].second, stream()));
        const double px = (double)d->N * d->H * d->W;
        probe.flops += 2.0 * 2.0 * px * d->K * d->C * 9.0;                              // both products, every tap
        probe.bytes += 4.0 * (2.0 * px * d->C + px * d->K + 2.0 * (double)d->K * d->C * 9.0);   // dy, x, dx, filter, dw once each
    }
    *done = true;
    if (b.splits > 1 && open_dw && b.quads) {   // the caller's next call adds the copies
        open_dw->partial = partial_b;
        open_dw->splits = b.splits;
        open_dw->elems = b.out_elems;
        open_dw->value = dw;
        open_dw->lanes = wgrad_sum_lanes(b.out_elems / 4);
        open_split_set(partial_b);
    } else if (b.splits > 1) {
        if (int rc2 = wgrad_split_sum(b, partial_b, dw)) return rc2;
    }
    if (splits_a > 1 && open) {   // the caller's next call adds the copies
        open->partial = partial_a;
        open->splits = splits_a;
        open->elems = pc.out_elems;
        open->C = (size_t)pc.Mout;
        open->inner = (size_t)pc.OH * pc.OW;
        open->bias = nullptr;
        open->value = dx;
        open_split_set(partial_a);
        return DOPT_HIP_OK;
    }
    if (splits_a > 1)
        return launch_splitk_reduce(pc.out_elems, splits_a, partial_a, dx, nullptr, (unsigned)pc.Mout, (unsigned)(pc.OH * pc.OW));
    return DOPT_HIP_OK;
}

using WgradSquare = Tile<128, 128, 4, 2>;
using WgradNarrow = Tile<64, 128, 2, 4>;  // K <= 64: two workgroups per CU

}  // namespace

extern "C" {

int dopt_hip_conv_fwd(const dopt_hip_conv_desc *d, const float *x, const float *w, float *y)
{
    size_t P, Q;
    if (int rc = check_desc(d, &P, &Q, "dopt_hip_conv_fwd")) return rc;
    DOPT_REQUIRE(x && w && y, "dopt_hip_conv_fwd: null argument");
    DOPT_ENSURE_INIT();
    return run_gather<false>(d, P, Q, x, w, y);
}

int dopt_hip_conv_fwd_bias(const dopt_hip_conv_desc *d, const float *x, const float *w, const float *bias, float *y)
{
    size_t P, Q;
    if (int rc = check_desc(d, &P, &Q, "dopt_hip_conv_fwd_bias")) return rc;
    DOPT_REQUIRE(x && w && bias && y, "dopt_hip_conv_fwd_bias: null argument");
    DOPT_ENSURE_INIT();
    return run_gather<false>(d, P, Q, x, w, y, bias);
}

int dopt_hip_conv_bwd_data(const dopt_hip_conv_desc *d, const float *dy, const float *w, float *dx)
{
    size_t P, Q;
    if (int rc = check_desc(d, &P, &Q, "dopt_hip_conv_bwd_data")) return rc;
    DOPT_REQUIRE(dy && w && dx, "dopt_hip_conv_bwd_data: null argument");
    DOPT_ENSURE_INIT();
    return run_gather<true>(d, P, Q, dy, w, dx);
}

size_t dopt_hip_conv_packed_bytes(const dopt_hip_conv_desc *d, int bwd_data)
{
    size_t P, Q;
    if (check_desc(d, &P, &Q, "dopt_hip_conv_packed_bytes") || !ensure_init()) return 0;
    if (!bwd_data && conv_smallc_takes(d)) return 0;   // that forward kernel reads the filter as it is
    if (direct2x2_takes(d) || (!bwd_data && few_setup(d, P, Q).ok)) return d->K * d->C * d->R * d->S * sizeof(float);   // the filter as it is
    if (dense2x2_takes(d)) return dense2x2_elems(d) * sizeof(float);
    const PatchSetup u = bwd_data ? patch_setup<true>(d, P, Q) : patch_setup<false>(d, P, Q);
    // PackJob keeps strides in 32 bits
    return u.ok && d->C * 9 < (1ull << 32) ? u.wp_elems * sizeof(float) : 0;
}

int dopt_hip_conv_packed_layout(const dopt_hip_conv_desc *d, int bwd_data)
{
    if (dopt_hip_conv_packed_bytes(d, bwd_data) == 0) return -1;
    if (direct2x2_takes(d)) return 3;  // the filter itself: such kernels read [K][C][3][3], and a caller may pass the filter
    size_t P, Q;
    if (!bwd_data && check_desc(d, &P, &Q, "dopt_hip_conv_packed_layout") == 0 && few_setup(d, P, Q).ok) return 3;
    if (dense2x2_takes(d)) return 2;   // the same matrix, read transposed by backward-data
    return bwd_data ? 1 : 0;
}

int dopt_hip_conv_pack_batch(int n, const dopt_hip_conv_desc *descs, const int *bwd_data, const float *const *w,
                             float *const *packed)
{
    if (n == 0) return DOPT_HIP_OK;
    DOPT_REQUIRE(n > 0 && descs && bwd_data && w && packed, "dopt_hip_conv_pack_batch: null argument");
    DOPT_ENSURE_INIT();
    PackBatch b{};
    unsigned blocks = 0;
    auto flush = [&]() -> int {
        if (b.njobs == 0) return DOPT_HIP_OK;
        hipLaunchKernelGGL(pack_batch_k, dim3(blocks), dim3(256), 0, stream(), b);
        DOPT_LAUNCH_CHECK();
        b.njobs = 0;
        blocks = 0;
        return DOPT_HIP_OK;
    };
    for (int i = 0; i < n; i++) {
        size_t P, Q;
        if (int rc = check_desc(&descs[i], &P, &Q, "dopt_hip_conv_pack_batch")) return rc;
        DOPT_REQUIRE(w[i] && packed[i] && aligned16(packed[i]), "dopt_hip_conv_pack_batch: filter %d: null or unaligned pointer", i);
        if (dopt_hip_conv_packed_layout(&descs[i], bwd_data[i]) == 3) {   // "packed" is a plain copy (callers that know pass the filter itself instead)
            if (int rc = flush()) return rc;
            if (packed[i] != w[i])
                if (int rc = dopt_hip_copy_d2d(packed[i], w[i], descs[i].K * descs[i].C * descs[i].R * descs[i].S * sizeof(float))) return rc;
            continue;
        }
        if (dense2x2_takes(&descs[i]) && !(!bwd_data[i] && conv_smallc_takes(&descs[i]))) {
            if (int rc = dense2x2_pack(&descs[i], w[i], packed[i])) return rc;   // a launch of its own: the matrix is large
            continue;
        }
        const PatchSetup u = bwd_data[i] ? patch_setup<true>(&descs[i], P, Q) : patch_setup<false>(&descs[i], P, Q);
        DOPT_REQUIRE(u.ok && dopt_hip_conv_packed_bytes(&descs[i], bwd_data[i]) > 0,
                     "dopt_hip_conv_pack_batch: convolution %d does not take a packed filter", i);
        PackJob j = bwd_data[i] ? pack_job<true>(&descs[i], u, w[i], packed[i]) : pack_job<false>(&descs[i], u, w[i], packed[i]);
        j.first_block = blocks;
        blocks += j.mblocks * (unsigned)u.pc.chunks_total;
        b.job[b.njobs++] = j;
        if (b.njobs == kPackJobs)
            if (int rc = flush()) return rc;
    }
    return flush();
}

int dopt_hip_conv_fwd_bias_packed_open(const dopt_hip_conv_desc *d, const float *x, const float *packed,
                                       const float *bias, float *y, dopt_hip_split_sum *open)
{
    size_t P, Q;
    if (open) {   // complete unless a kernel below leaves parts
        *open = dopt_hip_split_sum{};
        open->value = y;
    }
    if (int rc = check_desc(d, &P, &Q, "dopt_hip_conv_fwd_bias_packed")) return rc;
    DOPT_REQUIRE(x && packed && y, "dopt_hip_conv_fwd_bias_packed: null argument");
    DOPT_ENSURE_INIT();
    if (dopt_hip_conv_packed_layout(d, 0) == 3) {
        bool done = false;
        if (int rc = run_few(d, P, Q, x, packed, bias, y, &done, open)) return rc;
        if (done) return DOPT_HIP_OK;
        if (int rc = run_direct2x2<false>(d, x, packed, bias, y, &done)) return rc;
        if (done) return DOPT_HIP_OK;
        return run_dense2x2<false>(d, x, packed, nullptr, bias, y);   // operands it cannot read as quads: from the filter
    }
    if (dopt_hip_conv_packed_layout(d, 0) == 2) return run_dense2x2<false>(d, x, nullptr, packed, bias, y);
    bool done = false;
    if (int rc = run_patch<false>(d, P, Q, x, nullptr, bias, y, &done, packed, open)) return rc;
    DOPT_REQUIRE(done, "dopt_hip_conv_fwd_bias_packed: this convolution does not take a packed filter");
    return DOPT_HIP_OK;
}

int dopt_hip_conv_fwd_bias_packed(const dopt_hip_conv_desc *d, const float *x, const float *packed, const float *bias,
                                  float *y)
{
    return dopt_hip_conv_fwd_bias_packed_open(d, x, packed, bias, y, nullptr);
}

int dopt_hip_conv_bwd_data_packed_open(const dopt_hip_conv_desc *d, const float *dy, const float *packed, float *dx,
                                       dopt_hip_split_sum *open)
{
    size_t P, Q;
    if (open) {
        *open = dopt_hip_split_sum{};
        open->value = dx;
    }
    if (int rc = check_desc(d, &P, &Q, "dopt_hip_conv_bwd_data_packed")) return rc;
    DOPT_REQUIRE(dy && packed && dx, "dopt_hip_conv_bwd_data_packed: null argument");
    DOPT_ENSURE_INIT();
    if (dopt_hip_conv_packed_layout(d, 1) == 3) {
        bool done = false;
        if (int rc = run_direct2x2<true>(d, dy, packed, nullptr, dx, &done)) return rc;
        if (done) return DOPT_HIP_OK;
        return run_dense2x2<true>(d, dy, packed, nullptr, nullptr, dx);
    }
    if (dopt_hip_conv_packed_layout(d, 1) == 2) return run_dense2x2<true>(d, dy, nullptr, packed, nullptr, dx);
    bool done = false;
    if (int rc = run_patch<true>(d, P, Q, dy, nullptr, nullptr, dx, &done, packed, open)) return rc;
    DOPT_REQUIRE(done, "dopt_hip_conv_bwd_data_packed: this convolution does not take a packed filter");
    return DOPT_HIP_OK;
}

int dopt_hip_conv_bwd_data_packed(const dopt_hip_conv_desc *d, const float *dy, const float *packed, float *dx)
{
    return dopt_hip_conv_bwd_data_packed_open(d, dy, packed, dx, nullptr);
}

int dopt_hip_conv_bwd_pair_packed_open(const dopt_hip_conv_desc *d, const float *dy, const float *packed, const float *x,
                                       float *dx, float *dw, dopt_hip_split_sum *open, dopt_hip_split_sum *open_dw)
{
    size_t P, Q;
    if (int rc = check_desc(d, &P, &Q, "dopt_hip_conv_bwd_pair_packed_open")) return rc;
    DOPT_REQUIRE(dy && packed && x && dx && dw, "dopt_hip_conv_bwd_pair_packed_open: null argument");
    DOPT_ENSURE_INIT();
    if (open) {
        *open = dopt_hip_split_sum{};
        open->value = dx;
    }
    if (open_dw) {
        *open_dw = dopt_hip_split_sum{};
        open_dw->value = dw;
    }
    bool done = false;
    if (int rc = run_bwd_pair(d, P, Q, dy, packed, x, dx, dw, open, open_dw, &done)) return rc;
    if (done) return DOPT_HIP_OK;
    // not a pair the one-launch kernel takes: filter gradient first (it may use the workspace), then backward-data,
    // which may leave its result open in it
    if (int rc = dopt_hip_conv_bwd_filter(d, dy, x, dw)) return rc;
    if (open) return dopt_hip_conv_bwd_data_packed_open(d, dy, packed, dx, open);
    return dopt_hip_conv_bwd_data_packed(d, dy, packed, dx);
}

int dopt_hip_conv_pair_probe(int enable)
{
    DOPT_ENSURE_INIT();
    DOPT_REQUIRE(enable >= 0 && enable <= 2, "dopt_hip_conv_pair_probe: 0 off, 1 one-launch backward pairs, 2 Winograd launches");
    g_pair_probe.on = enable;
    if (enable) {
        g_pair_probe.used = 0;
        g_pair_probe.flops = g_pair_probe.bytes = 0.0;
    }
    return DOPT_HIP_OK;
}

int dopt_hip_conv_pair_probe_read(int *launches, double *total_us, double *flops, double *bytes)
{
    DOPT_REQUIRE(launches && total_us && flops && bytes, "dopt_hip_conv_pair_probe_read: null argument");
    DOPT_ENSURE_INIT();
    PairProbe &probe = g_pair_probe;
    double us = 0.0;
    for (size_t i = 0; i < probe.used; i++) {
        DOPT_HIP_CHECK(hipEventSynchronize(probe.events[i].second));
        float ms = 0.0f;
        DOPT_HIP_CHECK(hipEventElapsedTime(&ms, probe.events[i].first, probe.events[i].second));
        us += (double)ms * 1000.0;
    }
    *launches = (int)probe.used;
    *total_us = us;
    *flops = probe.flops;
    *bytes = probe.bytes;
    return DOPT_HIP_OK;
}

int dopt_hip_split_sum_close(const dopt_hip_split_sum *open)
{
    DOPT_REQUIRE(open != nullptr, "dopt_hip_split_sum_close: null argument");
    if (open->splits == 0) return DOPT_HIP_OK;
    DOPT_REQUIRE(open->splits > 1 && open->partial && open->value && open->elems % 4 == 0 &&
                     (open->lanes > 0 || (open->C > 0 && open->inner > 0)),
                 "dopt_hip_split_sum_close: malformed description");
    DOPT_ENSURE_INIT();
    open_split_clear(open->partial);
    if (open->lanes > 0) return launch_split_sum(open->elems / 4, open->splits, open->lanes, open->partial, open->value);
    return launch_splitk_reduce(open->elems, open->splits, open->partial, open->value, open->bias, (unsigned)open->C,
                                (unsigned)open->inner);
}

int dopt_hip_conv_bwd_filter_batch(int n, const dopt_hip_conv_desc *descs, const float *const *dy, const float *const *x,
                                   float *const *dw)
{
    DOPT_REQUIRE(n >= 0 && (n == 0 || (descs && dy && x && dw)), "dopt_hip_conv_bwd_filter_batch: null argument");
    DOPT_ENSURE_INIT();
    // the filter gradients of 2x2-image layers are one dense product each, all of the same kernel: up to 8 share a launch
    int i = 0;
    while (i < n) {
        int m = 0;
        size_t C[8], K[8], N[8];
        while (i + m < n && m < 8) {
            const dopt_hip_conv_desc *d = &descs[i + m];
            size_t P, Q;
            if (check_desc(d, &P, &Q, "dopt_hip_conv_bwd_filter_batch") || !dy[i + m] || !x[i + m] || !dw[i + m] ||
                conv_smallc_takes(d) || !dense2x2_takes(d))
                break;
            C[m] = d->C; K[m] = d->K; N[m] = d->N;
            m++;
        }
        clear_error();
        int rc = DOPT_HIP_OK;
        if (m >= 2 && sgemm_fold2x2_batch(m, C, K, N, x + i, dy + i, dw + i, &rc)) {
            if (rc) return rc;
            i += m;
            continue;
        }
        if (int rc1 = dopt_hip_conv_bwd_filter(&descs[i], dy[i], x[i], dw[i])) return rc1;
        i++;
    }
    return DOPT_HIP_OK;
}

int dopt_hip_conv_bwd_filter(const dopt_hip_conv_desc *d, const float *dy, const float *x, float *dw)
{
    size_t P, Q;
    if (int rc = check_desc(d, &P, &Q, "dopt_hip_conv_bwd_filter")) return rc;
    DOPT_REQUIRE(dy && x && dw, "dopt_hip_conv_bwd_filter: null argument");
    DOPT_ENSURE_INIT();
    {
        bool done = false;
        if (int rc = conv_smallc_wgrad(d, dy, x, dw, &done)) return rc;
        if (done) return DOPT_HIP_OK;
        if (dense2x2_takes(d)) return run_dense2x2_wgrad(d, dy, x, dw);
        if (int rc = run_wgrad_patch(d, dy, x, dw, &done)) return rc;
        if (done) return DOPT_HIP_OK;
    }
    FilterGrad f{};
    f.dy = dy;
    f.x = x;
    f.N = (int)d->N; f.C = (int)d->C; f.H = (int)d->H; f.W = (int)d->W;
    f.K = (int)d->K; f.P = (int)P; f.Q = (int)Q; f.R = (int)d->R; f.S = (int)d->S;
    f.padH = (int)d->padH; f.padW = (int)d->padW; f.strideH = (int)d->strideH; f.strideW = (int)d->strideW;
    const int taps = f.R * f.S;
    f.Cp = round_up(f.C, 16);
    f.ncols = taps * f.Cp;
    f.npix = f.N * f.P * f.Q;
    f.out_elems = (size_t)f.K * f.ncols;
    f.dy_bytes = (size_t)f.npix * f.K * sizeof(float);
    f.x_bytes = (size_t)f.N * f.C * f.H * f.W * sizeof(float);
    f.slabs_total = (f.npix + BK - 1) / BK;
    const bool big = f.K > 64;
    const int BM = big ? 128 : 64, BN = 128;
    f.mtiles = (f.K + BM - 1) / BM;
    f.ntiles = (f.ncols + BN - 1) / BN;
    const int tiles = f.mtiles * f.ntiles;
    // filter gradients are short and wide (small output, long pixel reduction): allow deep splits
    int splits = gather_splits(tiles, f.slabs_total, big ? num_cus() : 2 * num_cus(), BM, BN, f.out_elems, kGatherRate, 512, 3.0);
    f.slabs_per_split = (f.slabs_total + splits - 1) / splits;
    splits = (f.slabs_total + f.slabs_per_split - 1) / f.slabs_per_split;
    f.splits = splits;
    float *partial = (float *)workspace((size_t)splits * f.out_elems * sizeof(float));
    if (!partial) return DOPT_HIP_ERR_OOM;
    f.out = partial;
    // column groups of one tile that can fall on different taps
    int gw = BN;
    while (f.Cp % gw != 0) gw /= 2;  // largest power-of-two divisor of Cp not above BN (>= 16)
    const int tpt = BN / gw;         // 1, 2, 4 or 8
    dim3 grid(xcd_grid((unsigned)(tiles * splits)));
    auto run = [&](auto tile_tag) {
        using T = decltype(tile_tag);
        return tpt == 1 ? launch_wgrad<T, 1>(f, grid) : tpt == 2 ? launch_wgrad<T, 2>(f, grid) : tpt == 4 ? launch_wgrad<T, 4>(f, grid) : launch_wgrad<T, 8>(f, grid);
    };
    if (int rc = big ? run(WgradSquare{}) : run(WgradNarrow{})) return rc;
    return launch_wgrad_reduce(f.K, f.C, f.Cp, taps, splits, f.out_elems, partial, dw);
}

}  // extern "C"
