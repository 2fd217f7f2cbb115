// `matmul`: row-major C[M,N] = A[M,K] * B[K,N] in fp32 (alpha = 1, beta = 0, no transposes).
// Replaces cublasSgemm_v2 at cuda/source/dopt/cuda/math.d:234-235.
//
// The reference funnels far more than dense layers through matmul: every scalar or bias
// broadcast is a product with a ones vector (core/source/dopt/core/ops/basic.d:370-381,
// core/source/dopt/core/ops/package.d:96-103) and rank-2 row / column sums are products with a
// ones vector too (core/source/dopt/core/ops/math.d:257-279).  Those degenerate shapes are
// HBM-bound and get their own kernels here; everything else runs on matrix instructions: small outputs on the fp32 one, large
// ones on the bf16 one with each fp32 value split into three parts (mfma_core.h).
#include <vector>

#include "common.h"
#include "mfma_core.h"

namespace {

using namespace dopt;

constexpr int BK = 16;
constexpr int kGemmThreads = 256;

struct Gemm {
    const float *A, *B;
    float *C;  // or `splits` partial copies
    int M, N, K;
    int lda, ldb;  // row pitch of A and B as stored
    int mtiles, ntiles, slabs_total, slabs_per_split, splits;
    int slabs_per_pass;   // sgemm_rows_k: a split is added up in C in passes of so many slabs
    size_t out_elems;
};

// An operand tile is BR rows (of M or of N) by BK reduction steps, staged k-major in LDS:
// Xs[k][r].  In memory the operand is either "k-contiguous" -- element (r, k) at X[r*ld + k],
// which is A as given or B transposed -- or "r-contiguous" -- element (r, k) at X[k*ld + r],
// which is B as given or A transposed.
//   k-contiguous: 16 lanes run along k, 16 row groups; the LDS store does the transposition.
//   r-contiguous: float4 along r, copied straight into the k-major tile.
template <int BR>
struct KContig {
    static constexpr int N = BR / 16;
    float reg[N];
    __device__ void load(const float *X, int ld, int r_base, int r_max, int kk0, int k_max, int tid)
    {
        const int kl = tid & 15, r0 = tid >> 4;
        const bool kok = kk0 + kl < k_max;
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int r = r_base + r0 + 16 * i;
            reg[i] = (kok && r < r_max) ? X[(size_t)r * ld + kk0 + kl] : 0.0f;
        }
    }
    __device__ void store(float *Xs, int LD, int tid) const
    {
        const int kl = tid & 15, r0 = tid >> 4;
#pragma unroll
        for (int i = 0; i < N; i++) Xs[kl * LD + r0 + 16 * i] = reg[i];
    }
};

template <int BR, bool kVec>
struct RContig {
    static constexpr int N = BR * BK / 4 / kGemmThreads;
    float4 reg[N];
    __device__ void load(const float *X, int ld, int r_base, int r_max, int kk0, int k_max, int tid)
    {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int f = tid + kGemmThreads * i;
            const int row = f / (BR / 4), gr = r_base + (f % (BR / 4)) * 4;
            const int kk = kk0 + row;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (kk < k_max) {
                const float *src = X + (size_t)kk * ld + gr;
                if (kVec) {
                    if (gr < r_max) v = *(const float4 *)src;  // r_max % 4 == 0: a float4 never straddles the edge
                } else {
                    if (gr + 0 < r_max) v.x = src[0];
                    if (gr + 1 < r_max) v.y = src[1];
                    if (gr + 2 < r_max) v.z = src[2];
                    if (gr + 3 < r_max) v.w = src[3];
                }
            }
            reg[i] = v;
        }
    }
    __device__ void store(float *Xs, int LD, int tid) const
    {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int f = tid + kGemmThreads * i;
            *(float4 *)&Xs[(f / (BR / 4)) * LD + (f % (BR / 4)) * 4] = reg[i];
        }
    }
};

template <bool kCond, class T, class F>
struct Pick {
    using type = T;
};
template <class T, class F>
struct Pick<false, T, F> {
    using type = F;
};

// C = op(A) * op(B).  kTA: A is stored [K][M]; kTB: B is stored [N][K].
template <int BM, bool kTA, bool kTB, bool kVec>
__global__ __launch_bounds__(kGemmThreads, 2) void sgemm_k(Gemm p)
{
    constexpr int BN = BM == 128 ? 128 : 256, WN = BM == 128 ? 2 : 4;
    constexpr int LDA = BM + 4, LDB = BN + 4;
    __shared__ __attribute__((aligned(16))) float As[2][BK * LDA];
    __shared__ __attribute__((aligned(16))) float Bs[2][BK * LDB];

    // 1-D grid over (split, tile), tile fastest: the blocks an XCD receives work on neighbouring
    // tiles of the same slice of the reduction, whatever the ratio of tiles to splits
    unsigned L;
    const unsigned tiles = (unsigned)(p.mtiles * p.ntiles);
    if (!xcd_remap(blockIdx.x, tiles * (unsigned)p.splits, &L)) return;
    const int split = (int)(L / tiles);
    const unsigned tile = L - (unsigned)split * tiles;
    const int mt = (int)(tile % (unsigned)p.mtiles), nt = (int)(tile / (unsigned)p.mtiles);
    const int m0 = mt * BM, n0 = nt * BN;
    const int slab_begin = split * p.slabs_per_split;
    const int slab_end = min(slab_begin + p.slabs_per_split, p.slabs_total);

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm = w / WN, wn = w % WN;

    typename Pick<kTA, RContig<BM, kVec>, KContig<BM>>::type la;
    typename Pick<kTB, KContig<BN>, RContig<BN, kVec>>::type lb;
    auto load = [&](int slab) {
        la.load(p.A, p.lda, m0, p.M, slab * BK, p.K, tid);
        lb.load(p.B, p.ldb, n0, p.N, slab * BK, p.K, tid);
    };
    auto store = [&](int buf) {
        la.store(As[buf], LDA, tid);
        lb.store(Bs[buf], LDB, tid);
    };

    v16f acc[2][2];
    zero_acc(acc);
    load(slab_begin);
    store(0);
    __syncthreads();
    int cur = 0;
    for (int slab = slab_begin; slab < slab_end; ++slab) {
        const bool more = slab + 1 < slab_end;
        if (more) load(slab + 1);
        mma_slab<BK, LDA, LDB>(As[cur], Bs[cur], wm * 64, wn * 64, acc, lane);
        if (more) store(cur ^ 1);
        __syncthreads();
        cur ^= 1;
    }

    float *outp = p.C + (size_t)split * p.out_elems;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int col = n0 + wn * 64 + j * 32 + (lane & 31);
        if (col >= p.N) continue;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int m = m0 + wm * 64 + i * 32 + acc_row(v, lane);
                if (m < p.M) outp[(size_t)m * p.N + col] = acc[i][j][v];
            }
    }
}

// The same product on the bf16 matrix instructions (mfma_core.h): operands are split into three bf16 parts on their way
// into LDS.  Bound by the power the matrix cores may draw (4096 x 4096 x 4096: the cores busy 71 % of the cycles at 1.6 of
// 2.4 GHz), then by what a wavefront issues beside its matrix instructions - reading fragments, splitting, arranging
// operands - which must fit into the slots they leave (eight per instruction); it goes with the sides of a wavefront's
// tile.  Eight wavefronts of 128 x 64 in 256 x 256 tiles, one workgroup per CU: 1068 -> 640 us for 4096 x 4096 x 4096
// (129 -> 215 TFLOP/s); 64 x 64 in 128 x 256 and 256 x 128: 755 us; 64 x 32 in 128 x 128: 965 us, for outputs too small
// to give every CU a larger tile.  The smaller ones have registers for a second set of accumulators, the smallest for a third.
// In the largest tile half of the threads stage A, half B, each a block of four rows by four steps: of a k-contiguous operand four 16-byte
// pieces of four rows (four lanes per 64-byte row segment), of an r-contiguous one four 16-byte pieces of four steps
// (sixteen lanes per 256 bytes), which become the quads of four rows by naming the registers.
// It serves every product of more than 64 rows, whatever the operands' alignment and however they are transposed, so
// that one (M, N, K) always adds its terms in one order (a plan that reads a transposed operand in place gets the bits
// of the plan that copies it first).
//
// A row's 16 steps in LDS are a line of 128 bytes: four pieces of 16 bytes with the (h, m) parts of a quad each, then two
// pieces with the l parts of two quads each; piece p lies at place p ^ f(row), and the halves of an l piece change places
// with bit 3 of the row.  f exclusive-ors 4, 2 and 5 for the low three bits of the row, so that the lanes which the LDS
// serves in one cycle - one piece of eight rows or half a piece of sixteen when reading, four pieces of two rows four
// apart when writing - touch different banks (a pitch of 112 bytes without the exchange lost a quarter of the loop to
// conflicts).
constexpr int kRowBytes = 128, kRowsThreads = 512;
__device__ __forceinline__ int row_swap(int row) { return (row & 1) << 6 ^ (row & 2) << 4 ^ (row & 4) * 20; }   // 16 f(row)
__device__ __forceinline__ int hm_at(int row, int quad) { return row * kRowBytes + (16 * quad ^ row_swap(row)); }
__device__ __forceinline__ int l_at(int row, int quad)
{
    return row * kRowBytes + ((64 + 16 * (quad >> 1)) ^ row_swap(row)) + (8 * (quad & 1) ^ (row & 8));
}

// Loads go through a buffer resource: an element outside the tile's rows or past the end of the reduction is fetched
// from kOobOffset, where the hardware range check returns zero, so the loop holds no branch and every load of a slab is
// in flight at once (guarded plain loads compile to one exec-masked region each, with waits in between).
// Pieces are 16 bytes whatever their alignment, and the range check works dword by dword (measured), so a piece may also
// stick out of the buffer.  One that sticks out of the matrix without leaving the buffer brings rows nobody stores
// (r-contiguous) or steps past the end of the reduction (k-contiguous, K no multiple of four: kCut), which are zeroed.
template <bool kCut>
struct Stage3 {
    float4 q[4];        // kc: four steps of row i; else four rows of step i
    unsigned base;      // byte offset of the block at the slab's first step, or kOobOffset when it lies outside the matrix
    int left;           // kCut: steps of the loaded pieces that lie before the end of the reduction
    int k0, rows;       // the block's first step inside a slab; how many of its rows lie inside the matrix
    int hm, l;          // where the parts of its first row go
    unsigned step, line;   // bytes between consecutive steps; between pieces
    bool kc;
    __device__ void init(bool k_contig, int ld, int r_base, int r_max, int t)
    {
        kc = k_contig;
        line = (unsigned)ld * 4u;
        step = kc ? 4u : line;
        k0 = 4 * (t & 3);
        const int row = t >> 2 << 2, r = r_base + row;
        rows = r_max - r;
        hm = hm_at(row, t & 3);
        l = l_at(row, t & 3);
        base = rows > 0 ? (unsigned)r * (kc ? line : 4u) + (unsigned)k0 * step : kOobOffset;
    }
    // A slab wholly past the end of the reduction loads nothing (every offset out of range).
    __device__ void load(__amdgpu_buffer_rsrc_t rs, int k, int k_max)
    {
        const unsigned soff = (unsigned)k * step;
        const int steps = k_max - k - k0;
        const int pieces = !kc ? steps : steps > 0 ? rows : 0;
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = buffer_load_f32x4(rs, i < pieces ? base : kOobOffset, soff + i * line);
        if (kCut) left = kc ? steps : 4;
    }
    // Splits the four steps of the block's row e and stores them.
    __device__ void store(char *Xs, int e) const
    {
        auto pick = [&](int i) { const float4 v = q[i]; return e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w; };
        const float4 own = q[e], across = make_float4(pick(0), pick(1), pick(2), pick(3));
        float4 v = make_float4(kc ? own.x : across.x, kc ? own.y : across.y, kc ? own.z : across.z, kc ? own.w : across.w);
        if (kCut) v = make_float4(v.x, left > 1 ? v.y : 0.0f, left > 2 ? v.z : 0.0f, left > 3 ? v.w : 0.0f);
        v4u a;
        uint2 b;
        split_quad(make_float4(v.x * kSplitUp, v.y * kSplitUp, v.z * kSplitUp, v.w * kSplitUp), a, b);
        *(v4u *)(Xs + (hm ^ row_swap(e)) + e * kRowBytes) = a;
        *(uint2 *)(Xs + (l ^ row_swap(e)) + e * kRowBytes) = b;
    }
};

// WM x WN wavefronts of MI x NI 32 x 32 pieces each.
template <int WM_, int WN_, int MI_, int NI_>
struct RowsTile {
    static constexpr int WM = WM_, WN = WN_, MI = MI_, NI = NI_, BM = 32 * WM * MI, BN = 32 * WN * NI;
    static constexpr int kBuf = (BM + BN) * kRowBytes;   // a buffer: the lines of A, then those of B
    static constexpr bool kLow = MI * NI <= 4, kTotal = MI * NI <= 2;   // which sets of registers there are beside the accumulators
    static_assert(WM * WN * 64 == kRowsThreads && BM % 64 == 0 && BN % 64 == 0 && BM + BN <= kRowsThreads, "one block of four rows by four steps per thread");
};

template <class T, bool kTA, bool kTB, bool kCut>
__global__ __launch_bounds__(kRowsThreads, 2) void sgemm_rows_k(Gemm p)
{
    constexpr int MI = T::MI, NI = T::NI, kBuf = T::kBuf;
    extern __shared__ __attribute__((aligned(16))) char rows_lds[];

    unsigned L;
    const unsigned tiles = (unsigned)(p.mtiles * p.ntiles);
    if (!xcd_remap(blockIdx.x, tiles * (unsigned)p.splits, &L)) return;
    const int split = (int)(L / tiles);
    const unsigned tile = L - (unsigned)split * tiles;
    const int mt = (int)(tile % (unsigned)p.mtiles), nt = (int)(tile / (unsigned)p.mtiles);
    const int m0 = mt * T::BM, n0 = nt * T::BN;
    const int k_begin = split * p.slabs_per_split * BK;
    const int k_end = min(min(k_begin + p.slabs_per_split * BK, p.slabs_total * BK), p.K);

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, kh = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wm = w / T::WN, wn = w % T::WN;
    const int arow = wm * 32 * MI + l32, brow = wn * 32 * NI + l32;

    // low: the four smaller kinds of products, where there are registers for them
    // total: the finished passes, where there are registers for them too
    constexpr bool kLow = T::kLow, kTotal = T::kTotal;
    v16f acc[MI][NI], low[kLow ? MI : 1][kLow ? NI : 1], total[kTotal ? MI : 1][kTotal ? NI : 1];
    auto add_low = [&]() {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++)
#pragma unroll
                for (int v = 0; v < 16; v++)
                    if (kLow) acc[i][j][v] += low[i % (kLow ? MI : 1)][j % (kLow ? NI : 1)][v];
    };
    auto add_total = [&]() {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[i][j][v] += total[i % (kTotal ? MI : 1)][j % (kTotal ? NI : 1)][v];
    };
    // Slab s is multiplied out of one LDS buffer in two groups of 3 MI NI matrix instructions (quads 0 and 1, quads 2 and 3).
    // Between them slab s + 1, fetched an iteration ago, is split and stored into the other buffer, and slab s + 2 is
    // requested.  A group's fragments are read while the group before it is multiplied; those of the next slab's first
    // group after the one barrier of the slab, which stands a third into the second group: by then this slab has been
    // read whole and the next one is stored whole.  Loads behind the last slab fall out of range and fetch nothing, what
    // is made of them is never multiplied.
    // the first BM / 64 wavefronts stage A, the next BN / 64 stage B; wavefronts beyond repeat what the first ones do
    constexpr int kStagers = (T::BM + T::BN) / 64;
    const int sw = w < kStagers ? w : w - kStagers;
    const bool for_b = sw >= T::BM / 64;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(for_b ? p.B : p.A, (size_t)(for_b ? p.N : p.M) * p.K * sizeof(float));
    Stage3<kCut> st;
    st.init(kTA != kTB ? !kTA : for_b ? kTB : !kTA, for_b ? p.ldb : p.lda, for_b ? n0 : m0, for_b ? p.N : p.M,
            (for_b ? sw - T::BM / 64 : sw) * 64 + lane);
    char *const mine = rows_lds + (for_b ? T::BM * kRowBytes : 0);
    const int ahm = hm_at(arow, kh), al = l_at(arow, kh), bhm = hm_at(T::BM + brow, kh), bl = l_at(T::BM + brow, kh);
    // The fragments of a group: lane half kh takes quad 2g + kh of its rows.  Which quad differs from quad kh's place by
    // an exclusive or, made here so that the addresses do not hold registers.
    v4u fa[2][MI], fb[2][NI];
    uint2 la[MI], lb[NI];
    auto read_hm = [&](const char *buf, int g) {
        int x = 32 * g;
        asm volatile("" : "+s"(x));
        const char *const pa = buf + (ahm ^ x), *const pb = buf + (bhm ^ x);
#pragma unroll
        for (int i = 0; i < MI; i++) fa[g][i] = *(const v4u *)(pa + 32 * i * kRowBytes);
#pragma unroll
        for (int j = 0; j < NI; j++) fb[g][j] = *(const v4u *)(pb + 32 * j * kRowBytes);
    };
    auto read_l = [&](const char *buf, int g) {
        int x = 16 * g;
        asm volatile("" : "+s"(x));
        const char *const pa = buf + (al ^ x), *const pb = buf + (bl ^ x);
#pragma unroll
        for (int i = 0; i < MI; i++) la[i] = *(const uint2 *)(pa + 32 * i * kRowBytes);
#pragma unroll
        for (int j = 0; j < NI; j++) lb[j] = *(const uint2 *)(pb + 32 * j * kRowBytes);
    };
    // The matrix instructions of group g, in three parts: (l, h) . (h, l), (h, m) . (m, h), (h, m) . (h, m)
    auto part = [&](int g, int kind) {
        v4u b[NI];
#pragma unroll
        for (int j = 0; j < NI; j++) {
            const v4u h = fb[g][j];
            b[j] = kind == 0 ? h : kind == 1 ? v4u{h.z, h.w, h.x, h.y} : v4u{h.x, h.y, lb[j].x, lb[j].y};
        }
#pragma unroll
        for (int i = 0; i < MI; i++) {
            const v4u a = kind < 2 ? fa[g][i] : v4u{la[i].x, la[i].y, fa[g][i].x, fa[g][i].y};
#pragma unroll
            for (int j = 0; j < NI; j++) {
                v16f &c = kLow && kind ? low[i % (kLow ? MI : 1)][j % (kLow ? NI : 1)] : acc[i][j];
                c = mfma_bf16(a, b[j], c);
            }
        }
    };
    float *const outp = p.C + (size_t)split * p.out_elems + (size_t)(m0 + wm * 32 * MI) * p.N + n0 + brow;
    const bool whole = m0 + T::BM <= p.M && n0 + T::BN <= p.N;
    // C = the accumulators, plus what C holds when `add`; no guards inside the matrix, and a block's loads go out together
    auto put = [&](bool add) {
        int pitch = p.N;
        asm volatile("" : "+s"(pitch));   // no row address is held across the reduction
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++) {
                float *const at = outp + (size_t)(i * 32 + 4 * kh) * pitch + 32 * j;
                if (whole) {
                    float old[16];
                    if (add) {
#pragma unroll
                        for (int v = 0; v < 16; v++) old[v] = at[(size_t)(8 * (v >> 2) + (v & 3)) * pitch];
#pragma unroll
                        for (int v = 0; v < 16; v++) acc[i][j][v] += old[v];
                    }
#pragma unroll
                    for (int v = 0; v < 16; v++) at[(size_t)(8 * (v >> 2) + (v & 3)) * pitch] = acc[i][j][v];
                } else {
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const int m = m0 + wm * 32 * MI + i * 32 + acc_row(v, lane);
                        float *const c = at + (size_t)(8 * (v >> 2) + (v & 3)) * pitch;
                        if (m < p.M && n0 + brow + 32 * j < p.N) *c = add ? *c + acc[i][j][v] : acc[i][j][v];
                    }
                }
            }
    };
    // A split's sum is formed in passes (sgemm_route says how long they are), all but the last of which wait in `total` or in C.
    float top = 0.0f;   // NaN once anything is not finite: x * 0 is 0 for finite x only
#pragma clang loop unroll(disable)
    for (int from = k_begin, to; from < k_end; from = to) {
        to = kTotal ? k_end : min(from + p.slabs_per_pass * BK, k_end);
        int left = p.slabs_per_pass;   // kTotal: slabs until the end of the pass
        zero_acc(acc);
        zero_acc(low);
        zero_acc(total);
        st.load(rs, from, to);
#pragma unroll
        for (int e = 0; e < 4; e++) st.store(mine, e);
        st.load(rs, from + BK, to);
        __syncthreads();
        read_hm(rows_lds, 0);
        read_l(rows_lds, 0);
        for (int k0 = from; k0 < to; k0 += 2 * BK) {
#pragma unroll
            for (int cur = 0; cur < 2; cur++) {
                if (cur && k0 + BK >= to) break;   // uniform
                char *const now = rows_lds + cur * kBuf, *const next = mine + (cur ^ 1) * kBuf;
                st.store(next, 0);
                part(0, 2);
                __builtin_amdgcn_sched_barrier(0);
                read_hm(now, 1);
                st.store(next, 1);
                part(0, 1);
                __builtin_amdgcn_sched_barrier(0);
                read_l(now, 1);
                st.store(next, 2);
                part(0, 0);
                __builtin_amdgcn_sched_barrier(0);
                st.store(next, 3);
                st.load(rs, k0 + (cur + 2) * BK, to);
                part(1, 2);
                __syncthreads();
                read_hm(rows_lds + (cur ^ 1) * kBuf, 0);
                part(1, 1);
                __builtin_amdgcn_sched_barrier(0);
                read_l(rows_lds + (cur ^ 1) * kBuf, 0);
                part(1, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (kTotal && --left == 0) {   // uniform
                    add_low();
                    add_total();
#pragma unroll
                    for (int i = 0; i < (kTotal ? MI : 1); i++)
#pragma unroll
                        for (int j = 0; j < (kTotal ? NI : 1); j++) total[i][j] = acc[i][j];
                    zero_acc(acc);
                    zero_acc(low);
                    left = p.slabs_per_pass;
                }
            }
        }
        __syncthreads();   // the buffers are free for the next pass
        add_low();
        if (kTotal) add_total();
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    top = __fmaf_rn(acc[i][j][v], 0.0f, top);
                    acc[i][j][v] *= kSplitDown;
                }
        put(from != k_begin);
    }
    if (!__any(top != 0.0f)) return;
    {   // an operand or a sum that is not finite: this wavefront's part in fp32 instructions, of which those values are taken that
        // are not finite in C (the others have the bits that they have beside finite ones, whatever tile they lie in)
        const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.A, (size_t)p.M * p.K * sizeof(float));
        const __amdgpu_buffer_rsrc_t rb = make_rsrc(p.B, (size_t)p.K * p.N * sizeof(float));
        zero_acc(acc);
        for (int k = k_begin + kh; k - kh < k_end; k += 2) {
            float a[MI], b[NI];
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const int r = m0 + arow + 32 * i;
                const unsigned at = kTA ? (unsigned)k * (unsigned)p.lda + (unsigned)r : (unsigned)r * (unsigned)p.lda + (unsigned)k;
                a[i] = buffer_load_f32(ra, r < p.M && k < k_end ? at * 4u : kOobOffset, 0);
            }
#pragma unroll
            for (int j = 0; j < NI; j++) {
                const int c = n0 + brow + 32 * j;
                const unsigned bt = kTB ? (unsigned)c * (unsigned)p.ldb + (unsigned)k : (unsigned)k * (unsigned)p.ldb + (unsigned)c;
                b[j] = buffer_load_f32(rb, c < p.N && k < k_end ? bt * 4u : kOobOffset, 0);
            }
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NI; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int m = m0 + wm * 32 * MI + i * 32 + acc_row(v, lane);
                float *const c = outp + (size_t)(i * 32 + 4 * kh + 8 * (v >> 2) + (v & 3)) * p.N + 32 * j;
                if (m < p.M && n0 + brow + 32 * j < p.N && *c * 0.0f != 0.0f) *c = acc[i][j][v];
            }
}

// Small outputs (a dense layer at batch 128: 128 x 512 values from a 512-deep reduction).  The tile
// engine above would run four blocks plus a reduction launch; here one block owns a 32 x 32 tile of
// C, its eight wavefronts each take an eighth of K straight from memory into MFMA operands (no LDS
// staging: nothing is reused inside a 32-wide tile), and the eight partial tiles are summed through
// LDS in wavefront order.  Per step of 8 reductions a lane holds four k values for its row of A and
// four for its column of B; v_mfma_f32_32x32x2 number e pairs element e of lanes 0-31 (k = 8q + e)
// with element e of lanes 32-63 (k = 8q + 4 + e) - any pairing works as long as A and B agree.
//
// X is "k-contiguous" when element (r, k) sits at X[r * ld + k] (A as given, B transposed), else
// "r-contiguous" at X[k * ld + r].
//
// Loads go through buffer resources (an element outside the matrix or past the end of the wavefront's share of K
// comes from kOobOffset and reads as zero: no branch) and kSmallDepth steps are in flight per wavefront: with one
// step of prefetch every step waited a full memory latency, eight of them in a row for a 512-deep reduction -
// most of such a kernel's duration.  The order of the sums is that of the steps, whatever is in flight.
constexpr int kSmallWaves = 8, kSmallDepth = 4;
constexpr int kGroupJobs = 8;   // jobs one grouped launch may hold (its descriptions travel as kernel arguments)

// The lane's four reductions kk .. kk + 3 of row / column r.  `base`: byte offset of (r, reduction 0), or kOobOffset
// when r lies outside the matrix; `pitch`: bytes between consecutive reductions of an r-contiguous operand.
// A k-contiguous operand is loaded as one 16-byte piece whatever its alignment (see Stage3): word by word, each load touched a
// line per row, and [29 x 2146] x [2146 x 2424], B stored [2424][2146], took 49 us instead of 20.
template <bool kKContig>
__device__ __forceinline__ void small_load(__amdgpu_buffer_rsrc_t rs, unsigned base, unsigned pitch, int kk, int k_end,
                                           float (&v)[4])
{
    if (kKContig) {
        const float4 q = buffer_load_f32x4(rs, kk < k_end ? base + (unsigned)kk * 4u : kOobOffset, 0);
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = buffer_load_f32(rs, kk + e < k_end ? base + (unsigned)(kk + e) * pitch : kOobOffset, 0);
    }
}

// What the last pieces of a k-contiguous operand hold past the end of the reduction counts as zero.  kCut: a reduction of no
// multiple of four, whose last pieces do.
template <bool kKContig, bool kCut>
__device__ __forceinline__ float small_value(const float (&v)[4], int e, int kk, int k_end)
{
    return kKContig && kCut && e > 0 ? (kk + e < k_end ? v[e] : 0.0f) : v[e];
}

// kCut: a k-contiguous operand's rows are no whole quads.
template <bool kTA, bool kTB, bool kCut>
__device__ __forceinline__ void sgemm_small_body(int M, int N, int K, int lda, int ldb, int kslice, const float *A,
                                                 const float *B, float *C, const float *colbias, int bias_shift,
                                                 const float *rowvec, int relu, const float *mask, int bx, int by, int k0, int k1,
                                                 float (*red)[32 * 33])
{
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, r = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // the same in every lane: loop bounds stay scalar
    const int m0 = by * 32, n0 = bx * 32;
    const int row = m0 + r, col = n0 + r;
    const int k_begin = k0 + wave * kslice, k_end = min(k1, k_begin + kslice);   // the block's part of the reduction: [k0, k1)
    const __amdgpu_buffer_rsrc_t rsa = make_rsrc(A, (size_t)M * K * sizeof(float)), rsb = make_rsrc(B, (size_t)K * N * sizeof(float));
    // A is k-contiguous as given, B when it is read transposed
    const unsigned abase = row < M ? (kTA ? (unsigned)row * 4u : (unsigned)row * (unsigned)lda * 4u) : kOobOffset;
    const unsigned bbase = col < N ? (kTB ? (unsigned)col * (unsigned)ldb * 4u : (unsigned)col * 4u) : kOobOffset;
    const unsigned apitch = (unsigned)lda * 4u, bpitch = (unsigned)ldb * 4u;

    v16f acc;
#pragma unroll
    for (int v = 0; v < 16; v++) acc[v] = 0.0f;
    float a[kSmallDepth][4], b[kSmallDepth][4];
    const int nsteps = k_begin < k_end ? (k_end - k_begin + 7) / 8 : 0;
#pragma unroll
    for (int j = 0; j < kSmallDepth; j++) {   // steps past the end fetch nothing
        small_load<!kTA>(rsa, abase, apitch, k_begin + 8 * j + 4 * half, k_end, a[j]);
        small_load<kTB>(rsb, bbase, bpitch, k_begin + 8 * j + 4 * half, k_end, b[j]);
        __builtin_amdgcn_sched_barrier(0);   // in this order: the first step's operands are waited for first
    }
    auto value_a = [&](int j, int s, int e) { return small_value<!kTA, kCut>(a[j], e, k_begin + 8 * (s + j) + 4 * half, k_end); };
    auto value_b = [&](int j, int s, int e) { return small_value<kTB, kCut>(b[j], e, k_begin + 8 * (s + j) + 4 * half, k_end); };
    // Whole rounds of kSmallDepth steps without a branch inside (a branch per step made the compiler wait for every
    // load in flight at the top of the loop), then the steps left over, whose operands are in their registers or on
    // their way already.
    const int whole = nsteps / kSmallDepth * kSmallDepth;
    for (int s = 0; s < whole; s += kSmallDepth) {
#pragma unroll
        for (int j = 0; j < kSmallDepth; j++) {
#pragma unroll
            for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(value_a(j, s, e), value_b(j, s, e), acc, 0, 0, 0);
            const int kk = k_begin + 8 * (s + j + kSmallDepth) + 4 * half;   // this register set's next step
            small_load<!kTA>(rsa, abase, apitch, kk, k_end, a[j]);
            small_load<kTB>(rsb, bbase, bpitch, kk, k_end, b[j]);
            __builtin_amdgcn_sched_barrier(0);   // keep each refill behind its own step: sunk to the loop's end, all of them are waited for at once
        }
    }
#pragma unroll
    for (int j = 0; j < kSmallDepth - 1; j++)
        if (whole + j < nsteps) {
#pragma unroll
            for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(value_a(j, whole, e), value_b(j, whole, e), acc, 0, 0, 0);
        }
#pragma unroll
    for (int v = 0; v < 16; v++) red[wave][acc_row(v, lane) * 33 + r] = acc[v];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int idx = tid + i * 64 * kSmallWaves, rr = idx >> 5, cc = idx & 31;
        float sum = red[0][rr * 33 + cc];
#pragma unroll
        for (int w = 1; w < kSmallWaves; w++) sum += red[w][rr * 33 + cc];
        if (m0 + rr < M && n0 + cc < N) {
            if (colbias) {   // one value per group of 2^bias_shift columns, times the row's factor when there is one
                float add = colbias[(n0 + cc) >> bias_shift];
                if (rowvec) add = __fmul_rn(rowvec[m0 + rr], add);   // rounded on its own, as the separate product is
                sum += add;
            }
            if (relu) sum = sum < 0.0f ? 0.0f : sum;
            if (mask) sum = mask[(size_t)(m0 + rr) * N + n0 + cc] > 0.0f ? sum : 0.0f;   // reluGrad(product, ., mask)
            C[(size_t)(m0 + rr) * N + n0 + cc] = sum;
        }
    }
}

// blockIdx.z: the part of the reduction (8 kslice steps each); the parts' sums go to consecutive copies of C.
template <bool kTA, bool kTB, bool kCut>
__global__ __launch_bounds__(64 * kSmallWaves) void sgemm_small_k(int M, int N, int K, int lda, int ldb, int kslice,
                                                                   const float *A, const float *B, float *C,
                                                                   const float *colbias, int bias_shift,
                                                                   const float *rowvec, int relu, const float *mask)
{
    __shared__ float red[kSmallWaves][32 * 33];
    const int k0 = (int)blockIdx.z * kSmallWaves * kslice;
    sgemm_small_body<kTA, kTB, kCut>(M, N, K, lda, ldb, kslice, A, B, C + (size_t)blockIdx.z * M * N, colbias, bias_shift, rowvec, relu,
                                     mask, (int)blockIdx.x, (int)blockIdx.y, k0, min(K, k0 + kSmallWaves * kslice), red);
}

// Short reductions over large outputs with both operands stored k-major (A as [K][M], B as [K][N]:
// the product x^T * dy of a filter gradient).  With K <= 128 a 128 x 128 output tile needs 128 KB of
// operands, which fit in LDS whole: every load of the block is issued before the first multiply, so
// the memory latency is paid once per tile instead of once per slab, and each operand byte enters
// the CU once per 128 x 128 outputs (a quarter of what 32 x 32 tiles fetch).  The reduction runs in
// four chunks of 32; a chunk is multiplied as soon as it is in LDS while the later ones are still
// in flight.  Eight wavefronts as 2 x 4, 64 x 32 outputs each.
constexpr int kPanelK = 128, kPanelTile = 128, kPanelThreads = 512, kPanelLd = kPanelTile + 4;
constexpr size_t kPanelLds = (size_t)2 * kPanelK * kPanelLd * sizeof(float);

// Element (k, r .. r + 3) of an operand stored [K][R] (R % 4 == 0, 16-byte aligned), zero outside.
__device__ __forceinline__ float4 panel_load(const float *X, int ld, int k, int K, int r, int R)
{
    return (k < K && r < R) ? *(const float4 *)(X + (size_t)k * ld + r) : make_float4(0.f, 0.f, 0.f, 0.f);
}

// kFold: the product is the filter gradient of a 3x3, pad-1 convolution over 2x2 images written as a
// dense product -- row 4c + (input pixel), column 4k + (output pixel) -- and the kernel stores the
// nine tap sums of every (k, c) pair to C[k][c][3][3] instead of the 4 x 4 block itself: tap (a, b)
// collects the pixel pairs with 1 - iy + oy == a and 1 - ix + ox == b.
template <bool kFold>
__device__ __forceinline__ void sgemm_panel_body(int M, int N, int K, int mtiles, int ntiles, const float *A, const float *B,
                                                 float *C, unsigned bid)
{
    extern __shared__ __attribute__((aligned(16))) float panel_lds[];
    float *As = panel_lds, *Bs = panel_lds + kPanelK * kPanelLd;
    unsigned L;
    if (!xcd_remap(bid, (unsigned)(mtiles * ntiles), &L)) return;
    const int m0 = (int)(L % (unsigned)mtiles) * kPanelTile, n0 = (int)(L / (unsigned)mtiles) * kPanelTile;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wm = w >> 2, wn = w & 3;

    // chunk c = reduction steps [32c, 32c + 32): 1024 float4 per operand, two per thread
    float4 ra[4][2], rb[4][2];
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int f = tid + kPanelThreads * i, k = 32 * c + (f >> 5), r = (f & 31) * 4;
            ra[c][i] = panel_load(A, M, k, K, m0 + r, M);
            rb[c][i] = panel_load(B, N, k, K, n0 + r, N);
        }
    v16f acc[2][1];
    zero_acc(acc);
#pragma unroll
    for (int c = 0; c < 4; c++) {
        if (32 * c < K) {   // uniform
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int f = tid + kPanelThreads * i, o = (32 * c + (f >> 5)) * kPanelLd + (f & 31) * 4;
                *(float4 *)&As[o] = ra[c][i];
                *(float4 *)&Bs[o] = rb[c][i];
            }
            __syncthreads();
            mma_slab<32, kPanelLd, kPanelLd>(As + 32 * c * kPanelLd, Bs + 32 * c * kPanelLd, wm * 64, wn * 32, acc, lane);
        }
    }
    if constexpr (!kFold) {
        const int col = n0 + wn * 32 + (lane & 31);
        if (col < N) {
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int m = m0 + wm * 64 + i * 32 + acc_row(v, lane);
                    if (m < M) C[(size_t)m * N + col] = acc[i][0][v];
                }
        }
    } else {
        // the tile goes back through LDS (the operands are spent) so that one thread sees the 4 x 4
        // block of a (c, k) pair; threads run along c, which is contiguous in the filter gradient
        __syncthreads();
        float *tile = panel_lds;   // [128][kPanelLd]
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int v = 0; v < 16; v++)
                tile[(wm * 64 + i * 32 + acc_row(v, lane)) * kPanelLd + wn * 32 + (lane & 31)] = acc[i][0][v];
        __syncthreads();
        const int Cin = M / 4, Kout = N / 4;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int pair = tid + kPanelThreads * j, cl = pair & 31, kl = pair >> 5;
            const int c = m0 / 4 + cl, k = n0 / 4 + kl;
            if (c < Cin && k < Kout) {
                float q[4][4];   // [input pixel iy*2+ix][output pixel oy*2+ox]
#pragma unroll
                for (int pin = 0; pin < 4; pin++) {
                    const float4 v = *(const float4 *)&tile[(cl * 4 + pin) * kPanelLd + kl * 4];
                    q[pin][0] = v.x; q[pin][1] = v.y; q[pin][2] = v.z; q[pin][3] = v.w;
                }
                float *out = C + ((size_t)k * Cin + c) * 9;
#pragma unroll
                for (int a = 0; a < 3; a++)
#pragma unroll
                    for (int b = 0; b < 3; b++) {
                        float sum = 0.0f;
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
    }
}

template <bool kFold>
__global__ __launch_bounds__(kPanelThreads) void sgemm_panel_k(int M, int N, int K, int mtiles, int ntiles, const float *A,
                                                                const float *B, float *C)
{
    sgemm_panel_body<kFold>(M, N, K, mtiles, ntiles, A, B, C, blockIdx.x);
}

// Several such products in one launch (the filter gradients of consecutive 2x2-image layers wait for nothing but their
// own dy): job j owns the blocks from first[j] on, a multiple of 8 each, so a block's place among the XCDs is what it
// would be in a launch of its own.
struct PanelJob {
    int M, N, K, mtiles, ntiles;
    unsigned first;
    const float *A, *B;
    float *C;
};
struct PanelGroup {
    PanelJob j[kGroupJobs];
    int n;
};

template <bool kFold>
__global__ __launch_bounds__(kPanelThreads) void sgemm_panel_group_k(PanelGroup g)
{
    int j = 0;
    while (j + 1 < g.n && blockIdx.x >= g.j[j + 1].first) j++;
    const PanelJob &q = g.j[j];
    sgemm_panel_body<kFold>(q.M, q.N, q.K, q.mtiles, q.ntiles, q.A, q.B, q.C, blockIdx.x - q.first);
}

__global__ __launch_bounds__(256) void splitk_reduce_k(size_t n, int splits, const float *partial, float *out)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        // four loads in flight per round (indices clamped, surplus values dropped); adds in split order
        float acc = 0.f;
        const int last = splits - 1;
        for (int s = 0; s < splits; s += 4) {
            const float v0 = partial[(size_t)s * n + i], v1 = partial[(size_t)min(s + 1, last) * n + i];
            const float v2 = partial[(size_t)min(s + 2, last) * n + i], v3 = partial[(size_t)min(s + 3, last) * n + i];
            acc = (((acc + v0) + (s + 1 <= last ? v1 : 0.f)) + (s + 2 <= last ? v2 : 0.f)) + (s + 3 <= last ? v3 : 0.f);
        }
        out[i] = acc;
    }
}

// ... and the epilogue of sgemm_small_k behind it.
__global__ __launch_bounds__(256) void splitk_epilogue_k(size_t M, size_t N, int splits, const float *partial, float *out,
                                                          const float *colbias, int bias_shift, const float *rowvec, int relu,
                                                          const float *mask)
{
    const size_t n = M * N;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        float acc = 0.f;
        const int last = splits - 1;
        for (int s = 0; s < splits; s += 4) {
            const float v0 = partial[(size_t)s * n + i], v1 = partial[(size_t)min(s + 1, last) * n + i];
            const float v2 = partial[(size_t)min(s + 2, last) * n + i], v3 = partial[(size_t)min(s + 3, last) * n + i];
            acc = (((acc + v0) + (s + 1 <= last ? v1 : 0.f)) + (s + 2 <= last ? v2 : 0.f)) + (s + 3 <= last ? v3 : 0.f);
        }
        if (colbias) {
            const size_t row = i / N, col = i - row * N;
            float add = colbias[col >> bias_shift];
            if (rowvec) add = __fmul_rn(rowvec[row], add);
            acc += add;
        }
        if (relu) acc = acc < 0.0f ? 0.0f : acc;
        if (mask) acc = mask[i] > 0.0f ? acc : 0.0f;
        out[i] = acc;
    }
}

// K == 1: C[m][n] = a[m] * b[n] -- the broadcast product.  One rounding per element, so a
// product with 1.0f reproduces the broadcast value exactly.
__global__ __launch_bounds__(256) void outer_k(size_t M, size_t N, const float *a, const float *b, float *c)
{
    const size_t total = M * N;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const size_t m = i / N, n = i - m * N;
        c[i] = a[m] * b[n];
    }
}

// Matrix times vector, either way the matrix is stored, in one order: the reduction falls into slices of kGemvSlice steps; of a
// slice, chain l (of 64) adds the products l, l + 64, l + 128 .., the chains' sums meet in halves (l and l + 32, then l and
// l + 16 ..), and slices are added from the first on.  So a plan that reads a transposed matrix in place gets the bits of the
// plan that copies it first.  Bound by the matrix' bytes from a few MB on.
constexpr int kGemvSlice = 1024;

struct VectorEpilogue {   // + rowvec[row] * colbias[col >> shift], relu, mask, as sgemm_small_k's
    const float *colbias, *rowvec, *mask;
    int shift, relu;
    size_t N;   // columns of the result
    __device__ __forceinline__ float operator()(float sum, size_t i) const
    {
        if (colbias) {
            const size_t row = i / N, col = i - row * N;
            float add = colbias[col >> shift];
            if (rowvec) add = __fmul_rn(rowvec[row], add);
            sum += add;
        }
        if (relu) sum = sum < 0.0f ? 0.0f : sum;
        if (mask) sum = mask[i] > 0.0f ? sum : 0.0f;
        return sum;
    }
};

// The matrix is stored row by row along the reduction: a wavefront per result, a lane per chain.
// kSteps > 0: at most so many steps of 64, where all of the loops below is only what a wavefront has to go through.  Up to four one
// after the other (3 000 000 rows of 2 steps 437 us with the loops, 314 so; 30000 of 64 6.7 and 4.5, of 129 7.7 and 5.4), more all
// together (8333 rows of 512 4.5 us one after the other, 3.8 with the loops, 3.6 so; 6057 of 429 3.8, 3.8 and 3.1; 25648 of 272 9.1, 8.2 and 6.5).
template <int kSteps>
__global__ __launch_bounds__(256) void gemv_rows_k(size_t M, size_t K, const float *A, const float *b, float *c, VectorEpilogue ep)
{
    const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= M) return;
    const int lane = threadIdx.x & 63;
    const float *ar = A + row * K;
    if constexpr (kSteps > 0) {
        float acc = 0.0f;
        if constexpr (kSteps <= 4) {
            for (size_t k = lane; k < K; k += 64) acc += ar[k] * b[k];
        } else {
            const int last = (int)K - 1;
            float x[kSteps], y[kSteps];
#pragma unroll
            for (int u = 0; u < kSteps; u++) {   // (clamped, not branched)
                x[u] = ar[min(64 * u + lane, last)];
                y[u] = b[min(64 * u + lane, last)];
            }
#pragma unroll
            for (int u = 0; u < kSteps; u++)
                if (64 * u + lane <= last) acc += x[u] * y[u];
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
        if (lane == 0) c[row] = ep(acc, row);
        return;
    }
    float total = 0.0f;
    for (size_t k0 = 0; k0 < K; k0 += kGemvSlice) {
        const size_t k1 = min(K, k0 + kGemvSlice);
        float acc = 0.0f;
        size_t k = k0;
        for (; k + 512 <= k1; k += 512) {   // eight steps in flight
            float x[8], y[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                x[u] = ar[k + 64 * u + lane];
                y[u] = b[k + 64 * u + lane];
            }
#pragma unroll
            for (int u = 0; u < 8; u++) acc += x[u] * y[u];
        }
        // what is left, as many steps as there are
        const int left = (int)(k1 - k);
        float x[8], y[8];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (64 * u < left) {   // (the same in every lane)
                const size_t at = min(k + 64 * u + lane, k1 - 1);
                x[u] = ar[at];
                y[u] = b[at];
            }
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (64 * u + lane < left) acc += x[u] * y[u];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
        total = k0 == 0 ? acc : total + acc;
    }
    if (lane == 0) c[row] = ep(total, row);
}

// The matrix is stored [K][N]: a block of 256 threads folds one slice of 256 / kGroups columns, a thread every kGroups-th chain of a
// column, so that all halves but the last are added in its registers and one value a thread meets the others' in LDS (with
// neighbouring chains, all of which met there, 2855 columns of 64 steps 2.8 us, 2.5 so; 7182 of 799 9.7 and 8.9).  kLive: a reduction of so many steps at most; chains
// beyond them are zeros that change nothing.
template <int kGroups, int kLive = kGemvSlice>
struct GemvLds {
    static constexpr int kCols = 256 / kGroups, kChains = (kLive < 64 ? kLive : 64) / kGroups;
    float sum[kGroups][kCols];
};
// (`on`: false for the threads of a larger block that only keep the barrier company)
template <int kGroups, int kLive = kGemvSlice, class Store>
__device__ __forceinline__ void gemv_cols_body(int K, int N, const float *a, const float *B, int bx, int k0, bool on, GemvLds<kGroups, kLive> &lds, Store &&store)
{
    constexpr int kCols = GemvLds<kGroups, kLive>::kCols, kChains = GemvLds<kGroups, kLive>::kChains;
    constexpr int kSteps = kLive > 64 && kChains < 16 ? 16 / kChains : 1;   // sixteen loads in flight
    const int col = threadIdx.x % kCols, g = threadIdx.x / kCols % kGroups, k1 = min(K, k0 + kGemvSlice);
    const int n = min(bx * kCols + col, N - 1);
    float acc[kChains];
#pragma unroll
    for (int j = 0; j < kChains; j++) acc[j] = 0.0f;
    if (on) {
        auto steps = [&](int k, auto whole) {   // (the last ones clamped, not branched)
            float av[kSteps][kChains], bv[kSteps][kChains];
#pragma unroll
            for (int u = 0; u < kSteps; u++)
#pragma unroll
                for (int j = 0; j < kChains; j++) {
                    const int step = k + 64 * u + kGroups * j + g, at = whole ? step : min(step, k1 - 1);
                    av[u][j] = a[at];
                    bv[u][j] = B[(size_t)at * N + n];
                }
#pragma unroll
            for (int u = 0; u < kSteps; u++)
#pragma unroll
                for (int j = 0; j < kChains; j++)
                    if (whole || k + 64 * u + kGroups * j + g < k1) acc[j] += av[u][j] * bv[u][j];
        };
        int k = k0;
        if constexpr (kLive > 64)
            for (; k + 64 * kSteps <= k1; k += 64 * kSteps) steps(k, std::true_type());
        if (kLive <= 64 || k < k1) steps(k, std::false_type());
    }
#pragma unroll
    for (int half = kChains / 2; half > 0; half >>= 1)   // chains 32 (fewer, if fewer are live) .. kGroups apart
#pragma unroll
        for (int j = 0; j < half; j++) acc[j] += acc[j + half];
    if (on && g > 0) lds.sum[g][col] = acc[0];
    __syncthreads();
    if (on && g == 0) {
        float s[kGroups];
        s[0] = acc[0];
#pragma unroll
        for (int i = 1; i < kGroups; i++) s[i] = lds.sum[i][col];
#pragma unroll
        for (int half = kGroups / 2; half > 0; half >>= 1)
#pragma unroll
            for (int i = 0; i < half; i++) s[i] += s[i + half];
        if (bx * kCols + col < N) store(bx * kCols + col, s[0]);
    }
}

// blockIdx.y: the slice.  With more than one their sums go to consecutive copies of the result, which splitk_epilogue_k adds
// (and `ep` does nothing).
template <int kGroups, int kLive>
__global__ __launch_bounds__(256) void gemv_cols_k(int K, int N, const float *a, const float *B, float *c, VectorEpilogue ep)
{
    __shared__ GemvLds<kGroups, kLive> lds;
    float *const to = c + (size_t)blockIdx.y * N;
    gemv_cols_body<kGroups, kLive>(K, N, a, B, (int)blockIdx.x, (int)blockIdx.y * kGemvSlice, true, lds,
                                   [&](int n, float v) { to[n] = ep(v, (size_t)n); });
}
// Eight groups, so that few columns make as many threads as they can.  Four where there are 64 columns a CU, a block of 64 for each
// (16913 columns of 679 steps 15.4 us with eight, 11.8 so; 22431 of 192 5.1 and 4.1; 14186 of 752 14.1 and 11.4, but 13302 of 244 4.1 and 4.7),
// but eight up to 96 columns a CU while they have all of the reduction in flight at once (18260 of 68 3.0 us with eight, 3.3 with four; 44921
// of 111 6.3 and 4.3), and for reductions of up to 64 steps, of which a thread takes no more chains than there are (3 000 000 columns of 2 steps 62 us
// with eight groups, 16 so; of 64 170 and 137; one group of all chains 13 and 139, but 300000 of 64 15.4, 13.8 with eight, 12.8 so).
constexpr int kGemvGroups = 8;

// Several independent small products in ONE launch: the weight and bias gradients of a dense head are six kernels of a
// few microseconds each that wait for nothing but the gradient in front of them, and a kernel boundary costs as much as
// one of them runs.  A block finds its job by its index; each job runs the body of the kernel it would have run alone
// (32 x 32-tile products of one template instance, and column sums of short reductions), so every value is what the
// separate launches give.
struct SmallJob {
    int M, N, K, lda, ldb, kslice, nx, first;   // nx: tiles per row of tiles; first: the job's first block
    const float *A, *B;
    float *C;
};
struct GemvJob {
    int K, N, first, pad;
    const float *a, *B;
    float *c;
};
struct SmallGroup {
    SmallJob s[kGroupJobs];
    GemvJob v[kGroupJobs];
    int ns, nv;
};

template <bool kTA, bool kTB, bool kCut>
__global__ __launch_bounds__(64 * kSmallWaves) void sgemm_small_group_k(SmallGroup g)
{
    __shared__ union {
        float red[kSmallWaves][32 * 33];
        GemvLds<kGemvGroups> gemv;
    } lds;
    const int b = (int)blockIdx.x;   // uniform: the scans below stay scalar
    if (g.nv > 0 && b >= g.v[0].first) {
        int j = 0;
        while (j + 1 < g.nv && b >= g.v[j + 1].first) j++;
        const GemvJob &q = g.v[j];
        gemv_cols_body<kGemvGroups>(q.K, q.N, q.a, q.B, b - q.first, 0, threadIdx.x < 256, lds.gemv, [&](int n, float v) { q.c[n] = v; });
        return;
    }
    int j = 0;
    while (j + 1 < g.ns && b >= g.s[j + 1].first) j++;
    const SmallJob &q = g.s[j];
    const int local = b - q.first;
    sgemm_small_body<kTA, kTB, kCut>(q.M, q.N, q.K, q.lda, q.ldb, q.kslice, q.A, q.B, q.C, nullptr, 0, nullptr, 0, nullptr,
                                     local % q.nx, local / q.nx, 0, q.K, lds.red);
}

// c[m][n] = relu?(c[m][n] + u[m] * v[n]): the epilogue of dopt_hip_sgemm_rank1 as a pass of its own, for the
// shapes whose product kernel has none.  Each step rounds on its own, like the separate operations.
__global__ __launch_bounds__(256) void rank1_epilogue_k(size_t M, size_t N, const float *u, const float *v, int relu, float *c)
{
    const size_t total = M * N;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const size_t m = i / N, n = i - m * N;
        float x = c[i];
        if (v) x += __fmul_rn(u[m], v[n]);
        if (relu) x = x < 0.0f ? 0.0f : x;
        c[i] = x;
    }
}

unsigned flat_grid(size_t n)
{
    size_t blocks = ceil_div(n, (size_t)256);
    size_t cap = (size_t)num_cus() * 16;
    return (unsigned)(blocks < 1 ? 1 : (blocks > cap ? cap : blocks));
}

// Steps of the reduction per wavefront of a 32 x 32-tile block that takes `depth` of them.
size_t small_slice(size_t depth) { return ceil_div(ceil_div(depth, (size_t)kSmallWaves), (size_t)8) * 8; }

// The LDS-resident kernel is taken where its 128 x 128 tiles give every CU one or two blocks and the operands take 128-bit loads.
// Against what those shapes take without it (an operand off the 16-byte grid): 2048 x 2048 x 64 11 and 18 us, 1024 x 4096 x
// 100 15 and 21, 2048 x 2048 x 128 17 and 17, 2880 x 2880 x 32 20 and 20; with two blocks on some CUs and 128 steps it is
// behind, 2816 x 2816 28 and 20, 2048 x 4096 27 and 20.
bool panel_shape(size_t M, size_t N, size_t K)
{
    const size_t tiles = ceil_div(M, (size_t)kPanelTile) * ceil_div(N, (size_t)kPanelTile);
    return K >= 1 && K <= (size_t)kPanelK && tiles >= (size_t)num_cus() && tiles <= (size_t)2 * num_cus() && M % 4 == 0 &&
           N % 4 == 0;
}

bool panel_takes(size_t M, size_t N, size_t K, const float *A, const float *B)
{
    return panel_shape(M, N, K) && aligned16(A) && aligned16(B);
}

int panel_launch(bool fold, size_t M, size_t N, size_t K, const float *A, const float *B, float *C)
{
    static bool raised = false;
    if (!raised) {   // above 64 KB of dynamic LDS a kernel has to be told once
        DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)sgemm_panel_k<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)kPanelLds));
        DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)sgemm_panel_k<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)kPanelLds));
        DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)sgemm_panel_group_k<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)kPanelLds));
        raised = true;
    }
    if (M == 0) return DOPT_HIP_OK;   // called for the attributes only
    const int mt = (int)ceil_div(M, (size_t)kPanelTile), nt = (int)ceil_div(N, (size_t)kPanelTile);
    const dim3 grid(xcd_grid((unsigned)(mt * nt))), block(kPanelThreads);
    if (fold) hipLaunchKernelGGL(sgemm_panel_k<true>, grid, block, kPanelLds, stream(), (int)M, (int)N, (int)K, mt, nt, A, B, C);
    else hipLaunchKernelGGL(sgemm_panel_k<false>, grid, block, kPanelLds, stream(), (int)M, (int)N, (int)K, mt, nt, A, B, C);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

// `n` folded filter-gradient products (all of them shapes panel_takes accepts) as one launch.
int panel_fold_group_launch(int n, const size_t *M, const size_t *N, const size_t *K, const float *const *A,
                            const float *const *B, float *const *C)
{
    if (int rc = panel_launch(true, 0, 0, 0, nullptr, nullptr, nullptr)) return rc;
    PanelGroup g{};
    unsigned blocks = 0;
    for (int i = 0; i < n; i++) {
        PanelJob &q = g.j[i];
        q.M = (int)M[i]; q.N = (int)N[i]; q.K = (int)K[i];
        q.mtiles = (int)ceil_div(M[i], (size_t)kPanelTile);
        q.ntiles = (int)ceil_div(N[i], (size_t)kPanelTile);
        q.first = blocks;
        q.A = A[i]; q.B = B[i]; q.C = C[i];
        blocks += xcd_grid((unsigned)(q.mtiles * q.ntiles));
    }
    g.n = n;
    hipLaunchKernelGGL(sgemm_panel_group_k<true>, dim3(blocks), dim3(kPanelThreads), kPanelLds, stream(), g);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

}  // namespace

namespace dopt {

// C[M,N] = op(A) * op(B) with op(X) = X or its transpose: transA means A is stored [K][M], transB
// means B is stored [N][K].

// C = op(A) * op(B), plus colbias[col >> bias_shift] on every element when colbias is given.  Returns
// *biased = false when the shape took a kernel without that epilogue (the caller adds the bias itself).
// What may ride in a product's epilogue besides the bias forms: a reluGrad mask (C = mask > 0 ? product : 0).
struct Extras {
    const float *mask = nullptr;
    bool written = false;   // see sgemm_route
};

// Whether a matrix times a vector finds the matrix stored row by row along the reduction (where both sides are vectors it does).
bool gemv_by_rows(int transA, int transB, size_t M, size_t N) { return (N == 1 && !transA) || (M == 1 && transB) || (M == 1 && N == 1); }

template <int kGroups, int kLive = kGemvSlice>
void launch_gemv_groups(int K, int N, size_t slices, const float *a, const float *B, float *c, const VectorEpilogue &ep)
{
    const dim3 grid((unsigned)ceil_div((size_t)N, (size_t)GemvLds<kGroups, kLive>::kCols), (unsigned)slices);
    hipLaunchKernelGGL((gemv_cols_k<kGroups, kLive>), grid, dim3(256), 0, stream(), K, N, a, B, c, ep);
}
int launch_gemv_cols(int K, int N, size_t slices, const float *a, const float *B, float *c, const VectorEpilogue &ep)
{
    if (K <= 16) launch_gemv_groups<4, 16>(K, N, slices, a, B, c, ep);
    else if (K <= 32) launch_gemv_groups<4, 32>(K, N, slices, a, B, c, ep);
    else if (K <= 64) launch_gemv_groups<4, 64>(K, N, slices, a, B, c, ep);
    else if (N >= (K <= 128 ? 96 : 64) * num_cus()) launch_gemv_groups<4>(K, N, slices, a, B, c, ep);
    else launch_gemv_groups<kGemvGroups>(K, N, slices, a, B, c, ep);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

int sgemm_epilogue(int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B, float *C,
                   const float *colbias, int bias_shift, const float *rowvec, int relu, bool *biased, const Extras &ex = Extras{});

int sgemm_bias(int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B, float *C,
               const float *colbias, int bias_shift, bool *biased)
{
    return sgemm_epilogue(transA, transB, M, N, K, A, B, C, colbias, bias_shift, nullptr, 0, biased);
}

// Which kernel a product takes and how it cuts the reduction: everything that decides the order in which an
// element's K terms are added.  It follows from the dimensions and the transposition flags alone - not from an epilogue
// being asked for, which a kernel without one leaves to a pass behind it; operand alignment picks between variants of a
// kernel that add in the same order (the LDS-resident kernel apart: panel_allowed = false is the route without it).
struct Route {
    enum Kind { kNone, kOuter, kGemv, kPanel = 5, kSmall, kTile64, kTile128, kRows, kRowsBig } kind;
    size_t cuts;    // partial sums per element that a second pass adds (gemv slices, tile-engine splits)
    size_t depth;   // reduction steps per partial sum (k per slice, slabs per split)
    size_t pass = 0;   // sgemm_rows_k: slabs that are added in its accumulators before they go to C
    size_t bm = 128, bn = 128;   // the tile engines' tile (no part of the order: every tile of a kind adds its elements' terms alike)
};

template <class T, bool kTA, bool kTB, bool kCut>
int rows_launch_one(dim3 grid, const Gemm &g)
{
    static bool raised = false;   // above 64 KB of dynamic LDS a kernel has to be told once
    if (!raised)
        DOPT_HIP_CHECK(hipFuncSetAttribute((const void *)sgemm_rows_k<T, kTA, kTB, kCut>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           2 * T::kBuf));
    raised = true;
    hipLaunchKernelGGL((sgemm_rows_k<T, kTA, kTB, kCut>), grid, dim3(kRowsThreads), 2 * T::kBuf, stream(), g);
    return DOPT_HIP_OK;
}

template <bool kTA, bool kTB, bool kCut>
int rows_launch(const Route &r, dim3 grid, const Gemm &g)
{
    if (r.bm == 256 && r.bn == 256) return rows_launch_one<RowsTile<2, 4, 4, 2>, kTA, kTB, kCut>(grid, g);
    if (r.bm == 256) return rows_launch_one<RowsTile<4, 2, 2, 2>, kTA, kTB, kCut>(grid, g);
    if (r.bn == 256) return rows_launch_one<RowsTile<2, 4, 2, 2>, kTA, kTB, kCut>(grid, g);
    return rows_launch_one<RowsTile<2, 4, 2, 1>, kTA, kTB, kCut>(grid, g);
}


// What a tile of sgemm_rows_k costs per 16 steps with every CU at work (4096 x 4096 x 4096: 630, 755 and 965 us); a
// workgroup's own start and end take about 4 us, split copies are written and read at about 5 TB/s, and another pass takes
// 3 us and its tile twice through a CU's 0.1 TB/s where it waits in C, half a microsecond where it waits in registers.
struct RowsShape {
    size_t bm, bn;
    double slab_us;
};
constexpr RowsShape kRowsShapes[] = {{256, 256, 2.4}, {128, 256, 1.45}, {256, 128, 1.45}, {128, 128, 0.93}};

// How many blocks share the reduction of a 32 x 32 tile: a few tiles over a long reduction leave most of the chip idle (a block
// takes 5.5 ns per step whatever runs beside it).  Another launch adds the parts.  [61 x 41] from 3673 steps: 21 us uncut, 8.6 in 29
// parts; [16 x 132] from 944 6.7 us uncut, 8.1 in eight.  The parts take no more space than the operands.  A round is one block per CU, as two
// on a CU share what it can load: [36 x 2052] from 4000 steps 22.6 us uncut, 29 in two parts (260 blocks), 22.4 in seven; [51 x 1500] from
// 3000 19.2 in three (282 blocks), 15.5 in five.
// `us`: what has to be undercut; `longest`: steps of a part.  Where rows off the 16-byte grid have raised `traffic_us` it hides what more
// parts give, so there they are also taken if they give half a microsecond without that ([64 x 640] from 8001 steps 24 us in three
// parts, 16 in six; [11 x 4459] from 5058 42 in two, 30 in five; [9 x 1538] from 4446 19 in two, 11 in five).
Route small_cuts(size_t M, size_t N, size_t K, size_t tiles, double traffic_us, double us, size_t longest = ~(size_t)0)
{
    Route r{Route::kSmall, 1, K, 0, 0, 0};
    const unsigned slots = (unsigned)num_cus(), k = (unsigned)K, t = (unsigned)tiles;
    const double copy_us = 8.0 * M * N / 5e6, grid_us = (double)tiles * 64 * K * sizeof(float) / 10e6;
    double on_grid = 0;
    for (unsigned cuts = 2; cuts <= 32; cuts++) {
        const unsigned depth = ((k + cuts - 1) / cuts + 63) / 64 * 64;
        if (depth < 128 || cuts * M * N > M * K + K * N) break;
        if (depth > longest || (k + depth - 1) / depth != cuts) continue;
        const unsigned rounds = (t * cuts + slots - 1) / slots;
        const double lasts = 5.5e-3 * depth * rounds, cost = 9.5 + std::max(traffic_us, lasts) + copy_us * cuts;
        const double even = std::max(grid_us, lasts) + copy_us * cuts;
        if (cost >= us && (r.cuts == 1 || even >= on_grid - 0.5)) continue;
        us = std::min(us, cost);
        on_grid = even;
        r.cuts = cuts;
        r.depth = depth;
    }
    return r;
}

// `written`: the product of a plan, whose reduction is cut the same however its operands are stored - one that reads a transposed
// matrix in place has to add its terms in the order of the product that was written, of a copy of it.
Route sgemm_route(int transA, int transB, size_t M, size_t N, size_t K, bool written, bool panel_allowed = true)
{
    Route r{Route::kNone, 1, K, 0, 0, 0};
    if (M * N == 0 || K == 0) return r;
    if (K == 1) { r.kind = Route::kOuter; return r; }
    if (M == 1 || N == 1) {   // matrix times vector: one order however the matrix is stored
        r.kind = Route::kGemv;
        r.depth = kGemvSlice;
        r.cuts = ceil_div(K, r.depth);
        return r;
    }
    // short reduction, both operands k-major, enough 128 x 128 tiles to fill the machine (alignment is checked at the
    // launch: the plan's buffers and every tensor of the pool are aligned)
    if (transA && !transB && panel_allowed && panel_shape(M, N, K)) { r.kind = Route::kPanel; return r; }
    // small and medium outputs: one block per 32 x 32 tile, the reduction split over its wavefronts.
    // Each tile reads its own 32 rows of A and 32 columns of B, so the operand traffic grows with the
    // number of tiles; it is served by the L2 at about 10 TB/s (1024 x 1024 x 256: 12 us against 20 us with the kernel
    // below), at half that when rows of a k-contiguous operand start off the 16-byte grid (91 x 1900 x 4674: 56 against 32 us).
    // A block by itself takes 5.5 ns per reduction step (256 x 256 x 8192: 49 against 28 us).
    const bool offsets32 = M * K < ((size_t)1 << 29) && K * N < ((size_t)1 << 29);
    const size_t tiles32 = ceil_div(M, (size_t)32) * ceil_div(N, (size_t)32);
    const double traffic = (double)tiles32 * 64 * K * sizeof(float);
    const bool small = offsets32 && tiles32 <= 4096 && traffic <= (double)(256 << 20);   // (32-bit byte offsets)
    // no operand's rows run along the reduction: whether that is whole quads changes nothing ([5112 x 19] from 2575 steps 30 us by
    // sgemm_rows_k, 24 in eleven parts here)
    const bool across = transA && !transB && !written;
    const double traffic_us = traffic / (K % 4 && !across ? 4.5e6 : 10e6);
    // (small_us, which decides between this kernel uncut and sgemm_rows_k, keeps the factor there too: without it [5112 x 19] ran here uncut in
    // 19 us, 3.3e-7 off float64 instead of 1.6e-7)
    const double small_us = 4 + (K % 4 ? 2 : 1) * std::max(traffic / 10e6, 5.5e-3 * K);
    const double uncut_us = across ? 4 + std::max(traffic / 10e6, 5.5e-3 * K) : small_us;
    const size_t slabs_total = ceil_div(K, (size_t)BK);
    if (M <= 64 || !offsets32) {
        if (small) return small_cuts(M, N, K, tiles32, traffic_us, uncut_us);
        r.kind = M <= 64 ? Route::kTile64 : Route::kTile128;
        r.bm = M <= 64 ? 64 : 128;
        r.bn = M <= 64 ? 256 : 128;
        const size_t tiles = ceil_div(M, r.bm) * ceil_div(N, r.bn);
        size_t splits = (2 * (size_t)num_cus() + tiles - 1) / tiles;
        if (splits > slabs_total / 4) splits = slabs_total / 4;
        if (splits > 32) splits = 32;
        if (splits < 1) splits = 1;
        r.depth = ceil_div(slabs_total, splits);
        r.cuts = ceil_div(slabs_total, r.depth);
        return r;
    }
    // How many steps may be added before a sum is rounded and put aside (a pass).  The bf16 instruction rounds down below its
    // guard bits, so a long sum drifts: 16384 products of non-negative values came out 1.2e-6 too small, 4096 by 2e-7.  And
    // no result is to be further off than with the fp32 instruction, for which the 32 x 32-tile kernel cuts a reduction in
    // eight and the tile engine cut it until there were two 128 x 128 tiles for each CU.  At equal lengths the error is 0.5
    // (A dense) to 0.7 (half of A zero, where the fp32 instruction rounds half as often) of the fp32 instruction's with the
    // small products in accumulators of their own, 0.7 to 1.15 with one accumulator: sums of twice and of half the length.
    // 469 x 5446 x 173, half of A zero, error against float64: fp32 8.7e-8, uncut 1.2e-7, so 8.3e-8 (25, 18 and 19 us);
    // 3818 x 1623 x 2673: 4.6e-7, 5.3e-7, 3.8e-7 (382, 199 and 234 us).
    const size_t tiles128 = ceil_div(M, (size_t)128) * ceil_div(N, (size_t)128);
    size_t finest = small ? (size_t)kSmallWaves : ceil_div((size_t)2 * num_cus(), tiles128);
    if (!small && finest > slabs_total / 4) finest = slabs_total / 4 ? slabs_total / 4 : 1;
    if (finest > 32) finest = 32;
    r.kind = Route::kRows;
    double best = 0;
    for (const RowsShape &t : kRowsShapes) {
        const size_t tiles = ceil_div(M, t.bm) * ceil_div(N, t.bn);
        const bool big = t.bm * t.bn == 256 * 256;
        if (big && K < 1024) continue;   // one accumulator per value: its passes have to be long
        size_t longest = big ? ceil_div(slabs_total, 2 * finest) : 2 * slabs_total / finest;
        if (longest > 4096 / BK) longest = 4096 / BK;
        if (longest < 1) longest = 1;
        for (size_t splits = 1; splits <= 32 && (splits == 1 || splits * 4 <= slabs_total); splits++) {
            const size_t depth = ceil_div(slabs_total, splits), cuts = ceil_div(slabs_total, depth);
            if (cuts != splits) continue;
            if (cuts > finest && cuts * M * N > M * K + K * N) break;   // more space than the operands take
            const size_t passes = ceil_div(depth, longest), pass = ceil_div(depth, passes);
            const double copy_us = (double)M * N * 4 / 5e6;
            const double pass_us = t.bm * t.bn == 128 * 128 ? 0.5 : 3 + t.bm * t.bn * 8 / 1e5;   // (the second through C)
            const double us = (double)ceil_div(tiles * cuts, (size_t)num_cus()) * (depth * t.slab_us + 4 + (passes - 1) * pass_us) +
                              copy_us * cuts + (cuts > 1 ? (cuts + 1) * copy_us + 5 : 0);
            if (best == 0 || us < best) {
                best = us;
                r.kind = big ? Route::kRowsBig : Route::kRows;
                r.bm = t.bm;
                r.bn = t.bn;
                r.depth = depth;
                r.cuts = cuts;
                r.pass = pass;
            }
        }
    }
    if (small && small_us < best) return small_cuts(M, N, K, tiles32, traffic_us, uncut_us);
    // Else the 32 x 32 tiles only where the reduction is cut into parts whose sums are as close as sgemm_rows_k's: 506 x 36 from 1127
    // steps 13 us and 1.2e-7 off float64; in parts of 256 steps 8 us and 1.2e-7; uncut 9 us and 2.2e-7.
    if (small) {
        const Route cut = small_cuts(M, N, K, tiles32, traffic_us, best, 256);
        if (cut.cuts > 1) return cut;
    }
    return r;
}

// The products with an epilogue: + rowvec[row] * colbias[col >> bias_shift] (rowvec optional), then relu.
// *biased says whether the kernel that ran applied it; if not, C holds the plain product.
int sgemm_epilogue(int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B, float *C,
                   const float *colbias, int bias_shift, const float *rowvec, int relu, bool *biased, const Extras &ex)
{
    *biased = false;
    if (M * N == 0) return DOPT_HIP_OK;
    DOPT_REQUIRE(C != nullptr, "dopt_hip_sgemm: C is null");
    DOPT_ENSURE_INIT();
    if (K == 0) return dopt_hip_memset(C, 0, M * N * sizeof(float));  // beta = 0
    DOPT_REQUIRE(A && B, "dopt_hip_sgemm: null operand");
    DOPT_REQUIRE(M < ((size_t)1 << 30) && N < ((size_t)1 << 30) && K < ((size_t)1 << 30) &&
                     M * N < ((size_t)1 << 40),
                 "dopt_hip_sgemm: dimensions too large");

    Route route = sgemm_route(transA, transB, M, N, K, ex.written);
    if (route.kind == Route::kPanel && !panel_takes(M, N, K, A, B))   // operands off the 16-byte grid: as if it were not there
        route = sgemm_route(transA, transB, M, N, K, ex.written, false);
    const Route::Kind kind = route.kind;
    if (kind == Route::kOuter) {  // vectors: a transposed vector is the same memory
        hipLaunchKernelGGL(outer_k, dim3(flat_grid(M * N)), dim3(256), 0, stream(), M, N, A, B, C);
        DOPT_LAUNCH_CHECK();
        return DOPT_HIP_OK;
    }
    if (kind == Route::kGemv) {
        const size_t R = N == 1 ? M : N, slices = route.cuts;
        const float *mat = N == 1 ? A : B, *vec = N == 1 ? B : A;
        const VectorEpilogue ep{colbias, rowvec, ex.mask, bias_shift, relu, N}, none{nullptr, nullptr, nullptr, 0, 0, 1};
        *biased = true;
        if (gemv_by_rows(transA, transB, M, N)) {
            const dim3 grid((unsigned)ceil_div(R, (size_t)4));
            if (K <= 256) hipLaunchKernelGGL(gemv_rows_k<4>, grid, dim3(256), 0, stream(), R, K, mat, vec, C, ep);
            else if (K <= 384) hipLaunchKernelGGL(gemv_rows_k<6>, grid, dim3(256), 0, stream(), R, K, mat, vec, C, ep);
            else if (K <= 512) hipLaunchKernelGGL(gemv_rows_k<8>, grid, dim3(256), 0, stream(), R, K, mat, vec, C, ep);
            else hipLaunchKernelGGL(gemv_rows_k<0>, grid, dim3(256), 0, stream(), R, K, mat, vec, C, ep);
            DOPT_LAUNCH_CHECK();
            return DOPT_HIP_OK;
        }
        float *to = C;
        if (slices > 1 && !(to = (float *)workspace(slices * R * sizeof(float)))) return DOPT_HIP_ERR_OOM;
        for (size_t s0 = 0; s0 < slices; s0 += 65535)   // (a grid's second dimension)
            if (int rc = launch_gemv_cols((int)(K - s0 * kGemvSlice), (int)R, std::min(slices - s0, (size_t)65535), vec + s0 * kGemvSlice,
                                          mat + s0 * kGemvSlice * R, to + s0 * R, slices > 1 ? none : ep))
                return rc;
        if (slices > 1) {
            hipLaunchKernelGGL(splitk_epilogue_k, dim3(flat_grid(R)), dim3(256), 0, stream(), M, N, (int)slices, to, C, colbias, bias_shift, rowvec, relu,
                               ex.mask);
            DOPT_LAUNCH_CHECK();
        }
        return DOPT_HIP_OK;
    }
    if (kind == Route::kPanel) return panel_launch(false, M, N, K, A, B, C);
    if (kind == Route::kSmall) {
        const int lda = (int)(transA ? M : K), ldb = (int)(transB ? K : N);
        const size_t cuts = route.cuts;
        const int kslice = (int)small_slice(route.depth);
        float *to = C;
        if (cuts > 1 && !(to = (float *)workspace(cuts * M * N * sizeof(float)))) return DOPT_HIP_ERR_OOM;
        const bool fused = cuts == 1;   // the epilogue runs behind the last sum
        const dim3 grid((unsigned)ceil_div(N, (size_t)32), (unsigned)ceil_div(M, (size_t)32), (unsigned)cuts), block(64 * kSmallWaves);
#define DOPT_SMALL(TA, TB, CUT)                                                                                          \
    hipLaunchKernelGGL((sgemm_small_k<TA, TB, CUT>), grid, block, 0, stream(), (int)M, (int)N, (int)K, lda, ldb, kslice, \
                       A, B, to, fused ? colbias : nullptr, bias_shift, fused ? rowvec : nullptr, fused ? relu : 0,      \
                       fused ? ex.mask : nullptr)
        const bool cut = K % 4 != 0;
        if (transA && transB) { if (cut) DOPT_SMALL(true, true, true); else DOPT_SMALL(true, true, false); }
        else if (transA) DOPT_SMALL(true, false, false);   // nothing k-contiguous to cut
        else if (transB) { if (cut) DOPT_SMALL(false, true, true); else DOPT_SMALL(false, true, false); }
        else { if (cut) DOPT_SMALL(false, false, true); else DOPT_SMALL(false, false, false); }
#undef DOPT_SMALL
        DOPT_LAUNCH_CHECK();
        if (!fused) {
            hipLaunchKernelGGL(splitk_epilogue_k, dim3(flat_grid(M * N)), dim3(256), 0, stream(), M, N, (int)cuts, to, C, colbias,
                               bias_shift, rowvec, relu, ex.mask);
            DOPT_LAUNCH_CHECK();
        }
        *biased = true;   // whatever epilogue was asked for (the extras included), it has been applied
        return DOPT_HIP_OK;
    }

    Gemm g{};
    g.A = A;
    g.B = B;
    g.M = (int)M;
    g.N = (int)N;
    g.K = (int)K;
    g.lda = (int)(transA ? M : K);
    g.ldb = (int)(transB ? K : N);
    g.out_elems = M * N;
    g.slabs_total = (int)ceil_div(K, (size_t)BK);
    const bool big = kind != Route::kTile64;
    g.mtiles = (int)ceil_div(M, route.bm);
    g.ntiles = (int)ceil_div(N, route.bn);
    const int tiles = g.mtiles * g.ntiles;
    const int splits = (int)route.cuts;
    g.slabs_per_split = (int)route.depth;
    g.slabs_per_pass = (int)route.pass;
    g.splits = splits;
    float *partial = nullptr;
    if (splits > 1) {
        partial = (float *)workspace((size_t)splits * g.out_elems * sizeof(float));
        if (!partial) return DOPT_HIP_ERR_OOM;
    }
    g.C = splits > 1 ? partial : C;
    // 128-bit loads for the operands stored with M (or N) contiguous
    const bool vec = (!transA || (M % 4 == 0 && aligned16(A))) && (transB || (N % 4 == 0 && aligned16(B)));
    dim3 grid(xcd_grid((unsigned)(tiles * splits)));
#define DOPT_SGEMM(BMV, TA, TB)                                                                               \
    do {                                                                                                      \
        if (vec) hipLaunchKernelGGL((sgemm_k<BMV, TA, TB, true>), grid, dim3(kGemmThreads), 0, stream(), g);   \
        else hipLaunchKernelGGL((sgemm_k<BMV, TA, TB, false>), grid, dim3(kGemmThreads), 0, stream(), g);      \
    } while (0)
#define DOPT_SGEMM_T(BMV)                                   \
    do {                                                    \
        if (!transA && !transB) DOPT_SGEMM(BMV, false, false); \
        else if (!transA) DOPT_SGEMM(BMV, false, true);     \
        else if (!transB) DOPT_SGEMM(BMV, true, false);     \
        else DOPT_SGEMM(BMV, true, true);                   \
    } while (0)
    if (kind == Route::kRows || kind == Route::kRowsBig) {
        const bool cut = K % 4 != 0;
#define DOPT_ROWS(TA, TB)                                                                                \
    do {                                                                                                 \
        if (int rc = cut ? rows_launch<TA, TB, true>(route, grid, g) : rows_launch<TA, TB, false>(route, grid, g)) return rc; \
    } while (0)
        if (!transA && !transB) DOPT_ROWS(false, false);
        else if (!transA) DOPT_ROWS(false, true);
        else if (!transB) { if (int rc = rows_launch<true, false, false>(route, grid, g)) return rc; }   // nothing k-contiguous to cut
        else DOPT_ROWS(true, true);
#undef DOPT_ROWS
    } else if (big) DOPT_SGEMM_T(128);
    else DOPT_SGEMM_T(64);
#undef DOPT_SGEMM_T
#undef DOPT_SGEMM
    DOPT_LAUNCH_CHECK();
    if (splits > 1) {
        hipLaunchKernelGGL(splitk_reduce_k, dim3(flat_grid(g.out_elems)), dim3(256), 0, stream(), g.out_elems, splits,
                           partial, C);
        DOPT_LAUNCH_CHECK();
    }
    return DOPT_HIP_OK;
}

// Filter gradient of a 3x3, pad-1, unit-stride convolution over 2x2 images in one launch:
// dw[K][C][3][3] from x[N][4C] and dy[N][4K].  Returns false (nothing launched) when the shape does
// not suit the LDS-resident kernel; the caller then takes the product and folds it itself.
bool sgemm_fold2x2(size_t C, size_t K, size_t N, const float *x, const float *dy, float *dw, int *rc)
{
    if (!panel_takes(4 * C, 4 * K, N, x, dy)) return false;
    *rc = panel_launch(true, 4 * C, 4 * K, N, x, dy, dw);
    return true;
}

// The same for `n` layers at once (n <= 8): one launch when every layer suits the LDS-resident kernel, else false with
// nothing launched.
bool sgemm_fold2x2_batch(int n, const size_t *C, const size_t *K, const size_t *N, const float *const *x,
                         const float *const *dy, float *const *dw, int *rc)
{
    if (n < 1 || n > kGroupJobs) return false;
    size_t M4[kGroupJobs], N4[kGroupJobs];
    for (int i = 0; i < n; i++) {
        if (!panel_takes(4 * C[i], 4 * K[i], N[i], x[i], dy[i])) return false;
        M4[i] = 4 * C[i];
        N4[i] = 4 * K[i];
    }
    *rc = panel_fold_group_launch(n, M4, N4, N, x, dy, dw);
    return true;
}

int product(bool written, int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B, float *C)
{
    Extras ex;
    ex.written = written;
    bool applied;
    return sgemm_epilogue(transA, transB, M, N, K, A, B, C, nullptr, 0, nullptr, 0, &applied, ex);
}

int product_batch(bool written, int n, const int *transA, const int *transB, const size_t *M, const size_t *N, const size_t *K, const float *const *A,
                  const float *const *B, float *const *C)
{
    DOPT_REQUIRE(n >= 0 && (n == 0 || (transA && transB && M && N && K && A && B && C)), "dopt_hip_sgemm_batch: null argument");
    DOPT_ENSURE_INIT();
    // Products that take the 32 x 32-tile kernel (grouped per template instance) or the short column sum share launches;
    // the others run one by one.  Outputs must not overlap any operand of the batch: the order inside it is not kept.
    struct Inst { bool ta, tb, cut; SmallGroup g; unsigned blocks; bool used; };
    std::vector<Inst> insts;
    std::vector<GemvJob> gemvs;
    std::vector<int> single;
    for (int i = 0; i < n; i++) {
        if (M[i] * N[i] == 0) continue;
        const bool plain = K[i] > 0 && A[i] && B[i] && C[i] && M[i] < ((size_t)1 << 30) && N[i] < ((size_t)1 << 30) && K[i] < ((size_t)1 << 30);
        const Route r = plain ? sgemm_route(transA[i], transB[i], M[i], N[i], K[i], written) : Route{Route::kNone, 1, 0, 0, 0, 0};
        if (r.kind == Route::kGemv && r.cuts == 1 && !gemv_by_rows(transA[i], transB[i], M[i], N[i]) && gemvs.size() < (size_t)kGroupJobs) {
            const size_t R = M[i] == 1 ? N[i] : M[i];
            GemvJob q{};
            q.K = (int)K[i]; q.N = (int)R;
            q.a = M[i] == 1 ? A[i] : B[i];
            q.B = M[i] == 1 ? B[i] : A[i];
            q.c = C[i];
            gemvs.push_back(q);
        } else if (r.kind == Route::kSmall && r.cuts == 1) {
            const int lda = (int)(transA[i] ? M[i] : K[i]), ldb = (int)(transB[i] ? K[i] : N[i]);
            const bool ta = transA[i] != 0, tb = transB[i] != 0, cut = K[i] % 4 != 0 && (!ta || tb);   // the instance the product would take alone
            Inst *in = nullptr;
            for (Inst &c : insts)
                if (c.ta == ta && c.tb == tb && c.cut == cut && c.g.ns < kGroupJobs) in = &c;
            if (!in) {
                insts.push_back(Inst{ta, tb, cut, SmallGroup{}, 0, false});
                in = &insts.back();
            }
            SmallJob &q = in->g.s[in->g.ns++];
            q.M = (int)M[i]; q.N = (int)N[i]; q.K = (int)K[i]; q.lda = lda; q.ldb = ldb;
            q.kslice = (int)small_slice(K[i]);
            q.nx = (int)ceil_div(N[i], (size_t)32);
            q.first = (int)in->blocks;
            q.A = A[i]; q.B = B[i]; q.C = C[i];
            in->blocks += (unsigned)(q.nx * ceil_div(M[i], (size_t)32));
        } else {
            single.push_back(i);
        }
    }
    for (size_t k = 0; k < insts.size(); k++) {
        Inst &in = insts[k];
        if (k == 0) {   // the column sums ride in the first launch
            for (const GemvJob &v : gemvs) {
                GemvJob &q = in.g.v[in.g.nv++];
                q = v;
                q.first = (int)in.blocks;
                in.blocks += (unsigned)ceil_div((size_t)v.N, (size_t)GemvLds<kGemvGroups>::kCols);
            }
            gemvs.clear();
        }
        const dim3 grid(in.blocks), block(64 * kSmallWaves);
#define DOPT_GROUP(TA, TB, CUT) hipLaunchKernelGGL((sgemm_small_group_k<TA, TB, CUT>), grid, block, 0, stream(), in.g)
        if (in.ta && in.tb) { if (in.cut) DOPT_GROUP(true, true, true); else DOPT_GROUP(true, true, false); }
        else if (in.ta) DOPT_GROUP(true, false, false);
        else if (in.tb) { if (in.cut) DOPT_GROUP(false, true, true); else DOPT_GROUP(false, true, false); }
        else { if (in.cut) DOPT_GROUP(false, false, true); else DOPT_GROUP(false, false, false); }
#undef DOPT_GROUP
        DOPT_LAUNCH_CHECK();
    }
    for (const GemvJob &v : gemvs) {   // no 32 x 32-tile launch to ride in
        if (int rc = launch_gemv_cols(v.K, v.N, 1, v.a, v.B, v.c, VectorEpilogue{nullptr, nullptr, nullptr, 0, 0, 1})) return rc;
    }
    for (int i : single)
        if (int rc = product(written, transA[i], transB[i], M[i], N[i], K[i], A[i], B[i], C[i])) return rc;
    return DOPT_HIP_OK;
}

int product_rank1(bool written, int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B, const float *u, const float *v, int relu,
                  float *C)
{
    DOPT_REQUIRE((u == nullptr) == (v == nullptr), "dopt_hip_sgemm_rank1: u and v go together");
    Extras ex;
    ex.written = written;
    bool applied = false;
    if (int rc = sgemm_epilogue(transA, transB, M, N, K, A, B, C, v, 0, u, relu, &applied, ex)) return rc;
    if (applied || M * N == 0 || (!v && !relu)) return DOPT_HIP_OK;
    hipLaunchKernelGGL(rank1_epilogue_k, dim3(flat_grid(M * N)), dim3(256), 0, stream(), M, N, u, v, relu, C);
    DOPT_LAUNCH_CHECK();
    return DOPT_HIP_OK;
}

int product_relu_grad(bool written, int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B, const float *x, float *C)
{
    DOPT_REQUIRE(x != nullptr || M * N == 0, "dopt_hip_sgemm_relu_grad: null argument");
    Extras ex;
    ex.mask = x;
    ex.written = written;
    bool applied = false;
    if (int rc = sgemm_epilogue(transA, transB, M, N, K, A, B, C, nullptr, 0, nullptr, 0, &applied, ex)) return rc;
    if (applied || M * N == 0) return DOPT_HIP_OK;
    return dopt_hip_relu_bwd(M * N, C, x, C);   // in place: every element is read before it is written
}

uint64_t product_order(bool written, int transA, int transB, size_t M, size_t N, size_t K)
{
    if (!ensure_init()) return 0;   // the cut of a reduction follows the device's size
    const Route r = sgemm_route(transA, transB, M, N, K, written);
    return (uint64_t)r.kind | (uint64_t)r.cuts << 8 | (uint64_t)r.depth << 24 | (uint64_t)r.pass << 52;
}

}  // namespace dopt

extern "C" {

int dopt_hip_sgemm_batch(int n, const int *transA, const int *transB, const size_t *M, const size_t *N, const size_t *K,
                         const float *const *A, const float *const *B, float *const *C)
{
    return product_batch(false, n, transA, transB, M, N, K, A, B, C);
}

int dopt_hip_sgemm_rank1(int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B,
                         const float *u, const float *v, int relu, float *C)
{
    return product_rank1(false, transA, transB, M, N, K, A, B, u, v, relu, C);
}

int dopt_hip_sgemm_relu_grad(int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B,
                             const float *x, float *C)
{
    return product_relu_grad(false, transA, transB, M, N, K, A, B, x, C);
}

uint64_t dopt_hip_sgemm_order(int transA, int transB, size_t M, size_t N, size_t K) { return product_order(false, transA, transB, M, N, K); }

int dopt_hip_sgemm_t(int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B, float *C)
{
    return product(false, transA, transB, M, N, K, A, B, C);
}

int dopt_hip_sgemm(size_t M, size_t N, size_t K, const float *A, const float *B, float *C)
{
    return dopt_hip_sgemm_t(0, 0, M, N, K, A, B, C);
}

}  // extern "C"
