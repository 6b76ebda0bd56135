// kernels_sample.hip -- multinomial sampling, bit-exact with the reference's
// streaming CPU sampler (reference src/zxh/src/measure/measure_general.cpp,
// measure_streaming_impl.h, measure_common.cpp).
//
// The reference builds, per segment of 2^I amplitudes, a CDF from a Blelloch
// exclusive scan of p_i = re^2 + im^2, offsets it by a binary-counter prefix
// of earlier segment totals, and resolves sorted thresholds with
// std::upper_bound.  Every value it compares is a node sum of ONE balanced
// binary tree over p (Blelloch up-sweep nodes, merge_prob_sum_range, and the
// binary counter all add left+right children of aligned power-of-two blocks),
// combined left to right in Fenwick order:
//     excl_j   = (((0 + N_{l1}[.]) + N_{l2}[.]) + ...)   set bits of j, high to low
//     prefix_s = same over segment indices, with levels >= I
//     cdf_j    = (prefix_s + excl_j) + p_j,   tail_s = prefix_s + N_I[s]
// So the GPU stores the tree levels >= LS (LS = min(4, I) for complex128,
// min(5, I) for complex64; lower levels are recomputed from the 256 bytes of
// amplitudes of a block: 16 complex128 or 32 complex64), and each shot performs
// libstdc++'s exact upper_bound probe sequence, evaluating cdf at each probe.
// A threshold belongs to the first segment whose running-max tail exceeds
// it, which is where the reference's sequential segment walk places it.
// No fused multiply-add is allowed anywhere on this path.
#include "dev.h"

#include <algorithm>
#include <cstring>
#include <functional>
#include <vector>

#pragma clang fp contract(off)

namespace zxa
{
namespace
{

constexpr int kThreads = 256;
constexpr int kSpanBits = 12; // input values per workgroup in the tree kernel
constexpr int kMaxLevels = 64;

struct Levels
{
    uint64_t off[kMaxLevels]; // offset of level l in the tree array (valid for LS <= l <= m)
};

__device__ __forceinline__ double p_of(const void *state, bool c64, uint64_t i)
{
    if (c64)
    {
        const float2 a = static_cast<const float2 *>(state)[i];
        const double x = a.x, y = a.y;
        return __dadd_rn(__dmul_rn(x, x), __dmul_rn(y, y));
    }
    const double2 a = static_cast<const double2 *>(state)[i];
    return __dadd_rn(__dmul_rn(a.x, a.x), __dmul_rn(a.y, a.y));
}

// One workgroup reduces up to 2^kSpanBits input values of level lin into the
// levels lin+1 .. lin+span_bits and stores every level in [LS, m] it owns.
// src_kind: 0 = c128 amplitudes, 1 = c64 amplitudes, 2 = tree nodes (f64).
// The root (level m) also goes to root[0] (host memory), and, when one segment
// is the whole state, to one[0..1] as that segment's prefix (0) and tail.
__global__ __launch_bounds__(kThreads) void tree_kernel(const void *__restrict__ src, int src_kind, int lin,
                                                        int span_bits, int LS, int m, double *__restrict__ tree,
                                                        const Levels lv, double *__restrict__ root,
                                                        double *__restrict__ one)
{
    __shared__ double buf[1 << kSpanBits];
    auto top = [&](double v) {
        if (root)
            root[0] = v;
        if (one)
        {
            one[0] = 0.0;
            one[1] = __dadd_rn(0.0, v);
        }
    };
    const int span = 1 << span_bits;
    const uint64_t g0 = static_cast<uint64_t>(blockIdx.x) << span_bits;
    for (int i = threadIdx.x; i < span; i += kThreads)
    {
        double v;
        if (src_kind == 2)
            v = static_cast<const double *>(src)[lv.off[lin] + g0 + i];
        else
            v = p_of(src, src_kind == 1, g0 + i);
        buf[i] = v;
        if (src_kind != 2 && lin >= LS)
            tree[lv.off[lin] + g0 + i] = v;
        if (lin == m)
            top(v);
    }
    __syncthreads();
    for (int r = 1; r <= span_bits; r++)
    {
        const int cnt = span >> r;
        const int l = lin + r;
        double vals[(1 << kSpanBits) / kThreads / 2 > 0 ? (1 << kSpanBits) / kThreads / 2 : 1];
        int nv = 0;
        for (int k = threadIdx.x; k < cnt; k += kThreads)
            vals[nv++] = __dadd_rn(buf[2 * k], buf[2 * k + 1]);
        __syncthreads();
        nv = 0;
        for (int k = threadIdx.x; k < cnt; k += kThreads)
        {
            const double v = vals[nv++];
            buf[k] = v;
            if (l >= LS && l <= m)
                tree[lv.off[l] + (g0 >> r) + k] = v;
            if (l == m)
                top(v);
        }
        __syncthreads();
    }
}

typedef double dvec2 __attribute__((ext_vector_type(2)));
typedef float fvec4 __attribute__((ext_vector_type(4)));

// tree_amp_kernel geometry: a wave tile is 16 loads of 16 bytes per lane,
// 1024 amplitudes (c128) or 2048 (c64); a workgroup holds four tiles.
template <bool kC64>
struct TreeGeo
{
    static constexpr int kTileBits = kC64 ? 11 : 10;
    static constexpr int kRounds = kC64 ? 2 : 1;     // 512 level-1 nodes per round
    static constexpr int kGroupBits = kTileBits + 2; // amplitudes per workgroup
};
constexpr int kRowPad = 9; // LDS doubles per row of 8 level-1 nodes (one pad)

// Orders this wave's LDS accesses (a wave executes in lockstep; the fences
// keep the compiler from moving accesses across the exchange).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The value of the neighbouring lane (lane ^ 1), by DPP quad permutation.
__device__ __forceinline__ double lane_xor1(double v)
{
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_mov_dpp(int(b), 0xB1, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(int(b >> 32), 0xB1, 0xF, 0xF, false);
    return __builtin_bit_cast(double, (static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}

// First tree pass when the stored levels start at the precision's low level
// (4 for complex128, 5 for complex64): one read of the state, that level
// written; the upper levels come from it in tree_kernel passes.
// Each wave reduces a tile.  All of the tile's loads (coalesced, 16 bytes per
// lane, nontemporal) are issued before any arithmetic.  Level 1 is formed in
// registers: inside the lane for complex64 (a 16-byte load holds two
// amplitudes), with the neighbouring lane by DPP for complex128.  Level-1
// nodes go to LDS in rows of 8 (16 amplitudes; padded to 9 doubles so that the
// row reads are conflict-free); each lane sums one row as the aligned-pair
// tree (levels 2..4) in registers; complex128 stores the level-4 node (a
// contiguous 512 bytes per wave), complex64 adds the neighbouring lane's (DPP)
// and stores level 5 from the even lanes (256 bytes per wave and round).  The
// stores are nontemporal: the state streams through without the tree's writes
// breaking up the reads.  Every node is
// left + right of the same two children as in the reference's balanced tree
// (IEEE addition is commutative, so the order of the two operands does not
// matter).
template <bool kC64>
__global__ __launch_bounds__(kThreads) void tree_amp_kernel(const void *__restrict__ state, double *__restrict__ tl)
{
    using G = TreeGeo<kC64>;
    __shared__ double rows[kThreads / 64][64 * kRowPad];
    const int w = threadIdx.x >> 6, L = threadIdx.x & 63;
    const uint64_t tile = uint64_t(blockIdx.x) * (kThreads / 64) + w;
    const uint64_t base = tile << G::kTileBits;
    double *rb = rows[w];
    if (kC64)
    {
        const fvec4 *src = static_cast<const fvec4 *>(state) + (base >> 1);
        fvec4 v[16];
#pragma unroll
        for (int k = 0; k < 16; k++)
            v[k] = __builtin_nontemporal_load(src + 64 * k + L);
#pragma unroll
        for (int r = 0; r < 2; r++)
        {
#pragma unroll
            for (int k = 0; k < 8; k++)
            {
                const fvec4 a = v[8 * r + k];
                const double x0 = a.x, y0 = a.y, x1 = a.z, y1 = a.w;
                const double n1 = __dadd_rn(__dadd_rn(__dmul_rn(x0, x0), __dmul_rn(y0, y0)),
                                            __dadd_rn(__dmul_rn(x1, x1), __dmul_rn(y1, y1)));
                const int j = 64 * k + L; // level-1 node within the round
                rb[(j >> 3) * kRowPad + (j & 7)] = n1;
            }
            wave_sync();
            double q[8];
#pragma unroll
            for (int c = 0; c < 8; c++)
                q[c] = rb[L * kRowPad + c];
            wave_sync();
#pragma unroll
            for (int c = 0; c < 4; c++)
                q[c] = __dadd_rn(q[2 * c], q[2 * c + 1]);
            // level 4 of row L, then level 5 with the neighbouring lane
            const double n4 = __dadd_rn(__dadd_rn(q[0], q[1]), __dadd_rn(q[2], q[3]));
            const double n5 = __dadd_rn(n4, lane_xor1(n4));
            if ((L & 1) == 0)
                __builtin_nontemporal_store(n5, tl + (base >> 5) + 32 * r + (L >> 1));
        }
    }
    else
    {
        const dvec2 *src = static_cast<const dvec2 *>(state) + base;
        dvec2 v[16];
#pragma unroll
        for (int k = 0; k < 16; k++)
            v[k] = __builtin_nontemporal_load(src + 64 * k + L);
#pragma unroll
        for (int k = 0; k < 16; k++)
        {
            const double p = __dadd_rn(__dmul_rn(v[k].x, v[k].x), __dmul_rn(v[k].y, v[k].y));
            const double n1 = __dadd_rn(p, lane_xor1(p));
            const int j = 32 * k + (L >> 1); // level-1 node within the tile
            if ((L & 1) == 0)
                rb[(j >> 3) * kRowPad + (j & 7)] = n1;
        }
        wave_sync();
        double q[8];
#pragma unroll
        for (int c = 0; c < 8; c++)
            q[c] = rb[L * kRowPad + c];
#pragma unroll
        for (int c = 0; c < 4; c++)
            q[c] = __dadd_rn(q[2 * c], q[2 * c + 1]);
        __builtin_nontemporal_store(__dadd_rn(__dadd_rn(q[0], q[1]), __dadd_rn(q[2], q[3])), tl + (base >> 4) + L);
    }
}

// Tree pass over stored nodes: level lin -> levels lin+1 .. lin+5, all
// stored.  A wave tile is 2048 level-lin nodes (16 loads of two nodes per
// lane); level lin+1 is the in-lane pair (stored from registers, 512
// contiguous bytes per load), then each lane sums a row of 16 level-(lin+1)
// nodes from LDS (rows padded to 17 doubles) as the aligned-pair tree and
// stores its 8 + 4 + 2 + 1 nodes of levels lin+2 .. lin+5, which are
// contiguous across the wave's lanes.  Needs 2^13 level-lin nodes per
// workgroup.
constexpr int kUpRowPad = 17;
__global__ __launch_bounds__(kThreads) void tree_up_kernel(const double *__restrict__ in, double *__restrict__ o1,
                                                           double *__restrict__ o2, double *__restrict__ o3,
                                                           double *__restrict__ o4, double *__restrict__ o5)
{
    __shared__ double rows[kThreads / 64][64 * kUpRowPad];
    const int w = threadIdx.x >> 6, L = threadIdx.x & 63;
    const uint64_t tile = uint64_t(blockIdx.x) * (kThreads / 64) + w; // 1024 level-(lin+1) nodes each
    const dvec2 *src = reinterpret_cast<const dvec2 *>(in) + (tile << 10);
    double *rb = rows[w];
    dvec2 v[16];
#pragma unroll
    for (int k = 0; k < 16; k++)
        v[k] = __builtin_nontemporal_load(src + 64 * k + L);
#pragma unroll
    for (int k = 0; k < 16; k++)
    {
        const double n = __dadd_rn(v[k].x, v[k].y);
        const int j = 64 * k + L;
        o1[(tile << 10) + j] = n;
        rb[(j >> 4) * kUpRowPad + (j & 15)] = n;
    }
    wave_sync();
    double q[16];
#pragma unroll
    for (int c = 0; c < 16; c++)
        q[c] = rb[L * kUpRowPad + c];
    const uint64_t r = (tile << 6) + L; // this lane's row: node index at level lin+5
#pragma unroll
    for (int c = 0; c < 8; c++)
        q[c] = __dadd_rn(q[2 * c], q[2 * c + 1]);
#pragma unroll
    for (int c = 0; c < 4; c++)
        reinterpret_cast<dvec2 *>(o2)[4 * r + c] = dvec2{q[2 * c], q[2 * c + 1]};
#pragma unroll
    for (int c = 0; c < 4; c++)
        q[c] = __dadd_rn(q[2 * c], q[2 * c + 1]);
#pragma unroll
    for (int c = 0; c < 2; c++)
        reinterpret_cast<dvec2 *>(o3)[2 * r + c] = dvec2{q[2 * c], q[2 * c + 1]};
    q[0] = __dadd_rn(q[0], q[1]);
    q[1] = __dadd_rn(q[2], q[3]);
    reinterpret_cast<dvec2 *>(o4)[r] = dvec2{q[0], q[1]};
    o5[r] = __dadd_rn(q[0], q[1]);
}

// prefix_s (Fenwick over levels >= I) and tail_s = prefix_s + N_I[s].
__global__ __launch_bounds__(kThreads) void tails_kernel(const double *__restrict__ tree, const Levels lv, int I, int m,
                                                         uint64_t nseg, double *__restrict__ prefix,
                                                         double *__restrict__ tail)
{
    const uint64_t s = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x;
    if (s >= nseg)
        return;
    double acc = 0.0;
    for (int l = m - I - 1; l >= 0; l--)
        if ((s >> l) & 1u)
            acc = __dadd_rn(acc, tree[lv.off[I + l] + ((s >> l) - 1)]);
    prefix[s] = acc;
    tail[s] = __dadd_rn(acc, tree[lv.off[I] + s]);
}

// In-place running maximum over nseg values (one workgroup; max is exact).
__global__ __launch_bounds__(kThreads) void cummax_kernel(double *__restrict__ v, uint64_t n)
{
    __shared__ double part[kThreads];
    const uint64_t per = (n + kThreads - 1) / kThreads;
    const uint64_t b = threadIdx.x * per;
    const uint64_t e = b + per < n ? b + per : n;
    double mx = -1.0;
    for (uint64_t i = b; i < e; i++)
        mx = fmax(mx, v[i]);
    part[threadIdx.x] = mx;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        double run = -1.0;
        for (int t = 0; t < kThreads; t++)
        {
            const double cur = part[t];
            part[t] = run; // exclusive running max
            run = fmax(run, cur);
        }
    }
    __syncthreads();
    double run = part[threadIdx.x];
    for (uint64_t i = b; i < e; i++)
    {
        run = fmax(run, v[i]);
        v[i] = run;
    }
}

// tails_kernel and cummax_kernel in one workgroup, for states of few
// segments: each thread's run of segments, then the running maximum across the
// threads by doubling (max is exact, so the order does not matter).
constexpr int kFewThreads = 1024;
constexpr uint64_t kFewSegs = 4096;
__global__ __launch_bounds__(kFewThreads) void few_tails_kernel(const double *__restrict__ tree, const Levels lv,
                                                                int I, int m, int nseg, double *__restrict__ prefix,
                                                                double *__restrict__ cmax)
{
    __shared__ double part[kFewThreads];
    constexpr int kPer = int(kFewSegs) / kFewThreads;
    double t[kPer];
    double mx = -1.0;
#pragma unroll
    for (int j = 0; j < kPer; j++)
    {
        const int s = int(threadIdx.x) * kPer + j;
        t[j] = -1.0;
        if (s < nseg)
        {
            double acc = 0.0;
            for (int l = m - I - 1; l >= 0; l--)
                if ((s >> l) & 1)
                    acc = __dadd_rn(acc, tree[lv.off[I + l] + uint64_t((s >> l) - 1)]);
            prefix[s] = acc;
            t[j] = __dadd_rn(acc, tree[lv.off[I] + uint64_t(s)]);
        }
        mx = fmax(mx, t[j]);
    }
    part[threadIdx.x] = mx;
    __syncthreads();
    for (int d = 1; d < kFewThreads; d <<= 1)
    {
        const double o = int(threadIdx.x) >= d ? part[threadIdx.x - d] : -1.0;
        __syncthreads();
        part[threadIdx.x] = fmax(part[threadIdx.x], o);
        __syncthreads();
    }
    double run = threadIdx.x ? part[threadIdx.x - 1] : -1.0;
#pragma unroll
    for (int j = 0; j < kPer; j++)
    {
        const int s = int(threadIdx.x) * kPer + j;
        run = fmax(run, t[j]);
        if (s < nseg)
            cmax[s] = run;
    }
}

// Virtual bits of a real address (pack_virtual_results_host,
// src/zxh/src/measure/measure_result_pack.h:24-44; the reference's GPU path
// does the same in map_real_to_virtual_words_kernel): virtual bit q = parity
// (real & row q) ^ b[q], the row's bit 63 holding b[q].  Up to 64 rows travel
// in the kernel arguments; more come from device memory.
constexpr int kArgRows = 64;
struct PackArgs
{
    uint64_t rows[kArgRows];
    const uint64_t *more; // all nq rows when nq > kArgRows
    uint64_t *out;        // nullptr: no packing
    int nq, wc;
};

// One shot per thread.
//
// The probes of libstdc++'s upper_bound over a segment's 2^I values are
// the midpoints of aligned blocks: after a right turn at mid the range is
// (mid, end of mid's block), 2^l - 1 values whose own midpoint is again the
// block's, and before the first right turn it is the block from 0.  So the
// walk is a descent: at block [P, P + 2^l) the probe is mid = P + 2^(l-1),
// whose prefix is that of P (carried, the same sums in the same order) plus
// one stored node, the left half's.  A probe loads that node and the
// amplitude at mid, both at once.  The last LB levels lie in one block of
// 256 bytes, read once; its pair sums come from registers.  (Re-reading every
// prefix node and a 256-byte block at each probe, 10^6 shots of a 30-qubit
// complex128 state took 1.88 ms, and 1024 shots of a 20-qubit one 82 us of
// dependent loads.)
template <bool kC64>
__global__ __launch_bounds__(kThreads) void search_kernel(const void *__restrict__ state,
                                                          const double *__restrict__ tree, const Levels lv, int I,
                                                          int LS, const double *__restrict__ cmax,
                                                          const double *__restrict__ prefix, uint64_t nseg,
                                                          const double *__restrict__ thr, uint64_t shots,
                                                          uint64_t *__restrict__ out, int *__restrict__ err,
                                                          const PackArgs pack)
{
    const uint64_t k = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x;
    if (k >= shots)
        return;
    const double tau = thr[k];
    // first segment whose running-max tail exceeds tau
    uint64_t lo = 0, len = nseg;
    while (len > 0)
    {
        const uint64_t half = len >> 1;
        if (tau < cmax[lo + half])
            len = half;
        else
        {
            lo = lo + half + 1;
            len = len - half - 1;
        }
    }
    if (lo >= nseg)
    {
        *err = 1;
        return;
    }
    const uint64_t seg = lo;
    const uint64_t sbase = seg << I;
    const double head = prefix[seg];
    const int LB = LS < I ? LS : I; // low levels recomputed from amplitudes
    const uint64_t valid = uint64_t(1) << I;

    uint64_t P = 0;
    double acc = 0.0;
    for (int l = I; l > LB; l--)
    {
        const uint64_t mid = P + (uint64_t(1) << (l - 1));
        const double left = tree[lv.off[l - 1] + ((sbase + P) >> (l - 1))];
        const double pm = p_of(state, kC64, sbase + mid);
        const double excl = __dadd_rn(acc, left);
        if (!(tau < __dadd_rn(__dadd_rn(head, excl), pm)))
        {
            P = mid;
            acc = excl;
        }
    }
    // the block of 2^LB amplitudes from P on and its aligned pair sums; a turn
    // halves the window they cover, which stays at the arrays' front
    constexpr int kLBM = kC64 ? 5 : 4;
    constexpr int NB = 1 << kLBM;
    double q[kLBM][NB];
#pragma unroll
    for (int i = 0; i < NB; i++)
        q[0][i] = i < (1 << LB) ? p_of(state, kC64, sbase + P + i) : 0.0;
#pragma unroll
    for (int r = 1; r < kLBM; r++)
#pragma unroll
        for (int i = 0; i < (NB >> r); i++)
            q[r][i] = __dadd_rn(q[r - 1][2 * i], q[r - 1][2 * i + 1]);
    const double p0 = q[0][0];
#pragma unroll
    for (int l = kLBM; l > 0; l--)
    {
        if (l > LB)
            continue;
        const int half = 1 << (l - 1);
        const double excl = __dadd_rn(acc, q[l - 1][0]);
        const bool right = !(tau < __dadd_rn(__dadd_rn(head, excl), q[0][half]));
        P = right ? P + half : P;
        acc = right ? excl : acc;
#pragma unroll
        for (int r = 0; r < l - 1; r++)
#pragma unroll
            for (int i = 0; i < (half >> r); i++)
                q[r][i] = right ? q[r][i + (half >> r)] : q[r][i];
    }
    // without a right turn value 0 is still to be probed
    uint64_t first = P + 1;
    if (P == 0 && tau < __dadd_rn(__dadd_rn(head, 0.0), p0))
        first = 0;
    const uint64_t real = sbase + (first == valid ? valid - 1 : first);
    out[k] = real;
    if (pack.out)
        for (int w = 0; w < pack.wc; w++)
        {
            uint64_t word = 0;
            const int hi = min(64, pack.nq - 64 * w);
            for (int j = 0; j < hi; j++)
            {
                const uint64_t row = pack.more ? pack.more[64 * w + j] : pack.rows[j];
                word |= uint64_t((__popcll(real & row & ~(uint64_t(1) << 63)) & 1) ^ int(row >> 63)) << j;
            }
            pack.out[k * uint64_t(pack.wc) + w] = word;
        }
}

// Lowest stored tree level: below it the search recomputes from amplitudes
// (256 bytes of state per block in both precisions).
inline unsigned low_level(int prec, unsigned I)
{
    return std::min(prec == C64 ? 5u : 4u, I);
}

int build_tree(Ctx &ctx, const void *state, int prec, unsigned m, unsigned LS, Levels &lv, double **tree_out,
               double *root, double *one)
{
    uint64_t total = 0;
    for (unsigned l = 0; l < kMaxLevels; l++)
        lv.off[l] = 0;
    for (unsigned l = LS; l <= m; l++)
    {
        lv.off[l] = total;
        total += uint64_t(1) << (m - l);
    }
    ZXA_TRY(ctx.scratch_b.ensure(total * sizeof(double)));
    double *tree = static_cast<double *>(ctx.scratch_b.ptr);
    // level 0 -> up to kSpanBits, then from level kSpanBits, ...
    int lin = 0;
    bool first = true;
    ZXA_TRY(ctx.tic());
    const int gbits = prec == C64 ? TreeGeo<true>::kGroupBits : TreeGeo<false>::kGroupBits;
    const unsigned amp_level = prec == C64 ? 5u : 4u;
    if (LS == amp_level && int(m) >= gbits)
    {
        // amplitudes -> level 4 (c128) or 5 (c64) in one read of the state
        const unsigned groups = static_cast<unsigned>(uint64_t(1) << (int(m) - gbits));
        double *tl = tree + lv.off[amp_level];
        if (prec == C64)
            hipLaunchKernelGGL(tree_amp_kernel<true>, dim3(groups), dim3(kThreads), 0, ctx.stream, state, tl);
        else
            hipLaunchKernelGGL(tree_amp_kernel<false>, dim3(groups), dim3(kThreads), 0, ctx.stream, state, tl);
        ZXA_HIP(hipGetLastError());
        first = false;
        lin = int(amp_level);
    }
    // stored levels -> five more levels per pass while a pass fills its grid
    while (!first && int(m) - lin >= 13 + 5)
    {
        const unsigned groups = static_cast<unsigned>(uint64_t(1) << (int(m) - lin - 13));
        hipLaunchKernelGGL(tree_up_kernel, dim3(groups), dim3(kThreads), 0, ctx.stream, tree + lv.off[lin],
                           tree + lv.off[lin + 1], tree + lv.off[lin + 2], tree + lv.off[lin + 3],
                           tree + lv.off[lin + 4], tree + lv.off[lin + 5]);
        ZXA_HIP(hipGetLastError());
        lin += 5;
    }
    while (first || lin < int(m))
    {
        const int span_bits = std::min<int>(kSpanBits, int(m) - lin);
        const uint64_t groups = uint64_t(1) << (int(m) - lin - span_bits);
        const int kind = first ? (prec == C64 ? 1 : 0) : 2;
        const void *src = first ? state : static_cast<const void *>(tree);
        // a non-first pass reads level lin, which must be stored
        if (!first && unsigned(lin) < LS)
        {
            set_error("sampler tree: unstored intermediate level");
            return EINVAL_;
        }
        hipLaunchKernelGGL(tree_kernel, dim3(static_cast<unsigned>(groups)), dim3(kThreads), 0, ctx.stream, src, kind,
                           lin, span_bits, int(LS), int(m), tree, lv, root, one);
        ZXA_HIP(hipGetLastError());
        first = false;
        lin += span_bits;
        if (span_bits == 0)
            break;
    }
    // algorithmic bytes: one read of the state and one write of the stored
    // levels (the passes above the first read stored levels back; not counted)
    ZXA_TRY(ctx.toc(F_TREE, (uint64_t(1) << m) * elem_bytes(prec) + total * sizeof(double)));
    *tree_out = tree;
    return OK;
}

} // namespace

// What the sampler's kernels tell the host: in pinned, coherent memory.
struct Told
{
    double total;
    int err;
};

int told(Ctx &ctx, Told **t)
{
    ZXA_TRY(ctx.sample_total_pin.ensure(sizeof(Told)));
    *t = static_cast<Told *>(ctx.sample_total_pin.ptr);
    return OK;
}

int prob_total(Ctx &ctx, const void *state, int prec, unsigned m, double *out)
{
    Levels lv;
    double *tree = nullptr;
    Told *t = nullptr;
    ZXA_TRY(told(ctx, &t));
    const unsigned LS = low_level(prec, m);
    ctx.sample_ready = false; // the tree of a launch before this one is overwritten
    ZXA_TRY(build_tree(ctx, state, prec, m, LS, lv, &tree, &t->total, nullptr));
    ZXA_HIP(hipStreamSynchronize(ctx.stream));
    *out = t->total;
    return OK;
}

int sample_launch(Ctx &ctx, const void *state, int prec, unsigned m, unsigned seg_bits)
{
    if (m > 40)
    {
        set_error("sampler: state wider than 40 bits");
        return EINVAL_;
    }
    ctx.sample_ready = false;
    const unsigned I = std::min(m, seg_bits);
    const unsigned LS = low_level(prec, I);
    Levels &lv = ctx.sample_levels_as<Levels>();
    double *tree = nullptr;
    Told *t = nullptr;
    ZXA_TRY(told(ctx, &t));
    const uint64_t nseg = uint64_t(1) << (m - I);
    ZXA_TRY(ctx.scratch_d.ensure(2 * nseg * sizeof(double)));
    double *prefix = static_cast<double *>(ctx.scratch_d.ptr);
    double *cmax = prefix + nseg;
    ZXA_TRY(build_tree(ctx, state, prec, m, LS, lv, &tree, &t->total, nseg == 1 ? prefix : nullptr));
    if (nseg > kFewSegs)
    {
        hipLaunchKernelGGL(tails_kernel, dim3(static_cast<unsigned>((nseg + kThreads - 1) / kThreads)),
                           dim3(kThreads), 0, ctx.stream, tree, lv, int(I), int(m), nseg, prefix, cmax);
        ZXA_HIP(hipGetLastError());
        hipLaunchKernelGGL(cummax_kernel, dim3(1), dim3(kThreads), 0, ctx.stream, cmax, nseg);
        ZXA_HIP(hipGetLastError());
    }
    else if (nseg > 1)
    {
        hipLaunchKernelGGL(few_tails_kernel, dim3(1), dim3(kFewThreads), 0, ctx.stream, tree, lv, int(I), int(m),
                           int(nseg), prefix, cmax);
        ZXA_HIP(hipGetLastError());
    }
    ctx.sample_m = m;
    ctx.sample_I = I;
    ctx.sample_ready = true;
    return OK;
}

int sample_total(Ctx &ctx, double *total)
{
    if (!ctx.sample_ready)
    {
        set_error("sampler: total before launch");
        return ESTATE;
    }
    ZXA_HIP(hipStreamSynchronize(ctx.stream));
    *total = static_cast<const Told *>(ctx.sample_total_pin.ptr)->total;
    return OK;
}

// Resolves the thresholds of a sampler launch.  thr, real and pack->out are
// pinned host memory (the kernel reads and writes them in place); next, when
// given, forms thresholds [from, to) just before they are searched, so that
// the search of one piece runs while the host forms the next.
int sample_search(Ctx &ctx, const void *state, int prec, const double *thr, size_t shots, uint64_t *real,
                  const PackSpec *pack, const std::function<void(size_t, size_t)> &next)
{
    if (shots == 0)
        return OK;
    if (!ctx.sample_ready)
    {
        set_error("sampler: search before launch");
        return ESTATE;
    }
    const unsigned m = ctx.sample_m, I = ctx.sample_I;
    const unsigned LS = low_level(prec, I);
    const Levels &lv = ctx.sample_levels_as<Levels>();
    const double *tree = static_cast<const double *>(ctx.scratch_b.ptr);
    const uint64_t nseg = uint64_t(1) << (m - I);
    const double *prefix = static_cast<const double *>(ctx.scratch_d.ptr);
    const double *cmax = prefix + nseg;
    Told *t = nullptr;
    ZXA_TRY(told(ctx, &t));
    t->err = 0;
    PackArgs pa = {};
    std::vector<uint64_t> rows;
    if (pack)
    {
        pa.nq = int(pack->nq);
        pa.wc = (pa.nq + 63) / 64;
        rows.resize(size_t(pa.nq));
        for (int q = 0; q < pa.nq; q++)
            rows[size_t(q)] = pack->rows[q] | (uint64_t(pack->b[q] & 1u) << 63);
        if (pa.nq <= kArgRows)
            std::copy(rows.begin(), rows.end(), pa.rows);
        else
        {
            ZXA_TRY(ctx.scratch_c.ensure(rows.size() * sizeof(uint64_t)));
            ZXA_HIP(hipMemcpyAsync(ctx.scratch_c.ptr, rows.data(), rows.size() * sizeof(uint64_t),
                                   hipMemcpyHostToDevice, ctx.stream));
            pa.more = static_cast<const uint64_t *>(ctx.scratch_c.ptr);
        }
    }
    // pieces of 128 K shots: 0.2 ms of threshold recurrence each, several
    // times what the search of one takes, so only the last is not hidden
    constexpr size_t kPiece = size_t(1) << 17;
    ZXA_TRY(ctx.tic());
    for (size_t o = 0; o < shots; o += kPiece)
    {
        const size_t cnt = next ? std::min(kPiece, shots - o) : shots;
        if (next)
            next(o, o + cnt);
        pa.out = pack ? pack->out + o * size_t(pa.wc) : nullptr;
        const unsigned grid = static_cast<unsigned>((cnt + kThreads - 1) / kThreads);
        if (prec == C64)
            hipLaunchKernelGGL(search_kernel<true>, dim3(grid), dim3(kThreads), 0, ctx.stream, state, tree, lv,
                               int(I), int(LS), cmax, prefix, nseg, thr + o, uint64_t(cnt), real + o, &t->err, pa);
        else
            hipLaunchKernelGGL(search_kernel<false>, dim3(grid), dim3(kThreads), 0, ctx.stream, state, tree, lv,
                               int(I), int(LS), cmax, prefix, nseg, thr + o, uint64_t(cnt), real + o, &t->err, pa);
        ZXA_HIP(hipGetLastError());
        if (!next)
            break;
    }
    ZXA_TRY(ctx.toc(F_SAMPLE, 0));
    ZXA_HIP(hipStreamSynchronize(ctx.stream));
    if (t->err)
    {
        set_error("measure failed to resolve all local samples");
        return EUNRESOLVED;
    }
    return OK;
}

// The whole draw: the tree builds while the host forms the uniforms'
// factors, which do not depend on the total; then the recurrence, piece by
// piece ahead of the search.
int sample_draw(Ctx &ctx, const void *state, int prec, unsigned m, unsigned seg_bits, uint64_t stream_seed,
                size_t shots, double *thr, uint64_t *real, const PackSpec *pack)
{
    ZXA_TRY(sample_launch(ctx, state, prec, m, seg_bits));
    threshold_draws(stream_seed, shots, thr);
    threshold_factors(thr, shots);
    double total = 0.0;
    ZXA_TRY(sample_total(ctx, &total));
    if (!(total > 0.0))
    {
        set_error("state has zero total probability");
        return EZEROPROB;
    }
    double lo = 0.0;
    return sample_search(ctx, state, prec, thr, shots, real, pack,
                         [&](size_t b, size_t e) { lo = threshold_apply(thr + b, e - b, lo, total); });
}

// measure (measure_common.cpp:73-92) on a caller's state and affine map;
// nq = 0: real addresses only.
int measure_affine(Ctx &ctx, const void *state, int prec, unsigned m, unsigned seg_bits, unsigned nq,
                   const uint64_t *rows, const uint8_t *b, uint64_t stream_seed, size_t shots, uint64_t *packed,
                   uint64_t *out_real)
{
    if (shots == 0)
        return OK;
    const size_t wc = (size_t(nq) + 63) / 64;
    ZXA_TRY(ctx.sample_thr_pin.ensure(shots * sizeof(double)));
    ZXA_TRY(ctx.sample_out_pin.ensure(shots * (1 + wc) * sizeof(uint64_t)));
    uint64_t *real = static_cast<uint64_t *>(ctx.sample_out_pin.ptr);
    PackSpec ps;
    ps.nq = nq;
    ps.rows = rows;
    ps.b = b;
    ps.out = real + shots;
    ZXA_TRY(sample_draw(ctx, state, prec, m, seg_bits, stream_seed, shots,
                        static_cast<double *>(ctx.sample_thr_pin.ptr), real, nq ? &ps : nullptr));
    if (nq)
        std::memcpy(packed, ps.out, shots * wc * sizeof(uint64_t));
    if (out_real)
        std::memcpy(out_real, real, shots * sizeof(uint64_t));
    return OK;
}

int sample_apply(Ctx &ctx, const void *state, int prec, unsigned m, unsigned seg_bits, const double *thresholds,
                 size_t shots, uint64_t *out_real)
{
    if (shots == 0)
        return OK;
    ZXA_TRY(ctx.sample_thr_pin.ensure(shots * sizeof(double)));
    ZXA_TRY(ctx.sample_out_pin.ensure(shots * sizeof(uint64_t)));
    std::memcpy(ctx.sample_thr_pin.ptr, thresholds, shots * sizeof(double));
    ZXA_TRY(sample_launch(ctx, state, prec, m, seg_bits));
    double total = 0.0;
    ZXA_TRY(sample_total(ctx, &total));
    ZXA_TRY(sample_search(ctx, state, prec, static_cast<const double *>(ctx.sample_thr_pin.ptr), shots,
                          static_cast<uint64_t *>(ctx.sample_out_pin.ptr), nullptr, nullptr));
    std::memcpy(out_real, ctx.sample_out_pin.ptr, shots * sizeof(uint64_t));
    return OK;
}

} // namespace zxa
