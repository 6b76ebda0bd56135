// kernels_circuit.hip -- circuits executed out of LDS (see circuit.h).
#include "circuit.h"
#include "poly.h"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace zxa
{
namespace
{

template <bool kC64>
struct CGeo;
template <>
struct CGeo<false>
{
    using T = double2;
    using R = double;
    static constexpr int kTileBits = 12;
    static constexpr int kSwz = 4; // sixteen 16-byte LDS words to a row of banks
};
template <>
struct CGeo<true>
{
    using T = float2;
    using R = float;
    static constexpr int kTileBits = 13;
    static constexpr int kSwz = 5; // thirty-two 8-byte words
};

// LDS index of a tile coordinate: its low bits (the banks' 256 bytes) XORed
// with the bits three above them, so that the lanes of an access, whose
// coordinates skip up to three consecutive bits, land in distinct banks
// wherever those bits are.  Linear over XOR: an element's index is the base's
// XOR the offset's.
template <bool kC64>
__host__ __device__ __forceinline__ uint32_t lds_index(uint32_t a)
{
    return a ^ ((a >> 3) & ((1u << CGeo<kC64>::kSwz) - 1));
}

__device__ __forceinline__ uint32_t par32(uint32_t x)
{
    return __popc(x) & 1u;
}

__device__ __forceinline__ uint32_t odd(uint32_t sel, uint32_t x)
{
    return par32(x & sel & 0x7fffffffu) ^ (sel >> 31);
}

__host__ __device__ __forceinline__ uint32_t insert_zero(uint32_t x, uint32_t p)
{
    const uint32_t lo = x & ((1u << p) - 1);
    return ((x >> p) << (p + 1)) | lo;
}

// Steps are read through the scalar cache: offsets, selectors and matrices
// are the same for every thread, and the LDS is left to the amplitudes.  A
// step's first line (all but the matrices) is loaded at once.
#define ZXA_STEP const __attribute__((address_space(4))) LdsStep

struct StepHead
{
    uint32_t kind, count, pivot, ctrl;
    uint32_t slot[4], sel[3], full[4];
    StepHead() = default;
    __device__ __forceinline__ explicit StepHead(ZXA_STEP &st)
        : kind(st.kind), count(st.count), pivot(st.pivot), ctrl(st.ctrl),
          slot{st.slot[0], st.slot[1], st.slot[2], st.slot[3]}, sel{st.sel[0], st.sel[1], st.sel[2]},
          full{st.full[0], st.full[1], st.full[2], st.full[3]}
    {
    }
};

template <bool kC64>
__device__ __forceinline__ typename CGeo<kC64>::R entry(ZXA_STEP &st, int j, int e)
{
    if constexpr (kC64)
        return st.uf[j][e];
    else
        return st.u[j][e];
}

// K commuting gates on every coset of their offsets in the tile: a thread
// reads the coset's 2^K amplitudes, applies the gates in registers and writes
// them back.  A gate's offset changes its own selector and no other's, so the
// thread starts from the coset's element that every gate's selector leaves
// out: the pairs are then (even, odd) throughout and the matrices uniform.
template <bool kC64, int K, bool kCtrl>
__device__ __forceinline__ void gates_step(typename CGeo<kC64>::T *amp, const StepHead &h, ZXA_STEP &st,
                                           uint32_t bits, uint32_t base)
{
    using T = typename CGeo<kC64>::T;
    using R = typename CGeo<kC64>::R;
    constexpr int N = 1 << K;
    const uint32_t total = 1u << (bits - K);
    uint32_t sel[K], side[K];
#pragma unroll
    for (int j = 0; j < K; j++)
    {
        sel[j] = h.sel[j] & 0x7fffffffu;
        side[j] = __builtin_popcount(h.full[j] & base) + (h.sel[j] >> 31);
    }
    for (uint32_t b = threadIdx.x; b < total; b += blockDim.x)
    {
        uint32_t l = b;
#pragma unroll
        for (int j = 0; j < K; j++)
            l = insert_zero(l, (h.pivot >> (8 * j)) & 0xffu);
        uint32_t off[N];
        off[0] = lds_index<kC64>(l);
        bool on = true;
#pragma unroll
        for (int j = 0; j < K; j++)
        {
            const uint32_t f = (__popc(l & sel[j]) + side[j]) & 1u;
            off[0] ^= f ? h.slot[j] : 0u;
            if constexpr (kCtrl)
            {
                // the pair's even-side element decides
                const uint32_t e = f ? l ^ h.slot[3] : l;
                on = ((__popc(e & h.ctrl & 0x7fffffffu) + (h.ctrl >> 31) + __builtin_popcount(h.full[3] & base)) &
                      1u) != 0;
            }
        }
        if (kCtrl && !on)
            continue;
#pragma unroll
        for (int j = 0; j < K; j++)
#pragma unroll
            for (int c = 0; c < (1 << j); c++)
                off[(1 << j) + c] = off[c] ^ h.slot[j];
        T v[N];
#pragma unroll
        for (int c = 0; c < N; c++)
            v[c] = amp[off[c]];
#pragma unroll
        for (int j = 0; j < K; j++)
        {
            R m[8];
#pragma unroll
            for (int e = 0; e < 8; e++)
                m[e] = entry<kC64>(st, j, e);
#pragma unroll
            for (int c = 0; c < N; c++)
            {
                if (c & (1 << j))
                    continue;
                const T p = v[c], q = v[c | (1 << j)];
                T np, nq;
                np.x = m[0] * p.x - m[1] * p.y + m[2] * q.x - m[3] * q.y;
                np.y = m[0] * p.y + m[1] * p.x + m[2] * q.y + m[3] * q.x;
                nq.x = m[4] * p.x - m[5] * p.y + m[6] * q.x - m[7] * q.y;
                nq.y = m[4] * p.y + m[5] * p.x + m[6] * q.y + m[7] * q.x;
                v[c] = np;
                v[c | (1 << j)] = nq;
            }
        }
#pragma unroll
        for (int c = 0; c < N; c++)
            amp[off[c]] = v[c];
    }
}

// A window's phase factors, every window of some passes at once and over the
// whole chip, so that the circuit kernel evaluates no selector and no sine.
// Blocks below tblocks: the phases by the tile coordinates alone, exp(i sum
// of the gates' angles at base 0), 2^bits entries per window.  The others (a
// state of several tiles): per window and tile 64 factors of exp(i (C + sum_i
// c_i l_i)), by groups of coordinate bits, 32 for bits 0-4 (with C), 16 for
// bits 5-8 and 16 for bits 9-12.
// A window whose selectors do not split so has a table of every tile, formed
// by a launch of its own over tile index and coordinates together (bits: the
// state's), and factors of 1.
struct WinTask
{
    uint64_t gates; // const LdsDiag *
    uint64_t count;
    uint64_t win;   // const LdsWin *
    uint64_t out;   // the table's first entry; kNoTable: formed by the other launch
};
constexpr uint64_t kNoTable = ~uint64_t(0);
constexpr int kFactors = 64;
// Gates of a table's sum, read together into LDS (one by one from memory, each
// waiting for the one before, a gate took 0.25 us).
constexpr int kTabGates = 128;
static_assert(sizeof(LdsDiag) == 32 && 2 * kTabGates == 256, "two 16-byte loads a gate, one per thread");

template <bool kC64>
__global__ __launch_bounds__(256) void window_kernel(const WinTask *__restrict__ tasks, uint32_t bits,
                                                     uint32_t tblocks, uint32_t outer,
                                                     typename CGeo<kC64>::T *__restrict__ out,
                                                     double2 *__restrict__ factors)
{
    __shared__ LdsWin W;
    __shared__ LdsDiag sh[kTabGates];
    const WinTask task = tasks[blockIdx.y];
    if (blockIdx.x < tblocks)
    {
        if (task.out == kNoTable)
            return;
        const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
        const uint32_t count = uint32_t(task.count);
        // the angles' sum with its rounding errors carried beside it
        double th = 0.0, lo = 0.0;
        for (uint32_t g0 = 0; g0 < count; g0 += kTabGates)
        {
            const uint32_t n = min(uint32_t(kTabGates), count - g0);
            const float4 *src = reinterpret_cast<const float4 *>(task.gates) + 2 * g0;
            __syncthreads();
            if (threadIdx.x < 2 * n)
                reinterpret_cast<float4 *>(sh)[threadIdx.x] = src[threadIdx.x];
            __syncthreads();
#pragma unroll 4
            for (uint32_t g = 0; g < n; g++)
            {
                const double a = (odd(sh[g].s0, x) & odd(sh[g].s1, x)) ? sh[g].theta : 0.0;
                const double t = th + a, b = t - th;
                lo += (th - (t - b)) + (a - b);
                th = t;
            }
        }
        if (x >> bits)
            return;
        double s, c;
        sincos(th + lo, &s, &c);
        typename CGeo<kC64>::T r;
        r.x = c;
        r.y = s;
        out[task.out + x] = r;
        return;
    }
    static_assert(sizeof(LdsWin) / sizeof(double) <= 256, "one load per thread");
    if (threadIdx.x < sizeof(LdsWin) / sizeof(double))
        reinterpret_cast<double *>(&W)[threadIdx.x] = reinterpret_cast<const double *>(task.win)[threadIdx.x];
    __syncthreads();
    const uint32_t tile = (blockIdx.x - tblocks) * (256 / kFactors) + threadIdx.x / kFactors;
    if (tile >> outer)
        return;
    const uint32_t j = threadIdx.x % kFactors;
    const uint32_t i0 = j < 32 ? 0u : j < 48 ? 5u : 9u;
    const uint32_t x = j < 32 ? j : j & 15u;
    double a = 0.0;
    for (uint32_t k = 0; k < outer; k++)
    {
        if (!((tile >> k) & 1u))
            continue;
#pragma unroll
        for (uint32_t b = 0; b < 5; b++)
            a += ((x >> b) & 1u) ? W.m[i0 + b][k] : 0.0;
        if (j < 32)
        {
            a += W.m[13][k];
            for (uint32_t l = k + 1; l < outer; l++)
                a += ((tile >> l) & 1u) ? W.q[k][l] : 0.0;
        }
    }
    double s, c;
    sincos(a, &s, &c);
    factors[((uint64_t(blockIdx.y) << outer) + tile) * kFactors + j] = make_double2(c, s);
}

// The steps' lines into the scalar cache (16 KiB), every wave its share and
// sixteen loads at a time, while the tile's amplitudes are on their way: a
// step that found its table in memory would wait a microsecond for it.
__device__ __forceinline__ void warm_steps(const LdsStep *steps, uint32_t nsteps)
{
    const uint32_t waves = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lines = min(nsteps * uint32_t(sizeof(LdsStep) / 64), 224u);
    using Line = const __attribute__((address_space(4))) uint32_t;
    Line *p = (Line *)steps;
    for (uint32_t i = wave; i < lines; i += 16 * waves)
    {
        uint32_t t[16];
#pragma unroll
        for (uint32_t j = 0; j < 16; j++)
            t[j] = p[16 * min(i + j * waves, lines - 1)];
#pragma unroll
        for (uint32_t j = 0; j < 16; j++)
            asm volatile("" ::"s"(t[j]));
    }
}

// Kernel arguments of a pass.  A tile is the coset of the span of vec[0 ..
// bits): coordinate l stands for the offsets of its bits, the tile index is
// deposited into the address bits that are no pivot.
struct CPass
{
    uint32_t vec[14];
    uint32_t piv[14]; // ascending
    uint32_t bits, ntiles, outer;
    uint32_t nsteps, nwin;
    uint32_t fresh; // the state is |0...0>, not yet written
    uint32_t wfull; // bit k: window k has a table per tile
};

// The circuit, or a pass of it.  A workgroup holds a tile in LDS from the
// first step to the last; the steps come through the scalar cache
// (warm_steps) and a window's table entries are loaded before the steps ahead
// of it run, so no step waits for memory.
// Bound by its steps.  One of three gates reads and writes the tile once
// (4096 complex128 amplitudes: 2 x 64 KiB at 128 bytes a cycle, 0.43 us), takes
// 1536 FP64 cycles (0.64 us) and a barrier, and 1.9 us in all: a compute unit
// holds one workgroup, two waves per SIMD, since two would need four waves and
// the registers (164; complex64 211) allow three (two), so that little of it
// overlaps.  20 and 18 bits, 256 and 64 tiles, take the same 1.9 us, 21 bits
// twice that; complex64, 8192 amplitudes, 2.1; a whole state of 13 bits
// (complex64 14) 2.3 (3.9).  What counts is that a launch, its tables and the
// state's way to memory and back are paid once for many layers: 20 layers of 20
// qubits took 41 tile passes at 16 to 21 us, each with a table copy and a
// factor launch, 980 us in all, and take 11 passes and 620 us here; 10 qubits
// and 3 layers, whose state is one tile, 30 launches and 205 us, now one and 46
// us.
// kTile: a state of one tile is 2^13 (complex64 2^14) amplitudes, 128 KiB;
// tiles of a wider one 64 KiB.
constexpr int kLogThreads = 9;
constexpr int kThreads = 1 << kLogThreads;
// kFull: some window has a table of every tile (P.wfull).
template <bool kC64, bool kTile, bool kFull = false>
__global__ __launch_bounds__(kThreads) void circuit_kernel(typename CGeo<kC64>::T *__restrict__ state, const CPass P,
                                                           const LdsStep *__restrict__ steps,
                                                           const LdsDiag *__restrict__ diags,
                                                           const typename CGeo<kC64>::T *__restrict__ tabs,
                                                           const double2 *__restrict__ factors)
{
    using G = CGeo<kC64>;
    using T = typename G::T;
    using R = typename G::R;
    constexpr int kBits = G::kTileBits + (kTile ? 0 : 1);
    constexpr int kPer = (1 << kBits) / kThreads; // amplitudes per thread of a full tile
    __shared__ T amp[1 << kBits];
    __shared__ double2 dt[kTile ? kLdsWindows * kFactors : 1];
    const uint32_t tid = threadIdx.x, nt = blockDim.x, size = 1u << P.bits;
    uint32_t toff = 0; // the address offset of coordinate tid
    if constexpr (kTile)
    {
#pragma unroll
        for (int j = 0; j < kLogThreads; j++)
            toff ^= ((tid >> j) & 1u) ? P.vec[j] : 0u;
    }
    // the address of this thread's k-th amplitude (coordinate tid + k nt)
    auto address = [&](uint32_t base, int k) {
        if constexpr (kTile)
        {
            uint32_t o = base ^ toff;
#pragma unroll
            for (int j = 0; j < kBits - kLogThreads; j++)
                o ^= ((k >> j) & 1) ? P.vec[kLogThreads + j] : 0u;
            return o;
        }
        return tid + uint32_t(k) * nt;
    };
    warm_steps(steps, P.nsteps);
    for (uint32_t tile = blockIdx.x; tile < P.ntiles; tile += gridDim.x)
    {
        uint32_t base = 0;
        if constexpr (kTile)
        {
            base = tile;
#pragma unroll
            for (int j = 0; j < kBits; j++)
                base = insert_zero(base, P.piv[j]);
        }
        // (a whole state's amplitudes go to LDS as they come)
        T v[kTile ? kPer : 1];
#pragma unroll
        for (int k = 0; k < kPer; k++)
        {
            const uint32_t i = tid + k * nt;
            T &z = v[kTile ? k : 0];
            z.x = (tile == 0 && i == 0);
            z.y = 0;
            if (!P.fresh && (kTile || i < size))
                z = state[address(base, k)];
            if (!kTile && i < size)
                amp[lds_index<kC64>(i)] = z;
        }
        if constexpr (kTile)
            for (uint32_t e = tid; e < P.nwin * kFactors; e += nt)
                dt[e] = factors[((uint64_t(e / kFactors) << P.outer) + tile) * kFactors + e % kFactors];
        if constexpr (kTile)
        {
#pragma unroll
            for (int k = 0; k < kPer; k++)
                amp[lds_index<kC64>(tid + k * nt)] = v[k];
        }
        __syncthreads();
        constexpr int kPf = kPer < 16 ? kPer : kTile ? 16 : 8; // loaded ahead; the rest at their use
        uint32_t s = 0;
        // a step's first line is loaded one step ahead
        StepHead h, next;
        if (P.nsteps)
            next = StepHead(((ZXA_STEP *)steps)[0]);
        for (uint32_t win = 0;; win++)
        {
            // the next window's table entries, on their way under the gates
            // before it (past the last window those of the first amplitudes'
            // worth of any window, or of the state, unused)
            T pf[kPf];
            const T *src = state;
            if (P.nwin)
            {
                const uint32_t wi = min(win, P.nwin - 1);
                uint64_t table = wi;
                if constexpr (kFull)
                    table += uint64_t(__builtin_popcount(P.wfull & ((1u << wi) - 1))) * (P.ntiles - 1) +
                             ((P.wfull >> wi) & 1u ? tile : 0u);
                src = tabs + (table << P.bits);
            }
#pragma unroll
            for (int k = 0; k < kPf; k++)
                pf[k] = src[kTile ? tid + k * nt : min(tid + k * nt, size - 1)];
            for (; s < P.nsteps; s++)
            {
                ZXA_STEP &st = ((ZXA_STEP *)steps)[s];
                h = next;
                if (h.kind == 2)
                    break;
                next = StepHead(((ZXA_STEP *)steps)[min(s + 1, P.nsteps - 1)]);
                if (h.kind == 0)
                {
                    if (h.count == 3)
                        gates_step<kC64, 3, false>(amp, h, st, P.bits, base);
                    else if (h.count == 2)
                        gates_step<kC64, 2, false>(amp, h, st, P.bits, base);
                    else
                        gates_step<kC64, 1, false>(amp, h, st, P.bits, base);
                }
                else if (h.kind == 1)
                    gates_step<kC64, 1, true>(amp, h, st, P.bits, base);
                else if constexpr (kTile)
                {
                    // a window whose selectors do not split by tile and
                    // coordinate, of a state wider than lds_table_bits: gate by
                    // gate
                    const uint32_t g0 = h.slot[0], g1 = h.slot[1];
                    double th[kPer] = {};
                    for (uint32_t g = g0; g < g1; g++)
                    {
                        const LdsDiag d = diags[g];
                        const uint32_t b0 = par32(d.f0 & base), b1 = par32(d.f1 & base);
#pragma unroll
                        for (int k = 0; k < kPer; k++)
                        {
                            const uint32_t i = tid + k * nt;
                            th[k] += ((odd(d.s0, i) ^ b0) & (odd(d.s1, i) ^ b1)) ? d.theta : 0.0;
                        }
                    }
#pragma unroll 1
                    for (int k = 0; k < kPer; k++)
                    {
                        double a = th[0];
#pragma unroll
                        for (int j = 1; j < kPer; j++)
                            a = k == j ? th[j] : a;
                        double sn, cs;
                        sincos(a, &sn, &cs);
                        const uint32_t at = lds_index<kC64>(tid + k * nt);
                        const T z = amp[at];
                        T r;
                        r.x = z.x * R(cs) - z.y * R(sn);
                        r.y = z.x * R(sn) + z.y * R(cs);
                        amp[at] = r;
                    }
                }
                __syncthreads();
            }
            if (s >= P.nsteps)
                break;
            // coordinate bits 0-8 are the thread's
            static_assert(kLogThreads == 9, "the factors' third group starts at bit 9");
            double2 w01 = make_double2(1.0, 0.0);
            if constexpr (kTile)
            {
                const double2 a = dt[win * kFactors + (tid & 31u)], b = dt[win * kFactors + 32 + (tid >> 5)];
                w01 = make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
            }
#pragma unroll
            for (int k = 0; k < kPer; k++)
            {
                const uint32_t i = tid + k * nt;
                if (!kTile && i >= size)
                    continue;
                const uint32_t a = lds_index<kC64>(i);
                T p = k < kPf ? pf[k < kPf ? k : 0] : tabs[(uint64_t(win) << P.bits) + i];
                if constexpr (kTile)
                {
                    // in double in both precisions: one rounding to the
                    // amplitudes' precision at the end
                    const double2 d = dt[win * kFactors + 48 + k];
                    const double dx = w01.x * d.x - w01.y * d.y, dy = w01.x * d.y + w01.y * d.x;
                    const double px = p.x, py = p.y;
                    p.x = R(px * dx - py * dy);
                    p.y = R(px * dy + py * dx);
                }
                const T z = amp[a];
                T r;
                r.x = z.x * p.x - z.y * p.y;
                r.y = z.x * p.y + z.y * p.x;
                amp[a] = r;
            }
            s++;
            if (s < P.nsteps)
                next = StepHead(((ZXA_STEP *)steps)[s]);
            __syncthreads();
        }
#pragma unroll
        for (int k = 0; k < kPer; k++)
        {
            const uint32_t i = tid + k * nt;
            if (kTile || i < size)
                state[address(base, k)] = amp[lds_index<kC64>(i)];
        }
        __syncthreads(); // the tile's amplitudes are read before the next tile's are written
    }
}

constexpr uint64_t kAlpha = (uint64_t(1) << 63) - 1;
constexpr uint32_t kAlpha32 = 0x7fffffffu;
constexpr uint32_t kTrue = 0x80000000u;          // the constant selector
constexpr size_t kTabBytes = size_t(32) << 20;   // window tables of one pass
constexpr size_t kMaxLot = 8;                    // passes planned and staged together
constexpr size_t kMaxSteps = 512;                // of one pass (128 KiB of its slot)
constexpr size_t kMaxDiags = 2560;               // 80 KiB
constexpr size_t kMergeFrom = 64;                // gates of a window above which equal ones are looked for
constexpr size_t kMaxScan = 8192;                // operations looked at for one pass
constexpr size_t kMaxDeferred = 192;             // of them deferred, where each is compared

uint32_t pack32(uint64_t sel)
{
    return uint32_t(sel & kAlpha32) | (uint32_t(sel >> 63) << 31);
}

// An angle within half a turn: the sums of many stay small, and so do their
// rounding errors.
double turn(double a)
{
    // 2 pi = 6.283185307179586 (rounded to double) + 2.4492935982947064e-16
    constexpr double kHi = 6.283185307179586, kLo = 2.4492935982947064e-16;
    const double m = std::fabs(a);
    if (m <= 0.5 * kHi)
        return a;
    if (m <= 2.0 * kHi) // the difference is exact
        return a - std::copysign(kHi, a) - std::copysign(kLo, a);
    const double r = std::remainder(a, kHi);
    return r - std::round((a - r) / kHi) * kLo;
}

bool parity(uint64_t x)
{
    return (__builtin_popcountll(x) & 1) != 0;
}

} // namespace

void LdsCircuit::begin(unsigned bits, int prec)
{
    bits_ = bits;
    prec_ = prec;
    simple_ = true;
    ops_.clear();
    mats_.clear();
}

int LdsCircuit::push(const U3Gate &g, const uint64_t *ctrl)
{
    const uint64_t a = g.packed_sel & kAlpha;
    if (g.delta == 0 || (g.delta >> bits_) != 0 || (a >> bits_) != 0 || !parity(a & g.delta) ||
        (ctrl && ((*ctrl & kAlpha) >> bits_) != 0))
    {
        set_error("circuit: a selector does not separate its pair, or reaches outside the state");
        return EINVAL_;
    }
    simple_ = simple_ && a == g.delta && (a & (a - 1)) == 0;
    Op o = {ctrl ? 1u : 0u, uint32_t(g.delta), pack32(g.packed_sel), ctrl ? pack32(*ctrl) : 0u, 0.0,
            uint32_t(mats_.size())};
    std::array<double, 8> m;
    std::copy(g.u, g.u + 8, m.begin());
    mats_.push_back(m);
    ops_.push_back(o);
    return OK;
}

int LdsCircuit::gate(const U3Gate &g)
{
    return push(g, nullptr);
}

int LdsCircuit::swap(uint64_t delta, uint64_t sel, const uint64_t *ctrl)
{
    const U3Gate g = {sel, delta, {0, 0, 1, 0, 1, 0, 0, 0}};
    return push(g, ctrl);
}

// Of a long window, gates with the same selectors become one, its angle their
// sum with the rounding errors carried: a table takes time by the gate (3000
// CP gates on 20 qubits, 190 of them different, took 0.8 ms).
int LdsCircuit::window(const DiagGate *gates, size_t ngates)
{
    const bool merge = ngates > kMergeFrom;
    const size_t first = ops_.size();
    unsigned shift = 64;
    std::vector<double> low;
    if (merge)
    {
        while ((size_t(1) << (64 - shift)) < 2 * ngates)
            shift--;
        seen_.assign(size_t(1) << (64 - shift), 0u);
    }
    for (size_t i = 0; i < ngates; i++)
    {
        const DiagGate &d = gates[i];
        if (((d.s0 & kAlpha) >> bits_) != 0 || (d.s1 != kNoSel && ((d.s1 & kAlpha) >> bits_) != 0))
        {
            set_error("circuit: diagonal selector outside the state");
            return EINVAL_;
        }
        Op o = {2u, 0u, pack32(d.s0), d.s1 == kNoSel ? kTrue : pack32(d.s1), d.theta, 0u};
        if (merge)
        {
            if (o.s1 != kTrue && o.s0 > o.s1)
                std::swap(o.s0, o.s1);
            uint64_t h = ((uint64_t(o.s0) << 32 | o.s1) * 0x9e3779b97f4a7c15ull) >> shift;
            for (; seen_[h] != 0; h = (h + 1) & (seen_.size() - 1))
                if (ops_[seen_[h] - 1].s0 == o.s0 && ops_[seen_[h] - 1].s1 == o.s1)
                    break;
            if (seen_[h] != 0)
            {
                double &th = ops_[seen_[h] - 1].theta;
                const double t = th + o.theta, b = t - th;
                low[seen_[h] - 1 - first] += (th - (t - b)) + (o.theta - b);
                th = t;
                continue;
            }
            seen_[h] = uint32_t(ops_.size() + 1);
            low.push_back(0.0);
        }
        ops_.push_back(o);
    }
    for (size_t i = 0; i < low.size(); i++)
        ops_[first + i].theta = turn(ops_[first + i].theta) + low[i];
    return OK;
}

// One pass: the operations of rest_ from head_ on, in order, that the tile can
// take and that commute with every earlier one that it cannot; the others stay.  The tile's offsets are the lowest address bits (whole 128-byte
// lines) and then the offsets of the gates as they come, while there is room.
// Diagonal gates wait until a gate that does not commute with them, so that
// few windows carry them.
void LdsCircuit::plan()
{
    const unsigned w = std::min(bits_, bits_ <= lds_state_bits(prec_) ? bits_ : lds_tile_bits(prec_));
    const bool whole = w == bits_;
    const unsigned run = whole ? bits_ : (prec_ == C64 ? 4u : 3u);
    const size_t max_windows =
        whole ? std::max<size_t>(1, kTabBytes / (elem_bytes(prec_) << bits_)) : size_t(kLdsWindows);
    vec_.clear();
    piv_.clear();
    red_.clear();
    for (unsigned b = 0; b < run; b++)
    {
        vec_.push_back(1u << b);
        piv_.push_back(b);
        red_.push_back(1u << b);
    }
    order_.clear();
    drafts_.clear();
    later_.clear();
    pending_.clear();
    group_.clear();
    dgates_.clear();
    ddiags_.clear();
    uint32_t ddelta = 0, dalpha = 0, dsel = 0, pend = 0; // unions over what is deferred, and waiting
    size_t windows = 0, diags = 0;
    const uint32_t all = bits_ >= 32 ? ~0u : (1u << bits_) - 1;

    auto close = [&]() {
        if (group_.empty())
            return;
        drafts_.push_back({0u, uint32_t(order_.size()), uint32_t(group_.size())});
        order_.insert(order_.end(), group_.begin(), group_.end());
        group_.clear();
    };
    auto flush = [&]() {
        if (pending_.empty())
            return;
        close();
        drafts_.push_back({2u, uint32_t(order_.size()), uint32_t(pending_.size())});
        order_.insert(order_.end(), pending_.begin(), pending_.end());
        diags += pending_.size();
        windows++;
        pending_.clear();
        pend = 0;
    };
    auto diag_free = [&](const Op &d) {
        if (((d.s0 | d.s1) & ddelta) == 0)
            return true;
        if (simple_)
            return false;
        for (const auto &g : dgates_)
            if (parity(d.s0 & kAlpha32 & g[0]) || parity(d.s1 & kAlpha32 & g[0]))
                return false;
        return true;
    };
    auto gate_free = [&](const Op &g) {
        const uint32_t a = g.s0 & kAlpha32;
        if ((a & ddelta) == 0 && (dalpha & g.delta) == 0 && (dsel & g.delta) == 0)
            return true;
        if (simple_)
            return false;
        for (const auto &o : dgates_)
            if (parity(a & o[0]) || parity(o[1] & g.delta))
                return false;
        for (const auto &d : ddiags_)
            if (parity(d[0] & g.delta) || parity(d[1] & g.delta))
                return false;
        return true;
    };
    auto in_tile = [&](uint32_t delta) {
        if (whole)
            return true;
        uint32_t x = delta;
        for (size_t i = 0; i < red_.size(); i++)
            if ((x >> piv_[i]) & 1u)
                x ^= red_[i];
        if (x == 0)
            return true;
        if (vec_.size() == w)
            return false;
        // the pivot leaves every other row: rows stay fully reduced
        const uint32_t p = 31u - uint32_t(__builtin_clz(x));
        for (size_t i = 0; i < red_.size(); i++)
            if ((red_[i] >> p) & 1u)
                red_[i] ^= x;
        vec_.push_back(x);
        piv_.push_back(p);
        red_.push_back(x);
        return true;
    };

    size_t at = head_;
    for (; at < rest_.size(); at++)
    {
        if (at - head_ >= kMaxScan || drafts_.size() + 4 > kMaxSteps || diags + pending_.size() >= kMaxDiags ||
            dgates_.size() + ddiags_.size() > kMaxDeferred ||
            // every address bit has a deferred gate (a state of no address
            // bits, whose phase gates have constant selectors, has neither)
            (simple_ && ddelta != 0 && ddelta == all))
            break;
        const Op &o = ops_[rest_[at]];
        if (o.kind == 2u)
        {
            if (diag_free(o))
            {
                pending_.push_back(rest_[at]);
                pend |= (o.s0 | o.s1) & kAlpha32;
            }
            else
            {
                later_.push_back(rest_[at]);
                dsel |= (o.s0 | o.s1) & kAlpha32;
                if (!simple_)
                    ddiags_.push_back({o.s0 & kAlpha32, o.s1 & kAlpha32});
            }
            continue;
        }
        if (o.kind == 1u)
        {
            // a controlled gate commutes with nothing here: it takes the
            // pass when nothing is deferred, and ends it otherwise
            if (!later_.empty() || (!pending_.empty() && windows + 2 > max_windows) || !in_tile(o.delta))
                break;
            flush();
            close();
            drafts_.push_back({1u, uint32_t(order_.size()), 1u});
            order_.push_back(rest_[at]);
            continue;
        }
        bool take = gate_free(o);
        if (take)
        {
            bool waits = (pend & o.delta) != 0;
            if (waits && !simple_)
            {
                waits = false;
                for (uint32_t d : pending_)
                    waits = waits || parity(ops_[d].s0 & kAlpha32 & o.delta) || parity(ops_[d].s1 & kAlpha32 & o.delta);
            }
            // the pass's last window is kept for what is still waiting
            if (waits && windows + 2 > max_windows)
                take = false;
            else if (!in_tile(o.delta))
                take = false;
            else
            {
                if (waits)
                    flush();
                bool joins = group_.size() < size_t(kLdsGates);
                for (uint32_t k : group_)
                    joins = joins && !parity(o.s0 & kAlpha32 & ops_[k].delta) &&
                            !parity(ops_[k].s0 & kAlpha32 & o.delta);
                if (!joins)
                    close();
                group_.push_back(rest_[at]);
            }
        }
        if (!take)
        {
            later_.push_back(rest_[at]);
            ddelta |= o.delta;
            dalpha |= o.s0 & kAlpha32;
            if (!simple_)
                dgates_.push_back({o.delta, o.s0 & kAlpha32});
        }
    }
    close();
    flush();
    // what was deferred goes right before the operations not looked at, which
    // stay where they are (moved for every pass, the host's time grew with the
    // square of a circuit's length: 6.1 s for 800 thousand two-bit gates, 0.39
    // now)
    head_ = at - later_.size();
    std::copy(later_.begin(), later_.end(), rest_.begin() + long(head_));
    place();
}

// The pass's coordinates: offsets above the run in ascending order of their
// pivots, the room left taken by the lowest address bits that are no pivot.
void LdsCircuit::place()
{
    const unsigned w = bits_ <= lds_state_bits(prec_) ? bits_ : lds_tile_bits(prec_);
    for (unsigned b = 0; vec_.size() < w; b++)
    {
        if (std::find(piv_.begin(), piv_.end(), b) != piv_.end())
            continue;
        uint32_t x = 1u << b;
        for (size_t i = 0; i < red_.size(); i++)
            if ((red_[i] >> b) & 1u)
                red_[i] ^= x;
        vec_.push_back(x);
        piv_.push_back(b);
        red_.push_back(x);
    }
    // fully reduced rows: row i alone has pivot i, so a vector of the span has
    // coordinate i iff its pivot bit i is set
    std::vector<size_t> idx(w);
    for (size_t i = 0; i < w; i++)
        idx[i] = i;
    std::sort(idx.begin(), idx.end(), [&](size_t a, size_t b) { return piv_[a] < piv_[b]; });
    std::vector<uint32_t> p(w), r(w);
    for (size_t i = 0; i < w; i++)
    {
        p[i] = piv_[idx[i]];
        r[i] = red_[idx[i]];
    }
    piv_.swap(p);
    vec_ = r;
}

struct LdsCircuit::Pass
{
    CPass P;
    const char *steps, *diags, *wins;
    std::vector<std::pair<uint32_t, uint32_t>> ranges; // per window with a table: its diagonal gates
    // tables of 2^P.bits entries that window k comes after
    size_t tables(size_t k) const
    {
        return k + size_t(__builtin_popcount(P.wfull & ((1u << std::min<size_t>(k, 31)) - 1))) * (P.ntiles - 1);
    }
    size_t tables() const
    {
        return tables(ranges.size());
    }
};

int LdsCircuit::stage(Ctx &ctx, bool fresh, Pass &out)
{
    const unsigned w = unsigned(vec_.size());
    const bool tile = w != bits_;
    const bool c64 = prec_ == C64;
    auto coords = [&](uint32_t x) { // of a vector of the span
        if (!tile)
            return x;
        uint32_t l = 0;
        for (unsigned i = 0; i < w; i++)
            l |= ((x >> piv_[i]) & 1u) << i;
        return l;
    };
    auto form = [&](uint32_t sel) { // a selector over the coordinates
        if (!tile)
            return sel;
        uint32_t l = sel & kTrue;
        for (unsigned i = 0; i < w; i++)
            l |= uint32_t(parity(sel & kAlpha32 & vec_[i])) << i;
        return l;
    };
    auto index = [&](uint32_t l) { return c64 ? lds_index<true>(l) : lds_index<false>(l); };
    bool units = true;
    for (unsigned i = 0; i < w; i++)
        units = units && vec_[i] == (1u << piv_[i]);
    CPass &P = out.P;
    std::memset(&P, 0, sizeof(P));
    uint32_t mask = 0;
    for (unsigned i = 0; i < w; i++)
    {
        P.vec[i] = vec_[i];
        P.piv[i] = piv_[i];
        mask |= 1u << piv_[i];
    }
    P.bits = w;
    P.outer = bits_ - w;
    P.ntiles = 1u << P.outer;
    P.fresh = fresh;
    std::vector<int> outer;
    for (unsigned b = 0; b < bits_; b++)
        if (!((mask >> b) & 1u))
            outer.push_back(int(b));

    std::vector<LdsStep> steps(drafts_.size());
    std::vector<LdsDiag> diags;
    std::vector<LdsWin> wins;
    std::vector<DiagGate> win;
    Poly poly;
    for (size_t s = 0; s < drafts_.size(); s++)
    {
        const Draft &d = drafts_[s];
        LdsStep &st = steps[s];
        std::memset(&st, 0, sizeof(st));
        st.kind = d.kind;
        st.count = d.count;
        if (d.kind != 2u)
        {
            uint32_t pv[kLdsGates] = {}, rd[kLdsGates] = {};
            for (uint32_t j = 0; j < d.count; j++)
            {
                const Op &o = ops_[order_[d.first + j]];
                const uint32_t l = coords(o.delta);
                st.slot[j] = index(l);
                st.sel[j] = form(o.s0);
                st.full[j] = tile ? o.s0 & kAlpha32 : 0u;
                for (int e = 0; e < 8; e++)
                {
                    if (c64)
                        st.uf[j][e] = float(mats_[o.mat][size_t(e)]);
                    else
                        st.u[j][e] = mats_[o.mat][size_t(e)];
                }
                uint32_t x = l;
                for (uint32_t k = 0; k < j; k++)
                    if ((x >> pv[k]) & 1u)
                        x ^= rd[k];
                pv[j] = uint32_t(__builtin_ctz(x));
                rd[j] = x;
                if (d.kind == 1u)
                {
                    st.ctrl = form(o.s1);
                    st.slot[3] = l;
                    st.full[3] = tile ? o.s1 & kAlpha32 : 0u;
                }
            }
            std::sort(pv, pv + d.count);
            for (uint32_t j = 0; j < d.count; j++)
                st.pivot |= pv[j] << (8 * j);
            continue;
        }
        const uint32_t g0 = uint32_t(diags.size());
        win.clear();
        for (uint32_t j = 0; j < d.count && tile; j++)
        {
            const Op &o = ops_[order_[d.first + j]];
            win.push_back({uint64_t(o.s0 & kAlpha32) | (uint64_t(o.s0 >> 31) << 63),
                           o.s1 == kTrue ? kNoSel : uint64_t(o.s1 & kAlpha32) | (uint64_t(o.s1 >> 31) << 63),
                           o.theta});
        }
        const bool table = !tile || (units && window_is_polynomial(bits_, win.data(), win.size()));
        // (over the tile index and the coordinates, where a table has them all)
        const bool full = !table && bits_ <= lds_table_bits(prec_);
        auto index_form = [&](uint32_t sel) {
            uint32_t t = 0;
            for (size_t k = 0; k < outer.size() && full; k++)
                t |= ((sel >> outer[k]) & 1u) << (w + k);
            return t;
        };
        for (uint32_t j = 0; j < d.count; j++)
        {
            const Op &o = ops_[order_[d.first + j]];
            const uint32_t s0 = form(o.s0) | index_form(o.s0), s1 = form(o.s1) | index_form(o.s1);
            if (!table || (s0 != 0 && s1 != 0)) // (a table's gate that needs a bit outside the tile holds nowhere in it)
                diags.push_back({s0, s1, tile ? o.s0 & kAlpha32 : 0u, tile ? o.s1 & kAlpha32 : 0u, turn(o.theta), 0.0});
        }
        if (!table && !full)
        {
            st.kind = 3u;
            st.slot[0] = g0;
            st.slot[1] = uint32_t(diags.size());
            continue;
        }
        P.wfull |= uint32_t(full) << (tile ? out.ranges.size() : 0);
        out.ranges.push_back({g0, uint32_t(diags.size())});
        if (!tile)
            continue;
        wins.emplace_back();
        LdsWin &W = wins.back();
        std::memset(&W, 0, sizeof(W));
        if (full)
            continue;
        window_polynomial(bits_, win.data(), win.size(), poly);
        for (size_t k = 0; k < outer.size(); k++)
        {
            for (unsigned i = 0; i < w; i++)
                W.m[i][k] = turn(poly.q(int(piv_[i]), outer[k]));
            W.m[13][k] = turn(poly.L[size_t(outer[k])]);
            for (size_t l = k + 1; l < outer.size(); l++)
                W.q[k][l] = turn(poly.q(outer[k], outer[l]));
        }
    }
    P.nsteps = uint32_t(steps.size());
    P.nwin = uint32_t(out.ranges.size());

    const size_t diag_off = steps.size() * sizeof(LdsStep);
    const size_t win_off = diag_off + diags.size() * sizeof(LdsDiag);
    std::vector<char> blob(win_off + wins.size() * sizeof(LdsWin));
    auto put = [&](size_t off, const void *src, size_t bytes) {
        if (bytes)
            std::memcpy(blob.data() + off, src, bytes);
    };
    put(0, steps.data(), diag_off);
    put(diag_off, diags.data(), diags.size() * sizeof(LdsDiag));
    put(win_off, wins.data(), wins.size() * sizeof(LdsWin));
    void *d = nullptr;
    if (!blob.empty())
        ZXA_TRY(ctx.ring.stage(blob.data(), blob.size(), ctx.stream, &d));
    out.steps = static_cast<const char *>(d);
    out.diags = out.steps + diag_off;
    out.wins = out.steps + win_off;
    return OK;
}

// Launches staged passes: their tables' copy, every window table at once, and
// the passes one after the other.
int LdsCircuit::launch(Ctx &ctx, void *state, const std::vector<Pass> &passes)
{
    const bool c64 = prec_ == C64;
    const uint32_t w = passes[0].P.bits;
    const bool tile = w != bits_;
    // (a window with a table per tile twice: its factors, and its table)
    std::vector<WinTask> tasks, wide;
    size_t ntab = 0;
    for (const Pass &p : passes)
    {
        for (size_t k = 0; k < p.ranges.size(); k++)
        {
            WinTask t = {reinterpret_cast<uint64_t>(p.diags) + p.ranges[k].first * sizeof(LdsDiag),
                         p.ranges[k].second - p.ranges[k].first,
                         reinterpret_cast<uint64_t>(p.wins) + (tile ? k * sizeof(LdsWin) : 0),
                         uint64_t(ntab + p.tables(k)) << w};
            if (tile && ((p.P.wfull >> k) & 1u))
            {
                wide.push_back(t);
                t.out = kNoTable;
            }
            tasks.push_back(t);
        }
        ntab += p.tables();
    }
    const size_t nwin = tasks.size();
    tasks.insert(tasks.end(), wide.begin(), wide.end());
    void *dr = nullptr;
    if (!tasks.empty())
        ZXA_TRY(ctx.ring.stage(tasks.data(), tasks.size() * sizeof(WinTask), ctx.stream, &dr));
    ZXA_TRY(ctx.ring.flush(ctx.stream));
    // tables, then factors
    char *tabs = nullptr;
    double2 *factors = nullptr;
    if (!tasks.empty())
    {
        const uint32_t outer = passes[0].P.outer;
        auto need = [&](size_t tables, size_t windows) {
            return (tables << w) * elem_bytes(prec_) + (tile ? (windows << outer) * kFactors * sizeof(double2) : 0);
        };
        // passes to come: the largest lot's at once (an allocation that grows
        // under way waits for the device, 1 ms of a first run in all)
        size_t bytes = need(ntab, nwin);
        if (left())
        {
            const size_t most = kMaxLot * kLdsWindows;
            bytes = std::max(bytes, need(most, most));
            if (tile && !wide.empty())
                bytes = std::max(bytes, need((kTabBytes >> w) / elem_bytes(prec_) + (size_t(kLdsWindows) << outer), most));
        }
        ZXA_TRY(ctx.scratch_a.ensure(bytes));
        tabs = static_cast<char *>(ctx.scratch_a.ptr);
        factors = reinterpret_cast<double2 *>(tabs + (ntab << w) * elem_bytes(prec_));
        const WinTask *tk = static_cast<const WinTask *>(dr);
        auto run = [&](uint32_t tblocks, uint32_t fblocks, size_t first, size_t count, uint32_t bits) {
            const dim3 grid(tblocks + fblocks, unsigned(count));
            if (c64)
                hipLaunchKernelGGL(window_kernel<true>, grid, dim3(256), 0, ctx.stream, tk + first, bits, tblocks,
                                   outer, reinterpret_cast<float2 *>(tabs), factors);
            else
                hipLaunchKernelGGL(window_kernel<false>, grid, dim3(256), 0, ctx.stream, tk + first, bits, tblocks,
                                   outer, reinterpret_cast<double2 *>(tabs), factors);
            return hip_check(hipGetLastError(), "window kernel launch");
        };
        ZXA_TRY(run(((1u << w) + 255u) / 256u, tile ? ((1u << outer) + 3u) / 4u : 0u, 0, nwin, w));
        if (!wide.empty())
            ZXA_TRY(run(((1u << bits_) + 255u) / 256u, 0, nwin, wide.size(), bits_));
    }
    for (const Pass &p : passes)
    {
        const LdsStep *ds = reinterpret_cast<const LdsStep *>(p.steps);
        const LdsDiag *dd = reinterpret_cast<const LdsDiag *>(p.diags);
        // (LDS holds two workgroups per compute unit; the registers run them
        // one after the other)
        const uint32_t nt = std::min(uint32_t(kThreads), std::max(64u, (1u << w) >> 3));
        const uint32_t grid = std::min(p.P.ntiles, 2u * uint32_t(ctx.num_cus > 0 ? ctx.num_cus : 256));
        ZXA_TRY(ctx.tic());
        const bool full = p.P.wfull != 0;
        if (c64 && tile)
            hipLaunchKernelGGL((full ? circuit_kernel<true, true, true> : circuit_kernel<true, true, false>),
                               dim3(grid), dim3(nt), 0, ctx.stream,
                               static_cast<float2 *>(state), p.P, ds, dd, reinterpret_cast<const float2 *>(tabs),
                               factors);
        else if (c64)
            hipLaunchKernelGGL((circuit_kernel<true, false>), dim3(1), dim3(nt), 0, ctx.stream,
                               static_cast<float2 *>(state), p.P, ds, dd, reinterpret_cast<const float2 *>(tabs),
                               factors);
        else if (tile)
            hipLaunchKernelGGL((full ? circuit_kernel<false, true, true> : circuit_kernel<false, true, false>),
                               dim3(grid), dim3(nt), 0, ctx.stream,
                               static_cast<double2 *>(state), p.P, ds, dd,
                               reinterpret_cast<const double2 *>(tabs), factors);
        else
            hipLaunchKernelGGL((circuit_kernel<false, false>), dim3(1), dim3(nt), 0, ctx.stream,
                               static_cast<double2 *>(state), p.P, ds, dd,
                               reinterpret_cast<const double2 *>(tabs), factors);
        ZXA_HIP(hipGetLastError());
        ZXA_TRY(ctx.toc(F_FUSED, (p.P.fresh ? 1ull : 2ull) * (uint64_t(1) << bits_) * elem_bytes(prec_)));
        if (tabs)
        {
            tabs += (p.tables() << w) * elem_bytes(prec_);
            factors += tile ? (size_t(p.P.nwin) << p.P.outer) * kFactors : 0;
        }
    }
    return ctx.ring.done(ctx.stream);
}

void LdsCircuit::start()
{
    rest_.resize(ops_.size());
    for (size_t i = 0; i < ops_.size(); i++)
        rest_[i] = uint32_t(i);
    head_ = 0;
}

int LdsCircuit::next_pass()
{
    const size_t before = head_;
    plan();
    if (head_ == before && left())
    {
        set_error("circuit: no operation fits a pass");
        return ESTATE;
    }
    return OK;
}

int LdsCircuit::schedule(uint32_t *order, uint32_t *pass_of)
{
    size_t at = 0;
    uint32_t pass = 0;
    for (start(); left(); pass++)
    {
        ZXA_TRY(next_pass());
        for (uint32_t o : order_)
        {
            order[at] = o;
            pass_of[at++] = pass;
        }
    }
    return OK;
}

int LdsCircuit::run(Ctx &ctx, void *state)
{
    start();
    // the first pass by itself, then three and up to eight with one table
    // copy and one table launch: the device works on one lot while the host
    // plans the next
    bool fresh = true;
    size_t lot = 1;
    std::vector<Pass> passes;
    while (fresh || left())
    {
        struct Batch // dropped on an error return
        {
            ParamRing &r;
            ~Batch()
            {
                r.end_batch();
            }
        } batch{ctx.ring};
        ZXA_TRY(ctx.ring.begin_batch());
        passes.clear();
        size_t tabs = 0;
        while ((fresh || left()) && passes.size() < lot && tabs < kTabBytes)
        {
            ZXA_TRY(next_pass());
            passes.emplace_back();
            ZXA_TRY(stage(ctx, fresh, passes.back()));
            tabs += (passes.back().tables() << passes.back().P.bits) * elem_bytes(prec_);
            fresh = false;
        }
        ZXA_TRY(launch(ctx, state, passes));
        lot = std::min(kMaxLot, lot * 3);
    }
    return OK;
}

} // namespace zxa
