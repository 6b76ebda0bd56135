// kernels_small.hip -- whole circuits on a state held in one compute unit's
// LDS (complex128 to 13 bits, complex64 to 14; see small.h).
#include "small.h"

#include <algorithm>
#include <cstring>

namespace zxa
{
namespace
{

constexpr int kMaxThreads = 1024;

template <bool kC64>
struct SGeo;
template <>
struct SGeo<false>
{
    using T = double2;
    using R = double;
    static constexpr int kBits = 13;
    static constexpr int kPer = 8;  // amplitudes per thread at 2^kBits
    static constexpr int kSwz = 3;  // 16-byte LDS words: eight to 128 bytes
};
template <>
struct SGeo<true>
{
    using T = float2;
    using R = float;
    static constexpr int kBits = 14;
    static constexpr int kPer = 16;
    static constexpr int kSwz = 4; // 8-byte LDS words: sixteen to 128 bytes
};

// LDS index of an amplitude: the address with its low bits (one 128-byte row)
// XORed with the fields above them, so that lanes whose addresses differ in
// any kSwz consecutive bits touch different banks.  Linear over XOR: an
// element's index is the base's XOR the offset's.
template <bool kC64>
__host__ __device__ __forceinline__ uint32_t lds_index(uint32_t a)
{
    constexpr int S = SGeo<kC64>::kSwz;
    const uint32_t f = (a >> S) ^ (a >> (2 * S)) ^ (a >> (3 * S)) ^ (a >> (4 * S));
    return a ^ (f & ((1u << S) - 1));
}

__device__ __forceinline__ uint32_t odd(uint32_t sel, uint32_t x)
{
    return (__popc(x & sel & 0x7fffffffu) & 1u) ^ (sel >> 31);
}

__device__ __forceinline__ uint32_t insert_zero(uint32_t x, uint32_t p)
{
    const uint32_t lo = x & ((1u << p) - 1);
    return ((x >> p) << (p + 1)) | lo;
}

// K commuting gates on every coset of their offsets: a thread reads the
// coset's 2^K amplitudes, applies the gates in registers and writes them back.
// Gate i pairs the elements that differ in its offset; because the other
// gates' offsets leave its selector unchanged, the side of the pair's first
// element is the selector's parity over the coset's base, so one lookup per
// gate (the matrix or its mirror, by address) serves every pair.
template <bool kC64, int K, bool kCtrl>
__device__ __forceinline__ void gates_step(typename SGeo<kC64>::T *amp, const SmallStep &st, uint32_t bits)
{
    using T = typename SGeo<kC64>::T;
    using R = typename SGeo<kC64>::R;
    constexpr int N = 1 << K;
    const uint32_t total = 1u << (bits - K);
    for (uint32_t b = threadIdx.x; b < total; b += blockDim.x)
    {
        uint32_t base = b;
        const uint32_t pv = st.pivot;
#pragma unroll
        for (int j = 0; j < K; j++)
            base = insert_zero(base, (pv >> (8 * j)) & 0xffu);
        const uint32_t a0 = lds_index<kC64>(base);
        uint32_t off[N];
        off[0] = a0;
#pragma unroll
        for (int j = 0; j < K; j++)
        {
            const uint32_t d = st.slot[j];
#pragma unroll
            for (int c = 0; c < (1 << j); c++)
                off[(1 << j) + c] = off[c] ^ d;
        }
        T v[N];
#pragma unroll
        for (int c = 0; c < N; c++)
            v[c] = amp[off[c]];
#pragma unroll
        for (int j = 0; j < K; j++)
        {
            const uint32_t f = odd(st.sel[j], base);
            if constexpr (kCtrl)
            {
                // the even-side element decides (its unswizzled address is
                // the base, or the base XOR the offset kept in slot[3])
                if (!odd(st.ctrl, f ? base ^ st.slot[3] : base))
                    continue;
            }
            const double2 *u = reinterpret_cast<const double2 *>(st.u[j]);
            const uint32_t m = f ? 3u : 0u;
            const double2 d00 = u[0 ^ m], d01 = u[1 ^ m], d10 = u[2 ^ m], d11 = u[3 ^ m];
            const R m00x = R(d00.x), m00y = R(d00.y), m01x = R(d01.x), m01y = R(d01.y);
            const R m10x = R(d10.x), m10y = R(d10.y), m11x = R(d11.x), m11y = R(d11.y);
#pragma unroll
            for (int c = 0; c < N; c++)
            {
                if (c & (1 << j))
                    continue;
                const T p = v[c], q = v[c | (1 << j)];
                T np, nq;
                np.x = m00x * p.x - m00y * p.y + m01x * q.x - m01y * q.y;
                np.y = m00x * p.y + m00y * p.x + m01x * q.y + m01y * q.x;
                nq.x = m10x * p.x - m10y * p.y + m11x * q.x - m11y * q.y;
                nq.y = m10x * p.y + m10y * p.x + m11x * q.y + m11y * q.x;
                v[c] = np;
                v[c | (1 << j)] = nq;
            }
        }
#pragma unroll
        for (int c = 0; c < N; c++)
            amp[off[c]] = v[c];
    }
}

// The window phases exp(i sum of the gates' angles), one table of 2^bits
// entries per window: every window of the circuit at once, over the whole
// chip, so that the circuit kernel (one compute unit) evaluates no selector
// and no sine.
template <bool kC64>
__global__ __launch_bounds__(256) void small_phase_kernel(const uint32_t *__restrict__ wins,
                                                          const uint4 *__restrict__ gates, uint32_t bits,
                                                          typename SGeo<kC64>::T *__restrict__ out)
{
    const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >> bits)
        return;
    const uint32_t w = blockIdx.y;
    const uint32_t g0 = wins[w], g1 = wins[w + 1];
    double th = 0.0;
    for (uint32_t g = g0; g < g1; g++)
    {
        const uint4 e = gates[g]; // s0, s1, theta
        const double t = __hiloint2double(int(e.w), int(e.z));
        th += (odd(e.x, x) & odd(e.y, x)) ? t : 0.0;
    }
    double s, c;
    sincos(th, &s, &c);
    typename SGeo<kC64>::T r;
    r.x = c;
    r.y = s;
    out[(uint64_t(w) << bits) + x] = r;
}

// The circuit: one workgroup, the state in LDS from the first step to the
// last.  A step costs one LDS read and write of the state and a barrier
// (three gates per step: 8192 complex128 amplitudes are 2 x 128 KiB per step
// at 128 bytes a cycle, and about as many FP64 cycles), so the step count
// decides; a launch per gate, as the pair kernel did it, costs more than a
// step even on one compute unit.  10 qubits, 40 gates: 30 launches of 1.8 us
// and their gaps before.  The steps come through LDS in chunks, and a
// window's phases are loaded before the steps ahead of it run, so no step
// waits for memory.  Above 2^13 (2^14) amplitudes the state leaves LDS and
// the tile passes take over.
constexpr int kChunk = 112;
template <bool kC64>
__global__ __launch_bounds__(kMaxThreads) void small_circuit_kernel(typename SGeo<kC64>::T *__restrict__ state,
                                                                    uint32_t bits,
                                                                    const uint4 *__restrict__ steps, uint32_t nsteps,
                                                                    const typename SGeo<kC64>::T *__restrict__ phases,
                                                                    uint32_t nwin, int fresh)
{
    using G = SGeo<kC64>;
    using T = typename G::T;
    __shared__ T amp[1 << G::kBits];
    __shared__ uint4 buf[kChunk * (sizeof(SmallStep) / 16)];
    const uint32_t tid = threadIdx.x, nt = blockDim.x, size = 1u << bits;
    T pf[G::kPer];
    uint32_t win = 0;
    auto fetch = [&]() {
        if (win < nwin)
        {
            const T *src = phases + (uint64_t(win) << bits);
#pragma unroll
            for (int k = 0; k < G::kPer; k++)
            {
                const uint32_t i = tid + k * nt;
                if (i < size)
                    pf[k] = src[i];
            }
        }
    };
    fetch();
    for (uint32_t i = tid; i < size; i += nt)
    {
        T z;
        z.x = (i == 0);
        z.y = 0;
        amp[lds_index<kC64>(i)] = fresh ? z : state[i];
    }
    constexpr uint32_t kUnits = sizeof(SmallStep) / 16;
    for (uint32_t s0 = 0; s0 < nsteps; s0 += kChunk)
    {
        const uint32_t ns = min(nsteps - s0, uint32_t(kChunk));
        // (the last step of the previous chunk ended with a barrier)
        for (uint32_t i = tid; i < ns * kUnits; i += nt)
            buf[i] = steps[s0 * kUnits + i];
        __syncthreads();
        for (uint32_t s = 0; s < ns; s++)
        {
            const SmallStep &st = reinterpret_cast<const SmallStep *>(buf)[s];
            const uint32_t kind = __builtin_amdgcn_readfirstlane(st.kind);
            const uint32_t count = __builtin_amdgcn_readfirstlane(st.count);
            if (kind == 0)
            {
                if (count == 3)
                    gates_step<kC64, 3, false>(amp, st, bits);
                else if (count == 2)
                    gates_step<kC64, 2, false>(amp, st, bits);
                else
                    gates_step<kC64, 1, false>(amp, st, bits);
            }
            else if (kind == 1)
                gates_step<kC64, 1, true>(amp, st, bits);
            else
            {
#pragma unroll
                for (int k = 0; k < G::kPer; k++)
                {
                    const uint32_t i = tid + k * nt;
                    if (i < size)
                    {
                        const uint32_t a = lds_index<kC64>(i);
                        const T v = amp[a], p = pf[k];
                        T r;
                        r.x = v.x * p.x - v.y * p.y;
                        r.y = v.x * p.y + v.y * p.x;
                        amp[a] = r;
                    }
                }
                win++;
                fetch();
            }
            __syncthreads();
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < size; i += nt)
        state[i] = amp[lds_index<kC64>(i)];
}

template <bool kC64>
int launch(Ctx &ctx, void *state, uint32_t bits, const char *blob, size_t nsteps, size_t nwin, size_t win_off,
           size_t diag_off, bool fresh)
{
    using T = typename SGeo<kC64>::T;
    T *phases = nullptr;
    if (nwin)
    {
        ZXA_TRY(ctx.scratch_a.ensure((nwin << bits) * sizeof(T)));
        phases = static_cast<T *>(ctx.scratch_a.ptr);
        const uint32_t nt = std::min(256u, std::max(64u, 1u << bits));
        const dim3 grid(((1u << bits) + nt - 1) / nt, unsigned(nwin));
        hipLaunchKernelGGL(small_phase_kernel<kC64>, grid, dim3(nt), 0, ctx.stream,
                           reinterpret_cast<const uint32_t *>(blob + win_off),
                           reinterpret_cast<const uint4 *>(blob + diag_off), bits, phases);
        ZXA_HIP(hipGetLastError());
    }
    const uint32_t nt = std::max(64u, (1u << bits) / uint32_t(SGeo<kC64>::kPer));
    hipLaunchKernelGGL(small_circuit_kernel<kC64>, dim3(1), dim3(nt), 0, ctx.stream, static_cast<T *>(state), bits,
                       reinterpret_cast<const uint4 *>(blob), uint32_t(nsteps), phases, uint32_t(nwin), int(fresh));
    return hip_check(hipGetLastError(), "small_circuit_kernel launch");
}

constexpr uint64_t kAlpha = (uint64_t(1) << 63) - 1;
constexpr size_t kPhaseBytes = size_t(32) << 20; // window tables of one run

uint32_t pack32(uint64_t sel)
{
    return uint32_t(sel & 0x7fffffffu) | (uint32_t(sel >> 63) << 31);
}

bool parity(uint64_t x)
{
    return (__builtin_popcountll(x) & 1) != 0;
}

} // namespace

void SmallCircuit::begin(unsigned bits, int prec)
{
    bits_ = bits;
    prec_ = prec;
    fresh_ = true;
    steps_.clear();
    diags_.clear();
    wins_.clear();
    group_.clear();
}

size_t SmallCircuit::blob_bytes() const
{
    return steps_.size() * sizeof(SmallStep) + diags_.size() * sizeof(Diag) +
           (wins_.size() + 1) * sizeof(uint32_t) + 64;
}

// Runs what is pending when `more` bytes would not fit the parameter slot.
int SmallCircuit::room(Ctx &ctx, void *state, size_t more)
{
    const size_t esz = elem_bytes(prec_);
    if (blob_bytes() + 2 * sizeof(SmallStep) + more > ParamRing::kSlotBytes ||
        (((wins_.size() + 1) << bits_) * esz > kPhaseBytes && !wins_.empty()))
        return run(ctx, state);
    return OK;
}

// The step of the pending group: pivots by elimination over the offsets.
void SmallCircuit::close()
{
    if (group_.empty())
        return;
    SmallStep st;
    std::memset(&st, 0, sizeof(st));
    st.count = uint32_t(group_.size());
    uint32_t piv[3] = {0, 0, 0};
    uint32_t red[3];
    for (size_t i = 0; i < group_.size(); i++)
    {
        const uint32_t d = uint32_t(group_[i].delta);
        st.slot[i] = prec_ == C64 ? lds_index<true>(d) : lds_index<false>(d);
        st.sel[i] = pack32(group_[i].packed_sel);
        std::memcpy(st.u[i], group_[i].u, sizeof(st.u[i]));
        uint32_t r = d;
        for (size_t j = 0; j < i; j++)
            if ((r >> piv[j]) & 1u)
                r ^= red[j];
        piv[i] = uint32_t(__builtin_ctz(r));
        red[i] = r;
    }
    std::sort(piv, piv + group_.size());
    for (size_t i = 0; i < group_.size(); i++)
        st.pivot |= piv[i] << (8 * i);
    steps_.push_back(st);
    group_.clear();
}

int SmallCircuit::push(const U3Gate &g, const uint64_t *ctrl)
{
    const uint64_t a = g.packed_sel & kAlpha;
    if (g.delta == 0 || (g.delta >> bits_) != 0 || (a >> bits_) != 0 || !parity(a & g.delta))
    {
        set_error("small circuit: the selector does not separate the pair, or reaches outside the state");
        return EINVAL_;
    }
    bool joins = !ctrl && group_.size() < 3;
    for (const U3Gate &o : group_)
        joins = joins && !parity(a & o.delta) && !parity(o.packed_sel & kAlpha & g.delta);
    if (!joins)
        close();
    group_.push_back(g);
    if (ctrl)
    {
        close();
        steps_.back().kind = 1;
        steps_.back().ctrl = pack32(*ctrl);
        steps_.back().slot[3] = uint32_t(g.delta);
    }
    return OK;
}

int SmallCircuit::gate(Ctx &ctx, void *state, const U3Gate &g)
{
    ZXA_TRY(room(ctx, state, sizeof(SmallStep)));
    return push(g, nullptr);
}

int SmallCircuit::swap(Ctx &ctx, void *state, uint64_t delta, uint64_t sel, const uint64_t *ctrl)
{
    ZXA_TRY(room(ctx, state, sizeof(SmallStep)));
    const U3Gate g = {sel, delta, {0, 0, 1, 0, 1, 0, 0, 0}};
    return push(g, ctrl);
}

int SmallCircuit::window(Ctx &ctx, void *state, const DiagGate *gates, size_t ngates)
{
    // a window larger than a quarter of a parameter slot goes in parts
    const size_t per = ParamRing::kSlotBytes / 4 / sizeof(Diag);
    for (size_t o = 0; o < ngates; o += per)
    {
        const size_t n = std::min(per, ngates - o);
        ZXA_TRY(room(ctx, state, sizeof(SmallStep) + n * sizeof(Diag)));
        close();
        wins_.push_back(uint32_t(diags_.size()));
        for (size_t i = o; i < o + n; i++)
        {
            const DiagGate &d = gates[i];
            if (((d.s0 & kAlpha) >> bits_) != 0 || (d.s1 != kNoSel && ((d.s1 & kAlpha) >> bits_) != 0))
            {
                set_error("small circuit: diagonal selector outside the state");
                return EINVAL_;
            }
            // a missing second selector is the constant one (alpha 0, beta 1)
            diags_.push_back({pack32(d.s0), d.s1 == kNoSel ? 0x80000000u : pack32(d.s1), d.theta});
        }
        SmallStep st;
        std::memset(&st, 0, sizeof(st));
        st.kind = 2;
        steps_.push_back(st);
    }
    return OK;
}

int SmallCircuit::run(Ctx &ctx, void *state)
{
    close();
    if (!fresh_ && steps_.empty())
        return OK;
    static_assert(sizeof(Diag) == 16 && sizeof(SmallStep) % 16 == 0, "16-byte units");
    const size_t diag_off = steps_.size() * sizeof(SmallStep);
    const size_t win_off = diag_off + diags_.size() * sizeof(Diag);
    const size_t nwin = wins_.size(), nsteps = steps_.size();
    std::vector<char> blob(win_off + (nwin + 1) * sizeof(uint32_t));
    if (nsteps)
        std::memcpy(blob.data(), steps_.data(), diag_off);
    if (!diags_.empty())
        std::memcpy(blob.data() + diag_off, diags_.data(), diags_.size() * sizeof(Diag));
    wins_.push_back(uint32_t(diags_.size()));
    std::memcpy(blob.data() + win_off, wins_.data(), wins_.size() * sizeof(uint32_t));
    const bool fresh = fresh_;
    fresh_ = false;
    steps_.clear();
    diags_.clear();
    wins_.clear();
    void *d = nullptr;
    ZXA_TRY(ctx.ring.stage(blob.data(), blob.size(), ctx.stream, &d));
    ZXA_TRY(ctx.tic());
    const char *p = static_cast<const char *>(d);
    ZXA_TRY(prec_ == C64 ? launch<true>(ctx, state, bits_, p, nsteps, nwin, win_off, diag_off, fresh)
                         : launch<false>(ctx, state, bits_, p, nsteps, nwin, win_off, diag_off, fresh));
    ZXA_TRY(ctx.toc(F_FUSED, (fresh ? 1ull : 2ull) * (uint64_t(1) << bits_) * elem_bytes(prec_)));
    return ctx.ring.done(ctx.stream);
}

} // namespace zxa
