// small.h -- circuits on states that fit one compute unit's LDS.
//
// The engine's fused policy hands every operation of such a circuit to a
// SmallCircuit instead of launching it; run() executes them all in one
// launch (and one before it that tabulates the diagonal windows).
#pragma once

#include "dev.h"

#include <cstdint>
#include <vector>

namespace zxa
{

// Widest state (address bits) of a SmallCircuit: 128 KiB of amplitudes.
constexpr unsigned small_max_bits(int prec)
{
    return prec == C64 ? 14u : 13u;
}

// A step of the kernel: up to three gates that commute pairwise, or one
// gate with a control selector, or a diagonal window.  Selectors are packed
// as alpha | beta << 31.  16-byte aligned: the kernel copies steps in 16-byte
// units.
struct alignas(16) SmallStep
{
    uint32_t kind;     // 0: gates, 1: controlled gate, 2: window
    uint32_t count;    // gates
    uint32_t pivot;    // byte j: j-th pivot bit (ascending) of the gates' offsets
    uint32_t ctrl;     // kind 1: the control selector
    uint32_t slot[4];  // per gate: its offset as an LDS index (swizzled)
    uint32_t sel[4];   // per gate: its selector
    double u[3][8];    // per gate: u00, u01, u10, u11 (re, im)
};

class SmallCircuit
{
  public:
    void begin(unsigned bits, int prec);
    // One U3 (any offset, any selector with alpha . delta = 1).
    int gate(Ctx &ctx, void *state, const U3Gate &g);
    // Swaps each pair of x (delta, sel): where ctrl is given, only the pairs
    // whose even-side element the control selects.
    int swap(Ctx &ctx, void *state, uint64_t delta, uint64_t sel, const uint64_t *ctrl);
    int window(Ctx &ctx, void *state, const DiagGate *gates, size_t ngates);
    // Runs what is pending on the state (2^bits amplitudes); the first run
    // after begin() starts from |0...0>, which need not have been written.
    int run(Ctx &ctx, void *state);

  private:
    struct Diag
    {
        uint32_t s0, s1;
        double theta;
    };
    int push(const U3Gate &g, const uint64_t *ctrl);
    void close();
    int room(Ctx &ctx, void *state, size_t more);
    size_t blob_bytes() const;
    unsigned bits_ = 0;
    int prec_ = 0;
    bool fresh_ = true;
    std::vector<SmallStep> steps_;
    std::vector<Diag> diags_;
    std::vector<uint32_t> wins_; // first gate of each window, in order
    std::vector<U3Gate> group_;  // gates of the step being formed
};

} // namespace zxa
