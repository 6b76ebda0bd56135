// circuit.h -- circuits executed out of LDS.
//
// The engine's fused policy hands the operations of a circuit on a small or
// middling state to an LdsCircuit instead of launching them; run() plans them
// into passes and launches those.  A state that fits one compute unit's LDS
// takes one pass for the whole circuit.  A wider state is swept tile by tile, a
// pass applying every operation, of whatever layer, that its tile's address
// bits allow.
#pragma once

#include "dev.h"

#include <array>
#include <cstdint>
#include <vector>

namespace zxa
{

// Widest state (address bits) held whole: 128 KiB of amplitudes.
constexpr unsigned lds_state_bits(int prec)
{
    return prec == C64 ? 14u : 13u;
}
// Address bits of a tile of a wider state: 64 KiB of amplitudes.
constexpr unsigned lds_tile_bits(int prec)
{
    return prec == C64 ? 13u : 12u;
}
// Widest state whose windows that do not split by tile and coordinate (after
// CX transport) are tabulated over all amplitudes, by every compute unit before
// the pass, rather than summed gate by gate in the tiles, by as many as there
// are tiles.  Four layers with 100 transported CP gates each, in us, gate by
// gate and tabulated (and in tile passes): complex128, 14 bits 339, 200 (295),
// 18 bits 391, 294 (351); complex64, 16 bits 575, 250 (358), 20 bits 658, 503
// (600).  A table of 2^20 complex128 or 2^21 complex64 amplitudes, 16 MiB each,
// takes the whole chip as long as the tiles take, which have a compute unit
// each there (0.6 and 0.44 us a gate).
constexpr unsigned lds_table_bits(int prec)
{
    return prec == C64 ? 20u : 18u;
}
constexpr int kLdsOuter = 10;  // most address bits outside a tile
constexpr int kLdsWindows = 8; // most windows of a pass over tiles

constexpr int kLdsGates = 3;   // most gates of a step (four, at 256 threads, ran 7% slower)

// A step of the kernel: up to three gates that commute pairwise, or one gate
// with a control selector, or a diagonal window.  Offsets and selectors are
// in tile coordinates, selectors packed as alpha | beta << 31.  Read through
// the scalar cache.
struct alignas(64) LdsStep
{
    uint32_t kind;    // 0: gates, 1: controlled gate, 2: window, 3: window gate by gate
    uint32_t count;   // gates
    uint32_t pivot;   // byte j: j-th pivot bit (ascending) of the gates' offsets
    uint32_t ctrl;    // kind 1: the control selector
    uint32_t slot[4];         // per gate: its offset as an LDS index (kind 1: slot[3] unswizzled;
                              // kind 3: first and one past the last of the pass's diagonal gates)
    uint32_t sel[4];          // per gate: its selector
    uint32_t full[4];         // per gate: its selector over the tile's base address (kind 1: full[3] the control's)
    union                     // per gate: u00, u01, u10, u11 (re, im), in the state's precision
    {
        double u[kLdsGates][8];
        float uf[kLdsGates][8];
    };
};

// A diagonal gate in tile coordinates: theta where both selectors hold; f0,
// f1 are the selectors over the tile's base address.
struct alignas(16) LdsDiag
{
    uint32_t s0, s1, f0, f1;
    double theta, pad;
};

// A window's phase in a tile: T[l] (by the coordinates alone, tabulated) times
// exp(i (C + sum_i c_i l_i)), c and C linear and quadratic in the tile index's
// bits: c_i = sum_k m[i][k], C = sum_k (m[13][k] + sum_{l > k} q[k][l]).
struct LdsWin
{
    double m[14][kLdsOuter];
    double q[kLdsOuter][kLdsOuter];
};

class LdsCircuit
{
  public:
    void begin(unsigned bits, int prec);
    // One U3 (any offset, any selector with alpha . delta = 1).
    int gate(const U3Gate &g);
    // Swaps each pair of x (delta, sel): where ctrl is given, only the pairs
    // whose even-side element the control selects.
    int swap(uint64_t delta, uint64_t sel, const uint64_t *ctrl);
    int window(const DiagGate *gates, size_t ngates);
    // Runs the operations on the state (2^bits amplitudes), from |0...0>,
    // which need not have been written.
    int run(Ctx &ctx, void *state);
    // The plan alone, on the host: the operations in the order they are
    // applied, and the pass of each.
    int schedule(uint32_t *order, uint32_t *pass_of);

  private:
    struct Op
    {
        uint32_t kind;  // 0: gate, 1: controlled gate, 2: diagonal gate
        uint32_t delta; // gates
        uint32_t s0;    // the gate's selector, or the first of a diagonal gate
        uint32_t s1;    // the control, or the second selector
        double theta;
        uint32_t mat;
    };
    // Steps before the tile's coordinates are known.
    struct Draft
    {
        uint32_t kind; // as LdsStep, windows as 2
        uint32_t first, count;
    };
    // A planned pass: its kernel arguments and where its tables are.
    struct Pass;
    int push(const U3Gate &g, const uint64_t *ctrl);
    void start();
    int next_pass();
    void plan();
    void place();
    int stage(Ctx &ctx, bool fresh, Pass &out);
    int launch(Ctx &ctx, void *state, const std::vector<Pass> &passes);
    unsigned bits_ = 0;
    int prec_ = 0;
    bool simple_ = true; // every gate on one address bit, its selector that bit
    std::vector<Op> ops_;
    std::vector<std::array<double, 8>> mats_;
    std::vector<uint32_t> seen_; // a window's hash table: 0, or one past an operation
    // planning of a pass
    std::vector<uint32_t> rest_;                  // from head_ on: operations not yet in a pass
    std::vector<uint32_t> later_;                 // of those, looked at for a pass and deferred
    size_t head_ = 0;
    bool left() const
    {
        return head_ < rest_.size();
    }
    std::vector<uint32_t> order_;                 // operations of the pass, by draft
    std::vector<Draft> drafts_;
    std::vector<uint32_t> vec_, piv_, red_;       // the tile's offsets; elimination
    std::vector<uint32_t> pending_, group_;
    std::vector<std::array<uint32_t, 2>> dgates_, ddiags_;
};

} // namespace zxa
