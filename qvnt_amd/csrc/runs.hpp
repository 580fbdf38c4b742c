// Runs of the plain form: consecutive SingleOps applied in one pass over the
// state, in queue order and with the rounding of one kernel per SingleOp.
//
// The reference applies a MultiOp one SingleOp at a time
// (src/operator/multi/mod.rs:96-114), one pass over the state each.  A run
// keeps the amplitudes of a tile on the chip instead: the tile's qubits T
// hold every bit that the run's gates mix, so each SingleOp maps the tile
// onto itself, and applying the queue's next gates one after the other to
// each tile gives what applying them one after the other to the state
// gives, to the last bit (the formulas are those of device.hpp, FP32
// amplitudes rounded once per SingleOp).  Gates are never reordered.
//
// This header: the layout of a run's program and the planner (runs.cpp,
// host only).  runs_ops.hpp: the gates on 16 amplitudes.  runs.hip: the
// kernel.
#pragma once

#include <cstddef>
#include <cstdint>

#include "common.hpp"

namespace qvnt {
namespace runs {

constexpr unsigned kRegBits = 4;             // register qubits of a phase, at most
constexpr unsigned kRegs = 1u << kRegBits;   // amplitudes per thread, at most
constexpr unsigned kMaxTile = 13;
constexpr unsigned kMinQubits = kRegBits;    // 2^4 amplitudes
constexpr unsigned kMaxOps = 78;             // a run's program fits in 4 KiB of kernel arguments
constexpr unsigned kMaxPhases = 24;

// Register qubits of a phase on 2^ns amplitudes.  At 16 amplitudes a thread a
// state of 2^20 has one wave for each SIMD, and one wave alone issues an FP64
// instruction every 8 cycles, not every 4: 8 amplitudes a thread double the
// waves, for a third more phases.  200 random gates and a QFT, FP64: 20
// qubits 293 and 150 us with 16, 273 and 123 with 8; 21 qubits 325 and 192,
// 321 and 177; 22 qubits 464 and 286, 583 and 334.
constexpr unsigned kSmallQubits = 21;
constexpr unsigned reg_bits(unsigned ns) { return ns <= kSmallQubits ? 3u : 4u; }

// Tile qubits at most.  Large states: both components of a tile of 2^13 FP32
// or 2^12 FP64 amplitudes are exchanged through 32 KiB of LDS, one after the
// other.  States of few tiles leave most of the chip idle and each tile's ops
// and exchanges are the time, so the tiles are smaller, though a run then
// holds fewer gates.  200 random gates with tiles of 10, 11, 12, 13: 16
// qubits FP64 166, 166, 184 us, FP32 170, 169, 191, 257; 18 qubits FP64 193,
// 191, 208, FP32 192, 192, 201, 271; 20 qubits FP64 304, 284, 279, FP32 263,
// 250, 240, 313.
constexpr unsigned kTinyQubits = 18;
constexpr unsigned max_tile(unsigned ns, bool fp64) { return ns <= kTinyQubits ? 11u : ns <= kSmallQubits || fp64 ? 12u : 13u; }
// The low qubits that every tile holds: one 128-byte line.
constexpr unsigned row_bits(bool fp64) { return fp64 ? 3u : 4u; }

// Codes: a family and, where it has them, the register bits it works on
// (one bit: j; two bits j0 < j1: pair_variant).
enum Family : uint32_t {
    F_PH = 0,      // phase (re, im) on the amplitudes of `pc`
    F_I1, F_I2, F_I3,  // i, -1, -i on the amplitudes of `pc`
    F_T, F_TD,     // t and its dagger on the amplitudes of `pc`
    F_RZ,          // rz / rzz: conjugate phases by the parity of the act bits; variant: the register bits among them
    F_X, F_Y, F_RX, F_RY, F_H1,   // one register bit
    F_RXX, F_RYY, F_SWAP, F_ISWAP, F_ISWAPD, F_SQSW, F_SQSWD, F_SQIS, F_SQISD, F_H2, F_H2R,  // two
    F_COUNT
};
constexpr uint32_t code_of(uint32_t family, uint32_t variant) { return family * 16u + variant; }
// variant of a pair of register bits: the two-bit mask itself (3, 5, 6, 9, 10, 12)
constexpr uint32_t pair_variant(unsigned j0, unsigned j1) { return (1u << j0) | (1u << j1); }

struct ROp {            // 32 bytes
    uint32_t code_pc;   // code << 16 | pc: register indices the gate acts on
    uint32_t lbits;     // parity bits << 16 | control bits among the tile's thread bits (local positions)
    uint32_t live;      // set per tile by the kernel: bit 0 the controls outside the tile hold, bit 1 the parity there
    uint32_t pad;
    double re, im;      // phase
};
struct ROut {           // 16 bytes: the op's bits outside the tile (global positions)
    uint64_t ctrl, parity;
};
struct RPhase {         // 8 bytes
    uint8_t rpos[kRegBits];   // local positions of the register bits, ascending
    uint16_t op_end;
    uint16_t pad;
};
struct Run {
    uint32_t t;               // tile qubits
    uint32_t nphases, nops;
    uint32_t regs;            // register qubits of a phase: 3 or 4
    uint8_t tpos[16];         // global positions of the local bits, ascending
    uint8_t in[kRegBits], out[kRegBits];  // local positions of the register bits while the tile is read / written
    uint8_t gin[kRegBits], gout[kRegBits];  // their global positions
    RPhase phase[kMaxPhases];
    ROut outer[kMaxOps];
    ROp op[kMaxOps];
};
// (16 bytes: the launch's other arguments, psi and tiles)
static_assert(sizeof(Run) + 16 <= 4096, "a run is passed as kernel arguments");

// The next step of a plain apply of a validated queue on 2^ns amplitudes.
// Done: nothing is left.  RunStep: gates [from, from + count) as `run`.
// Single: gate `from` through its own kernel.  *pos moves past the step
// (and past gates that are the identity there).  regs, max_tile: of the run
// (reg_bits, max_tile).
enum class Kind { Done, RunStep, Single };
struct Step {
    Kind kind = Kind::Done;
    size_t from = 0, count = 0;
};
Step next(const qvnt_gate* g, size_t n, size_t* pos, unsigned ns, bool fp64, unsigned regs, unsigned max_tile, Run* run);

}  // namespace runs
}  // namespace qvnt
