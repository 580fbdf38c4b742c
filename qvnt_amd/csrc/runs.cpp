// Planner of the plain form's runs (runs.hpp).
#include "runs.hpp"

#include <cstring>

namespace qvnt {
namespace runs {
namespace {

// A SingleOp's part on one or two qubits.  Multi-bit x, y, z and s are
// tensor powers whose factors only move amplitudes or multiply them by
// powers of i, which is exact, so they split per bit; a multi-bit t is not
// (t.t rounds, s does not).
struct Prim {
    uint32_t family;
    uint64_t mix;        // qubits whose amplitudes it mixes: register bits of its phase
    uint64_t ctrl;       // qubits that have to be 1
    uint64_t parity;     // F_RZ: its act bits
    bool rev;            // F_H2: a is the higher bit
    double re, im;
};

constexpr size_t kMaxPrims = 64;
// From here on a queue's runs are weighed (Cost); below, a launch takes longer
// than a pass, and two SingleOps are a run (18 qubits FP64: 3 gates with 1
// control 4.8 us as a run, 10.9 alone; 20 with a control each 6.1 and 8.6).
constexpr unsigned kWeighedQubits = 20;

uint64_t low_bit(uint64_t x) { return x & (~x + 1); }

// The gate's parts on a buffer of 2^ns amplitudes: their number (0: the
// identity there), or -1 for a gate that only its own kernel takes.
int lower(const qvnt_gate& g, unsigned ns, Prim* out) {
    const uint64_t lmask = (1ull << ns) - 1u;
    if (g.kind == QVNT_ID || (g.ctrl & ~lmask)) return 0;
    Prim p{};
    p.ctrl = g.ctrl;
    p.re = g.re;
    p.im = g.im;
    const auto per_bit = [&](uint64_t bits, bool mixes) {
        int k = 0;
        for (uint64_t b = bits; b; b &= b - 1, ++k) {
            out[k] = p;
            if (mixes) out[k].mix = low_bit(b);
            else out[k].ctrl |= low_bit(b);
        }
        return k;
    };
    const auto mixing = [&](uint32_t family, uint64_t bits) {
        p.family = family;
        p.mix = bits;
        out[0] = p;
        return 1;
    };
    const bool d = g.dagger != 0;
    switch (g.kind) {
    case QVNT_X: p.family = F_X; return per_bit(g.a, true);
    case QVNT_Y: p.family = F_Y; return per_bit(g.a, true);
    // (a phase on |1>: the act bit is one more control)
    case QVNT_Z: p.family = F_I2; return per_bit(g.a & lmask, false);
    case QVNT_S: p.family = d ? F_I3 : F_I1; return per_bit(g.a & lmask, false);
    case QVNT_T:
        if (popc(g.a & lmask) > 1) return -1;
        p.family = d ? F_TD : F_T;
        return per_bit(g.a & lmask, false);
    case QVNT_PHI: p.family = F_PH; return per_bit(g.a & lmask, false);
    case QVNT_RZ: case QVNT_RZZ:
        p.family = F_RZ;
        p.parity = g.a & lmask;
        out[0] = p;
        return 1;
    case QVNT_RX: return mixing(F_RX, g.a);
    case QVNT_RY: return mixing(F_RY, g.a);
    case QVNT_H1: return mixing(F_H1, g.a);
    case QVNT_RXX: return mixing(F_RXX, g.a);
    case QVNT_RYY: return mixing(F_RYY, g.a);
    case QVNT_SWAP: return mixing(F_SWAP, g.a);
    case QVNT_ISWAP: return mixing(d ? F_ISWAPD : F_ISWAP, g.a);
    case QVNT_SQRT_SWAP: return mixing(d ? F_SQSWD : F_SQSW, g.a);
    case QVNT_SQRT_ISWAP: return mixing(d ? F_SQISD : F_SQIS, g.a);
    case QVNT_H2: return mixing(g.a < g.b ? F_H2 : F_H2R, g.a | g.b);
    default: return -1;  // U1, U2: their matrices do not fit beside the amplitudes
    }
}

// The share of the state that the gate's own kernel moves, in 1/64ths: the
// half where a control outside the 128-byte line is 1, and so on.
unsigned single_share(const qvnt_gate& g, unsigned ns, bool fp64) {
    const uint64_t line = (1ull << row_bits(fp64)) - 1u, lmask = (1ull << ns) - 1u;
    unsigned halves = popc(g.ctrl & ~line);
    const uint64_t a = g.a & lmask;
    if ((g.kind == QVNT_Z || g.kind == QVNT_S || g.kind == QVNT_T || g.kind == QVNT_PHI) && popc(a) == 1 && !(a & line))
        ++halves;
    if ((g.kind == QVNT_SWAP || g.kind == QVNT_ISWAP || g.kind == QVNT_SQRT_SWAP || g.kind == QVNT_SQRT_ISWAP) && !(low_bit(a) & line))
        ++halves;
    return halves < 6 ? 64u >> halves : 1u;
}

// What single kernels and a run take, in 1/64ths of a pass over the state
// (read and written at 6 TB/s).  Fitted to queues of 2 to 70 x, ry and rz with
// 0 to 6 controls, on the top qubits and in the tile, on 20 to 28 qubits in
// both precisions, each timed all as runs and all as single kernels (1248
// pairs): the choice takes 0.1 % longer than the better of the two on average,
// a third at most (26 qubits FP32, 70 x with 6 controls each, left single).
struct Cost {
    unsigned ns;
    bool fp64;
    double launch;
    Cost(unsigned n, bool f64)
        // 5.6 us from one kernel to the next
        : ns(n), fp64(f64), launch(5.6 * 64.0 * 6.0e6 / (double)((f64 ? 32ull : 16ull) << n)) {}
    double single(unsigned share) const { return share > launch / 2.0 ? share + launch / 2.0 : launch; }
    // An op's arithmetic: 28 qubits FP32 20 ry in 1.69 ms (a pass 0.77), 40 with
    // 4 controls in 3.27, with 5 in 2.11; 25 qubits, where each block has one
    // tile, 0.29 and 0.17 (0.09); FP64 28 qubits 1.70 for 20 and 2.21 for 40
    // (1.59).  Moves (x, swap): 40 with 4 controls FP32 1.52.
    double op(bool move, unsigned share) const {
        if (fp64) return move ? 0.7 : 1.4;
        if (move) return 1.7;
        const double most = ns <= 25 ? 5.0 : 6.3, part = 2.0 + (ns <= 25 ? 0.6 : 0.8) * share;
        return part < most ? part : most;
    }
    double run(double ops) const { return (ops + 20.0 > 70.0 ? ops + 20.0 : 70.0) + launch; }
};

}  // namespace

Step next(const qvnt_gate* g, size_t n, size_t* pos, unsigned ns, bool fp64, unsigned regs, unsigned max_tile, Run* run) {
    Prim prims[kMaxPrims];
    while (*pos < n && lower(g[*pos], ns, prims) == 0) ++*pos;
    Step step;
    step.from = *pos;
    if (*pos >= n) return step;
    step.kind = Kind::Single;
    step.count = 1;
    if (ns < kMinQubits) {
        ++*pos;
        return step;
    }
    const unsigned tmax = ns < max_tile ? ns : max_tile;
    const unsigned rows = row_bits(fp64) + regs < tmax ? row_bits(fp64) : tmax - regs;

    // The longest prefix of the queue that fits: its tile qubits, and its
    // phases' register qubits.  Where a pass takes longer than a launch, the
    // prefix that gains most over its gates' own kernels, if any does.  (By
    // the bytes alone, more than 1.25 passes' worth, gates with many controls
    // went into FP32 runs that took longer: 28 qubits, 20 ry with 4 controls
    // in the tile 1.70 ms as a run and 1.10 alone, 40 of them 3.27 and 2.19, 40
    // with 5 controls 2.11 and 1.57.)
    const Cost cost(ns, fp64);
    const bool weigh = ns >= kWeighedQubits;
    double alone = 0.0, ops = 0.0, best_gain = 0.0;
    struct Prefix {
        unsigned count, phases;
        uint64_t tile, mixed;   // mixed: of its last phase
        size_t last;
    } best{0, 0, 0, 0, 0};
    Prim list[kMaxOps];
    uint64_t mixed[kMaxPhases];
    unsigned ends[kMaxPhases];
    unsigned count = 0, phases = 1;
    uint64_t tile = (1ull << rows) - 1u;
    mixed[0] = 0;
    size_t gates = 0;
    for (size_t i = *pos; i < n; ++i) {
        const int k = lower(g[i], ns, prims);
        if (k < 0) break;
        if (k == 0) continue;
        unsigned c2 = count, ph2 = phases;
        uint64_t t2 = tile, r2 = mixed[phases - 1];
        uint64_t nmixed[kMaxPhases];
        unsigned nends[kMaxPhases];
        bool ok = true;
        for (int j = 0; j < k && ok; ++j) {
            const Prim& p = prims[j];
            t2 |= p.mix;
            ok = c2 < kMaxOps && popc(t2) <= tmax;
            if (!ok) break;
            if (popc(r2 | p.mix) > regs) {
                ok = ph2 < kMaxPhases;
                if (!ok) break;
                nmixed[ph2 - 1] = r2;
                nends[ph2 - 1] = c2;
                ++ph2;
                r2 = 0;
            }
            r2 |= p.mix;
            list[c2++] = p;
        }
        if (!ok) break;
        for (unsigned q = phases; q < ph2; ++q) {
            mixed[q - 1] = nmixed[q - 1];
            ends[q - 1] = nends[q - 1];
        }
        mixed[ph2 - 1] = r2;
        count = c2;
        phases = ph2;
        tile = t2;
        ++gates;
        const unsigned share = single_share(g[i], ns, fp64);
        alone += cost.single(share);
        for (int j = 0; j < k; ++j) ops += cost.op(prims[j].family == F_X || prims[j].family == F_SWAP, share);
        const double gain = alone - cost.run(ops);
        // (one SingleOp alone is its own kernel's work)
        if (gates >= 2 && (!weigh || gain >= best_gain)) {
            best_gain = gain;
            best = {count, phases, tile, r2, i + 1};
        }
    }
    if (best.last == 0) {
        ++*pos;
        return step;
    }
    count = best.count;
    phases = best.phases;
    tile = best.tile;
    mixed[phases - 1] = best.mixed;
    ends[phases - 1] = count;
    step.kind = Kind::RunStep;
    step.count = best.last - step.from;
    *pos = best.last;

    // the tile, filled with the lowest qubits
    for (unsigned q = 0; popc(tile) < tmax; ++q) tile |= 1ull << q;
    std::memset(run, 0, sizeof(Run));
    run->t = tmax;
    run->regs = regs;
    run->nphases = phases;
    run->nops = count;
    int local[64];
    unsigned t = 0;
    for (unsigned q = 0; q < ns; ++q) {
        local[q] = -1;
        if (!(tile >> q & 1)) continue;
        local[q] = (int)t;
        run->tpos[t++] = (uint8_t)q;
    }
    const auto local_mask = [&](uint64_t m) {
        uint32_t l = 0;
        for (; m; m &= m - 1)
            if (local[ctz(m)] >= 0) l |= 1u << local[ctz(m)];
        return l;
    };

    unsigned c = 0;
    for (unsigned ph = 0; ph < phases; ++ph) {
        // register bits: the phase's own, then the tile's top bits
        uint32_t rl = local_mask(mixed[ph]);
        for (int b = (int)t - 1; popc(rl) < regs; --b) rl |= 1u << b;
        int reg[kMaxTile];
        unsigned j = 0;
        for (unsigned b = 0; b < t; ++b) {
            reg[b] = -1;
            if (!(rl >> b & 1)) continue;
            reg[b] = (int)j;
            run->phase[ph].rpos[j++] = (uint8_t)b;
        }
        const auto reg_mask = [&](uint32_t l) {
            uint32_t m = 0;
            for (l &= rl; l; l &= l - 1) m |= 1u << reg[ctz(l)];
            return m;
        };
        for (; c < ends[ph]; ++c) {
            const Prim& p = list[c];
            ROp& op = run->op[c];
            const uint32_t lc = local_mask(p.ctrl), lp = local_mask(p.parity);
            const uint32_t rc = reg_mask(lc);
            uint32_t pc = 0;
            for (uint32_t r = 0; r < 1u << regs; ++r)
                if ((r & rc) == rc) pc |= 1u << r;
            uint32_t variant = reg_mask(local_mask(p.mix));
            if (p.family == F_RZ) variant = reg_mask(lp);
            else if (p.family >= F_X && p.family <= F_H1) variant = ctz(variant);
            op.code_pc = code_of(p.family, variant) << 16 | pc;
            op.lbits = (lp & ~rl) << 16 | (lc & ~rl);
            op.re = p.re;
            op.im = p.im;
            run->outer[c].ctrl = p.ctrl & ~tile;
            run->outer[c].parity = p.parity & ~tile;
        }
        run->phase[ph].op_end = (uint16_t)c;
    }
    // the tile is read and written in the first and last phase's layout
    // where that keeps the bits of a line among the threads, else with its
    // top bits in the registers
    const auto edge = [&](const RPhase& ph, uint8_t* to, uint8_t* global) {
        const bool own = ph.rpos[0] >= rows;
        for (unsigned j = 0; j < regs; ++j) {
            to[j] = own ? ph.rpos[j] : (uint8_t)(t - regs + j);
            global[j] = run->tpos[to[j]];
        }
    };
    edge(run->phase[0], run->in, run->gin);
    edge(run->phase[phases - 1], run->out, run->gout);
    return step;
}

}  // namespace runs
}  // namespace qvnt
