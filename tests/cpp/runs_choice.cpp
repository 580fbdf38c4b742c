// Which gates the plain form's planner (runs.hpp) puts into runs: queues whose
// gates' own kernels are faster stay single.
#include <cstdio>
#include <vector>

#include "../../oracle/qvnt_oracle.h"
#include "../../qvnt_amd/csrc/runs.hpp"

using namespace qvnt::runs;

static int failures = 0;

// `count` ry (or x) on qubits 14 and 15 with `controls` controls from qubit 4 on
static std::vector<qvnt_gate> queue(unsigned controls, unsigned count, bool x = false) {
    std::vector<qvnt_gate> out;
    for (unsigned k = 0; k < count; ++k) {
        qvnt_gate buf[8];
        const long m = x ? orc_op_x(1ull << (14 + k % 2), buf) : orc_op_ry(0.3 + k, 1ull << (14 + k % 2), buf);
        if (m != 1 || (controls && orc_op_c(buf, 1, ((1ull << controls) - 1u) << 4))) ++failures;
        out.push_back(buf[0]);
    }
    return out;
}
static std::vector<qvnt_gate> operator+(std::vector<qvnt_gate> a, const std::vector<qvnt_gate>& b) {
    a.insert(a.end(), b.begin(), b.end());
    return a;
}

// the queue's steps, as text: r<gates> for a run, s for a single
static void expect(const char* name, const std::vector<qvnt_gate>& g, unsigned n, bool fp64, size_t runs, size_t singles) {
    static Run run;
    size_t r = 0, s = 0, gates = 0;
    for (size_t pos = 0;;) {
        const Step step = next(g.data(), g.size(), &pos, n, fp64, reg_bits(n), max_tile(n, fp64), &run);
        if (step.kind == Kind::Done) break;
        (step.kind == Kind::RunStep ? r : s) += 1;
        gates += step.count;
    }
    if (r != runs || s != singles || gates != g.size()) {
        std::printf("%s, %u qubits %s: %zu runs and %zu singles, want %zu and %zu\n", name, n, fp64 ? "FP64" : "FP32", r, s, runs, singles);
        ++failures;
    }
}

int main() {
    // (times measured as one run and as single kernels beside each)
    expect("20 ry, 4 controls", queue(4, 20), 28, false, 0, 20);   // 1697 1102 us
    expect("40 ry, 4 controls", queue(4, 40), 28, false, 0, 40);   // 3272 2194
    expect("40 ry, 5 controls", queue(5, 40), 28, false, 0, 40);   // 2112 1566
    expect("40 ry, 4 controls", queue(4, 40), 26, false, 0, 40);   // 739 631
    expect("40 ry, 4 controls", queue(4, 40), 25, false, 1, 0);    // 290 361
    expect("40 ry, 5 controls", queue(5, 40), 25, false, 1, 0);    // 171 269
    expect("70 x, 5 controls", queue(5, 70, true), 28, false, 1, 0);   // 2388 2672
    expect("40 ry, 4 controls", queue(4, 40), 24, false, 1, 0);    // 154 244
    expect("40 ry, 4 controls", queue(4, 40), 22, false, 1, 0);    // 46 167
    expect("40 ry, 4 controls", queue(4, 40), 18, false, 1, 0);
    expect("20 ry, 3 controls", queue(3, 20), 28, false, 1, 0);    // 1712 2020
    expect("10 ry, 2 controls", queue(2, 10), 28, false, 1, 0);    // 1157 1802
    expect("20 ry", queue(0, 20), 28, false, 1, 0);                // 1686 13381
    expect("2 ry", queue(0, 2), 28, false, 1, 0);                  // 784 1341
    expect("20 x, 4 controls", queue(4, 20, true), 28, false, 1, 0);   // 877 1102
    expect("20 ry, 4 controls", queue(4, 20), 28, true, 1, 0);     // 1740 2753
    expect("70 ry, 5 controls", queue(5, 70), 28, true, 1, 0);     // 2523 4569
    expect("2 ry, 1 control", queue(1, 2), 28, true, 0, 2);        // 1593 1456 (on the top qubits)
    expect("5 ry, 2 controls", queue(2, 5), 28, true, 1, 0);       // 1630 1932
    expect("one ry", queue(0, 1), 28, true, 0, 1);
    // cheap gates behind a run stay out of it, between two halves of it they do not break it
    expect("20 ry, then 40 with 5 controls", queue(0, 20) + queue(5, 40), 28, false, 1, 40);
    expect("20 ry, 1 with 5 controls, 20 ry", queue(0, 20) + queue(5, 1) + queue(0, 20), 28, false, 1, 0);
    std::printf("%d failure(s)\n", failures);
    return failures ? 1 : 0;
}
