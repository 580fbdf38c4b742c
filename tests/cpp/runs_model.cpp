// A CPU model of the plain form's run kernel (qvnt_amd/csrc/runs.hip: k_run)
// driven by the real planner (runs.cpp) and the kernel's own gate code
// (runs_ops.hpp, compiled for the host).  For random circuits of every gate
// kind -- multi-bit masks, controls inside the registers, the tile and
// outside it, daggers, matrices, act bits and controls beyond the buffer --
// the final state must equal the oracle's, applied one SingleOp at a time,
// to the last bit; FP32 states the oracle's FP64 result on the widened
// amplitudes rounded once per SingleOp.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "../../oracle/qvnt_oracle.h"
#include "../../qvnt_amd/csrc/runs_ops.hpp"

using namespace qvnt;
using namespace qvnt::runs;

#define CHECK(c)                                                                     \
    do {                                                                             \
        if (!(c)) {                                                                  \
            std::fprintf(stderr, "CHECK failed %s:%d %s\n", __FILE__, __LINE__, #c); \
            std::exit(1);                                                            \
        }                                                                            \
    } while (0)

namespace qvnt {
bool is_diagonal_kind(uint32_t) { return false; }
}

static uint32_t swz(uint32_t e) { return e ^ (e >> 4); }
template <int B>
static uint32_t spread(uint32_t x, const uint8_t* p) {
    for (unsigned j = 0; j < B; ++j) {
        if (j) CHECK(p[j] > p[j - 1]);
        const uint32_t lo = x & ((1u << p[j]) - 1u);
        x = ((x ^ lo) << 1) | lo;
    }
    return x;
}
template <int B>
static uint32_t element(uint32_t tid, int i, const uint8_t* p) {
    uint32_t e = spread<B>(tid, p);
    for (unsigned j = 0; j < B; ++j)
        if (i >> j & 1) e |= 1u << p[j];
    return e;
}

static int seen[F_COUNT][2][2];

template <int B, class R>
static void run_step(std::vector<cplx<R>>& psi, unsigned ns, const Run& run) {
    const unsigned t = run.t, nth = 1u << (t - B);
    CHECK(run.regs == B && t >= B && t <= kMaxTile && t <= ns && run.nphases >= 1 && run.nphases <= kMaxPhases && run.nops <= kMaxOps);
    for (unsigned k = 0; k + 1 < t; ++k) CHECK(run.tpos[k] < run.tpos[k + 1] && run.tpos[k + 1] < ns);
    for (int j = 0; j < B; ++j) CHECK(run.gin[j] == run.tpos[run.in[j]] && run.gout[j] == run.tpos[run.out[j]]);
    std::vector<char> hit(1u << t, 0);
    for (uint32_t e = 0; e < 1u << t; ++e) {
        CHECK(swz(e) < 1u << t && !hit[swz(e)]);
        hit[swz(e)] = 1;
    }
    for (uint64_t n = 0; n < psi.size() >> t; ++n) {
        uint64_t tile = n;
        for (unsigned k = 0; k < t; ++k) {
            const uint64_t lo = tile & ((1ull << run.tpos[k]) - 1u);
            tile = ((tile ^ lo) << 1) | lo;
        }
        const auto global = [&](uint32_t e) {
            uint64_t i = tile;
            for (unsigned k = 0; k < t; ++k) i |= (uint64_t)(e >> k & 1) << run.tpos[k];
            return i;
        };
        std::vector<cplx<R>> local(1u << t);
        for (uint32_t tid = 0; tid < nth; ++tid)
            for (int i = 0; i < 1 << B; ++i) local[element<B>(tid, i, run.in)] = psi[global(element<B>(tid, i, run.in))];
        uint32_t o = 0;
        for (uint32_t ph = 0; ph < run.nphases; ++ph) {
            const RPhase& p = run.phase[ph];
            CHECK(p.op_end >= o && p.op_end <= run.nops && p.rpos[B - 1] < t);
            for (uint32_t tid = 0; tid < nth; ++tid) {
                cplx<R> v[1 << B];
                const uint32_t tb = spread<B>(tid, p.rpos);
                for (int i = 0; i < 1 << B; ++i) v[i] = local[element<B>(tid, i, p.rpos)];
                for (uint32_t k = o; k < p.op_end; ++k) {
                    const ROp& op = run.op[k];
                    const ROut& q = run.outer[k];
                    const uint32_t lc = op.lbits & 0xFFFFu, pc = op.code_pc & 0xFFFFu, code = op.code_pc >> 16;
                    CHECK(code >> 4 < F_COUNT);
                    const bool live = (tile & q.ctrl) == q.ctrl, on = (tb & lc) == lc;
                    const bool odd = ((dpopc(tb & (op.lbits >> 16)) + dpopc(tile & q.parity)) & 1u) != 0;
                    if (!live) continue;
                    // the kernel's two forms: whole waves, and lanes selected
                    const bool whole = on && pc == (1u << (1 << B)) - 1u && lc == 0;
                    seen[code >> 4][B - 3][whole ? 0 : 1] = 1;
                    if (whole) apply_op<B, false>(v, code, pc, true, odd, op.re, op.im);
                    else apply_op<B, true>(v, code, pc, on, odd, op.re, op.im);
                }
                for (int i = 0; i < 1 << B; ++i) local[element<B>(tid, i, p.rpos)] = v[i];
            }
            o = p.op_end;
        }
        CHECK(o == run.nops);
        for (uint32_t tid = 0; tid < nth; ++tid)
            for (int i = 0; i < 1 << B; ++i) psi[global(element<B>(tid, i, run.out))] = local[element<B>(tid, i, run.out)];
    }
}

static std::vector<qvnt_gate> circuit(std::mt19937_64& g, unsigned n, int count, bool local) {
    std::vector<qvnt_gate> out;
    const auto pick = [&](uint64_t m) { return std::uniform_int_distribution<uint64_t>(0, m - 1)(g); };
    std::uniform_real_distribution<double> ang(0.0, 6.2831853);
    while ((int)out.size() < count) {
        qvnt_gate q[64];
        std::vector<unsigned> bits(n);
        for (unsigned k = 0; k < n; ++k) bits[k] = k;
        std::shuffle(bits.begin(), bits.end(), g);
        // (local: neighbouring qubits, so that many gates share a run)
        if (local) std::sort(bits.begin(), bits.begin() + std::min(n, 6u));
        const auto mask = [&](unsigned c) {
            uint64_t m = 0;
            for (unsigned k = 0; k < c; ++k) m |= 1ull << bits[k];
            return m;
        };
        const unsigned many = 1 + (unsigned)pick(std::min(n, 3u));
        double m1[8];
        const double c = std::cos(ang(g)), s = std::sqrt(1 - c * c);
        const double h[8] = {c, 0, 0, -s, 0, -s, c, 0};
        std::memcpy(m1, h, sizeof m1);
        long k = 0;
        unsigned used = 2;
        switch (pick(21)) {
        case 0: k = orc_op_x(mask(used = many), q); break;
        case 1: k = orc_op_y(mask(used = many), q); break;
        case 2: k = orc_op_z(mask(used = many) | (pick(8) ? 0 : 1ull << 40), q); break;
        case 3: k = orc_op_s(mask(used = many), q); break;
        case 4: k = orc_op_t(mask(used = many), q); break;
        case 5: k = orc_op_rx(ang(g), mask(used = 1), q); break;
        case 6: k = orc_op_ry(ang(g), mask(used = 1), q); break;
        case 7: k = orc_op_rz(ang(g), pick(8) ? mask(used = 1) : 1ull << 41, q); break;
        case 8: k = orc_op_rxx(ang(g), mask(2), q); break;
        case 9: k = orc_op_ryy(ang(g), mask(2), q); break;
        case 10: k = orc_op_rzz(ang(g), pick(8) ? mask(2) : mask(1) | 1ull << 42, q); break;
        case 11: k = orc_op_phi(ang(g), mask(used = 1), q); break;
        case 12: k = orc_op_swap(mask(2), q); break;
        case 13: k = orc_op_i_swap(mask(2), q); break;
        case 14: k = orc_op_sqrt_swap(mask(2), q); break;
        case 15: k = orc_op_sqrt_i_swap(mask(2), q); break;
        case 16: k = orc_op_h(mask(used = many), q); break;
        case 17: k = orc_op_u3(ang(g), ang(g), ang(g), mask(used = 1), q); break;
        case 18: k = orc_op_qft(mask(used = many), q); break;
        case 19: k = pick(4) ? 0 : orc_op_matrix1(mask(used = 1), m1, q); break;
        default: k = orc_op_t(mask(used = 1), q); break;
        }
        if (k <= 0) continue;
        if (pick(4) == 0) orc_op_dgr(q, (size_t)k);
        unsigned nc = (unsigned)pick(3);
        if (used + nc > n) nc = n - used;
        uint64_t ctrl = 0;
        for (unsigned j = 0; j < nc; ++j) ctrl |= 1ull << bits[used + j];
        if (pick(24) == 0) ctrl |= 1ull << 43;
        if (ctrl) CHECK(orc_op_c(q, (size_t)k, ctrl) == 0);
        out.insert(out.end(), q, q + k);
        // h2 with a below b as well: the reference builds a above b
        if (pick(6) == 0 && n >= 2) {
            qvnt_gate e{};
            e.kind = QVNT_H2;
            e.a = 1ull << bits[0];
            e.b = 1ull << bits[1];
            e.act = e.a | e.b;
            if (n >= 3 && pick(2)) e.ctrl = 1ull << bits[2];
            out.push_back(e);
        }
    }
    return out;
}

template <class R>
static void check(std::mt19937_64& g, unsigned n, int count, bool local, unsigned regs, size_t* runs, size_t* singles, size_t* fused) {
    const std::vector<qvnt_gate> q = circuit(g, n, count, local);
    const uint64_t len = 1ull << n;
    std::vector<cplx<R>> psi(len);
    std::normal_distribution<double> d;
    for (auto& p : psi) p = {(R)d(g), (R)d(g)};
    // amplitudes that are zero, infinite or not a number follow the same formulas
    if (n > 5) {
        for (int k = 0; k < 6; ++k) psi[g() % len] = {(R)0, (R)-0.0};
        psi[g() % len].re = (R)INFINITY;
        psi[g() % len].im = (R)NAN;
    }
    orc_reg* ref = orc_reg_with_state(n, 0);
    double* w = orc_reg_psi(ref);
    for (uint64_t i = 0; i < len; ++i) w[2 * i] = psi[i].re, w[2 * i + 1] = psi[i].im;
    const auto single = [&](const qvnt_gate& gate) {
        orc_reg_apply(ref, &gate, 1);
        w = orc_reg_psi(ref);
        for (uint64_t i = 0; i < 2 * len; ++i) w[i] = (double)(R)w[i];
    };
    Run run;
    size_t done = 0;
    for (size_t pos = 0;;) {
        const Step s = next(q.data(), q.size(), &pos, n, sizeof(R) == 8, regs, regs == 3 ? max_tile(n, sizeof(R) == 8) : max_tile(64, sizeof(R) == 8), &run);
        if (s.kind == Kind::Done) break;
        CHECK(s.from >= done && s.count >= 1 && pos >= s.from + s.count);
        // (gates left out are the identity: the oracle applies them all the same)
        for (; done < s.from + s.count; ++done) single(q[done]);
        if (s.kind == Kind::Single) {
            for (uint64_t i = 0; i < len; ++i) psi[i] = {(R)w[2 * i], (R)w[2 * i + 1]};
            ++*singles;
            continue;
        }
        if (regs == 3) run_step<3>(psi, n, run);
        else run_step<4>(psi, n, run);
        ++*runs;
        *fused += s.count;
        for (uint64_t i = 0; i < len; ++i) {
            const double re = psi[i].re, im = psi[i].im;
            const bool ok = (re == w[2 * i] || (std::isnan(re) && std::isnan(w[2 * i]))) &&
                            (im == w[2 * i + 1] || (std::isnan(im) && std::isnan(w[2 * i + 1])));
            if (!ok) {
                std::fprintf(stderr, "n %u: amplitude %llu after gate %zu: (%.17g, %.17g), oracle (%.17g, %.17g)\n", n,
                             (unsigned long long)i, done, re, im, w[2 * i], w[2 * i + 1]);
                std::exit(1);
            }
        }
    }
    orc_reg_free(ref);
}

int main() {
    std::mt19937_64 g(20240229);
    size_t runs = 0, singles = 0, fused = 0;
    for (unsigned n = 3; n <= 15; ++n)
        for (int k = 0; k < (n < 13 ? 12 : 5); ++k) {
            for (unsigned regs = 3; regs <= 4; ++regs) {
                check<double>(g, n, 120, k & 1, regs, &runs, &singles, &fused);
                check<float>(g, n, 120, k & 1, regs, &runs, &singles, &fused);
            }
        }
    for (int f = 0; f < F_COUNT; ++f) {
        const bool whole_possible = f > F_TD;
        for (const auto& form : seen[f])
            if (!form[1] || (whole_possible && !form[0])) {
                std::fprintf(stderr, "family %d not run in every form\n", f);
                return 1;
            }
    }
    std::printf("%zu runs of %zu SingleOps, %zu singles: equal to the oracle\n", runs, fused, singles);
    return 0;
}
