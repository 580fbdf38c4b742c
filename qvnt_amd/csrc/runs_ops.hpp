// One SingleOp of a run on the 16 amplitudes a thread holds (runs.hpp): the
// formulas of device.hpp on the register array, every index known at
// compile time.
#pragma once

#include "device.hpp"
#include "runs.hpp"

namespace qvnt {
namespace runs {

QVNT_HD Par par_of(double re, double im, uint32_t a, bool dagger) {
    Par g{};
    g.a = a;
    g.re = re;
    g.im = im;
    g.dagger = dagger ? 1u : 0u;
    g.i_pow = 1u;  // one act bit (atomic/y.rs:11)
    return g;
}

// The new value of an amplitude, in its register: kept back on lanes that
// the gate does not act on (M: there may be some).  The empty asm ends the
// orbit's update: nothing of the next orbit is computed before.  Without it
// the scheduler holds the inputs and outputs of all 16 amplitudes at once,
// in FP64 more than the 128 registers of four waves per SIMD.
template <bool M, class R>
QVNT_HD void put(cplx<R>& x, cplx<R> now, bool on) {
    x.re = !M || on ? now.re : x.re;
    x.im = !M || on ? now.im : x.im;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(x.re), "+v"(x.im));
#endif
}

// one register bit J, at the register indices of pc (M: not all of them, or
// not on all lanes)
template <int K, int J, bool M, class R>
QVNT_HD void one_bit(cplx<R>* v, uint32_t pc, bool on, const Par& g) {
#pragma unroll
    for (int i = 0; i < (int)kRegs; ++i) {
        if (i & (1 << J)) continue;
        if (M && !((pc >> i) & 1u)) continue;
        const cplx<R> x0 = v[i], x1 = v[i | (1 << J)];
        put<M>(v[i], f_pair<K>(g, 0, x0, x1), on);
        put<M>(v[i | (1 << J)], f_pair<K>(g, 1, x1, x0), on);
    }
}
template <int K, bool M, class R>
QVNT_HD void one_bit_sel(cplx<R>* v, uint32_t j, uint32_t pc, bool on, const Par& g) {
    switch (j) {
    case 0: one_bit<K, 0, M>(v, pc, on, g); break;
    case 1: one_bit<K, 1, M>(v, pc, on, g); break;
    case 2: one_bit<K, 2, M>(v, pc, on, g); break;
    default: one_bit<K, 3, M>(v, pc, on, g); break;
    }
}

// two register bits, mask B: both parities' pairs (r, r ^ 3), or the odd one only
template <int K, int B, bool ODD, bool M, class R>
QVNT_HD void two_bit(cplx<R>* v, uint32_t pc, bool on, const Par& g) {
    constexpr int lo = B & -B, hi = B ^ lo;
#pragma unroll
    for (int i = 0; i < (int)kRegs; ++i) {
        if (i & B) continue;
        if (M && !((pc >> i) & 1u)) continue;
        if (!ODD) {
            const cplx<R> x0 = v[i], x3 = v[i | B];
            put<M>(v[i], f_pair<K>(g, 0, x0, x3), on);
            put<M>(v[i | B], f_pair<K>(g, 3, x3, x0), on);
        }
        const cplx<R> x1 = v[i | lo], x2 = v[i | hi];
        put<M>(v[i | lo], f_pair<K>(g, 1, x1, x2), on);
        put<M>(v[i | hi], f_pair<K>(g, 2, x2, x1), on);
    }
}
template <int K, bool ODD, bool M, class R>
QVNT_HD void two_bit_sel(cplx<R>* v, uint32_t b, uint32_t pc, bool on, const Par& g) {
    switch (b) {
    case 3: two_bit<K, 3, ODD, M>(v, pc, on, g); break;
    case 5: two_bit<K, 5, ODD, M>(v, pc, on, g); break;
    case 6: two_bit<K, 6, ODD, M>(v, pc, on, g); break;
    case 9: two_bit<K, 9, ODD, M>(v, pc, on, g); break;
    case 10: two_bit<K, 10, ODD, M>(v, pc, on, g); break;
    default: two_bit<K, 12, ODD, M>(v, pc, on, g); break;
    }
}

// h2 (h2.rs:22-38): slot bit 0 is the gate's a, the lower register bit
// unless REV
template <int B, bool REV, bool M, class R>
QVNT_HD void quad(cplx<R>* v, uint32_t pc, bool on) {
    constexpr int lo = B & -B, hi = B ^ lo, a = REV ? hi : lo, b = REV ? lo : hi;
#pragma unroll
    for (int i = 0; i < (int)kRegs; ++i) {
        if (i & B) continue;
        if (M && !((pc >> i) & 1u)) continue;
        const c64 x[4] = {up(v[i]), up(v[i | a]), up(v[i | b]), up(v[i | a | b])};
        put<M>(v[i], down<R>(f_h2_rel(0, x[0], x[1], x[2], x[3])), on);
        put<M>(v[i | a], down<R>(f_h2_rel(1, x[1], x[0], x[3], x[2])), on);
        put<M>(v[i | b], down<R>(f_h2_rel(2, x[2], x[3], x[0], x[1])), on);
        put<M>(v[i | a | b], down<R>(f_h2_rel(3, x[3], x[2], x[1], x[0])), on);
    }
}
template <bool REV, bool M, class R>
QVNT_HD void quad_sel(cplx<R>* v, uint32_t b, uint32_t pc, bool on) {
    switch (b) {
    case 3: quad<3, REV, M>(v, pc, on); break;
    case 5: quad<5, REV, M>(v, pc, on); break;
    case 6: quad<6, REV, M>(v, pc, on); break;
    case 9: quad<9, REV, M>(v, pc, on); break;
    case 10: quad<10, REV, M>(v, pc, on); break;
    default: quad<12, REV, M>(v, pc, on); break;
    }
}

// rz / rzz (rz.rs:19-25, rzz.rs:19-25): the phase's imaginary part is im
// where the act bits have odd parity, -im where even; imx is the value for
// even parity of the register bits among them, B
template <int B, bool M, class R>
QVNT_HD void parity_phase(cplx<R>* v, uint32_t pc, bool on, double re, double imx) {
#pragma unroll
    for (int i = 0; i < (int)kRegs; ++i) {
        if (M && !((pc >> i) & 1u)) continue;
        put<M>(v[i], down<R>(cmul(c64{re, (__builtin_popcount(i & B) & 1) ? -imx : imx}, up(v[i]))), on);
    }
}
template <bool M, class R>
QVNT_HD void parity_phase_sel(cplx<R>* v, uint32_t b, uint32_t pc, bool on, double re, double imx) {
    switch (b) {
    case 0: parity_phase<0, M>(v, pc, on, re, imx); break;
    case 1: parity_phase<1, M>(v, pc, on, re, imx); break;
    case 2: parity_phase<2, M>(v, pc, on, re, imx); break;
    case 3: parity_phase<3, M>(v, pc, on, re, imx); break;
    case 4: parity_phase<4, M>(v, pc, on, re, imx); break;
    case 5: parity_phase<5, M>(v, pc, on, re, imx); break;
    case 6: parity_phase<6, M>(v, pc, on, re, imx); break;
    case 8: parity_phase<8, M>(v, pc, on, re, imx); break;
    case 9: parity_phase<9, M>(v, pc, on, re, imx); break;
    case 10: parity_phase<10, M>(v, pc, on, re, imx); break;
    default: parity_phase<12, M>(v, pc, on, re, imx); break;
    }
}

// the kinds that scale the amplitudes of pc one by one
template <uint32_t F, class R>
QVNT_HD void phase(cplx<R>* v, uint32_t pc, bool on, double re, double im) {
#pragma unroll
    for (int i = 0; i < (int)kRegs; ++i) {
        if (!((pc >> i) & 1u)) continue;
        const c64 p = up(v[i]), e{kFrac1Sqrt2, kFrac1Sqrt2};
        put<true>(v[i], down<R>(F == F_PH ? cmul(c64{re, im}, p) : F == F_T ? cmul(e, p) : F == F_TD ? cmul(e, rotate(p, 3))
                                          : rotate(p, F == F_I1 ? 1u : F == F_I2 ? 2u : 3u)), on);
    }
}

// One op on v.  code, pc: uniform; on: whether the lane's bits satisfy the
// controls (M false: all lanes do, and pc is full); odd: the parity of the
// act bits outside the registers (per lane).
template <bool M, class R>
QVNT_HD void apply_op(cplx<R>* v, uint32_t code, uint32_t pc, bool on, bool odd, double re, double im) {
    const uint32_t f = code >> 4, var = code & 15u;
    const Par g1 = par_of(re, im, 1u, false), g2 = par_of(re, im, 3u, false), g2d = par_of(re, im, 3u, true);
    switch (f) {
    case F_PH: phase<F_PH>(v, pc, on, re, im); break;
    case F_I1: phase<F_I1>(v, pc, on, re, im); break;
    case F_I2: phase<F_I2>(v, pc, on, re, im); break;
    case F_I3: phase<F_I3>(v, pc, on, re, im); break;
    case F_T: phase<F_T>(v, pc, on, re, im); break;
    case F_TD: phase<F_TD>(v, pc, on, re, im); break;
    case F_RZ: parity_phase_sel<M>(v, var, pc, on, re, odd ? im : -im); break;
    case F_X: one_bit_sel<QVNT_X, M>(v, var, pc, on, g1); break;
    case F_Y: one_bit_sel<QVNT_Y, M>(v, var, pc, on, g1); break;
    case F_RX: one_bit_sel<QVNT_RX, M>(v, var, pc, on, g1); break;
    case F_RY: one_bit_sel<QVNT_RY, M>(v, var, pc, on, g1); break;
    case F_H1: one_bit_sel<QVNT_H1, M>(v, var, pc, on, g1); break;
    case F_RXX: two_bit_sel<QVNT_RXX, false, M>(v, var, pc, on, g2); break;
    case F_RYY: two_bit_sel<QVNT_RYY, false, M>(v, var, pc, on, g2); break;
    case F_SWAP: two_bit_sel<QVNT_SWAP, true, M>(v, var, pc, on, g2); break;
    case F_ISWAP: two_bit_sel<QVNT_ISWAP, true, M>(v, var, pc, on, g2); break;
    case F_ISWAPD: two_bit_sel<QVNT_ISWAP, true, M>(v, var, pc, on, g2d); break;
    case F_SQSW: two_bit_sel<QVNT_SQRT_SWAP, true, M>(v, var, pc, on, g2); break;
    case F_SQSWD: two_bit_sel<QVNT_SQRT_SWAP, true, M>(v, var, pc, on, g2d); break;
    case F_SQIS: two_bit_sel<QVNT_SQRT_ISWAP, true, M>(v, var, pc, on, g2); break;
    case F_SQISD: two_bit_sel<QVNT_SQRT_ISWAP, true, M>(v, var, pc, on, g2d); break;
    case F_H2: quad_sel<false, M>(v, var, pc, on); break;
    default: quad_sel<true, M>(v, var, pc, on); break;
    }
}

}  // namespace runs
}  // namespace qvnt
