// One SingleOp of a run on the 2^B amplitudes a thread holds (runs.hpp): the
// formulas of device.hpp on the register array, every index known at
// compile time.
#pragma once

#include "device.hpp"
#include "runs.hpp"
#include "tile.hpp"

namespace qvnt {
namespace runs {

using tile::put;

QVNT_HD Par par_of(double re, double im, uint32_t a, bool dagger) {
    Par g{};
    g.a = a;
    g.re = re;
    g.im = im;
    g.dagger = dagger ? 1u : 0u;
    g.i_pow = 1u;  // one act bit (atomic/y.rs:11)
    return g;
}

// one register bit J, at the register indices of pc (M: not all of them, or
// not on all lanes)
template <int B, int K, int J, bool M, class R>
QVNT_HD void one_bit(cplx<R>* v, uint32_t pc, bool on, const Par& g) {
#pragma unroll
    for (int i = 0; i < 1 << B; ++i) {
        if (i & (1 << J)) continue;
        if (M && !((pc >> i) & 1u)) continue;
        const cplx<R> x0 = v[i], x1 = v[i | (1 << J)];
        put<M>(v[i], f_pair<K>(g, 0, x0, x1), on);
        put<M>(v[i | (1 << J)], f_pair<K>(g, 1, x1, x0), on);
    }
}
template <int B, int K, bool M, class R>
QVNT_HD void one_bit_sel(cplx<R>* v, uint32_t j, uint32_t pc, bool on, const Par& g) {
    switch (j) {
    case 0: one_bit<B, K, 0, M>(v, pc, on, g); break;
    case 1: one_bit<B, K, 1, M>(v, pc, on, g); break;
    case 2: one_bit<B, K, 2, M>(v, pc, on, g); break;
    default: if constexpr (B > 3) one_bit<B, K, 3, M>(v, pc, on, g); break;
    }
}

// two register bits, mask P: both parities' pairs (r, r ^ 3), or the odd one only
template <int B, int K, int P, bool ODD, bool M, class R>
QVNT_HD void two_bit(cplx<R>* v, uint32_t pc, bool on, const Par& g) {
    constexpr int lo = P & -P, hi = P ^ lo;
#pragma unroll
    for (int i = 0; i < 1 << B; ++i) {
        if (i & P) continue;
        if (M && !((pc >> i) & 1u)) continue;
        if (!ODD) {
            const cplx<R> x0 = v[i], x3 = v[i | P];
            put<M>(v[i], f_pair<K>(g, 0, x0, x3), on);
            put<M>(v[i | P], f_pair<K>(g, 3, x3, x0), on);
        }
        const cplx<R> x1 = v[i | lo], x2 = v[i | hi];
        put<M>(v[i | lo], f_pair<K>(g, 1, x1, x2), on);
        put<M>(v[i | hi], f_pair<K>(g, 2, x2, x1), on);
    }
}
template <int B, int K, bool ODD, bool M, class R>
QVNT_HD void two_bit_sel(cplx<R>* v, uint32_t b, uint32_t pc, bool on, const Par& g) {
    switch (b) {
    case 3: two_bit<B, K, 3, ODD, M>(v, pc, on, g); break;
    case 5: two_bit<B, K, 5, ODD, M>(v, pc, on, g); break;
    case 6: two_bit<B, K, 6, ODD, M>(v, pc, on, g); break;
    case 9: if constexpr (B > 3) two_bit<B, K, 9, ODD, M>(v, pc, on, g); break;
    case 10: if constexpr (B > 3) two_bit<B, K, 10, ODD, M>(v, pc, on, g); break;
    default: if constexpr (B > 3) two_bit<B, K, 12, ODD, M>(v, pc, on, g); break;
    }
}

// h2 (h2.rs:22-38): slot bit 0 is the gate's a, the lower register bit
// unless REV
template <int B, int P, bool REV, bool M, class R>
QVNT_HD void quad(cplx<R>* v, uint32_t pc, bool on) {
    constexpr int lo = P & -P, hi = P ^ lo, a = REV ? hi : lo, b = REV ? lo : hi;
#pragma unroll
    for (int i = 0; i < 1 << B; ++i) {
        if (i & P) continue;
        if (M && !((pc >> i) & 1u)) continue;
        const c64 x[4] = {up(v[i]), up(v[i | a]), up(v[i | b]), up(v[i | a | b])};
        put<M>(v[i], down<R>(f_h2_rel(0, x[0], x[1], x[2], x[3])), on);
        put<M>(v[i | a], down<R>(f_h2_rel(1, x[1], x[0], x[3], x[2])), on);
        put<M>(v[i | b], down<R>(f_h2_rel(2, x[2], x[3], x[0], x[1])), on);
        put<M>(v[i | a | b], down<R>(f_h2_rel(3, x[3], x[2], x[1], x[0])), on);
    }
}
template <int B, bool REV, bool M, class R>
QVNT_HD void quad_sel(cplx<R>* v, uint32_t b, uint32_t pc, bool on) {
    switch (b) {
    case 3: quad<B, 3, REV, M>(v, pc, on); break;
    case 5: quad<B, 5, REV, M>(v, pc, on); break;
    case 6: quad<B, 6, REV, M>(v, pc, on); break;
    case 9: if constexpr (B > 3) quad<B, 9, REV, M>(v, pc, on); break;
    case 10: if constexpr (B > 3) quad<B, 10, REV, M>(v, pc, on); break;
    default: if constexpr (B > 3) quad<B, 12, REV, M>(v, pc, on); break;
    }
}

// rz / rzz (rz.rs:19-25, rzz.rs:19-25): the phase's imaginary part is im
// where the act bits have odd parity, -im where even; imx is the value for
// even parity of the register bits among them, P
template <int B, int P, bool M, class R>
QVNT_HD void parity_phase(cplx<R>* v, uint32_t pc, bool on, double re, double imx) {
#pragma unroll
    for (int i = 0; i < 1 << B; ++i) {
        if (M && !((pc >> i) & 1u)) continue;
        put<M>(v[i], down<R>(cmul(c64{re, (__builtin_popcount(i & P) & 1) ? -imx : imx}, up(v[i]))), on);
    }
}
template <int B, bool M, class R>
QVNT_HD void parity_phase_sel(cplx<R>* v, uint32_t b, uint32_t pc, bool on, double re, double imx) {
    switch (b) {
    case 0: parity_phase<B, 0, M>(v, pc, on, re, imx); break;
    case 1: parity_phase<B, 1, M>(v, pc, on, re, imx); break;
    case 2: parity_phase<B, 2, M>(v, pc, on, re, imx); break;
    case 3: parity_phase<B, 3, M>(v, pc, on, re, imx); break;
    case 4: parity_phase<B, 4, M>(v, pc, on, re, imx); break;
    case 5: parity_phase<B, 5, M>(v, pc, on, re, imx); break;
    case 6: parity_phase<B, 6, M>(v, pc, on, re, imx); break;
    case 8: if constexpr (B > 3) parity_phase<B, 8, M>(v, pc, on, re, imx); break;
    case 9: if constexpr (B > 3) parity_phase<B, 9, M>(v, pc, on, re, imx); break;
    case 10: if constexpr (B > 3) parity_phase<B, 10, M>(v, pc, on, re, imx); break;
    default: if constexpr (B > 3) parity_phase<B, 12, M>(v, pc, on, re, imx); break;
    }
}

// the kinds that scale the amplitudes of pc one by one
template <int B, uint32_t F, class R>
QVNT_HD void phase(cplx<R>* v, uint32_t pc, bool on, double re, double im) {
#pragma unroll
    for (int i = 0; i < 1 << B; ++i) {
        if (!((pc >> i) & 1u)) continue;
        const c64 p = up(v[i]), e{kFrac1Sqrt2, kFrac1Sqrt2};
        put<true>(v[i], down<R>(F == F_PH ? cmul(c64{re, im}, p) : F == F_T ? cmul(e, p) : F == F_TD ? cmul(e, rotate(p, 3))
                                          : rotate(p, F == F_I1 ? 1u : F == F_I2 ? 2u : 3u)), on);
    }
}

// One op on v.  code, pc: uniform; on: whether the lane's bits satisfy the
// controls (M false: all lanes do, and pc is full); odd: the parity of the
// act bits outside the registers (per lane).
template <int B, bool M, class R>
QVNT_HD void apply_op(cplx<R>* v, uint32_t code, uint32_t pc, bool on, bool odd, double re, double im) {
    const uint32_t f = code >> 4, var = code & 15u;
    const Par g1 = par_of(re, im, 1u, false), g2 = par_of(re, im, 3u, false), g2d = par_of(re, im, 3u, true);
    switch (f) {
    case F_PH: phase<B, F_PH>(v, pc, on, re, im); break;
    case F_I1: phase<B, F_I1>(v, pc, on, re, im); break;
    case F_I2: phase<B, F_I2>(v, pc, on, re, im); break;
    case F_I3: phase<B, F_I3>(v, pc, on, re, im); break;
    case F_T: phase<B, F_T>(v, pc, on, re, im); break;
    case F_TD: phase<B, F_TD>(v, pc, on, re, im); break;
    case F_RZ: parity_phase_sel<B, M>(v, var, pc, on, re, odd ? im : -im); break;
    case F_X: one_bit_sel<B, QVNT_X, M>(v, var, pc, on, g1); break;
    case F_Y: one_bit_sel<B, QVNT_Y, M>(v, var, pc, on, g1); break;
    case F_RX: one_bit_sel<B, QVNT_RX, M>(v, var, pc, on, g1); break;
    case F_RY: one_bit_sel<B, QVNT_RY, M>(v, var, pc, on, g1); break;
    case F_H1: one_bit_sel<B, QVNT_H1, M>(v, var, pc, on, g1); break;
    case F_RXX: two_bit_sel<B, QVNT_RXX, false, M>(v, var, pc, on, g2); break;
    case F_RYY: two_bit_sel<B, QVNT_RYY, false, M>(v, var, pc, on, g2); break;
    case F_SWAP: two_bit_sel<B, QVNT_SWAP, true, M>(v, var, pc, on, g2); break;
    case F_ISWAP: two_bit_sel<B, QVNT_ISWAP, true, M>(v, var, pc, on, g2); break;
    case F_ISWAPD: two_bit_sel<B, QVNT_ISWAP, true, M>(v, var, pc, on, g2d); break;
    case F_SQSW: two_bit_sel<B, QVNT_SQRT_SWAP, true, M>(v, var, pc, on, g2); break;
    case F_SQSWD: two_bit_sel<B, QVNT_SQRT_SWAP, true, M>(v, var, pc, on, g2d); break;
    case F_SQIS: two_bit_sel<B, QVNT_SQRT_ISWAP, true, M>(v, var, pc, on, g2); break;
    case F_SQISD: two_bit_sel<B, QVNT_SQRT_ISWAP, true, M>(v, var, pc, on, g2d); break;
    case F_H2: quad_sel<B, false, M>(v, var, pc, on); break;
    default: quad_sel<B, true, M>(v, var, pc, on); break;
    }
}

}  // namespace runs
}  // namespace qvnt
