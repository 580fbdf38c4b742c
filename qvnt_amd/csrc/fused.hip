// The fused form of QReg::apply: many SingleOps per pass over the state.
//
// The host compiler (fusion.cpp) turns the queue into passes; this kernel
// runs one pass.  One block per tile of 2^t amplitudes (the tile's t qubits
// are the pass's qubit set; blocks take tiles in XCD order, xcd_order).
// The tile is read once from HBM into registers, 16 amplitudes per thread,
// moves through LDS from one phase's register layout to the next
// (tile.hpp), and is written back once.  HBM traffic is one read and one
// write of the state per pass, whatever the number of
// gates in it.  Results agree with the plain form to rounding (FMA
// contraction is on in this file; 2x2 products are merged on the host).
#pragma clang fp contract(fast)

#include <hip/hip_cooperative_groups.h>

#include <cstring>
#include <vector>

#include "device.hpp"
#include "fusion.hpp"
#include "reg.hpp"
#include "tile.hpp"

namespace qvnt {
namespace {

using namespace fusion;
using tile::exchange;
using tile::layout_of;
using tile::put;
using tile::spread;
using Layout = tile::Layout<kRegBits>;
using tile::swz;

// the local offset behind an offset of the program, which are swizzled as
// fusion.hpp's lds_swizzle has it (its own inverse)
__device__ __forceinline__ uint32_t unswizzled(uint32_t e) { return e ^ ((e >> 4) & 15u); }

__device__ __forceinline__ double fmar(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmar(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// complex multiply(-add) as explicit FMA chains: 4 instructions each
template <class R>
__device__ __forceinline__ cplx<R> fma_c(cplx<R> acc, cplx<R> a, cplx<R> x) {
    acc.re = fmar(-a.im, x.im, fmar(a.re, x.re, acc.re));
    acc.im = fmar(a.im, x.re, fmar(a.re, x.im, acc.im));
    return acc;
}
template <class R>
__device__ __forceinline__ cplx<R> mul_c(cplx<R> a, cplx<R> x) {
    return {fmar(a.re, x.re, -(a.im * x.im)), fmar(a.re, x.im, a.im * x.re)};
}
template <class R>
__device__ __forceinline__ cplx<R> ld_coef(const double* __restrict__ c, int k) {
    return {(R)c[2 * k], (R)c[2 * k + 1]};
}

// In the ops below M is false when the op acts on every register index and
// every lane; otherwise pc is the uniform pattern of the register indices it
// acts on and `on` says whether this lane does (controls on lane bits).

// 2x2 on register bit J
template <int J, bool M, class R>
__device__ __forceinline__ void apply_m2(cplx<R>* v, const double* __restrict__ c, uint32_t pc, bool on) {
    const cplx<R> u00 = ld_coef<R>(c, 0), u01 = ld_coef<R>(c, 1), u10 = ld_coef<R>(c, 2), u11 = ld_coef<R>(c, 3);
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
        if (i & (1 << J)) continue;
        if (M && !((pc >> i) & 1u)) continue;
        const cplx<R> x0 = v[i], x1 = v[i | (1 << J)];
        put<M>(v[i], fma_c(mul_c(u00, x0), u01, x1), on);
        put<M>(v[i | (1 << J)], fma_c(mul_c(u10, x0), u11, x1), on);
    }
}

template <int J0, int J1, bool M, class R>
__device__ __forceinline__ void apply_m4(cplx<R>* v, const double* __restrict__ c, uint32_t pc, bool on) {
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
        if (i & ((1 << J0) | (1 << J1))) continue;
        if (M && !((pc >> i) & 1u)) continue;
        const int idx[4] = {i, i | (1 << J0), i | (1 << J1), i | (1 << J0) | (1 << J1)};
        cplx<R> x[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = v[idx[k]];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            cplx<R> acc = mul_c(ld_coef<R>(c, 4 * r), x[0]);
            acc = fma_c(acc, ld_coef<R>(c, 4 * r + 1), x[1]);
            acc = fma_c(acc, ld_coef<R>(c, 4 * r + 2), x[2]);
            acc = fma_c(acc, ld_coef<R>(c, 4 * r + 3), x[3]);
            put<M>(v[idx[r]], acc, on);
        }
    }
}

// anti-diagonal 2x2 (u00 = u11 = 0): out0 = u01 x1, out1 = u10 x0
template <int J, bool M, class R>
__device__ __forceinline__ void apply_a2(cplx<R>* v, const double* __restrict__ c, uint32_t pc, bool on) {
    const cplx<R> u01 = ld_coef<R>(c, 0), u10 = ld_coef<R>(c, 1);
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
        if (i & (1 << J)) continue;
        if (M && !((pc >> i) & 1u)) continue;
        const cplx<R> x0 = v[i], x1 = v[i | (1 << J)];
        put<M>(v[i], mul_c(u01, x1), on);
        put<M>(v[i | (1 << J)], mul_c(u10, x0), on);
    }
}

// the swap of the two halves (x, controlled x): no arithmetic
template <int J, bool M, class R>
__device__ __forceinline__ void apply_x2(cplx<R>* v, uint32_t pc, bool on) {
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
        if (i & (1 << J)) continue;
        if (M && !((pc >> i) & 1u)) continue;
        const cplx<R> x0 = v[i], x1 = v[i | (1 << J)];
        put<M>(v[i], x1, on);
        put<M>(v[i | (1 << J)], x0, on);
    }
}

// the real middle factor of a split 2x2 (fusion.hpp: OP_T2), one FMA per
// real output: out0 = x0 - a x1, out1 = x1 + a x0
template <int J, bool M, class R>
__device__ __forceinline__ void apply_t2(cplx<R>* v, R a, uint32_t pc, bool on) {
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
        if (i & (1 << J)) continue;
        if (M && !((pc >> i) & 1u)) continue;
        const cplx<R> x0 = v[i], x1 = v[i | (1 << J)];
        put<M>(v[i], cplx<R>{fmar(-a, x1.re, x0.re), fmar(-a, x1.im, x0.im)}, on);
        put<M>(v[i | (1 << J)], cplx<R>{fmar(a, x0.re, x1.re), fmar(a, x0.im, x1.im)}, on);
    }
}

// 4x4 pairing r with r ^ 3 only: out[r] = u[r][r] x[r] + u[r][r^3] x[r^3]
template <int J0, int J1, bool M, class R>
__device__ __forceinline__ void apply_p4(cplx<R>* v, const double* __restrict__ c, uint32_t pc, bool on) {
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
        if (i & ((1 << J0) | (1 << J1))) continue;
        if (M && !((pc >> i) & 1u)) continue;
        const int idx[4] = {i, i | (1 << J0), i | (1 << J1), i | (1 << J0) | (1 << J1)};
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const cplx<R> x = v[idx[r]], y = v[idx[r ^ 3]];
            put<M>(v[idx[r]], fma_c(mul_c(ld_coef<R>(c, 2 * r), x), ld_coef<R>(c, 2 * r + 1), y), on);
            put<M>(v[idx[r ^ 3]], fma_c(mul_c(ld_coef<R>(c, 2 * (r ^ 3)), y), ld_coef<R>(c, 2 * (r ^ 3) + 1), x), on);
        }
    }
}

// P4 with real diagonal and imaginary pairing coefficients (fusion.hpp:
// OP_P4R): out_r = c_r x_r + i s_r x_(r^3)
template <int J0, int J1, bool M, class R>
__device__ __forceinline__ void apply_p4r(cplx<R>* v, const double* __restrict__ c, uint32_t pc, bool on) {
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
        if (i & ((1 << J0) | (1 << J1))) continue;
        if (M && !((pc >> i) & 1u)) continue;
        const int idx[4] = {i, i | (1 << J0), i | (1 << J1), i | (1 << J0) | (1 << J1)};
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const cplx<R> x = v[idx[r]], y = v[idx[r ^ 3]];
            const cplx<R> k = ld_coef<R>(c, r), q = ld_coef<R>(c, r ^ 3);
            put<M>(v[idx[r]], cplx<R>{k.re * x.re - k.im * y.im, k.re * x.im + k.im * y.re}, on);
            put<M>(v[idx[r ^ 3]], cplx<R>{q.re * y.re - q.im * x.im, q.re * y.im + q.im * x.re}, on);
        }
    }
}

// diagonal: one phase per register (host tables, controls folded in)
template <bool M, class R>
__device__ __forceinline__ void apply_d(cplx<R>* v, const double* __restrict__ c, bool on) {
#pragma unroll
    for (int i = 0; i < kRegs; ++i) put<M>(v[i], mul_c(ld_coef<R>(c, i), v[i]), on);
}
// The same from a table of the lane's own: the phases are loaded before the
// first is used, AHEAD at a time: 16 in FP32; 8 in FP64, where no more
// registers are free, and in the persistent kernel, where 16 take FP32 from 92
// registers and five waves a SIMD to 118 and four.  (One at a time each waited for memory: k_fused of a 28-qubit QFT FP32
// 12.9 ms so, 11.9 now; of 15 random gates on 26 qubits 327 and 251 us; FP64
// 16 qubits QFT 72 and 65 us.)
template <int AHEAD, bool M, class R>
__device__ __forceinline__ void apply_d_lane(cplx<R>* v, const double* __restrict__ c, bool on) {
#pragma unroll
    for (int i = 0; i < kRegs; i += AHEAD) {
        cplx<double> d[AHEAD];
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) d[k] = cplx<double>{c[2 * (i + k)], c[2 * (i + k) + 1]};
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) asm volatile("" : "+v"(d[k].re), "+v"(d[k].im));
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) put<M>(v[i + k], mul_c(cplx<R>{(R)d[k].re, (R)d[k].im}, v[i + k]), on);
    }
}

// a phase on the amplitudes whose register bit J is 1 (fusion.hpp: OP_PH)
template <int J, bool M, class R>
__device__ __forceinline__ void apply_ph(cplx<R>* v, const cplx<R> g, bool on) {
#pragma unroll
    for (int i = 0; i < kRegs; ++i)
        if (i & (1 << J)) put<M>(v[i], mul_c(g, v[i]), on);
}

// the structured block (fusion.hpp: OP_S): diagonal, T2 on register bits
// 0..3, diagonal, either diagonal left out when the op's sel says so --
// each form is straight-line code, so the 16 amplitudes stay in registers
// from the first product to the last
template <bool D1, bool D2, class R>
__device__ __forceinline__ void apply_s(cplx<R>* v, const double* __restrict__ c) {
    if (D1) apply_d<false>(v, c, true);
    apply_t2<0, false>(v, (R)c[2 * kRegs + 0], 0u, true);
    apply_t2<1, false>(v, (R)c[2 * kRegs + 2], 0u, true);
    apply_t2<2, false>(v, (R)c[2 * kRegs + 4], 0u, true);
    apply_t2<3, false>(v, (R)c[2 * kRegs + 6], 0u, true);
    if (D2) apply_d<false>(v, c + 2 * (kRegs + kRegBits), true);
}

// T2's and PH's coefficient, carried in the op (fusion.hpp: FOp::ga, gb)
template <class R>
__device__ __forceinline__ cplx<R> inline_coef(const FOp& op) {
    return cplx<R>{(R)__longlong_as_double((long long)op.ga), (R)__longlong_as_double((long long)op.gb)};
}

// over the active lanes of the wave; uniform
__device__ __forceinline__ bool some(bool x) { return __builtin_amdgcn_ballot_w64(x) != 0; }
__device__ __forceinline__ bool every(bool x) { return __builtin_amdgcn_ballot_w64(!x) == 0; }

// One op other than G, S and D.
template <bool M, class R>
__device__ __forceinline__ void apply_op(cplx<R>* v, const FOp& op, const double* __restrict__ c, bool on) {
    switch (op.type) {
    case OP_PH:
        switch (op.sel) {
        case 0: apply_ph<0, M>(v, inline_coef<R>(op), on); break;
        case 1: apply_ph<1, M>(v, inline_coef<R>(op), on); break;
        case 2: apply_ph<2, M>(v, inline_coef<R>(op), on); break;
        default: apply_ph<3, M>(v, inline_coef<R>(op), on); break;
        }
        break;
    case OP_T2:
        switch (op.sel) {
        case 0: apply_t2<0, M>(v, inline_coef<R>(op).re, op.pc, on); break;
        case 1: apply_t2<1, M>(v, inline_coef<R>(op).re, op.pc, on); break;
        case 2: apply_t2<2, M>(v, inline_coef<R>(op).re, op.pc, on); break;
        default: apply_t2<3, M>(v, inline_coef<R>(op).re, op.pc, on); break;
        }
        break;
    case OP_M2:
        switch (op.sel) {
        case 0: apply_m2<0, M>(v, c, op.pc, on); break;
        case 1: apply_m2<1, M>(v, c, op.pc, on); break;
        case 2: apply_m2<2, M>(v, c, op.pc, on); break;
        default: apply_m2<3, M>(v, c, op.pc, on); break;
        }
        break;
    case OP_M4:
        switch (op.sel) {
        case 1: apply_m4<0, 1, M>(v, c, op.pc, on); break;
        case 2: apply_m4<0, 2, M>(v, c, op.pc, on); break;
        case 3: apply_m4<0, 3, M>(v, c, op.pc, on); break;
        case 6: apply_m4<1, 2, M>(v, c, op.pc, on); break;
        case 7: apply_m4<1, 3, M>(v, c, op.pc, on); break;
        default: apply_m4<2, 3, M>(v, c, op.pc, on); break;
        }
        break;
    case OP_P4:
        switch (op.sel) {
        case 1: apply_p4<0, 1, M>(v, c, op.pc, on); break;
        case 2: apply_p4<0, 2, M>(v, c, op.pc, on); break;
        case 3: apply_p4<0, 3, M>(v, c, op.pc, on); break;
        case 6: apply_p4<1, 2, M>(v, c, op.pc, on); break;
        case 7: apply_p4<1, 3, M>(v, c, op.pc, on); break;
        default: apply_p4<2, 3, M>(v, c, op.pc, on); break;
        }
        break;
    case OP_P4R:
        switch (op.sel) {
        case 1: apply_p4r<0, 1, M>(v, c, op.pc, on); break;
        case 2: apply_p4r<0, 2, M>(v, c, op.pc, on); break;
        case 3: apply_p4r<0, 3, M>(v, c, op.pc, on); break;
        case 6: apply_p4r<1, 2, M>(v, c, op.pc, on); break;
        case 7: apply_p4r<1, 3, M>(v, c, op.pc, on); break;
        default: apply_p4r<2, 3, M>(v, c, op.pc, on); break;
        }
        break;
    case OP_A2:
        switch (op.sel) {
        case 0: apply_a2<0, M>(v, c, op.pc, on); break;
        case 1: apply_a2<1, M>(v, c, op.pc, on); break;
        case 2: apply_a2<2, M>(v, c, op.pc, on); break;
        default: apply_a2<3, M>(v, c, op.pc, on); break;
        }
        break;
    default:
        switch (op.sel) {
        case 0: apply_x2<0, M>(v, op.pc, on); break;
        case 1: apply_x2<1, M>(v, op.pc, on); break;
        case 2: apply_x2<2, M>(v, op.pc, on); break;
        default: apply_x2<3, M>(v, op.pc, on); break;
        }
        break;
    }
}

// No branch in here diverges: a wave whose lanes all satisfy an op's lane
// controls runs it whole, one with none skips it, a mixed one selects per
// lane.  (A divergent branch around the op makes the compiler keep the 16
// amplitudes twice, old and new: 221 VGPRs in FP64.)
//
// `next` is the phase's first op on entry and the one after its last on
// exit: each op is loaded while the one before runs (its 64 bytes are a line
// of the scalar cache, and with one wave a SIMD nothing hides the miss: 16
// qubits FP64, 400 gates, k_fused 254 us without, 240 so).  The ops of a pass
// lie one after the other, and behind the last one the program's buffer goes
// on.
template <int AHEAD, class R>
__device__ __forceinline__ void run_phase(cplx<R>* v, uint32_t begin, uint32_t end, const FOp* __restrict__ ops,
                                          const double* __restrict__ coef, uint32_t tb, uint64_t tile, FOp& next) {
    // the product of the phase's G factors (uniform, accumulated in FP64)
    cplx<double> scal{1.0, 0.0};
    bool scaled = false;
    for (uint32_t o = begin; o < end; ++o) {
        const FOp op = next;
        next = ops[o + 1];
        // controls on lane bits (this thread's base) and on bits outside the
        // tile (which differ between the lanes of a wave only where it holds
        // several small tiles, see persist_unit)
        const bool on = (tb & op.lctrl) == op.lctrl && (tile & op.gctrl) == op.gctrl;
        if (!some(on)) continue;
        const bool all = every(on);
        const double* c = coef + op.coef;
        const uint32_t type = op.type;
        if (type == OP_S) {
            switch (op.sel) {
            case 0: apply_s<false, false>(v, c); break;
            case 1: apply_s<true, false>(v, c); break;
            case 2: apply_s<false, true>(v, c); break;
            default: apply_s<true, true>(v, c); break;
            }
        } else if (type == OP_G) {
            const uint32_t k = ((tile & op.ga) != 0 ? 1u : 0u) | ((tile & op.gb) != 0 ? 2u : 0u);
            const cplx<double> g = mul_c(ld_coef<double>(c, (int)(k * kRegs)), scal);
            scal.re = on ? g.re : scal.re;
            scal.im = on ? g.im : scal.im;
            scaled |= on;
        } else if (type == OP_D) {
            // table variant from the non-register operands
            const bool ea = (op.la | op.ga) != 0, eb = (op.lb | op.gb) != 0;
            const uint32_t k = ((((tb & op.la) | (tile & op.ga)) != 0) ? 1u : 0u) |
                               ((((tb & op.lb) | (tile & op.gb)) != 0) ? 2u : 0u);
            // dmode 1: the variant-0 table, then (waves whose operand bit is
            // set) the ratio table, both uniform loads; else each lane loads
            // its own variant
            if ((ea || eb) && op.dmode != 1) {
                apply_d_lane<AHEAD, true>(v, c + 2 * kRegs * k, on);
            } else {
                const uint32_t var = ea ? 1u : 2u;
                if (all) apply_d<false>(v, c, true);
                else apply_d<true>(v, c, on);
                const bool second = (ea || eb) && (k & var) != 0 && on;
                if (some(second)) {
                    if (every(second)) apply_d<false>(v, c + 2 * kRegs * var, true);
                    else apply_d<true>(v, c + 2 * kRegs * var, second);
                }
            }
        } else if (all && op.pc == 0xFFFFu) {
            apply_op<false>(v, op, c, true);
        } else {
            apply_op<true>(v, op, c, on);
        }
    }
    if (some(scaled)) {
        const cplx<R> f{(R)scal.re, (R)scal.im};
#pragma unroll
        for (int i = 0; i < kRegs; ++i) put<true>(v[i], mul_c(f, v[i]), scaled);
    }
}

typedef double mf64x4 __attribute__((ext_vector_type(4)));
typedef float mf32x4 __attribute__((ext_vector_type(4)));

// One 16x16x4 matrix-core step: acc(16x16) += A(16x4) * B(4x16).
// Lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16].  Element i of
// its accumulator is acc[l / 16 + 4 i][l % 16] for f64 and
// acc[4 (l / 16) + i][l % 16] for f32 (measured on gfx950).
__device__ __forceinline__ mf64x4 mfma(double a, double b, mf64x4 acc) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
}
__device__ __forceinline__ mf32x4 mfma(float a, float b, mf32x4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
}
template <class R> struct AccOf;
template <> struct AccOf<double> { typedef mf64x4 type; static constexpr bool hi_low_bits = true; };
template <> struct AccOf<float> { typedef mf32x4 type; static constexpr bool hi_low_bits = false; };

// The register layout of a dense phase (16x16 unitary U on the phase's
// register bits): the tile is a 16 x 2^(t-4) complex matrix X, row = register
// index of the phase, column = thread base, and each 64-lane wave owns the 64
// columns of its own threads.  Lane l holds, in register 4 c + s, the element
// of row 4 s + l / 16 and column 16 c + l % 16 of them: the matrix cores'
// B operand of step s for column tile c.
__device__ __forceinline__ Layout dense_layout(const FPhase& ph, uint32_t tid) {
    const uint32_t hi = (tid >> 4) & 3u;
    uint32_t e = spread<kRegBits>(tid & ~48u, ph.rpos);
    e |= ((hi & 1u) << ph.rpos[0]) | ((hi >> 1) << ph.rpos[1]);
    Layout l;
    l.base = swz(e);
    l.bit[0] = swz(1u << ph.rpos[2]);
    l.bit[1] = swz(1u << ph.rpos[3]);
    l.bit[2] = swz(spread<kRegBits>(16u, ph.rpos));
    l.bit[3] = swz(spread<kRegBits>(32u, ph.rpos));
    return l;
}

// X := U X in dense_layout, as a real 32x32 GEMM on the matrix cores:
//   Yre = Ure Xre - Uim Xim,   Yim = Ure Xim + Uim Xre.
// The result comes out in the layout it went in: element i of lane l's
// accumulator is row l / 16 + 4 i in f64, and in f32, where it is row
// 4 (l / 16) + i, U's rows are taken in the order that makes it so.
template <class R>
__device__ __forceinline__ void dense_phase(cplx<R>* v, const double* __restrict__ u, uint32_t tid) {
    typedef typename AccOf<R>::type Acc;
    const uint32_t lane = tid & 63u, hi = lane >> 4, m = lane & 15u;
    // A operands: row m (f32: of the reordered U) and column 4 s + hi
    const uint32_t row = AccOf<R>::hi_low_bits ? m : (m >> 2) | ((m & 3u) << 2);
    R ure[4], uim[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const uint32_t e = 16u * row + 4u * (uint32_t)s + hi;
        ure[s] = (R)u[2 * e];
        uim[s] = (R)u[2 * e + 1];
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        Acc yre = {0, 0, 0, 0}, yim = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const cplx<R> x = v[4 * c + s];
            yre = mfma(ure[s], x.re, yre);
            yim = mfma(ure[s], x.im, yim);
            yre = mfma(-uim[s], x.im, yre);
            yim = mfma(uim[s], x.re, yim);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) put<false>(v[4 * c + i], cplx<R>{yre[i], yim[i]}, true);
    }
}

// Global index of local element 0 of tile `tile_index` (the tiles
// enumerate the bits outside the tile's qubit set): zeros inserted at the
// tile's bit positions.
__device__ __forceinline__ uint64_t tile_base(const uint32_t* tp, uint32_t t, uint64_t tile_index) {
    uint64_t tile = tile_index;
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)kMaxTile; ++k) {
        if (k < t) {  // uniform
            const uint64_t lo = tile & ((1ull << tp[k]) - 1u);
            tile = ((tile ^ lo) << 1) | lo;
        }
    }
    return tile;
}

// The pass's local-bit positions from the packed copy (one byte each):
// four words read at once instead of a dependent scalar load per bit in
// the loops over them, and four scalar registers instead of thirteen.
__device__ __forceinline__ void load_tpos(const FPass& pass, uint32_t* tp) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = pass.tpack[i];
#pragma unroll
    for (int k = 0; k < kMaxTile; ++k) tp[k] = (w[k / 4] >> (8 * (k % 4))) & 63u;
}

// global offset of local index l (bits from t up are zero)
__device__ __forceinline__ uint64_t global_offset(const uint32_t* tp, uint32_t l) {
    uint64_t off = 0;
#pragma unroll
    for (int k = 0; k < kMaxTile; ++k) off |= (uint64_t)((l >> k) & 1u) << tp[k];
    return off;
}

// Where the tile is read from or written to HBM: the local bits the
// registers run over, and the thread's address.
template <class R>
struct Edge {
    bool own;
    uint32_t pos[kRegBits];
    uint32_t tb;              // local index of register 0
    uint64_t step[kRegBits];  // global offsets of the register bits (uniform)
    // The first (e 0) or last (1) phase's own layout where a whole 128-byte
    // line stays among the threads in it (local bits 0..2 in FP64, 0..3 in
    // FP32; saves one exchange), else the tile's top bits in the registers.
    __device__ __forceinline__ void set(const FPass& pass, int e, bool allow, uint32_t tid) {
        own = allow && !pass.edge_dense[e] && (pass.edge[e] & 63u) >= (sizeof(R) == 8 ? 3u : 4u);
        const uint32_t l = own ? pass.edge[e] : (pass.t - kRegBits) * 0x01010101u + 0x03020100u;
        const uint32_t g = own ? pass.edge_global[e] : pass.top_global;
#pragma unroll
        for (int j = 0; j < kRegBits; ++j) {
            pos[j] = (l >> (8 * j)) & 63u;
            step[j] = 1ull << ((g >> (8 * j)) & 63u);
        }
        tb = spread<kRegBits>(tid, pos);
    }
    __device__ __forceinline__ uint64_t off(int i) const {
        uint64_t o = 0;
#pragma unroll
        for (int j = 0; j < kRegBits; ++j)
            if (i >> j & 1) o |= step[j];
        return o;
    }
};

// Passes of at most this many tiles bring their program near first
// (warm_program).  With more, the blocks before have done so, and the touches
// only take time: 31-qubit Ising steps in FP32 96 ms without, 112 with.
constexpr uint32_t kWarmTiles = 2048;

// Brings the pass's phases, ops and coefficients into the L2 of this block's
// XCD: one load a line, all at once and beside the tile's own, where the op
// loop's scalar loads would wait for memory one after the other (16 qubits
// FP64, 400 gates: 370 us of k_fused without; with the ops' tables found
// through the ops, and the edges' layouts through the phases, three misses
// one after the other before the first op, 240; 216 so).
__device__ __forceinline__ uint32_t warm_program(const FPass& pass, const FPhase* __restrict__ phases, const FOp* __restrict__ ops,
                                                 const double* __restrict__ coef, uint32_t tid) {
    uint32_t seen = 0;
    const auto touch = [&](const void* from, const void* to) {
        const unsigned char* p = static_cast<const unsigned char*>(from);
        for (uint32_t k = tid * 128u; k < (uint32_t)(static_cast<const unsigned char*>(to) - p); k += pass.nthreads * 128u)
            seen ^= *reinterpret_cast<const uint32_t*>(p + k);
    };
    touch(ops + pass.op_begin, ops + pass.op_end);
    touch(coef + pass.coef_begin, coef + pass.coef_end);
    touch(phases + pass.phase_begin, phases + pass.phase_end);
    return seen;
}

// One tile of one pass: read 2^t amplitudes, run the pass's phases, write
// them back; the pass and program live in scalar-loadable memory.
// tiles: of the pass (kWarmTiles); tid: the thread's index within the tile (0 .. 2^(t-4) - 1); lds: 2^t
// reals.  ACTIVE false: the threads run the phases (and their barriers) on
// their own LDS region but neither read nor write HBM -- a block of the
// persistent batched kernel whose tile group has no tile (see
// k_batch_persist).
template <class R, bool GATED = false>
__device__ __forceinline__ void fused_tile(cplx<R>* __restrict__ psi, const FPass& pass, const FPhase* __restrict__ phases,
                                           const FOp* __restrict__ ops, const double* __restrict__ coef,
                                           uint64_t tile_index, uint32_t tiles, R* lds, uint32_t tid, bool active = true) {
    const bool warm = tiles <= kWarmTiles;
    uint32_t seen = 0;
    if (warm) seen = warm_program(pass, phases, ops, coef, tid);
    uint32_t tp[kMaxTile];
    load_tpos(pass, tp);
    const uint64_t tile = tile_base(tp, pass.t, tile_index);
    const uint32_t p0 = pass.phase_begin, p1 = pass.phase_end;
    cplx<R> v[kRegs];
    bool own_in;
    uint32_t tb;
    Layout cur;
    {
        Edge<R> in;
        in.set(pass, 0, true, tid);
        own_in = in.own;
        tb = in.tb;
        cur = layout_of<kRegBits>(tb, in.pos);
        const cplx<R>* p = psi + (tile | global_offset(tp, tb));
        // One branch around the 16 loads: with a branch each (uniform ones
        // stay branches in this file) every load waited for the one before
        // it.  k_batch_persist, 1024 registers of 10..20 qubits, FP32, tiles
        // of 12: 11.1 ms so, 8.9 now; FP64 12.2 and 10.4.
        if (!GATED || active) {
#pragma unroll
            for (int i = 0; i < kRegs; ++i) {
                const cplx<R>* q = p + in.off(i);
                v[i] = cplx<R>{__builtin_nontemporal_load(&q->re), __builtin_nontemporal_load(&q->im)};
            }
        } else {
#pragma unroll
            for (int i = 0; i < kRegs; ++i) v[i] = cplx<R>{(R)0, (R)0};
        }
    }
    if (warm) asm volatile("" ::"v"(seen));
    // (each phase's header, too, is loaded while the one before runs)
    FOp next = ops[pass.op_begin];
    FPhase ahead = phases[p0];
    for (uint32_t p = p0; p < p1; ++p) {
        const FPhase ph = ahead;
        ahead = phases[p + 1];
        if (ph.dense) {
            const Layout to = dense_layout(ph, tid);
            exchange<kRegBits>(v, lds, cur, to);
            cur = to;
            dense_phase(v, coef + ph.ucoef, tid);
            continue;
        }
        if (p != p0 || !(own_in || pass.direct_first)) {
            tb = spread<kRegBits>(tid, ph.rpos);
            const Layout to = layout_of<kRegBits>(tb, ph.rpos);
            exchange<kRegBits>(v, lds, cur, to);
            cur = to;
        }
        run_phase<(GATED || sizeof(R) == 8) ? 8 : 16>(v, ph.op_begin, ph.op_end, ops, coef, tb, tile, next);
    }
    Edge<R> out;
    out.set(pass, 1, !pass.permuted, tid);
    if (pass.permuted) {
        // through the pass's qubit permutation: the thread that stores local
        // index tid + j 2^(t-4) reads it from pimg / pout
        uint32_t s = 0;
#pragma unroll
        for (uint32_t k = 0; k < (uint32_t)(kMaxTile - kRegBits); ++k)
            if (k + kRegBits < pass.t) s ^= unswizzled(pass.pimg[k]) & (0u - ((tid >> k) & 1u));
        s = swz(s);
        exchange<kRegBits>(v, lds, cur, [&](int i) { return s ^ swz(unswizzled(pass.pout[i])); });
    } else if (!out.own && !pass.direct_last) {
        exchange<kRegBits>(v, lds, cur, layout_of<kRegBits>(out.tb, out.pos));
    }
    if (!GATED || active) {
        // every amplitude of the tile is read once and written once per
        // pass: non-temporal stores (streamed through the caches, evicted first)
        cplx<R>* p = psi + (tile | global_offset(tp, out.tb));
#pragma unroll
        for (int i = 0; i < kRegs; ++i) {
            cplx<R>* q = p + out.off(i);
            __builtin_nontemporal_store(v[i].re, &q->re);
            __builtin_nontemporal_store(v[i].im, &q->im);
        }
    }
}

// Four waves per SIMD: the exchange takes half a tile of LDS (32 KiB for
// 2^12 FP64 or 2^13 FP32 amplitudes), and the op code keeps one copy of the
// 16 amplitudes.  The persistent kernel's loop state does not fit beside them
// in 128 registers in FP64: three (137 VGPRs; FP32 takes 92, for five).
#define QVNT_FUSED_BOUNDS __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4)))
#define QVNT_PERSIST_BOUNDS __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(1, 3)))

// XCD-aware block order.  The dispatcher hands workgroups to the eight XCDs
// round robin (block b to XCD b mod 8), and each XCD has its own L2 and
// address translation.  With G = 8q + r blocks, block b < 8q runs work
// item (b mod 8) q + b / 8, so XCD x walks the contiguous range
// [x q, (x + 1) q): its concurrently running blocks touch neighbouring
// lines and pages.  The last r blocks keep their index.  A bijection on
// [0, G).
__device__ __forceinline__ uint32_t xcd_order(uint32_t b, uint32_t G) {
    const uint32_t q = G >> 3;
    return b < (q << 3) ? (b & 7u) * q + (b >> 3) : b;
}

template <class R>
__global__ QVNT_FUSED_BOUNDS void k_fused(cplx<R>* __restrict__ psi, FPass pass, const FPhase* __restrict__ phases,
                                               const FOp* __restrict__ ops, const double* __restrict__ coef) {
    extern __shared__ unsigned char smem[];
    fused_tile<R>(psi, pass, phases, ops, coef, xcd_order(blockIdx.x, gridDim.x), gridDim.x,
                  reinterpret_cast<R*>(smem), threadIdx.x);
}

// The batched form: the tiles of one pass of many registers in one launch
// (every item's pass has the launch's t).  Block b (in XCD order, xcd_order)
// runs tile b - items[map[b]].block0 of item map[b]; registers, passes and
// programs are addressed by offsets from the two base pointers.  (Two tiles a
// block share what the scalar cache holds of the program, which paid with two
// waves per SIMD; with four, 4096 registers FP64 take 30.6 ms with two tiles
// a block and 29.3 with one.)
template <class R>
__global__ QVNT_FUSED_BOUNDS void k_batch(cplx<R>* __restrict__ arena, const unsigned char* __restrict__ prog,
                                               const BItem* __restrict__ items, const uint32_t* __restrict__ map) {
    extern __shared__ unsigned char smem[];
    const uint32_t b = xcd_order(blockIdx.x, gridDim.x);
    const BItem it = items[map[b]];
    fused_tile<R>(arena + it.psi_off, *reinterpret_cast<const FPass*>(prog + it.pass_off),
                  reinterpret_cast<const FPhase*>(prog + it.phase_off), reinterpret_cast<const FOp*>(prog + it.op_off),
                  reinterpret_cast<const double*>(prog + it.coef_off), b - it.block0, it.tiles, reinterpret_cast<R*>(smem), threadIdx.x);
}

// One work unit of the persistent batched kernel (below): up to
// 2^(tmax-t) tiles of one register pass of tile size t, one tile per group
// of 2^(t-4) threads with its own 2^t-amplitude LDS region; all groups run
// the same program, so they pass the same barriers, and a group without a
// tile runs the phases without HBM traffic.  Groups of whole waves (t >= 10)
// take their tile index wave-uniform, as in k_batch, so the program's
// tile-dependent branches and table loads stay scalar.
template <class R>
__device__ __forceinline__ void persist_unit(cplx<R>* __restrict__ arena, const unsigned char* __restrict__ prog,
                                             const BItem* __restrict__ items, const PUnit& un, unsigned char* smem) {
    const BItem it = items[un.item];
    const FPass& pass = *reinterpret_cast<const FPass*>(prog + it.pass_off);
    const FPhase* ph = reinterpret_cast<const FPhase*>(prog + it.phase_off);
    const FOp* ops = reinterpret_cast<const FOp*>(prog + it.op_off);
    const double* coef = reinterpret_cast<const double*>(prog + it.coef_off);
    const uint32_t tbits = pass.t - kRegBits;                 // threads per tile: 2^tbits
    const uint32_t tid = threadIdx.x & ((1u << tbits) - 1u);
    if (tbits >= 6) {
        const uint32_t group = __builtin_amdgcn_readfirstlane(threadIdx.x >> tbits);
        const uint32_t tile = un.tile0 + group;
        fused_tile<R, true>(arena + it.psi_off, pass, ph, ops, coef, tile, ~0u,
                            reinterpret_cast<R*>(smem) + ((size_t)group << pass.t), tid, tile < un.tile_end);
    } else {
        const uint32_t group = threadIdx.x >> tbits;
        const uint32_t tile = un.tile0 + group;
        fused_tile<R, true>(arena + it.psi_off, pass, ph, ops, coef, tile, ~0u,
                            reinterpret_cast<R*>(smem) + ((size_t)group << pass.t), tid, tile < un.tile_end);
    }
}

// Units of each round (in thousandths) that blocks claim instead of taking
// them in a fixed order, kPersistChunk consecutive units per claim
// (4096-register batch, FP64, when a tile took twice the LDS and two waves a
// SIMD ran: 54.2 ms per run with none; one unit per claim: 51.6 with 100, 50.7
// with 150, 53.1 with 250; with 150, two units per claim 48.3, four 48.3; 300
// in fours 48.3, 400 in fours 48.5).
constexpr uint32_t kPersistClaimed = 150;
constexpr uint32_t kPersistChunk = 4;

// The batched form as one persistent launch (cooperative: every block is
// resident).  The blocks walk the rounds in order and meet at a grid
// barrier between rounds, which also makes a round's HBM writes visible to
// the next (cooperative groups' grid sync: release and acquire fences at
// device scope).  In each round, a whole number of strides of the round's
// first units go out in a fixed order: with a grid of 8q blocks, XCD x (the
// blocks b with b mod 8 = x, which the dispatcher places on XCD x) walks
// its own contiguous eighth of them, its q blocks q apart.  The rest (about
// kPersistClaimed thousandths) are claimed kPersistChunk consecutive units
// at a time from the round's counter, so blocks that finish early take
// more of the round's tail.
// status[1 + r] is round r's counter: zero when the launch starts, zeroed
// for round r + 1 by block 0 during round r (nobody claims from it before
// the barrier that ends round r), and round 0's zeroed again by block 0 at
// the end, after every block has left it; so the counters are zero again
// when the launch ends.
//
// The dynamic LDS array starts 16-byte aligned after the claim word (its
// elements are 4 or 8 bytes; at byte 4 the FP64 ones would be misaligned).
//
// The launch bounds ask for one wave a SIMD at least and three at most, so
// nothing pads the register allocation beyond what the kernel uses, which is
// what the runtime's occupancy query (and so the cooperative grid size) counts.
//
// A launch that is not cooperative (a graph node whose cooperative
// attribute the runtime did not honour) has no grid barrier: every block
// sees that alike, block 0 sets *status to 1, and all return before any
// barrier or HBM access.
template <class R>
__global__ QVNT_PERSIST_BOUNDS void k_batch_persist(cplx<R>* __restrict__ arena, const unsigned char* __restrict__ prog,
                                                  const BItem* __restrict__ items, const PUnit* __restrict__ units,
                                                  const uint32_t* __restrict__ round_begin, uint32_t rounds,
                                                  uint32_t* status) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ uint32_t claim;
    cooperative_groups::grid_group grid = cooperative_groups::this_grid();
    if (!grid.is_valid()) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *status = 1u;
        return;
    }
    uint32_t* count = status + 1;
    const uint32_t G = gridDim.x;
    const bool by_xcd = (G & 7u) == 0;
    const uint32_t xcd = blockIdx.x & 7u;
    for (uint32_t r = 0; r < rounds; ++r) {
        const uint32_t rb = round_begin[r], u_end = round_begin[r + 1], n = u_end - rb;
        if (blockIdx.x == 0 && threadIdx.x == 0 && r + 1 < rounds) count[r + 1] = 0u;
        const uint32_t claimed = (uint32_t)(((uint64_t)n * kPersistClaimed) / 1000u);
        const uint32_t fixed = ((n - claimed) / G) * G;       // whole strides
        // this block's units of the fixed part: [next, stop) in steps of step
        uint32_t next = rb + blockIdx.x, stop = rb + fixed, step = G;
        if (by_xcd) {
            next = rb + xcd * (fixed >> 3) + (blockIdx.x >> 3);
            stop = rb + (xcd + 1u) * (fixed >> 3);
            step = G >> 3;
        }
        // the claimed units in hand: [have, have_end)
        uint32_t have = 0, have_end = 0;
        for (;;) {
            uint32_t u;
            if (next < stop) {  // uniform
                u = next;
                next += step;
            } else {
                if (have >= have_end) {
                    if (threadIdx.x == 0) claim = atomicAdd(&count[r], 1u);
                    __syncthreads();
                    const uint64_t first = (uint64_t)claim * kPersistChunk;
                    __syncthreads();  // before the next claim overwrites it
                    if (first >= n - fixed) break;
                    have = rb + fixed + (uint32_t)first;
                    have_end = rb + fixed + (uint32_t)min((uint64_t)(n - fixed), first + kPersistChunk);
                }
                u = have++;
            }
            persist_unit<R>(arena, prog, items, units[u], smem);
            // the next unit's first LDS writes may hit elements other
            // threads still read in this unit's last phase
            __syncthreads();
        }
        grid.sync();
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) count[0] = 0u;
}

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

struct ProgramLayout {
    size_t ph_off, op_off, cf_off, total;
};
ProgramLayout program_layout(const Program& prog) {
    ProgramLayout L;
    L.ph_off = 0;
    L.op_off = align256(L.ph_off + prog.phases.size() * sizeof(FPhase));
    L.cf_off = align256(L.op_off + prog.ops.size() * sizeof(FOp));
    L.total = L.cf_off + prog.coef.size() * sizeof(double) + 256;
    return L;
}

}  // namespace

size_t program_bytes(const Program& prog) { return program_layout(prog).total; }

int batch_persist_grid(qvnt_prec prec, uint32_t tmax, uint32_t* blocks) {
    const size_t amp = prec == QVNT_F64 ? 16 : 8;
    const int threads = 1 << (tmax - kRegBits);
    const size_t lds = ((size_t)1 << tmax) * amp / 2;
    int per_cu = 0, dev = 0, cus = 0, coop = 0;
    QVNT_HIP(hipGetDevice(&dev));
    QVNT_HIP(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev));
    if (!coop) return fail(QVNT_E_HIP, "the device does not support cooperative launches");
    QVNT_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    if (prec == QVNT_F64)
        QVNT_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_batch_persist<double>, threads, lds));
    else
        QVNT_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_batch_persist<float>, threads, lds));
    if (per_cu <= 0) return fail(QVNT_E_HIP, "the persistent batched kernel does not fit a compute unit");
    *blocks = (uint32_t)per_cu * (uint32_t)cus;
    return QVNT_OK;
}

int launch_batch_persist(hipStream_t stream, qvnt_prec prec, void* arena, const void* prog, const BItem* items,
                         const PUnit* units, const uint32_t* round_begin, uint32_t rounds, uint32_t tmax,
                         uint32_t blocks, uint32_t* status, hipGraph_t* graph) {
    const size_t amp = prec == QVNT_F64 ? 16 : 8;
    const dim3 grid(blocks), block(1u << (tmax - kRegBits));
    const size_t lds = ((size_t)1 << tmax) * amp / 2;
    const unsigned char* p = static_cast<const unsigned char*>(prog);
    void* args[] = {&arena, &p, &items, &units, &round_begin, &rounds, &status};
    void* fn = prec == QVNT_F64 ? reinterpret_cast<void*>(k_batch_persist<double>)
                                : reinterpret_cast<void*>(k_batch_persist<float>);
    if (!graph) {
        QVNT_HIP(hipLaunchCooperativeKernel(fn, grid, block, args, (unsigned)lds, stream));
        return QVNT_OK;
    }
    // the cooperative launch captured from the stream into a graph (on
    // ROCm 7.2 a captured cooperative launch stays cooperative, while a
    // kernel node built by hand with the cooperative attribute does not;
    // the kernel's own check covers either)
    QVNT_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
    const hipError_t e = hipLaunchCooperativeKernel(fn, grid, block, args, (unsigned)lds, stream);
    hipGraph_t g = nullptr;
    const hipError_t end = hipStreamEndCapture(stream, &g);
    if (e != hipSuccess || end != hipSuccess || !g) {
        if (g) (void)hipGraphDestroy(g);
        (void)hipGetLastError();
        return fail(QVNT_E_HIP, "capturing the persistent batched launch");
    }
    *graph = g;
    return QVNT_OK;
}

int launch_batch(hipStream_t stream, qvnt_prec prec, void* arena, const void* prog, const BItem* items, const uint32_t* map,
                 uint32_t t, uint32_t blocks) {
    const size_t amp = prec == QVNT_F64 ? 16 : 8;
    const dim3 grid(blocks), block(1u << (t - kRegBits));
    const size_t lds = ((size_t)1 << t) * amp / 2;
    const unsigned char* p = static_cast<const unsigned char*>(prog);
    if (prec == QVNT_F64)
        hipLaunchKernelGGL(k_batch<double>, grid, block, lds, stream, static_cast<c64*>(arena), p, items, map);
    else
        hipLaunchKernelGGL(k_batch<float>, grid, block, lds, stream, static_cast<c32*>(arena), p, items, map);
    QVNT_HIP(hipGetLastError());
    return QVNT_OK;
}

void pack_program(const Program& prog, unsigned char* host) {
    const ProgramLayout L = program_layout(prog);
    std::memset(host, 0, L.total);
    if (!prog.phases.empty()) std::memcpy(host + L.ph_off, prog.phases.data(), prog.phases.size() * sizeof(FPhase));
    if (!prog.ops.empty()) std::memcpy(host + L.op_off, prog.ops.data(), prog.ops.size() * sizeof(FOp));
    if (!prog.coef.empty()) std::memcpy(host + L.cf_off, prog.coef.data(), prog.coef.size() * sizeof(double));
}

int launch_program(qvnt_reg* r, const Program& prog, const void* dev) {
    const ProgramLayout L = program_layout(prog);
    const unsigned char* d = static_cast<const unsigned char*>(dev);
    const FPhase* dph = reinterpret_cast<const FPhase*>(d + L.ph_off);
    const FOp* dop = reinterpret_cast<const FOp*>(d + L.op_off);
    const double* dcf = reinterpret_cast<const double*>(d + L.cf_off);
    for (const FPass& fp : prog.passes) {
        const uint64_t tiles = r->len >> fp.t;
        const size_t lds = ((size_t)1 << fp.t) * r->amp_bytes() / 2;
        Timed t(r, QVNT_K_FUSED, 2.0 * (double)r->amp_bytes() * (double)r->len);
        if (r->prec == QVNT_F64)
            hipLaunchKernelGGL(k_fused<double>, dim3((unsigned)tiles), dim3(fp.nthreads), lds, r->stream,
                               static_cast<c64*>(r->psi), fp, dph, dop, dcf);
        else
            hipLaunchKernelGGL(k_fused<float>, dim3((unsigned)tiles), dim3(fp.nthreads), lds, r->stream,
                               static_cast<c32*>(r->psi), fp, dph, dop, dcf);
        QVNT_HIP(hipGetLastError());
    }
    return QVNT_OK;
}

namespace {

// Uploads the program (stream-ordered, from pageable memory) and launches
// one kernel per pass.
int run_program(qvnt_reg* r, const Program& prog) {
    static thread_local std::vector<unsigned char> host;
    const size_t total = program_bytes(prog);
    if (total > r->prog_cap) {
        QVNT_HIP(hipStreamSynchronize(r->stream));
        void* old = r->prog;
        const size_t old_cap = r->prog_cap;
        r->prog = nullptr;
        r->prog_cap = 0;
        // (a register that owns its memory takes its blocks from the device's
        // cache and gives them back there; the stream is synchronized above)
        if (r->owns_memory) {
            dev_release(r->device, old, old_cap);
            if (dev_alloc(r->device, &r->prog, total) != QVNT_OK)
                return fail(QVNT_E_OOM, "device memory for the fused program");
        } else {
            if (old) QVNT_HIP(hipFree(old));
            if (hipMalloc(&r->prog, total) != hipSuccess) return fail(QVNT_E_OOM, "device memory for the fused program");
        }
        r->prog_cap = total;
    }
    host.resize(total);
    pack_program(prog, host.data());
    QVNT_HIP(hipMemcpyAsync(r->prog, host.data(), total, hipMemcpyHostToDevice, r->stream));
    return launch_program(r, prog, r->prog);
}

}  // namespace

// The steps of a fused apply on 2^ns (>= 2^kMinFused) amplitudes; returns
// the tile size.  max_qubits = 0 and no dense phases from kAutoTileQubits:
// the tile the run-time model picks; otherwise max_qubits (0: the default)
// clamped to what the precision's LDS tile and the buffer allow.
unsigned compile_fused(const qvnt_gate* g, size_t n, unsigned ns, bool fp64, uint32_t max_qubits, uint32_t dense_min,
                       std::vector<Step>& steps) {
    const bool single_plain = ns >= kSinglePlainQubits;
    if (!max_qubits && dense_min == 0 && ns >= kAutoTileQubits)
        return plan_auto(g, n, ns, fp64, steps, single_plain, true);
    const unsigned cap = max_tile(fp64);
    unsigned tq = max_qubits ? max_qubits : kDefaultTile;
    if (tq > cap) tq = cap;
    if (tq < (unsigned)kMinFused) tq = kMinFused;
    if (tq > ns) tq = ns;
    plan(g, n, ns, tq, steps, dense_min, single_plain, true, fp64 ? 16 : 8);
    return tq;
}

void fused_plan_stats(const qvnt_gate* g, size_t n, unsigned ns, bool fp64, uint32_t max_qubits, uint32_t dense_min,
                      double* out) {
    out[0] = out[1] = out[2] = out[3] = 0.0;
    if (ns < (unsigned)kMinFused) {  // the plain kernels, one launch per gate
        out[0] = (double)n;
        return;
    }
    std::vector<Step> steps;
    out[1] = compile_fused(g, n, ns, fp64, max_qubits, dense_min, steps);
    for (const Step& st : steps) {
        if (st.plain) {
            out[0] += 1.0;
            continue;
        }
        out[0] += (double)st.prog.passes.size();
        out[2] += (double)program_cost(st.prog);
        for (const FPhase& ph : st.prog.phases) out[3] += ph.dense;
    }
}

int apply_fused(qvnt_reg* r, const qvnt_gate* g, size_t n, uint32_t max_qubits, uint32_t* passes) {
    if (passes) *passes = 0;
    if (r->ns < (unsigned)kMinFused) {
        for (size_t i = 0; i < n; ++i)
            if (int rc = launch_gate(r, g[i])) return rc;
        if (passes) *passes = (uint32_t)n;
        return QVNT_OK;
    }
    std::vector<Step> steps;
    compile_fused(g, n, r->ns, r->prec == QVNT_F64, max_qubits, r->dense_min, steps);
    uint32_t count = 0;
    for (const Step& st : steps) {
        if (st.plain) {
            if (int rc = launch_gate(r, st.gate)) return rc;
            ++count;
        } else {
            if (int rc = run_program(r, st.prog)) return rc;
            count += (uint32_t)st.prog.passes.size();
        }
    }
    if (passes) *passes = count;
    return QVNT_OK;
}

}  // namespace qvnt
