// A tile of amplitudes held in registers, 2^B per thread, and its way through
// LDS from one register layout to the next: shared by the kernels that apply
// several gates per pass (runs.hip, fused.hip).
#pragma once

#include "device.hpp"

namespace qvnt {
namespace tile {

// LDS offset of local element e: bits 4.. folded onto the low bits, so that
// lanes which differ in bits 4..8 fall on different banks.  XOR-linear:
// offsets of disjoint bits combine by XOR.
__device__ __forceinline__ uint32_t swz(uint32_t e) { return e ^ (e >> 4); }

// zeros inserted into x at the ascending positions p
template <int B, class P>
__device__ __forceinline__ uint32_t spread(uint32_t x, const P* p) {
#pragma unroll
    for (int j = 0; j < B; ++j) {
        const uint32_t lo = x & ((1u << p[j]) - 1u);
        x = ((x ^ lo) << 1) | lo;
    }
    return x;
}

// A register layout: LDS offset of a thread's register 0, and what each bit
// of the register index adds to it (uniform).
template <int B>
struct Layout {
    uint32_t base;
    uint32_t bit[B];
    __device__ __forceinline__ uint32_t operator()(int i) const {
        uint32_t e = base;
#pragma unroll
        for (int j = 0; j < B; ++j)
            if (i >> j & 1) e ^= bit[j];
        return e;
    }
};
// registers over the local bits p, the thread's bits around them; tb: the
// local index of register 0
template <int B, class P>
__device__ __forceinline__ Layout<B> layout_of(uint32_t tb, const P* p) {
    Layout<B> l;
    l.base = swz(tb);
#pragma unroll
    for (int j = 0; j < B; ++j) l.bit[j] = __builtin_amdgcn_readfirstlane(swz(1u << p[j]));
    return l;
}

// Registers from one layout to another, one component after the other: half
// the LDS of a whole tile, so twice the blocks on a CU.  A thread writes the
// elements it read last, so between exchanges of one tile the first write
// needs no barrier; the first exchange of the block's next tile does.
// (With LDS for both components and one barrier instead of three no size ran
// faster, from 10 to 31 qubits: the barriers are not what bounds it.)
template <int B, class R, class From, class To>
__device__ __forceinline__ void exchange(cplx<R>* v, R* lds, const From& from, const To& to) {
#pragma unroll
    for (int i = 0; i < 1 << B; ++i) lds[from(i)] = v[i].re;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 1 << B; ++i) v[i].re = lds[to(i)];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 1 << B; ++i) lds[from(i)] = v[i].im;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 1 << B; ++i) v[i].im = lds[to(i)];
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

}  // namespace tile
}  // namespace qvnt
