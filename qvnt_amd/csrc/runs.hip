// The kernel of the plain form's runs (runs.hpp): one launch applies up to
// kMaxOps SingleOps, in queue order, to tiles of 2^t amplitudes.
//
// One kernel per SingleOp is bound by HBM above 20 qubits (one read and one
// write of the state each, 5.4 ms at 30 qubits FP64) and by the launches
// below (4-6 us each from one to the next).  A run reads and writes the
// state once for all its SingleOps, which leaves FP64 arithmetic beside the
// HBM stream: a rz, rx or ry is 6 operations an amplitude.  Measured, one
// call each, before (a kernel per SingleOp) and with runs:
//   30-qubit brickwork layer, FP64, 106 SingleOps   576 ms    36 ms
//   27-qubit Ising step, FP32, 135 SingleOps         45 ms   7.6 ms
//   15-qubit circuit, FP32, 300 gates               1.4 ms   0.4 ms
//   10-qubit QFT with register and readback         241 us    60 us
//
// 256 threads hold a tile of 2^12 FP64 amplitudes in registers, 16 each
// (2^13 in FP32: 512 threads); LDS only carries them from one phase's layout
// to the next, one component at a time (32 KiB), so four blocks fit a CU
// and, at 110 registers, four waves a SIMD: one block's HBM accesses overlap
// the others' arithmetic.  The program comes with the launch as kernel
// arguments: no upload, no device memory.
#pragma clang fp contract(off)

#include "reg.hpp"
#include "runs_ops.hpp"

namespace qvnt {
namespace {

using namespace runs;

constexpr unsigned kMaxThreads = 1u << (kMaxTile - kRegBits);

// LDS offset of local element e: bits 4.. folded onto the low bits, so that
// lanes which differ in bits 4..8 fall on different banks.  XOR-linear:
// offsets of disjoint bits combine by XOR.
__device__ __forceinline__ uint32_t swz(uint32_t e) { return e ^ (e >> 4); }

// zeros inserted into x at the ascending positions p
__device__ __forceinline__ uint32_t spread(uint32_t x, const uint8_t* p) {
#pragma unroll
    for (unsigned j = 0; j < kRegBits; ++j) {
        const uint32_t lo = x & ((1u << p[j]) - 1u);
        x = ((x ^ lo) << 1) | lo;
    }
    return x;
}

// A register layout: which local bits the 16 registers of a thread run over.
struct Layout {
    uint32_t tb;              // local index of register 0
    uint32_t s[kRegBits];     // swizzled offsets of the register bits (uniform)
};
__device__ __forceinline__ Layout layout_of(uint32_t tid, const uint8_t* p) {
    Layout l;
    l.tb = spread(tid, p);
#pragma unroll
    for (unsigned j = 0; j < kRegBits; ++j) l.s[j] = __builtin_amdgcn_readfirstlane(swz(1u << p[j]));
    return l;
}
__device__ __forceinline__ uint32_t at(const Layout& l, int i) {
    uint32_t e = swz(l.tb);
#pragma unroll
    for (unsigned j = 0; j < kRegBits; ++j)
        if (i >> j & 1) e ^= l.s[j];
    return e;
}

// Registers from one layout to another, through LDS, one component after the
// other: half the LDS of a whole tile, so twice the blocks on a CU.  A
// thread writes what it read last (the elements of its own layout), so the
// first write needs no barrier.
template <class R>
__device__ __forceinline__ void exchange(cplx<R>* v, R* lds, const Layout& from, const Layout& to) {
#pragma unroll
    for (int i = 0; i < (int)kRegs; ++i) lds[at(from, i)] = v[i].re;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (int)kRegs; ++i) v[i].re = lds[at(to, i)];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (int)kRegs; ++i) lds[at(from, i)] = v[i].im;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (int)kRegs; ++i) v[i].im = lds[at(to, i)];
}

__device__ __forceinline__ bool same(const uint8_t* a, const uint8_t* b) {
    return *reinterpret_cast<const uint32_t*>(a) == *reinterpret_cast<const uint32_t*>(b);
}

template <class R>
__global__ __launch_bounds__(kMaxThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
void k_run(cplx<R>* __restrict__ psi, uint32_t tiles, Run run) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ __align__(16) ROp ops[kMaxOps + 2];
    __shared__ __align__(16) RPhase phases[kMaxPhases];
    R* lds = reinterpret_cast<R*>(smem);
    const uint32_t tid = threadIdx.x, nth = blockDim.x;
    for (uint32_t k = tid; k < run.nops; k += nth) ops[k] = run.op[k];
    for (uint32_t k = tid; k < run.nphases; k += nth) phases[k] = run.phase[k];

    // global offsets of this thread's bits where the tile is read and written
    const uint32_t lin = spread(tid, run.in), lout = spread(tid, run.out);
    uint64_t gin = 0, gout = 0;
    for (uint32_t k = 0; k < run.t; ++k) {
        gin |= (uint64_t)((lin >> k) & 1u) << run.tpos[k];
        gout |= (uint64_t)((lout >> k) & 1u) << run.tpos[k];
    }

    // XCD x (the blocks b with b mod 8 = x) walks its own contiguous eighth
    // of the tiles
    const uint32_t G = gridDim.x, b = blockIdx.x;
    const bool by_xcd = ((G | tiles) & 7u) == 0;
    uint32_t n = by_xcd ? (b & 7u) * (tiles >> 3) + (b >> 3) : b;
    const uint32_t stop = by_xcd ? ((b & 7u) + 1u) * (tiles >> 3) : tiles, step = by_xcd ? G >> 3 : G;
    for (; n < stop; n += step) {
        uint64_t tile = n;
        for (uint32_t k = 0; k < run.t; ++k) {
            const uint64_t lo = tile & ((1ull << run.tpos[k]) - 1u);
            tile = ((tile ^ lo) << 1) | lo;
        }
        cplx<R> v[kRegs];
        {
            const cplx<R>* p = psi + (tile | gin);
#pragma unroll
            for (int i = 0; i < (int)kRegs; ++i) {
                uint64_t off = 0;
#pragma unroll
                for (unsigned j = 0; j < kRegBits; ++j)
                    if (i >> j & 1) off |= 1ull << run.tpos[run.in[j]];
                v[i] = cplx<R>{__builtin_nontemporal_load(&p[off].re), __builtin_nontemporal_load(&p[off].im)};
            }
        }
        // (the barrier also ends the previous tile's reads of LDS)
        __syncthreads();
        for (uint32_t k = tid; k < run.nops; k += nth) {
            const ROut q = run.outer[k];
            ops[k].live = ((tile & q.ctrl) == q.ctrl ? 1u : 0u) | ((dpopc(tile & q.parity) & 1u) << 1);
        }
        __syncthreads();

        Layout cur = layout_of(tid, run.in);
        uint32_t o = 0;
        for (uint32_t ph = 0; ph < run.nphases; ++ph) {
            const RPhase p = phases[ph];
            if (!(ph == 0 && same(run.in, run.phase[0].rpos))) {
                const Layout to = layout_of(tid, p.rpos);
                exchange(v, lds, cur, to);
                cur = to;
            }
            const uint32_t end = __builtin_amdgcn_readfirstlane((uint32_t)p.op_end);
            while (o < end) {
                const ROp& op = ops[o];
                const uint32_t cp = __builtin_amdgcn_readfirstlane(op.code_pc), lb = __builtin_amdgcn_readfirstlane(op.lbits),
                               live = __builtin_amdgcn_readfirstlane(op.live);
                // no divergent branch around the op: a wave whose lanes all
                // satisfy the controls runs it whole, one with none skips
                // it, and only a mixed one selects per lane
                const uint32_t lc = lb & 0xFFFFu, pc = cp & 0xFFFFu;
                const bool on = (cur.tb & lc) == lc;
                const bool odd = ((dpopc(cur.tb & (lb >> 16)) ^ (live >> 1)) & 1u) != 0;
                const bool all = __builtin_amdgcn_ballot_w64(!on) == 0;
                if ((live & 1u) && __builtin_amdgcn_ballot_w64(on) != 0) {
                    if (all && pc == 0xFFFFu) apply_op<false>(v, cp >> 16, pc, true, odd, op.re, op.im);
                    else apply_op<true>(v, cp >> 16, pc, on, odd, op.re, op.im);
                }
                ++o;
            }
        }
        if (!same(run.out, run.phase[run.nphases - 1].rpos)) exchange(v, lds, cur, layout_of(tid, run.out));
        {
            cplx<R>* p = psi + (tile | gout);
#pragma unroll
            for (int i = 0; i < (int)kRegs; ++i) {
                uint64_t off = 0;
#pragma unroll
                for (unsigned j = 0; j < kRegBits; ++j)
                    if (i >> j & 1) off |= 1ull << run.tpos[run.out[j]];
                __builtin_nontemporal_store(v[i].re, &p[off].re);
                __builtin_nontemporal_store(v[i].im, &p[off].im);
            }
        }
    }
}

// Each block walks several tiles of a large state, so its copy of the
// program is read once.
constexpr uint64_t kMaxBlocks = 4096;

template <class R>
int launch_run(qvnt_reg* r, const Run& run) {
    const uint64_t tiles = r->len >> run.t;
    const dim3 grid((unsigned)(tiles < kMaxBlocks ? tiles : kMaxBlocks)), block(1u << (run.t - kRegBits));
    Timed t(r, QVNT_K_FUSED, 2.0 * (double)r->amp_bytes() * (double)r->len);
    hipLaunchKernelGGL(k_run<R>, grid, block, sizeof(R) << run.t, r->stream, static_cast<cplx<R>*>(r->psi), (uint32_t)tiles, run);
    QVNT_HIP(hipGetLastError());
    return QVNT_OK;
}

}  // namespace

int apply_plain(qvnt_reg* r, const qvnt_gate* g, size_t n) {
    static thread_local Run run;
    for (size_t pos = 0;;) {
        const Step s = next(g, n, &pos, r->ns, r->prec == QVNT_F64, &run);
        if (s.kind == Kind::Done) return QVNT_OK;
        const int rc = s.kind == Kind::Single ? launch_gate(r, g[s.from])
                       : r->prec == QVNT_F64  ? launch_run<double>(r, run)
                                              : launch_run<float>(r, run);
        if (rc) return rc;
    }
}

}  // namespace qvnt
