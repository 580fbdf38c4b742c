// The kernel of the plain form's runs (runs.hpp): one launch applies up to
// kMaxOps SingleOps, in queue order, to tiles of 2^t amplitudes.
//
// One kernel per SingleOp is bound by HBM above 20 qubits (one read and one
// write of the state each, 5.4 ms at 30 qubits FP64) and by the launches
// below (4-6 us each from one to the next).  A run reads and writes the
// state once for all its SingleOps, which leaves FP64 arithmetic beside the
// HBM stream: a rz, rx or ry is 6 operations an amplitude.  Measured, one
// whole call each with reset and readout, before (a kernel per SingleOp) and
// with runs:
//   30-qubit brickwork layer, FP64, 106 SingleOps   579 ms    41 ms (runs alone 31)
//   27-qubit Ising step, FP32, 135 SingleOps         45 ms   7.4 ms
//   15-qubit circuit, FP32, 300 gates               1.4 ms  0.26 ms
//   10-qubit QFT with register and readback         238 us    41 us
//
// From 22 qubits 256 threads hold a tile of 2^12 FP64 amplitudes in
// registers, 16 each (2^13 in FP32: 512 threads); LDS only carries them from
// one phase's layout to the next, one component at a time (32 KiB), so four
// blocks fit a CU and, at 120 registers, four waves a SIMD: one block's HBM
// accesses overlap the others' arithmetic, which bounds it: 30 qubits, a third
// of a brickwork layer, 4.85e9 vector instructions on 1024 SIMDs in 10.8 ms,
// four cycles each, 73 % of the cycles at 2.4 GHz.  Below, 8 amplitudes a thread and
// smaller tiles (runs.hpp): there the time is each op's latency -- its load
// from LDS, the dispatch, 16 or 8 amplitudes' dependent FP64 -- some 0.3 us.
// The program comes with the launch as kernel arguments: no upload, no
// device memory.
#pragma clang fp contract(off)

#include "reg.hpp"
#include "runs_ops.hpp"

namespace qvnt {
namespace {

using namespace runs;

using tile::exchange;
using tile::layout_of;
using tile::spread;
template <int B>
using Layout = tile::Layout<B>;

// the B (at most 4) positions packed in a word, one byte each
template <int B>
__device__ __forceinline__ void unpack(uint32_t w, uint32_t* p) {
#pragma unroll
    for (int j = 0; j < B; ++j) p[j] = (w >> (8 * j)) & 63u;
}
__device__ __forceinline__ uint32_t word(const uint8_t* p) { return *reinterpret_cast<const uint32_t*>(p); }

// What the bits of a thread's register index add to its global index
// (uniform), from their positions.  Computed where it is used: held across
// the tiles, the offsets of all registers spill scalar registers.
template <int B>
struct Steps {
    uint64_t step[B];
    __device__ __forceinline__ explicit Steps(uint32_t w) {
        asm volatile("" : "+s"(w));
        uint32_t p[B];
        unpack<B>(w, p);
#pragma unroll
        for (int j = 0; j < B; ++j) step[j] = 1ull << p[j];
    }
    __device__ __forceinline__ uint64_t operator()(int i) const {
        uint64_t o = 0;
#pragma unroll
        for (int j = 0; j < B; ++j)
            if (i >> j & 1) o |= step[j];
        return o;
    }
};

constexpr unsigned max_threads(int B) { return 1u << (kMaxTile - B); }

template <class R, int B>
__global__ __launch_bounds__(max_threads(B)) __attribute__((amdgpu_waves_per_eu(4, 4)))
void k_run(cplx<R>* __restrict__ psi, uint32_t tiles, Run run) {
    constexpr int N = 1 << B;
    constexpr uint32_t kFull = (1u << N) - 1u;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ __align__(16) ROp ops[kMaxOps + 2];
    __shared__ __align__(16) ROut outer[kMaxOps];
    __shared__ __align__(16) RPhase phases[kMaxPhases];
    R* lds = reinterpret_cast<R*>(smem);
    const uint32_t tid = threadIdx.x, nth = blockDim.x, t = run.t;
    for (uint32_t k = tid; k < run.nops; k += nth) {
        ops[k] = run.op[k];
        outer[k] = run.outer[k];
    }
    for (uint32_t k = tid; k < run.nphases; k += nth) phases[k] = run.phase[k];

    // The tile's bits and this thread's offsets where the tile is read and
    // written.  The positions come as four words: a byte load for each, one
    // after the other from the launch's argument memory, took 2 us a launch
    // at 10 qubits and 4 us at 28.
    uint32_t tw[4], in[B], out[B];
#pragma unroll
    for (int k = 0; k < 4; ++k) tw[k] = word(run.tpos + 4 * k);
    const auto tp = [&](int k) { return (tw[k >> 2] >> (8 * (k & 3))) & 63u; };
    unpack<B>(word(run.in), in);
    unpack<B>(word(run.out), out);
    const uint32_t lin = spread<B>(tid, in), lout = spread<B>(tid, out);
    uint64_t gin = 0, gout = 0;
#pragma unroll
    for (int k = 0; k < (int)kMaxTile; ++k) {
        // (bits from t up are zero in lin and lout)
        gin |= (uint64_t)((lin >> k) & 1u) << tp(k);
        gout |= (uint64_t)((lout >> k) & 1u) << tp(k);
    }

    // XCD x (the blocks b with b mod 8 = x) walks its own contiguous eighth
    // of the tiles
    const uint32_t G = gridDim.x, b = blockIdx.x;
    const bool by_xcd = ((G | tiles) & 7u) == 0;
    uint32_t n = by_xcd ? (b & 7u) * (tiles >> 3) + (b >> 3) : b;
    const uint32_t stop = by_xcd ? ((b & 7u) + 1u) * (tiles >> 3) : tiles, step = by_xcd ? G >> 3 : G;
    for (; n < stop; n += step) {
        uint64_t tile = n;
        asm volatile("" : "+s"(tw[0]), "+s"(tw[1]), "+s"(tw[2]), "+s"(tw[3]));
#pragma unroll
        for (int k = 0; k < (int)kMaxTile; ++k) {
            if (k < (int)t) {  // uniform
                const uint64_t lo = tile & ((1ull << tp(k)) - 1u);
                tile = ((tile ^ lo) << 1) | lo;
            }
        }
        cplx<R> v[N];
        {
            const cplx<R>* p = psi + (tile | gin);
            const Steps<B> step_in(word(run.gin));
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const cplx<R>* q = p + step_in(i);
                v[i] = cplx<R>{__builtin_nontemporal_load(&q->re), __builtin_nontemporal_load(&q->im)};
            }
        }
        // (the barrier also ends the previous tile's reads of LDS)
        __syncthreads();
        for (uint32_t k = tid; k < run.nops; k += nth) {
            const ROut q = outer[k];
            ops[k].live = ((tile & q.ctrl) == q.ctrl ? 1u : 0u) | ((dpopc(tile & q.parity) & 1u) << 1);
        }
        __syncthreads();

        uint32_t tb = lin;
        Layout<B> cur = layout_of<B>(tb, in);
        uint32_t o = 0;
        // (one op ahead: its load from LDS runs beside the op before)
        ROp next = ops[0];
        for (uint32_t ph = 0; ph < run.nphases; ++ph) {
            const uint32_t w = __builtin_amdgcn_readfirstlane(word(phases[ph].rpos));
            const uint32_t end = __builtin_amdgcn_readfirstlane((uint32_t)phases[ph].op_end);
            if (ph != 0 || w != word(run.in)) {
                uint32_t pos[B];
                unpack<B>(w, pos);
                tb = spread<B>(tid, pos);
                const Layout<B> to = layout_of<B>(tb, pos);
                exchange<B>(v, lds, cur, to);
                cur = to;
            }
            while (o < end) {
                const uint32_t cp = __builtin_amdgcn_readfirstlane(next.code_pc), lb = __builtin_amdgcn_readfirstlane(next.lbits),
                               live = __builtin_amdgcn_readfirstlane(next.live);
                const double re = next.re, im = next.im;
                next = ops[++o];
                // no divergent branch around the op: a wave whose lanes all
                // satisfy the controls runs it whole, one with none skips
                // it, and only a mixed one selects per lane
                const uint32_t lc = lb & 0xFFFFu, pc = cp & 0xFFFFu;
                const bool on = (tb & lc) == lc;
                const bool odd = ((dpopc(tb & (lb >> 16)) ^ (live >> 1)) & 1u) != 0;
                const bool all = __builtin_amdgcn_ballot_w64(!on) == 0;
                if ((live & 1u) && __builtin_amdgcn_ballot_w64(on) != 0) {
                    if (all && pc == kFull) apply_op<B, false>(v, cp >> 16, pc, true, odd, re, im);
                    else apply_op<B, true>(v, cp >> 16, pc, on, odd, re, im);
                }
            }
        }
        if (word(run.out) != word(run.phase[run.nphases - 1].rpos)) exchange<B>(v, lds, cur, layout_of<B>(lout, out));
        {
            cplx<R>* p = psi + (tile | gout);
            const Steps<B> step_out(word(run.gout));
#pragma unroll
            for (int i = 0; i < N; ++i) {
                cplx<R>* q = p + step_out(i);
                __builtin_nontemporal_store(v[i].re, &q->re);
                __builtin_nontemporal_store(v[i].im, &q->im);
            }
        }
    }
}

// Each block walks several tiles of a large state, so its copy of the
// program is read once.
constexpr uint64_t kMaxBlocks = 4096;

template <class R, int B>
int launch_run(qvnt_reg* r, const Run& run) {
    const uint64_t tiles = r->len >> run.t;
    const dim3 grid((unsigned)(tiles < kMaxBlocks ? tiles : kMaxBlocks)), block(1u << (run.t - B));
    Timed t(r, QVNT_K_FUSED, 2.0 * (double)r->amp_bytes() * (double)r->len);
    hipLaunchKernelGGL((k_run<R, B>), grid, block, sizeof(R) << run.t, r->stream, static_cast<cplx<R>*>(r->psi), (uint32_t)tiles, run);
    QVNT_HIP(hipGetLastError());
    return QVNT_OK;
}

int launch_run(qvnt_reg* r, const Run& run) {
    if (r->prec == QVNT_F64) return run.regs == 3 ? launch_run<double, 3>(r, run) : launch_run<double, 4>(r, run);
    return run.regs == 3 ? launch_run<float, 3>(r, run) : launch_run<float, 4>(r, run);
}

}  // namespace

int apply_plain(qvnt_reg* r, const qvnt_gate* g, size_t n) {
    static thread_local Run run;
    const bool fp64 = r->prec == QVNT_F64;
    for (size_t pos = 0;;) {
        const Step s = next(g, n, &pos, r->ns, fp64, reg_bits(r->ns), max_tile(r->ns, fp64), &run);
        if (s.kind == Kind::Done) return QVNT_OK;
        const int rc = s.kind == Kind::Single ? launch_gate(r, g[s.from]) : launch_run(r, run);
        if (rc) return rc;
    }
}

}  // namespace qvnt
