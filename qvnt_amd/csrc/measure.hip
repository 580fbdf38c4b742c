// Measurement: QReg::get_absolute / get_probabilities / measure_mask
// (src/register/quant.rs:434-507) on the device.
//
// The reference sums |psi|^2 sequentially, builds rand's WeightedIndex
// cumulative array on the host thread and draws from an unseeded thread_rng
// (quant.rs:437-442, 496-497).  Its draw cannot be reproduced, so a
// deterministic contract replaces it (the CPU oracle implements the same):
//   w_i = re*re + im*im in FP64 (no FMA), node(0,j) = w_j,
//   node(l,j) = node(l-1,2j) + node(l-1,2j+1)        (pairwise tree),
//   draw: x = u * node(top,0); from the root, with children (L, R), go left
//   iff x < L or R == 0, else x -= L and go right; the leaf reached is r.
// Every eleventh level is stored (O(2^n / 2^11) doubles); a draw makes the
// levels between again on its way down.  FP32 registers are
// reduced, searched and rescaled in FP64 as well.
#pragma clang fp contract(off)

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "device.hpp"
#include "reg.hpp"

namespace qvnt {
namespace {

constexpr int kBlock = 256;
constexpr unsigned kLeafLog = 11;          // leaves per stored bottom node

template <class R>
__device__ __forceinline__ double weight(cplx<R> p) {
    const double re = (double)p.re, im = (double)p.im;
    return re * re + im * im;
}

// A dispatch carries its size in work-items as a 32-bit number: grids are
// capped at kMaxGrid blocks and kernels stride over their work.
constexpr uint64_t kMaxGrid = 1u << 20;
constexpr unsigned kWave = 64;
constexpr unsigned kBlockWaves = kBlock / kWave;
constexpr uint64_t kSpreadNodes = 1024;  // 18 qubits: k_leaf 5.2 us in blocks of four waves, 4.5 in blocks of one

// Values of the tree's next lower stored level, or the leaves.
struct Nodes {
    const double* p;
    __device__ __forceinline__ double operator()(uint64_t k) const { return p[k]; }
};
template <class R>
struct Leaves {
    const cplx<R>* p;
    __device__ __forceinline__ double operator()(uint64_t k) const { return weight(p[k]); }
};

// The value of lane ^ M.  Within a row of 16 lanes a DPP move where one does
// it, else an LDS swizzle; every lane of the wave is active.
template <int M>
__device__ __forceinline__ int xor_lane(int v) {
    if constexpr (M == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);         // quad_perm 1 0 3 2
    else if constexpr (M == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);    // quad_perm 2 3 0 1
    else if constexpr (M == 8) return __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, true);   // row_ror 8
    else if constexpr (M < 32) return __builtin_amdgcn_ds_swizzle(v, (M << 10) | 0x1F);
    else return __shfl_xor(v, M);
}
template <int M>
__device__ __forceinline__ double xor_lane(double v) {
    return __hiloint2double(xor_lane<M>(__double2hiint(v)), xor_lane<M>(__double2loint(v)));
}

// Pairwise tree of 64 consecutive values per register, 2^LC registers: at
// step S lanes whose bit S is 0 go on with the even registers and the others
// with the odd ones, so each step halves the registers and takes one
// exchange for two sums.  At the end lane l holds one value, the sum of 2^LC
// consecutive values: group l >> LC of chunk l & (2^LC - 1).  (All sums of
// all lanes, six exchanges a register, took k_leaf 4.2 ms in FP32 at 31
// qubits, 16 GiB: bound by LDS, not by HBM.)
template <int LC, int S = 0>
__device__ __forceinline__ void fold(double* a) {
    if constexpr (S < LC) {
        const bool odd = (threadIdx.x >> S) & 1u;
#pragma unroll
        for (int k = 0; k < 1 << (LC - S - 1); ++k) {
            const double keep = odd ? a[2 * k + 1] : a[2 * k], give = odd ? a[2 * k] : a[2 * k + 1];
            a[k] = keep + xor_lane<1 << S>(give);
        }
        fold<LC, S + 1>(a);
    }
}

// The rest of the tree: s[d], d = 0 .. 6: this lane's node d levels above
// fold's (lane bit (LC + d) % 6 pairs level d).
template <int LC, int D = 0>
__device__ __forceinline__ void rise(double* s) {
    if constexpr (D < 6) {
        s[D + 1] = s[D] + xor_lane<1 << ((LC + D) % 6)>(s[D]);
        rise<LC, D + 1>(s);
    }
}
// 2^(6 + LC) values (LC 0: 2^lg of them, lg <= 6)
template <int LC, class F>
__device__ __forceinline__ void levels(const F& node, uint64_t base, uint32_t lg, double* s) {
    const uint32_t lane = threadIdx.x & (kWave - 1u);
    double a[1 << LC];
#pragma unroll
    for (int c = 0; c < 1 << LC; ++c) a[c] = LC > 0 || lane < (1u << lg) ? node(base + (uint64_t)c * kWave + lane) : 0.0;
    fold<LC>(a);
    s[0] = a[0];
    rise<LC>(s);
}

// One wave per node of the lowest stored level: 2^11 leaves, all in flight
// at once, and no barrier.  Bound by HBM: 16 GiB in 2.8 ms, 6.1 TB/s, in FP64
// and FP32.
template <class R>
__global__ __launch_bounds__(kBlock) void k_leaf(const cplx<R>* __restrict__ psi, uint64_t nleaves, double* __restrict__ out) {
    const uint32_t lane = threadIdx.x & (kWave - 1u);
    const uint32_t waves = blockDim.x / kWave;
    for (uint64_t node = (uint64_t)blockIdx.x * waves + threadIdx.x / kWave; node < nleaves; node += (uint64_t)gridDim.x * waves) {
        double s[7];
        if constexpr (sizeof(R) == 8) {
            levels<5>(Leaves<R>{psi}, node << kLeafLog, kLeafLog, s);
        } else {
            // two leaves a load
            const float4* p = reinterpret_cast<const float4*>(psi + (node << kLeafLog)) + lane;
            double a[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                const float4 q = p[c * (int)kWave];
                a[c] = weight(c32{q.x, q.y}) + weight(c32{q.z, q.w});
            }
            fold<4>(a);
            s[0] = a[0];
            rise<4>(s);
        }
        if (lane == 0) out[node] = s[6];
    }
}

// A stored level from the one 2^11 below it, one wave per node.
__global__ __launch_bounds__(kBlock) void k_upper(const double* __restrict__ in, uint64_t n, double* __restrict__ out) {
    const uint64_t node = (uint64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (node >= n) return;  // uniform over the wave
    double s[7];
    levels<5>(Nodes{in}, node << kLeafLog, kLeafLog, s);
    if ((threadIdx.x & (kWave - 1u)) == 0) out[node] = s[6];
}

struct TreeInfo {
    uint32_t top;      // log2(count)
    uint32_t lb;       // lowest stored level, min(top, 11)
    uint64_t off[64];  // offset of level l in the tree array; levels 11, 22, 33 below the top are stored
};
// The highest stored level below the top (0: the leaves).
__host__ __device__ inline uint32_t top_stage(uint32_t top) { return top ? (top - 1u) / kLeafLog * kLeafLog : 0u; }

__device__ __forceinline__ double lane_value(double v, uint32_t lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane), __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// A draw's position: x, what is left of u * total in the node reached.
struct Draw {
    double u, x, total;
    bool first;
};

// Descends the tree over 2^lg values from node(base) (LC 0: lg <= 6, else lg
// = 6 + LC): the offset of the value reached.  Wave-uniform.
template <int LC, class F>
__device__ __forceinline__ uint32_t descend(const F& node, uint64_t base, uint32_t lg, Draw& d) {
    double s[7];
    levels<LC>(node, base, lg, s);
    const uint32_t n = LC ? 6u : lg;
    if (d.first) {
        double root = s[6];
        if (LC == 0) {
#pragma unroll
            for (int l = 0; l < 6; ++l) root = n == (uint32_t)l ? s[l] : root;
        }
        d.total = lane_value(root, 0);
        d.x = d.u * d.total;
        d.first = false;
    }
    uint32_t m = 0;
#pragma unroll
    for (int l = 5; l >= 0; --l) {
        if ((uint32_t)l >= n) continue;  // uniform
        // the lane that holds node q of level l
        const auto at = [&](uint32_t q) {
            const uint32_t i = q << l;
            return (uint32_t)__builtin_amdgcn_readfirstlane(((i >> (6 - LC)) | (i << LC)) & (kWave - 1u));
        };
        const double L = lane_value(s[l], at(2 * m)), R = lane_value(s[l], at(2 * m + 1));
        const bool left = d.x < L || R == 0.0;
        d.x = left ? d.x : d.x - L;
        m = 2 * m + (left ? 0u : 1u);
    }
    if constexpr (LC > 0) {
        const uint32_t first = m << LC;
        return first + descend<0>(node, base + first, LC, d);
    } else {
        return m;
    }
}
template <class F>
__device__ __forceinline__ uint32_t descend_any(const F& node, uint64_t base, uint32_t lg, Draw& d) {
    switch (lg) {  // uniform
    case 7: return descend<1>(node, base, lg, d);
    case 8: return descend<2>(node, base, lg, d);
    case 9: return descend<3>(node, base, lg, d);
    case 10: return descend<4>(node, base, lg, d);
    case 11: return descend<5>(node, base, lg, d);
    default: return descend<0>(node, base, lg, d);
    }
}

// One draw per wave: down the stored levels, 2^11 nodes at a time, then the
// leaves of the node reached.  The sums of both are made again in the wave's
// registers; no barrier, and no chain of loads from one level to the next.
// Draw k is u[k], or u0 when u is null (one draw, passed by value: no copy to
// the device before the launch).  1024 draws, FP64: 18 qubits 9.1 us with a block
// per draw and its levels in LDS, 6.0 now; 20 qubits 13.0 and 11.0; 30 qubits
// 20 and 17.
template <class R>
__global__ __launch_bounds__(kBlock) void k_sample(const cplx<R>* __restrict__ psi, const double* __restrict__ tree,
                                                   TreeInfo info, const double* __restrict__ u, double u0, uint32_t shots,
                                                   uint64_t* __restrict__ out, double* __restrict__ total) {
    const uint32_t shot = __builtin_amdgcn_readfirstlane(blockIdx.x * kBlockWaves + threadIdx.x / kWave);
    if (shot >= shots) return;
    Draw d{u ? u[shot] : u0, 0.0, 0.0, true};
    uint64_t j = 0;
    uint32_t l = info.top;
    for (uint32_t to = top_stage(info.top); to >= kLeafLog; to -= kLeafLog) {
        j <<= l - to;
        j += descend_any(Nodes{tree + info.off[to]}, j, l - to, d);
        l = to;
    }
    j <<= l;
    j += descend_any(Leaves<R>{psi}, j, l, d);
    if ((threadIdx.x & (kWave - 1u)) == 0) {
        out[shot] = j;
        if (shot == 0) total[0] = d.total;
    }
}

// The root: the sum over the highest stored level, or the leaves.
template <class R>
__global__ __launch_bounds__(kWave) void k_total(const cplx<R>* __restrict__ psi, const double* __restrict__ tree, TreeInfo info,
                                                 double* __restrict__ total) {
    Draw d{0.0, 0.0, 0.0, true};
    const uint32_t from = top_stage(info.top);
    if (from) (void)descend_any(Nodes{tree + info.off[from]}, 0, info.top - from, d);
    else (void)descend_any(Leaves<R>{psi}, 0, info.top, d);
    if (threadIdx.x == 0) total[0] = d.total;
}

// collapse_mask (quant.rs:468-486): zero every amplitude with
// (idx ^ r) & mask != 0; store-only.
template <class R>
__global__ __launch_bounds__(kBlock) void k_collapse(cplx<R>* __restrict__ psi, uint64_t len, uint64_t r, uint64_t mask) {
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < len; i += (uint64_t)gridDim.x * kBlock)
        if ((i ^ r) & mask) psi[i] = cplx<R>{(R)0, (R)0};
}

// Renormalisation of the kept subspace (the bits of `mask` fixed to r's),
// multiplied in FP64.
template <class R>
__global__ __launch_bounds__(kBlock) void k_rescale(cplx<R>* __restrict__ psi, uint64_t groups, Deposit dep, double scale) {
    for (uint64_t t = (uint64_t)blockIdx.x * kBlock + threadIdx.x; t < groups; t += (uint64_t)gridDim.x * kBlock) {
        const uint64_t i = deposit(t, dep);
        const cplx<R> p = psi[i];
        psi[i] = cplx<R>{(R)((double)p.re * scale), (R)((double)p.im * scale)};
    }
}

// get_probabilities (quant.rs:434-454): p_i = |psi_i|^2 * inv.
template <class R>
__global__ __launch_bounds__(kBlock) void k_probs(const cplx<R>* __restrict__ psi, uint64_t n, double inv, double* __restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) out[i] = weight(psi[i]) * inv;
}

// Comparison of two registers in FP64: per block, <a|b> (re, im), |a|^2,
// |b|^2 and max |a_i - b_i| over 4096 amplitudes; the host folds the
// partials in block order.
template <class RA, class RB>
__global__ __launch_bounds__(kBlock) void k_compare(const cplx<RA>* __restrict__ a, const cplx<RB>* __restrict__ b,
                                                    uint64_t len, double* __restrict__ part) {
    double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    const uint64_t base = (uint64_t)blockIdx.x * 4096u;
    for (uint32_t k = threadIdx.x; k < 4096u; k += kBlock) {
        const uint64_t i = base + k;
        if (i >= len) break;
        const double ar = (double)a[i].re, ai = (double)a[i].im, br = (double)b[i].re, bi = (double)b[i].im;
        s[0] += ar * br + ai * bi;   // <a|b> = conj(a) b
        s[1] += ar * bi - ai * br;
        s[2] += ar * ar + ai * ai;
        s[3] += br * br + bi * bi;
        const double dr = ar - br, di = ai - bi;
        s[4] = fmax(s[4], sqrt(dr * dr + di * di));
    }
    __shared__ double sh[5][kBlock];
    for (int q = 0; q < 5; ++q) sh[q][threadIdx.x] = s[q];
    __syncthreads();
    for (unsigned h = kBlock / 2; h > 0; h >>= 1) {
        if (threadIdx.x < h) {
            for (int q = 0; q < 4; ++q) sh[q][threadIdx.x] += sh[q][threadIdx.x + h];
            sh[4][threadIdx.x] = fmax(sh[4][threadIdx.x], sh[4][threadIdx.x + h]);
        }
        __syncthreads();
    }
    if (threadIdx.x < 5) part[(uint64_t)blockIdx.x * 5 + threadIdx.x] = sh[threadIdx.x][0];
}

template <class RA, class RB>
void launch_compare(const void* a, const void* b, uint64_t len, double* part, unsigned blocks, hipStream_t s) {
    hipLaunchKernelGGL((k_compare<RA, RB>), dim3(blocks), dim3(kBlock), 0, s, static_cast<const cplx<RA>*>(a),
                       static_cast<const cplx<RB>*>(b), len, part);
}

unsigned log2u(uint64_t x) { return 63u - (unsigned)__builtin_clzll(x); }

TreeInfo tree_info(uint64_t count) {
    TreeInfo t{};
    t.top = log2u(count);
    t.lb = t.top < kLeafLog ? t.top : kLeafLog;
    uint64_t off = 0;
    for (uint32_t l = t.lb; l <= t.top; ++l) {
        t.off[l] = off;
        off += count >> l;
    }
    return t;
}

// Workspace blocks of a register that owns its memory come from and go
// back to the device's block cache (reg.hip); the register's stream is
// synchronized before a block goes back, so nothing queued still uses it.
int ws_alloc(qvnt_reg* r, void** p, size_t bytes) {
    if (r->owns_memory) return dev_alloc(r->device, p, bytes);
    if (hipMalloc(p, bytes) == hipSuccess) return QVNT_OK;
    (void)hipGetLastError();
    *p = nullptr;
    return QVNT_E_OOM;
}

int ws_release(qvnt_reg* r, void* p, size_t bytes) {
    if (!p) return QVNT_OK;
    if (!r->owns_memory) {
        QVNT_HIP(hipFree(p));
        return QVNT_OK;
    }
    QVNT_HIP(hipStreamSynchronize(r->stream));
    dev_release(r->device, p, bytes);
    return QVNT_OK;
}

int ensure_workspace(qvnt_reg* r, size_t tree_doubles, size_t shots) {
    if (tree_doubles > r->tree_cap) {
        void* old = r->tree;
        const size_t old_bytes = r->tree_cap * sizeof(double);
        r->tree = nullptr;
        r->tree_cap = 0;
        if (int rc = ws_release(r, old, old_bytes)) return rc;
        void* p = nullptr;
        if (ws_alloc(r, &p, tree_doubles * sizeof(double)) != QVNT_OK)
            return fail(QVNT_E_OOM, "device memory for the measurement tree");
        r->tree = static_cast<double*>(p);
        r->tree_cap = tree_doubles;
    }
    if (shots > r->shots_cap || !r->dscratch) {
        const size_t cap = shots < 64 ? 64 : shots;
        // (both blocks were sized by shots_cap; it is cleared before either
        // goes, so a failure below leaves no block recorded at a wrong size)
        void* d_old = r->dscratch;
        void* i_old = r->iscratch;
        const size_t old_cap = r->shots_cap;
        r->dscratch = nullptr;
        r->iscratch = nullptr;
        r->shots_cap = 0;
        if (int rc = ws_release(r, d_old, (old_cap + 1) * sizeof(double))) return rc;
        if (int rc = ws_release(r, i_old, (old_cap + 1) * sizeof(uint64_t))) return rc;
        void* d = nullptr;
        void* i = nullptr;
        if (ws_alloc(r, &d, (cap + 1) * sizeof(double)) != QVNT_OK)
            return fail(QVNT_E_OOM, "device memory for measurement scratch");
        if (ws_alloc(r, &i, (cap + 1) * sizeof(uint64_t)) != QVNT_OK) {
            (void)ws_release(r, d, (cap + 1) * sizeof(double));
            return fail(QVNT_E_OOM, "device memory for measurement scratch");
        }
        r->dscratch = static_cast<double*>(d);
        r->iscratch = static_cast<uint64_t*>(i);
        r->shots_cap = cap;
    }
    return QVNT_OK;
}

// The stored levels of the first `count` weights into `tree` (laid out by
// tree_info(count)); timed: bracket the launches with the register's timing
// events (the allocation-free path passes false: it creates no events, and so
// does the norm, which brackets its last kernel with them).
template <class R>
int build_levels(qvnt_reg* r, double* tree, uint64_t count, const TreeInfo& info, bool timed) {
    if (info.top <= kLeafLog) return QVNT_OK;  // the leaves are the level below the top
    // (few nodes: a wave a block, so that they spread over the CUs)
    const auto threads = [](uint64_t nodes) { return nodes <= kSpreadNodes ? kWave : (unsigned)kBlock; };
    const auto grid = [&](uint64_t nodes) {
        const uint64_t waves = threads(nodes) / kWave, blocks = (nodes + waves - 1) / waves;
        return dim3((unsigned)(blocks < kMaxGrid ? blocks : kMaxGrid));
    };
    Timed t(timed ? r : nullptr, QVNT_K_REDUCE, (double)r->amp_bytes() * (double)count);
    hipLaunchKernelGGL(k_leaf<R>, grid(count >> kLeafLog), dim3(threads(count >> kLeafLog)), 0, r->stream, static_cast<const cplx<R>*>(r->psi),
                       count >> kLeafLog, tree + info.off[kLeafLog]);
    QVNT_HIP(hipGetLastError());
    for (uint32_t l = 2 * kLeafLog; l < info.top; l += kLeafLog) {
        hipLaunchKernelGGL(k_upper, grid(count >> l), dim3(threads(count >> l)), 0, r->stream, (const double*)(tree + info.off[l - kLeafLog]),
                           count >> l, tree + info.off[l]);
        QVNT_HIP(hipGetLastError());
    }
    return QVNT_OK;
}

// Tree levels plus one draw per u_dev[k] (u_dev null: the single draw u0)
// into out_dev, total into total_dev[0]; every pointer is device memory; no
// synchronisation.
int sample_into(qvnt_reg* r, double* tree, uint64_t count, const double* u_dev, double u0, size_t shots,
                uint64_t* out_dev, double* total_dev, bool timed) {
    const TreeInfo info = tree_info(count);
    int rc = r->prec == QVNT_F64 ? build_levels<double>(r, tree, count, info, timed)
                                 : build_levels<float>(r, tree, count, info, timed);
    if (rc) return rc;
    const dim3 grid((unsigned)((shots + kBlockWaves - 1) / kBlockWaves));
    Timed t(timed ? r : nullptr, QVNT_K_OTHER, 0.0);
    if (r->prec == QVNT_F64)
        hipLaunchKernelGGL(k_sample<double>, grid, dim3(kBlock), 0, r->stream, static_cast<const c64*>(r->psi), (const double*)tree,
                           info, u_dev, u0, (uint32_t)shots, out_dev, total_dev);
    else
        hipLaunchKernelGGL(k_sample<float>, grid, dim3(kBlock), 0, r->stream, static_cast<const c32*>(r->psi), (const double*)tree,
                           info, u_dev, u0, (uint32_t)shots, out_dev, total_dev);
    QVNT_HIP(hipGetLastError());
    return QVNT_OK;
}

}  // namespace

// The total goes straight to pinned host memory where a block is at hand
// (HostBlock), else through the tree array and a copy.
int tree_build(qvnt_reg* r, uint64_t count, double* total_out) {
    const TreeInfo info = tree_info(count);
    int rc = ensure_workspace(r, (size_t)(info.off[info.top] + 1), 1);
    if (rc) return rc;
    HostBlock host(r->device, kHostSmall);
    double* total_dev = host.p ? static_cast<double*>(host.p) : r->tree + info.off[info.top];
    hipError_t e = hipSuccess;
    {
        // (one reduction in the statistics: the stored levels, if any, and the root)
        Timed t(r, QVNT_K_REDUCE, (double)r->amp_bytes() * (double)count);
        rc = r->prec == QVNT_F64 ? build_levels<double>(r, r->tree, count, info, false)
                                 : build_levels<float>(r, r->tree, count, info, false);
        if (rc) return rc;
        if (r->prec == QVNT_F64)
            hipLaunchKernelGGL(k_total<double>, dim3(1), dim3(kWave), 0, r->stream, static_cast<const c64*>(r->psi),
                               (const double*)r->tree, info, total_dev);
        else
            hipLaunchKernelGGL(k_total<float>, dim3(1), dim3(kWave), 0, r->stream, static_cast<const c32*>(r->psi),
                               (const double*)r->tree, info, total_dev);
        e = hipGetLastError();
    }
    if (e == hipSuccess && !host.p) e = hipMemcpyAsync(total_out, total_dev, sizeof(double), hipMemcpyDeviceToHost, r->stream);
    const hipError_t end = hipStreamSynchronize(r->stream);
    if (e == hipSuccess) e = end;
    if (e != hipSuccess) {
        host.keep_out();
        return fail(QVNT_E_HIP, std::string("norm: ") + hipGetErrorString(e));
    }
    if (host.p) std::memcpy(total_out, host.p, sizeof(double));
    return QVNT_OK;
}

size_t tree_doubles(uint64_t count) {
    const TreeInfo info = tree_info(count);
    return (size_t)(info.off[info.top] + 1);
}

int sample_launch(qvnt_reg* r, uint64_t count, const double* u_dev, size_t shots, uint64_t* out_dev, double* total_dev) {
    if (tree_doubles(count) > r->tree_cap) return fail(QVNT_E_ARG, "measurement tree workspace too small");
    return sample_into(r, r->tree, count, u_dev, 0.0, shots, out_dev, total_dev, true);
}

// The draws come from, and the outcomes and the total go to, one block of
// pinned host memory that the kernel reads and writes itself, where the draws
// fit one (HostBlock): a copy each way cost more than the draws (1024 shots,
// whole call: 10 qubits 50 us with the copies, 26 without; 17 qubits 49 and
// 33; the norm alone 23 and 12, 27 and 16).  Otherwise the outcomes
// land in iscratch[0, shots) and the total right after them (iscratch holds
// shots_cap + 1 words), so one copy brings both back.  A single draw goes to
// the kernel by value.
int tree_sample(qvnt_reg* r, uint64_t count, const double* u, size_t shots, uint64_t* out, double* total_out) {
    if (shots == 0) return fail(QVNT_E_ARG, "no draws");
    const bool small = (2 * shots + 1) * sizeof(uint64_t) <= kHostSmall;
    HostBlock host(r->device, small ? kHostSmall : 0);
    int rc = ensure_workspace(r, tree_doubles(count), host.p ? 1 : shots);
    if (rc) return rc;
    if (tree_doubles(count) > r->tree_cap) return fail(QVNT_E_ARG, "measurement tree workspace too small");
    if (host.p) {
        uint64_t* words = static_cast<uint64_t*>(host.p);   // outcomes, total, draws
        double* total_dev = reinterpret_cast<double*>(words + shots);
        double* draws = total_dev + 1;
        if (shots > 1) std::memcpy(draws, u, shots * sizeof(double));
        rc = sample_into(r, r->tree, count, shots > 1 ? draws : nullptr, shots > 1 ? 0.0 : u[0], shots, words, total_dev, true);
        const hipError_t e = hipStreamSynchronize(r->stream);
        if (rc == QVNT_OK && e != hipSuccess) rc = fail(QVNT_E_HIP, std::string("draws: ") + hipGetErrorString(e));
        if (rc) {
            host.keep_out();
            return rc;
        }
        std::memcpy(out, words, shots * sizeof(uint64_t));
        std::memcpy(total_out, total_dev, sizeof(double));
        return QVNT_OK;
    }
    const double* u_dev = nullptr;
    if (shots > 1) {
        QVNT_HIP(hipMemcpyAsync(r->dscratch + 1, u, shots * sizeof(double), hipMemcpyHostToDevice, r->stream));
        u_dev = r->dscratch + 1;
    }
    double* total_dev = reinterpret_cast<double*>(r->iscratch + shots);
    rc = sample_into(r, r->tree, count, u_dev, shots > 1 ? 0.0 : u[0], shots, r->iscratch, total_dev, true);
    if (rc) return rc;
    std::vector<uint64_t> words(shots + 1);
    QVNT_HIP(hipMemcpyAsync(words.data(), r->iscratch, (shots + 1) * sizeof(uint64_t), hipMemcpyDeviceToHost, r->stream));
    QVNT_HIP(hipStreamSynchronize(r->stream));
    std::memcpy(out, words.data(), shots * sizeof(uint64_t));
    std::memcpy(total_out, words.data() + shots, sizeof(double));
    return QVNT_OK;
}

int collapse(qvnt_reg* r, uint64_t outcome, uint64_t mask, bool renorm) {
    {
        const uint64_t nb = (r->len + kBlock - 1) / kBlock;
        const dim3 grid((unsigned)(nb < kMaxGrid ? nb : kMaxGrid));
        Timed t(r, QVNT_K_COLLAPSE, 2.0 * (double)r->amp_bytes() * (double)r->len);
        if (r->prec == QVNT_F64)
            hipLaunchKernelGGL(k_collapse<double>, grid, dim3(kBlock), 0, r->stream, static_cast<c64*>(r->psi), r->len, outcome, mask);
        else
            hipLaunchKernelGGL(k_collapse<float>, grid, dim3(kBlock), 0, r->stream, static_cast<c32*>(r->psi), r->len, outcome, mask);
        QVNT_HIP(hipGetLastError());
    }
    if (!renorm) return QVNT_OK;
    double kept = 0.0;
    int rc = tree_build(r, r->len, &kept);
    if (rc) return rc;
    if (!(kept > 0.0) || !std::isfinite(kept)) return fail(QVNT_E_ZERO_NORM, "collapsed state has zero norm");
    const double scale = 1.0 / std::sqrt(kept);
    Deposit d{};
    d.zeros = mask;
    d.n = popc(mask);
    d.set = outcome & mask;
    const uint64_t groups = r->len >> d.n;
    const uint64_t nb = (groups + kBlock - 1) / kBlock;
    const dim3 grid((unsigned)(nb < kMaxGrid ? nb : kMaxGrid));
    Timed t(r, QVNT_K_COLLAPSE, 2.0 * (double)r->amp_bytes() * (double)groups);
    if (r->prec == QVNT_F64)
        hipLaunchKernelGGL(k_rescale<double>, grid, dim3(kBlock), 0, r->stream, static_cast<c64*>(r->psi), groups, d, scale);
    else
        hipLaunchKernelGGL(k_rescale<float>, grid, dim3(kBlock), 0, r->stream, static_cast<c32*>(r->psi), groups, d, scale);
    QVNT_HIP(hipGetLastError());
    return QVNT_OK;
}

int rescale(qvnt_reg* r, double scale) {
    const Deposit d{};  // no fixed bits: every amplitude of the buffer
    const uint64_t nb = (r->len + kBlock - 1) / kBlock;
    const dim3 grid((unsigned)(nb < kMaxGrid ? nb : kMaxGrid));
    Timed t(r, QVNT_K_COLLAPSE, 2.0 * (double)r->amp_bytes() * (double)r->len);
    if (r->prec == QVNT_F64)
        hipLaunchKernelGGL(k_rescale<double>, grid, dim3(kBlock), 0, r->stream, static_cast<c64*>(r->psi), r->len, d, scale);
    else
        hipLaunchKernelGGL(k_rescale<float>, grid, dim3(kBlock), 0, r->stream, static_cast<c32*>(r->psi), r->len, d, scale);
    QVNT_HIP(hipGetLastError());
    return QVNT_OK;
}

int probabilities(qvnt_reg* r, double inv_total, double* dst, uint64_t n) {
    // To pinned memory the staging buffer and one copy win above 256 KiB: 512
    // KiB 46 us, through the ring 48; 1 MiB 55 and 64, 8 MiB 193 and 303.
    const Memory at = memory_of(dst);
    const bool copy = at == Memory::Device || (at == Memory::Pinned && n * sizeof(double) > kHostChunk / 2);
    const int done = copy ? kNoBlock : read_back(r, dst, n * sizeof(double), [&](void* block, size_t off, size_t bytes) {
        const uint64_t first = off / sizeof(double), m = bytes / sizeof(double);
        const dim3 grid((unsigned)((m + kBlock - 1) / kBlock));
        if (r->prec == QVNT_F64)
            hipLaunchKernelGGL(k_probs<double>, grid, dim3(kBlock), 0, r->stream, static_cast<const c64*>(r->psi) + first, m, inv_total,
                               static_cast<double*>(block));
        else
            hipLaunchKernelGGL(k_probs<float>, grid, dim3(kBlock), 0, r->stream, static_cast<const c32*>(r->psi) + first, m, inv_total,
                               static_cast<double*>(block));
        return hipGetLastError();
    });
    if (done != kNoBlock) return done;
    // bounded device staging: chunks of up to 2^24 probabilities
    const uint64_t chunk = n < (1ull << 24) ? n : (1ull << 24);
    void* vbuf = nullptr;
    if (dev_alloc(r->device, &vbuf, chunk * sizeof(double)) != QVNT_OK)
        return fail(QVNT_E_OOM, "probability staging buffer");
    double* buf = static_cast<double*>(vbuf);
    int rc = QVNT_OK;
    for (uint64_t off = 0; off < n && rc == QVNT_OK; off += chunk) {
        const uint64_t m = (n - off) < chunk ? (n - off) : chunk;
        const dim3 grid((unsigned)((m + kBlock - 1) / kBlock));
        if (r->prec == QVNT_F64)
            hipLaunchKernelGGL(k_probs<double>, grid, dim3(kBlock), 0, r->stream, static_cast<const c64*>(r->psi) + off, m, inv_total, buf);
        else
            hipLaunchKernelGGL(k_probs<float>, grid, dim3(kBlock), 0, r->stream, static_cast<const c32*>(r->psi) + off, m, inv_total, buf);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipMemcpyAsync(dst + off, buf, m * sizeof(double), hipMemcpyDeviceToHost, r->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(r->stream);
        if (e != hipSuccess) rc = fail(QVNT_E_HIP, std::string("probabilities: ") + hipGetErrorString(e));
    }
    // (every chunk ended with a synchronization; after a failure, wait here)
    if (rc != QVNT_OK) (void)hipStreamSynchronize(r->stream);
    dev_release(r->device, buf, chunk * sizeof(double));
    return rc;
}

int compare(qvnt_reg* a, qvnt_reg* b, double* out) {
    const uint64_t len = a->len;
    const unsigned blocks = (unsigned)((len + 4095) / 4096);
    QVNT_HIP(hipStreamSynchronize(b->stream));
    void* vpart = nullptr;
    if (dev_alloc(a->device, &vpart, (size_t)blocks * 5 * sizeof(double)) != QVNT_OK)
        return fail(QVNT_E_OOM, "comparison partials");
    double* part = static_cast<double*>(vpart);
    if (a->prec == QVNT_F64 && b->prec == QVNT_F64) launch_compare<double, double>(a->psi, b->psi, len, part, blocks, a->stream);
    else if (a->prec == QVNT_F64) launch_compare<double, float>(a->psi, b->psi, len, part, blocks, a->stream);
    else if (b->prec == QVNT_F64) launch_compare<float, double>(a->psi, b->psi, len, part, blocks, a->stream);
    else launch_compare<float, float>(a->psi, b->psi, len, part, blocks, a->stream);
    std::vector<double> host((size_t)blocks * 5);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(host.data(), part, host.size() * sizeof(double), hipMemcpyDeviceToHost, a->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(a->stream);
    if (e != hipSuccess) (void)hipStreamSynchronize(a->stream);
    dev_release(a->device, part, (size_t)blocks * 5 * sizeof(double));
    if (e != hipSuccess) return fail(QVNT_E_HIP, std::string("compare: ") + hipGetErrorString(e));
    double s[5] = {0, 0, 0, 0, 0};
    for (unsigned k = 0; k < blocks; ++k) {
        for (int q = 0; q < 4; ++q) s[q] += host[(size_t)k * 5 + q];
        s[4] = std::max(s[4], host[(size_t)k * 5 + 4]);
    }
    for (int q = 0; q < 5; ++q) out[q] = s[q];
    return QVNT_OK;
}

}  // namespace qvnt

// ------------------------------------------------ allocation-free shots
// qvnt_reg_sample_mask_noalloc: the shots of qvnt_reg_sample_mask with the
// tree levels, draws, outcomes and total in `scratch`, a file-scope device
// array of kScratchBytes that every GPU the library runs on holds until the
// process ends.  In host code `scratch` names a host-side stand-in, not a
// device address: the device address comes from hipGetSymbolAddress, taken
// once per device with that device current and kept in g_scratch.  Every
// call on one GPU shares that GPU's array, so calls that overlap on one GPU
// race.  Nothing in it needs to start at zero: each call writes the levels,
// the draws, every outcome and the total before reading them.
namespace qvnt {
namespace {

constexpr size_t kScratchBytes = size_t(16) << 20;  // 16 MiB: registers up to 30 qubits
constexpr int kMaxDevices = 64;

__device__ __align__(256) unsigned char scratch[kScratchBytes];

std::mutex g_scratch_mu;
void* g_scratch[kMaxDevices] = {};

int scratch_address(int device, unsigned char** out) {
    if (device < 0 || device >= kMaxDevices) return fail(QVNT_E_ARG, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[device]) {
        int cur = 0;
        QVNT_HIP(hipGetDevice(&cur));
        if (cur != device) QVNT_HIP(hipSetDevice(device));
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess || !p)
            return fail(QVNT_E_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch[device] = p;
    }
    *out = static_cast<unsigned char*>(g_scratch[device]);
    return QVNT_OK;
}

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

}  // namespace
}  // namespace qvnt

extern "C" int qvnt_reg_sample_mask_noalloc(qvnt_reg* r, uint64_t mask, const double* u, size_t shots, uint64_t* out) {
    using namespace qvnt;
    if (!r) return fail(QVNT_E_ARG, "null register");
    if (shots == 0) return QVNT_OK;
    if (!u || !out) return fail(QVNT_E_ARG, "null draws or outcomes");
    if (shots > (1u << 20)) return fail(QVNT_E_ARG, "at most 2^20 shots per call");
    mask &= (1ull << r->q_num) - 1u;
    if (mask == 0) {
        for (size_t k = 0; k < shots; ++k) out[k] = 0;
        return QVNT_OK;
    }
    for (size_t k = 0; k < shots; ++k)
        if (!(u[k] >= 0.0 && u[k] < 1.0)) return fail(QVNT_E_ARG, "draws must lie in [0, 1)");
    // workspace layout: [tree levels | total | draws | outcomes], 256-byte aligned
    const uint64_t count = 1ull << r->q_num;
    const size_t off_total = align256(tree_doubles(count) * sizeof(double));
    const size_t off_u = off_total + 256;
    const size_t off_out = off_u + align256(shots * sizeof(double));
    const size_t need = off_out + align256(shots * sizeof(uint64_t));
    if (need > kScratchBytes)
        return fail(QVNT_E_ARG, "allocation-free shots need " + std::to_string(need) + " bytes of workspace; the "
                                "fixed workspace holds " + std::to_string(kScratchBytes) +
                                " (registers up to 30 qubits, fewer shots at 30)");
    unsigned char* ws = nullptr;
    if (int rc = scratch_address(r->device, &ws)) return rc;
    double* tree = reinterpret_cast<double*>(ws);
    double* total_dev = reinterpret_cast<double*>(ws + off_total);
    double* u_dev = reinterpret_cast<double*>(ws + off_u);
    uint64_t* out_dev = reinterpret_cast<uint64_t*>(ws + off_out);
    QVNT_HIP(hipMemcpyAsync(u_dev, u, shots * sizeof(double), hipMemcpyHostToDevice, r->stream));
    if (int rc = sample_into(r, tree, count, u_dev, 0.0, shots, out_dev, total_dev, false)) return rc;
    double total = 0.0;
    QVNT_HIP(hipMemcpyAsync(out, out_dev, shots * sizeof(uint64_t), hipMemcpyDeviceToHost, r->stream));
    QVNT_HIP(hipMemcpyAsync(&total, total_dev, sizeof(double), hipMemcpyDeviceToHost, r->stream));
    QVNT_HIP(hipStreamSynchronize(r->stream));
    if (!(total > 0.0) || !std::isfinite(total)) return fail(QVNT_E_ZERO_NORM, "measurement of a zero-norm or non-finite state");
    for (size_t k = 0; k < shots; ++k) out[k] &= mask;
    return QVNT_OK;
}
