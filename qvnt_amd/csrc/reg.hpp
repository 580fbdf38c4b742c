// The device register (the reference's QReg, src/register/quant.rs:103-108)
// and the launch helpers shared by the HIP translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstring>
#include <string>
#include <vector>

#include "common.hpp"

#define QVNT_HIP(call)                                                                       \
    do {                                                                                     \
        hipError_t qvnt_e_ = (call);                                                         \
        if (qvnt_e_ != hipSuccess)                                                           \
            return ::qvnt::fail(QVNT_E_HIP, std::string(#call) + ": " + hipGetErrorString(qvnt_e_)); \
    } while (0)

struct qvnt_reg {
    uint32_t q_num = 0;      // qubits of the register
    uint32_t ns = 0;         // storage qubits: log2(len) = max(q_num, 3)
    uint64_t len = 0;        // stored amplitudes, max(2^q_num, 8) (quant.rs:15,116)
    qvnt_prec prec = QVNT_F64;
    int device = 0;
    void* psi = nullptr;     // device amplitudes, interleaved complex
    hipStream_t stream = nullptr;

    // measurement workspace: stored levels of the |psi|^2 pairwise tree
    double* tree = nullptr;
    size_t tree_cap = 0;     // doubles
    double* dscratch = nullptr;      // small device scratch (draws, totals)
    uint64_t* iscratch = nullptr;    // small device scratch: shots_cap outcomes + the total
    size_t shots_cap = 0;

    // fused-form program (phases, micro-ops, coefficients) on the device
    void* prog = nullptr;
    size_t prog_cap = 0;
    uint32_t dense_min = 0;  // fused form: phases of >= this many ops run as dense 16x16 (0: never)

    // per-kernel-class timing
    bool owns_memory = true;  // false: state, workspace and stream belong to a server slot
    bool timing = false;
    struct Pending { int kclass; hipEvent_t a, b; double bytes; };
    std::vector<Pending> pending;
    std::vector<hipEvent_t> event_pool;
    qvnt_kstats stats[QVNT_KCLASS_COUNT] = {};

    size_t amp_bytes() const { return prec == QVNT_F64 ? 16 : 8; }
};

namespace qvnt {

// Brackets one launch with timing events when the register has timing on.
struct Timed {
    qvnt_reg* r;
    int kclass;
    double bytes;
    hipEvent_t a = nullptr, b = nullptr;
    Timed(qvnt_reg* reg, int kc, double by);
    ~Timed();
};

// reg.hip: device blocks and streams that registers reuse.  Creating and
// destroying a stream and allocating and freeing the state and workspace
// cost more than the gates of a short-lived register (a 20-qubit register
// with a few gates and a measurement: most of ~290 us).  dev_alloc returns a
// cached block of exactly `bytes` of the device (current) or a new one;
// dev_release keeps a block of at most kCacheBlock bytes while the
// device's cache holds at most kCacheTotal, and frees the rest.  The caller
// of dev_release guarantees that no queued work still uses the block (its
// stream synchronized).  An allocation that fails frees every cached block
// of the device and tries once more.  stream_acquire / stream_release do
// the same for idle streams (default priority, non-blocking).
constexpr size_t kCacheBlock = size_t(64) << 20;
constexpr size_t kCacheTotal = size_t(256) << 20;
int dev_alloc(int device, void** p, size_t bytes);
void dev_release(int device, void* p, size_t bytes);
// HostBlock: a block of exactly `bytes` of pinned host memory for one call,
// that kernels read and write directly; p is null when there is none (0
// bytes, or the allocation failed).  The blocks are cached per device like the
// others, at most kHostTotal of them.  The owner's stream is synchronized
// before it ends, or, where that failed, keep_out() keeps the block from
// being used again.
constexpr size_t kHostSmall = size_t(64) << 10;
constexpr size_t kHostTotal = size_t(32) << 20;
struct HostBlock {
    int device;
    size_t bytes;
    void* p = nullptr;
    HostBlock(int device, size_t bytes);
    ~HostBlock();
    HostBlock(const HostBlock&) = delete;
    HostBlock& operator=(const HostBlock&) = delete;
    void keep_out() { p = nullptr; }
};
int stream_acquire(int device, hipStream_t* s);
void stream_release(int device, hipStream_t s);

// Where the caller's destination lies.  Device memory (managed memory with
// it) takes a copy of the runtime's, as no host thread may write it; pinned
// memory the same, from the size on where one copy over the bus beats the ring
// below and its second copy by a host thread.
enum class Memory { Pageable, Pinned, Device };
Memory memory_of(const void* p);

// `bytes` of results from the register's stream to pageable memory:
// fill(block, offset, n) enqueues the next n of them into a pinned block.
// Several blocks, so that one is copied to dst while the next ones fill.  The runtime's
// own copy to pageable memory does one after the other: 20 qubits FP64,
// probabilities 8 MiB 510 us, state 16 MiB 950 us; so 310 and 540 (the bus
// alone: 155 and 310), in pieces of 256 KiB 400 and 730, of 1 MiB 390 and 670.
// 10 qubits: 51 and 28 us, so 26 and 13.  (States of 32 to 512 KiB take the
// runtime 3 to 4 us less once it has its copy queue, 10.5 and 14.4 us for 32
// KiB; making the queue takes the process's first call 6 ms.)
// kNoBlock: no pinned memory, nothing done.
constexpr size_t kHostChunk = size_t(512) << 10;
constexpr int kNoBlock = -1;
constexpr int kHostRing = 4;
template <class Fill>
int read_back(qvnt_reg* r, void* dst, size_t bytes, const Fill& fill) {
    const size_t chunk = bytes <= kHostSmall ? kHostSmall : kHostChunk, chunks = (bytes + chunk - 1) / chunk;
    const auto size_for = [&](size_t k) { return k < chunks ? chunk : 0; };
    HostBlock ring[kHostRing] = {{r->device, size_for(0)}, {r->device, size_for(1)}, {r->device, size_for(2)}, {r->device, size_for(3)}};
    size_t depth = 0;
    while (depth < kHostRing && ring[depth].p) ++depth;
    if (depth < (chunks < 2 ? chunks : 2)) return kNoBlock;
    unsigned char* to = static_cast<unsigned char*>(dst);
    hipEvent_t full[kHostRing] = {};
    hipError_t e = hipSuccess;
    for (size_t k = 0; k < depth && chunks > 1 && e == hipSuccess; ++k) e = hipEventCreateWithFlags(&full[k], hipEventDisableTiming);
    const auto size = [&](size_t c) { return c + 1 < chunks ? chunk : bytes - c * chunk; };
    for (size_t asked = 0, c = 0; c < chunks && e == hipSuccess; ++c) {
        for (; asked < chunks && asked < c + depth && e == hipSuccess; ++asked) {
            e = fill(ring[asked % depth].p, asked * chunk, size(asked));
            if (e == hipSuccess && chunks > 1) e = hipEventRecord(full[asked % depth], r->stream);
        }
        if (e == hipSuccess) e = chunks > 1 ? hipEventSynchronize(full[c % depth]) : hipStreamSynchronize(r->stream);
        if (e == hipSuccess) std::memcpy(to + c * chunk, ring[c % depth].p, size(c));
    }
    if (e != hipSuccess && hipStreamSynchronize(r->stream) != hipSuccess)
        for (HostBlock& h : ring) h.keep_out();
    for (hipEvent_t ev : full)
        if (ev) (void)hipEventDestroy(ev);
    return e == hipSuccess ? QVNT_OK : fail(QVNT_E_HIP, std::string("copy to the host: ") + hipGetErrorString(e));
}

// plain.hip
// Validates a gate against a buffer of `len` amplitudes (bit counts, control
// overlap, qubits beyond the buffer); *noop is set for gates that are the
// identity there (Id, a control bit beyond the buffer).
int check_gate(uint64_t len, const qvnt_gate& g, bool* noop);
int launch_gate(qvnt_reg* r, const qvnt_gate& g);
int launch_init(qvnt_reg* r, uint64_t state);

// runs.hip: a validated queue in the plain form: runs of SingleOps in one
// pass each (runs.hpp), the others through launch_gate
int apply_plain(qvnt_reg* r, const qvnt_gate* g, size_t n);

// measure.hip
int tree_build(qvnt_reg* r, uint64_t count, double* total_out);
int tree_sample(qvnt_reg* r, uint64_t count, const double* u, size_t shots, uint64_t* out, double* total_out);
// doubles of tree workspace the draws over `count` weights need
size_t tree_doubles(uint64_t count);
// enqueues the tree levels and one draw per u_dev[k] into out_dev (device
// pointers; r->tree must hold tree_doubles(count)); no synchronisation
int sample_launch(qvnt_reg* r, uint64_t count, const double* u_dev, size_t shots, uint64_t* out_dev, double* total_dev);
int collapse(qvnt_reg* r, uint64_t outcome, uint64_t mask, bool renorm);
int probabilities(qvnt_reg* r, double inv_total, double* dst, uint64_t n);
// every amplitude of the buffer times `scale` (FP64 multiply)
int rescale(qvnt_reg* r, double scale);
int compare(qvnt_reg* a, qvnt_reg* b, double* out);

// fused.hip
int apply_fused(qvnt_reg* r, const qvnt_gate* g, size_t n, uint32_t max_qubits, uint32_t* passes);
// the steps of a fused apply on 2^ns (>= 2^kMinFused) amplitudes (host
// only; returns the tile size): the tile the run-time model picks when
// max_qubits = 0 and dense_min = 0 from 28 qubits, else max_qubits (0: the
// default) clamped to the precision's LDS tile and the buffer
namespace fusion { struct Step; }
unsigned compile_fused(const qvnt_gate* g, size_t n, unsigned ns, bool fp64, uint32_t max_qubits, uint32_t dense_min,
                       std::vector<fusion::Step>& steps);
// what apply_fused would compile for a buffer of 2^ns amplitudes (host
// only): out = {passes, tile qubits, summed op cost, dense phases}
void fused_plan_stats(const qvnt_gate* g, size_t n, unsigned ns, bool fp64, uint32_t max_qubits, uint32_t dense_min,
                      double* out);
namespace fusion { struct Program; }
size_t program_bytes(const fusion::Program& prog);
void pack_program(const fusion::Program& prog, unsigned char* host);
int launch_program(qvnt_reg* r, const fusion::Program& prog, const void* dev);
namespace fusion { struct BItem; }
// one batched launch: `blocks` tiles of 2^t amplitudes (block -> item by map)
int launch_batch(hipStream_t stream, qvnt_prec prec, void* arena, const void* prog, const fusion::BItem* items,
                 const uint32_t* map, uint32_t t, uint32_t blocks);
namespace fusion { struct PUnit; }
// the persistent batched kernel: blocks resident at once for tiles up to
// 2^tmax, and its cooperative launch over `rounds` rounds of work units
// (units [round_begin[r], round_begin[r+1]) form round r; device pointers)
int batch_persist_grid(qvnt_prec prec, uint32_t tmax, uint32_t* blocks);
// (status: 1 + rounds device words, zero at the first launch: the kernel
// sets status[0] to 1 if its launch was not cooperative, and uses
// status[1 + r] as round r's claim counter, leaving it zero; graph
// non-null: capture the launch into *graph instead of running it)
int launch_batch_persist(hipStream_t stream, qvnt_prec prec, void* arena, const void* prog, const fusion::BItem* items,
                         const fusion::PUnit* units, const uint32_t* round_begin, uint32_t rounds, uint32_t tmax,
                         uint32_t blocks, uint32_t* status, hipGraph_t* graph);

}  // namespace qvnt
