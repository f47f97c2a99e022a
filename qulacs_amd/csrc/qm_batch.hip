// Batched executor: many small circuits, each run from |0...0> and reduced to
// the expectation value of its observable, in one launch.
//
// What it replaces: for each circuit, QuantumCircuit::update_quantum_state
// (src/cppsim/circuit.cpp:46-57, one kernel launch and synchronisation per gate
// on the GPU backend) and Observable::get_expectation_value
// (src/cppsim/observable.cpp:56-58 -> general_quantum_operator.cpp:105-141, one
// reduction per term).
//
// Design:
//   * one work-group (1024 threads, 512 at K = 4) per circuit, circuits taken from a queue
//     (an atomic counter) in descending-cost order, so one launch covers a batch
//     of uneven sizes; every work-group leaves the loop once the queue is empty;
//   * the state lives in LDS: 2^lq complex128 with lq = min(n, 13) (128 KiB at
//     13 qubits); circuits of 14..20 qubits keep the state in device memory and
//     are processed in 2^13-amplitude tiles, one "stage" at a time: a stage is a
//     set of gates whose qubits all lie in one 13-qubit window (qubits 0..3 are
//     always in the window, so a tile is made of 256-byte contiguous runs);
//   * inside a stage the gates are grouped into passes: each pass names K
//     "block" qubits; a thread loads the 2^K amplitudes that differ in those
//     bits into registers, applies every gate of the pass (dense gates on block
//     qubits, diagonal gates and CZ on any local qubits) and writes them back,
//     so one LDS round trip serves several gates;
//   * LDS slots are XOR-swizzled (slot = i ^ fold3(i)) so that the 16-byte
//     accesses of a wave spread over the banks whichever block bits a pass uses;
//     fold3 is linear over GF(2), so slot(base | off) = slot(base) ^ slot(off);
//   * the observable sum_k c_k <P_k> is reduced per work-group in a fixed order
//     (deterministic), with P_k in the mask form of the reference
//     (src/csim/utility.cpp:12-43): P|x> = i^rot (-1)^popcount(x & pf) |x ^ bf>.
//
// Scheduling (host): gates are scanned in order; a gate joins the current
// stage / pass unless it touches a qubit of a gate skipped earlier in the same
// scan (then it is skipped too and its qubits are blocked) or it does not fit
// the window / block.  A gate is therefore only moved ahead of gates it
// commutes with trivially (disjoint qubits), and every scan schedules at least
// its first gate.
#include <cstring>

#include "qm_tile.hpp"

namespace qm {
namespace {

// Work-group size per register-block width: 8 waves at K = 4 (the register
// block limits a SIMD to 2 waves), 16 waves below, so a CU holding one
// 128 KiB tile still has 4 waves per SIMD to hide LDS latency.
template <int K>
constexpr u32 block_threads() { return K >= 4 ? 512u : 1024u; }
constexpr u32 kMaxBlockThreads = 1024;
struct DCirc {
    u32 n, lq, nstage, stage0, term0, nterm;
    u64 state_off;  // complex128 offset of the circuit's state in the scratch buffer
};
// This thread's share of sum_k c_k Re <psi|P_k|psi>, reading the state from LDS
// (swizzled slots) or from device memory.
template <bool FROM_LDS>
__device__ __forceinline__ double energy_sum(const double2* __restrict__ gs, const double2* st, const DCirc& c,
                                             const DTerm* __restrict__ terms) {
    double acc = 0.0;
    const u64 dim = 1ULL << c.n;
    for (u64 x = threadIdx.x; x < dim; x += blockDim.x) {
        const double2 px = FROM_LDS ? st[slot_of((u32)x)] : gs[x];
        for (u32 k = 0; k < c.nterm; ++k) {
            const DTerm tm = terms[c.term0 + k];
            const u64 y = x ^ tm.bf;
            const double2 py = FROM_LDS ? st[slot_of((u32)y)] : gs[y];  // y == x when bf == 0
            // psi_x * conj(psi_y) * i^rot * (-1)^popcount(x & pf)
            const double re0 = px.x * py.x + px.y * py.y, im0 = px.y * py.x - px.x * py.y;
            double re;
            switch (tm.rot & 3u) {
                case 0: re = re0; break;
                case 1: re = -im0; break;
                case 2: re = -re0; break;
                default: re = im0; break;
            }
            if (__popcll(x & tm.pf) & 1) re = -re;
            acc = fma(tm.coef, re, acc);
        }
    }
    return acc;
}

__global__ void k_batch_reset(int* counter) {
    if (threadIdx.x == 0) *counter = 0;
}

// Tiles of one stage of a batched circuit held in device memory (every stage
// after the first), the next tile loaded into registers while the passes run
// on the current one.  P amplitudes per thread, T threads.  The loop is laid
// out as in stage_tiles: unconditional loads of the next tile at the top, the
// LDS fill from them after the stores of the current tile.
constexpr u32 kBatchTile = 1u << kMaxLocal;
template <int K, u32 P, u32 T, int G>
__device__ __forceinline__ void batch_tiles(double2* st, double2* __restrict__ gs, const u32* hi_tab, u32 lq, u32 tl,
                                            const DStage& sg, const DPass* __restrict__ passes,
                                            const DSub* __restrict__ subs, const double2* __restrict__ pool) {
    const u32 tid = threadIdx.x, ntiles = 1u << tl;
    {
        const u64 tb = tile_base(0, tl, sg);
#pragma unroll
        for (u32 k = 0; k < P; ++k) st[slot_of(tid + k * T)] = gs[tile_index(tb, hi_tab, tid + k * T)];
        __syncthreads();
    }
    for (u32 t = 0;; ++t) {
        double rx[P], ry[P];
        const bool more = t + 1 < ntiles;
        {
            const u64 tb = tile_base(t + 1, tl, sg);
#pragma unroll
            for (u32 k = 0; k < P; ++k) {
                const double2 a = gs[more ? tile_index(tb, hi_tab, tid + k * T) : 0];
                rx[k] = a.x;
                ry[k] = a.y;
            }
        }
        run_passes<K, T, G>(st, lq, passes, sg.pass0, sg.npass, subs, pool);
        const u64 tb = tile_base(t, tl, sg);
#pragma unroll
        for (u32 k = 0; k < P; ++k) gs[tile_index(tb, hi_tab, tid + k * T)] = st[slot_of(tid + k * T)];
        __syncthreads();
        if (!more) break;
#pragma unroll
        for (u32 k = 0; k < P; ++k) st[slot_of(tid + k * T)] = make_double2(rx[k], ry[k]);
        __syncthreads();
    }
}

// The program arrays arrive as separate read-only, non-aliasing arguments so the
// compiler reads them through the scalar cache (inside a by-value struct they
// became per-lane vector loads).
template <int K>
__global__ __launch_bounds__(block_threads<K>()) void k_batch(
    const DCirc* __restrict__ circs, const DStage* __restrict__ stages, const DPass* __restrict__ passes,
    const DSub* __restrict__ subs, const double2* __restrict__ pool, const DTerm* __restrict__ terms,
    const u32* __restrict__ order, double2* __restrict__ scratch, double* __restrict__ energies, int* counter,
    u32 ncirc, int keep) {
    extern __shared__ double2 st[];
    __shared__ u32 hi_tab[1u << (kMaxLocal - kLowFixed)];
    __shared__ double red[16];
    __shared__ int s_slot;
    const u32 tid = threadIdx.x, bd = blockDim.x;

    for (;;) {
        if (tid == 0) s_slot = atomicAdd(counter, 1);
        __syncthreads();
        const int slot = s_slot;
        __syncthreads();
        if (slot >= (int)ncirc) break;  // uniform: every thread read the same slot
        const u32 ci = order[slot];
        const DCirc c = circs[ci];
        const u32 lq = c.lq, L = 1u << lq, tl = c.n - lq;
        double2* gs = scratch + c.state_off;

        for (u32 s = 0; s < c.nstage; ++s) {
            const DStage sg = stages[c.stage0 + s];
            if (tl > 0) {
                build_hi_tab(hi_tab, lq, sg);
                __syncthreads();
            }
            if (tl > 0 && s > 0 && L == kBatchTile) {
                // one register block per thread (two measured slower here)
                batch_tiles<K, kBatchTile / block_threads<K>(), block_threads<K>(), 1>(st, gs, hi_tab, lq, tl,
                                                                                        sg, passes, subs, pool);
                continue;
            }
            for (u32 t = 0; t < (1u << tl); ++t) {
                const u64 tb = tile_base(t, tl, sg);
                if (s == 0) {
                    // |0...0>: slot_of(0) == 0 and amplitude 0 lies in tile 0
                    for (u32 i = tid; i < L; i += bd) st[i] = make_double2((i == 0 && t == 0) ? 1.0 : 0.0, 0.0);
                } else {
                    for (u32 i = tid; i < L; i += bd) st[slot_of(i)] = gs[tile_index(tb, hi_tab, i)];
                }
                __syncthreads();
                run_passes<K, block_threads<K>(), 1>(st, lq, passes, sg.pass0, sg.npass, subs, pool);
                if (tl > 0) {
                    for (u32 i = tid; i < L; i += bd) gs[tile_index(tb, hi_tab, i)] = st[slot_of(i)];
                } else if (keep) {
                    for (u32 i = tid; i < L; i += bd) gs[i] = st[slot_of(i)];
                }
                __syncthreads();
            }
        }

        // sum_k c_k Re <psi| P_k |psi>
        const double acc = tl ? energy_sum<false>(gs, st, c, terms) : energy_sum<true>(gs, st, c, terms);
        const double total = block_sum(acc, red);
        if (tid == 0) energies[ci] = total;
        __syncthreads();
    }
}

// One stage of a single-state circuit: every work-group takes tiles of 2^lq
// amplitudes (grid-stride), runs the stage's passes on each in LDS and writes
// it back in place.  Tiles of one stage are disjoint, so work-groups never
// touch the same amplitudes.  The next tile is loaded into registers while the
// passes run on the current one (a barrier does not wait for global loads), so
// the HBM traffic of consecutive tiles overlaps the arithmetic.
//
// Work-group size and register blocks per thread: at K = 3, 512 threads with
// two 8-amplitude blocks each (a 13-qubit tile is 1024 groups), so every
// sub-operation is decoded once per two blocks and the FP64 chains of the two
// interleave; K = 2: 1024 threads with two 4-amplitude blocks; K = 4: 512
// threads with one 16-amplitude block.
template <int K>
constexpr u32 stage_threads() { return K == 2 ? 1024u : 512u; }
template <int K>
constexpr int stage_blocks() { return K <= 3 ? 2 : 1; }

// Tiles of exactly P * T amplitudes, P per thread, with prefetch.  Each
// iteration issues the loads of the next tile, runs the passes on the tile in
// LDS, stores it and only then moves the prefetched registers into LDS, so the
// wait for the loads follows the stores in program order and lets the stores
// stay in flight (the vector memory counter returns in order); with the LDS
// fill at the top of the loop the compiler's wait there has to hold for the
// first entry too and would drain the previous tile's stores.  The loads are
// unconditional (after the last tile every lane reads amplitude 0, one cache
// line, and the values are not used): a conditional load merged with the old
// values makes the compiler copy the loaded registers, i.e. wait, at once.
template <int K, u32 P, u32 T = stage_threads<K>()>
__device__ __forceinline__ void stage_tiles(double2* __restrict__ state, double2* st, const u64* hi_tab, u32 lq, u32 tl,
                                            const DStage& sg, const DPass* __restrict__ passes,
                                            const DSub* __restrict__ subs, const double2* __restrict__ pool) {
    const u32 tid = threadIdx.x;
    const u64 ntiles = 1ULL << tl;
    u64 t = blockIdx.x;
    if (t >= ntiles) return;
    {
        const u64 tb = tile_base(t, tl, sg);
#pragma unroll
        for (u32 k = 0; k < P; ++k) st[slot_of(tid + k * T)] = state[tile_index(tb, hi_tab, tid + k * T)];
        __syncthreads();
    }
    for (;;) {
        double rx[P], ry[P];  // the prefetched tile (separate scalars keep it in registers)
        const u64 tn = t + gridDim.x;
        const bool more = tn < ntiles;
        {
            const u64 tb = tile_base(tn, tl, sg);
#pragma unroll
            for (u32 k = 0; k < P; ++k) {
                const double2 x = state[more ? tile_index(tb, hi_tab, tid + k * T) : 0];
                rx[k] = x.x;
                ry[k] = x.y;
            }
        }
        run_passes<K, T, stage_blocks<K>()>(st, lq, passes, sg.pass0, sg.npass, subs, pool);
        const u64 tb = tile_base(t, tl, sg);
#pragma unroll
        for (u32 k = 0; k < P; ++k) state[tile_index(tb, hi_tab, tid + k * T)] = st[slot_of(tid + k * T)];
        if (!more) break;
        __syncthreads();  // the tile has been read out of LDS
#pragma unroll
        for (u32 k = 0; k < P; ++k) st[slot_of(tid + k * T)] = make_double2(rx[k], ry[k]);
        __syncthreads();
        t = tn;
    }
}

template <int K>
__global__ __launch_bounds__(stage_threads<K>()) void k_stage(double2* __restrict__ state, u32 lq, u32 tl, DStage sg,
                                                         const DPass* __restrict__ passes,
                                                         const DSub* __restrict__ subs,
                                                         const double2* __restrict__ pool) {
    extern __shared__ double2 st[];
    __shared__ u64 hi_tab[1u << (kMaxLocal - kLowFixed)];  // offsets of states above 32 qubits exceed 32 bits
    const u32 L = 1u << lq;
    build_hi_tab(hi_tab, lq, sg);
    __syncthreads();
    constexpr u32 T = stage_threads<K>();
    // the prefetched tile needs 4 P registers per thread on top of the register
    // blocks (at K = 4: 64 beside ~165, within the 256 of a 512-thread group)
    if constexpr (K >= 3) {
        if (L == 16 * T) {
            stage_tiles<K, 16>(state, st, hi_tab, lq, tl, sg, passes, subs, pool);
            return;
        }
    }
    if constexpr (K <= 3) {
        if (L == 8 * T) {
            stage_tiles<K, 8>(state, st, hi_tab, lq, tl, sg, passes, subs, pool);
            return;
        }
        if (L == 4 * T) {
            stage_tiles<K, 4>(state, st, hi_tab, lq, tl, sg, passes, subs, pool);
            return;
        }
    }
    const u64 ntiles = 1ULL << tl;
    for (u64 t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const u64 tb = tile_base(t, tl, sg);
        for (u32 i = threadIdx.x; i < L; i += T) st[slot_of(i)] = state[tile_index(tb, hi_tab, i)];
        __syncthreads();
        run_passes<K, T, stage_blocks<K>()>(st, lq, passes, sg.pass0, sg.npass, subs, pool);
        for (u32 i = threadIdx.x; i < L; i += T) state[tile_index(tb, hi_tab, i)] = st[slot_of(i)];
        __syncthreads();
    }
}

template <class T>
bool dev_upload(T** dst, const std::vector<T>& src) {
    *dst = nullptr;
    if (src.empty()) return true;
    if (!hip_ok(hipMalloc((void**)dst, src.size() * sizeof(T)), "qm_batch_compile: hipMalloc")) return false;
    return hip_ok(hipMemcpy(*dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice),
                  "qm_batch_compile: hipMemcpy");
}

// Grows *dst to hold `bytes` (contents not kept); capacity in *cap.
bool dev_reserve(void** dst, size_t* cap, size_t bytes, const char* what) {
    if (*cap >= bytes && *dst) return true;
    if (*dst) {
        if (!hip_ok(hipFree(*dst), what)) return false;
        *dst = nullptr;
        *cap = 0;
    }
    if (!hip_ok(hipMalloc(dst, std::max<size_t>(bytes, 256)), what)) return false;
    *cap = std::max<size_t>(bytes, 256);
    return true;
}

template <class T>
bool dev_put(T** dst, size_t* cap, const std::vector<T>& src, const char* what) {
    if (!dev_reserve((void**)dst, cap, src.size() * sizeof(T), what)) return false;
    return src.empty() || hip_ok(hipMemcpy(*dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice), what);
}

}  // namespace
}  // namespace qm

struct qm_batch {
    std::vector<qm::HCirc> circs;
    // compiled
    int device = -1;
    unsigned K = 0;
    int keep = 0;
    unsigned lq_max = 0;
    std::vector<qm::DCirc> h_circs;
    qm::u64 n_stages = 0, n_passes = 0, n_subs = 0;
    qm::DCirc* d_circs = nullptr;
    qm::DStage* d_stages = nullptr;
    qm::DPass* d_passes = nullptr;
    qm::DSub* d_subs = nullptr;
    double2* d_pool = nullptr;
    qm::DTerm* d_terms = nullptr;
    qm::u32* d_order = nullptr;
    double2* d_scratch = nullptr;
    double* d_energies = nullptr;
    int* d_counter = nullptr;
    size_t cap[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};  // bytes held by each device buffer above
    int grid = 0;                       // work-groups of the launch (computed once per compile)
    unsigned lq_cap = 13;               // qubits held in LDS per tile (qm_batch_set_local_qubits)
    hipGraph_t graph = nullptr;         // captured launch (qm_batch_capture)
    hipGraphExec_t graph_exec = nullptr;
    void drop_graph() {
        if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
        if (graph) (void)hipGraphDestroy(graph);
        graph_exec = nullptr;
        graph = nullptr;
    }

    void release() {
        drop_graph();
        grid = 0;
        if (device >= 0) {
            (void)hipSetDevice(device);
            void* ptrs[] = {d_circs, d_stages, d_passes, d_subs, d_pool, d_terms, d_order, d_scratch, d_energies, d_counter};
            for (void* p : ptrs)
                if (p) (void)hipFree(p);
        }
        d_circs = nullptr; d_stages = nullptr; d_passes = nullptr; d_subs = nullptr; d_pool = nullptr;
        d_terms = nullptr; d_order = nullptr; d_scratch = nullptr; d_energies = nullptr; d_counter = nullptr;
        for (size_t& c : cap) c = 0;
        device = -1;
        h_circs.clear();
    }
};

struct qm_circuit {
    unsigned n = 0, K = 4, lq = 13;
    std::vector<qm::DStage> stages;
    std::vector<qm::DPass> passes;
    std::vector<qm::DSub> subs;
    std::vector<double2> pool;
    int device = -1;
    int per_cu = 0, cus = 0;
    qm::DPass* d_passes = nullptr;
    qm::DSub* d_subs = nullptr;
    double2* d_pool = nullptr;
    void release() {
        if (device >= 0) {
            (void)hipSetDevice(device);
            void* ptrs[] = {d_passes, d_subs, d_pool};
            for (void* p : ptrs)
                if (p) (void)hipFree(p);
        }
        d_passes = nullptr; d_subs = nullptr; d_pool = nullptr;
        device = -1;
        per_cu = 0;
    }
};

namespace qm {
namespace {

// Sets the kernel's LDS limit and sizes the grid (resident work-groups, at most
// one per circuit).  Kept out of the launch path so a graph capture only sees
// stream operations.
bool batch_prepare_launch(qm_batch* b, unsigned dev, const char* what) {
    const size_t lds = sizeof(double2) << b->lq_max;
    const void* fn = b->K == 2 ? (const void*)k_batch<2> : b->K == 3 ? (const void*)k_batch<3> : (const void*)k_batch<4>;
    if (!hip_ok(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), what)) return false;
    int per_cu = 0, cus = 0;
    const int threads = (int)(b->K == 2 ? block_threads<2>() : b->K == 3 ? block_threads<3>() : block_threads<4>());
    if (!hip_ok(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, threads, lds), what)) return false;
    if (!hip_ok(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, (int)dev), what)) return false;
    if (per_cu < 1) {
        set_error(QM_ERR_HIP, "%s: the kernel does not fit a compute unit with %zu bytes of LDS", what, lds);
        return false;
    }
    b->grid = (int)std::min<u64>(b->h_circs.size(), (u64)per_cu * cus);
    return true;
}

bool batch_ok(qm_batch* b, const char* what) {
    if (!b) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: null batch", what);
        return false;
    }
    return true;
}

}  // namespace
}  // namespace qm

using namespace qm;

extern "C" {

qm_batch* qm_batch_create(void) { return new qm_batch(); }

void qm_batch_destroy(qm_batch* b) {
    if (!b) return;
    b->release();
    delete b;
}

int qm_batch_add_circuit(qm_batch* b, UINT n, const qm_batch_gate* gates, UINT gate_count, const ITYPE* bf,
                         const ITYPE* pf, const UINT* rot, const double* coefs, UINT term_count) {
    const char* what = "qm_batch_add_circuit";
    if (!batch_ok(b, what)) return -1;
    if (n < 1 || n > QM_BATCH_MAX_QUBITS) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: qubit count %u outside 1..%u", what, n, QM_BATCH_MAX_QUBITS);
        return -1;
    }
    if ((gate_count && !gates) || (term_count && (!bf || !pf || !rot || !coefs))) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: null gate or term array", what);
        return -1;
    }
    HCirc c;
    if (!convert_gates(n, gates, gate_count, c, what)) return -1;
    for (UINT t = 0; t < term_count; ++t) {
        if ((bf[t] >> n) || (pf[t] >> n)) {
            set_error(QM_ERR_INVALID_ARGUMENT, "%s: term %u acts beyond %u qubits", what, t, n);
            return -1;
        }
        DTerm tm{};
        tm.bf = bf[t];
        tm.pf = pf[t];
        tm.rot = rot[t];
        tm.coef = coefs[t];
        c.terms.push_back(tm);
    }
    b->circs.push_back(std::move(c));
    return (int)b->circs.size() - 1;
}

int qm_batch_compile(qm_batch* b, UINT block_qubits, int keep_states, unsigned dev) {
    const char* what = "qm_batch_compile";
    if (!batch_ok(b, what)) return QM_ERR_INVALID_ARGUMENT;
    const u32 K = block_qubits ? block_qubits : 4;
    if (K < 2 || K > 4) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: block_qubits %u outside 2..4", what, K);
        return QM_ERR_INVALID_ARGUMENT;
    }
    for (const HCirc& c : b->circs)
        for (const HOp& o : c.ops)
            if (o.type == 0 && o.q.size() > K) {
                set_error(QM_ERR_INVALID_ARGUMENT, "%s: a %zu-qubit dense gate needs block_qubits >= %zu", what,
                          o.q.size(), o.q.size());
                return QM_ERR_INVALID_ARGUMENT;
            }
    if (b->device >= 0 && b->device != (int)dev) b->release();
    b->drop_graph();  // device buffers and the queue length may change
    b->grid = 0;
    b->h_circs.clear();
    if (!use_device(dev)) return QM_ERR_HIP;
    Flat f;    std::vector<DTerm> terms;
    std::vector<DCirc> dc;
    u64 state_off = 0;
    u32 lq_max = kMinQubits;
    for (const HCirc& c : b->circs) {
        DCirc d{};
        d.n = c.ne;
        d.lq = std::min(c.ne, (u32)b->lq_cap);
        d.stage0 = (u32)f.stages.size();
        d.nstage = schedule_circuit(f, c, K, b->lq_cap);
        d.term0 = (u32)terms.size();
        d.nterm = (u32)c.terms.size();
        terms.insert(terms.end(), c.terms.begin(), c.terms.end());
        d.state_off = state_off;
        if (c.ne > b->lq_cap || keep_states) state_off += 1ULL << c.ne;
        lq_max = std::max(lq_max, d.lq);
        dc.push_back(d);
    }
    // descending cost: amplitudes x (passes + terms)
    std::vector<u32> order(dc.size());
    std::vector<double> cost(dc.size());
    for (size_t i = 0; i < dc.size(); ++i) {
        u64 np = 0;
        for (u32 s = 0; s < dc[i].nstage; ++s) np += f.stages[dc[i].stage0 + s].npass;
        cost[i] = std::ldexp(1.0, (int)dc[i].n) * (double)(np + dc[i].nterm + 1);
        order[i] = (u32)i;
    }
    std::stable_sort(order.begin(), order.end(), [&](u32 x, u32 y) { return cost[x] > cost[y]; });
    if (f.pool.empty()) f.pool.push_back(make_double2(0, 0));
    if (f.subs.empty()) f.subs.push_back(DSub{});
    if (f.passes.empty()) f.passes.push_back(DPass{});
    if (terms.empty()) terms.push_back(DTerm{});
    b->device = (int)dev;
    bool ok = dev_put(&b->d_circs, &b->cap[0], dc, what) && dev_put(&b->d_stages, &b->cap[1], f.stages, what) &&
              dev_put(&b->d_passes, &b->cap[2], f.passes, what) && dev_put(&b->d_subs, &b->cap[3], f.subs, what) &&
              dev_put(&b->d_pool, &b->cap[4], f.pool, what) && dev_put(&b->d_terms, &b->cap[5], terms, what) &&
              dev_put(&b->d_order, &b->cap[6], order, what);
    if (ok && state_off) {
        ok = dev_reserve((void**)&b->d_scratch, &b->cap[7], state_off * sizeof(double2), what);
        if (!ok) set_error(QM_ERR_OUT_OF_MEMORY, "%s: %llu bytes of state memory", what, state_off * 16ULL);
    }
    if (ok) ok = dev_reserve((void**)&b->d_energies, &b->cap[8], std::max<size_t>(1, dc.size()) * sizeof(double), what);
    if (ok) ok = dev_reserve((void**)&b->d_counter, &b->cap[9], sizeof(int), what);
    if (!ok) {
        b->release();
        return QM_ERR_HIP;
    }
    b->K = K;
    b->keep = keep_states ? 1 : 0;
    b->lq_max = lq_max;
    b->h_circs = dc;
    b->n_stages = f.stages.size();
    b->n_passes = 0;
    for (const DStage& s : f.stages) b->n_passes += s.npass;
    b->n_subs = 0;
    for (const DPass& p : f.passes) b->n_subs += p.nsub;
    return QM_OK;
}

const double* qm_batch_run_async(qm_batch* b, void* stream, unsigned dev) {
    const char* what = "qm_batch_run";
    if (!batch_ok(b, what)) return nullptr;
    if (b->device < 0 || b->device != (int)dev) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: batch not compiled for device %u", what, dev);
        return nullptr;
    }
    if (!use_device(dev)) return nullptr;
    hipStream_t st = stream_of(stream);
    const u32 ncirc = (u32)b->h_circs.size();
    if (ncirc == 0) return b->d_energies;
    const size_t lds = sizeof(double2) << b->lq_max;
    if (b->grid == 0 && !batch_prepare_launch(b, dev, what)) return nullptr;
    const u32 grid = (u32)b->grid;
#define QM_BATCH_ARGS                                                                                       \
    b->d_circs, b->d_stages, b->d_passes, b->d_subs, b->d_pool, b->d_terms, b->d_order, b->d_scratch, b->d_energies, \
        b->d_counter, ncirc, b->keep
    k_batch_reset<<<1, 64, 0, st>>>(b->d_counter);
    switch (b->K) {
        case 2: k_batch<2><<<grid, block_threads<2>(), lds, st>>>(QM_BATCH_ARGS); break;
        case 3: k_batch<3><<<grid, block_threads<3>(), lds, st>>>(QM_BATCH_ARGS); break;
        default: k_batch<4><<<grid, block_threads<4>(), lds, st>>>(QM_BATCH_ARGS); break;
    }
#undef QM_BATCH_ARGS
    if (!hip_ok(hipGetLastError(), what)) return nullptr;
    return b->d_energies;
}

int qm_batch_run(qm_batch* b, double* energies, void* stream, unsigned dev) {
    const double* d = qm_batch_run_async(b, stream, dev);
    if (!d) return QM_ERR_HIP;
    hipStream_t st = stream_of(stream);
    const size_t n = b->h_circs.size();
    if (n && energies) {
        if (!hip_ok(hipMemcpyAsync(energies, d, n * sizeof(double), hipMemcpyDeviceToHost, st), "qm_batch_run"))
            return QM_ERR_HIP;
    }
    if (!hip_ok(hipStreamSynchronize(st), "qm_batch_run")) return QM_ERR_HIP;
    return QM_OK;
}

int qm_batch_get_state(qm_batch* b, UINT index, qm_complex* out, void* stream, unsigned dev) {
    const char* what = "qm_batch_get_state";
    if (!batch_ok(b, what)) return QM_ERR_INVALID_ARGUMENT;
    if (!b->keep || index >= b->h_circs.size() || !out || b->device != (int)dev) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: no kept state %u (compile with keep_states, then run)", what, index);
        return QM_ERR_INVALID_ARGUMENT;
    }
    if (!use_device(dev)) return QM_ERR_HIP;
    hipStream_t st = stream_of(stream);
    const DCirc& c = b->h_circs[index];
    const u32 n = b->circs[index].n;  // the circuit's own size: extra qubits stay |0>, so the state is the prefix
    if (!hip_ok(hipMemcpyAsync(out, b->d_scratch + c.state_off, sizeof(double2) << n, hipMemcpyDeviceToHost, st), what))
        return QM_ERR_HIP;
    if (!hip_ok(hipStreamSynchronize(st), what)) return QM_ERR_HIP;
    return QM_OK;
}

int qm_batch_capture(qm_batch* b, void* stream, unsigned dev) {
    const char* what = "qm_batch_capture";
    if (!batch_ok(b, what)) return QM_ERR_INVALID_ARGUMENT;
    if (!stream || b->device != (int)dev || b->h_circs.empty()) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: needs a compiled, non-empty batch and a created stream", what);
        return QM_ERR_INVALID_ARGUMENT;
    }
    if (!use_device(dev)) return QM_ERR_HIP;
    if (b->grid == 0 && !batch_prepare_launch(b, dev, what)) return QM_ERR_HIP;
    b->drop_graph();
    hipStream_t st = stream_of(stream);
    if (!hip_ok(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal), what)) return QM_ERR_HIP;
    const double* d = qm_batch_run_async(b, stream, dev);
    hipGraph_t g = nullptr;
    const bool ended = hip_ok(hipStreamEndCapture(st, &g), what);
    if (!d || !ended || !g) {
        if (g) (void)hipGraphDestroy(g);
        return QM_ERR_HIP;
    }
    b->graph = g;
    if (!hip_ok(hipGraphInstantiate(&b->graph_exec, g, nullptr, nullptr, 0), what)) {
        b->drop_graph();
        return QM_ERR_HIP;
    }
    return QM_OK;
}

int qm_batch_run_graph(qm_batch* b, double* energies, void* stream, unsigned dev) {
    const char* what = "qm_batch_run_graph";
    if (!batch_ok(b, what)) return QM_ERR_INVALID_ARGUMENT;
    if (!b->graph_exec || b->device != (int)dev) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: capture the batch first (qm_batch_capture)", what);
        return QM_ERR_INVALID_ARGUMENT;
    }
    if (!use_device(dev)) return QM_ERR_HIP;
    hipStream_t st = stream_of(stream);
    if (!hip_ok(hipGraphLaunch(b->graph_exec, st), what)) return QM_ERR_HIP;
    const size_t n = b->h_circs.size();
    if (energies && n &&
        !hip_ok(hipMemcpyAsync(energies, b->d_energies, n * sizeof(double), hipMemcpyDeviceToHost, st), what))
        return QM_ERR_HIP;
    if (!hip_ok(hipStreamSynchronize(st), what)) return QM_ERR_HIP;
    return QM_OK;
}

int qm_batch_set_local_qubits(qm_batch* b, UINT local_qubits) {
    if (!batch_ok(b, "qm_batch_set_local_qubits")) return QM_ERR_INVALID_ARGUMENT;
    if (local_qubits < 8 || local_qubits > kMaxLocal) {
        set_error(QM_ERR_INVALID_ARGUMENT, "qm_batch_set_local_qubits: %u outside 8..%u", local_qubits, kMaxLocal);
        return QM_ERR_INVALID_ARGUMENT;
    }
    b->lq_cap = local_qubits;
    return QM_OK;
}

void qm_batch_clear(qm_batch* b) {
    if (!b) return;
    b->circs.clear();
    b->h_circs.clear();
}

void* qm_batch_state_device_ptr(qm_batch* b, UINT index) {
    if (!b || !b->keep || index >= b->h_circs.size()) {
        set_error(QM_ERR_INVALID_ARGUMENT, "qm_batch_state_device_ptr: no kept state %u", index);
        return nullptr;
    }
    return b->d_scratch + b->h_circs[index].state_off;
}

qm_circuit* qm_circuit_create(UINT n, const qm_batch_gate* gates, UINT gate_count, UINT block_qubits,
                              UINT local_qubits) {
    const char* what = "qm_circuit_create";
    // Defaults (0): up to 19 qubits a 13-qubit window leaves at most 64 tiles
    // per stage for 256 CUs; 12-qubit windows with 3-qubit blocks were 11-28 %
    // faster there on brickwork circuits (13 q: 0.198 -> 0.149 ms, 14 q: 0.130
    // -> 0.093 ms, 18 q: 0.179 -> 0.133 ms; 10-12 q, one stage: 15-20 % from the
    // block width alone), equal at 20 and slower from 21 qubits up.
    const bool small_state = n <= 19;
    u32 K = block_qubits ? block_qubits : (small_state ? 3 : 4);
    const u32 lq = local_qubits ? local_qubits : (small_state ? 12 : kMaxLocal);
    if (n < kMinQubits || n > QM_CIRCUIT_MAX_QUBITS || K < 2 || K > 4 || lq < 8 || lq > kMaxLocal ||
        (gate_count && !gates)) {
        set_error(QM_ERR_INVALID_ARGUMENT,
                  "%s: need %u <= qubits (%u) <= %u, block_qubits (%u) in 2..4, local_qubits (%u) in 8..%u and a gate array",
                  what, kMinQubits, n, QM_CIRCUIT_MAX_QUBITS, K, lq, kMaxLocal);
        return nullptr;
    }
    auto* c = new qm_circuit();
    HCirc hc;
    if (!convert_gates(n, gates, gate_count, hc, what)) {
        delete c;
        return nullptr;
    }
    if (!block_qubits)  // the default width widens to the largest dense gate (at most 4 qubits)
        for (const HOp& o : hc.ops)
            if (o.type == 0 && o.q.size() > K && o.q.size() <= 4) K = (u32)o.q.size();
    for (const HOp& o : hc.ops)
        if (o.type == 0 && o.q.size() > K) {
            set_error(QM_ERR_INVALID_ARGUMENT, "%s: a %zu-qubit dense gate needs block_qubits >= %zu", what, o.q.size(),
                      o.q.size());
            delete c;
            return nullptr;
        }
    c->n = n;
    c->K = K;
    c->lq = std::min(n, lq);
    Flat f;
    schedule_circuit(f, hc, K, lq);
    c->stages = f.stages;
    c->passes = f.passes;
    c->subs = f.subs;
    c->pool = f.pool;
    if (c->pool.empty()) c->pool.push_back(make_double2(0, 0));
    if (c->subs.empty()) c->subs.push_back(DSub{});
    if (c->passes.empty()) c->passes.push_back(DPass{});
    return c;
}

void qm_circuit_destroy(qm_circuit* c) {
    if (!c) return;
    c->release();
    delete c;
}

int qm_circuit_apply(qm_circuit* c, void* state, ITYPE dim, void* stream, unsigned dev) {
    const char* what = "qm_circuit_apply";
    if (!c || !state || dim != (1ULL << c->n)) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: null circuit/state or dim is not 2^%u", what, c ? c->n : 0u);
        return QM_ERR_INVALID_ARGUMENT;
    }
    if (!use_device(dev)) return QM_ERR_HIP;
    hipStream_t st = stream_of(stream);
    if (!qm::circuit_enqueue(c, state, dim, st, dev)) return QM_ERR_HIP;
    finish_update(st, what);
    return QM_OK;
}

}  // extern "C"

namespace qm {
bool circuit_prepare(qm_circuit* c, unsigned dev) {
    if (c->device != (int)dev) {
        c->release();
        bool ok = dev_upload(&c->d_passes, c->passes) && dev_upload(&c->d_subs, c->subs) &&
                  dev_upload(&c->d_pool, c->pool);
        if (!ok) {
            c->release();
            return false;
        }
        c->device = (int)dev;
    }
    return true;
}

bool circuit_enqueue(qm_circuit* c, void* state, u64 dim, hipStream_t st, unsigned dev) {
    const char* what = "qm_circuit_apply";
    if (!c || !state || dim != (1ULL << c->n)) {
        set_error(QM_ERR_INVALID_ARGUMENT, "%s: null circuit/state or dim is not 2^%u", what, c ? c->n : 0u);
        return false;
    }
    if (!circuit_prepare(c, dev)) return false;
    const size_t lds = sizeof(double2) << c->lq;
    const void* fn = c->K == 2 ? (const void*)k_stage<2> : c->K == 3 ? (const void*)k_stage<3> : (const void*)k_stage<4>;
    if (c->per_cu == 0) {
        int per_cu = 0, cus = 0;
        if (!hip_ok(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), what) ||
            !hip_ok(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, (int)(c->K == 2 ? stage_threads<2>() : c->K == 3 ? stage_threads<3>() : stage_threads<4>()), lds), what) ||
            !hip_ok(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, (int)dev), what))
            return false;
        if (per_cu < 1) {
            set_error(QM_ERR_HIP, "%s: the kernel does not fit a compute unit with %zu bytes of LDS", what, lds);
            return false;
        }
        c->per_cu = per_cu;
        c->cus = cus;
    }
    const u32 tl = c->n - c->lq;
    const u64 ntiles = 1ULL << tl;
    const u32 grid = (u32)std::min<u64>(ntiles, (u64)c->per_cu * c->cus);
    for (const DStage& sg : c->stages) {
        if (sg.npass == 0) continue;
        switch (c->K) {
            case 2: k_stage<2><<<grid, stage_threads<2>(), lds, st>>>((double2*)state, c->lq, tl, sg, c->d_passes, c->d_subs, c->d_pool); break;
            case 3: k_stage<3><<<grid, stage_threads<3>(), lds, st>>>((double2*)state, c->lq, tl, sg, c->d_passes, c->d_subs, c->d_pool); break;
            default: k_stage<4><<<grid, stage_threads<4>(), lds, st>>>((double2*)state, c->lq, tl, sg, c->d_passes, c->d_subs, c->d_pool); break;
        }
    }
    return hip_ok(hipGetLastError(), what);
}
}  // namespace qm

extern "C" {

void qm_circuit_stats(const qm_circuit* c, ITYPE* stages, ITYPE* passes, ITYPE* subops) {
    ITYPE np = 0, ns = 0;
    if (c)
        for (const DStage& sg : c->stages) {
            np += sg.npass;
            for (u32 p = 0; p < sg.npass; ++p) ns += c->passes[sg.pass0 + p].nsub;
        }
    if (stages) *stages = c ? c->stages.size() : 0;
    if (passes) *passes = np;
    if (subops) *subops = ns;
}

void qm_batch_stats(const qm_batch* b, ITYPE* circuits, ITYPE* stages, ITYPE* passes, ITYPE* subops) {
    if (circuits) *circuits = b ? b->circs.size() : 0;
    if (stages) *stages = b ? b->n_stages : 0;
    if (passes) *passes = b ? b->n_passes : 0;
    if (subops) *subops = b ? b->n_subs : 0;
}

}  // extern "C"
